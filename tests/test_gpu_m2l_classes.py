"""The M2L of the FP64 and type-1 paths on the matrix cores: every order it takes
(each shape of its tiles), trees under and over the size at which a workgroup
takes one class instead of four, fields whose classes hold more targets than a
workgroup takes in one round (cells along a line, along the diagonal) and whose
sources exceed the rows staged in LDS (a full grid at order 16: 12 x 8 cells
have 252 sources, 210 rows fit).  Against the oracle, 1e-10 relative as the
other FP64 parity tests (the same sums in another order; measured under 1e-13)."""
import numpy as np
import pytest

from lsmps_vpm_v2_amd import FmmSolver

pytestmark = pytest.mark.gpu
TOL = 1e-10


def _rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(b))


def _field(kind, n):
    rng = np.random.default_rng(n)
    x, y = rng.random(n), rng.random(n)
    if kind == "line":
        y = 1e-3 * y
    elif kind == "diagonal":
        y = x + 1e-3 * y
    return x, y, np.full(n, 1e-4), rng.standard_normal(n), np.ones(n, np.uint8)


def _workgroups(solver):
    """96 cells of a level each; from 65 on a workgroup takes all four classes."""
    level = solver.tree_cells()["level"]
    return sum(-(-int(np.sum(level == k)) // 96) for k in range(2, 17))


def _check(oracle, f, many, **kw):
    print(f"classes n={len(f[0])} {kw}", flush=True)
    solver = FmmSolver(**kw)
    u, v = solver.velocity(*f)
    assert (_workgroups(solver) > 64) == many
    u0, v0 = oracle.velocity(*f, oracle.opts(**kw), 1.0, 0.0)
    assert _rel(u, u0) <= TOL and _rel(v, v0) <= TOL


@pytest.mark.parametrize("kind", ["grid", "line", "diagonal"])
@pytest.mark.parametrize("p", range(1, 17))
def test_orders_match_oracle(gpu, oracle, kind, p):
    _check(oracle, _field(kind, 3000), False, p=p, max_par=2, max_src=2, max_level=12)


@pytest.mark.parametrize("kind", ["grid", "line", "diagonal"])
@pytest.mark.parametrize("p", [3, 10, 12, 13, 16])
def test_larger_trees_match_oracle(gpu, oracle, kind, p):
    _check(oracle, _field(kind, 12000), True, p=p, max_par=2, max_src=2, max_level=14)


@pytest.mark.parametrize("kind,n", [("grid", 3000), ("line", 3000), ("grid", 12000)])
@pytest.mark.parametrize("ndp", [1, 2, 7, 8, 12, 13, 15, 16])
def test_type1_orders_match_oracle(gpu, oracle, kind, n, ndp):
    x, y, s, g, _ = _field(kind, n)
    kw = dict(n_s=2, lmax=10, ndp=ndp, icutoff=2, l2l_mode=0)
    print(f"classes type 1 {kind} n={n} {kw}", flush=True)
    solver = FmmSolver(u_inf=0.0, v_inf=0.0)
    u, v = solver.velocity_type1(x, y, s, g, **kw)
    assert (_workgroups(solver) > 64) == (n > 3000)
    u0, v0 = oracle.t1_velocity(x, y, s, g, oracle.t1_opts(**kw))
    assert _rel(u, u0) <= TOL and _rel(v, v0) <= TOL
