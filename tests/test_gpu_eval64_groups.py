"""The FP64 evaluation at the edges of its groups (leaves of up to 8, 16, 32,
64 and more particles), of its 128-source rounds, and on both sides of the
number of leaves up to which four wavefronts share a leaf: velocity, regularized
velocity and potential against the oracle, 1e-10 relative as the other FP64
parity tests (the same FP64 sums in another order; measured under 1e-14)."""
import numpy as np
import pytest

from lsmps_vpm_v2_amd import FmmSolver, VpmFmmError, workloads as W

pytestmark = pytest.mark.gpu
TOL = 1e-10


def _rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(b))


MANY = 8192  # leaves up to which four wavefronts share one
CASES = [(7, 4), (700, 7), (700, 8), (700, 9), (900, 16), (900, 17), (1500, 32), (1500, 33),
         (3000, 64), (3000, 65), (3000, 130), (4000, 300), (60001, 8)]


@pytest.mark.parametrize("n,cap", CASES, ids=[f"{n}-{c}" for n, c in CASES])
def test_groups_match_oracle(gpu, oracle, n, cap):
    f = W.random_clusters(n, seed=n + cap, active_frac=0.9)
    print(f"eval64 n={n} max_par={cap}", flush=True)
    kw = dict(max_par=cap, max_src=cap)
    a = [f[k] for k in ("x", "y", "s", "omega", "active")]
    for icut in (0, 1, 2, 3):
        solver = FmmSolver(icutoff=icut, u_inf=0.0, **kw)
        u, v = solver.velocity(*a)
        assert (solver.stats()["n_leaves"] > MANY) == (n > 60000)
        u0, v0 = oracle.velocity(*a, oracle.opts(icutoff=icut, **kw), 0.0, 0.0)
        assert _rel(np.hypot(u - u0, v - v0) + np.hypot(u0, v0), np.hypot(u0, v0)) <= TOL
    b = [f[k] for k in ("x", "y", "q", "active")]
    phi = FmmSolver(**kw).potential(*b)
    assert _rel(phi, oracle.fmm_potential(*b, oracle.opts(**kw))) <= TOL


@pytest.mark.parametrize("n", [3000, 60001])
def test_strength_that_is_not_finite_is_no_duplicate(gpu, n):
    """A NaN strength is not a DUPLICATE_POINTS error, and does not reach the
    particle that carries it through its own pair."""
    f = W.random_clusters(n, seed=3)
    w = f["omega"].copy()
    w[n // 3] = np.nan
    # one tree level, so that everything is near field, or many small leaves
    cap = 4096 if n < 4096 else 8
    for icut in (0, 2):
        s = FmmSolver(max_par=cap, max_src=cap, icutoff=icut)
        u, v = s.velocity(f["x"], f["y"], f["s"], w, f["active"])
        assert (s.stats()["n_leaves"] > MANY) == (n > 60000)
        bad = np.isnan(u)
        assert bad.any() and not bad[n // 3]


@pytest.mark.parametrize("n", [3000, 60001])
@pytest.mark.parametrize("strengths", ["both", "one", "none", "opposite"])
def test_duplicates_are_found(gpu, n, strengths):
    """Two particles at one point, whatever their strengths: the error and not a
    NaN, from the field and the potential; apart, neither."""
    f = W.random_clusters(n, seed=3)
    x, y, q = f["x"].copy(), f["y"].copy(), f["q"].copy()
    i, k = n // 3, n // 2
    x[k], y[k] = x[i], y[i]
    q[i], q[k] = dict(both=(1.0, 2.0), one=(0.0, 1.0), none=(0.0, 0.0),
                      opposite=(1.0, -1.0))[strengths]
    s = FmmSolver(max_par=8, max_src=8)
    print(f"duplicates n={n} {strengths}", flush=True)
    for call in (s.field, s.potential):
        with pytest.raises(VpmFmmError) as e:
            call(x, y, q, f["active"])
        assert e.value.status == "DUPLICATE_POINTS"
        assert np.isfinite(call(f["x"], f["y"], q, f["active"])).all()
        assert (s.stats()["n_leaves"] > MANY) == (n > 60000)


def test_sizes_of_zero(gpu, oracle):
    """Gaussian near field of point particles: the factor is 1."""
    f = W.random_clusters(2000, seed=9)
    z = np.zeros_like(f["s"])
    z[::2] = f["s"][::2]
    a = [f["x"], f["y"], z, f["omega"], f["active"]]
    u, v = FmmSolver(icutoff=2).velocity(*a)
    u0, v0 = oracle.velocity(*a, oracle.opts(icutoff=2), 1.0, 0.0)
    assert np.isfinite(u).all() and _rel(u, u0) <= TOL and _rel(v, v0) <= TOL


@pytest.mark.parametrize("n,cap", [(5, 7), (700, 9), (60001, 8)])
@pytest.mark.parametrize("icut", [1, 2, 3])
def test_single_size_of_zero(gpu, oracle, icut, n, cap):
    """A point particle among blobs, the last of its leaf (of a source round, whose
    padding follows it): every velocity is finite."""
    f = W.random_clusters(n, seed=cap, active_frac=1.0)
    solver = FmmSolver(max_par=cap, max_src=cap, icutoff=icut)
    a = [f["x"], f["y"], f["s"].copy(), f["omega"], f["active"]]
    solver.velocity(*a)
    _, poff, pidx = solver.tree_leaves(n)
    last = pidx[poff[1:] - 1]
    for k in last[:: max(1, len(last) // 3)]:
        print(f"point particle {k} of {n}, icutoff={icut}", flush=True)
        a[2] = f["s"].copy()
        a[2][k] = 0.0
        u, v = solver.velocity(*a)
        u0, v0 = oracle.velocity(*a, oracle.opts(icutoff=icut, max_par=cap, max_src=cap), 1.0, 0.0)
        assert bool(np.isfinite(u0).all()) and bool(np.isfinite(u).all())
        assert _rel(u, u0) <= TOL and _rel(v, v0) <= TOL
