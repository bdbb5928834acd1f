"""Fields whose cells are smaller than the list tests' absolute tolerance (1e-9):
every cell below a leaf's neighbours is adjacent to it, and a tree of unequal leaves
has more list-1 entries than the 17 per leaf that the arrays hold.  Such a call is
refused, and leaves the handle as it should be."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _field(scale):
    g = np.random.default_rng(1)
    n = 700
    r, t = 10.0 ** g.uniform(-4, 0, n), g.uniform(0, 2 * np.pi, n)
    return scale * r * np.cos(t), scale * r * np.sin(t), np.full(n, 0.01 * scale), \
        g.standard_normal(n), np.ones(n, np.uint8)


KW = dict(max_par=8, max_src=8)


@pytest.mark.parametrize("call", ["fp64", "gauss", "mixed", "potential", "type1"])
def test_too_many_list_entries_are_refused(gpu, oracle, call):
    from lsmps_vpm_v2_amd import FmmSolver, VpmFmmError
    x, y, s, q, a = _field(1e-100)
    if call != "type1":
        t = oracle.Tree(x, y, a, oracle.opts(**KW))
        c = t.cells()
        leaves = c["id"][c["is_leaf"] != 0]
        assert sum(len(t.int_list(i)[0]) for i in leaves) > 17 * len(leaves) + 1
    print(f"list capacity {call}", flush=True)
    solver = FmmSolver(precision="mixed" if call == "mixed" else "fp64",
                       icutoff=2 if call == "gauss" else 0,
                       binom_mode=0 if call == "mixed" else 1, **KW)

    def run(x, y, s, q, a):
        if call == "potential":
            return [solver.potential(x, y, q, a)]
        if call == "type1":
            return solver.velocity_type1(x, y, s, q, n_s=8, lmax=12)
        return solver.velocity(x, y, s, q, a)

    with pytest.raises(VpmFmmError) as e:
        run(x, y, s, q, a)
    assert e.value.status == "INTERNAL"
    with pytest.raises(VpmFmmError):
        solver.tree_cells()  # no lists to inspect
    for out in run(*_field(1.0)):
        assert np.isfinite(out).all()
    assert len(solver.tree_cells()["id"]) > 0
