"""The mixed upward and downward passes on both sides of the depth (three levels
below the first one of 1024 cells) up to which subtrees are walked by a workgroup, against the FP64 path (held to the
oracle by its own tests) on a jittered lattice, even or graded towards its middle
(subtrees of very different size): FP32 rounding of the pairs, kept 0.4 spacings
apart, and expansions, rel-L2 <= 5e-6 as the other mixed tests."""
import numpy as np
import pytest

from lsmps_vpm_v2_amd import FmmSolver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,graded,deep", [(200, False, False), (300, False, False),
                                           (500, False, True), (200, True, True),
                                           (500, True, True)])
@pytest.mark.parametrize("p", [3, 8, 16])
def test_tiers_match_fp64(gpu, m, graded, deep, p):
    rng = np.random.default_rng(m)
    g = (np.stack(np.divmod(np.arange(m * m), m)) + 0.5 + 0.6 * (rng.random((2, m * m)) - 0.5)) / m
    if graded:
        g = (2 * g - 1) ** 3 + 0.01 * (2 * g - 1)
    q, act = rng.standard_normal(m * m), (rng.random(m * m) < 0.9).astype(np.uint8)
    kw = dict(p=p, max_par=4, max_src=4, binom_mode=0, list4_mode=2)
    print(f"tiers m={m} p={p} graded={graded}", flush=True)
    s = FmmSolver(precision="mixed", **kw)
    ex, ey = s.field(g[0], g[1], q, act)
    cells = np.bincount(s.tree_cells()["level"])
    assert (len(cells) - 1 - np.argmax(cells >= 1024) > 3) == deep
    ex0, ey0 = FmmSolver(**kw).field(g[0], g[1], q, act)
    err = np.sqrt(np.sum((ex - ex0) ** 2 + (ey - ey0) ** 2) / np.sum(ex0 ** 2 + ey0 ** 2))
    print(f"  {err:.2e}")
    assert err <= 5e-6
