"""Particle ranges of the tree's cells on both sides of the cell count from which
8 lanes instead of a wavefront search a cell's end, and for leaves at the edges
of the search's first round (64 particles) and of its steps: every leaf holds its
particles, every other cell its children's, exactly."""
import numpy as np
import pytest

from lsmps_vpm_v2_amd import FmmSolver, workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cap,many", [
    (2, 1, False), (2000, 1, False), (30000, 15, False), (150000, 63, False), (150000, 64, False),
    (300000, 129, False), (60000, 6, True), (60000, 17, True), (300000, 15, True),
    (250000, 63, True), (900000, 64, True), (1200000, 129, True)])
def test_ranges_add_up(gpu, n, cap, many):
    f = W.random_clusters(n, seed=cap, active_frac=0.9)
    s = FmmSolver(max_par=cap, max_src=cap)
    print(f"ranges n={n} max_par={cap}", flush=True)
    s.field(f["x"], f["y"], f["q"], f["active"])
    c = s.tree_cells()
    assert (len(c["id"]) > 8192) == many
    lid, poff, pidx = s.tree_leaves(n)
    assert np.array_equal(np.sort(pidx), np.arange(n))
    leaf = c["is_leaf"] != 0
    pos = {int(i): k for k, i in enumerate(c["id"])}
    rows = np.array([pos[int(i)] for i in lid])
    assert leaf.sum() == len(lid) and leaf[rows].all()
    assert np.array_equal(c["par_num"][rows], np.diff(poff))
    act = np.concatenate([[0], np.cumsum(f["active"][pidx] != 0)])
    assert np.array_equal(c["src_num"][rows], np.diff(act[poff]))
    # a cell's parent: one level up, half the indices
    key = lambda L, x, y: (L.astype(np.int64) << 40) | (x.astype(np.int64) << 20) | y
    k = key(c["level"], c["ix"], c["iy"])
    order = np.argsort(k)
    sub = c["level"] > 0
    up = key(c["level"][sub] - 1, c["ix"][sub] >> 1, c["iy"][sub] >> 1)
    par = order[np.searchsorted(k[order], up)]
    assert np.array_equal(k[par], up)
    for name in ("par_num", "src_num"):
        got = np.bincount(par, weights=c[name][sub], minlength=len(k)).astype(np.int64)
        assert np.array_equal(got[~leaf], c[name][~leaf])
