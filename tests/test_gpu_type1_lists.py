"""Type-1 list-2 M2L where the rounding of the box bounds shows.

Sources beside their target: the type-1 box tests compare bounds that are rounded level by level, against an
absolute tolerance of 1e-15.  Where two neighbouring boxes' bounds part by more
than that, the reference calls the boxes well separated and forms their whole
interaction by M2L, at a distance of one box side.  On the fields here this
holds along a whole row of level-3 boxes (a box that straddles the origin rounds
its upper bound away from its neighbour's), which the test asserts from the
oracle's lists; the velocity is then the oracle's only if these sources are
summed too.

Centres off the grid: the centres are rounded too, to 2^-53 of the coordinates,
which deep in a tree or far from the origin is a good part of a box side.  P2M,
M2M, L2L and L2P use the rounded centres, so the rounding cancels in the velocity
if M2L uses them as well."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-10


def _field(w, lo, n, seed):
    """n particles over [lo, lo + w] x [-w / 4, w / 4], the extremes included."""
    g = np.random.default_rng(seed)
    x, y = g.uniform(lo, lo + w, n), g.uniform(-w / 4, w / 4, n)
    x[:2], y[2:4] = (lo, lo + w), (-w / 4, w / 4)
    return x, y, np.full(n, 0.01 * w), g.normal(0, 1e-3, n)


def _beside(oracle, x, y, o):
    """List-2 entries whose box touches the target's."""
    t = oracle.T1Tree(x, y, o)
    b = t.boxes()
    return sum(max(abs(b["ix"][e] - b["ix"][k]), abs(b["iy"][e] - b["iy"][k])) <= 1
               for k in range(t.nboxes) if b["level"][k] >= 2 for e in t.list(k, 2))


@pytest.mark.parametrize("w, lo", [(1053.080880327208, -23.790051421199692),
                                   (128.6897492015798, -3.1167964408478293)])
@pytest.mark.parametrize("ndp, icutoff, mode", [(1, 2, 0), (5, 0, 0), (10, 2, 1), (12, 3, 1),
                                                (16, 2, 0), (17, 2, 0)])
def test_type1_sources_beside_the_target(gpu, oracle, w, lo, ndp, icutoff, mode):
    from lsmps_vpm_v2_amd import FmmSolver
    x, y, sz, g = _field(w, lo, 2000, 7)
    o = oracle.t1_opts(n_s=20, lmax=6, ndp=ndp, icutoff=icutoff, l2l_mode=mode)
    assert _beside(oracle, x, y, o) == 20
    ur, vr = oracle.t1_velocity(x, y, sz, g, o)
    u, v = FmmSolver(u_inf=0.0, v_inf=0.0).velocity_type1(x, y, sz, g, n_s=20, lmax=6, ndp=ndp,
                                                          icutoff=icutoff, l2l_mode=mode)
    err = np.max(np.hypot(u - ur, v - vr)) / np.sqrt(np.mean(ur ** 2 + vr ** 2))
    print(f"w {w:.0f} ndp {ndp} icutoff {icutoff} l2l {mode}: {err:.2e}")
    assert err <= TOL


# An M2L from grid offsets alone differs from the oracle by eps = 2^-53
# |coordinate| / side: 6e-14 (rel-L2) at offset 1e3, 6e-11 at 1e6, 3e-13 at level
# 16.  The stored-centre form differs by the rounding of sums of some hundred
# terms, 3e-15 at most on these fields; 1e-14 is 45 units of the last place.
REL = 1e-14


def _rel(u, v, ur, vr):
    return float(np.sqrt(np.mean((u - ur) ** 2 + (v - vr) ** 2) / np.mean(ur ** 2 + vr ** 2)))


def _check(oracle, x, y, sz, g, n_s, lmax, ndp, icutoff):
    from lsmps_vpm_v2_amd import FmmSolver
    ur, vr = oracle.t1_velocity(x, y, sz, g, oracle.t1_opts(n_s=n_s, lmax=lmax, ndp=ndp,
                                                            icutoff=icutoff, l2l_mode=0))
    u, v = FmmSolver(u_inf=0.0, v_inf=0.0).velocity_type1(x, y, sz, g, n_s=n_s, lmax=lmax,
                                                          ndp=ndp, icutoff=icutoff, l2l_mode=0)
    err = _rel(u, v, ur, vr)
    print(f"lmax {lmax} ndp {ndp}: {err:.2e}")
    assert err <= REL


@pytest.mark.parametrize("ndp", [2, 4, 6, 8, 10, 13, 16])
@pytest.mark.parametrize("offset", [0.0, 60.0, 1e3, 1e4, 1e6])
def test_type1_far_from_the_origin(gpu, oracle, offset, ndp):
    from lsmps_vpm_v2_amd import workloads as W
    c = W.random_clusters(7000, seed=51)
    for lmax in (7, 10):
        _check(oracle, c["x"] * 11 + offset, c["y"] * 11 - offset, np.full(7000, 0.04), c["q"],
               8, lmax, ndp, 2)


@pytest.mark.parametrize("ndp", [2, 4, 10, 16])
@pytest.mark.parametrize("lmax", [12, 13, 14, 16])
def test_type1_deep_trees(gpu, oracle, lmax, ndp):
    """Particles crowding towards a point, down to the deepest level."""
    g = np.random.default_rng(11)
    n = 9000
    r, th = 10.0 ** g.uniform(-6, 0, n), g.uniform(0, 2 * np.pi, n)
    x, y = r * np.cos(th) + 0.3, r * np.sin(th) - 0.2
    _check(oracle, x, y, np.full(n, 1e-4), g.normal(0, 1e-3, n), 10, lmax, ndp, 2)


@pytest.mark.parametrize("ndp", [4, 10, 16])
@pytest.mark.parametrize("scale", [1e-100, 1e-30, 1e6, 1e9])
def test_type1_scales(gpu, oracle, scale, ndp):
    """Fields of any size.  Below the box tests' tolerance no boxes are well
    separated (the oracle refuses such a field): only near pairs are summed, the
    same at every order."""
    from lsmps_vpm_v2_amd import FmmSolver
    g = np.random.default_rng(3)
    x, y, gz = scale * g.random(3000), scale * g.random(3000), scale * g.standard_normal(3000)
    sz = np.full(3000, 0.01 * scale)
    s = FmmSolver(u_inf=0.0, v_inf=0.0)
    kw = dict(n_s=20, lmax=8, icutoff=2, l2l_mode=0)
    u, v = s.velocity_type1(x, y, sz, gz, ndp=ndp, **kw)
    if scale < 1e-20:
        ur, vr = s.velocity_type1(x, y, sz, gz, ndp=20, **kw)
        assert np.isfinite(ur).all()
    else:
        ur, vr = oracle.t1_velocity(x, y, sz, gz, oracle.t1_opts(ndp=ndp, **kw))
    err = _rel(u, v, ur, vr)
    print(f"scale {scale:g} ndp {ndp}: {err:.2e}")
    assert err <= TOL
