"""The 3-D evaluation's groups of 8 targets, queues of 64 cells and rounds of
16 sources, at the sizes where they fill, spill over or stay partial: against
the 3-D oracle, max |d(u, v, w)| / rms(rotational velocity) <= 1e-11 (the same
FP64 sums in another order; measured under 1e-13)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-11


def _field(n, seed):
    g = np.random.Generator(np.random.PCG64(seed))
    p = g.uniform(-1.0, 1.0, (3, n))
    m = n // 2  # half of it clustered: leaves of every level
    p[:, :m] = 0.3 + 0.05 * g.standard_normal((3, m))
    s = 0.02 * (1 + g.uniform(0, 1, n))
    w = g.standard_normal((3, n))
    act = (g.random(n) < 0.8).astype(np.uint8)
    return [p[0].copy(), p[1].copy(), p[2].copy(), s, *(c.copy() for c in w)], act


def _check(cols, act, **o):
    from lsmps_vpm_v2_amd import FmmSolver
    from oracle import oracle as O
    print(f"3-D groups n={len(act)} {o}", flush=True)
    solver = FmmSolver()
    got = np.stack(solver.velocity3d(*cols, act, **o), 1)
    solver.close()
    ref = np.stack(O.o3_velocity(*cols, act, O.o3_opts(**o), 1.0, 0.0, 0.0), 1)
    return got, ref


CASES = [(n, dict(crit_num=c)) for n in (2, 7, 8, 9, 63, 65, 513) for c in (2, 5)] + [
    (1031, dict(crit_num=2, support=0.7)), (3000, dict(crit_num=30, support=9.0)),
    (5003, dict(crit_num=200)), (9001, dict(crit_num=1500, support=1.5)),
    (6000, dict(type=2, max_par=300, max_src=70)), (4001, dict(type=2, max_par=9, max_src=5))]


@pytest.mark.parametrize("n,o", CASES, ids=[f"{n}-" + "-".join(map(str, o.values())) for n, o in CASES])
def test_groups_match_oracle(gpu, n, o):
    got, ref = _check(*_field(n, n), **o)
    rot = ref - np.array([1.0, 0.0, 0.0])
    sc = max(np.sqrt(np.mean((rot ** 2).sum(1))), 1e-300)
    assert np.max(np.linalg.norm(got - ref, axis=1)) <= TOL * sc + 1e-15


def test_inactive_source_without_finite_strength(gpu):
    """Type 2 sums the inactive particles of near leaves: one whose strength is
    not finite reaches exactly the targets that take its leaf directly."""
    cols, act = _field(4000, 5)
    k = 3000
    act[k] = 0
    cols[5][k] = np.nan
    got, ref = _check(cols, act, type=2)
    assert 0 < np.isnan(ref).any(1).sum() < 2000
    assert np.array_equal(np.isnan(got), np.isnan(ref))


@pytest.mark.parametrize("type", [1, 2])
def test_infinite_strength(gpu, type):
    """An infinite x vorticity leaves u as it is; v and w become infinite where the
    particle is summed directly and NaN or infinite where a cell's moments carry it,
    target by target as in the oracle; the particle itself stays finite."""
    cols, act = _field(4000, 5)
    k = 3000
    act[k] = 1
    cols[4][k] = np.inf
    got, ref = _check(cols, act, type=type)
    sc = np.sqrt(np.mean((ref[:, 0] - 1.0) ** 2))
    assert np.max(np.abs(got[:, 0] - ref[:, 0])) <= TOL * sc
    assert np.max(np.abs(got[k] - ref[k])) <= TOL * sc
    for c in (1, 2):
        inf = np.isinf(ref[:, c])
        assert inf.sum() > 50
        assert np.array_equal(np.isnan(got[:, c]), np.isnan(ref[:, c]))
        assert np.array_equal(got[inf, c], ref[inf, c])


@pytest.mark.parametrize("n", [5, 8192, 8193, 20001])
def test_work_counts(gpu, n):
    """Pairs and far-cell terms as a walk over the oracle's tree counts them, on
    both sides of the 1024 records (of 8 targets) one workgroup adds up, and the
    same again for a second call on the handle."""
    from lsmps_vpm_v2_amd import FmmSolver
    from oracle import oracle as O
    cols, act = _field(n, n)
    act[:] = 1
    o = dict(crit_num=30, support=2.0)
    t = O.O3Tree(*cols[:3], act, O.o3_opts(**o))
    kids = {}
    for c in range(len(t.level)):
        kids.setdefault((int(t.level[c]) - 1, int(t.key[c]) >> 3), []).append(c)
    p = np.stack(cols[:3], 1)
    pairs = far = 0
    walk = [(c, np.arange(n)) for c in range(len(t.level)) if t.level[c] == 1 and not t.leaf[c]]
    while walk:
        c, tgt = walk.pop()
        for k in kids.get((int(t.level[c]), int(t.key[c])), []):
            r2 = ((p[tgt] - t.centre[k]) ** 2).sum(1)
            near = tgt[~(r2 > (o["support"] * t.size[k]) ** 2)]
            far += len(tgt) - len(near)
            if t.leaf[k]:
                own = t.particles(k)
                pairs += len(near) * len(own) - len(np.intersect1d(near, own))
            else:
                walk.append((k, near))
    s = FmmSolver()
    for _ in range(2):
        s.velocity3d(*cols, act, **o)
        st = s.fmm3d_stats()
        print(f"work n={n}: {st['pairs']} pairs, {st['m2p']} far", flush=True)
        assert (st["pairs"], st["m2p"]) == (pairs, far)


def test_strength_near_the_range(gpu):
    """A strength whose product with the distance of a target overflows, where only
    nearer targets sum it directly and the farther ones by its cell's moments:
    everything stays finite."""
    from lsmps_vpm_v2_amd import FmmSolver
    from oracle import oracle as O
    g = np.random.default_rng(2)
    n = 400
    p = g.uniform(-8.0, 8.0, (3, n))
    a = 1e290 * g.standard_normal((3, n))
    k = np.argmax(p.sum(0))
    a[:, k] = 0.0
    a[0, k] = 1.6e307
    act = np.ones(n, np.uint8)
    ref = np.stack(O.o3_velocity_alpha(*p, *a, act, O.o3_opts()), 1)
    assert np.isfinite(ref).all()
    got = np.stack(FmmSolver(u_inf=0.0, v_inf=0.0).velocity3d_alpha(*p, *a, act), 1)
    assert np.isfinite(got).all()
    # (scaled: the squares overflow)
    err = np.linalg.norm(got / 1e300 - ref / 1e300, axis=1)
    assert np.max(err) <= TOL * np.sqrt(np.mean(((ref / 1e300) ** 2).sum(1)))
