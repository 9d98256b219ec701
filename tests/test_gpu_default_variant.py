"""The step variant a pool takes when none was set: by the number of patches,
on both sides of every line of the rule (256 CUs), the results of every
variant; the captured graph follows the choice; a step in place keeps one tile
per patch."""
import numpy as np
import pytest

from _parity import assert_same

pytestmark = pytest.mark.gpu

SMALL, LARGE = (16, 16, 384, 1), (32, 32, 768, 1)


def _state(rng, lay, mx, m, n):
    h = 1.0 + rng.random((n * mx, m * mx))
    h[:, m * mx // 2:] *= rng.random((n * mx, m * mx - m * mx // 2)) < 0.5
    u = rng.normal(size=(2,) + h.shape) * h
    return h, u[0], u[1], rng.normal(0.0, 0.2, h.shape)


@pytest.mark.parametrize("mx,m,n,expect", [(8, 1, 1, (8, 8, 128, 1)), (16, 48, 32, SMALL), (16, 53, 29, (16, 16, 192, 1)),
                                           (32, 16, 8, SMALL), (32, 43, 3, LARGE), (64, 8, 4, SMALL), (64, 11, 3, LARGE)])
def test_default_equals_every_variant(gf, mx, m, n, expect):
    from geoflood_amd.pool import BrickLayout, Pool
    lay = BrickLayout(m, n, mx, mx, 1.0, 1.0)
    state = _state(np.random.default_rng(mx * m + n), lay, mx, m, n)
    out = []
    count = 1
    v = -1
    while v < count:
        pool = Pool(mx, mx, lay.npatch)
        pool.set_layout([lay])
        pool.upload_global(lay, *state)
        sid = pool.add_scenario(lay, dt0=0.02)
        cur, vs = pool.variants()
        count = len(vs)
        if v < 0:
            assert vs[cur][:4] == expect
        elif v < count:
            pool.set_variant(v)
        else:
            pool.close()
            break
        pool.run(3)
        rec = pool.scenario(sid)
        out.append((pool.download_global(lay, rec["cur"]), rec))
        pool.close()
        v += 1
    assert len(out) == count + 1
    for got, rec in out[1:]:
        assert rec == out[0][1]
        for a, r in zip(out[0][0], got):
            assert_same(a, r)


def test_graph_follows_the_population(gf):
    """More patches described between two captured runs: the second run is
    captured again with the variant for them, and equals an uncaptured one."""
    from geoflood_amd.pool import BrickLayout, Pool
    one, two = BrickLayout(4, 2, 32, 32, 1.0, 1.0), BrickLayout(13, 10, 32, 32, 1.0, 1.0)
    s1, s2 = (_state(np.random.default_rng(k), None, 32, *mn) for k, mn in enumerate([(4, 2), (13, 10)]))
    out = []
    for use_graph in (True, False):
        seen = []
        for lays in ([one], [two]):
            pool = Pool(32, 32, 130) if not seen else pool
            pool.set_layout(lays)
            pool.upload_global(lays[0], *(s1 if lays[0] is one else s2))
            sid = pool.add_scenario(lays[0], dt0=0.02)
            cur, vs = pool.variants()
            pool.run(2, graph=use_graph)
            pool.run(1, graph=use_graph)
            rec = pool.scenario(sid)
            seen.append((vs[cur][:4], pool.download_global(lays[0], rec["cur"]), rec))
        pool.close()
        out.append(seen)
    for a, b in zip(*out):
        assert a[0] == b[0] and a[2] == b[2]
        for x, y in zip(a[1], b[1]):
            assert_same(x, y)
    assert [s[0] for s in out[0]] == [SMALL, LARGE]


@pytest.mark.parametrize("mx", [8, 16, 32])
def test_default_steps_in_place(gf, mx):
    from geoflood_amd.pool import Pool
    rng = np.random.default_rng(mx)
    n, w = 3, mx + 4
    q = rng.normal(0.0, 0.3, (n, w, w, 3))
    q[..., 0] = 1.0 + rng.random((n, w, w))
    aux = rng.normal(0.0, 0.2, (n, w, w, 1))
    pool = Pool(mx, mx, n)
    pool.set_patches(np.full(n, 1.0), np.full(n, 1.0), np.zeros(n), np.zeros(n))
    out = []
    for dst in (0, 1):
        pool.upload_aos(0, q, aux, buf=0)
        c, _ = pool.step(0.02, src=0, dst=dst)
        out.append((c, pool.download_aos(0, n, buf=dst)[:, 2:-2, 2:-2]))
    pool.close()
    assert out[0][0] == out[1][0]
    assert_same(out[0][1], out[1][1])
