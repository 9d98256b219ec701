"""The persistent step kernel's item queues: a workgroup's first item is its
own index and the rest come from its queue, so populations below, at and
above the number of workgroups (256 CUs times the variant's occupancy) must
step every patch exactly once.  Batched attempts against the per-patch launch
loop, bit for bit."""
import numpy as np
import pytest

from _parity import assert_same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mx,m,n", [(8, 1, 1), (8, 7, 1), (8, 9, 1), (8, 45, 45), (8, 89, 23), (8, 89, 46), (8, 70, 61),
                                    (16, 16, 32), (16, 27, 19), (32, 16, 16), (32, 257, 1), (64, 8, 8), (64, 13, 5)])
def test_batched_equals_plain(gf, mx, m, n):
    from geoflood_amd.pool import BrickLayout, Pool
    rng = np.random.default_rng(mx * m + n)
    ny, nx = n * mx, m * mx
    h = 1.0 + rng.random((ny, nx))
    h[:, nx // 2:][rng.random((ny, nx - nx // 2)) < 0.9] = 0.0   # wet, front and dry patches
    if m > 4:
        h[:, 3 * nx // 4:] = 0.0
    u = rng.normal(size=(2, ny, nx)) * h
    b = rng.normal(0.0, 0.2, (ny, nx))
    lay = BrickLayout(m, n, mx, mx, 1.0, 1.0)
    out = []
    for plain in (False, True):
        pool = Pool(mx, mx, lay.npatch)
        pool.set_layout([lay])
        pool.upload_global(lay, h, u[0], u[1], b)
        sid = pool.add_scenario(lay, dt0=0.02)
        (pool.run_plain if plain else pool.run)(3)
        rec = pool.scenario(sid)
        out.append((pool.download_global(lay, rec["cur"]), rec))
        pool.close()
    assert out[0][1] == out[1][1]
    for a, r in zip(out[0][0], out[1][0]):
        assert_same(a, r)
