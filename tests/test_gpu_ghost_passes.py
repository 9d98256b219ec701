"""The resident ghost update (gf_pool_ghost_update) shares a launch between
items of different levels that do not wait for each other.  Over arbitrary
accepted links -- also those a balanced forest never has, where a patch's links
read ghost cells that a coarser patch's links have just written -- and
hydrograph sides it equals the transfers called one by one: all averages, then
per level the hydrograph sides and that level's interpolation."""
from types import SimpleNamespace

import numpy as np
import pytest

from geoflood_amd import GF_NB_INFLOW, GF_NB_STORED

pytestmark = pytest.mark.gpu

LEVELS, PER = 4, 8


def _links(rng, density):
    """Links between neighbouring levels; a fine slot takes two opposite faces
    or one corner, so that no cell is written by two links."""
    out, seen = [], set()
    for l in range(LEVELS - 1):
        for f in range((l + 1) * PER, (l + 2) * PER):
            kind = int(rng.integers(3))
            for side in ((0, 1), (2, 3), (int(rng.integers(4, 8)),))[kind]:
                c, ig = l * PER + int(rng.integers(PER)), int(rng.integers(2)) if side < 4 else 0
                if rng.random() < density and (c, side, ig) not in seen:
                    seen.add((c, side, ig))
                    out.append((c, f, side, ig))
    return np.array(out, dtype=np.int32).reshape(-1, 4)


@pytest.mark.parametrize("mx,density,inflow,seed", [(8, 0.9, 0.0, 1), (8, 0.9, 0.4, 2), (16, 0.9, 0.4, 3), (16, 0.3, 0.2, 4),
                                                    (32, 0.9, 0.3, 5), (64, 0.6, 0.3, 6)])
def test_equals_level_order(gf, mx, density, inflow, seed):
    from geoflood_amd.pool import Pool
    rng = np.random.default_rng(seed)
    n, w = LEVELS * PER, mx + 4
    level = np.repeat(np.arange(LEVELS), PER)
    dx = 1.0 / 2 ** level
    nbr = np.full((n, 8), GF_NB_STORED, dtype=np.int32)
    nbr[rng.random(n) < inflow, 0] = GF_NB_INFLOW
    links = _links(rng, density)
    q = rng.normal(0.0, 0.5, (n, w, w, 3))
    q[..., 0] = (1.0 + rng.random((n, w, w))) * (rng.random((n, w, w)) < 0.8)
    aux = rng.normal(0.0, 0.2, (n, w, w, 1))
    out = []
    for resident in (True, False):
        pool = Pool(mx, mx, n)
        pool.set_patches(dx, dx, np.zeros(n), np.zeros(n), nbr)
        sid = pool.add_scenario(SimpleNamespace(first=0, npatch=n), dt0=0.1)
        if (nbr[:, 0] == GF_NB_INFLOW).any():
            pool.set_inflow(sid, [0.0, 10.0], [0.4, 0.9], 0.5 * mx, 0.0, 0.3 * mx)
        pool.upload_aos(0, q, aux, buf=0)
        if resident:
            pool.set_levels(0, level)
            pool.set_cf_links(*links.T)
            pool.ghost_update(0, 3.0)
        else:
            pool.average_ghost(*links.T, buf=0)
            for l in range(LEVELS):
                pool.ghost_fill(l * PER, PER, buf=0, t=3.0)
                here = links[level[links[:, 0]] == l]
                if len(here):
                    pool.interpolate_ghost(*here.T, buf=0)
        out.append((pool.download_aos(0, n), pool.download_aux(0, n)))
        pool.close()
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
