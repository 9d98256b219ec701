"""The ghost update as the captured attempt runs it (each scenario's current
buffer and time, the discharge looked up once per scenario), and its level order
when levels were given anew after the links: the state it leaves equals that of
the transfers called one by one."""
from types import SimpleNamespace

import numpy as np
import pytest

from geoflood_amd import GF_NB_INFLOW, GF_NB_STORED
from test_gpu_ghost_passes import LEVELS, PER, _links

pytestmark = pytest.mark.gpu

N = LEVELS * PER


def _forest(mx, density, inflow, seed):
    rng = np.random.default_rng(seed)
    w = mx + 4
    nbr = np.full((N, 8), GF_NB_STORED, dtype=np.int32)
    nbr[rng.random(N) < inflow, 0] = GF_NB_INFLOW
    q = rng.normal(0.0, 0.5, (N, w, w, 3))
    q[..., 0] = (1.0 + rng.random((N, w, w))) * (rng.random((N, w, w)) < 0.8)
    return nbr, _links(rng, density), q, rng.normal(0.0, 0.2, (N, w, w, 1))


def _pool(mx, forest, t0):
    from geoflood_amd.pool import Pool
    nbr, _, q, aux = forest
    pool = Pool(mx, mx, N)
    dx = 1.0 / 2 ** np.repeat(np.arange(LEVELS), PER)
    pool.set_patches(dx, dx, np.zeros(N), np.zeros(N), nbr)
    sid = pool.add_scenario(SimpleNamespace(first=0, npatch=N), dt0=1e-3, t0=t0)
    if (nbr[:, 0] == GF_NB_INFLOW).any():
        pool.set_inflow(sid, [0.0, 10.0], [0.4, 0.9], 0.5 * mx, 0.0, 0.3 * mx)
    pool.upload_aos(0, q, aux, buf=0)
    return pool


def _state(pool):
    out = pool.download_aos(0, N), pool.download_aux(0, N)
    pool.close()
    return out


@pytest.mark.parametrize("mx,density,inflow,seed", [(8, 0.9, 0.4, 2), (16, 0.9, 0.4, 3), (32, 0.9, 0.3, 5), (64, 0.6, 0.3, 6)])
@pytest.mark.parametrize("shift", [0, 1])  # 1: every level given anew, one deeper, after the links
@pytest.mark.parametrize("graph", [True, False])
def test_attempt_equals_transfers_one_by_one(gf, mx, density, inflow, seed, shift, graph):
    print(f"case ghost captured {mx} {seed} {shift} {graph}", flush=True)
    forest = _forest(mx, density, inflow, seed)
    links = forest[1]
    level = np.repeat(np.arange(LEVELS), PER)
    pool = _pool(mx, forest, 3.0)
    pool.set_levels(0, level)
    pool.set_cf_links(*links.T)
    if shift:
        pool.set_levels(0, level + 1)
    pool.run(1, graph=graph)
    got = _state(pool)     # buffer 0: the attempt's source, with its ghost cells
    pool = _pool(mx, forest, 3.0)
    pool.average_ghost(*links.T, buf=0)
    for l in range(LEVELS + shift):
        if 0 <= l - shift:
            pool.ghost_fill((l - shift) * PER, PER, buf=0, t=3.0)   # hydrograph sides by the levels as they are
        here = links[level[links[:, 0]] == l]                       # links by the levels as they were
        if len(here):
            pool.interpolate_ghost(*here.T, buf=0)
    want = _state(pool)
    for a, b in zip(got, want):
        np.testing.assert_array_equal(a, b)
