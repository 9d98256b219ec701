"""A regrid that keeps the passes of the ghost update keeps the captured attempt
graph: moving a scenario to the other half of its pool (gf_pool_set_scenario_
slots) and setting the new half's links (gf_pool_set_cf_links) captures nothing,
although between the two calls the scenario's slots have no links."""
from types import SimpleNamespace

import numpy as np
import pytest

from geoflood_amd import GF_NB_INFLOW, GF_NB_STORED

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mx", [8, 16, 32])
def test_changing_halves_keeps_the_graph(gf, mx):
    """One coarse patch and, on its left half a level finer, a patch with a
    hydrograph side, which the coarse one writes to: passes 0 and 1."""
    from geoflood_amd.pool import Pool
    print(f"case graph captures {mx}", flush=True)
    half, w = 4, mx + 4
    pool = Pool(mx, mx, 2 * half)
    dx = np.tile([1.0, 0.5], 4)
    nbr = np.full((2 * half, 8), GF_NB_STORED, dtype=np.int32)
    nbr[1::half, 0] = GF_NB_INFLOW
    pool.set_patches(dx, dx, np.zeros(2 * half), np.zeros(2 * half), nbr)
    q = np.zeros((2 * half, w, w, 3))
    q[..., 0] = 1.0 + np.random.default_rng(mx).random((2 * half, w, w))
    for buf in (0, 1):
        pool.upload_aos(0, q, np.zeros((2 * half, w, w, 1)), buf=buf)
    sid = pool.add_scenario(SimpleNamespace(first=0, npatch=2), dt0=1e-4)
    pool.set_inflow(sid, [0.0, 10.0], [0.4, 0.9], 0.5 * mx, 0.0, 0.3 * mx)
    pool.set_levels(0, np.tile([0, 1], 4))

    def use(base):
        pool.set_scenario_slots(sid, base, 2)
        pool.set_cf_links([base], [base + 1], [0], [0])
        pool.run(1)

    captures = lambda: gf.load().gf_pool_graph_captures(pool.h)
    assert captures() == 0
    use(0)
    use(half)
    before = captures()
    for k in range(6):
        use(half * (k % 2))
    assert before >= 1 and captures() == before
    assert pool.scenario(sid)["attempts"] == 8
    pool.close()
