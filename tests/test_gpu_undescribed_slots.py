"""gf_pool_describe above the slots described so far leaves a gap, and a scenario
may cover it: the gap's slots read their own cells (every ghost region stored),
as their neighbours in the scenario step as they do without them."""
import numpy as np
import pytest

from _parity import assert_same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mx", [8, 16, 32, 64])
@pytest.mark.parametrize("graph", [False, True])
def test_gap_reads_its_own_cells(gf, mx, graph):
    from geoflood_amd.pool import BrickLayout, Pool
    print(f"case undescribed slots {mx} {graph}", flush=True)
    rng = np.random.default_rng(mx)
    gap, n, w = 3, 2, mx + 4
    q = np.zeros((gap + n, w, w, 3))
    q[:gap, ..., 0] = 1e-4 * rng.random((gap, w, w))       # below dry_tolerance: the step keeps the depths
    q[gap:, ..., 0] = 1.0 + rng.random((n, w, w))
    aux = np.zeros((gap + n, w, w, 1))
    out = []
    for skip in (gap, 0):
        pool = Pool(mx, mx, 8)
        lay = BrickLayout(n, 1, mx, mx, 1.0, 1.0)
        pool.describe(lay, skip)
        for buf in (0, 1):
            pool.upload_aos(0, q[gap - skip:], aux[gap - skip:], buf=buf)
        sid = pool.add_scenario(_Range(0, skip + n), dt0=0.01)
        pool.run(3, graph=graph)
        rec = pool.scenario(sid)
        out.append((pool.download_aos(0, skip + n, buf=rec["cur"]), rec["t"], rec["dt"], rec["nsteps"]))
        pool.close()
    inner = (slice(None), slice(2, -2), slice(2, -2))
    assert out[0][1:] == out[1][1:] and out[0][3] > 0
    assert_same(out[0][0][:gap][inner], q[:gap][inner], "gap")
    assert_same(out[0][0][gap:][inner], out[1][0][inner], "described")


class _Range:
    def __init__(self, first, npatch):
        self.first, self.npatch = first, npatch
