"""Tiles outside the range of the fast quotients (gf_exact.h) take the general
operations on the device, in the host batch's kernel and in the batched one, in
every variant: on inputs where the two forms give different cells (asserted on
the host first) the device's equal the oracle's."""
import numpy as np
import pytest

from _parity import assert_same
from _physlib import host_step
from test_general_step import INNER, SPECIAL, special

pytestmark = pytest.mark.gpu

DX, DY, DT = 0.1, 0.2, 0.005


@pytest.mark.parametrize("mx", [8, 16, 32, 64])
@pytest.mark.parametrize("kind", SPECIAL)
def test_out_of_range_tiles_equal_oracle(gf, oracle_c, mx, kind):
    from geoflood_amd import GF_NB_STORED
    from geoflood_amd.pool import Pool
    from oracle.oracle import Params
    print(f"case general path {kind} {mx}", flush=True)
    n = 5   # an ordinary patch among them; not a multiple of the patches per workgroup
    patches = [special(kind, seed, mx + 4) for seed in range(n)]
    params = patches[0][0]
    p = Params(**params)
    patches[2] = (params,) + special("film 1", 2, mx + 4)[1:]
    q = np.stack([x[1] for x in patches])
    bed = np.stack([x[2] for x in patches])
    gf.set_params(**params)
    oracle_c.set_params(p)
    try:
        ref, differ = q.copy(), 0
        cfl = [oracle_c.patch_update(mx, mx, 2, r, b, DX, DY, 0.0, DT) for r, b in zip(ref, bed)]
        for k in range(n):
            fast = q[k].copy()
            host_step(p, fast, bed[k], DX, DY, DT, fast=True)
            differ += not np.array_equal(fast[INNER], ref[k][INNER], equal_nan=True)
        assert differ, "an input that both forms step alike shows nothing"
        finite = bool(np.isfinite(ref[:, 2:-2, 2:-2]).all())

        got = [a.copy() for a in q]
        c = gf.step2_batch(got, list(bed.copy()), DX, DY, 0.0, DT)
        assert c == max(cfl) if finite else np.isnan(c)
        for k in range(n):
            assert_same(got[k][INNER], ref[k][INNER], f"batch, patch {k}")

        pool = Pool(mx, mx, n)
        try:
            for v in range(len(pool.variants()[1])):
                pool.set_patches(np.full(n, DX), np.full(n, DY), np.zeros(n), np.zeros(n),
                                 np.full((n, 8), GF_NB_STORED, dtype=np.int32))
                pool.set_variant(v)
                for buf in (0, 1):
                    pool.upload_aos(0, q, bed, buf=buf)
                sid = pool.add_scenario(_All(n), dt0=DT, max_cfl=1e300)
                pool.run(1)
                out = pool.download_aos(0, n, buf=1)
                for k in range(n):
                    assert_same(out[k][INNER], ref[k][INNER], f"variant {v}, patch {k}")
                assert pool.scenario(sid)["active"] == finite
        finally:
            pool.close()
    finally:
        gf.set_params()
        oracle_c.set_params(Params())


class _All:
    def __init__(self, n):
        self.first, self.npatch = 0, n
