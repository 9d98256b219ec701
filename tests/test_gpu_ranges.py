"""The step's fast quotients (gf_exact.h) and the general operations that
tiles outside their range take: identical values to the oracle on both sides
of every bound (momenta and bathymetry around 2^-240, products of waves that
underflow, large depths and momenta, dry tolerances and gravities outside the
range), and on mantissas next to a power of two, the hard reciprocals."""
import numpy as np
import pytest

from _parity import assert_same

pytestmark = pytest.mark.gpu


def _patch(rng, mx, kind):
    n = mx + 4
    h = 1.0 + rng.random((n, n))
    hu, hv = rng.normal(size=(2, n, n))
    b = rng.normal(0.0, 0.3, (n, n))
    if kind == "fronts":
        h[rng.random(h.shape) < 0.3] = 0.0
    elif kind == "edge":       # both sides of the smallest momentum and bathymetry of the fast range
        hu = hu * 2.0 ** rng.integers(-244, -236, h.shape)
        hv[:] = np.where(rng.random(h.shape) < 0.5, 0.0, 2.0 ** -240)
        b = b * 2.0 ** -238.0
    elif kind == "calm":       # equal depths and discharge: waves that are products of two small momenta
        h[:], b[:] = 1.5, 0.0
        hu[:] = 1e-70
        hv *= 1e-70
    elif kind == "cascade":    # a lake with a disturbance that decays below every bound
        h[:], b[:] = 2.0, 0.0
        hu = hu * 10.0 ** -rng.integers(0, 300, h.shape)
        hv = hv * 10.0 ** -rng.integers(0, 300, h.shape)
    elif kind == "large":
        h = h * 2.0 ** rng.integers(0, 34, h.shape)
        hu, hv = hu * 2.0 ** rng.integers(0, 24, h.shape), hv * 2.0 ** rng.integers(0, 24, h.shape)
        b = b * 2.0 ** rng.integers(0, 34, h.shape)
    elif kind == "mantissas":  # 2 - k ulp and 2 + k ulp
        h = 2.0 + rng.integers(-6, 6, h.shape) * 2.0 ** -52
        hu, hv = rng.choice([0.0, 1.0 - 2.0 ** -53, 1.0 + 2.0 ** -52], (2, n, n))
    h[h < 0] = 0.0
    q = np.stack([h, np.where(h > 0, hu, 0.0), np.where(h > 0, hv, 0.0)], -1)
    return np.ascontiguousarray(q), np.ascontiguousarray(b[..., None])


@pytest.mark.parametrize("mx", [8, 16, 32, 64])
@pytest.mark.parametrize("kind,params", [
    ("fronts", {}), ("edge", {}), ("calm", {}), ("cascade", {}), ("large", {}), ("mantissas", {}),
    ("fronts", dict(dry_tolerance=1e-6)), ("fronts", dict(grav=0.05)), ("fronts", dict(grav=300.0)),
    ("cascade", dict(mthlim=(3, 2, 1))),
])
def test_values_identical_to_oracle(gf, oracle_c, mx, kind, params):
    from oracle.oracle import Params
    rng = np.random.default_rng(mx)
    gf.set_params(**params)
    oracle_c.set_params(Params(**params))
    try:
        patches = [_patch(rng, mx, kind) for _ in range(3)]
        q, aux = [p[0] for p in patches], [p[1] for p in patches]
        ref = [a.copy() for a in q]
        dt = 1e-3 if kind != "large" else 1e-9
        cfl = max(oracle_c.patch_update(mx, mx, 2, r, a, 0.5, 0.25, 0.0, dt) for r, a in zip(ref, aux))
        got = gf.step2_batch(q, aux, 0.5, 0.25, 0.0, dt)
        assert got == cfl
        for a, r in zip(q, ref):
            assert_same(a[2:-2, 2:-2], r[2:-2, 2:-2], kind)
    finally:
        gf.set_params()
        oracle_c.set_params(Params())
