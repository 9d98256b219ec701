"""The step's scalar routines on the host (_physlib: the device's own sources).

The general operations (gf_physics.h) equal the oracle for every value: a NaN
or an infinity reaches exactly the cells that it reaches there, films under a
zero dry_tolerance stay finite, products that overflow go to the same side.
The forms of the range of gf_exact.h (gf_physics_fast.h) equal the general ones
inside it, over its whole extent: momenta and bathymetry from 2^-240, depths at
dry_tolerance and up to 2^30, gravities and tolerances at both ends, every
limiter, order and transverse setting."""
import numpy as np
import pytest

from _parity import assert_same
from _physlib import host_step

INNER = (slice(2, -2), slice(2, -2))
W = 20


def special(kind, seed, W=W):
    """(parameters, q, bed) of a patch (W cells wide with its ghost cells)
    outside the range."""
    rng = np.random.default_rng(seed)
    h = 1.0 + rng.random((W, W))
    u = rng.normal(size=(2, W, W))
    b = rng.normal(0.0, 0.3, (W, W, 1))
    params = {}
    if kind == "nan ghost":
        u[0][:, 0] = np.nan
    elif kind == "nan depth":
        h[3, 5] = np.nan
    elif kind == "nan bed":
        b[3, 5] = np.nan
    elif kind == "inf ghost":
        u[0][:, 0] = np.inf
    elif kind == "inf transverse ghost":
        u[1][:, 0] = np.inf
    elif kind == "inf momentum":
        u[1][9, 9] = np.inf
    elif kind == "inf depth":
        h[9, 9] = np.inf
    elif kind == "inf bed":
        b[9, 9] = np.inf
    elif kind == "-inf bed":
        b[9, 9] = -np.inf
    elif kind == "overflow":      # its square, and with it a wave, is infinite
        u[0][9, 9] = 1e155
    elif kind.startswith("film"):  # depths down to 1e-250 or 1e-300, all of them wet
        params = dict(dry_tolerance=0.0)
        h = 10.0 ** rng.uniform(-float(kind[5:]), 0.0, (W, W))
        u = u * h * np.sqrt(9.81 * h)
        b[:] = 0.0
    elif kind == "tolerance 1e-250":
        params = dict(dry_tolerance=1e-250)
        h = 10.0 ** rng.uniform(-250.0, 0.0, (W, W))
        u = u * h * np.sqrt(9.81 * h)
    else:
        raise ValueError(kind)
    return params, np.ascontiguousarray(np.stack([h, u[0], u[1]], -1)), b


SPECIAL = ["nan ghost", "nan depth", "nan bed", "inf ghost", "inf transverse ghost", "inf momentum", "inf depth", "inf bed",
           "-inf bed", "overflow", "film 250", "film 300", "tolerance 1e-250"]


@pytest.fixture
def ora(oracle_c):
    from oracle.oracle import Params
    oracle_c.set_pow_mode(True)
    yield oracle_c
    oracle_c.set_pow_mode(False)
    oracle_c.set_params(Params())


@pytest.mark.parametrize("kind", SPECIAL)
def test_general_operations_equal_oracle(ora, kind):
    from oracle.oracle import Params
    for seed in range(4):
        params, q, bed = special(kind, seed)
        p = Params(**params)
        ora.set_params(p)
        ref, got = q.copy(), q.copy()
        ora.patch_update(16, 16, 2, ref, bed, 0.1, 0.2, 0.0, 0.005)
        _, in_range = host_step(p, got, bed, 0.1, 0.2, 0.005, fast=False)
        assert not in_range
        assert_same(got[INNER], ref[INNER], f"{kind} {seed}")


def _in_range(rng):
    """A patch somewhere in the range, structured so that sums cancel."""
    from oracle.oracle import Params
    tol = 2.0 ** rng.uniform(-14, 10) if rng.random() < 0.5 else 1e-3
    params = Params(grav=2.0 ** rng.uniform(-4, 8) if rng.random() < 0.5 else 9.81, dry_tolerance=tol,
                    mthlim=tuple(int(x) for x in rng.integers(0, 6, 3)) if rng.random() < 0.5 else (4, 4, 4),
                    order=int(rng.integers(1, 3)), transverse=int(rng.integers(0, 3)),
                    manning_n=float(rng.choice([0.0, 0.025, 1e-8, 1e3])))
    shape = (W, W)
    kind = rng.integers(6)
    if kind == 0:
        h = tol * (0.9 + 0.4 * rng.random(shape))
    elif kind == 1:
        h = np.full(shape, tol * 2.0 ** rng.uniform(0, 10))
    elif kind == 2:
        h = tol * 2.0 ** rng.uniform(-1, min(19.0, 29.0 - np.log2(tol)), shape)
    elif kind == 3:
        h = tol * (3.0 + rng.integers(-3, 4, shape) * 2.0 ** -52)
    else:
        h = 1.0 + rng.random(shape)
        if kind == 5:
            h[rng.random(shape) < 0.3] = 0.0
    h = np.minimum(h, 2.0 ** 30)

    def momentum():
        kind, sign = rng.integers(6), rng.choice([-1.0, 1.0], shape)
        if kind == 0:
            return sign * 2.0 ** rng.uniform(-240, 19.9, shape)
        if kind == 1:
            return sign * 2.0 ** rng.uniform(-240, -230)
        if kind == 2:
            return np.zeros(shape)
        if kind == 3:
            return sign * 2.0 ** (rng.uniform(-239, 0) + rng.uniform(-0.5, 0.5, shape))
        if kind == 4:
            return np.clip(rng.normal(size=shape) * h * 0.5, 1.0 - 2.0 ** 20, 2.0 ** 20 - 1.0)
        return np.where(rng.random(shape) < 0.5, 0.0, sign * 2.0 ** rng.uniform(-239, -100, shape))

    kind = rng.integers(5)
    bed = (np.zeros(shape) if kind == 0 else rng.normal(0.0, 0.3, shape) if kind == 1
           else 2.0 ** rng.uniform(-240, -200) * rng.choice([-1.0, 0.0, 1.0], shape) if kind == 2
           else rng.choice([-1.0, 1.0], shape) * 2.0 ** rng.uniform(-240, 29, shape) if kind == 3 else 2.0 - h)
    return params, np.ascontiguousarray(np.stack([h, momentum(), momentum()], -1)), np.ascontiguousarray(bed[..., None])


@pytest.mark.parametrize("block", range(4))
def test_fast_forms_equal_general_in_their_range(block):
    tested = 0
    for n in range(400):
        rng = np.random.default_rng([block, n])
        params, q, bed = _in_range(rng)
        dx = 2.0 ** rng.uniform(-5, 5)
        dt = dx * 10.0 ** rng.uniform(-6, 0)
        a, b = q.copy(), q.copy()
        ca, in_range = host_step(params, a, bed, dx, 1.5 * dx, dt, fast=True)
        cb, _ = host_step(params, b, bed, dx, 1.5 * dx, dt, fast=False)
        if not in_range:
            continue
        tested += 1
        assert ca == cb, (block, n, ca, cb)
        assert_same(a[INNER], b[INNER], f"{block} {n}")
    assert tested > 350
