"""The step's powers on the device over the whole range of its own cube root and
logarithm (2^-100 to 2^60), on both sides of both ends and of the logarithm's
reduction, and beyond, where the library's take over: bit-identical to the host
build (correctly rounded)."""
import numpy as np
import pytest

from _powlib import host_powers
from test_pow_own_root import arguments

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("which", [0, 1])
def test_device_powers_over_their_range(gf, which):
    print(f"case device powers, whole range, {which}", flush=True)
    rng = np.random.default_rng(200 + which)
    x = arguments(rng, 1 << 19)
    ends = np.array([2.0 ** -100, 2.0 ** 60])
    x = np.concatenate([x, (ends[:, None] * (1.0 + rng.integers(-4096, 4096, (2, 4096)) * 2.0 ** -52)).ravel(),
                        2.0 ** rng.uniform(-299.0, -100.0, 4096), 2.0 ** rng.uniform(60.0, 299.0, 4096)])
    dev = np.zeros_like(x)
    assert gf.load().gf_eval_powers(which, len(x), gf.dptr(x), gf.dptr(dev)) == 0
    want = host_powers(which, x)
    bad = np.flatnonzero(dev != want)
    assert len(bad) == 0, (len(bad), x[bad[:5]], dev[bad[:5]], want[bad[:5]])
