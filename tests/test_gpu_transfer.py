"""Downloads (csrc/isph_transfer.hip) return what was uploaded, for sizes at
the edges of the 64-row groups and of the chunks that the threads share."""
import ctypes

import numpy as np
import pytest

from beach_slope_confined_amd import capi, configs

pytestmark = pytest.mark.gpu

CHUNK = (1280 * 1024 // 76) & ~63  # rows of a chunk with all eleven columns


def _sim(n):
    rng = np.random.default_rng(n)
    parts = {k: rng.uniform(0.5, 1.5, n) for k in ("vx", "vy", "mass", "density", "oden",
                                                   "pressure")}
    parts["x"], parts["y"] = rng.uniform(0.0, 1.6, n), rng.uniform(0.0, 0.6, n)
    parts["tid"] = rng.integers(1, 4, n).astype(np.int32)
    parts["flags"] = (rng.integers(0, 2, n) * 2).astype(np.int32)
    parts["pid"] = rng.permutation(n).astype(np.int32)
    sim = capi.IsphSim(configs.dam_break(0.05)["params"], n, 1)
    sim.set_particles(parts)
    return sim, parts


@pytest.mark.parametrize("n", [1, 63, 64, 65, CHUNK, CHUNK + 1, 2 * CHUNK + 64, 11 * CHUNK - 1])
def test_round_trip(require_gpu, n):
    sim, parts = _sim(n)
    q = sim.get_particles()
    order = np.argsort(parts["pid"])[q["pid"]]
    for k in parts:
        assert np.array_equal(q[k], parts[k][order]), k
    for k in ("x", "y", "vx", "vy", "pressure", "mass"):
        assert np.array_equal(sim.get_field(k), q[k]), k
    assert np.array_equal(sim.get_field("coff"), np.tile([1.0, 0.0, 0.0, 1.0], (n, 1)))
    sim.close()


def test_some_columns(require_gpu):
    """Arrays that the caller does not want stay untouched."""
    n = 3 * CHUNK + 7
    sim, _ = _sim(n)
    q = sim.get_particles()
    y, flags, nn = np.empty(n), np.empty(n, np.int32), ctypes.c_int32()
    rc = sim._fn("get_particles")(sim._h, ctypes.byref(nn), None, capi._dp(y), *[None] * 7,
                                  capi._ip(flags), None)
    assert rc == 0 and nn.value == n
    assert np.array_equal(y, q["y"]) and np.array_equal(flags, q["flags"])
    sim.close()
