"""Checkpoint slots copy their arrays in one launch (csrc/isph_copy.hip): every
array comes back, at sizes around the 16 KB pieces of 16-, 8- and 4-byte rows
and the 16-byte words."""
import numpy as np
import pytest

from beach_slope_confined_amd import capi, configs

pytestmark = pytest.mark.gpu


def _particles(n, seed):
    rng = np.random.default_rng(seed)
    parts = {k: rng.uniform(0.5, 1.5, n) for k in ("vx", "vy", "mass", "density", "oden",
                                                   "pressure")}
    parts["x"], parts["y"] = rng.uniform(0.0, 1.6, n), rng.uniform(0.0, 0.6, n)
    parts["tid"] = rng.integers(1, 4, n).astype(np.int32)
    parts["flags"] = (rng.integers(0, 2, n) * 2).astype(np.int32)
    parts["pid"] = rng.permutation(n).astype(np.int32)
    return parts


@pytest.mark.parametrize("n", [1, 2, 3, 1023, 1024, 1025, 2047, 2049, 4095, 4096, 4097, 9001])
def test_slots_return_their_state(require_gpu, n):
    sim = capi.IsphSim(configs.dam_break(0.05)["params"], n, 1)
    fields = ("x", "y", "vx", "vy", "pressure", "mass", "density", "porosity")
    kept = []
    for slot in (0, 1):
        sim.set_particles(_particles(n, 10 * n + slot))
        sim.checkpoint(slot)
        kept.append((sim.get_particles(), {k: sim.get_field(k) for k in fields}))
    assert not np.array_equal(kept[0][0]["x"], kept[1][0]["x"])
    for slot in (0, 1, 0):
        sim.restore(slot)
        q = sim.get_particles()
        for k, v in kept[slot][0].items():
            assert np.array_equal(q[k], v), (slot, k)
        for k, v in kept[slot][1].items():
            assert np.array_equal(sim.get_field(k), v), (slot, k)
    sim.close()
