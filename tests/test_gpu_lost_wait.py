"""Cooperative solves whose blocks have waited for each other in vain, forced
from the host (isph_lose_solves; no kernel waits).  The launched kernels carry
on from the state the launch began with, bit for bit, and the errors that
earlier stages of the step have raised are still reported."""
import numpy as np
import pytest

from beach_slope_confined_amd import capi, configs
from beach_slope_confined_amd.params import PREC_FP64, PREC_MIXED_V64

pytestmark = pytest.mark.gpu


# without a leader, with one in blocks of 512 and of 1024 rows, streamed
@pytest.mark.parametrize("nside", [40, 330, 430, 520])
@pytest.mark.parametrize("precision", [PREC_FP64, PREC_MIXED_V64])
def test_the_launched_kernels_take_over(require_gpu, nside, precision):
    out = []
    cfg = configs.tank_1m(nside)
    cfg["params"] = cfg["params"].copy(precision=precision, tol=1e-4)
    for lose in (0, 1):
        sim = configs.make_sim(cfg, capi.IsphSim)
        sim.lose_solves(lose)
        sim.step(1)
        f = sim.solve_forms()
        one = f["resident"] + f["streamed"]
        if lose:
            assert f["lost"] == 1 and f["launched"] and not one
        else:
            assert one and not f["launched"] and not f["lost"]
        out.append((sim.scalars(), sim.get_particles()))
        sim.close()
    assert out[0][0] == out[1][0]
    for k, v in out[0][1].items():
        assert np.array_equal(v, out[1][1][k]), k


@pytest.mark.parametrize("lose", [0, 1])
@pytest.mark.parametrize("precision", [PREC_FP64, PREC_MIXED_V64])
def test_pending_errors_are_reported(require_gpu, lose, precision):
    cfg = configs.dam_break(0.01)
    cfg["params"] = cfg["params"].copy(precision=precision, tol=1e-4)
    sim = configs.make_sim(cfg, capi.IsphSim)
    sim.neighbour()
    longest = int(np.diff(sim.get_neighbours()[0]).max())
    sim.close()
    cfg["params"] = cfg["params"].copy(max_nbr=longest - 1)
    sim = configs.make_sim(cfg, capi.IsphSim)
    sim.lose_solves(lose)
    with pytest.raises(capi.IsphError, match="ISPH_E_CAPACITY"):
        sim.step(1)
    assert sim.solve_forms()["lost"] == lose
    sim.close()
