"""Cooperative solves whose blocks have waited for each other in vain, forced
from the host (isph_lose_solves; no kernel waits).  The launched kernels carry
on from the state the launch began with, bit for bit, and the errors that
earlier stages of the step have raised are still reported."""
import numpy as np
import pytest

from beach_slope_confined_amd import capi, configs
from beach_slope_confined_amd.params import PREC_FP64, PREC_MIXED_V64

from parity_util import STAGES, run_stage

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


def overflow_before_the_solve(cfg, seed=1):
    """The configuration with fluid velocities of up to 0.1 dx a step, and its
    longest neighbour list of the search before the solve, which must be longer
    than any of the one after: with max_nbr one less, the step's only error is
    raised before its solve."""
    p, parts = cfg["params"], {k: v.copy() for k, v in cfg["parts"].items()}
    fluid = np.flatnonzero(parts["tid"] == 3)
    v, rng = 0.1 * p.dl / p.dt, np.random.default_rng(seed)
    parts["vx"][fluid] = rng.uniform(-v, v, len(fluid))
    parts["vy"][fluid] = rng.uniform(-v, v, len(fluid))
    cfg = dict(cfg, parts=parts)
    sim = configs.make_sim(cfg, capi.IsphSim)
    longest = []
    for name in STAGES[:STAGES.index("freesurf")]:
        run_stage(sim, name)
        if name == "neighbour":
            longest.append(int(np.diff(sim.get_neighbours()[0]).max()))
    sim.close()
    assert longest[0] > longest[1]
    return dict(cfg, params=p.copy(max_nbr=longest[0] - 1))


@pytest.mark.parametrize("lose", [0, 1])
@pytest.mark.parametrize("precision", [PREC_FP64, PREC_MIXED_V64])
def test_pending_errors_are_reported(require_gpu, lose, precision):
    cfg = configs.dam_break(0.01)
    cfg["params"] = cfg["params"].copy(precision=precision, tol=1e-4)
    sim = configs.make_sim(overflow_before_the_solve(cfg), capi.IsphSim)
    sim.lose_solves(lose)
    with pytest.raises(capi.IsphError, match="ISPH_E_CAPACITY"):
        sim.step(1)
    assert sim.solve_forms()["lost"] == lose
    sim.close()


def test_one_launch_again_after_a_while(require_gpu):
    """Two lost launches in a row keep 64 and then 128 solves kernel by kernel;
    the next one runs in one launch again, and one that is lost later counts
    from 64 anew.  The run's bits are those of one that lost none."""
    sims = [configs.make_sim(configs.dam_break(0.01), capi.IsphSim) for _ in range(2)]
    for lose, launched in ((2, (1 + 64) + (1 + 128)), (1, 1 + 64)):
        before = sims[1].solve_forms()
        sims[1].lose_solves(lose)
        for _ in range(launched + 1):
            for sim in sims:
                sim.step(1)
            now = sims[1].solve_forms()
            if now["resident"] > before["resident"]:
                break
        assert now["lost"] - before["lost"] == lose
        assert now["launched"] - before["launched"] == launched
    a, b = (sim.get_particles() for sim in sims)
    for k in a:
        assert np.array_equal(a[k], b[k]), k
