"""Multigrid solves whose kernels finish the reductions themselves (up to 1024
partials) and those of k_finish beyond: iterations and pressures' bits are
those recorded with k_finish's launches at every size, at few partials, at
the edges of a wave of them and on both sides of the limit."""
import hashlib

import pytest

from beach_slope_confined_amd import capi, configs
from beach_slope_confined_amd.params import PREC_MIXED_MG

pytestmark = pytest.mark.gpu

PRE = ("projection", "cellshift", "resetid", "neighbour", "effpor", "eddyvis", "int_vel")
# (side of the tank, particles, iterations, pressures)
RECORDED = [
    (12, 270, 11, "fa55dcfda8c3ed43"),
    (119, 15250, 15, "c77b11ef144db209"),
    (120, 15498, 16, "2800daa7dd5daf66"),
    (124, 16510, 19, "b677e9195d9ba4a1"),
    (250, 64768, 17, "4ef2ced0b06997dc"),
    (507, 261630, 20, "9e0b4ade22e6f4c5"),
    (508, 262654, 19, "ab66c3baab8e664d"),
]


@pytest.mark.parametrize("side,n,iters,digest", RECORDED)
def test_partials(require_gpu, side, n, iters, digest):
    cfg = dict(configs.tank_1m(side))
    cfg["params"] = cfg["params"].copy(precision=PREC_MIXED_MG, tol=1e-9)
    sim = configs.make_sim(cfg, capi.IsphSim)
    s = sim.scalars()
    sim.set_scalars(s["umax"], s["dt"], s["t"] + s["dt"])
    for st in PRE:
        getattr(sim, st)()
    assert sim.count() == n
    assert sim.ppesolve()[0] == iters
    x = sim.get_field("pressure")
    assert hashlib.sha256(x.tobytes()).hexdigest()[:16] == digest
    sim.close()


@pytest.mark.parametrize("maxit", [1, 3, 4, 5, 9])
def test_iteration_limit(require_gpu, maxit):
    """The limit holds wherever it falls in the iterations enqueued at once."""
    cfg = dict(configs.tank_1m(120))
    cfg["params"] = cfg["params"].copy(precision=PREC_MIXED_MG, tol=1e-9, maxit=maxit)
    sim = configs.make_sim(cfg, capi.IsphSim)
    s = sim.scalars()
    sim.set_scalars(s["umax"], s["dt"], s["t"] + s["dt"])
    for st in PRE:
        getattr(sim, st)()
    with pytest.raises(capi.IsphError, match="NOCONV"):
        sim.ppesolve()
    assert sim.scalars()["iters"] == maxit
    sim.close()
