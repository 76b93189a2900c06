"""Multigrid solves with wide cells: more rows in a block's cells than it keeps
in LDS (k_mg_down0).  The iterations and the pressures' bits are those of the
kernels that formed and restricted the residual in two launches, recorded
before the two were joined."""
import hashlib

import pytest

from beach_slope_confined_amd import capi, configs
from beach_slope_confined_amd.params import PREC_FP64_MG, PREC_MIXED_MG

pytestmark = pytest.mark.gpu

PRE = ("projection", "cellshift", "resetid", "neighbour", "effpor", "eddyvis", "int_vel")
# at most 9, 16, 47 and 121 particles a cell: 64 cells fill the LDS from 17 on
RECORDED = [
    (1.0, PREC_MIXED_MG, 20, "af7526e952e38b3f"),
    (1.5, PREC_FP64_MG, 22, "ee0b1744f63eb15e"),
    (2.5, PREC_MIXED_MG, 38, "10e19348e75a53eb"),
    (4.0, PREC_MIXED_MG, 59, "b246d93149f9168a"),
    (4.0, PREC_FP64_MG, 64, "b728b4d901b55ad7"),
]


@pytest.mark.parametrize("wide,precision,iters,digest", RECORDED)
def test_wide_cells(require_gpu, wide, precision, iters, digest):
    cfg = dict(configs.dam_break(0.005))
    p = cfg["params"]
    cfg["params"] = p.copy(precision=precision, tol=1e-9, maxit=20000,
                           cell_size=wide * p.cell_size)
    sim = configs.make_sim(cfg, capi.IsphSim)
    s = sim.scalars()
    sim.set_scalars(s["umax"], s["dt"], s["t"] + s["dt"])
    for st in PRE:
        getattr(sim, st)()
    assert sim.ppesolve()[0] == iters
    x = sim.get_field("pressure")
    assert hashlib.sha256(x.tobytes()).hexdigest()[:16] == digest
    sim.close()
