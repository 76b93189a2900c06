"""Solves that find column offsets beyond 16 bits and read the int32 columns:
an error that the neighbour search of the same step has raised is still
reported."""
import pytest

from beach_slope_confined_amd import capi, configs
from beach_slope_confined_amd.params import (PREC_FP64, PREC_FP64_MG, PREC_MIXED_MG,
                                             PREC_MIXED_V64)

from test_gpu_errors import tall_column
from test_gpu_lost_wait import overflow_before_the_solve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [PREC_FP64, PREC_MIXED_V64, PREC_MIXED_MG, PREC_FP64_MG])
def test_pending_errors_are_reported(require_gpu, precision):
    cfg = tall_column()
    cfg["params"] = cfg["params"].copy(tol=0.3)
    cfg = overflow_before_the_solve(cfg)
    cfg["params"] = cfg["params"].copy(precision=precision)
    sim = configs.make_sim(cfg, capi.IsphSim)
    with pytest.raises(capi.IsphError, match="ISPH_E_CAPACITY"):
        sim.step(1)
    sim.close()
