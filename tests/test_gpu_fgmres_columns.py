"""GMRES cycles that end at the edges of the dots' chunks of 8 basis vectors
and of the back substitution's rows of 64 lanes: bit-identical with the
oracle."""
import numpy as np
import pytest

from beach_slope_confined_amd import configs
from beach_slope_confined_amd.params import PREC_FGMRES

from parity_util import STAGES, pair, run_stage

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("restart", [1, 7, 8, 9, 63, 64, 65, 129, 400])
def test_cycle_lengths_bitwise(require_gpu, restart):
    gpu, ora = pair(configs.dam_break(0.01), precision=PREC_FGMRES,
                    tol=1e-2 if restart == 1 else 1e-4 if restart < 60 else 1e-10,
                    maxit=5000, inner_maxit=restart)
    for name in STAGES[:STAGES.index("ppesolve") + 1]:
        print(f"fgmres restart {restart} {name}", flush=True)
        rg = run_stage(gpu, name)
        ro = run_stage(ora, name)
    assert rg == ro
    assert gpu.scalars()["iters"] == ora.scalars()["iters"] >= min(restart, 130)
    assert np.array_equal(gpu.get_particles()["pressure"], ora.get_particles()["pressure"])
