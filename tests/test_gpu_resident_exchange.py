"""The resident BiCGSTAB's exchanges with and without a leader: the same bits
as the launched kernels (csrc/isph_resident.hip) on both sides of the grid
sizes where one gives way to the other."""
import pytest

from beach_slope_confined_amd import configs
from beach_slope_confined_amd.params import PREC_FP64, PREC_IR, PREC_MIXED_V64

from test_gpu_resident import _same

pytestmark = pytest.mark.gpu


# (nside + 6)(nside + 3) rows: 1, 64 and 65, 128 and 129, 159 and 161, 255 and
# 257, 384 and 387 groups of 256
@pytest.mark.parametrize("nside", [10, 123, 124, 176, 177, 197, 198, 251, 252, 309, 310])
def test_grids(require_gpu, nside):
    _same(configs.tank_1m(nside), precision=PREC_FP64)


# FP32 vectors do not converge on the larger tanks, launched or resident
@pytest.mark.parametrize("precision,nside", [(PREC_MIXED_V64, 100), (PREC_MIXED_V64, 150),
                                             (PREC_MIXED_V64, 220), (PREC_MIXED_V64, 300),
                                             (PREC_IR, 100), (PREC_IR, 150)])
def test_values_of_32_bits(require_gpu, precision, nside):
    _same(configs.tank_1m(nside), precision=precision)
