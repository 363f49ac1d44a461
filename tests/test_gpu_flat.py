"""Single steps on 3-D grids whose rows do not fill the sweep's tiles take 256 consecutive cells of an
x-plane per block (step_body's FLAT form), with stores by row alignment: parity with the oracle at
the sizes about those edges, with the tolerances of tests/test_gpu_stepper.py."""

import pytest

import lbm_cases
import xlb_amd as xa
from lbm_cases import Pair
from test_gpu_stepper import compare

pytestmark = pytest.mark.gpu

P = xa.PrecisionPolicy


# ny * nz below, at and above 256 cells; nz about 64, 128 and 256 and at multiples of 32 (whole lines)
@pytest.mark.parametrize("shape", [(4, 5, 7), (3, 8, 32), (5, 4, 63), (3, 5, 65), (4, 3, 127), (2, 6, 129), (3, 4, 255),
                                   (4, 5, 257), (3, 7, 96), (2, 9, 320)])
@pytest.mark.parametrize("lattice,collision,bcs,init", [("D3Q19", "BGK", "periodic", "random"),
                                                        ("D3Q19", "SmagorinskyLESBGK", "cavity_halfway", "random"),
                                                        ("D3Q27", "BGK", "cavity_fullway", "rest")])
@pytest.mark.parametrize("policy", [P.FP32FP32, P.FP64FP64, P.FP32FP16_SHIFTED])
def test_ragged_rows_match_oracle(monkeypatch, shape, lattice, collision, bcs, init, policy):
    monkeypatch.setitem(lbm_cases.LARGE_CASES, "ragged", (lattice, shape, collision, 1.6, init))
    monkeypatch.setitem(lbm_cases.BC_SET, "ragged", bcs)
    compare(Pair("ragged", policy), 6)
