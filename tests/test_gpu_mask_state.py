"""The state a stepper derives from its masks whenever they change."""

import warnings

import pytest
import torch

import xlb_amd as xa
from xlb_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lattice,shape", [("D2Q9", (40, 24)), ("D3Q19", (24, 12, 16))])
@pytest.mark.parametrize("corners", [False, True])
def test_deriving_it_waits_for_the_gpu_twice_at_most(lattice, shape, corners):
    """Walls and an outflow, with and without the corners whose sources are far away: the look-ups
    (any cell, any solid cell, far outflows) come back together; the other wait is the upload of the table."""
    BC = xa.operator.boundary_condition
    policy = xa.PrecisionPolicy.FP32FP32
    vs = getattr(xa.velocity_set, lattice)(policy, xa.ComputeBackend.MI355X)
    xa.init(velocity_set=vs, default_backend=xa.ComputeBackend.MI355X, default_precision_policy=policy)
    grid = xa.grid.grid_factory(shape, compute_backend=xa.ComputeBackend.MI355X)
    box, inner = grid.bounding_box_indices(), grid.bounding_box_indices(remove_edges=True)
    bcs = [BC.ExtrapolationOutflowBC(indices=(box if corners else inner)["right"]), BC.HalfwayBounceBackBC(indices=inner["bottom"])]
    st = xa.operator.stepper.IncompressibleNavierStokesStepper(grid, bcs)
    _, _, bm, mm = st.prepare_fields()
    bm.add_(0)  # another version of the mask
    torch.cuda.synchronize()
    with warnings.catch_warnings(record=True) as caught:
        warnings.simplefilter("always")
        torch.cuda.set_sync_debug_mode("warn")
        try:
            st._sync_state(bm, mm)
        finally:
            torch.cuda.set_sync_debug_mode("default")
    assert len([w for w in caught if "called a synchronizing" in str(w.message)]) <= 2
    assert st._has_bc_cells is True and st._has_solid is False
    assert bool(st._mask_holds & _lib.MASK_FAR_OUTFLOW) == (corners or lattice != "D2Q9")
    assert not st._mask_holds & _lib.MASK_SOLID
    bm[0, 5, 6] = 255
    st._sync_state(bm, mm)
    assert st._has_solid is True and st._mask_holds & _lib.MASK_SOLID
