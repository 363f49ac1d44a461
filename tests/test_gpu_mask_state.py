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


def test_a_new_missing_mask_in_the_place_of_a_freed_one():
    """A tensor that takes the id, the memory and the version of one that was freed is another tensor."""
    BC = xa.operator.boundary_condition
    policy = xa.PrecisionPolicy.FP32FP32
    vs = xa.velocity_set.D2Q9(policy, xa.ComputeBackend.MI355X)
    xa.init(velocity_set=vs, default_backend=xa.ComputeBackend.MI355X, default_precision_policy=policy)
    grid = xa.grid.grid_factory((40, 24), compute_backend=xa.ComputeBackend.MI355X)
    bc = BC.HalfwayBounceBackBC(indices=grid.bounding_box_indices(remove_edges=True)["bottom"])
    st = xa.operator.stepper.IncompressibleNavierStokesStepper(grid, [bc])
    f_0, f_1, bm, mm = st.prepare_fields()
    masks = [mm.cpu(), torch.zeros_like(mm).cpu()]
    taken = set()
    for i in range(20):
        want = masks[i % 2]
        missing = want.cuda()
        place = (id(missing), missing.data_ptr(), missing._version)
        again = place in taken
        taken.add(place)
        st(f_0, f_1, bm, missing, 1.2, 0)
        bits = sum((want[l].reshape(-1).int() << l) for l in range(9))
        assert torch.equal(st._bits.cpu(), bits), (i, again)
        del missing
    assert again  # it did happen here


def test_a_stepper_with_state_can_be_copied_and_pickled():
    """The copy derives its state from the masks it is given; results are the same."""
    import copy
    import pickle

    BC = xa.operator.boundary_condition
    policy = xa.PrecisionPolicy.FP32FP32
    vs = xa.velocity_set.D2Q9(policy, xa.ComputeBackend.MI355X)
    xa.init(velocity_set=vs, default_backend=xa.ComputeBackend.MI355X, default_precision_policy=policy)
    grid = xa.grid.grid_factory((40, 24), compute_backend=xa.ComputeBackend.MI355X)
    inner = grid.bounding_box_indices(remove_edges=True)
    bcs = [BC.HalfwayBounceBackBC(indices=inner["bottom"]), BC.ExtrapolationOutflowBC(indices=inner["right"])]
    st = xa.operator.stepper.IncompressibleNavierStokesStepper(grid, bcs)
    f_0, f_1, bm, mm = st.prepare_fields()
    f_0.mul_(1 + 0.02 * torch.rand(f_0.shape, generator=torch.Generator().manual_seed(1)).cuda())
    want = st.run(f_0.clone(), f_1.clone(), bm, mm, 1.3, 7)[0]
    for other in (copy.deepcopy(st), pickle.loads(pickle.dumps(st))):
        assert torch.equal(other.run(f_0.clone(), f_1.clone(), bm, mm, 1.3, 7)[0], want)
