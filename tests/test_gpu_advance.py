"""advance (xlbh_advance) leaves what run leaves on two copies of its start."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lattice,shape", [("D2Q9", (40, 33)), ("D3Q19", (12, 10, 70)), ("D3Q27", (9, 8, 11))])
@pytest.mark.parametrize("policy", ["FP32FP32", "FP64FP64", "FP32FP16_SHIFTED", "FP32I16_BLOCK"])
def test_solid_cells_keep_their_populations(lattice, shape, policy):
    """The buffers hold anything; a solid cell next to fluid is read by it in every step."""
    import xlb_amd as xa

    policy = xa.PrecisionPolicy[policy]
    vs = getattr(xa.velocity_set, lattice)(policy, xa.ComputeBackend.MI355X)
    xa.init(velocity_set=vs, default_backend=xa.ComputeBackend.MI355X, default_precision_policy=policy)
    grid = xa.grid.grid_factory(shape, compute_backend=xa.ComputeBackend.MI355X)
    inner = grid.bounding_box_indices(remove_edges=True)
    bc = xa.operator.boundary_condition.HalfwayBounceBackBC(indices=inner["bottom"])
    st = xa.operator.stepper.IncompressibleNavierStokesStepper(grid, [bc], collision_type="BGK")
    f, scratch, bm, mm = st.prepare_fields()
    bm = bm.clone()
    bm[0, 3:6, 4:6] = 255
    f, _ = st.run(f, scratch, bm, mm, 1.2, 3)

    def copy(seed=None):
        t = st.prepare_fields()[0]
        xa.grid.copy_population(t, f)
        if seed is not None:
            noise = torch.rand(t.shape, generator=torch.Generator().manual_seed(seed))
            t.copy_((noise * (1000 if policy.block else 1)).to(t.dtype))
        return t

    for steps in (1, 2, 5):
        a, _ = st.run(copy(), copy(), bm, mm, 1.2, steps)
        b, _ = st.advance(f, copy(1), copy(2), bm, mm, 1.2, steps)
        assert torch.equal(a, b), steps
        if policy.block:
            assert torch.equal(xa.grid.block_exponents(a), xa.grid.block_exponents(b))
