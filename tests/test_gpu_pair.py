"""Runs of more than four steps on larger grids update two steps per launch (xlb_amd/csrc/pair.hpp).
Each case compares ``run`` with the caller's loop of single steps, which must agree bit for bit in
both buffers: the same arithmetic is applied to every cell, so no tolerance is needed."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _stepper(shape, policy, collision, walls, dense):
    import xlb_amd as xa

    BC = xa.operator.boundary_condition
    vs = xa.velocity_set.D3Q19(policy, xa.ComputeBackend.MI355X)
    xa.init(velocity_set=vs, default_backend=xa.ComputeBackend.MI355X, default_precision_policy=policy)
    BC.boundary_condition_registry.reset()
    grid = xa.grid.grid_factory(shape, compute_backend=xa.ComputeBackend.MI355X)
    bcs = []
    if walls:
        box, inner = grid.bounding_box_indices(), grid.bounding_box_indices(remove_edges=True)

        def faces(*names):
            return torch.unique(torch.cat([torch.tensor(box[n]) for n in names], 1), dim=1).tolist()

        # ids from 90 on: both sides of the table of constants kept on chip
        BC.boundary_condition_registry.next_id = 90
        kinds = {"halfway": BC.HalfwayBounceBackBC, "fullway": BC.FullwayBounceBackBC, "nothing": BC.DoNothingBC}
        bcs = [BC.EquilibriumBC(rho=1.0, u=(0.02, 0.01, 0.0), indices=inner["top"]),
               kinds[walls](indices=faces("bottom", "left", "front"))]
        BC.boundary_condition_registry.next_id = 200
        rest, taken = torch.tensor(faces("right", "back")), torch.tensor(bcs[1].indices)
        flat = [(t[0] * shape[1] + t[1]) * shape[2] + t[2] for t in (rest, taken)]
        keep = ~torch.isin(*flat)
        bcs.append(BC.HalfwayBounceBackBC(indices=rest[:, keep].tolist()))
        centre = torch.tensor(shape).view(3, 1) // 3
        block = torch.stack(torch.meshgrid(*[torch.arange(5)] * 3, indexing="ij")).reshape(3, -1) + centre
        bcs.append(BC.EquilibriumBC(rho=1.01, u=(0.0, 0.0, -0.01), indices=block.tolist()))
    st = xa.operator.stepper.IncompressibleNavierStokesStepper(grid, bcs, collision_type=collision)
    f_0, f_1, bm, mm = st.prepare_fields()
    gen = torch.Generator(device="cuda").manual_seed(7)
    noise = 1 + 0.05 * torch.rand(f_0.shape, generator=gen, device="cuda", dtype=torch.float64)
    f_0.copy_((f_0.double() * noise).to(f_0.dtype))
    f_1.copy_(f_0.flip(0))  # an older buffer of its own
    if dense:
        f_0, f_1 = f_0.contiguous(), f_1.contiguous()
    return st, f_0, f_1, bm, mm


# nz about whole and part tiles of 64; ny about multiples of the 13 (FP64: 5) rows of a tile; nx odd
@pytest.mark.parametrize("shape", [(101, 130, 128), (97, 118, 129), (131, 117, 127), (64, 13, 2047), (40, 1201, 66)])
@pytest.mark.parametrize("walls", [None, "halfway", "fullway", "nothing"])
@pytest.mark.parametrize("policy,collision", [("FP32FP32", "BGK"), ("FP32FP32", "SmagorinskyLESBGK"),
                                              ("FP32FP32_DEVIATION", "BGK"), ("FP64FP64", "BGK"),
                                              ("FP64FP64", "SmagorinskyLESBGK")])
def test_run_equals_single_steps(shape, walls, policy, collision):
    import xlb_amd as xa

    st, f_0, f_1, bm, mm = _stepper(shape, xa.PrecisionPolicy[policy], collision, walls, dense=shape[0] == 97)
    for steps in (9, 10):
        a0, a1 = f_0.clone(), f_1.clone()
        b0, b1 = f_0.clone(), f_1.clone()
        a0, a1 = st.run(a0, a1, bm, mm, 1.7, steps)
        for t in range(steps):
            b0, b1 = st(b0, b1, bm, mm, 1.7, t)
            b0, b1 = b1, b0
        assert torch.equal(a0, b0) and torch.equal(a1, b1), (steps, (a0 - b0).abs().max(), (a1 - b1).abs().max())
        assert torch.isfinite(a0).all()


def test_short_runs_and_other_kinds_equal_single_steps():
    """Step counts around the switch, and a mask that holds a kind the two-step launch does not take."""
    import xlb_amd as xa

    for extra in (False, True):
        st, f_0, f_1, bm, mm = _stepper((64, 96, 160), xa.PrecisionPolicy.FP32FP32, "BGK", "halfway", False)
        if extra:  # one cell becomes solid
            bm = bm.clone()
            bm[0, 30, 40, 50] = 255
        for steps in range(0, 9):
            a0, a1, b0, b1 = f_0.clone(), f_1.clone(), f_0.clone(), f_1.clone()
            a0, a1 = st.run(a0, a1, bm, mm, 1.3, steps)
            for t in range(steps):
                b0, b1 = st(b0, b1, bm, mm, 1.3, t)
                b0, b1 = b1, b0
            assert torch.equal(a0, b0) and torch.equal(a1, b1), (extra, steps)
