"""Runs and recordings of D2Q9 update several steps per launch (xlb_amd/csrc/steps2d.hpp).  Each case
compares them with the caller's loop of single steps, which must agree bit for bit: the same
arithmetic is applied to every cell, so no tolerance is needed."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _stepper(shape, policy, collision, flow, force):
    import xlb_amd as xa

    BC = xa.operator.boundary_condition
    vs = xa.velocity_set.D2Q9(policy, xa.ComputeBackend.MI355X)
    xa.init(velocity_set=vs, default_backend=xa.ComputeBackend.MI355X, default_precision_policy=policy)
    BC.boundary_condition_registry.reset()
    grid = xa.grid.grid_factory(shape, compute_backend=xa.ComputeBackend.MI355X)
    box, inner = grid.bounding_box_indices(), grid.bounding_box_indices(remove_edges=True)

    def faces(*names):
        return torch.unique(torch.cat([torch.tensor(box[n]) for n in names], 1), dim=1).tolist()

    if flow == "periodic":
        bcs = []
    elif flow == "cavity":
        bcs = [BC.EquilibriumBC(rho=1.0, u=(0.03, 0.0), indices=inner["top"]),
               BC.FullwayBounceBackBC(indices=faces("bottom", "left", "right"))]
    elif flow == "still":
        bcs = [BC.DoNothingBC(indices=box["bottom"]), BC.HalfwayBounceBackBC(indices=box["top"])]
    else:
        walls = BC.HalfwayBounceBackBC(indices=faces("bottom", "top"))
        inlet = {"channel": lambda: BC.RegularizedBC("velocity", prescribed_value=(0.04, 0.0), indices=inner["left"]),
                 "zouhe": lambda: BC.ZouHeBC("velocity", prescribed_value=(0.04, 0.0), indices=inner["left"]),
                 "pressure": lambda: BC.RegularizedBC("pressure", prescribed_value=1.01, indices=inner["left"]),
                 "corners": lambda: BC.ZouHeBC("pressure", prescribed_value=1.01, indices=inner["left"])}[flow]()
        bcs = [walls, inlet, BC.ExtrapolationOutflowBC(indices=inner["right"])]
        if flow == "corners":  # an outlet with its corners, whose sources lie up to two cells away
            bcs = [inlet, BC.ExtrapolationOutflowBC(indices=box["right"])]
    kw = {}
    if force == "uniform":
        kw = dict(force_vector=(1e-5, -2e-5))
    elif force == "field":
        gen = torch.Generator().manual_seed(3)
        field = 1e-5 * torch.randn((2,) + shape + (1,), generator=gen, dtype=torch.float64)
        kw = dict(force_field=field.to(policy.compute_precision.torch_dtype).cuda())
    st = xa.operator.stepper.IncompressibleNavierStokesStepper(grid, bcs, collision_type=collision, **kw)
    f_0, f_1, bm, mm = st.prepare_fields()
    gen = torch.Generator().manual_seed(5)
    f_0.copy_((f_0.double() * (1 + 0.05 * torch.rand(f_0.shape, generator=gen, dtype=torch.float64).cuda())).to(f_0.dtype))
    f_1.copy_(f_0.flip(0))  # an older buffer of its own
    return st, f_0, f_1, bm, mm


# grids smaller than a block, at and about its 32 cells and the 8 to 30 it advances, and longer ones
@pytest.mark.parametrize("shape", [(5, 4), (31, 33), (64, 64), (17, 300), (259, 101)])
@pytest.mark.parametrize("flow", ["periodic", "cavity", "still", "channel", "zouhe", "pressure", "corners"])
@pytest.mark.parametrize("policy", ["FP32FP32", "FP64FP64"])
@pytest.mark.parametrize("collision,force", [("BGK", None), ("BGK", "field"), ("BGK", "uniform"),
                                             ("SmagorinskyLESBGK", None), ("KBC", "field")])
def test_run_and_record_equal_single_steps(shape, flow, policy, collision, force):
    import xlb_amd as xa

    st, f_0, f_1, bm, mm = _stepper(shape, xa.PrecisionPolicy[policy], collision, flow, force)
    if flow == "corners":
        from xlb_amd import _lib

        assert st._mask_holds & _lib.MASK_FAR_OUTFLOW
    for steps in (1, 2, 3, 4, 7, 13, 26):
        a0, a1, b0, b1 = f_0.clone(), f_1.clone(), f_0.clone(), f_1.clone()
        a0, a1 = st.run(a0, a1, bm, mm, 1.6, steps)
        kept = st.record(f_0, st.state_buffer(steps, f_0), bm, mm, 1.6, steps)
        for t in range(steps):
            b0, b1 = st(b0, b1, bm, mm, 1.6, t)
            b0, b1 = b1, b0
            assert torch.equal(kept[t], b0), (steps, t, (kept[t] - b0).abs().max())
        assert torch.equal(a0, b0) and torch.equal(a1, b1), (steps, (a0 - b0).abs().max(), (a1 - b1).abs().max())


@pytest.mark.parametrize("lattice,shape", [("D2Q9", (64, 50)), ("D3Q19", (64, 70, 130)), ("D3Q27", (12, 10, 14))])
def test_advance_equals_run_and_leaves_its_start(lattice, shape):
    import xlb_amd as xa

    policy = xa.PrecisionPolicy.FP32FP32
    vs = getattr(xa.velocity_set, lattice)(policy, xa.ComputeBackend.MI355X)
    xa.init(velocity_set=vs, default_backend=xa.ComputeBackend.MI355X, default_precision_policy=policy)
    grid = xa.grid.grid_factory(shape, compute_backend=xa.ComputeBackend.MI355X)
    st = xa.operator.stepper.IncompressibleNavierStokesStepper(grid, [], collision_type="BGK")
    f, _, bm, mm = st.prepare_fields()
    f.mul_(1 + 0.05 * torch.rand(f.shape, generator=torch.Generator().manual_seed(1)).cuda())
    kept = f.clone()
    for steps in (1, 2, 3, 5, 8):
        a, _ = st.run(f.clone(), torch.empty_like(f), bm, mm, 1.5, steps)
        b, other = st.advance(f, torch.empty_like(f), torch.empty_like(f), bm, mm, 1.5, steps)
        assert torch.equal(a, b) and torch.equal(f, kept) and other.data_ptr() != b.data_ptr()
    with pytest.raises(RuntimeError):
        st.advance(f, torch.empty_like(f), f, bm, mm, 1.5, 2)
    with pytest.raises(RuntimeError):
        st.advance(f, torch.empty_like(f), torch.empty_like(f), bm, mm, 1.5, 0)
