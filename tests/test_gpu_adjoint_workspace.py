"""The fused reverse sweep's workspace: its contents before the sweep do not matter, and its segments
may have different masks.  Compared with the two-kernel reverse step, which carries nothing from step
to step, in FP64: 1e-12 of the norm, some thousand roundings."""

import pytest
import torch

import xlb_amd as xa

pytestmark = pytest.mark.gpu

SHAPES = {"D2Q9": (23, 18), "D3Q19": (9, 8, 70), "D3Q27": (7, 6, 9)}


def _stepper(lattice, collision="BGK", bcs=None, policy=xa.PrecisionPolicy.FP64FP64, shape=None):
    vs = getattr(xa.velocity_set, lattice)(policy, xa.ComputeBackend.MI355X)
    xa.init(velocity_set=vs, default_backend=xa.ComputeBackend.MI355X, default_precision_policy=policy)
    grid = xa.grid.grid_factory(shape or SHAPES[lattice], compute_backend=xa.ComputeBackend.MI355X)
    st = xa.operator.stepper.IncompressibleNavierStokesStepper(grid, bcs(grid) if bcs else [], collision_type=collision)
    f, _, bm, mm = st.prepare_fields()
    noise = 0.05 * torch.rand(f.shape, generator=torch.Generator().manual_seed(2), dtype=torch.float64)
    return st, f.contiguous() * (1 + noise.cuda()).to(f.dtype), bm, mm


def _nan_workspace(st, bm):
    return st.adjoint_workspace(bm).fill_(255)  # every value in it reads as NaN


@pytest.mark.parametrize("lattice", sorted(SHAPES))
@pytest.mark.parametrize("later", ["no mask", "fewer walls"])
def test_segments_with_different_masks(lattice, later):
    """Walls that are there in the first segment only: the later one, which the sweep goes through
    first, leaves nothing at their cells."""
    BC = xa.operator.boundary_condition

    def walls(grid):
        inner = grid.bounding_box_indices(remove_edges=True)
        return [BC.HalfwayBounceBackBC(indices=inner["bottom"]), BC.HalfwayBounceBackBC(indices=inner["top"])]

    st, f, bm, mm = _stepper(lattice, bcs=walls)
    gone = torch.zeros_like(bm) if later == "no mask" else torch.where(bm == 1, bm, torch.zeros_like(bm))
    assert (gone != bm).any()
    n, omega = 4, 1.3
    masks = [bm, gone]  # of the earlier and of the later segment
    starts, states = [f], []
    for m in masks:
        states.append(st.record(starts[-1], st.state_buffer(n, f), m, mm, omega, n))
        starts.append(states[-1][n - 1].clone())
    lam = torch.randn(f.shape, generator=torch.Generator().manual_seed(3), dtype=torch.float64).cuda()
    want = lam.clone()
    for seg in (1, 0):
        for j in range(n - 1, -1, -1):
            f_t = starts[seg] if j == 0 else states[seg][j - 1]
            want = st.adjoint_step(f_t, want, torch.empty_like(want), masks[seg], mm, omega)
    ws = _nan_workspace(st, bm)
    a, b = lam.clone(), torch.empty_like(lam)
    for seg in (1, 0):
        out = st.adjoint_run(starts[seg], states[seg], a, b, masks[seg], mm, omega, n, timestep=seg * n, recompute=False,
                             workspace=ws, begin=seg == 1, end=seg == 0)
        a, b = (a, b) if out is a else (b, a)
    assert ((a - want).norm() / want.norm()).item() <= 1e-12


# rows of z: part of a wave, several waves with a ragged end, whole 128-byte lines
@pytest.mark.parametrize("lattice,shape", [("D2Q9", (23, 18)), ("D2Q9", (9, 130)), ("D3Q19", (6, 5, 77)),
                                           ("D3Q19", (5, 6, 130)), ("D3Q19", (4, 5, 96)), ("D3Q27", (5, 4, 33))])
@pytest.mark.parametrize("collision", ["BGK", "SmagorinskyLESBGK"])
@pytest.mark.parametrize("walls", [False, True])
@pytest.mark.parametrize("every", [1, 2, 4])
def test_sweep_equals_two_kernel_steps_whatever_the_workspace_held(monkeypatch, lattice, shape, collision, walls, every):
    BC = xa.operator.boundary_condition

    def channel(grid):
        box, inner = grid.bounding_box_indices(), grid.bounding_box_indices(remove_edges=True)
        two = [torch.tensor(box[k]) for k in ("bottom", "top")]
        return [BC.HalfwayBounceBackBC(indices=torch.unique(torch.cat(two, 1), dim=1).tolist()),
                BC.ExtrapolationOutflowBC(indices=inner["right"])]

    st, f, bm, mm = _stepper(lattice, collision, channel if walls else None, shape=shape)
    monkeypatch.setattr(st, "adjoint_workspace", lambda m, make=st.adjoint_workspace: make(m).fill_(255))
    lam = torch.randn(f.shape, generator=torch.Generator().manual_seed(3), dtype=torch.float64).cuda()
    got = []
    for fused in (True, False):
        f0 = f.clone().requires_grad_()
        out = xa.autodiff.rollout(st, f0, bm, mm, 1.4, 9, checkpoint_every=every, fused=fused)
        got.append(torch.autograd.grad(out, f0, lam)[0])
    assert ((got[0] - got[1]).norm() / got[1].norm()).item() <= 1e-12
