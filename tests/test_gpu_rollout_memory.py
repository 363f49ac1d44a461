"""Memory of a rollout's forward pass."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["store", "bf16", "bf16_shifted"])
def test_forward_pass_holds_two_fields_beside_its_checkpoints(mode):
    """The peak of the forward pass: its checkpoints and two population fields, and while a shifted
    checkpoint is encoded one more (its temporary).  Every allocation is a whole number of MB, so that
    the allocator's rounding of large blocks adds nothing."""
    import xlb_amd as xa

    policy = xa.PrecisionPolicy.FP32FP32
    vs = xa.velocity_set.D3Q19(policy, xa.ComputeBackend.MI355X)
    xa.init(velocity_set=vs, default_backend=xa.ComputeBackend.MI355X, default_precision_policy=policy)
    grid = xa.grid.grid_factory((64, 64, 128), compute_backend=xa.ComputeBackend.MI355X)
    st = xa.operator.stepper.IncompressibleNavierStokesStepper(grid, [])
    f, _, bm, mm = st.prepare_fields()
    f = f.contiguous().requires_grad_()
    field = f.numel() * f.element_size()
    xa.autodiff.rollout(st, f, bm, mm, 1.2, 4, checkpoint_every=2, checkpoint_dtype=mode)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    base = torch.cuda.memory_allocated()
    out = xa.autodiff.rollout(st, f, bm, mm, 1.2, 4, checkpoint_every=2, checkpoint_dtype=mode)
    kept = torch.cuda.memory_allocated() - base - field  # all but the output
    peak = torch.cuda.max_memory_allocated() - base
    assert out.shape == f.shape and kept > 0
    slack = field if mode == "bf16_shifted" else 0
    assert peak <= kept + 2 * field + slack + (1 << 20), (peak / field, kept / field)
