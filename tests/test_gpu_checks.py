"""Calls that are refused before anything is launched."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["store", "bf16", "bf16_shifted"])
@pytest.mark.parametrize("wrong", ["host", "planes", "extents"])
def test_rollout_checks_its_state_before_the_first_checkpoint(mode, wrong):
    """A state on the host, or of another shape than the masks', is refused for every checkpoint
    format (the codec's kernel would read the missing planes)."""
    import xlb_amd as xa

    policy = xa.PrecisionPolicy.FP32FP32
    vs = xa.velocity_set.D2Q9(policy, xa.ComputeBackend.MI355X)
    xa.init(velocity_set=vs, default_backend=xa.ComputeBackend.MI355X, default_precision_policy=policy)
    grid = xa.grid.grid_factory((20, 12), compute_backend=xa.ComputeBackend.MI355X)
    st = xa.operator.stepper.IncompressibleNavierStokesStepper(grid, [])
    f, _, bm, mm = st.prepare_fields()
    bad = {"host": f.cpu(), "planes": f[:8].contiguous(), "extents": f[:, :19].contiguous()}[wrong]
    with pytest.raises(ValueError):
        xa.autodiff.rollout(st, bad, bm, mm, 1.2, 3, checkpoint_dtype=mode)
