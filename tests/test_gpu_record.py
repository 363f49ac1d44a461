"""Recordings that start inside the buffer they write (xlbh_record)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lattice,shape", [("D2Q9", (1500, 1100)), ("D2Q9", (40, 31)), ("D3Q19", (24, 20, 36))])
@pytest.mark.parametrize("at", [1, -1])
def test_a_recording_may_start_from_a_state_it_overwrites(lattice, shape, at):
    """states[at] is read by the first step only, so recording over it gives what recording into
    another buffer gives, bit for bit (1500 x 1100: more blocks than run at once, so that some would
    read it after others wrote it)."""
    import xlb_amd as xa

    policy = xa.PrecisionPolicy.FP32FP32
    vs = getattr(xa.velocity_set, lattice)(policy, xa.ComputeBackend.MI355X)
    xa.init(velocity_set=vs, default_backend=xa.ComputeBackend.MI355X, default_precision_policy=policy)
    grid = xa.grid.grid_factory(shape, compute_backend=xa.ComputeBackend.MI355X)
    st = xa.operator.stepper.IncompressibleNavierStokesStepper(grid, [], collision_type="BGK")
    f, _, bm, mm = st.prepare_fields()
    f = f.contiguous() * (1 + 0.05 * torch.rand(f.shape, generator=torch.Generator().manual_seed(1)).cuda())
    n = 9
    want = st.record(f, st.state_buffer(n, f), bm, mm, 1.5, n)
    states = st.state_buffer(n, f)
    states[at].copy_(f)
    st.record(states[at], states, bm, mm, 1.5, n)
    assert torch.equal(states, want)
