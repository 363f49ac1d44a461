"""The moments of states larger than the memory-side cache, whose populations are read past the caches,
against sums in float64; vorticity and Q-criterion on velocities large enough for streamed outputs and
for slab-wise blocks, against the same calls on the grid cut into windows that take neither (the sizes
that test_gpu_postprocess.py holds against the oracle, with its tolerances)."""

import numpy as np
import pytest
import torch

import xlb_amd as xa

pytestmark = pytest.mark.gpu

MI = xa.ComputeBackend.MI355X
P = xa.PrecisionPolicy


# the sum of q <= 27 positive terms and its differences: q rounding errors each, and one division
@pytest.mark.parametrize("lattice,shape,policy,tol", [
    ("D3Q19", (173, 151, 137), P.FP32FP32, 2e-6), ("D3Q19", (96, 288, 128), P.FP32FP32, 2e-6),
    ("D3Q19", (211, 190, 181), P.FP32FP16_SHIFTED, 2e-6), ("D3Q19", (149, 113, 107), P.FP64FP64, 5e-15),
    ("D3Q27", (137, 151, 128), P.FP32FP32, 2e-6), ("D2Q9", (3000, 2501), P.FP32FP32, 2e-6),
])
def test_moments_of_large_states(lattice, shape, policy, tol):
    vs = getattr(xa.velocity_set, lattice)(policy, MI)
    xa.init(velocity_set=vs, default_backend=MI, default_precision_policy=policy)
    g = xa.grid.grid_factory(shape)
    f = g.create_field(vs.q, dtype=policy.store_precision)
    gen = torch.Generator(device="cuda").manual_seed(3)
    w, c = np.asarray(vs.w, dtype=np.float64), np.asarray(vs.c)
    shifted = policy == P.FP32FP16_SHIFTED
    rho = torch.zeros(shape, dtype=torch.float64, device="cuda")
    mom = torch.zeros((vs.d,) + tuple(shape), dtype=torch.float64, device="cuda")
    for l in range(vs.q):
        f[l] = (w[l] * 0.2 * torch.rand(f[l].shape, generator=gen, device="cuda") + (0.0 if shifted else w[l])).to(f.dtype)
        v = f[l].reshape(shape).double() + (w[l] if shifted else 0.0)
        rho += v
        for d in range(vs.d):
            if c[d][l]:
                mom[d] += float(c[d][l]) * v
    field = policy.compute_precision
    r, u = xa.operator.macroscopic.Macroscopic()(f, g.create_field(1, dtype=field), g.create_field(vs.d, dtype=field))
    assert ((r.reshape(shape).double() - rho).abs() / rho).max() <= tol
    assert (u.reshape(mom.shape).double() - mom / rho).abs().max() <= tol


# velocities just under and over 16 MB, in slabs with blocks left over, and above 256 MB
@pytest.mark.parametrize("shape,dtype,tol", [
    ((113, 103, 119), torch.float32, 1e-5), ((131, 119, 97), torch.float32, 1e-5), ((3, 701, 700), torch.float32, 1e-5),
    ((101, 83, 97), torch.float64, 1e-13), ((40, 700, 810), torch.float32, 1e-5),
])
@pytest.mark.parametrize("masked", [True, False])
def test_stencils_on_large_velocities(shape, dtype, tol, masked):
    gen = torch.Generator(device="cuda").manual_seed(4)
    u = 0.05 * torch.randn((3,) + shape, generator=gen, device="cuda", dtype=dtype)
    bc = 7 * (torch.rand((1,) + shape, generator=gen, device="cuda") < 0.03).to(torch.uint8) if masked else None
    sentinel = -3.0

    def both(u, bc):
        new = lambda n: torch.full((n,) + tuple(u.shape[1:]), sentinel, dtype=dtype, device="cuda")
        out = [new(3), new(1), new(1), new(1)]
        xa.operator.postprocess.Vorticity()(u, bc, out[0], out[1])
        xa.operator.postprocess.QCriterion()(u, bc, out[2], out[3])
        return out

    whole = both(u, bc)
    side = 128
    for y0 in range(0, shape[1] - 2, side - 2):
        for x0 in range(0, shape[0] - 2, 10):
            x, y = slice(x0, x0 + 12), slice(y0, y0 + side)
            window = both(u[:, x, y].contiguous(), bc[:, x, y].contiguous() if masked else None)
            for got, ref in zip(whole, window):
                got, ref = got[:, x, y][:, 1:-1, 1:-1], ref[:, 1:-1, 1:-1]
                assert torch.equal(got == sentinel, ref == sentinel)
                assert (got - ref).abs().max() <= tol * ref[ref != sentinel].abs().max()
    for got in whole:
        for edge in (got[:, 0], got[:, -1], got[:, :, 0], got[:, :, -1], got[..., 0], got[..., -1]):
            assert bool((edge == sentinel).all())
