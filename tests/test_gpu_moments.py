"""Density, velocity and second moment at the edges of the launch (k_moments takes one cell after
another): cell counts about whole blocks of 256, single rows, dense and padded planes, every store."""

import numpy as np
import pytest
import torch

import xlb_amd as xa

pytestmark = pytest.mark.gpu

MI = xa.ComputeBackend.MI355X


@pytest.mark.parametrize("lattice,shape", [("D2Q9", (1, 1)), ("D2Q9", (5, 51)), ("D2Q9", (16, 16)), ("D2Q9", (1, 257)),
                                           ("D3Q19", (1, 1, 2)), ("D3Q19", (5, 3, 17)), ("D3Q19", (4, 2, 129)),
                                           ("D3Q27", (2, 2, 64)), ("D3Q27", (3, 7, 73))])
@pytest.mark.parametrize("policy", ["FP32FP32", "FP64FP64", "FP64FP32", "FP32FP16", "FP32BF16_SHIFTED", "FP32I16_BLOCK"])
@pytest.mark.parametrize("padded", [False, True])
def test_moments_against_sums(lattice, shape, policy, padded):
    """q <= 27 terms below 1 and their differences, then one division: 2e-6 in FP32, 5e-15 in FP64."""
    policy = xa.PrecisionPolicy[policy]
    vs = getattr(xa.velocity_set, lattice)(policy, MI)
    xa.init(velocity_set=vs, default_backend=MI, default_precision_policy=policy)
    grid = xa.grid.grid_factory(shape, compute_backend=MI)
    three = tuple(shape) + (1,) * (3 - len(shape))
    w, c = torch.tensor(np.asarray(vs.w), dtype=torch.float64).cuda(), torch.tensor(np.asarray(vs.c)).double().cuda()
    gen = torch.Generator().manual_seed(4)
    value = w.view(-1, 1, 1, 1) * (1 + 0.2 * torch.rand((vs.q,) + three, generator=gen, dtype=torch.float64).cuda())
    f = grid.create_field(vs.q, dtype=policy.store_precision, padded=True) if padded or policy.block else grid.create_field(
        vs.q, dtype=policy.store_precision)
    if policy.block:
        flat = torch.zeros((vs.d,) + three, device="cuda")
        xa.operator.equilibrium.QuadraticEquilibrium()(1 + 0.1 * torch.rand((1,) + three, generator=gen).cuda(), flat, f)
    else:
        f.copy_((value - (w.view(-1, 1, 1, 1) if policy.shifted else 0.0)).to(f.dtype))
    value = xa.grid.decode_populations(f, vs.w, block=policy.block, shifted=policy.shifted)
    tol = 5e-15 if policy.compute_precision == xa.Precision.FP64 else 2e-6
    new = lambda n: torch.full((n,) + three, float("nan"), dtype=policy.compute_precision.torch_dtype, device="cuda")
    rho, u = xa.operator.macroscopic.Macroscopic()(f, new(1), new(vs.d))
    want = value.sum(0, keepdim=True)
    mom = torch.stack([(c[d].view(-1, 1, 1, 1) * value).sum(0) for d in range(vs.d)])
    assert (rho.double() - want).abs().max() <= tol and (u.double() - mom / want).abs().max() <= tol
    alone = xa.operator.macroscopic.ZeroMoment()(f, new(1))
    given = xa.operator.macroscopic.FirstMoment()(f, rho, new(vs.d))
    assert torch.equal(alone, rho) and (given.double() - mom / want).abs().max() <= tol
    pairs = [(a, b) for a in range(vs.d) for b in range(a, vs.d)]
    pi = xa.operator.macroscopic.SecondMoment()(f, new(len(pairs)))
    for t, (a, b) in enumerate(pairs):
        ref = ((c[a] * c[b]).view(-1, 1, 1, 1) * value).sum(0)
        assert (pi[t].double() - ref).abs().max() <= tol
