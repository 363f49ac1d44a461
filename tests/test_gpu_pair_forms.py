"""The two-step launches of D3Q19 (xlb_amd/csrc/pair.hpp) on grids that take them: every case first asks
xlbh_run_launches whether its run is in pairs (from five steps on: the last one is single, and the
number of launches keeps the parity of the steps), then compares it with single steps, bit for bit."""

import pytest
import torch

import xlb_amd as xa
from test_gpu_pair import _stepper
from xlb_amd import _lib

pytestmark = pytest.mark.gpu


def _launches(st, shape, steps):
    return _lib.lib().xlbh_run_launches(st.lattice_id, st._collision_id(), st.precision_policy.store_format, st.compute_id,
                                        int(st._has_bc_cells), _lib.FORCE_NONE, *shape, steps, st._mask_holds, 0)


def _laid_out(f, layout):
    """A copy of f with dense planes, or with planes 192 elements longer."""
    n = f[0].numel()
    plane = n + (192 if layout == "padded" else 0)
    t = torch.full((f.shape[0] * plane,), float("nan"), dtype=f.dtype, device="cuda")
    t = t.as_strided(f.shape, (plane, f.shape[2] * f.shape[3], f.shape[3], 1))
    return t.copy_(f)


def _single(st, f_0, f_1, bm, mm, omega, steps):
    for t in range(steps):
        f_0, f_1 = st(f_0, f_1, bm, mm, omega, t)
        f_0, f_1 = f_1, f_0
    return f_0, f_1


# tiles of z of one, two and 63 cells at the end, of y of a few rows; a whole tile
CASES = [("FP32FP32", (120, 180, 129)), ("FP32FP32", (120, 178, 130)), ("FP32FP32", (40, 199, 193)), ("FP32FP32", (64, 98, 127)),
         ("FP32FP32_DEVIATION", (64, 75, 191)), ("FP64FP64", (120, 138, 129)), ("FP64FP64", (64, 209, 130)),
         ("FP64FP64", (97, 44, 193)), ("FP64FP64", (64, 39, 128))]


@pytest.mark.parametrize("policy,shape", CASES)
@pytest.mark.parametrize("walls", [None, "halfway", "fullway", "nothing"])
@pytest.mark.parametrize("layout", ["dense", "padded"])
def test_pairs_equal_single_steps(policy, shape, walls, layout):
    st, f_0, f_1, bm, mm = _stepper(shape, xa.PrecisionPolicy[policy], "BGK", walls, True)
    for steps in (4, 5, 6, 9):
        assert steps < 5 or _launches(st, shape, steps) < steps
        a = st.run(_laid_out(f_0, layout), _laid_out(f_1, layout), bm, mm, 1.7, steps)
        b = _single(st, f_0.clone(), f_1.clone(), bm, mm, 1.7, steps)
        assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1]), (steps, (a[0] - b[0]).abs().max())
        assert torch.isfinite(a[0]).all()
        assert layout == "dense" or torch.isnan(a[0].as_strided((18, 192), (a[0].stride(0), 1), f_0[0].numel())).all()


@pytest.mark.parametrize("policy,shape", CASES[1:8:3])
@pytest.mark.parametrize("collision", ["BGK", "SmagorinskyLESBGK"])
@pytest.mark.parametrize("walls", [None, "halfway"])
def test_advance_in_pairs(policy, shape, collision, walls):
    if policy == "FP32FP32_DEVIATION" and collision != "BGK":
        policy = "FP32FP32"
    st, f_0, f_1, bm, mm = _stepper(shape, xa.PrecisionPolicy[policy], collision, walls, True)
    kept = f_0.clone()
    for steps in (2, 3, 7):
        assert _launches(st, shape, 5) < 5  # advance has no single step at its end: pairs from two steps on
        a, _ = st.advance(f_0, torch.full_like(f_0, float("nan")), torch.full_like(f_0, float("nan")), bm, mm, 1.7, steps)
        b, _ = _single(st, f_0.clone(), f_1.clone(), bm, mm, 1.7, steps)
        assert torch.equal(a, b) and torch.equal(f_0, kept), steps


@pytest.mark.parametrize("what", ["solid", "outflow"])
def test_other_cells_go_to_single_steps(what):
    """A solid cell, or a kind that the two-step launch does not take, on a grid that would be in pairs."""
    shape = (64, 98, 127)
    st, f_0, f_1, bm, mm = _stepper(shape, xa.PrecisionPolicy.FP32FP32, "BGK", "halfway", True)
    assert _launches(st, shape, 8) < 8
    if what == "solid":
        bm = bm.clone()
        bm[0, 30, 40, 50] = 255
    else:
        outflow = xa.operator.boundary_condition.ExtrapolationOutflowBC(indices=[[30], [40], [50]])
        st.boundary_conditions.append(outflow)
        bm, mm = bm.clone(), mm.clone()
        bm[0, 30, 40, 50] = outflow.id
        mm[1, 30, 40, 50] = True
    for steps in range(0, 9):
        a = st.run(f_0.clone(), f_1.clone(), bm, mm, 1.3, steps)
        assert _launches(st, shape, steps) == steps
        b = _single(st, f_0.clone(), f_1.clone(), bm, mm, 1.3, steps)
        assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1]), steps
