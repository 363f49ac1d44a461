"""Runs whose caller says what the boundary mask holds (xlbh_run_known, xlbh_record_known): for every
boundary kind the populations are those of xlbh_run and xlbh_record, bit for bit."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lattice,shape", [("D2Q9", (70, 45)), ("D3Q19", (101, 130, 128))])
@pytest.mark.parametrize("kind", range(11))
def test_every_kind_as_without_the_knowledge(lattice, shape, kind):
    """One plane of cells of each kind id, through the C entries with the bit of that kind alone: a
    kind that a launch of several steps does not implement has to go to single steps."""
    import xlb_amd as xa
    from xlb_amd import _lib

    policy = xa.PrecisionPolicy.FP32FP32
    vs = getattr(xa.velocity_set, lattice)(policy, xa.ComputeBackend.MI355X)
    xa.init(velocity_set=vs, default_backend=xa.ComputeBackend.MI355X, default_precision_policy=policy)
    grid = xa.grid.grid_factory(shape, compute_backend=xa.ComputeBackend.MI355X)
    inner = grid.bounding_box_indices(remove_edges=True)
    bc = xa.operator.boundary_condition.HalfwayBounceBackBC(indices=inner["left"])
    st = xa.operator.stepper.IncompressibleNavierStokesStepper(grid, [bc], collision_type="BGK")
    f, _, bm, mm = st.prepare_fields()
    f = f.contiguous() * (1 + 0.02 * torch.rand(f.shape, generator=torch.Generator().manual_seed(1)).cuda())
    nx, ny, nz, plane, masks, mode, _, _, _ = st._launch_args(f, None, bm, mm)
    table = (_lib.BcDesc * 256)()
    table[bc.id].kind, table[bc.id].rho = kind, 1.01
    table[bc.id].u[0] = 0.02
    table = torch.frombuffer(bytearray(bytes(table)), dtype=torch.uint8).cuda()
    aux = torch.full((nx * ny * nz,), 0.03 if kind in (_lib.BC_ZOUHE_VELOCITY, _lib.BC_REGULARIZED_VELOCITY) else 1.01,
                     device="cuda")
    args = (masks[0], masks[1], _lib.ptr(aux), _lib.ptr(table), mode, None, None, nx, ny, nz, plane, 1.6, 0.0, 0)
    known, L, s = 1 << _lib.BC_NONE | 1 << kind, _lib.lib(), _lib.stream_of(f)
    ids = (st.lattice_id, st._collision_id(), policy.store_format, policy.compute_id)
    steps = 11
    a, b, c, d = f.clone(), f.flip(0), f.clone(), f.flip(0)
    _lib.check(L.xlbh_run(*ids, _lib.ptr(a), _lib.ptr(b), *args, steps, s))
    _lib.check(L.xlbh_run_known(*ids, _lib.ptr(c), _lib.ptr(d), *args, steps, known, s))
    assert torch.isfinite(a).all()
    assert torch.equal(a, c) and torch.equal(b, d)
    kept, known_kept = st.state_buffer(steps, f), st.state_buffer(steps, f)
    _lib.check(L.xlbh_record(*ids, _lib.ptr(f), _lib.ptr(kept), *args, steps, s))
    _lib.check(L.xlbh_record_known(*ids, _lib.ptr(f), _lib.ptr(known_kept), *args, steps, known, s))
    assert torch.equal(kept, known_kept)
