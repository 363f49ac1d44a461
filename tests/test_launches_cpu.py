"""How many steps a launch does (xlbh_run_launches, which needs no GPU): the rules behind xlbh_run_known
and xlbh_record_known."""

import pytest

from xlb_amd import _lib

L = _lib.lib()
KINDS = (1 << 10) - 1  # ids without an entry and every boundary kind but Grad's approximation


def launches(shape, n, lattice=_lib.D2Q9, collision=_lib.BGK, store=_lib.F32, compute=_lib.COMPUTE_F32, mask=0,
             force=_lib.FORCE_NONE, known=KINDS, keep=0):
    shape = tuple(shape) + (1,) * (3 - len(shape))
    return L.xlbh_run_launches(lattice, collision, store, compute, mask, force, *shape, n, known, keep)


F64 = dict(store=_lib.F64, compute=_lib.COMPUTE_F64)


@pytest.mark.parametrize("shape,options", [((64, 64), {}), ((64, 64), F64), ((512, 256), dict(mask=1)),
                                           ((256, 256, 256), dict(lattice=_lib.D3Q19)), ((40, 30, 20), dict(lattice=_lib.D3Q27))])
def test_runs_keep_the_parity_of_their_steps(shape, options):
    """As many launches as steps modulo two, so that the newest state is in the buffer that the number of
    steps selects; never more launches than steps, and for a recording as few as the steps per launch."""
    for n in range(60):
        got = launches(shape, n, **options)
        assert 0 < got <= n or got == n == 0
        assert (got - n) % 2 == 0
        assert (n > 0) <= launches(shape, n, keep=1, **options) <= n


@pytest.mark.parametrize("shape", [(64, 64), (200, 200), (512, 256), (1024, 512)])
@pytest.mark.parametrize("options", [{}, F64, dict(mask=1), dict(mask=1, force=_lib.FORCE_FIELD)])
def test_several_steps_where_the_launch_takes_the_time(shape, options):
    assert launches(shape, 100, **options) <= 40


# a block covers little of a thin grid; KBC is bound by its arithmetic on large ones
@pytest.mark.parametrize("shape,options", [
    ((1, 60000), {}), ((2, 50569), F64), ((4, 26001), F64),
    ((2, 44327), dict(collision=_lib.KBC, **F64)), ((1728, 2331), dict(collision=_lib.KBC, mask=1)),
    ((1994, 1252), dict(collision=_lib.KBC, mask=1, **F64)),
])
def test_single_steps_where_they_take_less_time(shape, options):
    assert launches(shape, 50, **options) == 50


@pytest.mark.parametrize("shape", [(1728, 1331), (1684, 1228)])
@pytest.mark.parametrize("options", [{}, dict(mask=1), F64])
def test_large_recordings_write_each_state_once(shape, options):
    """Every state is written in segments of a block's rows, which costs more than the launches saved."""
    assert launches(shape, 50, keep=1, **options) == 50


@pytest.mark.parametrize("shape,lattice", [((64, 64), _lib.D2Q9), ((256, 256, 256), _lib.D3Q19)])
def test_only_kinds_the_kernels_implement(shape, lattice):
    few = 1 << _lib.BC_NONE | 1 << _lib.BC_HALFWAY_BB
    assert launches(shape, 50, lattice=lattice, mask=1, known=few) < 50
    for more in (_lib.MASK_SOLID, _lib.MASK_FAR_OUTFLOW, 1 << _lib.BC_GRADS_APPROXIMATION, 0xFFFFFFFF):
        assert launches(shape, 50, lattice=lattice, mask=1, known=few | more) == 50
        assert launches(shape, 50, lattice=lattice, mask=0, known=few | more) < 50  # no mask, nothing to know
    assert launches(shape, 50, lattice=lattice, store=_lib.F16) == 50
    assert launches(shape, -1, lattice=lattice) == -1 and b"n_steps" in L.xlbh_last_error()
    assert launches(shape, 5, lattice=7) == -1 and b"lattice" in L.xlbh_last_error()
