"""How an AXPY is launched, on the CPU: the rule reads no array."""
from ctypes import c_uint32

import pytest

LINE = 1 << 20          # an address on a 128-byte line


def plan_of(xs, n, guarded=0, offset=0, units=256):
    """(chunks, long-lived waves or 0, first chunk that is stored through the L2 or None)"""
    out = (c_uint32 * 3)()
    xs.check(xs.halhip().HipAxpyPlanOf(LINE + 4 * offset, n, guarded, units, out))
    return out[0], out[1], None if out[2] == out[0] else out[2]


@pytest.mark.parametrize("offset,least", [(0, 1 << 21), (1, 1 << 20), (31, 1 << 20)])
def test_short_arrays_are_stored_through_the_l2_where_that_gains(xs, offset, least):
    """One wave per chunk: the shortest lose by it, the kernel then waits for its stores' way to memory."""
    for n in (1, 31, 32, 1 << 12, 1 << 16, 1 << 18, least - 1, least):
        assert plan_of(xs, n, offset=offset)[1:] == (0, None), n
    for n in (least + 1, 3 << 20, 1 << 22):
        assert plan_of(xs, n, offset=offset)[1:] == (0, 0), n
    for n in ((1 << 22) + 1, (1 << 23) - 5000):
        assert plan_of(xs, n, offset=offset)[1:] == (0, None), n


@pytest.mark.parametrize("guarded", [0, 1])
@pytest.mark.parametrize("units", [256, 64, 32])
def test_longer_arrays_are_stored_through_the_l2_by_eight_waves_per_unit_alone(xs, units, guarded):
    """Only their last three quarters: all of it is a loss to arrays that are not in the last-level cache. On fewer compute
    units the sizes are smaller in proportion, so that these stores never meet few waves."""
    least, most = 32768 * units, 65536 * units
    for n in (least + 1024, 3 * least // 2, most):
        chunks, waves, through = plan_of(xs, n, guarded, units=units)
        if waves != 0:          # a plain launch of few chunks has a wave for each
            assert (waves, through) == (8 * units, chunks // 4), n
    for n in (least // 2, least, most + 1024, 2 * most, 16 * most):
        chunks, waves, through = plan_of(xs, n, guarded, units=units)
        assert waves == 0 or through is None, n
        if n > most and waves != 0:
            assert waves == 2 * units, n
    assert plan_of(xs, most, 1, units=units)[2] is not None
