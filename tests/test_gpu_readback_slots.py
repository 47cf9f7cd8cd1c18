"""The pinned slots K2's host result goes to."""

import pytest

from minispeed_amd import _native
from minispeed_amd.boundary import HostReadback, _PinnedSlots

pytestmark = pytest.mark.gpu


def test_slots_are_apart_and_come_back():
    many = [HostReadback() for _ in range(3 * _PinnedSlots.SLAB // _PinnedSlots.SLOT)]
    starts = sorted(r.ptr for r in many)
    assert all(b - a >= _native.SCALARS_BYTES for a, b in zip(starts, starts[1:]))
    assert all(p % _PinnedSlots.SLOT == 0 for p in starts) and all(r.host.is_pinned() for r in many)
    last = many.pop()
    ptr, r = last.ptr, None
    del last
    assert ptr in {r.ptr for r in [HostReadback() for _ in range(_PinnedSlots.SLAB // _PinnedSlots.SLOT)]}


def test_a_slot_that_a_kernel_may_still_write_is_not_reused():
    r = HostReadback()
    r.arm()
    ptr = r.ptr
    del r
    assert ptr not in {r.ptr for r in [HostReadback() for _ in range(200)]}


def test_a_result_is_read_and_frees_its_slot():
    r = HostReadback()
    r.arm()
    r._ready[0] = 1
    assert r.wait(0).ready == 1 and not r._pending[0]
