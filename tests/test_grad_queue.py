"""The queue of contiguous gradients (csrc/walk.cpp): K5's rows, which
gradient is a window's first, and what is left to the caller."""

import numpy as np
import pytest
import torch

from minispeed_amd.contiguous import ACCUM_ROW
from minispeed_amd.flat import _walk

SIZES, OFFSETS, TILE0 = [5, 0, 4100], [0, 5, 5], [0, 1, 1]
ACCUM, SUMSQ, FLAG = 1 << 20, 1 << 30, 1 << 31


def _queue(groups=1):
    q = _walk().GradQueue()
    for g in range(groups):
        q.add_group(0, SIZES, OFFSETS, TILE0, ACCUM + (g << 24), SUMSQ, FLAG)
    return q


def _rows(batch):
    return batch[2].view(ACCUM_ROW).reshape(-1)


@pytest.mark.parametrize("dtype,code", [(torch.float32, 0), (torch.float16, 1), (torch.bfloat16, 2)])
def test_rows(dtype, code):
    q = _queue(2)
    grads = {}
    total = 0
    for gi, k in [(1, 2), (0, 0), (0, 1), (0, 2)]:
        grads[gi, k] = torch.zeros(SIZES[k], dtype=dtype)
        total += SIZES[k]
        assert q.put(gi, k, grads[gi, k]) == total
        assert q.put(gi, k, grads[gi, k]) == q.AGAIN
    (batch,) = q.rows()
    assert batch[0] == 0 and batch[1] == code and q.empty() and q.rows() == []
    order = sorted(grads, key=lambda x: x[0])       # by group, then as they came
    assert [t.data_ptr() for t in batch[3]] == [grads[x].data_ptr() for x in order]
    for row, (gi, k) in zip(_rows(batch), order):
        want = np.array([(ACCUM + (gi << 24) + 4 * OFFSETS[k], grads[gi, k].data_ptr(), SIZES[k], 1, 0,
                          SUMSQ + 8 * TILE0[k], FLAG + 4 * TILE0[k])], dtype=ACCUM_ROW)
        assert row == want[0]


def test_first_of_a_window_and_pointers():
    q, g = _queue(), torch.zeros(5)
    ptrs = np.full(4, 7, dtype=np.int64)
    for window in range(2):
        q.pointers(0, ptrs)
        assert ptrs.tolist() == [0, 0, 0, 7]
        for micro in range(2):
            q.put(0, 0, g)
            (batch,) = q.rows()
            assert _rows(batch)["first"].tolist() == [1 if micro == 0 else 0]
        q.pointers(0, ptrs)
        assert ptrs.tolist() == [ACCUM, 0, 0, 7]
        q.put(0, 2, torch.zeros(4100))      # dropped with its window
        q.next_window()
        assert q.empty()


def test_batches_per_dtype_in_order_of_arrival():
    q = _queue()
    q.put(0, 2, torch.zeros(4100, dtype=torch.bfloat16))
    q.put(0, 0, torch.zeros(5))
    q.put(0, 1, torch.zeros(0, dtype=torch.bfloat16))
    assert [(b[1], len(b[2]), len(b[3])) for b in q.rows()] == [(2, 2, 2), (0, 1, 1)]


def test_left_to_the_caller():
    q, p = _queue(), torch.nn.Parameter(torch.zeros(5))
    assert q.take(0, 0, p) == q.NONE
    p.grad = torch.ones(5)
    assert q.take(0, 0, p) == q.SLOW and p.grad is not None     # a host gradient
    class Sub(torch.Tensor):
        pass
    assert q.take(0, 0, torch.zeros(5).as_subclass(Sub)) == q.SLOW
    assert q.take(0, 0, object()) == q.SLOW
    for bad in (torch.zeros(6), torch.zeros(5, dtype=torch.float64), torch.zeros(10)[::2]):
        with pytest.raises(ValueError):
            q.put(0, 0, bad)
    with pytest.raises(IndexError):
        q.take(1, 0, p)
    assert q.empty()


def test_slots_that_an_earlier_window_left():
    q = _queue()
    assert q.stale_slots(0, 2048) == []
    for k in range(3):
        q.put(0, k, torch.zeros(SIZES[k]))
    q.rows()
    assert q.stale_slots(0, 2048) == []               # all of this window
    q.next_window()
    q.put(0, 2, torch.zeros(4100))
    q.rows()
    assert q.stale_slots(0, 2048) == [(0, 1)]
    q.next_window()
    assert q.stale_slots(0, 2048) == [(1, 4)]         # the first one stays clear
    assert q.stale_slots(0, 2048) == []
    q.put(0, 0, torch.zeros(5))
    q.put(0, 2, torch.zeros(4100))
    q.rows()
    q.next_window()
    assert q.stale_slots(0, 2048) == [(0, 4)]         # neighbours in one range


def test_a_copy_of_the_buffers_has_its_own_queue():
    q = _queue()
    for k in (0, 2):
        q.put(0, k, torch.zeros(SIZES[k]))
    with pytest.raises(ValueError):
        q.rebased([(8, 16, 24)])                      # something is queued
    q.rows()
    with pytest.raises(ValueError):
        q.rebased([])
    c, ptrs = q.rebased([(ACCUM + 64, SUMSQ + 64, FLAG + 64)]), np.zeros(3, dtype=np.int64)
    c.pointers(0, ptrs)
    assert ptrs.tolist() == [ACCUM + 64, 0, ACCUM + 64 + 4 * OFFSETS[2]]
    g = torch.zeros(SIZES[2])
    c.put(0, 2, g)
    assert q.empty()
    (batch,) = c.rows()
    assert _rows(batch).tolist() == [(ACCUM + 64 + 4 * OFFSETS[2], g.data_ptr(), SIZES[2], 0, 0,
                                      SUMSQ + 64 + 8 * TILE0[2], FLAG + 64 + 4 * TILE0[2])]
    c.next_window()
    assert c.stale_slots(0, 2048) == [(0, 4)] and q.stale_slots(0, 2048) == []
