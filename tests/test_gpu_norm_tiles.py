"""K2 reading the tile statistics of small groups itself
(``ms_norm_clip_tiles``): bit for bit the fold into partial slots followed by
``ms_norm_clip``, on both sides of the line (``ms_stats_blocks()`` tiles), for
one group and for more groups than travel in the kernel arguments; and the
reading K1 on both sides of its short-scan line (6144 tiles), whose tile
slots must equal the writing K1's; and K1 over one contiguous buffer without a
segment table (``ms_buffer_tile_stats``, ``ms_buffer_scale``), bit for bit the
scan of a one-row table, torch's ``div_`` and ``mul_``."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from minispeed_amd import _native

DEV = "cuda:0"


def test_arguments_refused_on_the_host():
    lib = _native.load()
    nb = _native.stats_blocks()
    tail = (0, 0.0, 0, 1.0, 0, 0, 1, 1.0, 1.0)
    groups = (_native.TileStats * 1)(_native.TileStats(None, None, 5))
    call = lib.ms_norm_clip_tiles
    assert call(groups, 1, 8, 8, nb, *tail, 8, None, None) == -1          # tiles without slots
    groups[0] = _native.TileStats(8, 8, -1)
    assert call(groups, 1, 8, 8, nb, *tail, 8, None, None) == -1
    groups[0] = _native.TileStats(8, 8, 5)
    assert call(None, 1, 8, 8, nb, *tail, 8, None, None) == -1
    assert call(groups, 1, None, 8, nb, *tail, 8, None, None) == -1
    assert call(groups, 1, 8, 8, nb, *tail, None, None, None) == -1
    assert call(groups, 1, 8, 8, nb - 1, *tail, 8, None, None) == -3
    assert call(groups, 1, 8, 8, nb, *tail[:6], 0, *tail[7:], 8, None, None) == -1   # window 0
    scan = lib.ms_grad_tile_stats
    assert scan(8, 1, 1, 0, 10, 0, 10, 0, 1.0, None, None, 8, 1, None) == -1
    assert scan(8, 1, 1, 0, 2049, 0, 10, 0, 1.0, None, 8, 8, 1, None) == -3
    assert scan(None, 0, 1, 0, 10, 0, 10, 0, 1.0, None, 8, 8, 1, None) == -2
    assert scan(None, 0, 1, 4, 4, 4, 4, 0, 1.0, None, 8, 8, 0, None) == 0
    stats, scale = lib.ms_buffer_tile_stats, lib.ms_buffer_scale
    assert stats(8, 7, 10, 8, 8, 1, None) == -1 and stats(8, 0, -1, 8, 8, 1, None) == -1
    assert stats(None, 0, 10, 8, 8, 1, None) == -1 and stats(8, 0, 10, 8, None, 1, None) == -1
    assert stats(8, 0, 2049, 8, 8, 1, None) == -3 and stats(None, 0, 0, 8, 8, 0, None) == 0
    assert scale(None, 10, 1, 2.0, None) == -1 and scale(8, -1, 1, 2.0, None) == -1
    assert scale(8, 10, 3, 2.0, None) == -1 and scale(8, 10, 1, 0.0, None) == -1
    assert scale(None, 0, 2, 0.0, None) == 0 and scale(8, 10, 0, 2.0, None) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("counts", [[1], [63], [1024], [1025], [16383], [16384], [16385], [40000],
                                    [0], [5, 0, 20000, 16384], [7] * 35 + [16385]])
@pytest.mark.parametrize("bad", [None, "flag", "inf"])
def test_norm_from_tiles_equals_fold_and_norm(counts, bad):
    lib = _native.load()
    nb, n = _native.stats_blocks(), len(counts)
    gen = torch.Generator(device=DEV).manual_seed(sum(counts))
    tiles = [(torch.rand(max(c, 1), generator=gen, device=DEV, dtype=torch.float64) * 3,
              torch.zeros(max(c, 1), dtype=torch.int32, device=DEV)) for c in counts]
    if bad and counts[-1]:
        (tiles[-1][1] if bad == "flag" else tiles[-1][0])[counts[-1] - 1] = (
            1 if bad == "flag" else float("inf"))
    args = (1, 2.5, 1, 1024.0, 3, 1, 7, 1.0, 2.0 ** 20)

    def buffers():
        return (torch.full((n * nb,), 7.0, dtype=torch.float64, device=DEV),
                torch.full((n * nb,), 3, dtype=torch.int32, device=DEV),
                torch.zeros(_native.SCALARS_BYTES, dtype=torch.uint8, device=DEV))
    ps, pf, want = buffers()
    for g, (c, (ts, tf)) in enumerate(zip(counts, tiles)):
        _native.check(lib.ms_reduce_tile_stats(ts.data_ptr(), tf.data_ptr(), c,
                                               ps.data_ptr() + 8 * g * nb, pf.data_ptr() + 4 * g * nb,
                                               nb, None), "fold")
    _native.check(lib.ms_norm_clip(ps.data_ptr(), pf.data_ptr(), nb, n, *args, want.data_ptr(), None,
                                   None), "norm")
    ps, pf, got = buffers()
    groups = (_native.TileStats * n)(*[_native.TileStats(ts.data_ptr(), tf.data_ptr(), c)
                                       for c, (ts, tf) in zip(counts, tiles)])
    _native.check(lib.ms_norm_clip_tiles(groups, n, ps.data_ptr(), pf.data_ptr(), nb, *args,
                                         got.data_ptr(), None, None), "norm from tiles")
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    s = _native.StepScalars.from_buffer_copy(got.cpu().numpy().tobytes())
    assert s.overflow == (1 if bad == "flag" and counts[-1] else 0)
    if bad is None:
        exact = float(np.sum([float(ts[:c].sum()) for c, (ts, _) in zip(counts, tiles)]))
        # one fp32 rounding per group and one per add of the group sums
        assert abs(s.sumsq - exact) <= exact * 2.0 ** -24 * 2 * n


@pytest.mark.gpu
@pytest.mark.parametrize("counts", [[1025], [5000, 16384], [40000]])
@pytest.mark.parametrize("extra", [1024, 16384, 37])
def test_more_slots_a_group_than_the_fold_needs(counts, extra):
    """nblk above ms_stats_blocks() spreads the tiles over other slots, so
    the fold adds them in another order: the result follows it."""
    lib = _native.load()
    nb, n = _native.stats_blocks() + extra, len(counts)
    gen = torch.Generator(device=DEV).manual_seed(extra + sum(counts))
    # sums of very different sizes: their total depends on the order
    tiles = [(torch.exp(40 * torch.rand(c, generator=gen, device=DEV, dtype=torch.float64)),
              torch.zeros(c, dtype=torch.int32, device=DEV)) for c in counts]
    args = (1, 2.5, 1, 1024.0, 3, 1, 7, 1.0, 2.0 ** 20)
    ps = torch.empty(n * nb, dtype=torch.float64, device=DEV)
    pf = torch.empty(n * nb, dtype=torch.int32, device=DEV)
    want, got = (torch.zeros(_native.SCALARS_BYTES, dtype=torch.uint8, device=DEV) for _ in range(2))
    for g, (ts, tf) in enumerate(tiles):
        _native.check(lib.ms_reduce_tile_stats(ts.data_ptr(), tf.data_ptr(), counts[g],
                                               ps.data_ptr() + 8 * g * nb, pf.data_ptr() + 4 * g * nb,
                                               nb, None), "fold")
    _native.check(lib.ms_norm_clip(ps.data_ptr(), pf.data_ptr(), nb, n, *args, want.data_ptr(), None,
                                   None), "norm")
    folded = ps.clone(), pf.clone()
    ps.fill_(7.0)
    pf.fill_(3)
    groups = (_native.TileStats * n)(*[_native.TileStats(ts.data_ptr(), tf.data_ptr(), c)
                                       for c, (ts, tf) in zip(counts, tiles)])
    _native.check(lib.ms_norm_clip_tiles(groups, n, ps.data_ptr(), pf.data_ptr(), nb, *args,
                                         got.data_ptr(), None, None), "norm from tiles")
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    # every group was folded into its slots (the fp32 rounding of the sums
    # hides most changes of order from the scalars)
    assert torch.equal(ps, folded[0]) and torch.equal(pf, folded[1])


@pytest.mark.gpu
@pytest.mark.parametrize("n", [6144 * 2048 - 5, 6144 * 2048, 6144 * 2048 + 1])
def test_reading_scan_equals_the_writing_scan_at_the_short_scan_line(n):
    lib = _native.load()
    g = torch.randn(n, device=DEV, generator=torch.Generator(device=DEV).manual_seed(1)).to(torch.float16)
    table = torch.tensor([[0, 1000, g.data_ptr(), 0], [1000, n - 1000, g.data_ptr() + 2000, 0]],
                         dtype=torch.int64, device=DEV)
    nt = _native.scan_tiles(n)
    flat = torch.empty(n, device=DEV)
    out = []
    for target in (None, flat.data_ptr()):
        ts = torch.full((nt,), -1.0, dtype=torch.float64, device=DEV)
        tf = torch.full((nt,), 9, dtype=torch.int32, device=DEV)
        _native.check(lib.ms_grad_tile_stats(table.data_ptr(), 2, _native.DTYPE_F16, 0, n, 0, n,
                                             _native.SCALE_DIVIDE, 1024.0, target, ts.data_ptr(),
                                             tf.data_ptr(), nt, None), "K1")
        out.append((ts, tf))
    torch.cuda.synchronize()
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
    assert torch.equal(flat, g.float() / 1024.0)
    assert int(out[0][1].max()) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 7, 2047, 2048, 2049, 3 * 2048 + 5, 6200 * 2048 + 1])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("off", [0, 1])
def test_buffer_scan_equals_the_one_row_table(n, dtype, off):
    lib = _native.load()
    gen = torch.Generator(device=DEV).manual_seed(n + off)
    x = torch.randn(n + off, generator=gen, device=DEV).to(dtype)[off:]
    if n > 1:
        x[n // 2] = float("nan" if n % 2 else "inf")
    nt = _native.scan_tiles(n)
    table = torch.tensor([[0, n, x.data_ptr(), 0]], dtype=torch.int64, device=DEV)
    out = []
    for one in (True, False):
        ts = torch.full((nt,), -1.0, dtype=torch.float64, device=DEV)
        tf = torch.full((nt,), 9, dtype=torch.int32, device=DEV)
        args = (ts.data_ptr(), tf.data_ptr(), nt, None)
        d = _native.ms_dtype(dtype)
        rc = (lib.ms_buffer_tile_stats(x.data_ptr(), d, n, *args) if one else
              lib.ms_grad_tile_stats(table.data_ptr(), 1, d, 0, n, 0, n, 0, 1.0, None, *args))
        _native.check(rc, "K1")
        out.append((ts, tf))
    torch.cuda.synchronize()
    assert torch.equal(out[0][0].view(torch.int64), out[1][0].view(torch.int64))
    assert torch.equal(out[0][1], out[1][1])
    assert int(out[0][1].sum()) == (1 if n > 1 else 0)
    if dtype is not torch.float32:
        return
    for mode, factor in ((_native.SCALE_DIVIDE, 1024.0), (_native.SCALE_DIVIDE, 3.0),
                         (_native.SCALE_MULTIPLY, 1.0 / 3.0)):
        want = x.cpu()
        want.div_(factor) if mode == _native.SCALE_DIVIDE else want.mul_(factor)
        y = torch.cat([torch.full((8 + off,), 5.0, device=DEV), x, torch.full((8,), 5.0, device=DEV)])
        inner = y[8 + off:8 + off + n]
        _native.check(lib.ms_buffer_scale(inner.data_ptr(), n, mode, float(np.float32(factor)), None),
                      "scale")
        torch.cuda.synchronize()
        assert torch.equal(torch.nan_to_num(inner.cpu()), torch.nan_to_num(want))
        assert bool((y[:8 + off] == 5.0).all()) and bool((y[8 + off + n:] == 5.0).all())
