"""K5's launches: packed rows, rows with full addresses, and the limits
between them, against the fp32 sums and fp64 statistics of the same rows; the
statistics of parameters that some windows leave out."""

import numpy as np
import pytest
import torch
from torch import nn

import minispeed_amd as ms
from minispeed_amd import _native
from minispeed_amd.contiguous import ACCUM_ROW, accumulate_rows

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
N = _native.ACCUM_ROWS_PER_LAUNCH


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("nrows", [1, N - 1, N, N + 1, 2 * N + 3])
@pytest.mark.parametrize("where", ["together", "buffers", "apart"])
def test_rows_of_a_call(dtype, nrows, where):
    """where: every row in one buffer, turn by turn in six (more than the
    bases of a launch), or with flag slots that are not in step with the
    sums' (full addresses)."""
    rng = np.random.default_rng(nrows)
    gen = torch.Generator(device=DEV).manual_seed(nrows)
    sizes = rng.choice([0, 1, 5, 2047, 2048, 2049, 4097], size=nrows)
    tiles = (sizes + 2047) // 2048
    nbuf = 6 if where == "buffers" else 1
    starts = np.concatenate([[0], np.cumsum(sizes + 3)])
    t0 = np.concatenate([[0], np.cumsum(tiles)])
    f0 = t0[:-1] if where != "apart" else t0[-1] - t0[1:]      # from the back
    bufs = [torch.full((int(starts[-1]) + 8,), -3.0, device=DEV) for _ in range(nbuf)]
    ts = [torch.full((int(t0[-1]) + 1,), -1.0, dtype=torch.float64, device=DEV) for _ in range(nbuf)]
    tf = [torch.full((int(t0[-1]) + 1,), -1, dtype=torch.int32, device=DEV) for _ in range(nbuf)]
    want = [b.clone() for b in bufs]
    for first in (True, False):
        rows, srcs = np.zeros(nrows, dtype=ACCUM_ROW), []
        for r, n in enumerate(sizes):
            x = torch.randn(int(n), generator=gen, device=DEV).to(dtype)
            if n > 2 and r % 9 == 4 and not first:
                x[1] = float("inf")
            srcs.append(x)
            b = r % nbuf
            rows[r] = (bufs[b].data_ptr() + 4 * int(starts[r]), x.data_ptr(), n, first, 0,
                       ts[b].data_ptr() + 8 * int(t0[r]), tf[b].data_ptr() + 4 * int(f0[r]))
            w = want[b][int(starts[r]):int(starts[r]) + int(n)]
            w.copy_(x.float() if first else w + x.float())
        accumulate_rows(rows, _native.ms_dtype(dtype), DEV, _native.SCALE_DIVIDE, 4.0)
    torch.cuda.synchronize()
    for b in range(nbuf):
        assert torch.equal(bufs[b].view(torch.int32), want[b].view(torch.int32))
    sums, flags = [t.cpu().numpy() for t in ts], [t.cpu().numpy() for t in tf]
    for r, n in enumerate(sizes):
        b = r % nbuf
        w = want[b][int(starts[r]):int(starts[r]) + int(n)].cpu().double().numpy() / 4.0
        for k in range(tiles[r]):
            part = w[2048 * k:2048 * (k + 1)]
            bad = not np.isfinite(part).all()
            assert (flags[b][f0[r] + k] != 0) == bad, (r, k)
            if not bad:
                ref = float(np.sum(part * part))
                # at most 2048 fp64 additions in another order
                assert abs(sums[b][t0[r] + k] - ref) <= 2048 * 2.0 ** -52 * ref, (r, k)


def test_parameters_that_some_windows_leave_out():
    shapes = [(300, 70), (5,), (2048,), (4100,), (33, 9)]

    def engine(stats):
        gen = torch.Generator().manual_seed(3)
        params = [nn.Parameter(torch.randn(*s, generator=gen).cuda()) for s in shapes]
        e = ms.initialize(model=nn.ParameterList(params), config={
            "train_micro_batch_size_per_gpu": 1, "gradient_clipping": 1.0, "dtype": "bf16",
            "optimizer": {"type": "AdamW", "params": {"lr": 1e-2}},
            "zero_optimization": {"stage": 1}, "hip_boundary": {"contiguous_gradients": True}})
        e.contiguous.use_tile_stats = stats
        return e
    a, b = engine(True), engine(False)
    for window, given in enumerate([(0, 1, 2, 3, 4), (0, 2), (), (3,), (1, 3, 4), (0, 1, 2, 3, 4)]):
        for e in (a, b):
            for k in given:
                p = e.flat_groups[0].params[k]
                gen = torch.Generator(device="cuda").manual_seed(10 * window + k)
                p.grad = torch.randn(p.shape, generator=gen, device="cuda").to(p.dtype)
                e.contiguous.accumulate(0, k, p)
            e.contiguous.flush()
            if window == 1:          # an abandoned window in between
                p = e.flat_groups[0].params[4]
                p.grad = torch.ones_like(p)
                e.contiguous.accumulate(0, 4, p)
                e.contiguous.flush()
                e.zero_grad()
                continue
            e.micro_steps += 1
            assert e.step()
        if window != 1:
            # the fp64 partial sums in two partitions: one fp32 rounding
            assert abs(a.grad_norm - b.grad_norm) <= 1.2e-7 * b.grad_norm, window
