"""The tile statistics of parameters that some windows of contiguous gradients
leave out."""

import pytest
import torch
from torch import nn

import minispeed_amd as ms

pytestmark = pytest.mark.gpu


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
