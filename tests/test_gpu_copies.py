"""copy.deepcopy of an engine that has taken steps: the copy steps on as the
original does, and neither touches the other's buffers."""

import copy

import pytest
import torch
from torch import nn

import minispeed_amd as ms

pytestmark = pytest.mark.gpu


def _engine(stage, contiguous):
    torch.manual_seed(7)
    model = nn.Sequential(nn.Linear(16, 40), nn.Tanh(), nn.Linear(40, 3))
    engine, *_ = ms.initialize(model=model, config={
        "train_micro_batch_size_per_gpu": 4, "gradient_accumulation_steps": 2,
        "optimizer": {"type": "AdamW", "params": {"lr": 1e-2}},
        "fp16": {"enabled": True, "initial_scale_power": 8, "loss_scale_window": 3},
        "zero_optimization": {"stage": stage}, "gradient_clipping": 0.5,
        "hip_boundary": {"contiguous_gradients": contiguous}})
    return engine


def _micro(engine, seed):
    x = torch.randn(4, 16, generator=torch.Generator().manual_seed(seed)).cuda()
    engine.backward(engine(x).float().pow(2).mean())
    engine.step()


def _masters(engine):
    return [g.data.clone() for g in engine.flat_groups]


@pytest.mark.parametrize("stage", [0, 2, 3])
@pytest.mark.parametrize("contiguous", [False, True])
def test_copy_steps_as_the_original(stage, contiguous):
    engine = _engine(stage, contiguous)
    for i in range(5):                     # two windows and a half
        _micro(engine, i)
    twin = copy.deepcopy(engine)
    if not contiguous:                     # (torch copies no param.grad)
        for p, q in zip(engine.module.parameters(), twin.module.parameters()):
            q.grad = None if p.grad is None else p.grad.clone()
    before = _masters(engine)
    for i in range(5, 10):
        _micro(twin, i)
    assert all(torch.equal(a, b) for a, b in zip(_masters(engine), before))
    for i in range(5, 10):
        _micro(engine, i)
    assert all(torch.equal(a, b) for a, b in zip(_masters(engine), _masters(twin)))
    assert not any(torch.equal(a, b) for a, b in zip(_masters(engine), before))
    assert engine.grad_norm == twin.grad_norm and engine.loss_scale == twin.loss_scale
    assert engine.global_steps == twin.global_steps == 5
