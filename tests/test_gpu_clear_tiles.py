"""Statistics slots of parameters that a window leaves out: the clearing
kernel, and how many launches a window with many of them takes."""

import numpy as np
import pytest
import torch

import minispeed_amd
from minispeed_amd import _native

CLEAR_RANGES = 224      # MS_CLEAR_RANGES_PER_LAUNCH


def test_argument_errors():
    call = _native.load().ms_clear_tiles
    assert call(None, 0, None, None, 0, None) == 0
    assert call(None, 1, 8, 8, 4, None) == -1
    for bad in ([-1, 2], [2, 2], [3, 2], [0, 5]):
        assert call(np.array(bad, dtype=np.int64).ctypes.data, 1, 8, 8, 4, None) == -1


@pytest.mark.gpu
@pytest.mark.parametrize("count", [1, CLEAR_RANGES, CLEAR_RANGES + 1, 3 * CLEAR_RANGES])
def test_ranges(count):
    rng = np.random.default_rng(count)
    cuts = np.cumsum(rng.integers(1, 700, size=2 * count + 1))
    ranges, n = np.ascontiguousarray(cuts[1:].reshape(count, 2)), int(cuts[-1]) + 3
    ranges[0, 0], ranges[-1, 1] = 0, n - (count > 1)
    sums = torch.ones(n, dtype=torch.float64, device="cuda")
    flags = torch.ones(n, dtype=torch.int32, device="cuda")
    want = torch.ones(n)
    for begin, end in ranges:
        want[begin:end] = 0
    _native.check(_native.load().ms_clear_tiles(
        ranges.ctypes.data, count, sums.data_ptr(), flags.data_ptr(), n,
        _native.stream_handle(sums.device)), "ms_clear_tiles")
    assert torch.equal(sums.cpu().float(), want) and torch.equal(flags.cpu().float(), want)


@pytest.mark.gpu
def test_alternating_parameters_take_one_launch(monkeypatch):
    """Windows over every second parameter: the slots and the norm are those
    of the present gradients, with one clearing launch where any is stale."""
    sizes = [3000 + 7 * k for k in range(40)]
    params = [torch.nn.Parameter(torch.randn(n, device="cuda")) for n in sizes]
    engine = minispeed_amd.initialize(model=torch.nn.ParameterList(params), config={
        "train_micro_batch_size_per_gpu": 1, "dtype": "fp32",
        "optimizer": {"type": "AdamW", "params": {"lr": 1e-3}},
        "hip_boundary": {"contiguous_gradients": True}})
    lib, calls = _native.load(), []

    class Spy:
        def __getattr__(self, name):
            calls.append(name)
            return getattr(lib, name)

    monkeypatch.setattr(_native, "load", lambda: Spy())
    from torch.utils._python_dispatch import TorchDispatchMode

    class Fills(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            calls.append(str(func))
            return func(*args, **(kwargs or {}))

    for window in range(4):
        present = [k for k in range(40) if window == 0 or k % 2 == window % 2]
        total = 0.0
        for k in present:
            grad = torch.randn(sizes[k], device="cuda")
            total += grad.double().square().sum().item()
            params[k].grad = grad
            engine.contiguous.accumulate(0, k, params[k])
        calls.clear()
        with Fills():
            engine.micro_steps += 1
            assert engine.step()
        assert calls.count("ms_clear_tiles") == (window > 0)
        assert not [c for c in calls if "zero" in c or "fill" in c]
        assert abs(engine.get_gradient_norm() / total ** 0.5 - 1) < 1e-6
        at = 0
        slots = engine.contiguous.tile_sumsq[0].cpu()
        for k, n in enumerate(sizes):
            tiles = -(-n // _native.ACCUM_TILE)
            assert bool((slots[at:at + tiles] != 0).all()) == (k in present)
            assert bool((slots[at:at + tiles] == 0).all()) == (k not in present)
            at += tiles
