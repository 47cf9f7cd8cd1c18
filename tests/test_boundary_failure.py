"""A boundary that fails before its launch, on the CPU: the gradients, the
parameters and ZeRO-3's gathered state are as they were, so the caller can
free memory and step again."""

import types

import numpy as np
import pytest
import torch

from minispeed_amd import boundary
from minispeed_amd.flat import FlatLayout, FlatParamGroup
from minispeed_amd.precision import DynamicLossScaler
from minispeed_amd.zero.stage_1_and_2 import ZeROOptimizer
from minispeed_amd.zero.stage_3 import ZeROStage3Optimizer

SHAPES = [(3,), (43, 3), (64,)]


class _Table:
    def __init__(self, fail):
        self.fail = fail

    def find(self, table, stream):
        return (64, len(table)) if self.fail == "table behind K1" else None

    def upload(self, table, stream=None):
        if self.fail in ("table", "table behind K1"):
            raise torch.OutOfMemoryError("table")
        return 64, len(table)


class _Group(FlatParamGroup):
    """A group over host tensors, with what needs a GPU stood in for."""

    def __init__(self, stage, fail):
        self.params = [torch.nn.Parameter(torch.randn(s)) for s in SHAPES]
        self.layout = lay = FlatLayout([p.numel() for p in self.params], rank=0, world_size=1,
                                       zero_stage=stage)
        self.numel, self.numel_padded = lay.numel, lay.numel_padded
        self.shard_start, self.shard_end = lay.shard_start, lay.shard_end
        self._numels, self._shapes = list(lay.numels), SHAPES
        self._numels_np = np.asarray(self._numels, dtype=np.int64)
        self._offsets = list(zip(lay.offsets, self.params))
        self.device, self._device_index = torch.device("cuda:0"), 0
        self.data, self.zero_stage = torch.zeros(self.numel_padded), stage
        self._partitioned = self._materialized = stage == 3
        self._rows = self._native_rows = self._shard_views = None
        self.model_shard = torch.zeros(self.numel_padded) if stage == 3 else None
        self.fail = fail

    def table(self, key):
        return _Table(self.fail)

    def grad_pointers(self):
        grads = [p.grad for p in self.params]
        return np.array([g.data_ptr() for g in grads] + [0], dtype=np.int64), grads, None

    def flat_grad_for_overwrite(self):
        if self.fail == "flat_grad":
            raise torch.OutOfMemoryError("flat gradient")
        return torch.zeros(self.numel_padded)


class _Stream:
    device_type, device_index, stream_id, cuda_stream = 1, 0, 0, 0


class _Workspace:
    def __init__(self, fail):
        from minispeed_amd import _native
        self.fail, self.norm = fail, _native.NormArgs()
        self.tile_stats, self.groups = (_native.TileStats * 1)(), (_native.BoundaryGroup * 1)()
        self.readback = types.SimpleNamespace(arm=lambda: None)
        self.waits = 0

    def enter(self):
        return _Stream()

    def finish_readback(self):
        self.waits += 1

    def tile_ptrs(self, ntiles, cur):
        if self.fail == "tiles":
            raise torch.OutOfMemoryError("tile slots")
        return 64, 64


@pytest.mark.parametrize("stage,fail", [
    (1, "tiles"), (1, "model"), (3, "tiles"), (3, "flat_grad"), (3, "table"),
    (3, "table behind K1"), (3, "moments"), (3, "scan"), (3, "update")])
def test_nothing_is_released(stage, fail, monkeypatch):
    opt = object.__new__(ZeROStage3Optimizer if stage == 3 else ZeROOptimizer)
    group = _Group(stage, fail)
    opt.flat_groups, opt.contiguous, opt.launch_timer = [group], None, None
    opt._workspace = _Workspace(fail)
    opt._gathered, opt._boundary_freed = True, False
    n = group.numel_padded - (fail == "moments")
    opt.adam = types.SimpleNamespace(
        param_groups=[{"lr": 0.1, "betas": (0.9, 0.99), "eps": 1e-8, "weight_decay": 0.0}],
        state=[{"step": 4, "exp_avg": torch.zeros(n), "exp_avg_sq": torch.zeros(n)}])
    monkeypatch.setattr(boundary, "record_streams", lambda tensors, stream: None)
    scans = []

    def scan(*args):
        scans.append(args)
        return -2 if fail == "scan" else 0

    lib = types.SimpleNamespace(ms_boundary_scan=scan, ms_error_string=lambda rc: b"no table",
                                ms_boundary_update=lambda *args: -2)
    monkeypatch.setattr(boundary._native, "load", lambda: lib)
    grads = [torch.randn_like(p) for p in group.params]
    for p, g in zip(group.params, grads):
        p.grad = g
    where = [p.data_ptr() for p in group.params]
    # host storage is what the model walk refuses at stage 1
    with pytest.raises((torch.OutOfMemoryError, RuntimeError)):
        opt.boundary_step(DynamicLossScaler(enabled=False), None, materialize_flat_grad=True)
    assert all(p.grad is g for p, g in zip(group.params, grads))
    assert [tuple(p.shape) for p in group.params] == SHAPES
    assert [p.data_ptr() for p in group.params] == where
    assert opt._gathered and not opt._boundary_freed
    assert opt.adam.state[0]["step"] == 4
    # a K2 that was launched is waited for: its result is not the next boundary's
    behind = fail in ("table behind K1", "moments", "update")
    assert len(scans) == (behind or fail == "scan") and opt._workspace.waits == behind


def test_gathered_parameters_are_written_where_their_placeholders_lie():
    group = _Group(3, None)
    group.dematerialize_params()
    assert group.shard_pointers().tolist() == [p.data_ptr() for p in group.params] + [0]
