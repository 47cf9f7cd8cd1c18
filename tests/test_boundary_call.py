"""ms_boundary_step, its two halves and the table they are launched with: struct layouts,
argument errors and the table's columns on the CPU; on the GPU the one call
against the entry points it stands for, bit for bit."""

import ctypes
import gc
import os
import shutil
import subprocess
import weakref

import numpy as np
import pytest
import torch

import minispeed_amd
from minispeed_amd import _native, boundary
from minispeed_amd.boundary import LaunchTimer, adamw_params
from minispeed_amd.flat import FlatParamGroup, _walk
from minispeed_amd.precision import DynamicLossScaler

INCLUDE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include")
STRUCTS = {"ms_boundary_group_t": _native.BoundaryGroup, "ms_norm_args_t": _native.NormArgs,
           "ms_tile_stats_t": _native.TileStats}


@pytest.mark.skipif(shutil.which("gcc") is None, reason="gcc not available")
def test_struct_layouts(tmp_path):
    lines = []
    for cname, cls in STRUCTS.items():
        lines.append(f'printf("{cname} %zu\\n", sizeof({cname}));')
        lines += [f'printf("{cname}.{f} %zu\\n", offsetof({cname}, {f}));' for f, *_ in cls._fields_]
    src = tmp_path / "probe.c"
    src.write_text('#include <stddef.h>\n#include <stdio.h>\n#include "minispeed_boundary.h"\n'
                   "int main(void) {\n" + "\n".join(lines) + "\nreturn 0; }\n")
    exe = tmp_path / "probe"
    subprocess.run(["gcc", "-I", INCLUDE, str(src), "-o", str(exe)], check=True)
    for line in subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split("\n"):
        if line:
            key, value = line.split(" ")
            cname, _, field = key.partition(".")
            cls = STRUCTS[cname]
            assert (getattr(cls, field).offset if field else ctypes.sizeof(cls)) == int(value), key


def test_argument_errors_launch_nothing():
    lib = _native.load()
    groups, stats, norm = _native.BoundaryGroup(), _native.TileStats(), _native.NormArgs()
    call = lib.ms_boundary_step
    assert call(groups, stats, -1, norm, None, None) == -1
    assert call(None, stats, 1, norm, None, None) == -1
    assert call(groups, None, 1, norm, None, None) == -1
    assert call(groups, stats, 1, None, None, None) == -1
    assert call(groups, stats, 0, norm, None, None) == -1          # K2's own checks
    groups.grad_dtype = 9
    assert call(groups, stats, 1, norm, None, None) == -1          # K1's own checks
    groups.grad_dtype, groups.numel = 1, 5
    assert call(groups, stats, 1, norm, None, None) == -2          # no table
    update, scalars = lib.ms_boundary_update, ctypes.create_string_buffer(_native.SCALARS_BYTES)
    assert update(groups, -1, scalars, None, None) == -1
    assert update(None, 1, scalars, None, None) == -1
    assert update(groups, 1, None, None, None) == -1
    groups.update_from_flat = 1                                    # no flat gradient
    assert update(groups, 1, scalars, None, None) == -1


def test_rows_in_a_cycle_are_collected():
    """Parameters that refer to the engine's objects (an owner attribute, a
    gradient hook) close a cycle through the rows; it goes when dropped."""
    class Owner:
        pass

    for link in ("attribute", "hook"):
        owner = Owner()
        owner.params = [torch.nn.Parameter(torch.zeros(3)) for _ in range(2)]
        for p in owner.params:
            if link == "attribute":
                p.owner = owner
            else:
                p.register_hook(lambda grad, owner=owner: None)
        base = np.array([[0, 3, 0, 0], [3, 3, 0, 0]], dtype=np.int64)
        owner.rows = _walk().BoundaryRows(owner.params, [3, 3], 0, base, [0, 1])
        gone = weakref.ref(owner)
        del owner, p
        gc.collect()
        assert gone() is None, link


def test_rows_on_the_host():
    params = [torch.nn.Parameter(torch.zeros(n)) for n in (3, 0, 5)]
    base = np.array([[0, 3, 7, 7], [3, 5, 7, 7], [8, 2, 7, 7]], dtype=np.int64)
    rows = _walk().BoundaryRows(params, [3, 0, 5], 0, base, [0, 2, 3])
    rows.set_grads(np.array([11, 12, 13, 0], dtype=np.int64))
    assert rows.table[:, 2].tolist() == [11, 13, 0]
    assert rows.models(True) == 0                        # host storage: the caller's to refuse
    assert rows.models(False) == -1 and rows.table[:, 3].tolist() == [0, 0, 0]
    params[2].grad = torch.zeros(5)
    assert rows.grads(1, 0, 0) == 2 and rows.table[:, 2].tolist() == [11, 13, 0]
    with pytest.raises(ValueError):
        rows.set_grads(np.zeros(3, dtype=np.int64))
    with pytest.raises(ValueError):
        _walk().BoundaryRows(params, [3, 0, 5], 0, base, [0, 2, 4])
    _walk().release_grads(params)
    assert params[2].grad is None
    same = _walk().same_table
    assert same(base, base.copy()) and not same(base, base[:2])
    params.pop()
    with pytest.raises(ValueError):
        rows.models(True)


def _host_group(sizes):
    """A group over host tensors, as far as its pointer walk goes."""
    g = FlatParamGroup.__new__(FlatParamGroup)
    g.params = [torch.nn.Parameter(torch.zeros(n)) for n in sizes]
    g.device, g._device_index, g._partitioned = torch.device("cuda:0"), 0, False
    g._numels, g._numels_np = list(sizes), np.asarray(sizes, dtype=np.int64)
    return g


def test_storage_of_another_size_is_named():
    g = _host_group((3, 129))
    for n in (7, 130):
        g.params[0].data = torch.zeros(n)
        with pytest.raises(RuntimeError, match=f"parameter 0 of its group has {n} elements, expected 3"):
            g.model_pointers()
    with pytest.raises(ValueError):
        _walk().model_pointers(g.params, 0, np.zeros(3, dtype=np.int64), np.zeros(3, dtype=np.int64))


class _Group:
    """One group's arrays on the GPU: n flat indices in two segments."""

    def __init__(self, n, own, dtype, seed, inf=False):
        gen = torch.Generator(device="cuda").manual_seed(seed)
        self.n, self.own = n, own
        self.grad = torch.randn(n, generator=gen, device="cuda").to(dtype)
        if inf:
            self.grad[n // 2] = float("inf")
        self.model = torch.zeros(n, dtype=dtype, device="cuda")
        k, size = own[1] - own[0], self.grad.element_size()
        self.state = [torch.randn(k, generator=gen, device="cuda").abs_() for _ in range(3)]
        cut = n // 3
        rows = [[0, cut, self.grad.data_ptr(), self.model.data_ptr()],
                [cut, n - cut, self.grad.data_ptr() + cut * size, self.model.data_ptr() + cut * size]]
        self.k1 = torch.tensor(rows, dtype=torch.int64, device="cuda")
        lo, hi = own
        self.k3 = torch.tensor([[max(b, lo), min(b + m, hi) - max(b, lo), g + (max(b, lo) - b) * size,
                                 p + (max(b, lo) - b) * size] for b, m, g, p in rows
                                if min(b + m, hi) > max(b, lo)], dtype=torch.int64, device="cuda")
        nt = _native.scan_tiles(n)
        self.sums = torch.zeros(nt, dtype=torch.float64, device="cuda")
        self.flags = torch.zeros(nt, dtype=torch.int32, device="cuda")

    def out(self):
        return [self.model, self.sums, self.flags, *self.state]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("inf", [False, True])
@pytest.mark.parametrize("sizes", [[(1, (0, 1))], [(2049, (0, 2049)), (5000, (512, 4096)), (700, (0, 0))]])
def test_one_call_is_the_three_entry_points(dtype, inf, sizes):
    lib, code = _native.load(), _native.ms_dtype(dtype)
    hp = adamw_params(1e-2, (0.9, 0.99), 1e-8, 0.1, 3, grad_scale=8.0, unscale=True)
    stream = torch.cuda.current_stream().cuda_stream
    results = []
    for one in (False, True):
        groups = [_Group(n, own, dtype, 5 + i, inf and i == 0) for i, (n, own) in enumerate(sizes)]
        nblk, n = _native.stats_blocks(), len(groups)
        partials = torch.zeros(n * nblk, dtype=torch.float64, device="cuda")
        flags = torch.zeros(n * nblk, dtype=torch.int32, device="cuda")
        scalars = torch.zeros(_native.SCALARS_BYTES, dtype=torch.uint8, device="cuda")
        stats = (_native.TileStats * n)(*[(g.sums.data_ptr(), g.flags.data_ptr(), g.sums.numel())
                                          for g in groups])
        if one:
            norm = _native.NormArgs(
                block_sumsq=partials.data_ptr(), block_flag=flags.data_ptr(), nblk=nblk, has_clip=1,
                scaler_enabled=1, max_norm=1.0, scale=8.0, good_steps=1, skipped_steps=2, window=9,
                min_scale=1.0, max_scale=64.0, out=scalars.data_ptr())
            args = (_native.BoundaryGroup * n)()
            for b, g in zip(args, groups):
                b.segs, b.nseg = g.k1.data_ptr(), len(g.k1)
                b.own_segs, b.own_nseg = g.k3.data_ptr(), len(g.k3)
                b.grad_dtype = b.model_dtype = code
                b.numel, (b.own_begin, b.own_end) = g.n, g.own
                b.master, b.exp_avg, b.exp_avg_sq = (t.data_ptr() for t in g.state)
                b.hp = hp
            timer = LaunchTimer()
            k3 = sum(g.own[1] > g.own[0] for g in groups)
            events = timer.pairs(["k1"] * n + ["k2"] + ["k3"] * k3)
            _native.check(lib.ms_boundary_step(args, stats, n, norm, events, stream), "step")
            torch.cuda.synchronize()
            for name, count in (("k1", n), ("k2", 1), ("k3", k3)):
                ms = timer.durations_ms(name)
                assert len(ms) == count and all(t >= 0.0 for t in ms)
        else:
            for g, st in zip(groups, stats):
                _native.check(lib.ms_grad_tile_stats(
                    g.k1.data_ptr(), len(g.k1), code, 0, g.n, *g.own, _native.SCALE_DIVIDE, 8.0, None,
                    st.sumsq, st.flag, st.ntiles, stream), "K1")
            _native.check(lib.ms_norm_clip_tiles(
                stats, n, partials.data_ptr(), flags.data_ptr(), nblk, 1, 1.0, 1, 8.0, 1, 2, 9, 1.0, 64.0,
                scalars.data_ptr(), None, stream), "K2")
            for g in groups:
                if g.own[1] > g.own[0]:
                    _native.check(lib.ms_fused_adamw(
                        *(t.data_ptr() for t in g.state), None, g.k3.data_ptr(), len(g.k3), code, code,
                        *g.own, hp, scalars.data_ptr(), stream), "K3")
            torch.cuda.synchronize()
        results.append([scalars, *[t for g in groups for t in g.out()]])
    for a, b in zip(*results):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
    assert (results[0][0][:4].view(torch.int32).item() != 0) == inf


@pytest.mark.gpu
def test_rows_are_the_pointer_walks():
    """Addresses as grad_pointers / model_pointers give them; what those look
    at more closely is left to them."""
    params = [torch.nn.Parameter(torch.randn(n, device="cuda").half()) for n in (3, 129, 64)]
    g = FlatParamGroup(params, device=torch.device("cuda:0"), rank=0, world_size=1, zero_stage=1)
    cur = torch.cuda.current_stream()
    stream = int(cur.device_type), int(cur.device_index), int(cur.stream_id)
    both = torch.randn(193, device="cuda").half()     # two gradients of one storage
    params[1].grad, params[2].grad = both[:129], both[129:]
    rows = g.boundary_rows()
    assert rows.grads(*stream) == -1 and rows.models(True) == -1
    want = g.boundary_table(0, g.numel_padded, g.grad_pointers()[0], g.model_pointers())
    assert np.array_equal(rows.table, want)
    params[2].grad = torch.randn(128, device="cuda").half()[::2]
    assert rows.grads(*stream) == 2
    params[1].data = params[1].data[:7].clone()
    assert rows.models(True) == 1
    params[1].data = torch.zeros(129, device="cuda")
    assert rows.models(True) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("through_rows", [False, True])
@pytest.mark.parametrize("views", [False, True])
def test_recorded_memory_waits_for_the_stream(through_rows, views):
    """A gradient allocated on another stream and dropped while the recorded
    stream is busy: its memory is not handed out again before that is done."""
    params = [torch.nn.Parameter(torch.zeros(1 << 20, device="cuda")) for _ in range(2)]
    g = FlatParamGroup(params, device=torch.device("cuda:0"), rank=0, world_size=1, zero_stage=1)
    side, cur = torch.cuda.Stream(), torch.cuda.current_stream()
    ids = int(cur.device_type), int(cur.device_index), int(cur.stream_id)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        if views:
            both = torch.zeros(1 << 21, device="cuda")
            grads = [both[:1 << 20], both[1 << 20:]]
            del both
        else:
            grads = [torch.zeros(1 << 20, device="cuda") for _ in params]
    held = {t.untyped_storage().data_ptr(): t.untyped_storage().nbytes() for t in grads}
    torch.cuda.synchronize()
    torch.cuda._sleep(50_000_000)
    if through_rows:
        for p, t in zip(params, grads):
            p.grad = t
        rows = g.boundary_rows()
        assert rows.grads(*ids) == -1
        g.release_grads()
        rows.drop()
    else:
        _walk().record_streams(grads, *ids)
    grads = t = p = None
    with torch.cuda.stream(side):
        again = [torch.empty(n, dtype=torch.uint8, device="cuda") for n in held.values()]
    assert not cur.query()                      # the stream was still busy
    assert not {t.data_ptr() for t in again} & set(held)
    torch.cuda.synchronize()


@pytest.mark.gpu
@pytest.mark.parametrize("lead", [304, 3])
def test_gradients_that_view_the_flat_gradient(lead):
    """K1, writing the flat gradient, unscales such gradients in place; K3
    then takes them from there, once unscaled."""
    results = []
    for views in (False, True):
        gen = torch.Generator(device="cuda").manual_seed(1)
        params = [torch.nn.Parameter(torch.randn(n, generator=gen, device="cuda"))
                  for n in (lead, 5000, 77)]
        engine = minispeed_amd.initialize(model=torch.nn.ParameterList(params), config={
            "train_micro_batch_size_per_gpu": 1, "dtype": "fp32",
            "optimizer": {"type": "AdamW", "params": {"lr": 0.1, "eps": 1.0}}})
        g = engine.flat_groups[0]
        for p, off, n in zip(g.params, g.layout.offsets, g.layout.numels):
            grad = torch.randn(n, generator=gen, device="cuda")
            p.grad = g.grad[off:off + n].copy_(grad) if views else grad
        scalars = engine.optimizer.boundary_step(DynamicLossScaler(enabled=True, init_scale=8.0), 0.5,
                                                 materialize_flat_grad=True)
        results.append([g.data, g.grad, torch.tensor(scalars.norm),
                        *[engine.optimizer.state[0][k] for k in ("exp_avg", "exp_avg_sq")]])
    for a, b in zip(*results):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [7, 130])
def test_replaced_storage_of_another_size_is_refused(n):
    """Every kernel that reads or writes whole parameters refuses storage of
    another size before it is launched."""
    params = [torch.nn.Parameter(torch.randn(k, device="cuda").half()) for k in (3, 129, 64)]
    engine = minispeed_amd.initialize(model=torch.nn.ParameterList(params), config={
        "train_micro_batch_size_per_gpu": 1, "dtype": "fp16",
        "optimizer": {"type": "AdamW", "params": {"lr": 0.1}}})
    g = engine.flat_groups[0]
    before = g.data.clone()
    params[1].data = torch.zeros(n, dtype=torch.float16, device="cuda")
    for call in (lambda: engine.optimizer.boundary_step(engine.loss_scaler, None),
                 g.copy_model_to_flat, g.copy_flat_to_model):
        with pytest.raises(RuntimeError, match=f"parameter 1 of its group has {n} elements, expected 129"):
            call()
    torch.cuda.synchronize()
    assert torch.equal(g.data, before) and not params[1].any()


@pytest.mark.gpu
@pytest.mark.parametrize("stage,long_scan,grads_move", [(1, 1 << 26, False), (3, 1 << 26, False),
                                                        (1, 1, False), (1, 1, True), (1, 1 << 26, True)])
def test_model_storage_moves(stage, long_scan, grads_move, monkeypatch):
    """K1 then reads the last boundary's table, or one with its model column;
    K3 writes the new storage."""
    monkeypatch.setattr(boundary, "_LONG_SCAN", long_scan)
    shapes, results = [(3,), (43, 30), (64,)], []
    for move in (False, True):
        gen = torch.Generator(device="cuda").manual_seed(2)
        params = [torch.nn.Parameter(torch.randn(s, generator=gen, device="cuda")) for s in shapes]
        engine = minispeed_amd.initialize(model=torch.nn.ParameterList(params), config={
            "train_micro_batch_size_per_gpu": 1, "dtype": "bf16",
            "optimizer": {"type": "AdamW", "params": {"lr": 0.1}}, "zero_optimization": {"stage": stage}})
        grads = [torch.randn(s, generator=gen, device="cuda").bfloat16() for s in shapes]
        for step in range(3):
            engine.optimizer.gather_parameters()
            if move and step:
                for p in params:
                    p.data = p.data.clone()
            if grads_move:
                grads = [t.clone() for t in grads]
            for p, t in zip(params, grads):
                p.grad = t
            engine.micro_steps += 1
            assert engine.step()
        engine.optimizer.gather_parameters()
        results.append([p.detach().clone() for p in params] + [engine.flat_groups[0].shard])
    for a, b in zip(*results):
        assert torch.equal(a, b)
