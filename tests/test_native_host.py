"""The host side of the calls in native code (kvax_amd/csrc/host.cpp): the plain case gives what the general path in Python
gives, bit for bit, and everything else is left to that path."""
import re
import shutil
import subprocess
import sys
import threading
import warnings

import pytest
import torch

import kvax_amd
from kvax_amd import FlashAttentionParamsConfig, Mesh, _native, attention_specs, create_attention_mask, flash_attention

ONE = (("data", None, "model", None), ("data", None, "model", None))
CP = (("data", "context", None, None), ("data", None, None, None))


class _Spy:
    """The native module; `taken` counts the calls it took, with `off` it takes none."""

    def __init__(self, real, off):
        self.real, self.off, self.taken = real, off, []

    def __getattr__(self, name):
        def call(*args):
            done = None if self.off else getattr(self.real, name)(*args)
            if done is not None:
                self.taken.append(name)
            return done
        return call


def test_what_is_not_on_the_gpu_is_left_alone():
    host = _native.host()
    ids = torch.zeros((1, 64), dtype=torch.int32)
    x = torch.zeros((1, 64, 2, 64), dtype=torch.bfloat16)
    mask = (torch.zeros((1, 1, 1), dtype=torch.int32),) * 4
    assert host.masks(ids, ids, ids, ids, ((64, 64, False),), 1, 1, 0, 0) is None
    assert host.forward(x, x, x, ids, ids, ids, ids, mask, 1.0, 64, 64, 64, 64, 0, 0) is None
    assert host.backward(x, x, x, ids, ids, ids, ids, mask, mask, x, x, x, 1.0, 64, 64, 64, 64, 1, 0, 0) is None
    for bad in (None, 3, "x"):
        assert host.masks(bad, ids, ids, ids, ((64, 64, False),), 1, 1, 0, 0) is None
        assert host.forward(bad, x, x, ids, ids, ids, ids, mask, 1.0, 64, 64, 64, 64, 0, 0) is None
    with pytest.raises(TypeError):
        host.forward(x)


def test_without_the_extension_the_calls_go_through_python(monkeypatch):
    """A torch that it was not built for, or no build of it: the library is still there."""
    monkeypatch.setattr(_native, "_host", None)
    monkeypatch.delattr(kvax_amd, "_host", raising=False)
    monkeypatch.setitem(sys.modules, "kvax_amd._host", None)
    with pytest.warns(RuntimeWarning, match="cannot be used"):
        host = _native.host()
    ids = torch.zeros((1, 64), dtype=torch.int32)
    assert host.masks(ids, ids, ids, ids, ((64, 64, False),), 1, 1, 0, 0) is None
    assert host.forward(*[None] * 15) is None and host.backward(*[None] * 20) is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert _native.host() is host


@pytest.mark.parametrize("which", range(4), ids=["abi_version", "fa_args", "mask_desc", "torch"])
def test_an_extension_built_for_something_else_is_not_used(which, monkeypatch):
    """It fills in structures for functions it gets as bare addresses and reads torch's tensors through inline code."""
    real = _native.host()
    key = list(_native._host_key(_native.lib()))
    key[which] = key[which] + (1 if which < 3 else ".post1")
    monkeypatch.setattr(_native, "_host_key", lambda l: tuple(key))
    monkeypatch.setattr(_native, "_host", None)
    with pytest.warns(RuntimeWarning, match=re.escape(str(key[which]))):
        host = _native.host()
    assert host is not real and host.forward(*[None] * 15) is None


@pytest.mark.parametrize("missing", ["torch", "g++", "headers"])
def test_the_library_is_built_without_what_only_the_extension_needs(missing, monkeypatch, tmp_path, capsys):
    from kvax_amd.csrc import build

    commands = []

    def run(cmd, **kwargs):
        commands.append(cmd)
        broken = cmd[0] == "g++" and missing == "headers"
        return subprocess.CompletedProcess(cmd, int(broken), "", "no headers" if broken else "")

    monkeypatch.setattr(build, "LIB", tmp_path / "lib.so")
    monkeypatch.setattr(build, "OBJ", tmp_path / "obj")
    monkeypatch.setattr(build.subprocess, "run", run)
    monkeypatch.setattr(shutil, "which", lambda name: None if name == missing else f"/usr/bin/{name}")
    if missing == "torch":
        monkeypatch.setitem(sys.modules, "torch", None)
    if missing == "headers":
        with pytest.raises(RuntimeError, match="no headers"):
            build.build()
    else:
        assert build.build() == tmp_path / "lib.so"
        assert not any(cmd[0] == "g++" for cmd in commands) and missing in capsys.readouterr().err
    assert any("-o" in cmd and cmd[cmd.index("-o") + 1] == str(tmp_path / "lib.so") for cmd in commands), "not linked"


# name -> (batch, q_len, kv_len, heads, kv heads, head_dim, value head_dim, shards, forward, backward in native code)
CASES = {
    "plain": (2, 192, 192, 4, 2, 64, 64, 1, True, True),
    "one_row": (1, 128, 128, 4, 4, 128, 128, 1, True, True),
    "values_narrower": (1, 128, 128, 4, 2, 192, 128, 1, True, True),
    "ragged_forward": (3, 77, 130, 4, 1, 128, 128, 1, True, None),
    "shards": (1, 256, 256, 4, 2, 128, 128, 2, True, True),
    "transposed_views": (2, 128, 128, 4, 2, 64, 64, 1, True, True),
    "int64_ids": (2, 128, 128, 4, 2, 64, 64, 1, False, True),
    "ids_not_contiguous": (2, 128, 128, 4, 2, 64, 64, 1, False, True),
    "mask_not_contiguous": (2, 128, 128, 4, 2, 64, 64, 1, False, False),
    "gradient_expanded": (1, 128, 128, 4, 2, 64, 64, 1, True, False),
    "half": (2, 192, 192, 4, 2, 128, 128, 1, True, True),
    "block_sizes": (3, 256, 384, 4, 2, 64, 64, 1, True, True),
    "block_sizes_shards": (2, 512, 384, 4, 2, 64, 64, 2, True, True),
}
IDS_TO_CONVERT = ("int64_ids", "ids_not_contiguous")  # masks from the Python code, as the forward


@pytest.mark.gpu
@pytest.mark.parametrize("name", CASES)
def test_same_bits_as_the_general_path(name, monkeypatch):
    b, sq, sk, hq, hkv, d, dv, cp, fwd_native, bwd_native = CASES[name]
    g = torch.Generator(device="cuda").manual_seed(1)
    dtype = torch.float16 if name == "half" else torch.bfloat16
    draw = lambda *s: torch.randn(s, generator=g, device="cuda", dtype=dtype)
    q, k, v = draw(b, sq, hq, d), draw(b, sk, hkv, d), draw(b, sk, hkv, dv)
    if name == "transposed_views":
        q, k, v = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v))
    dout = torch.ones((), device="cuda", dtype=torch.bfloat16).expand(b, sq, hq, dv) if name == "gradient_expanded" else draw(b, sq, hq, dv)
    ids = []
    for n in (sq, sk):
        pos = torch.arange(n, device="cuda", dtype=torch.int32).expand(b, n).contiguous()
        ids += [pos, (pos >= 50).int() - (pos >= n - 5).int() * 2]  # two documents and padding
    if name == "int64_ids":
        ids = [x.long() for x in ids]
    if name == "ids_not_contiguous":
        ids = [torch.stack([x, x], 2)[..., 0] for x in ids]
    # (apart: every size another, so that none can stand for another)
    apart = name.startswith("block_sizes")
    fwd_params = FlashAttentionParamsConfig(query_block_size=64 if not apart else 32, kv_block_size=64 if not apart else 16)
    bwd_params = FlashAttentionParamsConfig(query_block_size=64, kv_block_size=64 if not apart else 128)
    mesh = Mesh({"data": 1, "context": cp, "model": 1}) if cp > 1 else None
    real = _native.host()

    def run(spy):
        monkeypatch.setattr(_native, "host", lambda: spy)
        with attention_specs(*(CP if cp > 1 else ONE)):
            masks = create_attention_mask(*ids, fwd_params=fwd_params, bwd_params=bwd_params, calc_bwd_mask=True, mesh=mesh)
            arrays = [a for m in masks for a in m.flatten()]
            if name == "mask_not_contiguous":
                masks = tuple(type(m)(*[torch.stack([a, a], -1)[..., 0] for a in m.flatten()]) for m in masks)
            x = [t.detach().requires_grad_(True) for t in (q, k, v)]
            out = flash_attention(*x, *ids, masks, scale=d ** -0.5, fwd_params=fwd_params, bwd_params=bwd_params, mesh=mesh)
            grads = torch.autograd.grad(out, x, dout) if bwd_native is not None else []
        return arrays + [out.detach(), *grads]

    spy = _Spy(real, off=False)
    got, want = run(spy), run(_Spy(real, off=True))
    assert ("masks" in spy.taken) == (name not in IDS_TO_CONVERT)
    assert ("forward" in spy.taken) == fwd_native and ("backward" in spy.taken) == bool(bwd_native)
    for a, e in zip(got, want):
        assert a.shape == e.shape and a.stride() == e.stride() and a.dtype == e.dtype and torch.equal(a, e)


@pytest.mark.gpu
def test_errors_of_the_library_reach_the_caller():
    q = torch.zeros((1, 64, 2, 68), device="cuda", dtype=torch.bfloat16)[..., :64]  # rows not of 16-byte pieces
    ids = torch.zeros((1, 64), device="cuda", dtype=torch.int32)
    params = FlashAttentionParamsConfig(query_block_size=64, kv_block_size=64)
    with attention_specs(*ONE):
        mask = create_attention_mask(ids, ids, ids, ids, fwd_params=params)
        with pytest.raises(_native.KvaxNativeError, match="multiples of 8"):
            flash_attention(q, q, q, ids, ids, ids, ids, mask, fwd_params=params, bwd_params=params)


class _Tagged(torch.Tensor):
    """A subclass whose torch functions are seen, and give tensors of the subclass, as torch.Tensor's default does."""
    seen = []

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        cls.seen.append(getattr(func, "__name__", str(func)))
        return super().__torch_function__(func, types, args, kwargs or {})


class _Watch(torch.overrides.TorchFunctionMode):
    def __init__(self):
        super().__init__()
        self.seen = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.seen.append(getattr(func, "__name__", str(func)))
        return func(*args, **(kwargs or {}))


@pytest.mark.gpu
def test_subclasses_and_function_modes_see_the_calls(monkeypatch):
    """What overrides torch functions sees the allocations of a call, and a subclass's results are of the subclass; parameters
    and the mode of a default device are plain."""
    n, params = 128, FlashAttentionParamsConfig(query_block_size=64, kv_block_size=64)
    g = torch.Generator(device="cuda").manual_seed(1)
    data = [torch.randn((1, n, h, 64), generator=g, device="cuda", dtype=torch.bfloat16) for h in (4, 2, 2, 4)]
    pos = torch.arange(n, device="cuda", dtype=torch.int32).expand(1, n).contiguous()
    ids = (pos, pos // 50, pos, pos // 50)
    real = _native.host()

    def run(wrap):
        spy = _Spy(real, off=False)
        monkeypatch.setattr(_native, "host", lambda: spy)
        x = [wrap(t.clone()).requires_grad_(True) for t in data[:3]]
        with attention_specs(*ONE):
            masks = create_attention_mask(*ids, fwd_params=params, bwd_params=params, calc_bwd_mask=True)
            out = flash_attention(*x, *ids, masks, scale=0.125, fwd_params=params, bwd_params=params)
            grads = torch.autograd.grad(out, x, data[3])
        return spy.taken, (out, *grads)

    plain = lambda t: t
    taken, want = run(plain)
    assert taken == ["masks", "forward", "backward"]
    as_bits = lambda ts: [t.detach().as_subclass(torch.Tensor).view(torch.int16) for t in ts]
    same = lambda got: all(torch.equal(a, b) for a, b in zip(as_bits(got), as_bits(want)))

    taken, got = run(torch.nn.Parameter)
    assert taken == ["masks", "forward", "backward"] and same(got)
    with torch.device("cuda"):
        taken, got = run(plain)
    assert taken == ["masks", "forward", "backward"] and same(got)

    _Tagged.seen.clear()
    taken, got = run(lambda t: t.as_subclass(_Tagged))
    assert taken == ["masks"] and same(got)
    assert type(got[0]) is _Tagged and "empty_like" in _Tagged.seen
    with _Watch() as mode:
        taken, got = run(plain)
    # (the backward runs in autograd's thread of the device, where the mode is not active)
    assert taken == ["backward"] and same(got)
    assert {"empty", "empty_like"} <= set(mode.seen)


def _training_pass(seed, hq, hkv, d, n):
    """(inputs, a function of them that builds the masks and runs forward and backward)"""
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = [torch.randn((2, n, h, d), generator=g, device="cuda", dtype=torch.bfloat16) for h in (hq, hkv, hkv, hq)]
    pos = torch.arange(n, device="cuda", dtype=torch.int32).expand(2, n).contiguous()
    ids = (pos, pos // 300, pos, pos // 300)
    params = FlashAttentionParamsConfig(query_block_size=64, kv_block_size=64)

    def run(q, k, v, dout):
        q, k, v = (t.detach().requires_grad_(True) for t in (q, k, v))
        masks = create_attention_mask(*ids, fwd_params=params, bwd_params=params, calc_bwd_mask=True)
        out = flash_attention(q, k, v, *ids, masks, scale=d ** -0.5, fwd_params=params, bwd_params=params)
        return (*(a for m in masks for a in m.flatten()), out.detach(), *torch.autograd.grad(out, (q, k, v), dout))

    return x, run


@pytest.mark.gpu
def test_two_threads_on_streams_of_their_own(monkeypatch):
    """The interpreter lock is released in the launches, and memory and kernels are those of each thread's current stream."""
    spy = _Spy(_native.host(), off=False)
    monkeypatch.setattr(_native, "host", lambda: spy)
    with attention_specs(*ONE):
        passes = [_training_pass(1, 8, 2, 128, 1024), _training_pass(2, 4, 4, 64, 768)]
        want = [run(*x) for x, run in passes]
        torch.cuda.synchronize()
        got, errors = [[], []], []

        def worker(i):
            try:
                x, run = passes[i]
                stream = torch.cuda.Stream()
                with torch.cuda.stream(stream):
                    for _ in range(20):
                        # (what ran on the stream before may lie where the next pass allocates: all are kept and compared)
                        got[i].append(run(*x))
                stream.synchronize()
            except Exception as e:  # surfaced below
                errors.append(e)

        threads = [threading.Thread(target=worker, args=(i,)) for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join(60)
    assert not errors and all(len(x) == 20 for x in got)
    assert {name: spy.taken.count(name) for name in ("masks", "forward", "backward")} == dict.fromkeys(("masks", "forward", "backward"), 42)
    for results, ref in zip(got, want):
        assert all(torch.equal(a, b) for result in results for a, b in zip(result, ref))


@pytest.mark.gpu
def test_graph_replays_match_eager(monkeypatch):
    """A step recorded into a graph through the native calls and replayed on new inputs, with eager work between the replays."""
    spy = _Spy(_native.host(), off=False)
    monkeypatch.setattr(_native, "host", lambda: spy)
    with attention_specs(*ONE):
        x, run = _training_pass(3, 8, 2, 128, 1024)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            run(*x)  # the kernels' LDS limits, autograd's thread
        torch.cuda.current_stream().wait_stream(side)
        static = [t.clone() for t in x]
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            results = run(*static)
        assert spy.taken == ["masks", "forward", "backward"] * 2
        for seed in (4, 5, 6):
            g = torch.Generator(device="cuda").manual_seed(seed)
            new = [torch.randn(t.shape, generator=g, device="cuda", dtype=t.dtype) for t in x]
            for to, t in zip(static, new):
                to.copy_(t)
            graph.replay()
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(results, run(*new))), f"replay {seed}"
