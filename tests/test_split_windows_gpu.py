"""Split forward with windows of up to eight tiles, whose tiles the work-groups summarise themselves, and the first longer
one: against the dense CPU oracle, with windows that lie across the words of the live-tile bitmap, documents, padding, and
NaN in the keys of a document inside the windows that no row attends to."""
import ctypes
import sys

import numpy as np
import pytest
import torch

from kvax_amd import _native, create_attention_mask
from kvax_amd.ops.flash_attention import flash_attention_forward
from kvax_amd.utils import FlashAttentionParamsConfig, attention_specs
from oracle import attention_oracle as ao
from tests.tolerances import check_close

pytestmark = pytest.mark.gpu
flash_attention_module = sys.modules["kvax_amd.ops.flash_attention"]  # (the package exports a function of that name)


def check_lse(got, ref, keys=500):
    """Base 2 against natural.  fp32 sums: a logit is off by at most (D + 1) 2^-24 sum |q k| scale = 1.6e-4 at D = 256 and normal
    inputs, the sum over the keys by keys x 2^-24, v_exp_f32 and v_log_f32 by an ulp."""
    assert np.abs(got.cpu().numpy() * np.log(2.0) - ref).max() <= 1e-3 + keys * 2.0 ** -24


@pytest.mark.parametrize("d, dv", [(64, 64), (128, 128), (192, 128), (256, 256)])
@pytest.mark.parametrize("sq, sk, hq, hkv", [
    (40, 4480, 4, 1),     # windows of 4 tiles
    (40, 20500, 4, 1),    # of 6: some lie across a 64-tile word
    (40, 32700, 4, 1),    # of 8
    (40, 33000, 4, 1),    # of 9: a launch summarises the sequence
    (130, 65, 4, 2),      # one window, less than two tiles
    (777, 777, 8, 2),
])
def test_short_windows(device, sq, sk, hq, hkv, d, dv):
    rng = np.random.default_rng(sq + sk)
    kv_pos = np.arange(sk, dtype=np.int32)[None]
    kv_seg = (np.arange(sk) >= sk // 3).astype(np.int32)[None]
    kv_seg[:, sk - sk // 8:] = -1
    q_pos = (sk - 1 - np.arange(sq)[::-1] % sk).astype(np.int32)[None]
    q_seg = np.where(np.arange(sq) % 97 < 9, 0, 1).astype(np.int32)[None]
    q_seg = np.sort(q_seg, axis=1)
    q_seg[:, -3:] = -1
    ids = [torch.from_numpy(np.ascontiguousarray(x)).to(device) for x in (q_pos, q_seg, kv_pos, kv_seg)]
    draw = lambda *s: torch.from_numpy(rng.standard_normal(s, dtype=np.float32)).to(torch.bfloat16).to(device)
    q, k, v = draw(1, sq, hq, d), draw(1, sk, hkv, d), draw(1, sk, hkv, dv)
    p = FlashAttentionParamsConfig(64, 64)
    spec = ("data", None, "model", None)
    with attention_specs(spec, spec):
        mask = create_attention_mask(*ids, fwd_params=p)
    ref, ref_lse = ao.attention_forward(*(x.float().cpu().numpy() for x in (q, k, v)), q_pos, q_seg, kv_pos, kv_seg, d ** -0.5)
    if sk > 1000:  # whole tiles of padding beyond the block mask: not in any window, whatever they hold
        first = -(-(sk - sk // 8) // 64) * 64
        k[:, first:], v[:, first:] = float("nan"), float("nan")
    out, lse = flash_attention_forward(q, k, v, *ids, mask[0], d ** -0.5, p, p)
    check_close("out", out, ref)
    check_lse(lse, ref_lse, sk)
    assert not out[ids[1] == -1].any()


# One resident set of work-groups (512, or 256 above head_dim 128) summarises its windows itself, with more a launch does:
# the summaries at the start of the workspace are left alone or written.
@pytest.mark.parametrize("d, dv, resident", [(64, 64, 512), (128, 128, 512), (192, 128, 256), (256, 256, 256)])
@pytest.mark.parametrize("more", [0, 1])
def test_more_work_groups_than_resident_take_summaries_from_a_launch(device, d, dv, resident, more):
    hkv, sq, sk = 8, 40, 130
    b = resident // hkv + more
    seg = (np.arange(sk) >= 70).astype(np.int32)
    seg[-9:] = -1
    kv = [np.broadcast_to(x, (b, sk)).copy() for x in (np.arange(sk, dtype=np.int32), seg)]
    ids = [x[:, 45:45 + sq].copy() for x in kv] + kv
    on_gpu = [torch.from_numpy(x).to(device) for x in ids]
    g = torch.Generator(device=device).manual_seed(7)
    q, k, v = (torch.randn(s, generator=g, device=device, dtype=torch.bfloat16) for s in ((b, sq, hkv, d), (b, sk, hkv, d), (b, sk, hkv, dv)))
    p = FlashAttentionParamsConfig(64, 64)
    spec = ("data", None, "model", None)
    with attention_specs(spec, spec):
        mask = create_attention_mask(*on_gpu, fwd_params=p)[0]
    a = flash_attention_module._base_args(q, k, v, *on_gpu, d ** -0.5, p, p)
    out, lse = q.new_empty((b, sq, hkv, dv)), torch.empty((b, hkv, sq), device=device)
    a.out, a.lse, a.o_strides = out.data_ptr(), lse.data_ptr(), flash_attention_module._strides3(out)
    a.fwd_mask = flash_attention_module._mask_ptrs(mask)
    lib = _native.lib()
    ws = torch.full((lib.kvax_fa_fwd_workspace_bytes(ctypes.byref(a)),), 0x5A, dtype=torch.uint8, device=device)
    assert ws.numel() >= 32 * b * 3
    rc = lib.kvax_fa_fwd(ctypes.byref(a), ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)
    _native.check(rc, "kvax_fa_fwd")
    assert bool((ws[:32 * b * 3] != 0x5A).any()) == bool(more)
    rows = [0, b - 1]
    ref, ref_lse = ao.attention_forward(*(t[rows].float().cpu().numpy() for t in (q, k, v)), *(x[rows] for x in ids), d ** -0.5)
    check_close("out", out[rows], ref)
    check_lse(lse[rows], ref_lse)


@pytest.mark.parametrize("d, dv", [(64, 64), (128, 128), (192, 128), (256, 256)])
def test_short_windows_of_rows_without_any_key(device, d, dv):
    """Work-groups whose block mask names no key at all (queries of padding, keys of padding) beside ones with keys."""
    b, sq, sk, hq, hkv = 3, 130, 300, 4, 2
    seg = np.zeros((b, sk), np.int32)
    q_seg = np.zeros((b, sq), np.int32)
    q_seg[0], seg[1] = -1, -1
    pos = np.broadcast_to(np.arange(sk, dtype=np.int32), (b, sk)).copy()
    ids = [pos[:, sk - sq:].copy(), q_seg, pos, seg]
    on_gpu = [torch.from_numpy(x).to(device) for x in ids]
    g = torch.Generator(device=device).manual_seed(9)
    q, k, v = (torch.randn(s, generator=g, device=device, dtype=torch.bfloat16) for s in ((b, sq, hq, d), (b, sk, hkv, d), (b, sk, hkv, dv)))
    p = FlashAttentionParamsConfig(64, 64)
    spec = ("data", None, "model", None)
    with attention_specs(spec, spec):
        mask = create_attention_mask(*on_gpu, fwd_params=p)[0]
    out, lse = flash_attention_forward(q, k, v, *on_gpu, mask, d ** -0.5, p, p)
    ref, ref_lse = ao.attention_forward(*(t.float().cpu().numpy() for t in (q, k, v)), *ids, d ** -0.5)
    check_close("out", out, ref)
    check_lse(lse, ref_lse)
    assert not out[:2].any() and not lse[:2].any()


# The document in the middle of the keys has no queries: its tiles lie inside [lower, upper) of the block mask, whose blocks hold
# queries of the documents on either side, and are passed over for what the work-groups know of them.  Its whole tiles hold
# NaN, which would reach the results through 0 x NaN of any tile that is worked on.
@pytest.mark.parametrize("d, dv, dtype", [(64, 64, torch.bfloat16), (128, 128, torch.float16), (192, 128, torch.bfloat16),
                                          (256, 256, torch.float16)])
@pytest.mark.parametrize("b, sq, sk, hq, hkv", [
    (1, 40, 4480, 4, 1),     # windows of 4 tiles
    (2, 40, 20500, 4, 1),    # of 6
    (1, 40, 32700, 4, 1),    # of 8
    (1, 40, 33000, 4, 1),    # of 9: a launch summarises the sequence
    (2, 777, 777, 4, 2),
])
def test_dead_tiles_inside_the_windows(device, b, sq, sk, hq, hkv, d, dv, dtype):
    first, last = sk * 3 // 10, sk * 7 // 10  # the document without queries
    kv_pos = np.broadcast_to(np.arange(sk, dtype=np.int32), (b, sk)).copy()
    kv_seg = ((kv_pos >= first).astype(np.int32) + (kv_pos >= last)).astype(np.int32)
    kv_seg[:, sk - 20:] = -1
    q_pos = np.maximum(kv_pos[:, sk - sq:], last + 64)  # every query sees the first document and some of the last
    q_seg = np.where(np.arange(sq) < 16, 0, 2).astype(np.int32) * np.ones((b, 1), np.int32)
    q_seg[:, -3:] = -1
    if b > 1:
        q_seg[1] = np.where(np.arange(sq) < 9, 0, 2)  # rows of the batch differ
    host = (q_pos, q_seg, kv_pos, kv_seg)
    ids = [torch.from_numpy(x).to(device) for x in host]
    g = torch.Generator().manual_seed(sq + sk + d)
    q, k, v = (torch.randn(s, generator=g).to(dtype).to(device) for s in ((b, sq, hq, d), (b, sk, hkv, d), (b, sk, hkv, dv)))
    p = FlashAttentionParamsConfig(64, 64)
    spec = ("data", None, "model", None)
    with attention_specs(spec, spec):
        mask = create_attention_mask(*ids, fwd_params=p)[0]
    ref, ref_lse = ao.attention_forward(*(x.float().cpu().numpy() for x in (q, k, v)), *host, d ** -0.5)
    dead = slice(-(-first // 64), last // 64)  # its whole tiles
    lower, upper = (x[:, 0, 0].cpu().numpy() for x in (mask.lower_bounds, mask.upper_bounds))
    assert dead.stop > dead.start and (lower <= dead.start).all() and (upper >= dead.stop).all()
    k[:, dead.start * 64:dead.stop * 64], v[:, dead.start * 64:dead.stop * 64] = float("nan"), float("nan")
    out, lse = flash_attention_forward(q, k, v, *ids, mask, d ** -0.5, p, p)
    check_close("out", out, ref)
    check_lse(lse, ref_lse, sk)
    assert not out[ids[1] == -1].any() and not lse.transpose(1, 2)[ids[1] == -1].any()
