"""dK/dV of launches with few work items, where several work-groups share the steps of an item and their
fp32 results are added: against the dense CPU oracle, at uneven shares, shares without any step, ragged
lengths, padding, strided outputs' types and at the largest number of parts."""
import numpy as np
import pytest
import torch

from kvax_amd import create_attention_mask
from kvax_amd.ops.flash_attention import backward_workspace_bytes, flash_attention_backward, flash_attention_forward
from kvax_amd.ops.mask_creator import build_masks
from kvax_amd.utils import FlashAttentionParamsConfig, attention_specs
from kvax_amd.utils.benchmarking import generate_random_segments_lengths, make_random_attention_inputs
from oracle import attention_oracle as ao
from tests.tolerances import OPERAND_ROUNDING, check_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b, sq, sk, hq, hkv, d, pad, docs, fp32", [
    (1, 512, 512, 8, 1, 64, 0, 1, False),     # 8 parts of 8 steps
    (1, 2048, 2048, 8, 1, 128, 100, 1, True),  # 16 parts, one causal document: the last keys have a few steps only
    (2, 1000, 1000, 6, 2, 128, 77, 9, True),  # ragged; 6 parts of 48 (head, tile) pairs, documents leave most without a step
    (1, 777, 300, 12, 4, 64, 0, 1, False),    # more queries than keys, uneven shares
    (3, 640, 640, 4, 1, 256, 65, 3, True),
    (1, 512, 512, 16, 16, 64, 0, 1, False),   # too few steps to share: one part
    (1, 65, 129, 32, 1, 128, 0, 1, True),     # as few tiles as possible
    (1, 129, 65, 4, 4, 256, 0, 1, False),     # head_dim 256 takes half tiles: the second half of the last one holds no row
    (2, 96, 96, 4, 2, 256, 0, 2, False),
])
def test_shared_items_match_dense_oracle(device, b, sq, sk, hq, hkv, d, pad, docs, fp32):
    data, scale = make_random_attention_inputs(
        b, sq, sk, hq, hkv, d, d, seed=sq + hq + d, num_pad_tokens=pad, start_query_position=max(sk - sq, 0),
        list_of_segment_lengths=generate_random_segments_lengths(min(sq, sk), docs), device=device)
    q, k, v, *ids = data
    dout = torch.randn(q.shape, generator=torch.Generator().manual_seed(2)).to(q.dtype).to(device)
    p = FlashAttentionParamsConfig(64, 64)
    spec = ("data", None, "model", None)
    with attention_specs(spec, spec):
        masks = create_attention_mask(*ids, fwd_params=p, bwd_params=p, calc_bwd_mask=True)
    out, lse = flash_attention_forward(q, k, v, *ids, masks[0], scale, p, p)
    _, dk, dv = flash_attention_backward(q, k, v, *ids, masks[1], masks[2], out, lse, dout, scale, p, p, dkdv_fp32=fp32)
    host = [x.cpu().numpy() for x in ids]
    refs = ao.attention_backward(*(x.float().cpu().numpy() for x in (q, k, v)), *host, scale,
                                 dout.float().cpu().numpy(), dtype=np.float64)
    for name, got, ref in (("dk", dk, refs[1]), ("dv", dv, refs[2])):
        # P and dS enter the sums rounded to 16 bits, whatever the number of heads that share a key
        check_close(name, got, ref, rel=OPERAND_ROUNDING)
        assert not got[torch.from_numpy(host[3] == -1)].any(), "padding rows must be zero"


# With 257 to 512 items of up to 160 steps or more the device decides from the documents: one long document in the batch (its first
# items are longer than a compute unit's share: two parts), or equally long items (one part), ragged, with padding and without
# any key.
@pytest.mark.parametrize("layout, fp32", [("one_long", False), ("one_long", True), ("equal", False), ("equal", True),
                                          ("one_long_padded", False), ("nothing", False)])
@pytest.mark.parametrize("hkv, d, dv", [(8, 64, 64), (8, 128, 128), (8, 192, 128), (4, 256, 256)])
def test_device_decides_whether_items_are_shared(device, layout, fp32, hkv, d, dv):
    b, n, group = 2, 2600, 4  # 41 tiles of 64 tokens
    seg = np.zeros((b, n), np.int32)
    pos = np.zeros((b, n), np.int32) if layout == "equal" else np.broadcast_to(np.arange(n, dtype=np.int32), (b, n)).copy()
    if layout.startswith("one_long"):
        seg[1] = np.arange(n) // 70
        if layout == "one_long_padded":
            seg[:, -200:] = -1
    elif layout == "nothing":
        seg[:] = -1
    ids = [torch.from_numpy(x).to(device) for x in (pos, seg, pos, seg)]
    g = torch.Generator().manual_seed(3)
    shapes = [(b, n, hkv * group, d), (b, n, hkv, d), (b, n, hkv, dv), (b, n, hkv * group, dv)]
    q, k, v, dout = (torch.randn(s, generator=g).to(torch.bfloat16).to(device) for s in shapes)
    p = FlashAttentionParamsConfig(64, 64)
    spec = ("data", None, "model", None)
    with attention_specs(spec, spec):
        masks = create_attention_mask(*ids, fwd_params=p, bwd_params=p, calc_bwd_mask=True)
    scale = d ** -0.5
    out, lse = flash_attention_forward(q, k, v, *ids, masks[0], scale, p, p)
    run = lambda: flash_attention_backward(q, k, v, *ids, masks[1], masks[2], out, lse, dout, scale, p, p, dkdv_fp32=fp32)[1:]
    grads, again = run(), run()
    # one kv head of each row; the dense computation in fp32 (its error of 1e-5 of the sums is far below that of the
    # rounded operands)
    for row, head in ((0, hkv - 1), (1, 0)):
        hs = slice(head * group, (head + 1) * group)
        f = lambda t, h: t[row:row + 1, :, h].float().cpu().numpy()
        kv = slice(head, head + 1)
        refs = ao.attention_backward(f(q, hs), f(k, kv), f(v, kv), *(x[row:row + 1] for x in (pos, seg, pos, seg)), scale, f(dout, hs),
                                     dtype=np.float32)[1:]
        for name, got, repeat, ref in zip(("dk", "dv"), grads, again, refs):
            assert torch.equal(got, repeat)
            check_close(name, got[row:row + 1, :, kv], ref, rel=OPERAND_ROUNDING)
            assert not got[ids[3] == -1].any(), "padding rows must be zero"


def _dense_kv_head(q, k, v, dout, q_pos, q_seg, kv_pos, kv_seg, scale):
    """dK and dV of one kv head of one row, float64, from the heads of its group."""
    k, v = k.double(), v.double()
    allowed = (q_seg[:, None] == kv_seg) & (q_seg != -1)[:, None] & (q_pos[:, None] >= kv_pos)
    dk, dv = torch.zeros_like(k), torch.zeros_like(v)
    for h in range(q.shape[1]):
        qh, do = q[:, h].double(), dout[:, h].double()
        s = (qh @ k.t().contiguous() * scale).masked_fill_(~allowed, float("-inf"))
        s = torch.softmax(s, 1).nan_to_num_(0.0)  # (rows without any key)
        dv += s.t().contiguous() @ do
        dp = do @ v.t().contiguous()
        ds = s.mul_(dp.sub_((s * dp).sum(1, keepdim=True)))
        dk += ds.t().contiguous() @ qh * scale
    return dk, dv


# The ways the items are dealt to the XCDs that a deciding launch can have (see ItemMap: at least 8 (row, kv head) pairs; a
# number that divides 8; another one), context shards, fp16, values of 192, and more queries than the list of live tiles
# holds (2048 tiles of 64 at head_dim 128).  Whether the items were shared shows in the workspace, at whose end the parts lie.
# (The device decides for 257 to 512 items of 128 keys, 64 at 256, for which the shapes alone give one part.)
@pytest.mark.parametrize("shared", [True, False])
@pytest.mark.parametrize("b, sq, sk, group, hkv, d, dv, dtype, shards", [
    (1, 25600, 25550, 1, 2, 64, 64, torch.bfloat16, 1),
    (1, 13000, 13000, 2, 2, 256, 256, torch.bfloat16, 1),
    (1, 17152, 17100, 1, 3, 128, 128, torch.bfloat16, 1),
    (2, 2600, 2600, 4, 8, 128, 128, torch.float16, 1),
    (2, 2600, 2600, 4, 8, 192, 192, torch.bfloat16, 1),
    (2, 2688, 2688, 4, 8, 64, 64, torch.bfloat16, 2),
    (2, 2688, 2688, 4, 8, 192, 128, torch.float16, 3),
    (1, 131200, 2100, 1, 24, 128, 128, torch.bfloat16, 1),
])
def test_the_decision_and_what_follows_from_it(device, shared, b, sq, sk, group, hkv, d, dv, dtype, shards):
    rng = np.random.default_rng(5)
    long_queries = sq > 100_000
    if long_queries:  # every query sees its document: of nine tenths of the queries and the first 600 keys, or all of all
        q_seg, kv_seg = (np.arange(sq) >= 120_000) * shared, (np.arange(sk) >= 600) * shared
        q_pos, kv_pos = np.full(sq, sk), np.arange(sk)
    else:  # one causal document, or short ones
        q_seg, kv_seg = (np.arange(n) // (n if shared else 70) for n in (sq, sk))
        q_pos, kv_pos = np.arange(sq) + max(sk - sq, 0), np.arange(sk)
    host = [np.broadcast_to(x.astype(np.int32), (b, x.size)).copy() for x in (q_pos, q_seg, kv_pos, kv_seg)]
    if b > 1 and shared:  # (the other row's items are short)
        host[1][1], host[3][1] = np.arange(sq) // 70, np.arange(sk) // 70
    host[1][:, -40:] = host[3][:, -40:] = -1
    ids = [torch.from_numpy(x).to(device) for x in host]
    g = torch.Generator(device=device).manual_seed(3)
    shapes = [(b, sq, hkv * group, d), (b, sk, hkv, d), (b, sk, hkv, dv), (b, sq, hkv * group, dv)]
    q, k, v, dout = (torch.randn(s, generator=g, device=device, dtype=dtype) for s in shapes)
    p = FlashAttentionParamsConfig(64, 64)
    spec = ("data", None, "model", None)
    with attention_specs(spec, spec):
        fwd, dq_mask, dkdv_mask = build_masks(*ids, [(64, 64, False), (64, 64, False), (64, 64, True)], num_q_shards=shards)
    scale = d ** -0.5
    out, lse = flash_attention_forward(q, k, v, *ids, fwd, scale, p, p)
    parts = 2 * b * sk * hkv * (d + dv) * 4
    grads = []
    for fill in (0x5A, 0xA5):  # nothing depends on what the workspace held
        ws = torch.full((backward_workspace_bytes(q, k, v),), fill, dtype=torch.uint8, device=device)
        assert ws.numel() > parts
        buffers = (torch.empty_like(q), torch.empty_like(k), torch.empty_like(v), ws)
        flash_attention_backward(q, k, v, *ids, dq_mask, dkdv_mask, out, lse, dout, scale, p, p, buffers=buffers, dkdv_shards=shards)
        assert bool((ws[-parts:] != fill).any()) == shared
        grads.append(buffers[1:3])
    for name, got, again in zip(("dk", "dv"), *grads):
        assert torch.equal(got, again)
        assert not got[ids[3] == -1].any(), "padding rows must be zero"
    for row, head in {(0, hkv - 1), (b - 1, rng.integers(hkv))}:
        hs = slice(head * group, (head + 1) * group)
        refs = _dense_kv_head(q[row, :, hs], k[row, :, head], v[row, :, head], dout[row, :, hs], *(x[row] for x in ids), scale)
        for name, got, ref in zip(("dk", "dv"), grads[0], refs):
            check_close(name, got[row, :, head], ref.cpu().numpy(), rel=OPERAND_ROUNDING)
