"""dK/dV of launches with few work items, where several work-groups share the steps of an item and their
fp32 results are added: against the dense CPU oracle, at uneven shares, shares without any step, ragged
lengths, padding, strided outputs' types and at the largest number of parts."""
import numpy as np
import pytest
import torch

from kvax_amd import create_attention_mask
from kvax_amd.ops.flash_attention import flash_attention_backward, flash_attention_forward
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
