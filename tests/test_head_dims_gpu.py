"""The kernels built for query/key head_dim 192, with value head_dim 128 and 192 (tiles of 384-byte rows, operand
sizes that differ between the two contractions), and for 256: every forward path (one query, short and long query
sequences), the backward, ragged lengths, padding, strided tensors and the pairs that are padded to them, against
the dense CPU oracle."""
import numpy as np
import pytest
import torch

from kvax_amd import create_attention_mask, flash_attention
from kvax_amd.ops.flash_attention import flash_attention_backward, flash_attention_forward
from kvax_amd.utils import FlashAttentionParamsConfig, attention_specs
from kvax_amd.utils.benchmarking import generate_random_segments_lengths, make_random_attention_inputs
from oracle import attention_oracle as ao
from tests.tolerances import OPERAND_ROUNDING, check_close

pytestmark = pytest.mark.gpu
SPEC = ("data", None, "model", None)
P = FlashAttentionParamsConfig(64, 64)


def _inputs(b, sq, sk, hq, hkv, d, dv, pad, docs, device, dtype=torch.bfloat16):
    data, scale = make_random_attention_inputs(
        b, sq, sk, hq, hkv, d, dv, seed=sq + sk + d + dv, num_pad_tokens=pad, start_query_position=max(sk - sq, 0),
        list_of_segment_lengths=generate_random_segments_lengths(min(sq, sk), docs), device=device)
    return [t.to(dtype) for t in data[:3]], data[3:], scale


def _host(tensors):
    return [t.detach().float().cpu().numpy() if t.dtype.is_floating_point else t.cpu().numpy() for t in tensors]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b, sq, sk, hq, hkv, d, dv, pad, docs", [
    (2, 1, 5000, 8, 2, 192, 128, 0, 1),      # one query: four wavefronts share a tile, partial results of 128 and 192 columns
    (2, 1, 5000, 8, 2, 192, 192, 0, 1),
    (1, 48, 2000, 16, 4, 192, 128, 0, 1),    # split, two row tiles
    (1, 200, 3001, 4, 2, 192, 192, 0, 1),
    (2, 640, 640, 32, 32, 192, 128, 60, 4),  # work-groups of four wavefronts, ragged query tile
    (2, 520, 1111, 32, 16, 192, 192, 30, 3),
    (2, 640, 640, 32, 32, 256, 256, 60, 4),
    (2, 300, 300, 4, 2, 128, 160, 0, 2),     # padded to 192
    (1, 300, 300, 4, 2, 192, 40, 0, 2),
    (1, 300, 300, 4, 2, 64, 224, 0, 2),      # padded to 256
])
def test_forward(device, b, sq, sk, hq, hkv, d, dv, pad, docs, dtype):
    qkv, ids, scale = _inputs(b, sq, sk, hq, hkv, d, dv, pad, docs, device, dtype)
    with attention_specs(SPEC, SPEC):
        mask = create_attention_mask(*ids, fwd_params=P)
        out = flash_attention(*qkv, *ids, mask, scale=scale, fwd_params=P)
    assert out.shape == (b, sq, hq, dv)
    ref, _ = ao.attention_forward(*_host(qkv), *_host(ids), scale)
    check_close("out", out, ref)
    assert not out[ids[1] == -1].any()


@pytest.mark.parametrize("b, sq, sk, hq, hkv, d, dv, pad, docs, fp32", [
    (2, 640, 640, 4, 2, 192, 128, 65, 3, True),
    (1, 1000, 1000, 6, 2, 192, 192, 77, 9, True),   # ragged
    (1, 129, 65, 4, 4, 192, 128, 0, 1, False),      # the smallest number of tiles and a row beyond
    (3, 1280, 1280, 32, 32, 192, 128, 100, 4, False),  # more items than compute units: one part each
    (3, 1280, 1280, 32, 32, 256, 256, 100, 4, False),
    (1, 1000, 1000, 6, 2, 256, 256, 77, 9, True),
])
def test_backward(device, b, sq, sk, hq, hkv, d, dv, pad, docs, fp32):
    _check_backward(device, b, sq, sk, hq, hkv, d, dv, pad, docs, fp32, torch.bfloat16)


# Work-groups of the forward and of dQ take one, two, four or eight heads of a group (the largest power of two that divides it
# and is no more than the wavefronts): every group size with a remainder, rows that end inside a 32-row block, whole tiles of
# padding.  (dK and dV come from a kernel that does not know of it.)
@pytest.mark.parametrize("group", [1, 2, 3, 4, 6, 8, 16])
@pytest.mark.parametrize("n, d, dv", [(173, 64, 64), (173, 128, 128), (173, 192, 128), (397, 192, 128)])
def test_heads_of_a_group_share_a_work_group(device, group, n, d, dv):
    hkv = 2
    batch = -(-320 // (hkv * group * -(-n // 256)))  # so many that eight wavefronts run, and the key sequence is not divided
    (q, k, v), ids, scale = _inputs(batch, n, n, hkv * group, hkv, d, dv, 44, 3, device)
    dout = torch.randn((batch, n, hkv * group, dv), generator=torch.Generator().manual_seed(2)).to(q.dtype).to(device)
    with attention_specs(SPEC, SPEC):
        masks = create_attention_mask(*ids, fwd_params=P, bwd_params=P, calc_bwd_mask=True)
    out, lse = flash_attention_forward(q, k, v, *ids, masks[0], scale, P, P)
    dq = flash_attention_backward(q, k, v, *ids, masks[1], masks[2], out, lse, dout, scale, P, P)[0]
    rows = [0, batch - 1]
    q, k, v, dout, out, dq = (t[rows] for t in (q, k, v, dout, out, dq))
    ids = [t[rows] for t in ids]
    heads = sorted({0, hkv * group // 2 - 1, hkv * group // 2, hkv * group - 1})
    ref, _ = ao.attention_forward(*_host((q, k, v)), *_host(ids), scale)
    check_close("out", out, ref)
    ref = ao.attention_backward(*_host((q, k, v)), *_host(ids), scale, *_host([dout]), dtype=np.float64, heads=heads)[0]
    check_close("dq", dq[:, :, heads], ref[:, :, heads], rel=OPERAND_ROUNDING)
    assert not out[ids[1] == -1].any() and not dq[ids[1] == -1].any()


def _check_backward(device, b, sq, sk, hq, hkv, d, dv, pad, docs, fp32, dtype):
    (q, k, v), ids, scale = _inputs(b, sq, sk, hq, hkv, d, dv, pad, docs, device, dtype)
    # heads before the sequence in memory, as a caller with [batch, heads, seq, dim] tensors passes them
    q, v = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, v))
    dout = torch.randn((b, sq, hq, dv), generator=torch.Generator().manual_seed(2)).to(q.dtype).to(device)
    with attention_specs(SPEC, SPEC):
        masks = create_attention_mask(*ids, fwd_params=P, bwd_params=P, calc_bwd_mask=True)
    out, lse = flash_attention_forward(q, k, v, *ids, masks[0], scale, P, P)
    grads = flash_attention_backward(q, k, v, *ids, masks[1], masks[2], out, lse, dout, scale, P, P, dkdv_fp32=fp32)
    heads = None if hq < 32 else [1, hq - 1]
    refs = ao.attention_backward(*_host((q, k, v)), *_host(ids), scale, *_host([dout]), dtype=np.float64, heads=heads)
    if heads:
        grads, refs = ([x[:, :, heads] for x in grads], [r[:, :, heads] for r in refs])
    for name, got, ref in zip(("dq", "dk", "dv"), grads, refs):
        check_close(name, got, ref, rel=OPERAND_ROUNDING)
    assert not grads[0][ids[1] == -1].any() and not grads[1][ids[3] == -1].any() and not grads[2][ids[3] == -1].any()


# Work-groups of eight wavefronts: more than 256 of them (3 x 32 heads x 3 tiles of 256 rows, the last one ragged).


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d, dv", [(192, 128), (192, 192), (256, 256)])
def test_forward_with_eight_wavefronts(device, d, dv, dtype):
    (q, k, v), ids, scale = _inputs(3, 640, 640, 32, 32, d, dv, 60, 4, device, dtype)
    with attention_specs(SPEC, SPEC):
        mask = create_attention_mask(*ids, fwd_params=P)
    out, lse = flash_attention_forward(q, k, v, *ids, mask[0], scale, P, P)
    ref, ref_lse = ao.attention_forward(*_host((q, k, v)), *_host(ids), scale)
    check_close("out", out, ref)
    # in units of log2; fp32 sums of 256 products of 16-bit numbers of magnitude 1 (256 * 2^-24 * 256 * 0.64 / 16) and of 640 weights
    np.testing.assert_allclose(lse.cpu().numpy() * np.log(2.0), ref_lse, rtol=0, atol=2e-4)
    assert not out[ids[1] == -1].any()


def test_backward_with_eight_wavefronts_float16(device):
    _check_backward(device, 3, 640, 640, 32, 32, 192, 128, 60, 4, True, torch.float16)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_weight_of_the_largest_score_is_exact(device, dtype):
    """The key with a row's largest score enters with weight 1, which the 16-bit P holds exactly, also where the tile is worked
    on by halves and the key lies in the second one, with little above the first one's maximum."""
    b, sq, sk, h, d, top = 3, 640, 64, 32, 256, 41  # eight wavefronts, one tile
    g = torch.Generator(device=device).manual_seed(3)
    q, k, v = (torch.randn((b, n, h, d), generator=g, device=device, dtype=dtype) for n in (sq, sk, sk))
    q *= 0.25
    q[..., 0] = 4.0
    k[..., 0] = 0.0
    k[:, top] = 0.0
    k[:, top, :, 0] = 8.0  # score 2 for every row; the others are N(0, 1/16)
    v[:, :top] = v[:, top + 1:] = 0.0
    ids = [torch.zeros((b, n), dtype=torch.int32, device=device) for n in (sq, sq, sk, sk)]
    with attention_specs(SPEC, SPEC):
        out = flash_attention(q, k, v, *ids, create_attention_mask(*ids, fwd_params=P), scale=d ** -0.5, fwd_params=P)
    scores = [torch.mm(q[i, :, j].double(), k[i, :, j].double().t().contiguous()) * d ** -0.5 for i in range(b) for j in range(h)]
    assert all((s.argmax(dim=1) == top).all() for s in scores)
    weights = torch.stack([torch.softmax(s, dim=1)[:, top] for s in scores]).reshape(b, h, sq).transpose(1, 2)
    ref = (weights[..., None] * v[:, top:top + 1].double()).cpu().numpy()
    # what remains is the fp32 sum of the weights and the rounding of the result
    check_close("out", out, ref, atol=1e-5)


def _odd_rows(t):  # a slice of rows of width + 4
    return torch.nn.functional.pad(t, (0, 4))[..., :t.shape[3]]


def _odd_offset(t):
    return torch.nn.functional.pad(t.reshape(-1), (1, 0))[1:].view(t.shape)


def _columns(t):  # the head_dim axis is not contiguous
    return t.transpose(2, 3).contiguous().transpose(2, 3)


def _expanded(t):  # one row for all
    return t[:, :1, :1, :1].expand(t.shape)


@pytest.mark.parametrize("d, dv", [(192, 128), (192, 192), (64, 192)])
@pytest.mark.parametrize("view_q, view_k, view_v, view_dout", [
    (_odd_rows, _odd_rows, _odd_rows, _odd_rows), (_odd_offset,) * 4, (_columns,) * 4,
    (_odd_rows, _odd_offset, _columns, _expanded),
])
def test_any_strides_at_192(device, d, dv, view_q, view_k, view_v, view_dout):
    """Rows that the kernels cannot address, in the inputs and in the gradient of the output: the same bits as from contiguous
    tensors."""
    (q, k, v), ids, scale = _inputs(1, 128, 192, 4, 2, d, dv, 0, 2, device)
    dout = torch.randn((1, 128, 4, dv), generator=torch.Generator().manual_seed(2)).to(q.dtype).to(device)
    with attention_specs(SPEC, SPEC):
        masks = create_attention_mask(*ids, fwd_params=P, bwd_params=P, calc_bwd_mask=True)

        def run(q, k, v, dout):
            leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
            out = flash_attention(*leaves, *ids, masks, scale=scale, fwd_params=P, bwd_params=P)
            return out.detach(), *torch.autograd.grad(out, leaves, dout)

        given = [view(t) for view, t in zip((view_q, view_k, view_v, view_dout), (q, k, v, dout))]
        for got, want in zip(run(*given), run(*(t.contiguous().clone() for t in given))):
            assert torch.equal(got, want)


# At head_dim 64 and 128 eight wavefronts run where the tile bitmaps of the keys leave no room for two work-groups on a compute
# unit (more than 6929 and 3402 tiles of 64).  They take one, two, four or eight heads
# of a group; the rows end inside a 32-row block, and the documents of the queries are spread over the keys.
@pytest.mark.parametrize("group, hkv", [(1, 8), (2, 4), (4, 2), (8, 1), (12, 1)])
@pytest.mark.parametrize("d, sk", [(64, 460_000), (128, 230_000)])
def test_heads_of_a_group_share_a_work_group_of_eight_wavefronts(device, group, hkv, d, sk):
    sq, hq = 300, group * hkv
    seg = torch.arange(sk, device=device, dtype=torch.int32) * 7 // sk
    kv_pos = torch.arange(sk, device=device, dtype=torch.int32)
    at = torch.arange(sq, device=device) * 97 % 29 + torch.arange(sq, device=device) * (sk // sq)  # keys the queries stand at
    q_pos, q_seg = at.int(), seg[at]
    seg[sk - 3 * 64:], q_seg[-11:] = -1, -1
    ids = [x[None].contiguous() for x in (q_pos, q_seg, kv_pos, seg)]
    g = torch.Generator(device=device).manual_seed(d + group)
    shapes = [(1, sq, hq, d), (1, sk, hkv, d), (1, sk, hkv, d), (1, sq, hq, d)]
    q, k, v, dout = (torch.randn(s, generator=g, device=device, dtype=torch.bfloat16) for s in shapes)
    with attention_specs(SPEC, SPEC):
        masks = create_attention_mask(*ids, fwd_params=P, bwd_params=P, calc_bwd_mask=True)
    scale = d ** -0.5
    out, lse = flash_attention_forward(q, k, v, *ids, masks[0], scale, P, P)
    dq = flash_attention_backward(q, k, v, *ids, masks[1], masks[2], out, lse, dout, scale, P, P)[0]
    allowed = (q_seg[:, None] == seg) & (q_seg != -1)[:, None] & (q_pos[:, None] >= kv_pos)
    for h in {0, hq // 2, hq - 1}:  # float64
        kt, vt = (t[0, :, h // group].double() for t in (k, v))
        s = (q[0, :, h].double() @ kt.t().contiguous() * scale).masked_fill_(~allowed, float("-inf"))
        w = torch.softmax(s, 1).nan_to_num_(0.0)
        dp = dout[0, :, h].double() @ vt.t().contiguous()
        check_close("out", out[0, :, h], (w @ vt).cpu().numpy())
        check_close("dq", dq[0, :, h], (w * (dp - (w * dp).sum(1, keepdim=True)) @ kt * scale).cpu().numpy(), rel=OPERAND_ROUNDING)
    assert not out[ids[1] == -1].any() and not dq[ids[1] == -1].any()
