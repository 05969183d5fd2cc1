"""All context shards in one call: the dK/dV kernel's walk over shard-local masks, and the chunk
permutation kernel."""
import pytest
import torch

from kvax_amd import FlashAttentionParamsConfig, Mesh, attention_specs, create_attention_mask, flash_attention
from kvax_amd.ops.flash_attention import flash_attention_backward, flash_attention_forward
from kvax_amd.utils.benchmarking import generate_random_segments_lengths, make_random_attention_inputs
from kvax_amd.utils.permutation import apply_permutation, generate_shard_indices

pytestmark = pytest.mark.gpu
CP_SPECS = (("data", "context", None, None), ("data", None, None, None))


@pytest.mark.parametrize("sq, sk, cp, block, heads, kv_heads, dim, pad, docs", [
    (96, 128, 3, 32, 2, 2, 64, 0, 1),         # shards of half a query tile: tiles straddle two shards
    (320, 320, 2, 32, 4, 1, 128, 40, 3),      # a shard that starts inside a tile, padding, several documents
    (1024, 1024, 8, 64, 4, 2, 128, 700, 2),   # shards that are padding only
    (512, 700, 4, 128, 2, 1, 256, 0, 4),      # ragged keys, head_dim 256
])
def test_shards_in_one_call_equal_shard_by_shard(device, sq, sk, cp, block, heads, kv_heads, dim, pad, docs):
    data, scale = make_random_attention_inputs(
        2, sq, sk, heads, kv_heads, dim, dim, seed=sq + cp, num_pad_tokens=pad,
        list_of_segment_lengths=generate_random_segments_lengths(min(sq, sk), docs), device=device)
    q, k, v, q_pos, q_seg, kv_pos, kv_seg = data
    dout = torch.randn(q.shape, generator=torch.Generator().manual_seed(1)).to(q.dtype).to(device)
    p = FlashAttentionParamsConfig(block, block)
    mesh = Mesh({"data": 1, "context": cp, "model": 1})
    with attention_specs(*CP_SPECS):
        masks = create_attention_mask(q_pos, q_seg, kv_pos, kv_seg, fwd_params=p, bwd_params=p, calc_bwd_mask=True,
                                      mesh=mesh)
    out, lse = flash_attention_forward(q, k, v, q_pos, q_seg, kv_pos, kv_seg, masks[0], scale, p, p)
    got = flash_attention_backward(q, k, v, q_pos, q_seg, kv_pos, kv_seg, masks[1], masks[2], out, lse, dout, scale, p, p,
                                   dkdv_fp32=True, dkdv_shards=cp)
    # shard by shard, each with its own slice of everything (what one device of the group computes)
    n, dqs, dk, dv = sq // cp, [], 0, 0
    for r in range(cp):
        sl, nb = slice(r * n, (r + 1) * n), masks[1].lower_bounds.shape[-1] // cp
        dq_mask = tuple(a[..., r * nb:(r + 1) * nb].contiguous() for a in masks[1].flatten())
        kv_mask = tuple(a[:, r:r + 1].contiguous() for a in masks[2].flatten())
        dq_r, dk_r, dv_r = flash_attention_backward(
            q[:, sl], k, v, q_pos[:, sl].contiguous(), q_seg[:, sl].contiguous(), kv_pos, kv_seg, dq_mask, kv_mask,
            out[:, sl], lse[:, :, sl].contiguous(), dout[:, sl], scale, p, p, dkdv_fp32=True)
        dqs.append(dq_r)
        dk, dv = dk + dk_r, dv + dv_r
    # the same products in the same precision; sums of fp32 terms in another order, and exponentials
    # of scores whose sums met other tile boundaries: far inside one unit in the last place of bf16
    for name, a, b in zip(("dq", "dk", "dv"), got, (torch.cat(dqs, 1), dk, dv)):
        a, b = a.float(), b.float()
        assert (a - b).abs().max() <= 2 ** -8 * b.abs().max() and (a - b).norm() <= 1e-3 * b.norm(), name
    if pad:
        assert not got[1][:, sk - pad:].any() and not got[2][:, sk - pad:].any()


@pytest.mark.parametrize("built_for", [1, 2, 8])
def test_masks_of_another_mesh_are_refused(device, built_for):
    data, scale = make_random_attention_inputs(2, 512, 512, 4, 2, 64, 64, seed=5, device=device)
    p = FlashAttentionParamsConfig(32, 32)
    meshes = [Mesh({"data": 1, "context": cp, "model": 1}) for cp in (built_for, 4)]
    leaf = data[0].requires_grad_(True)
    with attention_specs(*CP_SPECS):
        masks = create_attention_mask(*data[3:], fwd_params=p, bwd_params=p, calc_bwd_mask=True, mesh=meshes[0])
        out = flash_attention(*data, masks, scale=scale, fwd_params=p, bwd_params=p, mesh=meshes[1])
        with pytest.raises(ValueError, match="the dK/dV mask has shape"):
            out.backward(torch.ones_like(out))
    assert leaf.grad is None


@pytest.mark.parametrize("shape, chunks, dtype", [
    ((1, 2, 1), 2, torch.int32), ((3, 12, 5), 4, torch.int32), ((2, 16, 3, 8), 16, torch.bfloat16),
    ((2, 6, 1, 1), 2, torch.bfloat16), ((1, 4096, 2, 64), 8, torch.bfloat16), ((2, 10, 3), 10, torch.float64),
    ((1, 2, 100003), 2, torch.int32),
])
def test_chunk_permutation(device, shape, chunks, dtype):
    x = torch.arange(torch.Size(shape).numel(), device=device).reshape(shape).to(dtype)
    order = torch.tensor(generate_shard_indices(chunks), device=device)
    want = x.reshape(shape[0], chunks, -1)[:, order].reshape(shape)
    assert torch.equal(apply_permutation([x], chunks, False)[0], want)
    assert torch.equal(apply_permutation([want], chunks, True)[0], x)
    if dtype.is_floating_point:
        leaf, g = x.clone().requires_grad_(True), torch.randn_like(x)
        apply_permutation([leaf], chunks, False)[0].backward(g)
        assert torch.equal(leaf.grad, apply_permutation([g], chunks, True)[0])


def _by_index(x, chunks, reverse=False):
    order = torch.tensor(generate_shard_indices(chunks, reverse), device=x.device)
    return x.reshape(x.shape[0], chunks, -1).index_select(1, order).reshape(x.shape)


@pytest.mark.parametrize("dtype, width", [(torch.bfloat16, 2), (torch.bool, 4), (torch.int8, 4), (torch.float32, 1)])
def test_chunk_permutation_of_a_view_at_any_offset(device, dtype, width):
    """A batch of one is contiguous wherever it starts in its storage; so is its gradient."""
    base = (torch.randn((1, 1 + 8 * width), device=device) * 3).to(dtype)
    x = base[:, 1:].view(1, 8, width)
    assert x.is_contiguous() and (x.data_ptr() % 4 or dtype == torch.float32)
    assert torch.equal(apply_permutation([x], 4, False)[0], _by_index(x, 4))
    assert torch.equal(apply_permutation([x], 4, True)[0], _by_index(x, 4, True))
    if dtype.is_floating_point:
        leaf = torch.randn((1, 8, width), device=device).to(dtype).requires_grad_(True)
        apply_permutation([leaf], 4, False)[0].backward(x)
        assert torch.equal(leaf.grad, _by_index(x, 4, True))


def test_chunk_permutation_of_lazily_conjugated_and_negated_tensors(device):
    x = torch.randn((2, 8, 3), device=device, dtype=torch.complex64)
    for y in (x.conj(), x.conj().imag):
        assert y.is_conj() or y.is_neg()
        assert torch.equal(apply_permutation([y], 4, False)[0], _by_index(y.resolve_conj().resolve_neg(), 4))
    leaf = x.clone().requires_grad_(True)
    apply_permutation([leaf], 4, False)[0].backward(x.conj())
    assert torch.equal(leaf.grad, _by_index(x.conj().resolve_conj(), 4, True))


def test_chunk_permutation_under_transforms(device):
    """What an indexed copy composes with: function transforms, forward mode, batched gradients, second derivatives, tracing."""
    from torch.autograd import forward_ad
    from torch.fx.experimental.proxy_tensor import make_fx

    x, t = torch.randn((2, 2, 8, 3), device=device)
    many = torch.randn((5, 2, 8, 3), device=device)
    f = lambda y: apply_permutation([y], 4, False)[0]
    want = torch.stack([_by_index(y, 4) for y in many])
    assert torch.equal(torch.func.vmap(f)(many), want)
    assert torch.equal(torch.func.jvp(f, (x,), (t,))[1], _by_index(t, 4))
    assert torch.equal(torch.func.grad(lambda y: (f(y) * t).sum())(x), _by_index(t, 4, True))
    with forward_ad.dual_level():
        assert torch.equal(forward_ad.unpack_dual(f(forward_ad.make_dual(x, t))).tangent, _by_index(t, 4))
    leaf = x.clone().requires_grad_(True)
    got = torch.autograd.grad(f(leaf), leaf, many, is_grads_batched=True)[0]
    assert torch.equal(got, torch.stack([_by_index(y, 4, True) for y in many]))
    first = torch.autograd.grad((f(leaf) ** 2 * t).sum(), leaf, create_graph=True)[0]
    second = torch.autograd.grad(first.sum(), leaf)[0]
    torch.testing.assert_close(second, 2 * _by_index(t, 4, True))
    assert torch.equal(make_fx(f)(x)(t), _by_index(t, 4))
    assert torch.equal(torch.compile(f, backend="eager", fullgraph=True)(t), _by_index(t, 4))
    assert type(f(torch.nn.Parameter(x))) is torch.Tensor
