"""Load-balancing token permutation for causal context parallelism.

The sequence axis (axis 1) is cut into ``2*cp`` equal chunks which are reordered as
``[0, 2cp-1, 1, 2cp-2, ...]`` so that shard ``r`` of ``cp`` owns original chunks ``r`` and
``2cp-1-r``: one cheap and one expensive chunk under a causal mask.  Behaviour follows
kvax/utils/permutation.py:9-116.
"""
from __future__ import annotations

from typing import Sequence

import torch
from torch.autograd import forward_ad

from kvax_amd import _native
from kvax_amd.utils.sharding import get_query_context_mesh_axis_size
from kvax_amd.utils.typing import DeviceArray


def generate_shard_indices(num_shards: int, reverse: bool = False) -> list[int]:
    """Chunk order ``[(i, num_shards-1-i) for i < num_shards/2]`` flattened, or its inverse."""
    order = []
    for i in range(num_shards // 2):
        order += [i, num_shards - 1 - i]
    if not reverse:
        return order
    inverse = [0] * len(order)
    for dst, src in enumerate(order):
        inverse[src] = dst
    return inverse


def _permute_on_device(x: torch.Tensor, num_shards: int, reverse: bool) -> torch.Tensor:
    # bytes are copied: a conjugate or a negative must be in memory first
    x = x.resolve_conj().resolve_neg().contiguous()
    if x.data_ptr() % 4:  # a view may start anywhere in its storage
        x = x.clone()
    out = torch.empty_like(x)
    chunk_bytes = x.numel() // (x.shape[0] * num_shards) * x.element_size()
    with torch.cuda.device(x.device):
        rc = _native.lib().kvax_permute_chunks(
            x.data_ptr(), out.data_ptr(), x.shape[0], num_shards, chunk_bytes, int(reverse),
            torch.cuda.current_stream().cuda_stream)
    _native.check(rc, "kvax_permute_chunks")
    return out


class _PermuteChunks(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, num_shards, reverse):
        ctx.num_shards, ctx.reverse = num_shards, reverse
        return _permute_on_device(x, num_shards, reverse)

    @staticmethod
    def backward(ctx, grad):
        return _permute(grad, ctx.num_shards, not ctx.reverse), None, None


def _is_plain(x: torch.Tensor) -> bool:
    """Whether x is memory and nothing else: no subclass, and no transform (vmap, forward-mode, batched
    gradients) or tracer that has to see the operations applied to it."""
    if torch.compiler.is_compiling() or torch.jit.is_tracing():
        return False
    functorch = torch._C._functorch
    return type(x) in (torch.Tensor, torch.nn.Parameter) and x.layout is torch.strided and not (
        torch._C._are_functorch_transforms_active() or functorch.is_functorch_wrapped_tensor(x)
        or functorch.is_legacy_batchedtensor(x) or torch._C._len_torch_dispatch_stack()
        or x._is_zerotensor() or forward_ad.unpack_dual(x).tangent is not None)


def _permute(x: torch.Tensor, num_shards: int, reverse: bool) -> torch.Tensor:
    """One tensor, permuted by the copy kernel; tensors it does not take (on the host, in pieces that are
    not a multiple of 4 bytes, more than a grid holds, or not plain memory) by an index."""
    if x.is_cuda and _is_plain(x) and x.numel() and x.shape[0] <= 65535 and num_shards % 2 == 0 and \
            num_shards <= 65534 and x.numel() // (x.shape[0] * num_shards) * x.element_size() % 4 == 0:
        return _PermuteChunks.apply(x, num_shards, reverse)
    order = generate_shard_indices(num_shards, reverse=reverse)
    idx = torch.as_tensor(order, device=x.device, dtype=torch.long)
    chunks = x.reshape(x.shape[0], num_shards, x.shape[1] // num_shards, *x.shape[2:])
    return chunks.index_select(1, idx).reshape(x.shape)


def apply_permutation(
    inputs: Sequence[DeviceArray], num_shards: int, reverse_permutation: bool
) -> list[DeviceArray]:
    outputs = []
    for x in inputs:
        seq = x.shape[1]
        if seq % num_shards != 0:
            raise ValueError(
                f"sequence length {seq} is not divisible by the number of chunks {num_shards}"
            )
        outputs.append(_permute(x, num_shards, reverse_permutation))
    return outputs


def _run(inputs, mesh, reverse: bool):
    num_shards = 2 * get_query_context_mesh_axis_size(mesh)
    single = isinstance(inputs, torch.Tensor)
    if single:
        inputs = (inputs,)
    lead = tuple(inputs[0].shape[:2])
    for x in inputs:
        if tuple(x.shape[:2]) != lead:
            raise AssertionError(
                f"inputs must share their (batch, sequence) prefix, got {lead} and "
                f"{tuple(x.shape[:2])}"
            )
    outputs = apply_permutation(inputs, num_shards, reverse)
    return outputs[0] if single else outputs


def permute_tokens_context_parallelism(inputs, mesh=None):
    """Reorder tokens along axis 1 for balanced causal work across context shards."""
    return _run(inputs, mesh, reverse=False)


def unpermute_tokens_context_parallelism(inputs, mesh=None):
    """Inverse of :func:`permute_tokens_context_parallelism`."""
    return _run(inputs, mesh, reverse=True)
