"""What a user of this package has it do, as cases that can be timed: mask building, serving (prefill and decoding) and
training with packed documents, through ``create_attention_mask`` and ``flash_attention`` (and its gradients).

Sizes are those of the package's workloads, tests and command line, and generic ones between them.  The
document lengths of a case are a function of the case alone, so that its work is known exactly; their order along the
sequence, and every tensor, come from the seed (for a mask, whose work does not depend on them, the lengths too).
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from kvax_amd import (
    PADDING_SEGMENT_ID,
    FlashAttentionParamsConfig,
    Mesh,
    attention_specs,
    create_attention_mask,
    flash_attention,
    permute_tokens_context_parallelism,
)

ONE_DEVICE = (("data", None, "model", None), ("data", None, "model", None))
CONTEXT_PARALLEL = (("data", "context", None, None), ("data", None, None, None))

# (query heads, kv heads) of the package's workloads, tests and command line
HEADS = ((32, 8), (64, 8), (16, 16), (16, 4), (8, 2), (4, 1), (8, 8))


def _case(kind, **fields):
    case = dict(kind=kind, batch=1, q_len=1, kv_len=1, heads=32, kv_heads=8, d_qk=128, d_v=128, dtype="bf16",
                documents=0, spread="lognormal", causal=True, pad=0.0, block=128, layout=0, cp=1, mask="kept")
    case.update(fields)
    return case


def listed():
    return [
        # Three block masks (forward, dQ, dK/dV) of one packed 32k training batch: built once per batch, ahead of the
        # layers; a latency of a few launches.
        _case("mask", name="mask_32k", q_len=32768, kv_len=32768, documents=2048, pad=0.05),
        # A chat program's token: four short conversations, mask and one attention call. Host work and launches.
        _case("decode", name="token_2k", batch=4, kv_len=2048, mask="built"),
        # A token of eight long conversations, one of the layers that share a mask: reads the key cache, nothing else.
        _case("decode", name="token_32k", batch=8, kv_len=32768),
        # A short prompt of an odd length, mask and one attention call, head_dim 64.
        _case("prefill", name="prompt_777", q_len=777, kv_len=777, heads=8, kv_heads=2, d_qk=64, d_v=64, mask="built"),
        # A chunk of a long prompt against the cache that its beginning has filled.
        _case("prefill", name="chunk_512_of_24k", q_len=512, kv_len=24000),
        # One long prompt, float16.
        _case("prefill", name="prompt_8k", q_len=8192, kv_len=8192, dtype="fp16"),
        # A training step of a small model: one packed row, head_dim 64.
        _case("train", name="train_2k_d64", q_len=2048, kv_len=2048, heads=8, kv_heads=2, d_qk=64, d_v=64, documents=512,
              pad=0.0625, block=64),
        # Training with query/key heads wider than the value heads (low-rank key compression expands to this).
        _case("train", name="train_4k_d192", batch=2, q_len=4096, kv_len=4096, heads=16, kv_heads=16, d_qk=192, d_v=128,
              documents=1024),
        # Training at the widest head.
        _case("train", name="train_8k_d256", q_len=8192, kv_len=8192, heads=16, kv_heads=4, d_qk=256, d_v=256, documents=2048,
              pad=0.05),
        # Packed long-context training, the package's headline workload.
        _case("train", name="train_32k", q_len=32768, kv_len=32768, documents=2048, pad=0.05),
        # Bidirectional training over many short documents with a quarter of padding: the block mask skips most of it.
        _case("train", name="train_4x16k_short", batch=4, q_len=16384, kv_len=16384, heads=64, documents=512,
              spread="exponential", causal=False, pad=0.25),
        # Context parallelism: eight query shards, permuted for load balance, keys and values whole.
        _case("context", name="context_8x8k", q_len=65536, kv_len=65536, documents=4096, cp=8),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _head_dims(rng):
    """Mostly the common sizes; now and then each of the others that the package takes."""
    return rng.choice([(128, 128)] * 4 + [(64, 64)] * 2 + [(32, 32), (192, 128), (192, 192), (256, 256)])


def _drawn(rng):
    kind = rng.choice(["mask", "decode", "decode", "prefill", "prefill", "train", "train", "train", "train", "context"])
    heads, kv_heads = rng.choice(HEADS)
    d_qk, d_v = _head_dims(rng)
    common = dict(heads=heads, kv_heads=kv_heads, d_qk=d_qk, d_v=d_v, dtype=rng.choice(["bf16", "bf16", "fp16"]),
                  block=rng.choice([64, 128]), layout=rng.randrange(1 << 20), mask=rng.choice(["kept", "built"]))
    if kind == "mask":
        length = _log_int(rng, 2000, 131072)
        return _case(kind, **common, batch=rng.choice([1, 1, 2, 4, 8]), q_len=length, kv_len=length,
                     documents=_log_int(rng, 32, max(33, length // 8)), causal=rng.random() < 0.75, pad=rng.choice([0.0, 0.05, 0.25]))
    if kind == "decode":
        slots, batch = _log_int(rng, 200, 65536), _log_int(rng, 1, 32)
        return _case(kind, **common, batch=batch, q_len=rng.choice([1, 1, 1, rng.randint(2, 8)]), kv_len=slots)
    if kind == "prefill":
        if rng.random() < 0.4:  # a chunk against a filled cache
            chunk = _log_int(rng, 16, 2048)
            return _case(kind, **common, batch=rng.choice([1, 1, 2]), q_len=chunk, kv_len=chunk + _log_int(rng, 500, 60000))
        length = _log_int(rng, 40, 16384)
        return _case(kind, **common, batch=rng.choice([1, 1, 2, 4]), q_len=length, kv_len=length,
                     documents=rng.choice([0, 0, 1024]), pad=rng.choice([0.0, 0.0, 0.3]))
    if kind == "train":
        block = common["block"]
        length = block * _log_int(rng, 4, 32768 // block)
        batch = _log_int(rng, 1, max(1, min(16, 65536 // length)))
        causal = rng.random() < 0.75
        return _case(kind, **common, batch=batch, q_len=length, kv_len=length, documents=rng.choice([0, _log_int(rng, 200, 4096)]),
                     spread=rng.choice(["lognormal", "exponential"]), causal=causal, pad=rng.choice([0.0, 0.05, 0.25]))
    cp = rng.choice([2, 4, 8])
    length = 2 * cp * 128 * rng.randint(1, 65536 // (256 * cp))
    common.update(d_qk=128, d_v=128, mask="kept")
    return _case(kind, **common, q_len=length, kv_len=length, documents=rng.choice([0, 4096]), cp=cp)


def draw(rng: random.Random):
    most = max(work(c)["flops"] for c in listed())
    while True:
        case = _drawn(rng)
        size = work(case)
        # the key cache and the tensors of a drawn case stay within what the listed ones hold, too
        if size["flops"] <= most and size["bytes"] <= 3e9:
            return case


# ---- layout of the sequences -------------------------------------------------------------------------------------------------


def _filled(case):
    """Keys in the cache of each batch row (decoding: from half full to full; a chunk: all)."""
    if case["kind"] == "decode":
        return np.linspace(case["kv_len"] / 2, case["kv_len"], case["batch"] + 1)[1:].astype(np.int64).clip(case["q_len"])
    return np.full(case["batch"], case["kv_len"], np.int64)


def _lengths(case, seed=0):
    """Document lengths of each batch row; what they leave of the row is padding."""
    rng = np.random.default_rng((case["layout"], seed))
    rows = []
    for row in range(case["batch"]):
        # rows of a padded batch differ in how much of them is padding
        pad = case["pad"] * (0.8 + 0.4 * (row + 0.5) / case["batch"])
        left = case["kv_len"] - int(round(pad * case["kv_len"]))
        mean, lengths = case["documents"], []
        while left > 0:
            if mean == 0:
                n = left
            elif case["spread"] == "lognormal":  # `documents` is the median
                n = int(np.clip(rng.lognormal(math.log(mean), 1.0), 32, 8 * mean))
            else:
                n = int(max(32, rng.exponential(mean)))
            lengths.append(min(n, left))
            left -= lengths[-1]
        rows.append(lengths)
    return rows


def _packed(case):
    """Queries and keys are the same tokens (training, whole prompts, masks)."""
    return case["q_len"] == case["kv_len"] and case["kind"] != "decode"


def _ids(case, seed):
    """(query positions, query segment ids, kv positions, kv segment ids) as int32 [batch, length] arrays."""
    b, sq, sk = case["batch"], case["q_len"], case["kv_len"]
    rng = np.random.default_rng(seed)
    if _packed(case):
        pos, seg = np.zeros((b, sk), np.int32), np.full((b, sk), PADDING_SEGMENT_ID, np.int32)
        # the ids are all that a mask is made from
        for row, lengths in enumerate(_lengths(case, seed if case["kind"] == "mask" else 0)):
            at = 0
            for i, n in enumerate(rng.permutation(np.array(lengths, np.int64))):
                seg[row, at:at + n] = i
                if case["causal"]:  # positions restart in every document; constant ones attend both ways
                    pos[row, at:at + n] = np.arange(n)
                at += n
            if case["causal"]:
                pos[row, at:] = np.arange(sk - at)
        return pos, seg, pos.copy(), seg.copy()
    filled = rng.permutation(_filled(case))
    kv_pos = np.broadcast_to(np.arange(sk, dtype=np.int32), (b, sk)).copy()
    kv_seg = np.where(kv_pos < filled[:, None], 0, PADDING_SEGMENT_ID).astype(np.int32)
    q_pos = (filled[:, None] - sq + np.arange(sq)[None]).astype(np.int32)
    return q_pos, np.zeros((b, sq), np.int32), kv_pos, kv_seg


def _pairs(case):
    """(query, key) pairs that may attend, over the batch."""
    if _packed(case):
        return sum(n * (n + 1) // 2 if case["causal"] else n * n for row in _lengths(case) for n in row)
    sq = case["q_len"]
    return sum(int(f) * sq - sq * (sq - 1) // 2 for f in _filled(case))


# ---- one case -----------------------------------------------------------------------------------------------------------------


def _params(case):
    return FlashAttentionParamsConfig(query_block_size=case["block"], kv_block_size=case["block"])


def _build_mask(s):
    backward = s["case"]["kind"] in ("mask", "train", "context")
    return create_attention_mask(*s["ids"], fwd_params=s["params"], bwd_params=s["params"], calc_bwd_mask=backward,
                                 mesh=s["mesh"])


def prepare(case, seed):
    device = torch.device("cuda")
    s = dict(case=case, params=_params(case), mesh=None, specs=ONE_DEVICE, scale=case["d_qk"] ** -0.5)
    ids = [torch.from_numpy(x).to(device) for x in _ids(case, seed)]
    tensors = []
    if case["kind"] != "mask":
        g = torch.Generator(device=device).manual_seed(seed)
        dtype = {"bf16": torch.bfloat16, "fp16": torch.float16}[case["dtype"]]
        b, sq, sk, hq, hkv = (case[k] for k in ("batch", "q_len", "kv_len", "heads", "kv_heads"))
        shapes = [(b, sq, hq, case["d_qk"]), (b, sk, hkv, case["d_qk"]), (b, sk, hkv, case["d_v"])]
        if case["kind"] in ("train", "context"):
            shapes.append((b, sq, hq, case["d_v"]))  # the gradient of the output
        tensors = [torch.randn(shape, generator=g, device=device, dtype=dtype) for shape in shapes]
    if case["kind"] == "context":
        s["mesh"] = Mesh({"data": 1, "context": case["cp"], "model": 1})
        s["specs"] = CONTEXT_PARALLEL
        with attention_specs(*s["specs"]):
            q, k, v, dout = permute_tokens_context_parallelism(tensors, mesh=s["mesh"])
            ids[:2] = permute_tokens_context_parallelism(ids[:2], mesh=s["mesh"])
        tensors = [q, k, v, dout]
    s["ids"], s["qkv"], s["dout"] = ids, tensors[:3], tensors[3] if len(tensors) == 4 else None
    if s["dout"] is not None:
        for t in s["qkv"]:
            t.requires_grad_(True)
    if case["mask"] == "kept" and case["kind"] != "mask":
        # the layers of a model share the masks of a batch
        with attention_specs(*s["specs"]):
            s["mask"] = _build_mask(s)
    return s


def run(s):
    with attention_specs(*s["specs"]):
        if s["case"]["kind"] == "mask":
            return [m.flatten() for m in _build_mask(s)]
        mask = s["mask"] if "mask" in s else _build_mask(s)
        out = flash_attention(*s["qkv"], *s["ids"], mask, scale=s["scale"], fwd_params=s["params"], bwd_params=s["params"],
                              mesh=s["mesh"])
        if s["dout"] is None:
            return out
        return [out.detach(), *torch.autograd.grad(out, s["qkv"], s["dout"])]


def work(case):
    b, sq, sk = case["batch"], case["q_len"], case["kv_len"]
    blocks_q, blocks_k = -(-sq // case["block"]), -(-sk // case["block"])
    masks = 16 * b * (2 * blocks_q + case["cp"] * blocks_k)
    id_bytes = 8 * b * (sq + sk)
    if case["kind"] == "mask":
        return {"bytes": id_bytes + masks, "flops": 0}
    hq, hkv, dk, dv = case["heads"], case["kv_heads"], case["d_qk"], case["d_v"]
    keys = int(_filled(case).sum())
    data = 2 * (b * sq * hq * (dk + dv) + keys * hkv * (dk + dv))  # q and the output, keys and values
    pairs = _pairs(case) * hq
    if case["kind"] in ("decode", "prefill"):
        return {"bytes": id_bytes + data, "flops": 2 * (dk + dv) * pairs}
    # forward: q, k, v in, output out; backward: those and dout in, dq, dk, dv out
    data += 2 * (b * sq * hq * (2 * dk + 2 * dv) + 2 * keys * hkv * (dk + dv))
    return {"bytes": id_bytes + masks + data, "flops": 2 * (dk + dv) * pairs + 2 * (3 * dk + 2 * dv) * pairs}


def tolerance(case):
    if case["kind"] == "mask":
        return "exact"
    # Four times what the results differ from the same path in float64: relative 2.5e-3 (bf16) and 3.7e-4 (fp16); at most 0.036
    # of an output's rms and 0.1 of a gradient's in bf16, an eighth of that in fp16.
    bf16, forward = case["dtype"] == "bf16", case["kind"] in ("decode", "prefill")
    return {"rel": 1e-2 if bf16 else 1.5e-3, "max": (0.15 if forward else 0.4) / (1 if bf16 else 8)}
