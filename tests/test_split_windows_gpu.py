"""Split forward with windows of up to eight tiles, whose tiles the work-groups summarise themselves, and the first longer
one: against the dense CPU oracle, with windows that lie across the words of the live-tile bitmap, documents, padding and
NaN in keys of tiles that nothing attends to."""
import numpy as np
import pytest
import torch

from kvax_amd import create_attention_mask
from kvax_amd.ops.flash_attention import flash_attention_forward
from kvax_amd.utils import FlashAttentionParamsConfig, attention_specs
from oracle import attention_oracle as ao
from tests.tolerances import check_close

pytestmark = pytest.mark.gpu


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
    ref, _ = ao.attention_forward(*(x.float().cpu().numpy() for x in (q, k, v)), q_pos, q_seg, kv_pos, kv_seg, d ** -0.5)
    if sk > 1000:  # whole tiles of padding: dead, whatever they hold
        first = -(-(sk - sk // 8) // 64) * 64
        k[:, first:], v[:, first:] = float("nan"), float("nan")
    out, _ = flash_attention_forward(q, k, v, *ids, mask[0], d ** -0.5, p, p)
    check_close("out", out, ref)
    assert not out[ids[1] == -1].any()
