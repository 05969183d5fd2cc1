"""The mask builder's one-launch kernel and the line to the two-launch pair: edges of its groups of 16 lanes, of 64
outer blocks, of the number of blocks and of the lengths, block sizes that are no multiple of 16, and query shards,
bit for bit against the oracle."""
import numpy as np
import pytest
import torch

from kvax_amd.ops.mask_creator import build_masks
from oracle import mask_oracle as mo
from tests.test_oracle_mask import _random_ids

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sq, sk, qbs, kbs, batch, shards", [
    (1, 1, 1, 1, 1, 1), (17, 15, 16, 16, 3, 1), (1000, 333, 48, 100, 2, 1), (1040, 4096, 16, 128, 2, 1),
    (2048, 2048, 16, 16, 2, 1), (2048, 2049, 16, 16, 1, 1), (128, 128, 1, 1, 2, 1), (129, 128, 1, 1, 1, 1),  # 128 blocks, and one more
    (2048, 2048, 1, 1, 1, 1), (2049, 2048, 1, 16, 1, 1),
    (3000, 4000, 512, 512, 2, 1), (3000, 4000, 513, 129, 2, 1),
    (4096, 4096, 128, 128, 1, 1), (4096, 4097, 128, 128, 1, 1), (1, 4096, 128, 64, 4, 1),
    (4096, 3072, 64, 128, 2, 8), (32768, 32768, 128, 128, 1, 4),
])
@pytest.mark.parametrize("skip_pad", [True, False])
def test_against_oracle(device, sq, sk, qbs, kbs, batch, shards, skip_pad):
    rng = np.random.default_rng([sq, sk, qbs, int(skip_pad)])
    ids = [*_random_ids(rng, batch, sq, "restart"), *_random_ids(rng, batch, sk, "restart")]
    dev = [torch.from_numpy(np.ascontiguousarray(a)).to(device) for a in ids]
    requests = [(qbs, kbs, False), (kbs, qbs, False), (qbs, kbs, True)]
    if shards > 1:  # shards hold whole query blocks of every mask
        requests = [(qbs, kbs, False), (qbs, kbs, True)]
    got = build_masks(*dev, requests, skip_pad, num_q_shards=shards)
    for mask, (bq, bk, kv_outer) in zip(got, requests):
        if kv_outer and shards > 1:
            n = sq // shards
            parts = [mo.block_mask_c(ids[0][:, r * n:(r + 1) * n], ids[1][:, r * n:(r + 1) * n], *ids[2:], bq, bk, skip_pad, True)
                     for r in range(shards)]
            want = [np.concatenate([p[i] for p in parts], axis=1) for i in range(4)]
        else:
            want = mo.block_mask_c(*ids, bq, bk, skip_pad, kv_outer)
        for x, y in zip(mask.flatten(), want):
            np.testing.assert_array_equal(x.cpu().numpy(), y)
