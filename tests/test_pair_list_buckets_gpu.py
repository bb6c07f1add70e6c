"""Pair lists at the sizes where the number of latents per bucket changes: one latent per bucket, one block per compute unit
exactly, two batches of latents to a bucket, and one bucket more than that."""
import numpy as np
import pytest
import torch

import abi
import oracle

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("skew", [False, True])
@pytest.mark.parametrize("shape", [
    (1024, 64, 32768), (1777, 50, 24571),    # half the pairs to a bucket
    (4096, 64, 256), (4096, 64, 257),        # one latent to a bucket: 256 blocks; two
    (4096, 64, 65536), (4096, 64, 65537),    # 256 buckets; one more would be too many
    (2048, 64, 131072), (2048, 64, 131073),  # two batches of latents to a bucket: 256 blocks; as many as there were
    (31, 33, 1)])
def test_pair_list_where_buckets_change(shape, skew):
    B, K, F = shape
    g = torch.Generator().manual_seed(B + F + skew)
    idx = torch.randint(0, F, (B, K), generator=g)
    if skew:
        idx = torch.where(torch.rand(B, K, generator=g) < 0.5, torch.randint(0, 9, (B, K), generator=g) * 613 % F, idx)
    want_begin, want_map = oracle.csr(idx, F)
    rc, begin, mp = abi.csr_build(idx.to(DEV), F)
    torch.cuda.synchronize()
    assert rc == 0
    np.testing.assert_array_equal(abi.widen_u32(begin).cpu().numpy(), want_begin.astype(np.int64))
    np.testing.assert_array_equal(abi.widen_u32(mp).cpu().numpy(), want_map.astype(np.int64))
