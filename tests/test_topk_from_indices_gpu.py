"""TopK backward that makes its own pair list (flexsae_topk_bwd_from_indices): the values of flexsae_csr_build and
flexsae_topk_bwd, dvals and dbias rounded once to the leaves' types, bit for bit; at buckets of every kind (in registers, with
frequent latents, too large for registers, more latents than the bucketed construction takes), widths of every vector, rows
that do not fill a chunk, and indices out of range."""
import ctypes

import pytest
import torch

from flexsae_amd import _lib
from tests import abi

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


def _from_indices(indices, weight, vals, resid, grad, leaf_dtypes, flags, flag):
    lib = _lib.load()
    sh = abi.shape_of(indices, weight, vals)
    dW = torch.full((sh.F, sh.D), float("nan"), dtype=weight.dtype, device=DEV)
    dv = torch.full((sh.B, sh.K), float("nan"), dtype=leaf_dtypes[0], device=DEV)
    db = torch.full((sh.D,), float("nan"), dtype=leaf_dtypes[1], device=DEV)
    g = torch.tensor([grad], dtype=torch.float32, device=DEV)
    nbytes = lib.flexsae_topk_bwd_from_indices_workspace_bytes(ctypes.byref(sh), 0)
    ws = torch.full((nbytes,), 0xAB, dtype=torch.uint8, device=DEV)
    args = (abi.ptr(indices), abi.ptr(weight), abi.ptr(vals), abi.ptr(resid), abi.ptr(g), abi.ptr(dW), abi.DT[weight.dtype],
            abi.ptr(dv), abi.DT[leaf_dtypes[0]], abi.ptr(db), abi.DT[leaf_dtypes[1]], abi.ptr(ws))
    assert lib.flexsae_topk_bwd_from_indices(ctypes.byref(sh), *args, 256, flags, abi.ptr(flag),
                                             abi.stream()) == _lib.ERR_WORKSPACE
    rc = lib.flexsae_topk_bwd_from_indices(ctypes.byref(sh), *args, nbytes, flags, abi.ptr(flag), abi.stream())
    assert rc == 0
    return dW, dv, db


@pytest.mark.parametrize("dtype,leaf_dtypes,flags", [
    (torch.float32, (torch.float32, torch.float32), 0), (torch.bfloat16, (torch.bfloat16, torch.bfloat16), 0),
    (torch.bfloat16, (torch.float32, torch.float16), _lib.TOPK_BWD_FP32_RESIDUAL),
    (torch.float16, (torch.float16, torch.bfloat16), 0)], ids=["fp32", "bf16", "bf16_fp32_resid", "fp16"])
@pytest.mark.parametrize("B,K,F,D,kind", [
    (1, 1, 1, 1, "uniform"), (63, 3, 7, 9, "uniform"), (65, 32, 4096, 256, "uniform"), (130, 17, 501, 262, "uniform"),
    (777, 20, 3000, 515, "uniform"), (500, 40, 2048, 520, "frequent"), (1000, 100, 300, 68, "uniform"),
    (3000, 30, 5000, 36, "frequent"), (64, 5, 40000, 2, "uniform")])
def test_same_values(B, K, F, D, kind, dtype, leaf_dtypes, flags):
    print("[case]", B, K, F, D, kind, dtype, flush=True)
    g = torch.Generator().manual_seed(B + D)
    idx = torch.randint(0, F, (B, K), generator=g)
    if kind == "frequent":  # half of the pairs on five latents of one bucket
        idx = torch.where(torch.rand(B, K, generator=g) < 0.5, torch.randint(0, 5, (B, K), generator=g), idx)
    bad = torch.rand(B, K, generator=g) < 0.01
    idx[bad] = torch.tensor([-1, F, 2 ** 40])[torch.randint(0, 3, (int(bad.sum()),), generator=g)]
    W = torch.randn(F, D, generator=g).to(dtype).to(DEV)
    v = torch.randn(B, K, generator=g).to(leaf_dtypes[0]).to(DEV)
    resid = torch.randn(B, D, generator=g).to(DEV)
    idx_d = idx.to(DEV)
    flag = torch.zeros(1, dtype=torch.int32, device=DEV)
    rc, dW, dv, db = abi.topk_backward(idx_d, W, v, resid, 1.5, flags=flags)
    assert rc == 0
    got = _from_indices(idx_d, W, v, resid, 1.5, leaf_dtypes, flags, flag)
    torch.cuda.synchronize()
    assert int(flag.item()) == (_lib.FLAG_INDEX_RANGE if bad.any() else 0)
    for a, b in zip(got, (dW, dv.to(leaf_dtypes[0]), db.to(leaf_dtypes[1]))):
        assert torch.equal(a, b)


@pytest.mark.parametrize("F", [1 << 25, (1 << 25) + 1])  # 8192 buckets of 4096 latents, and one latent more
def test_more_latents_than_buckets_take(F):
    idx = torch.tensor([[0, F - 1, 5], [F - 1, 7, F]], device=DEV)
    W = torch.ones(F, 1, device=DEV)
    v = torch.tensor([[1.0, 2.0, 3.0], [4.0, 5.0, 6.0]], device=DEV)
    resid = torch.tensor([[1.0], [-2.0]], device=DEV)
    flag = torch.zeros(1, dtype=torch.int32, device=DEV)
    dW, dv, db = _from_indices(idx, W, v, resid, 1.0, (torch.float32, torch.float32), 0, flag)
    assert int(flag.item()) == _lib.FLAG_INDEX_RANGE
    at = torch.tensor([0, 5, 7, F - 1], device=DEV)
    assert dW[at, 0].tolist() == [1.0, 3.0, -10.0, 2.0 - 8.0] and int((dW != 0).sum()) == 4
    assert dv.tolist() == [[1.0, 1.0, 1.0], [-2.0, -2.0, -2.0]] and db.tolist() == [-1.0]
