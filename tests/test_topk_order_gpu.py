"""TopK forward in latent order: shapes at the edges of its tiles, row blocks and sort widths, against float64 and
against the walk in the order given (the smaller workspace)."""
import ctypes

import pytest
import torch

from flexsae_amd import _lib
from tests import abi

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


def _forward(ws_bytes, idx, W, v, b, t, flag=None):
    sh = abi.shape_of(idx, W, v, b.dtype, t.dtype)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=DEV)
    loss = torch.full((1,), float("nan"), device=DEV)
    resid = torch.full((sh.B, sh.D), float("nan"), device=DEV)
    rc = _lib.load().flexsae_topk_fwd(ctypes.byref(sh), abi.ptr(idx), abi.ptr(W), abi.ptr(v), abi.ptr(b), abi.ptr(t),
                                      abi.ptr(loss), abi.ptr(resid), abi.ptr(ws), ws_bytes, abi.ptr(flag), abi.stream())
    torch.cuda.synchronize()
    assert rc == 0, _lib.status_string(rc)
    return loss, resid


# (B, K, F, D): rows of one, two, four and eight keys per lane, full and not; blocks of 4, 8 and 16 wavefronts with a last
# one that is not full; 128- and 256-byte pieces with a last one that is half a piece
@pytest.mark.parametrize("shape,dtype", [
    ((512, 128, 16384, 512), torch.float32),
    ((1029, 65, 20011, 2080), torch.float32),
    ((2051, 100, 16385, 672), torch.float32),
    ((2048, 256, 16384, 96), torch.float32),
    ((515, 257, 65537, 576), torch.bfloat16),
    ((700, 512, 131072, 256), torch.float16),
    ((1030, 255, 16384, 320), torch.bfloat16),
    ((2049, 129, 32768, 576), torch.bfloat16),
    ((4100, 64, 40000, 1088), torch.float16),
], ids=str)
def test_order_changes_only_the_rounding(shape, dtype):
    B, K, F, D = shape
    print("[case]", shape, dtype, flush=True)
    g = torch.Generator(device=DEV).manual_seed(B + K)
    idx = torch.randint(0, F, (B, K), generator=g, device=DEV)
    idx[::3, K // 2:] = idx[::3, :1]  # rows that repeat one latent
    idx[1, :] = torch.arange(K, device=DEV).flip(0)
    idx[2, K - 1], idx[3, 0], idx[B - 1, K // 2] = F, -1, 1 << 40  # counted as latent 0 with a value of zero
    W = torch.randn(F, D, generator=g, device=DEV, dtype=dtype)
    v = torch.randn(B, K, generator=g, device=DEV).to(dtype)
    b = torch.randn(D, generator=g, device=DEV).to(dtype)
    t = torch.randn(B, D, generator=g, device=DEV).to(dtype)
    lib = _lib.load()
    sh = ctypes.byref(abi.shape_of(idx, W, v, b.dtype, t.dtype))
    small, large = lib.flexsae_fwd_workspace_bytes(sh), lib.flexsae_topk_fwd_workspace_bytes(sh)
    assert large >= small + 8 * B * K  # the shape is one of those walked in latent order
    flag = torch.zeros(1, dtype=torch.int32, device=DEV)
    loss, resid = _forward(large, idx, W, v, b, t, flag)
    assert flag.item() == _lib.FLAG_INDEX_RANGE
    loss2, resid2 = _forward(large, idx, W, v, b, t)
    assert torch.equal(loss, loss2) and torch.equal(resid, resid2)
    loss_given, resid_given = _forward(small, idx, W, v, b, t)
    # K + 2 roundings, each at most 2^-24 of the sum of the terms' magnitudes
    bad = (idx < 0) | (idx >= F)
    safe, vd = idx.masked_fill(bad, 0), v.double().masked_fill(bad, 0.0)
    exact = b.double() - t.double()
    size = b.double().abs() + t.double().abs()
    for k in range(K):
        term = W[safe[:, k]].double() * vd[:, k, None]
        exact += term
        size += term.abs()
    bound = (K + 2) * 2.0 ** -24 * size
    assert ((resid.double() - exact).abs() <= bound).all()
    assert ((resid_given.double() - exact).abs() <= bound).all()
    # the loss adds the squares in double and rounds once: it is that of its own residual
    for lo, re in ((loss, resid), (loss_given, resid_given)):
        assert abs(lo.item() / re.double().square().mean().item() - 1) < 2.0 ** -23


def test_infinite_weights_stay_out_of_other_steps():
    """A last group of steps that is not full re-reads a row without adding it: no 0 * inf."""
    B, K, F, D = 600, 129, 16384, 1024
    g = torch.Generator(device=DEV).manual_seed(3)
    idx = torch.randint(0, F - 1, (B, K), generator=g, device=DEV)
    idx[5, 7] = F - 1  # the last of its row in latent order
    W = torch.randn(F, D, generator=g, device=DEV)
    W[F - 1] = float("inf")
    v = torch.rand(B, K, generator=g, device=DEV) + 0.5
    b, t = torch.randn(D, generator=g, device=DEV), torch.randn(B, D, generator=g, device=DEV)
    sh = ctypes.byref(abi.shape_of(idx, W, v, b.dtype, t.dtype))
    _, resid = _forward(_lib.load().flexsae_topk_fwd_workspace_bytes(sh), idx, W, v, b, t)
    assert torch.isposinf(resid[5]).all()
    keep = torch.arange(B, device=DEV) != 5
    assert torch.isfinite(resid[keep]).all()


@pytest.mark.parametrize("shape,dtype,pays", [
    ((4096, 128, 65536, 2304), torch.bfloat16, True), ((4096, 256, 262144, 2304), torch.bfloat16, True),
    ((4096, 64, 131072, 2304), torch.bfloat16, True),
    ((8192, 192, 262144, 1024), torch.bfloat16, True), ((1024, 256, 65536, 1024), torch.bfloat16, False),
    ((1024, 128, 131072, 2304), torch.bfloat16, False), ((2048, 256, 262144, 4096), torch.float16, True),
    ((2048, 256, 131072, 1024), torch.float32, True), ((2048, 64, 65536, 1024), torch.float32, False),
    ((2048, 96, 65536, 1024), torch.float32, True), ((1024, 192, 32768, 1152), torch.float32, False),
    ((2048, 192, 524288, 1024), torch.float32, False),
    ((4096, 64, 65536, 2304), torch.bfloat16, True), ((8041, 128, 524288, 512), torch.float16, False), ((4096, 512, (1 << 20) - 1, 2304), torch.bfloat16, True),
    ((300, 128, 65536, 2304), torch.bfloat16, False)], ids=str)
def test_which_shapes_are_walked_in_latent_order(shape, dtype, pays):
    lib = _lib.load()
    sh = ctypes.byref(_lib.Shape(*shape, *[abi.DT[dtype]] * 4))
    small, large = lib.flexsae_fwd_workspace_bytes(sh), lib.flexsae_topk_fwd_workspace_bytes(sh)
    assert lib.flexsae_topk_fwd_best_workspace_bytes(sh) == (large if pays else small)
    assert (large > small) == (shape[0] >= 512)


def test_more_latents_than_seventeen_bits():
    """Keys of twenty latent bits over nine position bits: the last latents come last."""
    B, K, F, D = 512, 500, (1 << 20) - 1, 160
    g = torch.Generator(device=DEV).manual_seed(9)
    idx = torch.randint(F - 4000, F, (B, K), generator=g, device=DEV)
    W = torch.zeros(F, D, device=DEV)
    W[F - 4000:] = torch.randn(4000, D, generator=g, device=DEV)
    v = torch.randn(B, K, generator=g, device=DEV)
    b, t = torch.randn(D, generator=g, device=DEV), torch.randn(B, D, generator=g, device=DEV)
    sh = ctypes.byref(abi.shape_of(idx, W, v, b.dtype, t.dtype))
    large = _lib.load().flexsae_topk_fwd_workspace_bytes(sh)
    assert large >= 8 * B * K
    _, resid = _forward(large, idx, W, v, b, t)
    at, order = torch.sort(idx, dim=1, stable=True)
    want = (b - t).double()
    size = b.double().abs() + t.double().abs()
    for k in range(K):
        term = W[at[:, k]].double() * v.gather(1, order[:, k:k + 1]).double()
        want += term
        size += term.abs()
    assert ((resid.double() - want).abs() <= (K + 2) * 2.0 ** -24 * size).all()
