"""TopK backward, groups of neighbouring latents per wavefront: latents without pairs, with the most a group takes, and
with more than that (reduced apart) side by side; groups cut short by F, streams of more than 64 pairs; against float64."""
import pytest
import torch

from flexsae_amd import _lib
from tests import abi

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("D", [8, 64, 65, 77, 130, 260, 515, 520, 1028, 1030])
@pytest.mark.parametrize("dtype,vals_dtype,dw_dtype", [
    (torch.float32, torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16, torch.bfloat16),
    (torch.bfloat16, torch.float32, torch.float32), (torch.float16, torch.float16, torch.float16)], ids=str)
@pytest.mark.parametrize("counts", [
    [0, 64, 65, 1, 0, 0, 130, 64, 64, 64, 64, 64, 64, 64, 64, 64, 0, 0, 0, 0, 0, 0, 0, 0, 3],
    [5], [0, 0, 7, 66, 0, 8, 9, 1, 0], [66] * 8 + [2] * 33 + [0] * 7], ids=["edges", "one", "short", "runs"])
@pytest.mark.parametrize("flags", [0, _lib.TOPK_BWD_AS_LARGE], ids=["as_small", "whole_groups"])
def test_groups(flags, counts, dtype, vals_dtype, dw_dtype, D):
    print("[case]", flags, counts[:4], dtype, vals_dtype, dw_dtype, D, flush=True)
    F = len(counts)
    K = 4
    pairs = torch.cat([torch.full((c,), f, dtype=torch.long) for f, c in enumerate(counts)])
    B = -(-len(pairs) // K)
    g = torch.Generator().manual_seed(len(pairs) + D)
    pairs = torch.cat([pairs, torch.full((B * K - len(pairs),), F - 1)])
    idx = pairs[torch.randperm(B * K, generator=g)].view(B, K)
    W = torch.randn(F, D, generator=g).to(dtype)
    v = torch.randn(B, K, generator=g).to(vals_dtype)
    resid = torch.randn(B, D, generator=g)
    grad = 1.5
    rc, dW, dv, db = abi.topk_backward(idx.to(DEV), W.to(DEV), v.to(DEV), resid.to(DEV), grad, dw_dtype=dw_dtype,
                                       flags=flags)
    torch.cuda.synchronize()
    assert rc == 0
    gathered = resid.to(torch.bfloat16) if dtype == torch.bfloat16 else resid  # what the call gathers
    scale = grad * 2.0 / (B * D)
    rows = gathered.double().repeat_interleave(K, 0)
    flat = idx.reshape(-1)
    terms = v.double().reshape(-1, 1) * scale * rows
    exact = torch.zeros(F, D, dtype=torch.double).index_add_(0, flat, terms)
    size = torch.zeros(F, D, dtype=torch.double).index_add_(0, flat, terms.abs())
    # a rounding per pair and a few for the scale and the chunks' sums, then the one to dW's type
    n = torch.tensor(counts).double().max() + K + 8
    half_ulp = {  # of numbers of 8 and 11 significant bits
        torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dw_dtype]
    floor = 2.0 ** -25 if dw_dtype == torch.float16 else 0.0  # half of fp16's smallest number
    assert ((dW.cpu().double() - exact).abs() <= n * 2.0 ** -24 * size + 1.001 * half_ulp * exact.abs() + floor).all()
    prods = rows * W.double()[flat] * scale
    bound = (D + 8) * 2.0 ** -24 * prods.abs().sum(1)
    assert ((dv.cpu().double().reshape(-1) - prods.sum(1)).abs() <= bound).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("B,K,F,D", [(40, 30, 100, 264), (500, 4, 1001, 520), (300, 5, 12293, 72), (2048, 52, 8195, 264),
                                     (10, 4, 4097, 264)])
def test_groups_of_any_size_give_the_same_bits(B, K, F, D, dtype):
    """One, two, four or eight latents per wavefront, by size: as with whole groups."""
    print("[case]", B, K, F, D, dtype, flush=True)
    g = torch.Generator(device=DEV).manual_seed(B + D)
    idx = torch.randint(0, F, (B, K), generator=g, device=DEV)
    W = torch.randn(F, D, generator=g, device=DEV).to(dtype)
    v = torch.randn(B, K, generator=g, device=DEV).to(dtype)
    resid = torch.randn(B, D, generator=g, device=DEV)
    small, large = (abi.topk_backward(idx, W, v, resid, 1.5, flags=f) for f in (0, _lib.TOPK_BWD_AS_LARGE))
    torch.cuda.synchronize()
    assert small[0] == 0 and large[0] == 0
    assert all(torch.equal(x, y) for x, y in zip(small[1:], large[1:]))


@pytest.mark.parametrize("K", [20, 40])
@pytest.mark.parametrize("D", [1028, 1284, 1524])
def test_last_tile_of_few_columns(D, K):
    """Five and six tiles of 256 columns, the last one of four or of most: apart from the others or in step with them, by the
    number of tiles, its columns and the pairs per latent."""
    print("[case]", D, K, flush=True)
    B, F = 64, 1001
    g = torch.Generator().manual_seed(D + K)
    idx = torch.randint(0, F, (B, K), generator=g)
    W, v, resid = torch.randn(F, D, generator=g), torch.randn(B, K, generator=g), torch.randn(B, D, generator=g)
    rc, dW, dv, db = abi.topk_backward(idx.to(DEV), W.to(DEV), v.to(DEV), resid.to(DEV), 1.5)
    torch.cuda.synchronize()
    assert rc == 0
    scale = 1.5 * 2.0 / (B * D)
    rows, flat = resid.double().repeat_interleave(K, 0), idx.reshape(-1)
    terms = v.double().reshape(-1, 1) * scale * rows
    exact, size = (torch.zeros(F, D, dtype=torch.double).index_add_(0, flat, t) for t in (terms, terms.abs()))
    n = torch.bincount(flat, minlength=F).max() + 8  # a rounding per pair and a few for the scale
    assert ((dW.cpu().double() - exact).abs() <= n * 2.0 ** -24 * size).all()
    prods = rows * W.double()[flat] * scale
    assert ((dv.cpu().double().reshape(-1) - prods.sum(1)).abs() <= (D + 8) * 2.0 ** -24 * prods.abs().sum(1)).all()
