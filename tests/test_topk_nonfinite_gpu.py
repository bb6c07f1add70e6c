"""TopK backward with an infinite residual: what of it reaches the weight gradient's other columns."""
import pytest
import torch

from tests import abi

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


# rows of odd length, padded to whole vectors and not; even ones
@pytest.mark.parametrize("D", [63, 65, 129, 513, 1025, 64, 130, 516, 1032])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_infinite_residual(value, dtype, D):
    """Only the gradient's own column, and in rows of even length with bf16 weights and values the other one of its pair of
    columns (the packed product multiplies that by zero): not the rest of the row, and no other latent."""
    print("[case]", value, dtype, D, flush=True)
    B, K, F = 6, 4, 40
    g = torch.Generator().manual_seed(D)
    W, v = torch.randn(F, D, generator=g).to(dtype), (torch.rand(B, K, generator=g) + 0.5).to(dtype)
    idx = torch.arange(B * K).view(B, K)
    resid = torch.randn(B, D, generator=g)
    col = 21
    resid[2, col] = value
    rc, dW, dv, db = abi.topk_backward(idx.to(DEV), W.to(DEV), v.to(DEV), resid.to(DEV), 1.0)
    torch.cuda.synchronize()
    assert rc == 0
    hit = torch.zeros(F, D, dtype=torch.bool)
    hit[idx[2], col] = True
    pair = torch.zeros_like(hit)
    if dtype == torch.bfloat16 and D % 2 == 0:
        pair[idx[2], col - 1] = True
    bad = ~torch.isfinite(dW.cpu().float())
    assert bool(bad[hit].all()) and not bool((bad & ~hit & ~pair).any())
    assert not torch.isfinite(dv.cpu()[2]).any() and torch.isfinite(dv.cpu()[[0, 1, 3, 4, 5]]).all()
    assert torch.equal(~torch.isfinite(db.cpu()), hit[idx[2, 0]])
