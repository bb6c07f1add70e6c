"""dbias of the hierarchical step at the edges of its column sums: one block of rows or many, columns that no block of
32 (or of 256) divides, and the most rows that are summed in one launch."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 63, 65, 1025, 2048, 2049])
@pytest.mark.parametrize("D", [4, 20, 260, 1100])
def test_dbias_column_sums(B, D):
    import flexsae_amd as flex

    print(f"[case] hier end B={B} D={D}", flush=True)
    K, F = 6, 97
    g = torch.Generator().manual_seed(B * 7 + D)
    idx = torch.randint(0, F, (B, K), generator=g)
    vals = torch.randn(B, K, generator=g).abs()
    W, bias, target = (torch.randn(*s, generator=g) for s in ((F, D), (D,), (B, D)))
    Wd, vd, bd = (x.cuda().requires_grad_() for x in (W, vals, bias))
    loss = flex.triton_hierarchical_sae_loss(idx.cuda(), Wd, vd, bd, target.cuda())
    loss.backward()
    # the step's own definition in 64 bits: S[b] = coef * sum over the prefixes of (reconstruction - target)
    e = (bias - target).double()
    S = torch.zeros(B, D, dtype=torch.float64)
    size = torch.zeros(B, D, dtype=torch.float64)  # sum of the magnitudes that were added
    run = e.abs()
    for k in range(K):
        step = vals[:, k, None].double() * W[idx[:, k]].double()
        e, run = e + step, run + step.abs()
        S, size = S + e, size + run
    coef = 2.0 / (B * K * D)
    want, size = coef * S.sum(0), coef * size.sum(0)
    # every value passes through at most 2K + 3 roundings in its row, 64 in its chunk of rows, one per chunk
    roundings = 2 * K + 3 + 64 + (B + 63) // 64
    assert (bd.grad.double().cpu() - want).abs().le(roundings * 2.0 ** -24 * size).all()
