"""The training step where its wavefronts take the tiles of a row one after the other (few batch rows) and where they take the
rows of a tile: rows on either side of the line, a last tile of few columns, one tile and several, slices."""
import pytest
import torch

import flexsae_amd as flex
from tests.helpers import make_inputs

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("scratch", [None, 1])
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.bfloat16, 1e-2), (torch.float16, 1e-3)], ids=str)
@pytest.mark.parametrize("B,K,F,D", [(2047, 3, 700, 260), (2048, 3, 700, 260), (2047, 66, 90, 132), (1, 2, 5, 1028), (3, 70, 80, 100)])
def test_either_order(B, K, F, D, dtype, tol, scratch):
    print("[case]", B, K, F, D, dtype, scratch, flush=True)
    idx, W, v, b, t = (x.to(DEV) for x in make_inputs(B, K, F, D, dtype, seed=B + K))
    flex.set_hier_scratch_bytes(scratch)
    try:
        leaves = [x.clone().requires_grad_() for x in (W, v, b)]
        loss = flex.triton_hierarchical_sae_loss(idx, *leaves, t)
        (loss * B).backward()
    finally:
        flex.set_hier_scratch_bytes(None)
    wide = [x.double().requires_grad_() for x in (W, v, b)]
    rows = wide[0][idx] * wide[1][..., None]
    err = wide[2] + torch.cumsum(rows, 1) - t.double()[:, None]
    want = err.square().mean()
    (want * B).backward()
    assert abs(loss.item() - want.item()) <= 1e-5 * want.item()
    for x, y in zip(leaves, wide):
        assert (x.grad.double() - y.grad).norm() <= tol * y.grad.norm()
