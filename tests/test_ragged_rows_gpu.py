"""Training step on rows that no vector of four columns divides: the same gradients, bit for bit, as forward and sweep."""
import pytest
import torch

import flexsae_amd as flex
from flexsae_amd import _lib
from tests import abi
from tests.helpers import make_inputs, rel_err

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


# tiles with one pair of columns, full ones and one over; every number of steps a kernel is built for, full and not;
# latents in every row (long), in one row only, in none
@pytest.mark.parametrize("dtype,K,D", [
    (torch.bfloat16, 16, 2), (torch.bfloat16, 5, 130), (torch.bfloat16, 32, 258), (torch.bfloat16, 50, 1538),
    (torch.bfloat16, 64, 126), (torch.bfloat16, 128, 386), (torch.bfloat16, 130, 1030), (torch.bfloat16, 256, 254),
    (torch.float16, 31, 642), (torch.float16, 128, 262), (torch.float32, 16, 6), (torch.float32, 64, 258),
    (torch.float32, 65, 1), (torch.float32, 100, 63), (torch.float32, 128, 129), (torch.float32, 200, 1026),
    (torch.float32, 256, 321)], ids=str)
@pytest.mark.parametrize("F", [70, 4000])
def test_ragged_rows(F, dtype, K, D):
    print("[case]", F, dtype, K, D, flush=True)
    args = make_inputs(150, K, F, D, dtype, seed=K + D)
    args[0][:, 0] = 3
    idx, W, v, b, t = (x.to(DEV) for x in args)
    assert flex.ops._train_ragged(W, K)
    grads = []
    for fused in (True, False):
        leaves = [x.clone().requires_grad_() for x in (W, v, b)]
        flex.set_fused_training(fused)
        try:
            loss = flex.triton_hierarchical_sae_loss(idx, *leaves, t)
            loss.backward()
        finally:
            flex.set_fused_training(True)
        torch.cuda.synchronize()
        grads.append([loss.detach()] + [x.grad for x in leaves])
    assert rel_err(grads[0][0].cpu(), grads[1][0].cpu()) < 1e-6  # other partial sums, all beyond a column in double
    for x, y in zip(grads[0][1:], grads[1][1:]):
        assert torch.equal(x, y)


def test_ragged_rows_want_the_flag():
    idx, W, v, b, t = (x.to(DEV) for x in make_inputs(8, 8, 32, 6, seed=3))
    assert abi.hier_train(idx, W, v, b, t)[0] == _lib.ERR_UNSUPPORTED
    rc, loss, dW, dv, db = abi.hier_train(idx, W, v, b, t, flags=_lib.BWD_RAGGED_ROWS)
    torch.cuda.synchronize()
    assert rc == 0 and all(torch.isfinite(x).all() for x in (loss, dW, dv, db))
    # not deferred, and no odd columns where a lane holds two
    assert abi.hier_train(idx, W, v, b, t, slice_cols=1 << 20,
                          flags=_lib.BWD_RAGGED_ROWS | _lib.BWD_SWEEP_ONLY)[0] == _lib.ERR_UNSUPPORTED
    idx, W, v, b, t = (x.to(DEV) for x in make_inputs(8, 8, 32, 7, seed=3))
    assert abi.hier_train(idx, W, v, b, t, flags=_lib.BWD_RAGGED_ROWS)[0] == _lib.ERR_UNSUPPORTED
