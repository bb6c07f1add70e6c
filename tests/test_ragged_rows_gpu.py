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
def test_ragged_rows(F, dtype, K, D, monkeypatch):
    print("[case]", F, dtype, K, D, flush=True)
    args = make_inputs(150, K, F, D, dtype, seed=K + D)
    args[0][:, 0] = 3
    idx, W, v, b, t = (x.to(DEV) for x in args)
    assert flex.ops._train_ragged(W, K)
    monkeypatch.setattr(flex.ops, "_ragged_pays", lambda *_: True)  # (whatever is faster)
    monkeypatch.setattr(flex.ops, "_step_pays", lambda *_: True)
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


def test_which_ragged_rows_take_the_training_step():
    def pays(dtype, B, K, F, D=390):
        return flex.ops._ragged_pays(torch.empty(F, D, dtype=dtype, device="meta", requires_grad=True), B, K)

    for dtype in (torch.float32, torch.bfloat16):
        assert all(pays(dtype, 64, K, 4000) for K in (1, 128, 256)) and not any(pays(dtype, 64, K, 4000) for K in (129, 255))
    assert pays(torch.float16, 601, 10, 1000) and not pays(torch.float16, 600, 10, 1000)
    assert not pays(torch.float16, 6000, 200, 1000)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("K,D", [(128, 132), (129, 132), (129, 130), (255, 64), (256, 64)])
@pytest.mark.parametrize("needs", [(True, True, True), (False, True, True)])
def test_steps_between_the_kernels(needs, K, D, dtype, monkeypatch):
    """129 to 255 steps go by forward and sweep where the weight takes a gradient: the training step's gradients."""
    print("[case]", needs, K, D, dtype, flush=True)
    idx, W, v, b, t = (x.to(DEV) for x in make_inputs(70, K, 500, D, dtype, seed=K + D))
    monkeypatch.setattr(flex.ops, "_one_gather_pays", lambda *_: False)  # (whatever is faster)
    grads = []
    for forced in (False, True):
        if forced:
            monkeypatch.setattr(flex.ops, "_step_pays", lambda *_: True)
            monkeypatch.setattr(flex.ops, "_ragged_pays", lambda *_: True)
        leaves = [x.clone().requires_grad_(n) for x, n in zip((W, v, b), needs)]
        assert flex.ops._step_pays(leaves[0], K) == (forced or K in (128, 256) or not needs[0])
        loss = flex.triton_hierarchical_sae_loss(idx, *leaves, t)
        loss.backward()
        grads.append([loss.detach()] + [x.grad for x in leaves])
    assert rel_err(grads[0][0].cpu(), grads[1][0].cpu()) < 1e-6  # other partial sums, all beyond a column in double
    for x, y in zip(grads[0][1:], grads[1][1:]):
        assert (x is None and y is None) or torch.equal(x, y)


def test_which_steps_between_the_kernels_gather_once():
    def pays(dtype, B, K, F, D):
        return flex.ops._one_gather_pays(torch.empty(F, D, dtype=dtype, device="meta", requires_grad=True), B, K)

    bf16, fp16, fp32 = torch.bfloat16, torch.float16, torch.float32
    assert pays(bf16, 512, 160, 16384, 512) and pays(fp16, 192, 160, 8192, 512) and not pays(fp32, 512, 160, 16384, 512)
    assert not pays(bf16, 2048, 160, 65536, 1024) and not pays(fp16, 224, 168, 17816, 1160) and not pays(bf16, 64, 160, 8192, 512)
    assert pays(bf16, 412, 150, 478747, 4944) and pays(fp32, 488, 254, 407482, 1632) and pays(fp16, 182, 200, 221872, 5240)
    assert not pays(bf16, 2734, 168, 233249, 1768) and not pays(fp32, 200, 150, 202656, 736) and not pays(fp16, 531, 168, 85672, 7264)


@pytest.mark.parametrize("D", [128, 130])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
def test_frozen_weights_gather_once(dtype, D):
    """129 to 255 steps without a weight gradient take the training step, whether or not vectors of four divide the rows."""
    W = torch.empty(500, D, dtype=dtype, device="meta")
    assert flex.ops._step_pays(W, 150) and flex.ops._ragged_pays(W, 70, 150)
    W.requires_grad_()
    assert not flex.ops._step_pays(W, 150) and not flex.ops._ragged_pays(W, 70, 150)


@pytest.mark.parametrize("D", [65, 129, 321, 705])
def test_odd_bf16_rows_give_the_same_bits_in_any_slices(D):
    """Rows whose whole width is no whole number of pieces: cut into slices of whole pieces."""
    print("[case] odd rows in slices", D, flush=True)
    g = torch.Generator(device=DEV).manual_seed(D)
    B, K, F = 70, 20, (6 << 20) // D + 1  # (smaller gradients stay in one slice)
    idx = torch.randint(0, F, (B, K), generator=g, device=DEV)
    got = []
    for least, scratch in ((None, None), (64, 1)):
        W, v, b = (torch.randn(*s, generator=g.manual_seed(7), device=DEV).to(torch.bfloat16).requires_grad_()
                   for s in ((F, D), (B, K), (D,)))
        t = torch.randn(B, D, generator=g, device=DEV).to(torch.bfloat16)
        try:
            flex.set_hier_scratch_bytes(scratch)
            if least:
                flex.set_hier_min_slice_cols(least)
            flex.triton_hierarchical_sae_loss(idx, W, v, b, t).backward()
        finally:
            flex.set_hier_scratch_bytes(None)
            flex.set_hier_min_slice_cols(None)
        got.append((W.grad, v.grad, b.grad))
    assert all(torch.equal(x, y) for x, y in zip(*got))
    W, v, b, t = (x.detach().double().cpu() for x in (W, v, b, t))
    W.requires_grad_()
    flex.hierarchical_sae_loss(idx.cpu(), W, v, b, t).backward()
    assert (got[0][0].double().cpu() - W.grad).norm() < 1e-2 * W.grad.norm()
