"""fp16 weights of few pairs per latent: the step in the backward, with the upstream gradient, gives the bits of the unit
gradient scaled and rounded afterwards."""
import ctypes

import pytest
import torch

import flexsae_amd as flex
from flexsae_amd import _lib, ops
from tests import abi
from tests.helpers import make_inputs, rel_err

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


# hot: the frequent latents' accumulators; slices of one tile, so that second steps ride in the next launch; empty latents
@pytest.mark.parametrize("B,K,F,D,hot,zipf", [
    (40, 16, 400, 256, False, None), (33, 7, 90, 1032, False, None), (40, 64, 2000, 512, False, 1.1), (300, 64, 5000, 640, True, 1.1),
    (200, 32, 4000, 1028, True, 1.3), (20, 200, 2000, 390, False, None), (64, 100, 1600, 1026, False, 1.2)], ids=str)
@pytest.mark.parametrize("upstream", [65536.0, 1.7e5])
def test_same_bits_as_the_scaled_unit_gradient(B, K, F, D, hot, zipf, upstream, monkeypatch):
    print("[case]", B, K, F, D, hot, zipf, upstream, flush=True)
    args = make_inputs(B, K, F, D, torch.float16, seed=B + K, zipf_s=zipf)
    if zipf and not hot:
        args[0][:, 0] = 5  # a latent in every row: reduced in chunks
    idx, W, v, b, t = (x.to(DEV) for x in args)
    monkeypatch.setattr(ops, "_ragged_pays", lambda *_: True)
    monkeypatch.setattr(ops, "_step_pays", lambda *_: True)
    monkeypatch.setattr(ops, "_late_step", lambda *_: True)  # (whatever the size)
    flex.set_hot_latents(hot)
    flex.set_hier_scratch_bytes(1)
    flex.set_hier_min_slice_cols(128)
    grads = []
    try:
        for late in (True, False):
            leaves = [x.clone().requires_grad_() for x in (W, v, b)]
            if late:
                loss = flex.triton_hierarchical_sae_loss(idx, *leaves, t)
            else:
                loss = ops.hier_train_sliced(idx, *leaves, t, True, hot, False)[0]
            (loss * upstream).backward()
            torch.cuda.synchronize()
            grads.append([loss.detach()] + [x.grad for x in leaves])
    finally:
        flex.set_hot_latents("auto")
        flex.set_hier_scratch_bytes(None)
        flex.set_hier_min_slice_cols(None)
    assert rel_err(grads[0][0].cpu(), grads[1][0].cpu()) < 1e-6
    for x, y in zip(grads[0][1:], grads[1][1:]):
        assert torch.equal(x, y)
    assert (grads[0][1] != 0).any()


def test_graph_of_the_backward_and_flags(monkeypatch):
    monkeypatch.setattr(ops, "_ragged_pays", lambda *_: True)
    monkeypatch.setattr(ops, "_step_pays", lambda *_: True)
    monkeypatch.setattr(ops, "_late_step", lambda *_: True)
    idx, W, v, b, t = (x.to(DEV) for x in make_inputs(16, 8, 60, 128, torch.float16, seed=4))
    leaves = [x.clone().requires_grad_() for x in (W, v, b)]
    loss = flex.triton_hierarchical_sae_loss(idx, *leaves, t) * 1024.0
    plain = torch.autograd.grad(loss, leaves, retain_graph=True)
    for x, y in zip(torch.autograd.grad(loss, leaves, create_graph=True), plain):
        assert torch.equal(x.detach(), y)
    sh = abi.shape_of(idx, W, v, b.dtype, t.dtype)
    lib = _lib.load()
    ws = torch.empty(lib.flexsae_hier_fwd_bwd_workspace_bytes(ctypes.byref(sh), 0), dtype=torch.uint8, device=DEV)
    out = [torch.empty(n, device=DEV) for n in (1, 60 * 128, 128, 128)]
    g = torch.ones(1, device=DEV)

    def call(g_ptr, flags):
        return lib.flexsae_hier_fwd_bwd_scaled(ctypes.byref(sh), *(abi.ptr(x) for x in (idx, W, v, b, t)), g_ptr,
                                               abi.ptr(out[0]), abi.ptr(out[1]), _lib.F32, abi.ptr(out[2]), abi.ptr(out[3]),
                                               abi.ptr(ws), ws.numel(), flags, None, abi.stream())

    assert call(None, 0) == _lib.ERR_INVALID_ARGUMENT
    for flag in (_lib.BWD_NO_DW, _lib.BWD_SWEEP_ONLY, _lib.BWD_REDUCE_ONLY, _lib.BWD_SKIP_EPILOGUE):
        assert call(abi.ptr(g), flag) == _lib.ERR_INVALID_ARGUMENT
    assert call(abi.ptr(g), 0) == 0
    torch.cuda.synchronize()


def test_which_shapes_take_it():
    def late(dtype, B, K, F, D):
        return ops._late_step(torch.empty(F, D, dtype=dtype, device="meta"), B, K)

    assert late(torch.float16, 4096, 32, 65536, 2304) and late(torch.float16, 4096, 64, 65536, 1536)
    assert not late(torch.float16, 4097, 64, 65536, 1536) and not late(torch.float16, 64, 32, 65536, 1535)
    assert not late(torch.bfloat16, 4096, 32, 65536, 2304) and not late(torch.float32, 4096, 32, 65536, 2304)


def test_a_captured_backward_leaves_no_measurement(monkeypatch):
    """The forward runs before the capture, the step inside it: no replay writes what the pair list says about its indices, which
    would pass for that of a later step."""
    monkeypatch.setattr(ops, "_late_step", lambda *_: True)
    B, K, F, D = 40, 16, 411, 256
    idx, W, v, b, t = (x.to(DEV) for x in make_inputs(B, K, F, D, torch.float16, seed=6))
    up = torch.tensor(2.0, device=DEV)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    leaves = [x.clone().requires_grad_() for x in (W, v, b)]
    with torch.cuda.stream(stream):
        want = torch.autograd.grad(flex.triton_hierarchical_sae_loss(idx, *leaves, t), leaves, up)
        torch.cuda.synchronize()
        st = ops._hot_auto[ops._hot_key(DEV, B, K, F, D, torch.float16)]
        assert st["words"][3] == st["asked"]
        loss = flex.triton_hierarchical_sae_loss(idx, *leaves, t)
        torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        got = torch.autograd.grad(loss, leaves, up)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(got, want))
        assert st["words"][3] == st["asked"] - 1
        st["pinned"][3] = 0  # (eager work between the replays)
        torch.zeros(8, device=DEV).add_(1)
        torch.cuda.synchronize()
        st["pinned"][3] = st["asked"] - 1
