"""Ordinary eager calls go past the dispatcher: the same bits as through the ops, and the ops wherever something has to see
them (modes, transforms, a graph of the backward)."""
import contextlib
import ctypes

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

import flexsae_amd as flex
from flexsae_amd import _lib, ops
from tests import abi
from tests.helpers import make_inputs

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
LOSS = {"hier": flex.triton_hierarchical_sae_loss, "topk": flex.triton_topk_sae_loss}


class _Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.ops = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.ops.append(str(func))
        return func(*args, **(kwargs or {}))


def _step(loss, args, upstream, needs=(True, True, True), seen=None):
    idx, W, v, b, t = args
    leaves = [x.clone().requires_grad_(n) for x, n in zip((W, v, b), needs)]
    out = LOSS[loss](idx, *leaves, t)
    (out * upstream).backward()
    return [out.detach()] + [x.grad for x in leaves]


@pytest.mark.parametrize("loss,fused", [("topk", True), ("hier", True), ("hier", False)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("B,K,F,D", [(7, 9, 40, 132), (64, 32, 300, 256), (5, 3, 11, 35)])
def test_same_bits_as_through_the_ops(loss, fused, dtype, B, K, F, D):
    print("[case]", loss, fused, dtype, B, K, F, D, flush=True)
    args = [x.to(DEV) for x in make_inputs(B, K, F, D, dtype, seed=B + D)]
    flex.set_fused_training(fused)
    try:
        for upstream in (1.0, 3.25):
            for needs in ((True, True, True), (False, True, True), (True, False, False)):
                with _Seen() as seen:
                    want = _step(loss, args, upstream, needs)
                assert any("flexsae_amd" in o for o in seen.ops)
                got = _step(loss, args, upstream, needs)
                for x, y in zip(got[1:], want[1:]):
                    assert (x is None and y is None) or torch.equal(x, y)
                assert torch.equal(got[0], want[0])
        with torch.no_grad():
            quiet = LOSS[loss](*args)
            with _Seen() as seen:
                assert torch.equal(quiet, LOSS[loss](*args))
            assert any("flexsae_amd" in o for o in seen.ops) and not quiet.requires_grad
    finally:
        flex.set_fused_training(True)


@pytest.mark.parametrize("loss", ["topk", "hier"])
def test_graphs_hooks_and_transforms(loss):
    args = [x.to(DEV) for x in make_inputs(16, 8, 60, 128, seed=4)]
    idx, W, v, b, t = args
    want = _step(loss, args, 2.0)
    # twice through a retained graph, and with a graph of the backward
    leaves = [x.clone().requires_grad_() for x in (W, v, b)]
    out = LOSS[loss](idx, *leaves, t) * 2.0
    for kw in ({"retain_graph": True}, {"retain_graph": True}, {"create_graph": True}):
        for x, y in zip(torch.autograd.grad(out, leaves, **kw), want[1:]):
            assert torch.equal(x.detach(), y)
    # what is saved passes the hooks: as many tensors as the op saves, and the gradients are those of what they give back
    counts = []
    for mode in (None, _Seen()):
        packed = []
        leaves = [x.clone().requires_grad_() for x in (W, v, b)]
        with torch.autograd.graph.saved_tensors_hooks(lambda x: packed.append(1) or x.cpu(), lambda x: x.to(DEV)):
            if mode is None:
                out = LOSS[loss](idx, *leaves, t)
            else:
                with mode:
                    out = LOSS[loss](idx, *leaves, t)
        (out * 2.0).backward()
        counts.append(len(packed))
        for x, y in zip(leaves, want[1:]):
            assert torch.equal(x.grad, y)
    assert counts[0] == counts[1]
    # a weight changed between forward and backward is refused
    leaves = [x.clone().requires_grad_() for x in (W, v, b)]
    out = LOSS[loss](idx, *leaves, t)
    with torch.no_grad():
        leaves[0].add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.backward()
    # functional transforms are the ops' business, which refuse them
    with pytest.raises(RuntimeError, match="functorch transforms"):
        torch.func.grad(lambda w: LOSS[loss](idx, w, v, b, t) * 2.0)(W)


@pytest.mark.parametrize("loss,fused,dtype,size", [
    ("topk", True, torch.float32, (16, 8, 60, 128)), ("hier", False, torch.bfloat16, (16, 8, 60, 128)),
    ("hier", True, torch.float16, (16, 8, 60, 128)), ("hier", True, torch.float16, (16, 8, 200, 256))])
@pytest.mark.parametrize("late", [False, True])
def test_the_surroundings_of_the_backward_count(loss, fused, dtype, size, late, monkeypatch):
    """A backward over batched upstream gradients, and one under a mode that its forward did not see, go through the ops."""
    idx, W, v, b, t = (x.to(DEV) for x in make_inputs(*size, dtype, seed=6))
    monkeypatch.setattr(ops, "_late_step", lambda *_: late)
    flex.set_fused_training(fused)
    try:
        leaves = [x.clone().requires_grad_() for x in (W, v, b)]
        out = LOSS[loss](idx, *leaves, t)
        ups = torch.tensor([1.0, 2.0, -0.5], device=DEV)
        want = [torch.autograd.grad(out, leaves, u, retain_graph=True) for u in ups]
        got = torch.autograd.grad(out, leaves, ups, retain_graph=True, is_grads_batched=True)
        for i, grads in enumerate(want):
            assert all(torch.equal(x, y[i]) for x, y in zip(grads, got))
        with _Seen() as seen:
            again = torch.autograd.grad(out, leaves, ups[1])
        assert any("flexsae_amd" in o for o in seen.ops)
        assert all(torch.equal(x, y) for x, y in zip(again, want[1]))
    finally:
        flex.set_fused_training(True)


def _transposed(x):  # the same values in another order in memory
    return x.t().contiguous().t() if x.dim() == 2 else x.repeat_interleave(2)[::2]


def _odd(x):  # ... behind one element of another buffer
    return x.new_empty(x.numel() + 1)[1:].view_as(x).copy_(x)


@pytest.mark.parametrize("loss,fused,dtype,late", [
    ("topk", True, torch.float32, False), ("topk", True, torch.bfloat16, False), ("hier", False, torch.bfloat16, False),
    ("hier", True, torch.bfloat16, False), ("hier", True, torch.float16, True)])
@pytest.mark.parametrize("lists", [False, True])
def test_saved_tensors_are_what_hooks_hand_back(loss, fused, dtype, late, lists, monkeypatch):
    """Of another layout or alignment: the same gradients.  On the host, or of another shape: refused before any launch."""
    idx, W, v, b, t = (x.to(DEV) for x in make_inputs(16, 8, 60, 128, dtype, seed=7))
    monkeypatch.setattr(ops, "_late_step", lambda *_: late)
    flex.set_fused_training(fused)

    def grads(unpack):
        leaves = [x.clone().requires_grad_() for x in (W, v, b)]
        with torch.autograd.graph.saved_tensors_hooks(lambda x: x, unpack):
            out = LOSS[loss](idx, *leaves, t)
        with flex.shared_pair_list() if lists else contextlib.nullcontext():
            return torch.autograd.grad(out * 2.0, leaves)

    try:
        want = grads(lambda x: x)
        for other in (_transposed, _odd):
            assert all(torch.equal(x, y) for x, y in zip(grads(other), want))
        for other in (lambda x: x.cpu(), lambda x: x[:, :-1] if x.dim() == 2 and x.is_floating_point() else x):
            with pytest.raises((RuntimeError, ValueError)):
                grads(other)
    finally:
        flex.set_fused_training(True)


def test_the_fused_update_marks_the_weight():
    idx, W, v, b, t = (x.to(DEV) for x in make_inputs(16, 8, 60, 128, seed=4))
    W2 = W.clone()
    before = W._version
    got = flex.hierarchical_sae_sgd_step(idx, W, v, b, t, 0.5)
    assert W._version > before
    with _Seen():
        want = flex.hierarchical_sae_sgd_step(idx, W2, v, b, t, 0.5)
    assert torch.equal(W, W2) and all(torch.equal(x, y) for x, y in zip(got, want))


@pytest.mark.parametrize("shared", [False, True])
def test_a_refused_update_leaves_the_weight_as_it_was(shared):
    """Rows that the update does not take: the weight keeps its values and its version, and a graph that saved it its backward."""
    idx, W, v, b, t = (x.to(DEV) for x in make_inputs(16, 8, 60, 132, torch.bfloat16, seed=4))
    before, version = W.clone(), W._version
    vals = v.clone().requires_grad_()
    loss = flex.triton_topk_sae_loss(idx, W, vals, b, t)
    with flex.shared_pair_list() if shared else contextlib.nullcontext():
        with pytest.raises(_lib.FlexSAELibraryError):
            flex.hierarchical_sae_sgd_step(idx, W, v, b, t, 0.5)
    assert W._version == version and torch.equal(W, before)
    loss.backward()


def test_finish_grads_checks_its_arguments():
    fn = _lib.load().flexsae_finish_grads
    x = torch.zeros(64, device=DEV)
    p = abi.ptr(x)
    odd = ctypes.c_void_p(x.data_ptr() + 4)
    none = ctypes.c_void_p(0)
    assert fn(none, 0, none, 0, 0, none, 0, none, 0, none, 0, none, 0, none, abi.stream()) == 0
    assert fn(none, 0, p, 0, 4, none, 0, none, 0, none, 0, none, 0, none, abi.stream()) == _lib.ERR_INVALID_ARGUMENT
    assert fn(p, 1, p, 2, 4, none, 0, none, 0, none, 0, none, 0, none, abi.stream()) == _lib.ERR_INVALID_ARGUMENT
    assert fn(p, 1, p, 0, 4, none, 0, none, 0, none, 0, none, 0, none, abi.stream()) == _lib.ERR_INVALID_ARGUMENT  # in place
    assert fn(odd, 0, p, 0, 4, none, 0, none, 0, none, 0, none, 0, none, abi.stream()) == _lib.ERR_ALIGNMENT
    assert fn(p, 7, p, 0, 4, none, 0, none, 0, none, 0, none, 0, none, abi.stream()) == _lib.ERR_INVALID_ARGUMENT


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("through_ops", [False, True])
def test_batched_upstream_gradients_of_the_fused_step(dtype, through_ops):
    """Each gets a weight gradient of its own, and the step's buffer stays for the backward after them: the same with a graph
    of the backward."""
    idx, W, v, b, t = (x.to(DEV) for x in make_inputs(16, 8, 60, 128, dtype, seed=6))
    leaves = [x.clone().requires_grad_() for x in (W, v, b)]
    if through_ops:
        with _Seen():
            out = flex.triton_hierarchical_sae_loss(idx, *leaves, t)
    else:
        out = flex.triton_hierarchical_sae_loss(idx, *leaves, t)
    ups = torch.tensor([1.0, 2.0, -0.5], device=DEV)
    got = torch.autograd.grad(out, leaves, ups, retain_graph=True, is_grads_batched=True)
    graph = torch.autograd.grad(out, leaves, ups[1], create_graph=True)
    with _Seen() as seen:
        want = [torch.autograd.grad(out, leaves, ups[0], retain_graph=True)]
    assert not any("train_sliced" in o for o in seen.ops)  # from the buffer, not computed again
    want += [torch.autograd.grad(out, leaves, u, retain_graph=True) for u in ups[1:]]
    for i, grads in enumerate(want):
        assert all(torch.equal(x, y[i]) for x, y in zip(grads, got))
    assert all(torch.equal(x, y) for x, y in zip(want[1], graph))


@pytest.mark.parametrize("loss", ["topk", "hier"])
def test_tensors_whose_memory_is_not_their_values(loss):
    """Negative views, which the dispatcher resolves, go through the ops; zero tensors are given memory."""
    idx, W, v, b, t = (x.to(DEV) for x in make_inputs(16, 8, 60, 128, seed=7))
    for i in range(1, 5):
        args = [idx, W, v, b, t]
        plain = list(args)
        plain[i] = -plain[i]
        args[i] = torch._neg_view(args[i])
        assert torch.equal(LOSS[loss](*args), LOSS[loss](*plain))
        args[i] = torch._efficientzerotensor(plain[i].shape, dtype=plain[i].dtype, device=DEV)
        plain[i] = torch.zeros_like(plain[i])
        assert torch.equal(LOSS[loss](*args), LOSS[loss](*plain))
    leaves = [x.clone().requires_grad_() for x in (W, v, b)]
    out = LOSS[loss](idx, *leaves, t)
    grads = torch.autograd.grad(out, leaves, torch._efficientzerotensor((), device=DEV), retain_graph=True)
    assert not any(x.any() for x in grads)
    grads = torch.autograd.grad(out, leaves, torch._neg_view(torch.ones((), device=DEV)), retain_graph=True)
    want = torch.autograd.grad(out, leaves, -torch.ones((), device=DEV))
    assert all(torch.equal(x, y) for x, y in zip(grads, want))
    W2 = W.clone()
    got = flex.hierarchical_sae_sgd_step(idx, W, torch._neg_view(v), b, t, 0.5)
    want = flex.hierarchical_sae_sgd_step(idx, W2, -v, b, t, 0.5)
    assert torch.equal(W, W2) and all(torch.equal(x, y) for x, y in zip(got, want))
    with pytest.raises((ValueError, RuntimeError)):
        flex.hierarchical_sae_sgd_step(idx, torch._efficientzerotensor(W.shape, device=DEV), v, b, t, 0.5)


@pytest.mark.parametrize("entry", ["topk_loss", "hier_loss", "hier_sliced"])
def test_what_the_extension_module_takes(entry):
    """Plain tensors of fitting shapes, contiguous or not; the rest it leaves to the ops, which see it or say what is wrong."""
    args = [x.to(DEV) for x in make_inputs(16, 8, 60, 128, seed=8)]
    idx, W, v, b, t = args
    LOSS["topk"](*args)
    fn = getattr(ops._native(W), entry)
    more = {"topk_loss": (), "hier_loss": (128,), "hier_sliced": (True, 128, 0, 0, None, 0)}[entry]
    want = fn(*args, *more)
    assert torch.equal(want, LOSS["topk" if entry == "topk_loss" else "hier"](*args))
    strided = [x.repeat_interleave(2, -1)[..., ::2] for x in args]
    assert not strided[1].is_contiguous() and torch.equal(fn(*strided, *more), want)
    odd = W.new_empty(W.numel() + 1)[1:].view_as(W).copy_(W)
    assert odd.data_ptr() % 16 and torch.equal(fn(idx, odd, v, b, t, *more), want)

    class Sub(torch.Tensor):
        pass

    refused = [(idx, W.as_subclass(Sub), v, b, t), (idx, W, v, b, t.cpu()), (idx.int(), W, v, b, t), (idx, W.double(), v, b, t),
               (idx, W, v[:, :4], b, t), (idx, W, v, b[:64], t), (idx[:0], W, v[:0], b, t[:0]), (idx, W[0], v, b, t),
               (idx, torch._neg_view(W), v, b, t), (idx, torch._efficientzerotensor(W.shape, device=DEV), v, b, t)]
    for wrong in refused:
        assert fn(*wrong, *more) is None
    with _Seen():
        assert fn(*args, *more) is None
    with pytest.raises(TypeError):
        fn(*args)[0] if more else fn(*args, 1)
    seen = []
    torch.func.vmap(lambda x: seen.append(fn(idx, W, x, b, t, *more)) or x)(torch.stack([v, v]))
    assert seen == [None]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("entry", ["hier_sliced", "hier_late", "hier_sgd"])
def test_what_the_steps_of_the_extension_module_take(entry, dtype):
    """The step leaves its measurement, tagged, in pinned memory; a call that it does not take leaves the words and the weight."""
    print("[case]", entry, dtype, flush=True)
    B, K, F, D = 100, 8, 900, 128
    idx, W, v, b, t = make_inputs(B, K, F, D, dtype, seed=8)
    idx[:, 0] = 3  # a latent with more than 64 pairs
    counts = torch.bincount(idx.flatten(), minlength=F)
    long = counts[counts > 64]
    want = [long.numel(), int(((long + 63) // 64).sum()), int((counts == 0).sum()), 77]
    idx, W, v, b, t = (x.to(DEV) for x in (idx, W, v, b, t))
    LOSS["topk"](idx, W, v, b, t)
    fn = getattr(ops._native(W), entry)
    words = torch.full((4,), -5, dtype=torch.int32, pin_memory=True)
    first = torch.full((), 0.5, device=DEV) if entry == "hier_sgd" else True
    more = (first, 128, 0, 0, words, 77)

    def taken(args):
        words.fill_(-5)
        got = fn(*args, *more)
        if got is not None and entry == "hier_late":
            torch.cuda.synchronize()
            assert words.tolist() == [-5] * 4  # (the step comes with the backward)
            torch.autograd.grad(got, args[1])
        torch.cuda.synchronize()
        assert words.tolist() == ([-5] * 4 if got is None else want)
        return got is not None

    def fresh(x=W):
        return x.clone().requires_grad_(entry != "hier_sgd")

    old = fresh()
    assert taken((idx, old, v, b, t))
    changed = not torch.equal(old.detach(), W)
    assert changed == (entry == "hier_sgd")

    class Sub(torch.Tensor):
        pass

    weight = fresh()
    refused = [(idx, W.as_subclass(Sub), v, b, t), (idx, weight, v, b, t.cpu()), (idx.int(), weight, v, b, t),
               (idx, weight.double(), v, b, t), (idx, weight, v[:, :4], b, t), (idx, weight, v, b[:64], t),
               (idx[:0], weight, v[:0], b, t[:0]), (idx, torch._neg_view(W), v, b, t)]
    strided = W.repeat_interleave(2, -1)[..., ::2]
    odd = W.new_empty(W.numel() + 1)[1:].view_as(W).copy_(W)
    narrow = (idx, W[:, :126].contiguous(), v, b[:126], t[:, :126])
    deep = (idx.repeat(1, 33), W, v.repeat(1, 33), b, t)  # 264 steps
    if entry == "hier_sgd":  # in place: whole rows on whole vectors
        refused += [(idx, strided, v, b, t), (idx, odd, v, b, t), narrow, deep]
    else:
        for w in (strided, odd):
            assert taken((idx, w.detach().requires_grad_(), v, b, t))
    for args in refused:
        assert not taken(args)
    with _Seen():
        assert not taken((idx, weight, v, b, t))
    assert torch.equal(weight.detach(), W) and weight._version == 0
    with pytest.raises(TypeError):
        fn(idx, W, v, b, t)


@pytest.mark.parametrize("sgd", [False, True])
def test_a_call_that_the_module_left_to_the_ops_does_not_end_the_measurement(sgd):
    B, K, F, D = 24, 8, 613, 132
    idx, W, v, b, t = (x.to(DEV) for x in make_inputs(B, K, F, D, seed=9))

    def step():
        w = W.clone().requires_grad_(not sgd)
        if sgd:
            flex.hierarchical_sae_sgd_step(idx, w, v, b, t, 0.5)
        else:
            flex.triton_hierarchical_sae_loss(idx, w, v, b, t).backward()
        torch.cuda.synchronize()

    key = ops._hot_key(DEV, B, K, F, D, torch.float32)
    for _ in range(2):
        with _Seen():
            step()
        step()
        st = ops._hot_auto[key]
        assert st["words"][3] == st["asked"] != 0
        st["words"][2] = F  # (as if no latent had a pair)
        with _Seen():
            step()
        step()
        assert st["words"][3] == st["asked"] and st["words"][2] == F - idx.unique().numel()


@pytest.mark.parametrize("loss", ["topk", "hier"])
def test_other_threads_and_streams(loss):
    """Forward and backward on a stream and a thread of their own, several at once: each the same bits."""
    import threading

    args = [x.to(DEV) for x in make_inputs(64, 16, 300, 256, torch.bfloat16, seed=9)]
    want = _step(loss, args, 2.0)
    got = [None] * 4

    def work(i):
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.default_stream())
        with torch.cuda.stream(stream):
            for _ in range(5):
                got[i] = _step(loss, args, 2.0)
        stream.synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    torch.cuda.synchronize()
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    torch.cuda.synchronize()
    for grads in got:
        assert all(torch.equal(x, y) for x, y in zip(grads, want))
