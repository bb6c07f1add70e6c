"""Host-side logic of the python layer (no GPU): validation, public names, fake kernels, the
eager torch definitions, and that nothing in the package touches the oracle."""
import ctypes
import os
import re
import shutil
import weakref

import pytest
import torch

import flexsae_amd as flex
import oracle
from flexsae_amd import _lib, build, ops
from helpers import make_inputs

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_public_names_match_the_reference_package():
    # reference torch-ext/flex_sae/__init__.py:12-18
    for name in ("__kernel_metadata__", "topk_sae_loss", "triton_topk_sae_loss", "hierarchical_sae_loss",
                 "triton_hierarchical_sae_loss"):
        assert name in flex.__all__ and hasattr(flex, name)


@pytest.mark.parametrize("fn", [flex.triton_topk_sae_loss, flex.triton_hierarchical_sae_loss])
def test_fused_ops_fail_loudly_without_a_gpu_tensor(fn):
    args = make_inputs(4, 8, 16, 64)
    with pytest.raises(RuntimeError, match="AMD GPU only"):
        fn(*args)


def test_validation_errors():
    idx, W, v, b, t = make_inputs(4, 8, 16, 64)
    with pytest.raises(TypeError):
        ops._validate(idx.int(), W, v, b, t)
    with pytest.raises(TypeError):
        ops._validate(idx, W.double(), v, b, t)
    with pytest.raises(ValueError):
        ops._validate(idx, W, v[:, :4], b, t)
    with pytest.raises(ValueError):
        ops._validate(idx, W, v, b[:32], t)
    with pytest.raises(ValueError):
        ops._validate(idx[:0], W, v[:0], b, t[:0])
    with pytest.raises(ValueError):
        ops._validate(idx.flatten(), W, v, b, t)


@pytest.mark.parametrize("fn", [ops._topk_bwd_impl, ops._hier_bwd_impl])
def test_a_backward_refuses_saved_tensors_that_do_not_fit(fn, monkeypatch):
    """... before it asks for anything on the device."""
    monkeypatch.setattr(ops._lib, "load", lambda: None)
    idx, W, v, b, t = make_inputs(4, 8, 16, 64)
    for saved in ((idx, W, v, t), (idx, W, v[:, :7], t), (idx, W[:, :63], v, t), (idx, W, v, t.half()), (idx, W, v, t[0]),
                  (idx[:0], W, v[:0], t[:0])):
        with pytest.raises((RuntimeError, ValueError), match="AMD GPU only|shape mismatch|expected resid|empty"):
            fn(torch.ones(()), *saved)
    with pytest.raises(RuntimeError, match="a saved tensor is on cpu"):
        ops._finish_grads(None, W, None, v, v.dtype, b, b.dtype)


@pytest.mark.parametrize("mode,fn", [(oracle.TOPK, flex.topk_sae_loss), (oracle.HIER, flex.hierarchical_sae_loss)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_eager_definitions_agree_with_oracle(mode, fn, dtype):
    args = make_inputs(16, 16, 64, 128, dtype=dtype)
    L, *_ = oracle.loss_grads(mode, *args, want_grads=False)
    got = fn(*args)
    assert got.dtype == torch.float32 and got.dim() == 0
    assert abs(got.item() - L) <= 2e-6 * abs(L)


@pytest.mark.parametrize("name", ["hier_fwd", "topk_fwd"])
def test_fake_kernels_give_shapes_and_dtypes(name):
    op = getattr(torch.ops.flexsae_amd, name)
    meta = lambda *s, dt=torch.bfloat16: torch.empty(*s, dtype=dt, device="meta")
    loss, resid = op(meta(32, 8, dt=torch.int64), meta(100, 256), meta(32, 8), meta(256), meta(32, 256))
    assert loss.shape == () and loss.dtype == torch.float32
    assert resid.shape == (32, 256) and resid.dtype == torch.float32
    bop = getattr(torch.ops.flexsae_amd, name.replace("fwd", "bwd"))
    dW, dv, db = bop(torch.empty((), dtype=torch.float32, device="meta"), meta(32, 8, dt=torch.int64),
                     meta(100, 256), meta(32, 8), resid)
    assert dW.shape == (100, 256) and dW.dtype == torch.bfloat16
    assert dv.shape == (32, 8) and dv.dtype == torch.float32
    assert db.shape == (256,) and db.dtype == torch.float32


def test_the_build_id_covers_the_extension_module(tmp_path, monkeypatch):
    for f in os.listdir(build.CSRC):
        shutil.copy(os.path.join(build.CSRC, f), tmp_path)
    here = build.source_id()
    monkeypatch.setattr(build, "CSRC", str(tmp_path))
    assert build.source_id() == here
    with open(tmp_path / "eager.cpp", "a") as fh:
        fh.write("// another source\n")
    changed = build.source_id()
    monkeypatch.setattr(build, "EAGER_FLAGS", [*build.EAGER_FLAGS, "-DX"])
    assert len({here, changed, build.source_id()}) == 3


@pytest.mark.parametrize("build_id,torch_version,fits", [
    ("this", torch.__version__, True), ("another", torch.__version__, False), ("this", "1.0", False), (None, None, False)])
def test_a_stale_extension_module_is_refused(build_id, torch_version, fits, monkeypatch):
    class Module:
        bound = False

        def init(self, *args):
            self.bound = True

    module = Module()
    if build_id is not None:
        module.build_id, module.torch_version = build_id, torch_version
    monkeypatch.setattr(flex, "_eager", module, raising=False)
    monkeypatch.setattr(_lib, "_eager", None)
    monkeypatch.setattr(_lib, "load", lambda: None)
    monkeypatch.setattr(_lib, "build_id", lambda: "this")
    if fits:
        assert _lib.eager(None) is module and module.bound
    else:
        with pytest.raises(_lib.FlexSAELibraryError, match="rebuild"):
            _lib.eager(None)
        assert not module.bound


def test_package_never_imports_the_oracle():
    pkg = os.path.join(ROOT, "flexsae_amd")
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".hpp", ".h")):
                text = open(os.path.join(dirpath, f)).read()
                assert not re.search(r"^\s*(from|import)\s+oracle\b", text, flags=re.M), f
                assert "sae_oracle" not in text, f


@pytest.mark.parametrize("B,K,D,want", [
    (3866, 4, 120, 1), (4096, 4, 128, 1), (4096, 16, 128, 1), (4096, 64, 128, 2),  # many row blocks: their sums count
    (1024, 64, 1024, 2), (1024, 4, 128, 3), (256, 64, 2304, 2), (64, 16, 128, 3),    # within one round of blocks
    (4096, 64, 512, 1), (4096, 64, 1024, 0), (8192, 64, 4096, 0)])
def test_rows_per_block_of_the_hot_latent_step(B, K, D, want):
    got = ops._hot_halvings(B, K, D, 256)
    assert got == want
    blocks = -(-B // (128 >> got)) * -(-D // 128)
    assert got == 0 or blocks <= 256


@pytest.mark.parametrize("forget", [lambda: flex.set_hot_latents("auto"), lambda: flex.set_dense_latents("auto")])
def test_forgotten_index_statistics_keep_their_buffer(forget):
    """A step under way may still write the words of a shape whose statistics were dropped."""
    words = torch.zeros(4, dtype=torch.int32)
    alive = weakref.ref(words)
    ops._hot_auto["a shape"] = {"pinned": words}
    del words
    forget()
    assert "a shape" not in ops._hot_auto and alive() is not None
    ops._hot_retired.pop()


@pytest.mark.parametrize("late", [False, True])
def test_a_step_that_was_not_taken_leaves_the_measurement_alive(late, monkeypatch):
    """The extension module may refuse a call, or raise, after the call has been given its measurement to leave: the next step
    of the shape asks again, and what arrives is read."""
    words = torch.zeros(4, dtype=torch.int32)

    def new_stats(key):
        st = ops._hot_auto[key] = {"hot": False, "dense": False, "pinned": words, "event": None, "spare": None,
                                   "words": (ctypes.c_uint32 * 4).from_address(words.data_ptr()), "seen": 0, "asked": 0,
                                   "pending": False}
        return st

    monkeypatch.setattr(ops, "_new_stats", new_stats)
    monkeypatch.setattr(ops, "_hot_auto", {})
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    B, K, F, D = 64, 32, 4096, 256
    route = ops._Route.__new__(ops._Route)
    route._step(B, K, F, D, torch.float32, torch.device("cuda", 0), True, 0)
    route.late = late
    monkeypatch.setattr(ops, "_route", lambda *_: route)
    route.here, route.train = False, True
    args = make_inputs(B, K, F, D)
    args = (args[0], *(x.requires_grad_() for x in args[1:4]), args[4])
    asked = []

    class Module:
        def hier_sliced(self, *a):
            asked.append(a[-2:])
            if len(asked) == 1:
                return None
            if len(asked) == 2:
                raise RuntimeError("no memory")
            return torch.zeros(())

        hier_late = hier_sliced

    assert ops._native_hier(Module(), *args) is None
    with pytest.raises(RuntimeError):
        ops._native_hier(Module(), *args)
    ops._native_hier(Module(), *args)
    assert len({tag for _, tag in asked}) == 3 and 0 not in {tag for _, tag in asked}
    assert all(pinned is words for pinned, _ in asked)
    # the third was taken: the next is asked only if that one may never answer
    ops._native_hier(Module(), *args)
    assert asked[3] == ((words, 4) if late else (None, 0))
    words[:] = torch.tensor([0, 0, 100, asked[2][1]], dtype=torch.int32)  # (few latents without a pair)
    assert ops._index_stats(route.key, B, K, F)["dense"] is True
    ops._native_hier(Module(), *args)  # answered: asked again
    assert asked[4][0] is words and asked[4][1] not in {tag for _, tag in asked[:4]}
    # a shape that is forgotten while its step is refused
    Module.hier_sliced = Module.hier_late = lambda *_: ops._forget_stats()
    words[3] = asked[4][1]
    assert ops._native_hier(Module(), *args) is None and not ops._hot_auto
    ops._hot_retired.pop()
