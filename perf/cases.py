"""Performance cases of the fused SAE decoder-loss path.

A case is one call a user of this package has it do: a training step (loss, then ``backward()`` into
the decoder weight, the activations and the bias), an evaluation of the loss without gradients, or the
training step with the plain-SGD update of the decoder fused in.  Fields of a case:

    loss    "topk" or "hier"
    do      "step" (forward + backward), "eval" (loss under no_grad) or "sgd" (fused update, hier only)
    B, K    batch rows, active latents per row
    F, D    latents in the dictionary, columns of a row (width of the model)
    dtype   storage of weight, vals, bias and target: "fp32", "bf16" or "fp16"
    dist    how a row's latents are spread: "unique" (uniform, none twice), "randint" (uniform, repeats
            allowed) or "zipf" (exponent 1.1 over a random order of the latents, none twice, vals
            sorted descending: what a trained dictionary's top-k looks like)
    w_std   standard deviation of the weights
"""
import math

import numpy as np
import torch

import flexsae_amd as flex

_DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
_SIZES = {"fp32": 4, "bf16": 2, "fp16": 2}

# fp16 training scales its loss so that gradients do not vanish below fp16's range
_FP16_LOSS_SCALE = 65536.0


def _case(name, loss, do, B, K, F, D, dtype, dist, w_std=1.0):
    return {"name": name, "loss": loss, "do": do, "B": B, "K": K, "F": F, "D": D, "dtype": dtype, "dist": dist,
            "w_std": w_std}


def listed():
    return [
        # A notebook-sized problem (the repository's smallest configuration): a step is all launches
        # and host work, once per loss.
        _case("topk_step_small", "topk", "step", 64, 32, 4096, 256, "fp32", "randint"),
        _case("hier_step_small", "hier", "step", 64, 32, 4096, 256, "fp32", "randint"),
        # A small dictionary trained in small batches with the fused optimiser step: short kernels.
        _case("hier_sgd_zipf", "hier", "sgd", 1024, 64, 32768, 1024, "bf16", "zipf", 0.02),
        # The headline configuration (B = 4096, F = 65536, D = 2304, bf16) with the most latents per
        # row, both losses ...
        _case("topk_step_k128", "topk", "step", 4096, 128, 65536, 2304, "bf16", "unique"),
        _case("hier_step_k128", "hier", "step", 4096, 128, 65536, 2304, "bf16", "unique"),
        # ... the loss of a validation batch there, no gradients ...
        _case("hier_eval_k64", "hier", "eval", 4096, 64, 65536, 2304, "bf16", "unique"),
        # ... and the same dictionary kept in fp16 under a loss scale, with the fewest per row.
        _case("hier_step_fp16_k32", "hier", "step", 4096, 32, 65536, 2304, "fp16", "unique"),
        # fp32 parameters, the default of a training script (the workload of the timing example):
        # many steps per row over a wide dictionary.
        _case("topk_step_fp32_k256", "topk", "step", 2048, 256, 131072, 1024, "fp32", "randint"),
        _case("hier_step_fp32_k256", "hier", "step", 2048, 256, 131072, 1024, "fp32", "randint"),
        # Ragged on every axis: a last batch of an epoch, a K and an F that are no powers of two, rows
        # that are a multiple of two columns only.
        _case("hier_step_ragged", "hier", "step", 1777, 50, 24571, 1538, "bf16", "unique"),
        # A trained dictionary: a few latents in most rows, most latents in none.
        _case("hier_step_zipf", "hier", "step", 8192, 64, 262144, 4096, "bf16", "zipf", 0.02),
        # The largest: half a million latents of a wide model, 8.6 GB of weights.
        _case("hier_step_large", "hier", "step", 16384, 128, 524288, 8192, "bf16", "unique", 0.02),
    ]


def _cost(c):
    return c["B"] * c["K"] * c["D"] * (2 if c["loss"] == "hier" else 1) * _SIZES[c["dtype"]]


def draw(rng):
    """One more case: every axis over the whole range of the listed ones (sizes over their logarithm),
    about half of them off the powers of two."""
    def size(lo, hi, even=1):
        x = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        if rng.random() < 0.5:
            return min(hi, max(lo, 1 << round(math.log2(x))))
        return min(hi, max(lo, int(x) // even * even))

    largest = _cost(listed()[-1])
    while True:
        loss, do = rng.choice([("topk", "step")] * 4 + [("hier", "step")] * 5 + [("topk", "eval"), ("hier", "eval"),
                                                                                 ("hier", "sgd")])
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp32", "fp32", "fp16"])
        dist = rng.choice(["unique", "randint", "zipf"])
        # (the fused update wants rows of whole 16-byte vectors)
        c = {"loss": loss, "do": do, "B": size(64, 16384), "K": size(16, 256), "F": size(4096, 524288),
             "D": size(256, 8192, 8 if do == "sgd" else rng.choice([1, 2, 4, 64])), "dtype": dtype, "dist": dist,
             "w_std": rng.choice([1.0, 0.02])}
        if _cost(c) <= largest and c["F"] * c["D"] * _SIZES[dtype] <= 9e9:
            return c


def _zipf_p(F):
    p = np.arange(1, F + 1, dtype=np.float64) ** -1.1
    return p / p.sum()


def _indices(case, g):
    B, K, F = case["B"], case["K"], case["F"]
    dev = "cuda"
    if case["dist"] == "zipf":
        cdf = torch.from_numpy(np.cumsum(_zipf_p(F))).to(dev)
        order = torch.randperm(F, generator=g, device=dev)

        def sample(n):
            u = torch.rand(n, generator=g, device=dev, dtype=torch.float64)
            return order[torch.searchsorted(cdf, u).clamp_(max=F - 1)]
    else:
        def sample(n):
            return torch.randint(0, F, (n,), generator=g, device=dev, dtype=torch.long)

    idx = sample(B * K).view(B, K)
    if case["dist"] == "randint":
        return idx
    while True:  # without replacement: what a row has drawn already is drawn again
        s, at = torch.sort(idx, dim=1, stable=True)
        again = torch.zeros_like(idx, dtype=torch.bool)
        again.scatter_(1, at[:, 1:], s[:, 1:] == s[:, :-1])
        n = int(again.sum())
        if n == 0:
            return idx
        idx[again] = sample(n)


def prepare(case, seed):
    dt, dev = _DTYPES[case["dtype"]], "cuda"
    g = torch.Generator(device=dev).manual_seed(seed)
    B, K, F, D = case["B"], case["K"], case["F"], case["D"]
    idx = _indices(case, g)
    vals = torch.randn(B, K, generator=g, device=dev).abs_()
    if case["dist"] == "zipf":
        vals = vals.sort(dim=1, descending=True).values
    weight = torch.randn(F, D, generator=g, device=dev, dtype=dt)
    if case["w_std"] != 1.0:
        weight *= case["w_std"]
    s = {"do": case["do"], "idx": idx, "weight": weight, "vals": vals.to(dt),
         "bias": torch.randn(D, generator=g, device=dev, dtype=dt),
         "target": torch.randn(B, D, generator=g, device=dev, dtype=dt),
         "fn": flex.triton_hierarchical_sae_loss if case["loss"] == "hier" else flex.triton_topk_sae_loss,
         "scale": _FP16_LOSS_SCALE if case["dtype"] == "fp16" else 1.0,
         # a step that moves frequent latents visibly and stays well inside stability
         "lr": 0.004 * D}
    if case["do"] == "step":
        for k in ("weight", "vals", "bias"):
            s[k].requires_grad_()
    return s


def run(state):
    s = state
    args = (s["idx"], s["weight"], s["vals"], s["bias"], s["target"])
    if s["do"] == "eval":
        with torch.no_grad():
            return {"loss": s["fn"](*args)}
    if s["do"] == "sgd":
        loss, dvals, dbias = flex.hierarchical_sae_sgd_step(*args, s["lr"])
        return {"loss": loss, "dvals": dvals, "dbias": dbias, "weight": s["weight"]}
    leaves = args[1:4]
    for x in leaves:
        x.grad = None
    loss = s["fn"](*args)
    (loss if s["scale"] == 1.0 else loss * s["scale"]).backward()
    return {"loss": loss.detach(), "dweight": leaves[0].grad, "dvals": leaves[1].grad, "dbias": leaves[2].grad}


def _touched(case):
    """Expected number of latents that at least one pair selects."""
    n, F = case["B"] * case["K"], case["F"]
    if case["dist"] == "zipf":
        return float(np.sum(-np.expm1(n * np.log1p(-np.minimum(_zipf_p(F), 0.999)))))
    return -F * math.expm1(n * math.log1p(-1.0 / F))


def work(case):
    B, K, F, D = case["B"], case["K"], case["F"], case["D"]
    es = _SIZES[case["dtype"]]
    rows = _touched(case) * D * es
    read = rows + B * K * (8 + es) + D * es + B * D * es
    pairs = B * K * D
    forward = 4 * pairs if case["loss"] == "hier" else 2 * pairs  # multiply-add; the squared error of every prefix
    if case["do"] == "eval":
        return {"bytes": read + 4, "flops": forward}
    backward = 8 * pairs if case["loss"] == "hier" else 4 * pairs  # dvals, dW; the suffix sums and the walk back
    written = 4 + B * K * es + D * es + (rows if case["do"] == "sgd" else F * D * es)
    return {"bytes": read + written, "flops": forward + backward}


def tolerance(case):
    # Measured against the same path in 64 bits over all listed cases and ten drawn ones, largest seen:
    # fp32 3.3e-7 (one value 5.2e-6 of the root mean square), bf16 2.3e-3 (2.1e-2), fp16 2.1e-4 (9e-4);
    # four times that.
    return {"fp32": {"rel": 1.5e-6, "max": 3e-5}, "bf16": {"rel": 1e-2, "max": 8e-2},
            "fp16": {"rel": 1e-3, "max": 4e-3}}[case["dtype"]]
