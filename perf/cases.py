"""What a user of this package has it do, as cases of a performance comparison.

Training steps through ``Trainer``, loss and gradients through ``Transformer``, single blocks through
``TransformerBlock`` and the operators of ``ops`` that the host bindings call one by one, from calls that
are nothing but launch latency to multi-billion-parameter slices that fill the GPU for a tenth of a second.
Model widths are those of ``TransformerRecipe``; models that need more than a fraction of the GPU are cut
to a few layers with their embedding, LM head and loss kept whole.
"""
from __future__ import annotations

import dataclasses
import math

import torch

from olmax_amd import AdamWConfig, ConstantSchedule, Trainer, TransformerRecipe, ops
from olmax_amd.layer import TransformerBlock

BF16 = torch.bfloat16

MODELS = {
    "tiny_llama": lambda layers: TransformerRecipe.tiny_llama(),
    "llama_like_271M": lambda layers: dataclasses.replace(TransformerRecipe.llama_like_271M(), num_layers=layers),
    "llama_like_7B": lambda layers: dataclasses.replace(TransformerRecipe.llama_like_7B_bench(), num_layers=layers),
    "llama3_8B": lambda layers: dataclasses.replace(TransformerRecipe.llama3_8B(), num_layers=layers),
    "olmo2_7B": lambda layers: dataclasses.replace(TransformerRecipe.olmo2_7B(), num_layers=layers),
    "gemma2_like_27B": lambda layers: TransformerRecipe.gemma2_slice_bench(layers),
    "gemma3_like_27B": lambda layers: TransformerRecipe.gemma3_slice_bench(layers),
}


def listed():
    return [
        # the CPU-sized plumbing configuration: head_dim 64, a step of some hundred short launches
        {"name": "tiny-train", "kind": "train", "model": "tiny_llama", "layers": 4, "batch": 4, "seq": 512, "micro": 1, "clip": 0.0},
        # a small model, width 1024, activations kept, on full sequences
        {"name": "small-train", "kind": "train", "model": "llama_like_271M", "layers": 4, "batch": 8, "seq": 1024, "micro": 1, "clip": 0.0},
        # the same model with gradient accumulation and global-norm clipping on batches whose token count no tile divides
        {"name": "small-train-accumulate", "kind": "train", "model": "llama_like_271M", "layers": 4, "batch": 3, "seq": 1000, "micro": 2, "clip": 1.0},
        # the headline step (sequence 4096, micro-batch 2, full-block recompute, overlapped optimizer), two of its layers
        {"name": "7b-train", "kind": "train", "model": "llama_like_7B", "layers": 2, "batch": 2, "seq": 4096, "micro": 1, "clip": 0.0},
        # post-norm + QK-norm + a vocabulary (100278) whose rows are not 16-byte aligned; loss and gradients only
        {"name": "olmo2-grads", "kind": "grads", "model": "olmo2_7B", "layers": 1, "batch": 1, "seq": 2048},
        # soft-caps, GQA, a 256000-entry tied vocabulary, full-block recompute; the longest pass of the list
        {"name": "gemma2-grads", "kind": "grads", "model": "gemma2_like_27B", "layers": 2, "batch": 2, "seq": 4096},
        # sliding windows, QK-norm, tied 262144-entry vocabulary, optimizer included
        {"name": "gemma3-train", "kind": "train", "model": "gemma3_like_27B", "layers": 2, "batch": 1, "seq": 4096, "micro": 1, "clip": 0.0},
        # one block forward and backward in isolation, as the block-level binding calls it
        {"name": "olmo2-block", "kind": "block", "model": "olmo2_7B", "batch": 2, "seq": 4096, "backward": True},
        # the forward of a GQA block on one sequence of ragged length: evaluation
        {"name": "llama3-block-forward", "kind": "block", "model": "llama3_8B", "batch": 1, "seq": 1500, "backward": False},
        # attention alone, forward and backward, GQA, a length that ends inside a tile
        {"name": "attention", "kind": "attention", "batch": 2, "seq": 1777, "heads": 32, "kv_heads": 8, "head_dim": 128, "window": -1, "softcap": 0.0},
        # one linear layer with its two gradients on a handful of tokens
        {"name": "linear", "kind": "linear", "tokens": 77, "inner": 1024, "outer": 2816},
        # RMSNorm forward and backward on a few hundred rows: launch latency
        {"name": "norm", "kind": "norm", "tokens": 300, "width": 2048},
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tiny", "small", "large", "large", "grads", "block", "block", "attention", "attention", "linear", "norm"])
    if kind == "tiny":
        return {"kind": "train", "model": "tiny_llama", "layers": 4, "batch": rng.randint(2, 8), "seq": _log(rng, 128, 1024), "micro": rng.choice([1, 1, 2]),
                "clip": rng.choice([0.0, 1.0])}
    if kind == "small":  # small models run on whatever lengths the data has
        batch = rng.randint(1, 6)
        seq = _log(rng, 3000, 8192) // batch
        seq = seq if rng.random() < 0.5 else seq // 64 * 64
        return {"kind": "train", "model": "llama_like_271M", "layers": 4, "batch": batch, "seq": seq, "micro": rng.choice([1, 1, 2]),
                "clip": rng.choice([0.0, 1.0])}
    if kind == "large":  # the large recipes train on packed sequences: whole multiples of 128 tokens
        model, batch, least = rng.choice([("llama_like_7B", 2, 1536), ("gemma3_like_27B", 1, 2048)])
        return {"kind": "train", "model": model, "layers": 2, "batch": batch, "seq": _log(rng, least, 4096) // 128 * 128, "micro": 1,
                "clip": rng.choice([0.0, 0.0, 1.0])}
    if kind == "grads":
        model, layers, batch, least, most = rng.choice([("olmo2_7B", 1, 1, 1024, 2048), ("gemma2_like_27B", 2, 2, 2048, 4096), ("llama3_8B", 2, 1, 2048, 4096)])
        return {"kind": "grads", "model": model, "layers": layers, "batch": batch, "seq": _log(rng, least, most) // 128 * 128}
    if kind == "block":
        model = rng.choice(["llama_like_7B", "llama3_8B", "olmo2_7B", "gemma2_like_27B", "gemma3_like_27B"])
        if rng.random() < 0.5:
            return {"kind": "block", "model": model, "batch": rng.randint(1, 2), "seq": 128 * max(1, _log(rng, 256, 4096) // 128), "backward": rng.random() < 0.6}
        return {"kind": "block", "model": model, "batch": 1, "seq": _log(rng, 60, 1900), "backward": rng.random() < 0.6}
    if kind == "attention":
        if rng.random() < 0.3:
            return {"kind": "attention", "batch": rng.randint(1, 4), "seq": _log(rng, 64, 1024), "heads": 16, "kv_heads": rng.choice([4, 16]), "head_dim": 64,
                    "window": rng.choice([-1, 256]), "softcap": 0.0}
        heads, kv = rng.choice([(32, 32), (32, 16), (32, 8), (40, 8), (8, 8)])
        return {"kind": "attention", "batch": rng.randint(1, 2), "seq": _log(rng, 64, 6000), "heads": heads, "kv_heads": kv, "head_dim": 128,
                "window": rng.choice([-1, -1, 1024]), "softcap": rng.choice([0.0, 0.0, 50.0])}
    if kind == "linear":
        inner, outer = rng.choice([(1024, 1024), (1024, 2816), (2816, 1024), (4096, 4096), (4096, 11008), (5376, 4096)])
        return {"kind": "linear", "tokens": _log(rng, 16, 4096), "inner": inner, "outer": outer}
    return {"kind": "norm", "tokens": _log(rng, 32, 16384), "width": rng.choice([256, 1024, 2048, 4096, 4608, 5376])}


def _config(case):
    return MODELS[case["model"]](case.get("layers", 1))


def _normal(gen, *shape, std=1.0):
    return torch.empty(*shape, device="cuda", dtype=BF16).normal_(0.0, std, generator=gen)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind in ("train", "grads"):
        cfg = _config(case)
        model = cfg.build(batch_size=case["batch"], sequence_length=case["seq"], seed=seed)
        n = case["batch"] * case["seq"]
        token = lambda: torch.randint(0, cfg.vocab_size, (n,), device="cuda", dtype=torch.int32, generator=gen)  # noqa: E731
        batch = [(token(), token()) for _ in range(case.get("micro", 1))]
        state = {"case": case, "model": model, "batch": batch}
        if kind == "train":  # a rate of the early warm-up: a few steps on one batch leave the weights as they are met
            state["trainer"] = Trainer(model, AdamWConfig(lr=ConstantSchedule(1e-5), b1=0.9, b2=0.95, weight_decay=0.1,
                                                          no_decay_modules=["embedding.weight"], max_grad_norm=case["clip"] or None))
        return state
    if kind == "block":
        cfg = _config(case)
        block = TransformerBlock(cfg, batch_size=case["batch"], sequence_length=case["seq"])
        for w in (block.wqkv, block.wo, block.wgu, block.wdown):
            w.normal_(0.0, 0.02, generator=gen)
        n = case["batch"] * case["seq"]
        return {"case": case, "block": block, "x": _normal(gen, n, cfg.d_model), "dy": _normal(gen, n, cfg.d_model)}
    if kind == "attention":
        B, S, H, K, D = (case[k] for k in ("batch", "seq", "heads", "kv_heads", "head_dim"))
        qkv = _normal(gen, B * S, (H + 2 * K) * D)  # one projection's output, read in place
        return {"case": case, "q": qkv[:, :H * D], "k": qkv[:, H * D:(H + K) * D], "v": qkv[:, (H + K) * D:], "do": _normal(gen, B * S, H * D)}
    if kind == "linear":
        T, I, O = case["tokens"], case["inner"], case["outer"]
        return {"case": case, "x": _normal(gen, T, I), "w": _normal(gen, O, I, std=0.02), "dy": _normal(gen, T, O)}
    T, d = case["tokens"], case["width"]
    return {"case": case, "x": _normal(gen, T, d), "dy": _normal(gen, T, d), "w": 1.0 + _normal(gen, d, std=0.1)}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "train":
        m = state["model"]
        loss = state["trainer"].train_batch(state["batch"])
        return {"loss": loss, "master": m.master, "m": m.m, "v": m.v, "params": m.params_bf16, "grad": m.grad_bf16, "grad_f32": m.grad_f32}
    if kind == "grads":
        m = state["model"]
        loss = m.loss_and_grads(*state["batch"][0])
        return {"loss": loss, "grad": m.grad_bf16, "grad_f32": m.grad_f32}
    if kind == "block":
        block = state["block"]
        y = block.forward(state["x"])
        if not case["backward"]:
            return y
        dx = block.backward(state["dy"])
        return {"y": y, "dx": dx, **block.grads}
    if kind == "attention":
        kw = dict(B=case["batch"], S=case["seq"], H=case["heads"], KH=case["kv_heads"], D=case["head_dim"],
                  window=None if case["window"] < 0 else case["window"], softcap=case["softcap"])
        q, k, v = state["q"], state["k"], state["v"]
        o, lse = ops.attn_fwd(q, k, v, **kw)
        dq, dk, dv = ops.attn_bwd(q, k, v, o, lse, state["do"], **kw)
        return {"o": o, "lse": lse, "dq": dq, "dk": dk, "dv": dv}
    if kind == "linear":
        x, w, dy = state["x"], state["w"], state["dy"]
        return {"y": ops.linear_fwd(x, w), "dx": ops.linear_bwd_input(dy, w), "dw": ops.linear_bwd_weight(dy, x)}
    x, w, dy = state["x"], state["w"], state["dy"]
    y = ops.rms_norm_fwd(x, w, 1e-5)
    dx, dw = ops.rms_norm_bwd(x, w, dy, 1e-5)
    return {"y": y, "dx": dx, "dw": dw}


def _pairs(S, window):
    """Visible (query, key) pairs of one causal sequence; a window w shows w + 1 keys."""
    if window < 0 or window + 1 >= S:
        return S * (S + 1) // 2
    return (window + 1) * (window + 2) // 2 + (S - window - 1) * (window + 1)


def work(case):
    kind = case["kind"]
    if kind in ("train", "grads"):
        cfg = _config(case)
        tokens = case["batch"] * case["seq"]
        d, H, K, D, F, V = cfg.d_model, cfg.n_heads, cfg.n_kv_heads, cfg.head_dim, cfg.hidden_size, cfg.vocab_size
        n = cfg.num_layers * (d * (H + 2 * K) * D + H * D * d + 3 * d * F) + V * d * (1 if cfg.tie_embeddings else 2)
        micro = case.get("micro", 1)
        # bf16 weights in, gradients out (bf16; the embedding's in fp32); the optimizer reads and writes fp32 p, m, v
        # and writes the bf16 copy
        size = 4.0 * n + 2.0 * V * d + 8.0 * tokens
        if kind == "train":
            size = micro * size + 26.0 * n
        return {"bytes": size, "flops": micro * tokens * cfg.flops_per_token(case["seq"])}
    if kind == "block":
        cfg = _config(case)
        T, S = case["batch"] * case["seq"], case["seq"]
        d, H, K, D, F = cfg.d_model, cfg.n_heads, cfg.n_kv_heads, cfg.head_dim, cfg.hidden_size
        n = d * (H + 2 * K) * D + H * D * d + 3 * d * F
        flops = 2.0 * T * n + 4.0 * case["batch"] * H * D * _pairs(S, cfg.windows()[0])
        if not case["backward"]:
            return {"bytes": 2.0 * n + 4.0 * T * d, "flops": flops}
        attn = 4.0 * case["batch"] * H * D * _pairs(S, cfg.windows()[0])
        return {"bytes": 4.0 * n + 8.0 * T * d, "flops": 6.0 * T * n + 3.5 * attn}
    if kind == "attention":
        B, S, H, K, D = (case[k] for k in ("batch", "seq", "heads", "kv_heads", "head_dim"))
        return {"bytes": 2.0 * B * S * D * (4 * H + 4 * K) + 4.0 * B * H * S, "flops": 3.5 * 4.0 * B * H * D * _pairs(S, case["window"])}
    if kind == "linear":
        T, I, O = case["tokens"], case["inner"], case["outer"]
        return {"bytes": 4.0 * (T * I + T * O + I * O), "flops": 6.0 * T * I * O}
    return {"bytes": 8.0 * case["tokens"] * case["width"] + 6.0 * case["width"], "flops": 12.0 * case["tokens"] * case["width"]}


def tolerance(case):
    # Measured against the same computation in fp32, and against another bf16 implementation that rounds where this
    # one rounds; the bounds are about four times the differences, cut where the model's own noise is close to them.
    kind = case["kind"]
    if kind in ("train", "grads"):  # flat gradients: 0.006 to 0.016 (two N(0, 0.02) layers of width 4096 amplify every rounding)
        return {"rel": 0.03, "max": 0.99}  # max: 0.1 to 0.9 over an embedding gradient that is zero in most rows
    if kind == "block":  # 0.006 to 0.011, max 0.07
        return {"rel": 0.03, "max": 0.3}
    if kind == "attention":  # 0.0025, max 0.1
        return {"rel": 0.01, "max": 0.4}
    return {"rel": 0.007, "max": 0.02}  # one rounding to bf16: 0.0017, max 0.0039
