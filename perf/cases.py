"""The workloads this library's speed is measured on: what a LoRA fine-tuning job has it do, through its public
entry points (`Trainer`, `Lfm2Model`, `ComputeEngine`), from a two-layer toy model to the widest supported shapes.

A case is a dict of plain values; `prepare` builds the model or the operands from a seed, `run` is one pass.
Sizes are those of `bench.py`'s workloads and of the tests' projection and attention tables.
"""
import math

import numpy as np
import torch

from ferrotensor_amd import AdamParams, AttentionOptions, ComputeEngine, HipContext, UnifiedTensor
from ferrotensor_amd.trainer import Lfm2Model, ModelConfig, Trainer

ATTENTION = ("q_proj", "k_proj", "v_proj", "o_proj")
ALL = ATTENTION + ("gate_proj", "up_proj", "down_proj")


def _step(name, layers, hidden, heads, kv, ffn, vocab, sequences, tokens, rank=8, adapted="attention", weights="f16",
          checkpoint=False, micro=0, ragged=False, kind="step"):
    return {"name": name, "kind": kind, "layers": layers, "hidden": hidden, "heads": heads, "kv": kv, "ffn": ffn,
            "vocab": vocab, "sequences": sequences, "tokens": tokens, "rank": rank, "adapted": adapted,
            "weights": weights, "checkpoint": checkpoint, "micro": micro, "ragged": ragged}


def listed():
    return [
        # The headline: one optimizer step of the 360M shape on 8 sequences of 256 tokens, adapters on q/k/v/o.
        _step("step_360m_8x256", 32, 960, 15, 5, 2560, 49152, 8, 256),
        # The same recipe on the 135M shape: narrower products, fewer tiles than the chip has room for.
        _step("step_135m_8x256", 30, 576, 9, 3, 1536, 49152, 8, 256),
        # The reference's default regime (batch 1, eight accumulated sequences, one optimizer step): small launches.
        _step("step_360m_8_times_1x256", 32, 960, 15, 5, 2560, 49152, 8, 256, micro=1),
        # The largest: 1.7B-wide blocks (four of them), long sequences, adapters on all seven projections, blocks
        # recomputed in backward.
        _step("step_1p7b_4layers_8x1024", 4, 2048, 32, 32, 8192, 49152, 8, 1024, rank=16, adapted="all", checkpoint=True),
        # A data loader's batch: sequences of unequal length padded to a multiple of 32, base weights kept in f32.
        _step("step_135m_f32_ragged", 12, 576, 9, 3, 1536, 49152, 7, 391, weights="f32", ragged=True),
        # The smallest: a two-layer toy model, every launch a few microseconds.
        _step("step_tiny_2x32", 2, 64, 4, 2, 128, 256, 2, 32, rank=4),
        # Forward only (held-out evaluation, sampling from a prompt): logits of every position to the host.
        _step("forward_360m_1x96", 32, 960, 15, 5, 2560, 49152, 1, 96, kind="forward"),
        # One adapted linear, forward and backward, as an operator-level binding calls it.
        {"name": "linear_2048x576x1536", "kind": "linear", "rows": 2048, "in": 576, "out": 1536, "rank": 8, "weights": "f16"},
        # f32 products in the three layouts (a@b, a@b^T, a^T@b): trainable bases, ragged row count.
        {"name": "matmul_f32_1000x960x2560", "kind": "matmul", "m": 1000, "k": 960, "n": 2560},
        # Causal attention forward and backward at the 1.7B shape's sequence length, grouped heads.
        {"name": "attention_4x1024_15_5", "kind": "attention", "batch": 4, "seq": 1024, "heads": 15, "kv": 5, "dim": 64},
        # RMSNorm forward and backward with the scale's gradient.
        {"name": "norm_2048x960", "kind": "norm", "rows": 2048, "size": 960},
        # Masked cross-entropy over the vocabulary: loss and logits gradient of one batch's supervised rows.
        {"name": "loss_1446x49152", "kind": "loss", "rows": 1446, "vocab": 49152},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["step", "step", "step", "step", "forward", "linear", "linear", "matmul", "attention", "norm", "loss"])
    if kind in ("step", "forward"):
        heads, kv = rng.choice([(3, 1), (4, 2), (6, 2), (9, 3), (12, 4), (15, 5), (16, 16), (24, 8), (32, 32)])
        hidden = heads * 64
        ffn = 32 * int(round(hidden * rng.uniform(2.5, 4.0) / 32))
        wide = hidden > 1024
        layers = rng.randint(1, 3) if wide else _log(rng, 2, 16)
        sequences, tokens = rng.randint(1, 8), _log(rng, 24, 512 if wide else 700)
        vocab = 8 * _log(rng, 128, 6144)
        if kind == "forward":
            return {k: v for k, v in _step("", layers, hidden, heads, kv, ffn, vocab, rng.randint(1, 2),
                                           _log(rng, 8, 160), kind="forward").items() if k != "name"}
        rank = rng.choice([4, 8, 8, 16])
        ragged = rng.random() < 0.4
        micro = 0 if ragged else rng.choice([0, 0, 1, 2])
        tokens = tokens if ragged else (tokens + 31) // 32 * 32   # train_chunk takes rows that are padded already
        c = _step("", layers, hidden, heads, kv, ffn, vocab, sequences, tokens, rank, rng.choice(["attention", "attention", "all"]),
                  rng.choice(["f16", "f16", "f16", "f32"]), rng.random() < 0.25, micro, ragged)
        return {k: v for k, v in c.items() if k != "name"}
    if kind == "linear":
        return {"kind": "linear", "rows": _log(rng, 17, 8192), "in": 32 * _log(rng, 2, 64), "out": 8 * _log(rng, 8, 640),
                "rank": rng.choice([4, 8, 16]), "weights": rng.choice(["f16", "f16", "f16", "f32"])}
    if kind == "matmul":
        return {"kind": "matmul", "m": _log(rng, 31, 4096), "k": _log(rng, 32, 2560), "n": _log(rng, 32, 4096)}
    if kind == "attention":
        heads, kv = rng.choice([(9, 3), (15, 5), (32, 32), (4, 2), (8, 1)])
        return {"kind": "attention", "batch": rng.randint(1, 8), "seq": _log(rng, 17, 1024), "heads": heads, "kv": kv,
                "dim": rng.choice([64, 64, 64, 32])}
    if kind == "norm":
        return {"kind": "norm", "rows": _log(rng, 16, 8192), "size": 4 * _log(rng, 16, 512)}
    return {"kind": "loss", "rows": _log(rng, 16, 2048), "vocab": 4 * _log(rng, 64, 12288)}


# ---- inputs -----------------------------------------------------------------------------------------------


class _Random:
    """Normal values made on the GPU from a seed, as host arrays (what a loader hands over)."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 1)

    def normal(self, shape, scale=1.0):
        return (torch.randn(shape, generator=self.g, device="cuda") * scale).cpu().numpy()

    def integers(self, low, high, shape):
        return torch.randint(low, high, shape, generator=self.g, device="cuda").cpu().numpy()


class _DeviceArray:
    def __init__(self, t):
        self.t = t
        self.__cuda_array_interface__ = {"shape": tuple(t.shape), "typestr": "<f4", "data": (t.ptr, False), "version": 2}


def _as_torch(t):
    """A torch view of a library tensor (no copy)."""
    return torch.as_tensor(_DeviceArray(t), device="cuda")


def _dims(c):
    h, d = c["hidden"], c["hidden"] // c["heads"]
    return {"q_proj": (h, h), "k_proj": (h, c["kv"] * d), "v_proj": (h, c["kv"] * d), "o_proj": (h, h),
            "gate_proj": (h, c["ffn"]), "up_proj": (h, c["ffn"]), "down_proj": (c["ffn"], h)}


def _adapted(c):
    return ALL if c["adapted"] == "all" else ATTENTION


def _lengths(c):
    """Token counts of the sequences: all equal, or spread from a quarter of the longest up to it."""
    n, s = c["sequences"], c["tokens"]
    if not c["ragged"] or n == 1:
        return [s] * n
    return [s - (i * (s - s // 4)) // (n - 1) for i in range(n)]


def _prepare_model(c, rnd):
    ctx = HipContext(0)
    model = Lfm2Model(ctx, ModelConfig(
        vocab_size=c["vocab"], hidden_size=c["hidden"], intermediate_size=c["ffn"], num_hidden_layers=c["layers"],
        num_attention_heads=c["heads"], num_key_value_heads=c["kv"], rms_norm_eps=1e-5, rope_theta=100000.0,
        tie_word_embeddings=True, f16_linears=c["weights"] == "f16", checkpoint_blocks=c["checkpoint"]))
    ones = np.ones(c["hidden"], np.float32)
    model.set_tensor("model.embed_tokens.weight", rnd.normal((c["vocab"], c["hidden"]), 0.02))
    model.set_tensor("model.norm.weight", ones)
    for l in range(c["layers"]):
        p = "model.layers.%d." % l
        model.set_tensor(p + "input_layernorm.weight", ones)
        model.set_tensor(p + "post_attention_layernorm.weight", ones)
        for name, (i, o) in _dims(c).items():
            block = "mlp." if name in ("gate_proj", "up_proj", "down_proj") else "self_attn."
            model.set_tensor(p + block + name + ".weight", rnd.normal((o, i), 0.02))
    if c["kind"] == "forward":
        return {"ctx": ctx, "model": model, "rows": rnd.integers(0, c["vocab"], (c["sequences"], c["tokens"])).astype(np.uint32)}
    for name in model.linear_prefixes(_adapted(c)):
        i, o = model.linear_dims(name)
        model.set_lora(name, rnd.normal((i, c["rank"]), 0.02), rnd.normal((c["rank"], o), 0.02), 2.0 * c["rank"])
    # Next-token targets; a prompt of an eighth to a half of each sequence is not supervised.
    seqs = []
    for n in _lengths(c):
        ids = rnd.integers(0, c["vocab"], (n + 1,)).astype(np.uint32)
        prompt = int(rnd.integers(n // 8, n // 2 + 1, (1,))[0])
        seqs.append((ids[:-1], ids[1:], (np.arange(n) >= prompt).astype(np.uint8)))
    trainer = Trainer(model, lr=2e-4, weight_decay=0.0, clip_grad_norm=1.0, grad_accum_steps=c["sequences"])
    s = {"ctx": ctx, "model": model, "trainer": trainer}
    if c["ragged"]:
        s["seqs"] = seqs
    else:
        micro = c["micro"] or c["sequences"]
        stack = lambda k, at: np.stack([q[k] for q in seqs[at:at + micro]])
        s["chunks"] = [tuple(stack(k, at) for k in range(3)) for at in range(0, c["sequences"], micro)]
    return s


def prepare(case, seed):
    c, rnd = case, _Random(seed)
    if c["kind"] in ("step", "forward"):
        s = _prepare_model(c, rnd)
        s["kind"] = c["kind"]
        return s
    ctx = HipContext(0)
    s = {"kind": c["kind"], "ctx": ctx, "eng": ComputeEngine(ctx), "out": {}}

    def up(name, *shape, scale=1.0):
        s[name] = UnifiedTensor.new(ctx, rnd.normal(shape, scale), list(shape))

    def empty(name, *shape):
        s[name] = UnifiedTensor.empty(ctx, list(shape))
        s["out"][name] = _as_torch(s[name])

    if c["kind"] == "linear":
        m, k, n, r = c["rows"], c["in"], c["out"], c["rank"]
        up("x", m, k), up("dy", m, n, scale=1e-3), up("a", k, r, scale=0.02), up("b", r, n, scale=0.02)
        w = rnd.normal((k, n), 0.02)
        s["w"] = UnifiedTensor.from_f32_as_f16(ctx, w, [k, n]) if c["weights"] == "f16" else UnifiedTensor.new(ctx, w, [k, n])
        empty("t", m, r), empty("y", m, n), empty("dt", m, r), empty("dx", m, k), empty("da", k, r), empty("db", r, n)
    elif c["kind"] == "matmul":
        m, k, n = c["m"], c["k"], c["n"]
        up("a", m, k), up("b", k, n, scale=0.02)
        up("bt", n, k, scale=0.02), up("at", k, m)
        empty("ab", m, n), empty("abt", m, n), empty("atb", m, n)
    elif c["kind"] == "attention":
        b, q, h, g, d = c["batch"], c["seq"], c["heads"], c["kv"], c["dim"]
        up("q", b, q, h, d), up("k", b, q, g, d), up("v", b, q, g, d), up("do", b, q, h, d, scale=1e-2)
        empty("o", b, q, h, d), empty("dq", b, q, h, d), empty("dk", b, q, g, d), empty("dv", b, q, g, d)
        s["stats"] = UnifiedTensor.empty(ctx, [b * h * q, 2])
        s["opts"] = AttentionOptions(causal=True)
    elif c["kind"] == "norm":
        up("x", c["rows"], c["size"]), up("g", c["rows"], c["size"], scale=1e-2)
        s["w"] = UnifiedTensor.new(ctx, 1.0 + rnd.normal((c["size"],), 0.1), [c["size"]])
        empty("y", c["rows"], c["size"]), empty("gx", c["rows"], c["size"]), empty("gw", c["size"])
    else:
        up("logits", c["rows"], c["vocab"], scale=3.0)
        targets = rnd.integers(0, c["vocab"], (c["rows"],)).astype(np.uint32)
        s["targets"] = UnifiedTensor.from_bytes(ctx, targets, [c["rows"]])
        s["weights"] = UnifiedTensor.new(ctx, np.full(c["rows"], 1.0 / 180.0, np.float32), [c["rows"]])
        empty("grad", c["rows"], c["vocab"]), empty("row_loss", c["rows"])
    return s


def run(s):
    kind = s["kind"]
    if kind == "step":
        if "seqs" in s:
            stats = s["trainer"].train_batch(s["seqs"])
        else:
            stats = [s["trainer"].train_chunk(*chunk) for chunk in s["chunks"]]
        grads = s["model"].grads()
        return {"loss": [np.array([st.loss for st in stats]), np.concatenate([np.array(st.per_sequence) for st in stats])],
                "grad_norm": stats[-1].grad_norm, "grads": np.concatenate(list(grads.values()))}
    if kind == "forward":
        return s["model"].forward_batch(s["rows"])
    ctx, eng = s["ctx"], s["eng"]
    if kind == "linear":
        eng.lora_down(ctx, s["x"], s["a"], s["t"], 2.0)
        eng.lora_linear(ctx, s["x"], s["w"], s["t"], s["b"], s["y"])
        eng.lora_grad_down(ctx, s["dy"], s["b"], s["dt"], 2.0)
        eng.lora_linear_dx(ctx, s["dy"], s["w"], s["dt"], s["a"], s["dx"])
        eng.lora_grad_a(ctx, s["x"], s["dt"], s["da"])
        eng.lora_grad_b(ctx, s["t"], s["dy"], s["db"])
    elif kind == "matmul":
        eng.matmul(ctx, s["a"], s["b"], s["ab"])
        eng.matmul_bt(ctx, s["a"], s["bt"], s["abt"])
        eng.matmul_at(ctx, s["at"], s["b"], s["atb"])
    elif kind == "attention":
        eng.flash_attention_v2_with_stats(ctx, s["q"], s["k"], s["v"], s["o"], s["stats"], s["opts"])
        eng.flash_attention_v2_backward_with_stats(ctx, s["q"], s["k"], s["v"], s["o"], s["do"], s["dq"], s["dk"], s["dv"],
                                                   s["stats"], s["opts"])
    elif kind == "norm":
        eng.rms_norm_eps(ctx, s["x"], s["w"], s["y"], 1e-5)
        eng.rms_norm_backward(ctx, s["x"], s["w"], s["g"], s["gx"], s["gw"], 1e-5)
    else:
        eng.masked_cross_entropy_weighted(ctx, s["logits"], s["targets"], s["weights"], s["grad"], s["row_loss"], 0.125)
    return s["out"]


def _model_work(c):
    lens = _lengths(c)
    rows, heads, d = sum(lens), c["heads"], c["hidden"] // c["heads"]
    train = c["kind"] == "step"
    head_rows = rows * 11 / 16 if train else rows          # on average 11/16 of the positions are supervised
    size = 2 if c["weights"] == "f16" else 4
    head = c["hidden"] * c["vocab"]
    flops = 2.0 * head_rows * head * (2 if train else 1)
    params, lora = float(head), 0.0
    attn = sum(2.0 * heads * n * n * d for n in lens)       # causal: half of the two products over all pairs
    for l in range(c["layers"]):
        passes = 1 + (1 if train else 0) + (1 if train and c["checkpoint"] and l + 1 < c["layers"] else 0)
        for name, (i, o) in _dims(c).items():
            params += i * o
            first = train and l == 0 and name in ("q_proj", "k_proj", "v_proj")   # no input gradient: frozen embedding
            flops += 2.0 * rows * i * o * (passes - (1 if first else 0))
            if train and name in _adapted(c):
                lora += c["rank"] * (i + o)
                flops += 2.0 * rows * c["rank"] * (i + o) * 3
        flops += attn * ((3.5 if train else 1.0) + (passes - 2 if train else 0))
    out = 4.0 * rows * c["vocab"] if not train else 0.0
    # weights once per direction, the embedding rows, the adapters with both moments and gradients
    return {"bytes": size * params * (2 if train else 1) + 4.0 * rows * c["hidden"] + 28.0 * lora + out, "flops": flops}


def work(case):
    c = case
    if c["kind"] in ("step", "forward"):
        return _model_work(c)
    if c["kind"] == "linear":
        m, k, n, r = c["rows"], c["in"], c["out"], c["rank"]
        return {"bytes": 4.0 * m * (2 * k + 2 * n + 2 * r) + (2 if c["weights"] == "f16" else 4) * k * n + 8.0 * r * (k + n),
                "flops": 4.0 * m * k * n + 12.0 * m * r * (k + n)}
    if c["kind"] == "matmul":
        m, k, n = c["m"], c["k"], c["n"]
        return {"bytes": 4.0 * (2 * m * k + 2 * k * n + 3 * m * n), "flops": 6.0 * m * k * n}
    if c["kind"] == "attention":
        b, q, h, g, d = c["batch"], c["seq"], c["heads"], c["kv"], c["dim"]
        return {"bytes": 4.0 * b * q * d * (4 * h + 4 * g), "flops": 3.5 * 2.0 * b * h * q * q * d}
    if c["kind"] == "norm":
        return {"bytes": 4.0 * (4 * c["rows"] * c["size"] + 2 * c["size"]), "flops": 12.0 * c["rows"] * c["size"]}
    return {"bytes": 4.0 * (2 * c["rows"] * c["vocab"] + 3 * c["rows"]), "flops": 6.0 * c["rows"] * c["vocab"]}


def tolerance(case):
    return TOLERANCE[case["kind"]]


# About four times what was measured. "step", "forward": the batched pass against the same sequences passed one or
# two at a time, i.e. the same sums in another order (gradients: relative up to 7e-6, single values up to 1.1e-4 of
# the rms; logits 1.7e-6 and 1e-5). The others: against the operation in f64 (products 7e-7 and 5e-6, attention 6e-7
# and 1.1e-5, norm 1.4e-7 and 4e-7, loss 9e-8 and 1e-6).
TOLERANCE = {
    "step": {"rel": 3e-5, "max": 5e-4},
    "forward": {"rel": 7e-6, "max": 5e-5},
    "linear": {"rel": 3e-6, "max": 2e-5},
    "matmul": {"rel": 3e-6, "max": 2e-5},
    "attention": {"rel": 3e-6, "max": 5e-5},
    "norm": {"rel": 6e-7, "max": 2e-6},
    "loss": {"rel": 4e-7, "max": 4e-6},
}
