"""Performance cases of the library: what a training program has it do, through its public entry points.

Two kinds of user are covered. One trains a decoder with `cgpt_amd.model` (a recorded step: token upload, forward, loss,
backward, AdamW); the other keeps a model of its own and calls the operators of `cgpt_amd.ops` one by one, as the
reference's block code does. A case is a dict of plain values with the `path` it takes:

  step        one training step of a model, its next batch uploaded first
  block       forward and backward of one decoder block, operator by operator, in the reference's order
  attention   flash attention forward and backward
  linear      a projection forward and backward
  cut_loss    classifier and loss of a large vocabulary without stored logits
  dense_loss  loss (and its gradient) of stored logits
  embedding   token lookup forward and the scatter of its gradient
  adamw       the optimizer over a model's whole parameter list

Token ids follow a Zipf distribution (a few ids take a large share of a batch, most of the vocabulary little), as the
ids of a byte-pair vocabulary do in text; activations and output gradients are normal, weights are normal with the
initialisation's deviation of 0.02.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from cgpt_amd import ops
from cgpt_amd.model import LOSS_CUT, LOSS_DENSE, Model, ModelConfig, TokenUpload

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
EPSILON = 1e-5

# The two decoder shapes that the repository trains: the 104m preset and the 12 x 768 decoder.
PRESET = {"hidden": 1024, "inter": 2048, "heads": 8, "kv_heads": 2, "head_dim": 128}
NARROW = {"hidden": 768, "inter": 2048, "heads": 12, "kv_heads": 4, "head_dim": 64}


# ------------------------------------------------------------------------------------------------ cases
def listed():
    return [
        # The training run itself: the whole 104m preset at the batch it is trained with.
        {"name": "step_104m_b32_t1024", "path": "step", **PRESET, "layers": 8, "vocab": 32000, "batch": 32, "seq": 1024,
         "dtype": "bf16", "loss": "cut"},
        # Long context: few sequences of 4096 tokens, 64-wide heads. Two of the twelve layers.
        {"name": "step_768_b8_t4096", "path": "step", **NARROW, "layers": 2, "vocab": 32000, "batch": 8, "seq": 4096,
         "dtype": "bf16", "loss": "cut"},
        # The single-sequence fp32 configuration used to check numerics against the CPU path. Two of the eight layers.
        {"name": "step_1024_f32_b1_t256", "path": "step", **PRESET, "layers": 2, "vocab": 32000, "batch": 1, "seq": 256,
         "dtype": "f32", "loss": "dense"},
        # A first experiment: small model, small vocabulary, a sequence length that is no multiple of anything.
        {"name": "step_small_f16_b3_t100", "path": "step", "hidden": 256, "inter": 704, "heads": 4, "kv_heads": 2,
         "head_dim": 64, "layers": 2, "vocab": 5003, "batch": 3, "seq": 100, "dtype": "f16", "loss": "dense"},
        # A program's own block on one short sequence: many small launches, each paid for on the host.
        {"name": "block_768_f16_b1_t128", "path": "block", **NARROW, "batch": 1, "seq": 128, "dtype": "f16"},
        # The same with an ordinary micro-batch whose row count is ragged.
        {"name": "block_1024_bf16_b5_t1001", "path": "block", **PRESET, "batch": 5, "seq": 1001, "dtype": "bf16"},
        # Attention as the reference's own benchmark calls it: one sequence, 32:8 heads, not causal, no saved logsumexp.
        {"name": "attention_f16_b1_t512", "path": "attention", "batch": 1, "seq": 512, "heads": 32, "kv_heads": 8,
         "head_dim": 128, "causal": False, "lse": False, "dtype": "f16"},
        # A projection with bias over a micro-batch, gradients added to those of the micro-batch before it.
        {"name": "linear_bf16_r2000", "path": "linear", "rows": 2000, "inputs": 1024, "outputs": 2048, "bias": True,
         "accumulate": True, "dtype": "bf16"},
        # Classifier and loss for a vocabulary that is no multiple of anything.
        {"name": "cut_loss_bf16_v50257", "path": "cut_loss", "rows": 2048, "hidden": 768, "vocab": 50257, "dtype": "bf16"},
        # The reference's own loss benchmark: fp32 logits of one sequence.
        {"name": "dense_loss_f32_v50257", "path": "dense_loss", "rows": 512, "vocab": 50257, "gradient": True, "dtype": "f32"},
        # The training batch's token lookup and the scatter of its gradient into the tied table.
        {"name": "embedding_bf16_n32768", "path": "embedding", "tokens": 32768, "hidden": 1024, "vocab": 32000,
         "accumulate": True, "dtype": "bf16"},
        # The optimizer over the 12 x 768 decoder's 134 tensors.
        {"name": "adamw_768x12", "path": "adamw", **NARROW, "layers": 12, "vocab": 32000, "dtype": "bf16"},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _decoder(rng, widest):
    """Widths of a decoder: heads of 32, 64 or 128 in groups, a feed-forward two or 8/3 times as wide."""
    while True:
        head_dim, kv_heads, group = rng.choice((32, 64, 64, 128)), rng.choice((1, 2, 4)), rng.choice((1, 2, 3, 4))
        hidden = head_dim * kv_heads * group
        if 128 <= hidden <= widest:
            inter = 2 * hidden if rng.random() < 0.5 else (8 * hidden // 3 + 31) // 32 * 32
            return {"hidden": hidden, "inter": inter, "heads": kv_heads * group, "kv_heads": kv_heads, "head_dim": head_dim}


def _batch(rng, most_rows):
    seq = _log_int(rng, 16, 2048)
    rows = _log_int(rng, 32, most_rows)
    return {"batch": max(1, min(32, rows // seq)), "seq": min(seq, most_rows)}


def _width(rng, low, high):
    """A layer's width: a multiple of 64 as a rule, sometimes any number."""
    n = _log_int(rng, low, high)
    return max(64, n // 64 * 64) if rng.random() < 0.75 else n


def draw(rng):
    path = rng.choice(("step", "step", "step", "block", "block", "attention", "linear", "cut_loss", "dense_loss", "embedding",
                       "adamw"))
    dtype = rng.choice(("bf16", "bf16", "bf16", "f16", "f16", "f32"))
    small = dtype == "f32"  # fp32 is for checks on small batches
    if path == "step":
        return {"path": path, **_decoder(rng, 1024), "layers": rng.choice((1, 2)), "vocab": _log_int(rng, 256, 32000),
                **_batch(rng, 512 if small else 16384), "dtype": dtype, "loss": rng.choice(("cut", "dense"))}
    if path == "block":
        return {"path": path, **_decoder(rng, 1024), **_batch(rng, 512 if small else 16384), "dtype": dtype}
    if path == "attention":
        kv_heads, group = rng.choice((1, 2, 4, 8)), rng.choice((1, 2, 3, 4))
        seq = _log_int(rng, 16, 512 if small else 4096)
        tokens = _log_int(rng, 32, 512 if small else 16384)
        return {"path": path, "batch": max(1, min(64, tokens // seq)), "seq": seq, "heads": kv_heads * group,
                "kv_heads": kv_heads, "head_dim": rng.choice((32, 64, 80, 96, 128)), "causal": rng.random() < 0.8,
                "lse": rng.random() < 0.8, "dtype": dtype}
    if path == "linear":
        inputs, outputs = _width(rng, 64, 4096), _width(rng, 64, 4096)
        most = (2e10 if small else 1e11) / (inputs * outputs)
        return {"path": path, "rows": _log_int(rng, 1, max(2, min(32768, most))), "inputs": inputs, "outputs": outputs,
                "bias": rng.random() < 0.3, "accumulate": rng.random() < 0.3, "dtype": dtype}
    if path == "cut_loss":
        hidden, vocab = 64 * rng.randint(4, 16), _log_int(rng, 1000, 60000)
        most = (2e10 if small else 1e11) / (hidden * vocab)
        return {"path": path, "rows": _log_int(rng, 32, max(64, min(16384, most))), "hidden": hidden, "vocab": vocab,
                "dtype": dtype}
    if path == "dense_loss":
        return {"path": path, "rows": _log_int(rng, 16, 4096), "vocab": _log_int(rng, 1000, 60000),
                "gradient": rng.random() < 0.75, "dtype": dtype}
    if path == "embedding":
        return {"path": path, "tokens": _log_int(rng, 32, 32768), "hidden": 64 * rng.randint(2, 16),
                "vocab": _log_int(rng, 256, 60000), "accumulate": rng.random() < 0.5, "dtype": dtype}
    return {"path": path, **_decoder(rng, 1024), "layers": rng.randint(1, 12), "vocab": _log_int(rng, 256, 32000),
            "dtype": dtype}


# --------------------------------------------------------------------------------------------- preparation
class _Random:
    """Seeded tensors on the device."""

    def __init__(self, seed, dtype):
        self.generator = torch.Generator(device="cuda").manual_seed(seed)
        self.dtype = dtype

    def normal(self, *shape, scale=1.0):
        return torch.randn(*shape, device="cuda", generator=self.generator).mul_(scale).to(self.dtype)

    def gain(self, width):  # a norm's weight: one, moved a little by training
        return (1.0 + 0.1 * torch.randn(width, device="cuda", generator=self.generator)).to(self.dtype)

    def ids(self, count, vocab):
        u = torch.rand(count, device="cuda", generator=self.generator, dtype=torch.float64)
        return (torch.exp(u * math.log(vocab + 1)) - 1).floor_().clamp_(0, vocab - 1).to(torch.int32)

    def empty(self, *shape):
        return torch.empty(*shape, device="cuda", dtype=self.dtype)


@functools.lru_cache(maxsize=None)
def _training_stream():
    return torch.cuda.Stream()  # a recorded step needs a stream of its own, and a program has one


def _rotary_tables(seq, head_dim, dtype):
    position = torch.arange(seq, device="cuda", dtype=torch.float32)[:, None]
    exponent = torch.arange(head_dim // 2, device="cuda", dtype=torch.float32) * 2.0 / head_dim
    theta = position / torch.pow(torch.tensor(10000.0, device="cuda"), exponent)[None, :]
    return torch.cos(theta).to(dtype), torch.sin(theta).to(dtype)


def _optimizer_options(dtype):
    return ops.AdamWOptions(learning_rate=3e-4, beta1=0.9, beta2=0.95, epsilon=1e-8, weight_decay=0.1,
                            loss_scale=1024.0 if dtype == "f16" else 1.0, max_grad_norm=1.0)


def _prepare_step(case, seed):
    config = ModelConfig(vocabulary_size=case["vocab"], num_layers=case["layers"], hidden_size=case["hidden"],
                         intermediate_size=case["inter"], num_query_heads=case["heads"], num_kv_heads=case["kv_heads"],
                         head_dim=case["head_dim"], rotary_dim=case["head_dim"], rms_epsilon=EPSILON,
                         dtype=DTYPES[case["dtype"]])
    model = Model(config, case["batch"], case["seq"], seed=seed)
    rng = np.random.RandomState(seed)
    tokens = np.exp(rng.rand(case["batch"], case["seq"] + 1) * math.log(case["vocab"] + 1)) - 1
    tokens = np.minimum(tokens, case["vocab"] - 1).astype(np.uint32)
    # At most 64 outputs: every gradient and every updated parameter where they fit, the weight matrices' gradients and the
    # norms' of the first block in deeper models.
    parameters = model.parameters()
    gradients = {"gradient." + name: gradient for name, _, gradient in parameters}
    outputs = {"loss": model.activation("loss"), **gradients}
    if 2 * len(parameters) < 60:
        outputs.update({"parameter." + name: parameter for name, parameter, _ in parameters})
    elif len(outputs) > 64:
        outputs = {name: tensor for name, tensor in outputs.items()
                   if not (name.startswith("gradient.model.layers.") and "norm" in name) or
                   name.startswith("gradient.model.layers.0.")}
    for tensor in outputs.values():
        tensor.owner = model  # they are views of the model's memory
    return {"model": model, "upload": TokenUpload(case["batch"], case["seq"]), "outputs": outputs,
            "inputs": np.ascontiguousarray(tokens[:, :-1]).reshape(-1),
            "targets": np.ascontiguousarray(tokens[:, 1:]).reshape(-1),
            "options": _optimizer_options(case["dtype"]), "loss": LOSS_CUT if case["loss"] == "cut" else LOSS_DENSE}


def _prepare_block(case, seed):
    r = _Random(seed, DTYPES[case["dtype"]])
    batch, seq, hidden, inter = case["batch"], case["seq"], case["hidden"], case["inter"]
    heads, kv_heads, head_dim = case["heads"], case["kv_heads"], case["head_dim"]
    rows, kv_width = batch * seq, kv_heads * head_dim
    weights = {"attention_norm": r.gain(hidden), "q": r.normal(hidden, hidden, scale=0.02),
               "k": r.normal(kv_width, hidden, scale=0.02), "v": r.normal(kv_width, hidden, scale=0.02),
               "q_norm": r.gain(head_dim), "k_norm": r.gain(head_dim), "o": r.normal(hidden, hidden, scale=0.02),
               "ffn_norm": r.gain(hidden), "gate": r.normal(inter, hidden, scale=0.02),
               "up": r.normal(inter, hidden, scale=0.02), "down": r.normal(hidden, inter, scale=0.02)}
    shapes = {"norm_a": (rows, hidden), "q_pre": (rows, hidden), "k_pre": (rows, kv_width), "v": (rows, kv_width),
              "q": (rows, hidden), "k": (rows, kv_width), "attended": (rows, hidden), "projected": (rows, hidden),
              "norm_f": (rows, hidden), "gate": (rows, inter), "up": (rows, inter), "activated": (rows, inter),
              "ffn": (rows, hidden), "out": (rows, hidden),
              "d_activated": (rows, inter), "d_gate": (rows, inter), "d_up": (rows, inter), "d_norm": (rows, hidden),
              "d_branch": (rows, hidden), "d_attended": (rows, hidden), "d_q": (rows, hidden), "d_k": (rows, kv_width),
              "d_v": (rows, kv_width), "d_q_pre": (rows, hidden), "d_k_pre": (rows, kv_width), "d_x": (rows, hidden)}
    buffers = {name: r.empty(*shape) for name, shape in shapes.items()}
    cos, sin = _rotary_tables(seq, head_dim, r.dtype)
    return {"x": r.normal(rows, hidden), "d_out": r.normal(rows, hidden), "w": weights,
            "g": {name: torch.empty_like(w) for name, w in weights.items()}, "b": buffers, "cos": cos, "sin": sin,
            "lse": torch.empty(batch, seq, heads, device="cuda"), "rope": ops.RopeOptions(),
            "attention": ops.FlashAttentionOptions(heads, kv_heads, head_dim), "q4": (batch, seq, heads, head_dim),
            "k4": (batch, seq, kv_heads, head_dim)}


def _prepare_attention(case, seed):
    r = _Random(seed, DTYPES[case["dtype"]])
    q4 = (case["batch"], case["seq"], case["heads"], case["head_dim"])
    k4 = (case["batch"], case["seq"], case["kv_heads"], case["head_dim"])
    return {"q": r.normal(*q4), "k": r.normal(*k4), "v": r.normal(*k4), "d_o": r.normal(*q4), "o": r.empty(*q4),
            "d_q": r.empty(*q4), "d_k": r.empty(*k4), "d_v": r.empty(*k4),
            "lse": torch.empty(q4[:3], device="cuda") if case["lse"] else None,
            "options": ops.FlashAttentionOptions(case["heads"], case["kv_heads"], case["head_dim"], causal=case["causal"])}


def _prepare_linear(case, seed):
    r = _Random(seed, DTYPES[case["dtype"]])
    rows, inputs, outputs = case["rows"], case["inputs"], case["outputs"]
    # A sum over micro-batches starts from gradients of the size that one micro-batch gives; the program clears it itself.
    accumulate = case["accumulate"]
    return {"x": r.normal(rows, inputs), "w": r.normal(outputs, inputs, scale=0.02), "d_y": r.normal(rows, outputs),
            "bias": r.normal(outputs, scale=0.02) if case["bias"] else None, "y": r.empty(rows, outputs),
            "d_x": r.empty(rows, inputs), "d_w": r.normal(outputs, inputs, scale=math.sqrt(rows)),
            "d_b": r.normal(outputs, scale=math.sqrt(rows)) if case["bias"] else None,
            "options": ops.LinearBackwardOptions(accumulate_weight=accumulate, accumulate_bias=accumulate)}


def _prepare_cut_loss(case, seed):
    r = _Random(seed, DTYPES[case["dtype"]])
    x, classifier = r.normal(case["rows"], case["hidden"]), r.normal(case["vocab"], case["hidden"], scale=0.02)
    return {"x": x, "classifier": classifier, "targets": r.ids(case["rows"], case["vocab"]),
            "loss": torch.empty(1, device="cuda"), "d_x": torch.empty_like(x), "d_classifier": torch.empty_like(classifier),
            "scale": 1024.0 if case["dtype"] == "f16" else 1.0}


def _prepare_dense_loss(case, seed):
    r = _Random(seed, DTYPES[case["dtype"]])
    logits = r.normal(case["rows"], case["vocab"], scale=2.0)
    return {"logits": logits, "targets": r.ids(case["rows"], case["vocab"]), "loss": torch.empty(1, device="cuda"),
            "gradient": torch.empty_like(logits) if case["gradient"] else None,
            "scale": 1024.0 if case["dtype"] == "f16" else 1.0}


def _prepare_embedding(case, seed):
    r = _Random(seed, DTYPES[case["dtype"]])
    weight = r.normal(case["vocab"], case["hidden"], scale=0.02)
    return {"weight": weight, "ids": r.ids(case["tokens"], case["vocab"]), "x": r.empty(case["tokens"], case["hidden"]),
            "d_x": r.normal(case["tokens"], case["hidden"]), "d_weight": r.normal(case["vocab"], case["hidden"]),
            "options": ops.EmbeddingBackwardOptions(accumulate_weight=case["accumulate"])}


def _parameter_sizes(case):
    hidden, inter, kv_width = case["hidden"], case["inter"], case["kv_heads"] * case["head_dim"]
    block = (hidden, hidden * hidden, kv_width * hidden, case["head_dim"], case["head_dim"], kv_width * hidden,
             hidden * hidden, hidden, inter * hidden, inter * hidden, hidden * inter)
    return (case["vocab"] * hidden, hidden) + case["layers"] * block


def _prepare_adamw(case, seed):
    # Parameters, gradients and moments are slices of four flat buffers, each slice on a boundary of 64 elements.
    r = _Random(seed, DTYPES[case["dtype"]])
    sizes = _parameter_sizes(case)
    starts = np.concatenate([[0], np.cumsum([(n + 63) // 64 * 64 for n in sizes])]).tolist()
    total = starts[-1]
    options = _optimizer_options(case["dtype"])
    parameter = r.normal(total, scale=0.02)
    gradient = r.normal(total, scale=1e-3 * options.loss_scale)
    master = parameter.float()
    first, second = torch.zeros_like(master), torch.zeros_like(master)
    entries = []
    for n, start in zip(sizes, starts):
        part = slice(start, start + n)
        entries.append(ops.AdamWBatchEntry(parameter[part], gradient[part],
                                           ops.AdamWState(master[part], first[part], second[part])))
    return {"entries": entries, "workspace": ops.AdamWWorkspace(), "options": options, "parameter": parameter,
            "master": master, "first": first, "second": second}


_PREPARE = {"step": _prepare_step, "block": _prepare_block, "attention": _prepare_attention, "linear": _prepare_linear,
            "cut_loss": _prepare_cut_loss, "dense_loss": _prepare_dense_loss, "embedding": _prepare_embedding,
            "adamw": _prepare_adamw}


def prepare(case, seed):
    return {"path": case["path"], **_PREPARE[case["path"]](case, seed)}


# ---------------------------------------------------------------------------------------------- one pass
def _run_step(s):
    stream = _training_stream()
    inputs, targets = s["upload"].acquire()
    inputs[:] = s["inputs"]
    targets[:] = s["targets"]
    s["model"].upload_tokens(s["upload"], stream)
    s["model"].train_step(s["options"], s["loss"], use_graph=True, stream=stream)
    return s["outputs"]


def _run_block(s):
    x, d_out, w, g, b, lse = s["x"], s["d_out"], s["w"], s["g"], s["b"], s["lse"]
    q4, k4, attention = s["q4"], s["k4"], s["attention"]
    q, k, v, attended = b["q"].view(q4), b["k"].view(k4), b["v"].view(k4), b["attended"].view(q4)
    head_dim = q4[3]
    # Forward: attention and feed-forward branches of the same input, added to it.
    ops.rmsnorm_forward(b["norm_a"], x, w["attention_norm"], EPSILON)
    ops.linear_forward(b["q_pre"], b["norm_a"], w["q"])
    ops.linear_forward(b["k_pre"], b["norm_a"], w["k"])
    ops.linear_forward(b["v"], b["norm_a"], w["v"])
    ops.rmsnorm_forward(b["q"].view(-1, head_dim), b["q_pre"].view(-1, head_dim), w["q_norm"], EPSILON)
    ops.rmsnorm_forward(b["k"].view(-1, head_dim), b["k_pre"].view(-1, head_dim), w["k_norm"], EPSILON)
    ops.rope_forward(q, k, s["cos"], s["sin"], rope_options=s["rope"])
    ops.flash_gqa_attention_forward_with_lse(attended, lse, q, k, v, options=attention)
    ops.linear_forward(b["projected"], b["attended"], w["o"])
    ops.rmsnorm_forward(b["norm_f"], x, w["ffn_norm"], EPSILON)
    ops.linear_forward(b["gate"], b["norm_f"], w["gate"])
    ops.linear_forward(b["up"], b["norm_f"], w["up"])
    ops.swiglu_forward(b["activated"], b["gate"], b["up"])
    ops.linear_forward(b["ffn"], b["activated"], w["down"])
    ops.add_tensors(b["out"], x, b["projected"])
    ops.add_tensors(b["out"], b["out"], b["ffn"])
    # Backward.
    added = ops.LinearBackwardOptions(accumulate_input=True)
    ops.linear_backward(b["d_activated"], g["down"], None, d_out, b["activated"], w["down"])
    ops.swiglu_backward(b["d_gate"], b["d_up"], b["d_activated"], b["gate"], b["up"])
    ops.linear_backward(b["d_norm"], g["gate"], None, b["d_gate"], b["norm_f"], w["gate"])
    ops.linear_backward(b["d_norm"], g["up"], None, b["d_up"], b["norm_f"], w["up"], options=added)
    ops.rmsnorm_backward(b["d_branch"], g["ffn_norm"], b["d_norm"], x, w["ffn_norm"], EPSILON)
    ops.add_tensors(b["d_x"], d_out, b["d_branch"])
    ops.linear_backward(b["d_attended"], g["o"], None, d_out, b["attended"], w["o"])
    ops.flash_gqa_attention_backward_with_lse(b["d_q"].view(q4), b["d_k"].view(k4), b["d_v"].view(k4),
                                              b["d_attended"].view(q4), attended, lse, q, k, v, options=attention)
    ops.rope_backward(b["d_q_pre"].view(q4), b["d_k_pre"].view(k4), b["d_q"].view(q4), b["d_k"].view(k4), s["cos"], s["sin"],
                      rope_options=s["rope"])
    ops.rmsnorm_backward(b["d_q"].view(-1, head_dim), g["q_norm"], b["d_q_pre"].view(-1, head_dim),
                         b["q_pre"].view(-1, head_dim), w["q_norm"], EPSILON)
    ops.rmsnorm_backward(b["d_k"].view(-1, head_dim), g["k_norm"], b["d_k_pre"].view(-1, head_dim),
                         b["k_pre"].view(-1, head_dim), w["k_norm"], EPSILON)
    ops.linear_backward(b["d_norm"], g["q"], None, b["d_q"], b["norm_a"], w["q"])
    ops.linear_backward(b["d_norm"], g["k"], None, b["d_k"], b["norm_a"], w["k"], options=added)
    ops.linear_backward(b["d_norm"], g["v"], None, b["d_v"], b["norm_a"], w["v"], options=added)
    ops.rmsnorm_backward(b["d_branch"], g["attention_norm"], b["d_norm"], x, w["attention_norm"], EPSILON)
    ops.add_tensors(b["d_x"], b["d_x"], b["d_branch"])
    return {"out": b["out"], "d_x": b["d_x"], **g}


def _run_attention(s):
    if s["lse"] is not None:
        ops.flash_gqa_attention_forward_with_lse(s["o"], s["lse"], s["q"], s["k"], s["v"], options=s["options"])
        ops.flash_gqa_attention_backward_with_lse(s["d_q"], s["d_k"], s["d_v"], s["d_o"], s["o"], s["lse"], s["q"], s["k"],
                                                  s["v"], options=s["options"])
    else:
        ops.flash_gqa_attention_forward(s["o"], s["q"], s["k"], s["v"], options=s["options"])
        ops.flash_gqa_attention_backward(s["d_q"], s["d_k"], s["d_v"], s["d_o"], s["q"], s["k"], s["v"], options=s["options"])
    return [t for t in (s["o"], s["lse"], s["d_q"], s["d_k"], s["d_v"]) if t is not None]


def _run_linear(s):
    ops.linear_forward(s["y"], s["x"], s["w"], bias=s["bias"])
    ops.linear_backward(s["d_x"], s["d_w"], s["d_b"], s["d_y"], s["x"], s["w"], options=s["options"])
    return [t for t in (s["y"], s["d_x"], s["d_w"], s["d_b"]) if t is not None]


def _run_cut_loss(s):
    ops.cut_cross_entropy_forward_backward(s["loss"], s["d_x"], s["d_classifier"], s["x"], s["classifier"], s["targets"],
                                           s["x"].shape[0], gradient_scale=s["scale"])
    return s["loss"], s["d_x"], s["d_classifier"]


def _run_dense_loss(s):
    rows = s["logits"].shape[0]
    if s["gradient"] is None:
        ops.cross_entropy_forward(s["loss"], s["logits"], s["targets"], rows)
        return s["loss"]
    ops.cross_entropy_forward_backward(s["loss"], s["gradient"], s["logits"], s["targets"], rows, gradient_scale=s["scale"])
    return s["loss"], s["gradient"]


def _run_embedding(s):
    count = s["ids"].numel()
    ops.embedding_forward(s["x"], s["ids"], count, s["weight"])
    ops.embedding_backward(s["d_weight"], s["d_x"], s["ids"], count, options=s["options"])
    return s["x"], s["d_weight"]


def _run_adamw(s):
    ops.adamw_step_many_async(s["entries"], s["options"], s["workspace"])
    return s["parameter"], s["master"], s["first"], s["second"]


_RUN = {"step": _run_step, "block": _run_block, "attention": _run_attention, "linear": _run_linear, "cut_loss": _run_cut_loss,
        "dense_loss": _run_dense_loss, "embedding": _run_embedding, "adamw": _run_adamw}


def run(state):
    return _RUN[state["path"]](state)


# -------------------------------------------------------------------------------- work and tolerances
def _attention_flops(case, products):
    pairs = case["seq"] * (case["seq"] + 1) / 2 if case.get("causal", True) else case["seq"] ** 2
    return products * 2.0 * case["batch"] * case["heads"] * pairs * case["head_dim"]


def work(case):
    e = DTYPES[case["dtype"]].itemsize
    path = case["path"]
    if path in ("step", "block"):
        rows, hidden, inter, kv_width = case["batch"] * case["seq"], case["hidden"], case["inter"], case["kv_heads"] * case["head_dim"]
        matrices = 2 * hidden * hidden + 2 * kv_width * hidden + 3 * inter * hidden
        block_flops = 6.0 * rows * matrices + _attention_flops(case, 7)
        if path == "block":
            # x and its gradient, the result and the output gradient; every weight read, every gradient written
            return {"bytes": e * (4.0 * rows * hidden + 2.0 * matrices), "flops": block_flops}
        # Token ids in; fp32 master copy and two moments read and written, the parameter read and written.
        parameters = case["layers"] * matrices + case["vocab"] * hidden
        return {"bytes": 8.0 * rows + parameters * (24.0 + 2.0 * e),
                "flops": case["layers"] * block_flops + 6.0 * rows * case["vocab"] * hidden}
    if path == "attention":
        q, k = (case["batch"] * case["seq"] * n * case["head_dim"] for n in (case["heads"], case["kv_heads"]))
        # q, dO read, o, dQ written; k, v read, dK, dV written
        return {"bytes": e * (4.0 * q + 4.0 * k), "flops": _attention_flops(case, 7)}
    if path == "linear":
        rows, inputs, outputs = case["rows"], case["inputs"], case["outputs"]
        gradients = 2 if case["accumulate"] else 1
        return {"bytes": e * (2.0 * rows * (inputs + outputs) + (1.0 + gradients) * inputs * outputs),
                "flops": 6.0 * rows * inputs * outputs}
    if path == "cut_loss":
        rows, hidden, vocab = case["rows"], case["hidden"], case["vocab"]
        return {"bytes": e * 2.0 * hidden * (rows + vocab), "flops": 6.0 * rows * hidden * vocab}
    if path == "dense_loss":
        count = case["rows"] * case["vocab"]
        return {"bytes": e * (2.0 if case["gradient"] else 1.0) * count, "flops": 4.0 * count}
    if path == "embedding":
        rows, hidden = case["tokens"], case["hidden"]
        ids = min(rows, case["vocab"])
        # The lookup writes every token's row and reads each id's once; the scatter reads every token's row and writes
        # the whole table, or reads and writes the ids' rows when it adds to what is there.
        table = 2.0 * ids if case["accumulate"] else float(case["vocab"])
        return {"bytes": 8.0 * rows + e * hidden * (2.0 * rows + ids + table), "flops": 1.0 * rows * hidden}
    parameters = float(sum(_parameter_sizes(case)))
    # Gradient read, parameter written, master copy and two moments read and written.
    return {"bytes": parameters * (2.0 * e + 24.0), "flops": 12.0 * parameters}


def tolerance(case):
    path, dtype = case["path"], case["dtype"]
    if path == "embedding":
        return "exact"  # additions in token order, each rounded to the storage type: what the CPU operator gives
    if path == "step":
        # Every operator's result is rounded to the storage type, layer after layer, and AdamW's first updates turn small
        # gradients' signs into whole steps.
        return {"rel": {"bf16": 2e-2, "f16": 5e-3, "f32": 1e-4}[dtype], "max": 0.5}
    if path == "adamw":
        return {"rel": {"bf16": 2e-3, "f16": 3e-4, "f32": 1e-5}[dtype]}
    if path == "block":
        return {"rel": {"bf16": 1e-2, "f16": 2e-3, "f32": 2e-5}[dtype]}
    return {"rel": {"bf16": 6e-3, "f16": 1e-3, "f32": 1e-5}[dtype]}
