"""Workloads of this package as its users run them, for timing and comparing.

Each case is one call sequence through the public entry points:

  train      one training step of a decoder: forward under autocast over fp32 master weights, loss,
             backward (fp16: of the loss times 1024, as a training loop scales it), and with
             ``optimizer`` the fused AdamW step -- what the package exists for
  logits     a forward pass without gradients over fp16 weights: scoring a text, or one pass of a
             generation loop (there is no key/value cache: the prompt is run again)
  linear     one Linear of the operator layer, forward and backward, with any of its epilogues
  mlp        the two-Linear ReLU block as one operator, forward and backward
  attention  causal attention on (B, S, nh * hd) activations, without bias, with a dense (nh, S, S)
             bias or with ALiBi slopes, forward and backward
  loss       cross entropy of (N, V) logits, forward and backward
  layernorm  LayerNorm, forward and backward
  softmax    softmax over the last dimension, forward and backward

``listed`` are the cases that are always looked at; ``draw`` makes more of the same ranges.  The
decoder sizes are those of the benchmark and the tests, and mixtures of them; the operators' are the
ranges of the tests, up to the sizes the decoders call them with.
"""
import math

import torch

import tritonformer_amd as T
from tritonformer_amd.optim import AdamW
from tritonformer_amd.transformer import Transformer, TransformerConfig, generate_alibi_mask, get_slopes

_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
_PADDED_VOCAB = 50304
# no drawn case costs more than the largest listed step (35 TFLOP; odd extents run slower)
_MOST_FLOPS = 14e12


def _decoder(name, kind, layers, heads, head_dim, ffn, ctx, batch, vocab, bias, alibi, dtype, optimizer=False):
    c = {"name": name, "kind": kind, "layers": layers, "heads": heads, "head_dim": head_dim, "ffn": ffn, "ctx": ctx,
         "batch": batch, "vocab": vocab, "bias": bias, "alibi": alibi, "dtype": dtype}
    if kind == "train":
        c["optimizer"] = optimizer
    return c


def listed():
    return [
        # the smallest step anyone runs: debugging a model, a unit test, a toy data set -- launches count
        _decoder("train-tiny", "train", 4, 4, 64, 1024, 256, 2, _PADDED_VOCAB, True, False, "fp16"),
        # a small model at full context, biased MLP, with its optimizer: pre-training on one card
        _decoder("train-160m", "train", 12, 12, 64, 3072, 2048, 8, _PADDED_VOCAB, True, False, "fp16", True),
        # the benchmark's headline step
        _decoder("train-410m", "train", 24, 16, 64, 4096, 2048, 4, _PADDED_VOCAB, False, False, "fp16"),
        # long context with ALiBi, one sequence
        _decoder("train-840m-alibi", "train", 24, 24, 64, 6144, 4096, 1, _PADDED_VOCAB, False, True, "fp16"),
        # the largest step, bf16, head_dim 128
        _decoder("train-1.4b-bf16", "train", 24, 16, 128, 8192, 2048, 2, _PADDED_VOCAB, False, False, "bf16"),
        # fine-tuning a small model on short texts with its optimizer and a vocabulary that nobody padded
        _decoder("finetune-odd-vocab", "train", 12, 12, 64, 3072, 320, 3, 50257, True, False, "bf16", True),
        # one pass over a short prompt
        _decoder("logits-410m-short", "logits", 24, 16, 64, 4096, 128, 1, _PADDED_VOCAB, False, False, "fp16"),
        # a Linear none of whose extents a tile divides, bias and ReLU fused
        {"name": "linear-ragged", "kind": "linear", "variant": "biasrelu", "batch": 3, "rows": 1371, "k": 2051, "n": 1733,
         "dtype": "fp16"},
        # attention with an additive bias matrix
        {"name": "attention-dense-bias", "kind": "attention", "bias": "dense", "batch": 2, "heads": 12, "ctx": 1024,
         "head_dim": 64, "dtype": "fp16"},
        # the loss alone, vocabulary not padded, bf16
        {"name": "loss-odd-vocab", "kind": "loss", "rows": 4095, "vocab": 50257, "dtype": "bf16"},
        # LayerNorm of an odd width: upper end of the tests' draws
        {"name": "layernorm-odd", "kind": "layernorm", "batch": 31, "rows": 1023, "cols": 1021, "dtype": "fp16"},
        # softmax in full precision: attention scores of one head group
        {"name": "softmax-fp32", "kind": "softmax", "batch": 8, "rows": 500, "cols": 777, "dtype": "fp32"},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choices(["train", "logits", "linear", "mlp", "attention", "loss", "layernorm", "softmax"],
                       [8, 3, 4, 2, 3, 2, 2, 2])[0]
    while True:
        c = _DRAW[kind](rng, kind)
        if work(c)["flops"] <= _MOST_FLOPS and work(c)["bytes"] <= 16e9:
            return c


def _draw_decoder(rng, kind):
    head_dim = rng.choice([64, 64, 64, 128, 32])
    heads = rng.choice([2, 3, 4, 6, 8, 12, 16, 20, 24])
    d = heads * head_dim
    ctx = 64 * _log_int(rng, 1, 64)
    c = _decoder("", kind, _log_int(rng, 2, 24), heads, head_dim, rng.choice([4 * d, 4 * d, 3 * d, 2 * d + 8 * rng.randint(1, 99)]),
                 ctx, _log_int(rng, 1, max(1, 16384 // ctx)), rng.choice([_PADDED_VOCAB, 8 * rng.randint(64, 6000), rng.randint(512, 60000)]),
                 rng.random() < 0.4, rng.random() < 0.3, rng.choice(["fp16", "bf16"]), rng.random() < 0.3)
    del c["name"]
    return c


def _extent(rng, low, high):
    """An extent of an operator: half of them whole multiples of 64, the rest anything."""
    v = _log_int(rng, low, high)
    return max(64, v // 64 * 64) if rng.random() < 0.5 else v


def _draw_linear(rng, kind):
    c = {"kind": kind, "batch": _log_int(rng, 1, 8), "rows": _extent(rng, 1, 2048), "k": _extent(rng, 64, 4096),
         "n": _extent(rng, 64, 8192), "dtype": rng.choice(["fp16", "bf16"])}
    if kind == "linear":
        c["variant"] = rng.choice(["nobias", "bias", "relu", "biasrelu"])
    else:
        c["bias"] = rng.random() < 0.5
    return c


def _draw_attention(rng, kind):
    return {"kind": kind, "bias": rng.choice(["none", "none", "dense", "alibi"]), "batch": _log_int(rng, 1, 8),
            "heads": rng.randint(1, 24), "ctx": 64 * _log_int(rng, 1, 40), "head_dim": rng.choice([32, 64, 64, 128]),
            "dtype": rng.choice(["fp16", "bf16"])}


def _draw_loss(rng, kind):
    return {"kind": kind, "rows": _log_int(rng, 1, 8192), "vocab": rng.choice([_PADDED_VOCAB, _log_int(rng, 256, 131072)]),
            "dtype": rng.choice(["fp16", "bf16"])}


def _draw_rows(rng, kind):
    return {"kind": kind, "batch": _log_int(rng, 1, 31), "rows": _log_int(rng, 1, 2048), "cols": _extent(rng, 64, 8192),
            "dtype": rng.choice(["fp16", "bf16"] if kind == "layernorm" else ["fp32", "fp16", "bf16"])}


_DRAW = {"train": _draw_decoder, "logits": _draw_decoder, "linear": _draw_linear, "mlp": _draw_linear,
         "attention": _draw_attention, "loss": _draw_loss, "layernorm": _draw_rows, "softmax": _draw_rows}


# ------------------------------------------------------------------------------------------- inputs
def _randn(g, shape, dtype, scale=1.0, shift=0.0):
    return (torch.randn(shape, generator=g, device="cuda") * scale + shift).to(dtype)


def _token_ids(g, shape, vocab):
    """Token ids as texts have them: frequencies fall off as the inverse of the rank, from 3 % for the most
    frequent one on (the rank is the id under a fixed permutation, so frequent tokens are not neighbours)."""
    u = torch.rand(shape, generator=g, device="cuda")
    rank = torch.exp(u * math.log((vocab + 3) / 3)).mul_(3).long() - 3
    step = 7919 if vocab % 7919 else 7907
    return rank.clamp_(0, vocab - 1) * step % vocab


def _prepare_decoder(case, g, seed):
    train = case["kind"] == "train"
    dtype = _DTYPES[case["dtype"]]
    d = case["heads"] * case["head_dim"]
    cfg = TransformerConfig(case["vocab"], d, case["ctx"], case["heads"], case["head_dim"], case["ffn"], case["layers"],
                            case["bias"], case["alibi"])
    torch.manual_seed(seed)
    model = Transformer(cfg, device="cuda", param_dtype=torch.float32 if train else dtype)
    with torch.no_grad():
        model.logits_out.weight.normal_(0.0, 0.02)  # the LM head starts at zero; a step from there on has it live
        for name, p in model.named_parameters():
            if p.ndim == 1:                         # LayerNorm parameters and biases some way into a training
                p.add_(torch.randn(p.shape, generator=g, device="cuda").mul_(0.05).to(p.dtype))
    state = {"model": model, "ids": _token_ids(g, (case["batch"], case["ctx"]), case["vocab"]), "dtype": dtype}
    if train:
        state["scale"] = 1024.0 if case["dtype"] == "fp16" else None
        state["optimizer"] = AdamW(model.parameters(), lr=1e-4) if case["optimizer"] else None
        state["returned"], state["updated"] = _returned(model), _updated(model)
    else:
        model.eval()
    return state


def _returned(model):
    """The parameters whose gradients a step hands back: LM head, final LayerNorm and, of the last block, the
    input LayerNorm, the value projection and the second MLP weight.  These 16-bit arithmetic determines
    (1e-3 to 1.4e-2 between two orders of summation).  The others it does not: a ReLU unit whose
    input rounds to the other side of zero takes its whole gradient with it, and query / key gradients are
    small differences, so that below the last MLP two correct fp16 steps are 2e-2 to 4e-2 apart and two bf16
    steps up to 0.15."""
    block = model.layer_list[len(model.layer_list) - 1]
    down = block.mlp.dense_4h_to_h
    return [model.logits_out.weight, model.final_layernorm.weight, model.final_layernorm.bias,
            block.input_layernorm.weight, block.input_layernorm.bias, block.attention.v_proj.weight,
            down.weight] + ([] if down.bias is None else [down.bias])


def _updated(model):
    """The parameters whose new values a step with its optimizer hands back: everything outside the blocks, and
    the first, the middle and the last block."""
    n = len(model.layer_list)
    rest = [p for name, p in model.named_parameters() if not name.startswith("layer_list.")]
    return rest + [p for i in sorted({0, n // 2, n - 1}) for p in model.layer_list[i].parameters()]


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    kind = case["kind"]
    if kind in ("train", "logits"):
        return kind, _prepare_decoder(case, g, seed)
    dtype = _DTYPES[case["dtype"]]
    if kind in ("linear", "mlp"):
        b, r, k, n = case["batch"], case["rows"], case["k"], case["n"]
        s = {"x": _randn(g, (b, r, k), dtype), "w": _randn(g, (k, n), dtype, 0.02)}
        if kind == "linear":
            s["apply"] = {"nobias": T.linear_no_bias, "bias": T.linear_bias, "relu": T.linear_fused_relu,
                          "biasrelu": T.linear_fused_bias_relu}[case["variant"]].apply
            s["args"] = [s["x"], s["w"]] + ([_randn(g, (n,), dtype, 0.1)] if case["variant"].startswith("bias") else [])
            s["dy"] = _randn(g, (b, r, n), dtype, 0.1)
        else:
            w2 = _randn(g, (n, k), dtype, 0.02)
            b1, b2 = (_randn(g, (n,), dtype, 0.1), _randn(g, (k,), dtype, 0.1)) if case["bias"] else (None, None)
            s["apply"] = T.mlp_fused_relu.apply
            s["args"] = [s["x"], s["w"], b1, w2, b2]
            s["dy"] = _randn(g, (b, r, k), dtype, 0.1)
    elif kind == "attention":
        b, nh, ctx, hd = case["batch"], case["heads"], case["ctx"], case["head_dim"]
        # views of the projections' (B, S, nh * hd) outputs, as a model makes them
        q, k, v, dy = (_randn(g, (b, ctx, nh * hd), dtype).view(b, ctx, nh, hd).permute(0, 2, 1, 3) for _ in range(4))
        s = {"apply": T.fast_causal_attention.apply, "args": [q, k, v], "dy": dy}
        if case["bias"] == "dense":
            s["constant"] = generate_alibi_mask(ctx, nh, device="cuda", dtype=dtype)[0]
            s["constant"] += _randn(g, (nh, ctx, ctx), dtype, 0.5)
        elif case["bias"] == "alibi":
            s["constant"] = torch.tensor(get_slopes(nh), device="cuda", dtype=torch.float16)
        if "constant" in s:
            s["apply"] = T.fast_causal_attention_with_bias.apply
    elif kind == "loss":
        n, v = case["rows"], case["vocab"]
        s = {"apply": T.cross_entropy_loss.apply, "args": [_randn(g, (n, v), dtype, 2.0)],
             "constant": _token_ids(g, (n,), v),
             # what a mean over the rows hands back, scaled as a training loop in fp16 does
             "dy": torch.full((n,), (1024.0 if case["dtype"] == "fp16" else 1.0) / n, device="cuda", dtype=dtype)}
    elif kind == "layernorm":
        shape = (case["batch"], case["rows"], case["cols"])
        s = {"apply": T.layer_norm.apply,
             "args": [_randn(g, shape, dtype, 1.5, 0.3), _randn(g, shape[-1:], dtype, 0.1, 1.0), _randn(g, shape[-1:], dtype, 0.1)],
             "constant": 1e-5, "dy": _randn(g, shape, dtype, 0.1)}
    else:
        shape = (case["batch"], case["rows"], case["cols"])
        s = {"apply": T.Softmax.apply, "args": [_randn(g, shape, dtype, 2.0)], "dy": _randn(g, shape, dtype, 0.1)}
    s["args"] = [None if a is None else a.requires_grad_(True) for a in s["args"]]
    return kind, s


# ------------------------------------------------------------------------------------------- the calls
def run(state):
    kind, s = state
    if kind == "logits":
        with torch.no_grad():
            return s["model"](s["ids"], None)
    if kind == "train":
        model, optimizer = s["model"], s["optimizer"]
        model.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=s["dtype"]):
            logits, loss = model(s["ids"], s["ids"])
        (loss if s["scale"] is None else loss * s["scale"]).backward()
        out = [logits, loss] + [p.grad for p in s["returned"]]
        if optimizer is not None:
            optimizer.step()
            out += s["updated"]
        return out
    args = s["args"]
    for a in args:
        if a is not None:
            a.grad = None
    y = s["apply"](*args, s["constant"]) if "constant" in s else s["apply"](*args)
    y.backward(s["dy"])
    return [y] + [a.grad for a in args if a is not None]


# ------------------------------------------------------------------------------------------- work, tolerance
def work(case):
    """Multiply-adds as two operations, causal attention at its half of the square; inputs read once, results
    written once."""
    kind = case["kind"]
    if kind in ("train", "logits"):
        L, d, f, s, b, v = (case["layers"], case["heads"] * case["head_dim"], case["ffn"], case["ctx"], case["batch"],
                            case["vocab"])
        mat = L * (4 * d * d + 2 * d * f) + d * v
        par = mat + v * d + (0 if case["alibi"] else s * d)
        if kind == "logits":
            return {"bytes": 2.0 * mat + 2.0 * b * s * v, "flops": 2.0 * b * s * mat + 2.0 * L * b * s * s * d}
        per = 8.0 + (24.0 if case["optimizer"] else 0.0)  # weight read, gradient written; AdamW: 3 reads + 3 writes of 4 bytes
        return {"bytes": per * par + 2.0 * b * s * v, "flops": 6.0 * b * s * mat + 7.0 * L * b * s * s * d}
    e = 4.0 if case["dtype"] == "fp32" else 2.0
    if kind in ("linear", "mlp"):
        t, k, n = case["batch"] * case["rows"], case["k"], case["n"]
        if kind == "linear":
            return {"bytes": e * (2 * t * k + 2 * t * n + 2 * k * n), "flops": 6.0 * t * k * n}
        return {"bytes": e * (4 * t * k + 4 * k * n), "flops": 12.0 * t * k * n}
    if kind == "attention":
        b, nh, s, hd = case["batch"], case["heads"], case["ctx"], case["head_dim"]
        bias = nh * s * s / 2 if case["bias"] == "dense" else 0
        return {"bytes": e * (8 * b * nh * s * hd + bias), "flops": 7.0 * b * nh * s * s * hd}
    if kind == "loss":
        return {"bytes": 2 * e * case["rows"] * case["vocab"], "flops": 0.0}
    return {"bytes": 4 * e * case["batch"] * case["rows"] * case["cols"], "flops": 0.0}


# kind -> data type -> (relative 2-norm, largest difference): about four times what the path differs by from the same
# arithmetic in torch operations (16-bit operands and results, sums in 32 bits; softmax in fp32 against 64 bits) and
# from itself with every contraction summed in three slices, over the listed and 120 drawn cases.
#   measured: train 9e-3 / 9e-2 in fp16, 1.4e-2 / 0.5 in bf16 (logits after all layers; LM-head gradient);
#   logits 1.8e-3 / 1e-2, 1.2e-2 / 8e-2; linear and mlp 1.5e-4 / one rounding, with a ReLU 7e-4 / 0.18 (a unit that
#   rounds to the other side of zero); attention 5e-4 / 1.3e-2, 3.8e-3 / 0.12;
#   loss, layernorm, softmax: roundings that fall the other way, at 2e-6 to 3e-5 / one rounding; fp32 9e-8 / 2e-6
_TOLERANCE = {
    "train": {"fp16": (3e-2, 0.3), "bf16": (5e-2, 0.99)},
    "logits": {"fp16": (8e-3, 4e-2), "bf16": (5e-2, 0.4)},
    "linear": {"fp16": (5e-4, 4e-3), "bf16": (2e-3, 3e-2)},
    "attention": {"fp16": (2e-3, 5e-2), "bf16": (1.5e-2, 0.5)},
    "loss": {"fp16": (1e-4, 4e-3), "bf16": (4e-4, 3e-2)},
    "layernorm": {"fp16": (1e-4, 4e-3), "bf16": (4e-4, 3e-2)},
    "softmax": {"fp16": (1e-4, 4e-3), "bf16": (4e-4, 3e-2), "fp32": (1e-6, 1e-5)},
}


def tolerance(case):
    if case["kind"] == "mlp" or "relu" in case.get("variant", ""):
        rel, largest = 3e-3, 0.8
    else:
        rel, largest = _TOLERANCE[case["kind"]][case["dtype"]]
    return {"rel": rel, "max": largest}
