"""The workloads that this library's speed is judged by, through its Python entry points (nihilus_amd.q8_0).

What a program that runs a LLaMA-shaped model with Q8_0 weights asks of the library: one decode token of a sequence, one decode
step of a batch of sequences, the pass over a prompt, single projections on their own, and the layout conversion of a weight as
it is loaded.  The attention between the projections belongs to the caller; its output is stood in for by q, so that every
projection reads what an earlier one wrote, as in a model.

Sizes are those of the LLaMA-3-8B and 70B shapes (hidden 4096 / 8192, feed-forward 14336 / 28672, 1024-row k and v, 128256-row
output) and, in draw(), generic ones between and around them.
"""
import math

import torch

from nihilus_amd import q8_0

EPS = 1e-5
WEIGHT_STD = 0.02  # of a trained transformer's matrices: a block's contribution stays at the size of the residual stream

# hidden size, feed-forward size, rows of k and of v, rows of the output matrix
LLAMA_8B = {"embd": 4096, "ff": 14336, "kv": 1024, "vocab": 128256}
LLAMA_70B = {"embd": 8192, "ff": 28672, "kv": 1024, "vocab": 128256}


def listed():
    return [
        # The smallest call there is: one activation row against a k or v projection.  Latency and the host's path only.
        {"name": "kv_one_row", "kind": "projection", "rows": 1, "n": 1024, "k": 4096, "residual": False},
        # Attention output projection of a small batch, the residual added in the store.
        {"name": "attn_out_5_rows", "kind": "projection", "rows": 5, "n": 4096, "k": 4096, "residual": True},
        # Down projection at the 70B shapes for a batch of sequences: a quarter of a gigabyte of weights, long K.
        {"name": "down_70b_24_rows", "kind": "projection", "rows": 24, "n": 8192, "k": 28672, "residual": True},
        # One decode token of a whole model (32 blocks and the logits), and of a slice of a larger one.
        {"name": "token_8b", "kind": "token", "blocks": 32, **LLAMA_8B},
        {"name": "token_70b_4_blocks", "kind": "token", "blocks": 4, **LLAMA_70B},
        # One decode step of a server's batch: embedding rows, blocks, logits for every sequence.
        {"name": "batch_4_8b", "kind": "batch", "rows": 4, "blocks": 2, **LLAMA_8B},
        {"name": "batch_16_8b", "kind": "batch", "rows": 16, "blocks": 2, **LLAMA_8B},
        {"name": "batch_64_70b", "kind": "batch", "rows": 64, "blocks": 1, **LLAMA_70B},
        # The pass over a prompt: a short one of an odd length, the usual benchmark length, and a long one that is no round number.
        {"name": "prompt_117_8b", "kind": "prompt", "rows": 117, "blocks": 2, **LLAMA_8B},
        {"name": "prompt_512_8b", "kind": "prompt", "rows": 512, "blocks": 2, **LLAMA_8B},
        {"name": "prompt_3001_8b", "kind": "prompt", "rows": 3001, "blocks": 2, **LLAMA_8B},
        # A feed-forward weight on its way from the file's layout into the device layout, as each of a model's weights is at load.
        {"name": "load_gate_8b", "kind": "load", "n": 14336, "k": 4096},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _multiple(rng, low, high, step=128):
    return step * max(1, round(_log_int(rng, low, high) / step))


def _prompt_rows(rng, low, high):
    # An even number of 32-row strips: with an odd number the mat-mat that these cases were first timed on read past the end of its
    # activations, so there is nothing to compare those lengths with.
    strips = 2 * max(1, round(_log_int(rng, low, high) / 64))
    return 32 * strips - rng.randrange(32)


def _model(rng):
    if rng.random() < 0.4:
        return dict(rng.choice([LLAMA_8B, LLAMA_70B]))
    embd = _multiple(rng, 1024, 8192)
    return {"embd": embd, "ff": _multiple(rng, 2 * embd, min(4 * embd, 28672)), "kv": _multiple(rng, 256, min(embd, 2048)), "vocab": _log_int(rng, 32000, 130000)}


def draw(rng):
    kind = rng.choice(["projection", "projection", "token", "batch", "batch", "prompt", "prompt", "load"])
    if kind == "projection":
        # outputs of any row count, k and v sized to output-matrix sized; K as the hidden and feed-forward sizes
        case = {"kind": kind, "rows": _log_int(rng, 1, 64), "n": _log_int(rng, 1000, 28672), "k": _multiple(rng, 1024, 28672), "residual": rng.random() < 0.5}
    elif kind == "load":
        case = {"kind": kind, "n": _log_int(rng, 1000, 28672), "k": _multiple(rng, 1024, 28672)}
    else:
        case = {"kind": kind, **_model(rng)}
        large = case["embd"] > 4096
        if kind == "token":
            case["blocks"] = rng.randint(1, 4 if large else 16)
        else:
            case["rows"] = _log_int(rng, 2, 64) if kind == "batch" else _prompt_rows(rng, 40, 700 if large else 3000)
            case["blocks"] = 1 if large else rng.randint(1, 2)
    return case


class _Source:
    """Seeded inputs on the GPU."""

    def __init__(self, seed):
        self.generator = torch.Generator(device="cuda")
        self.generator.manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0):
        return torch.empty(shape, dtype=torch.float32, device="cuda").normal_(mean, std, generator=self.generator)

    def weight(self, n, k, std=WEIGHT_STD):
        return q8_0.quantize_row_q8_0(self.normal(n, k, std=std), tiled=True)

    def norm(self, k):
        return self.normal(k, std=0.1, mean=1.0)

    def tokens(self, count, vocab):
        return torch.randint(vocab, (count,), dtype=torch.int32, device="cuda", generator=self.generator)


def prepare(case, seed):
    source = _Source(seed)
    state = dict(case)
    if case["kind"] == "projection":
        state["w"] = source.weight(case["n"], case["k"])
        state["x"] = source.normal(case["rows"], case["k"])
        state["add"] = source.normal(case["rows"], case["n"]) if case["residual"] else None
        return state
    if case["kind"] == "load":
        state["blocks"] = q8_0.quantize_row_q8_0(source.normal(case["n"], case["k"], std=WEIGHT_STD))
        return state
    embd, ff, kv, vocab = case["embd"], case["ff"], case["kv"], case["vocab"]
    state["layers"] = [
        {
            "attn_norm": source.norm(embd),
            "q": source.weight(embd, embd),
            "k": source.weight(kv, embd),
            "v": source.weight(kv, embd),
            "o": source.weight(embd, embd),
            "ffn_norm": source.norm(embd),
            "gate": source.weight(ff, embd),
            "up": source.weight(ff, embd),
            "down": source.weight(embd, ff),
        }
        for _ in range(case["blocks"])
    ]
    state["embedding"] = source.weight(vocab, embd, std=1.0)
    state["out_norm"] = source.norm(embd)
    state["output"] = source.weight(vocab, embd)
    state["ids"] = source.tokens(1 if case["kind"] == "token" else case["rows"], vocab)
    return state


def _token(s):
    """One token of one sequence: the first block's q/k/v, then a launch per block from its attention to the next one's."""
    embd, ff, kv, vocab, layers = s["embd"], s["ff"], s["kv"], s["vocab"], s["layers"]
    x = q8_0.get_rows(s["embedding"], s["ids"], vocab, embd, tiled=True)[0]
    q, k, v = q8_0.gemv_f32([layers[0]["q"], layers[0]["k"], layers[0]["v"]], x, [embd, kv, kv], embd, norm_weight=layers[0]["attn_norm"], eps=EPS)
    cache = [k, v]
    for i, layer in enumerate(layers):
        if i + 1 < len(layers):
            after = layers[i + 1]
            weights, rows, norm = [after["q"], after["k"], after["v"]], [embd, kv, kv], after["attn_norm"]
        else:
            weights, rows, norm = [s["output"]], [vocab], s["out_norm"]
        _, x, ys = q8_0.decode_layer(layer["o"], q, x, layer["gate"], layer["up"], layer["down"], layer["ffn_norm"], weights, rows, norm, EPS, embd, ff)
        if i + 1 < len(layers):
            q = ys[0]
            if i < 8:
                cache += ys[1:]
    return {"hidden": x, "logits": ys[0], "cache": cache}


def _rows(s):
    """Several rows at once: a batch of sequences' decode step (logits of every row), or a prompt (logits of its last row)."""
    m, embd, ff, kv, vocab = s["rows"], s["embd"], s["ff"], s["kv"], s["vocab"]
    x = q8_0.get_rows(s["embedding"], s["ids"], vocab, embd, tiled=True)
    cache = []
    for layer in s["layers"]:
        a = q8_0.rms_norm_quantize(x, layer["attn_norm"], EPS, tiled=True)
        q = q8_0.gemm(layer["q"], a, m, embd, embd, tiled=True)
        k = q8_0.gemm(layer["k"], a, m, kv, embd, tiled=True)
        v = q8_0.gemm(layer["v"], a, m, kv, embd, tiled=True)
        cache += [k, v]
        h = q8_0.mul_mat(layer["o"], q, embd, embd, residual=x)
        a = q8_0.rms_norm_quantize(h, layer["ffn_norm"], EPS, tiled=True)
        act = q8_0.gate_up_silu(layer["gate"], layer["up"], a, m, ff, embd)
        x = q8_0.gemm_residual(layer["down"], act, h, m, embd, ff)
    if s["kind"] == "batch":
        logits = q8_0.gemm(s["output"], q8_0.rms_norm_quantize(x, s["out_norm"], EPS, tiled=True), m, vocab, embd, tiled=True)
    else:
        logits = q8_0.gemv_f32(s["output"], x[m - 1], vocab, embd, norm_weight=s["out_norm"], eps=EPS)
    return {"hidden": x, "logits": logits, "cache": cache}


def run(state):
    kind = state["kind"]
    if kind == "projection":
        return q8_0.mul_mat(state["w"], state["x"], state["n"], state["k"], residual=state["add"])
    if kind == "load":
        return q8_0.tile(state["blocks"], state["n"], state["k"])
    return _token(state) if kind == "token" else _rows(state)


def _matrix_bytes(n, k):
    return n * (k // 32) * 34


def work(case):
    kind = case["kind"]
    if kind == "load":
        return {"bytes": 2 * _matrix_bytes(case["n"], case["k"]), "flops": 0}
    if kind == "projection":
        m, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": _matrix_bytes(n, k) + 4 * m * (k + n * (2 if case["residual"] else 1)), "flops": 2 * m * n * k}
    embd, ff, kv, vocab, blocks = case["embd"], case["ff"], case["kv"], case["vocab"], case["blocks"]
    m = 1 if kind == "token" else case["rows"]
    logit_rows = m if kind == "batch" else 1
    layer = 2 * embd * embd + 2 * kv * embd + 3 * ff * embd  # weights of a block
    cached = min(blocks, 9) if kind == "token" else blocks
    values_out = m * embd + logit_rows * vocab + 2 * cached * m * kv
    return {
        "bytes": _matrix_bytes(blocks * layer + vocab * embd, 32) // 32 + m * _matrix_bytes(1, embd) + 4 * values_out + 4 * (2 * blocks + 1) * embd,
        "flops": 2 * m * blocks * layer + 2 * logit_rows * vocab * embd,
    }


def tolerance(case):
    """Four times what these paths differ from the same with every sum in 64 bits (and the library's own quantizers between them).

    A projection alone: 1.4e-7 at K = 28672, 1.0e-7 at 4096.  Through a model the quantizers decide: a last-bit difference in a value on
    a rounding tie moves a quant by one, and every further quantizer spreads that until the difference is of the size of the
    quantization itself: 0.006 behind two blocks, 0.017 behind four, 0.026 behind thirty-two.
    """
    if case["kind"] == "load":
        return "exact"  # a permutation of bytes
    if case["kind"] == "projection":
        return {"rel": 6e-7}
    return {"rel": 0.02 * math.sqrt(case["blocks"])}
