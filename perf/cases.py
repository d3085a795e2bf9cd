"""What a user of this package has it do, as cases that can be timed and whose outputs can be compared.

Three kinds of work, each through the public entry points:

``rows``       alpha-entmax of the rows of a matrix (``triton_entmax``): a sparse replacement for softmax in attention maps,
               gates and output layers; inference, or training with the gradient of the input.
``attention``  sparse entmax attention (``adasplash``): prefill or scoring of a batch, or a training step with the gradients
               of q, k and v; causal or not, grouped K/V heads, padded batches, all element types.
``dense``      ``slow_entmax_attention``: the options the fused kernels do not have, as a decoding loop uses them -- one or a
               few new queries against a left-padded cache of keys, with ALiBi slopes.

Lengths of padded batches are spread evenly over [N/4, N] in an order that the seed gives, so a case's work does not depend
on the seed.  Scores have the spread that ``q_scale`` gives: with unit-variance q and k the scaled scores have unit variance;
3 is a peaked distribution, 1/sqrt(D) a flat one.
"""

import math

import torch

import adasplash_amd as A
from adasplash_amd.dense import slow_entmax_attention

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def _rows(name, rows, cols, dtype, alpha, train):
    return {"name": name, "kind": "rows", "rows": rows, "cols": cols, "dtype": dtype, "alpha": alpha, "train": train}


def _attention(name, B, Hq, Hkv, N, D, dtype, alpha, causal, padded, q_scale, k_scale, train):
    return {"name": name, "kind": "attention", "B": B, "Hq": Hq, "Hkv": Hkv, "N": N, "D": D, "dtype": dtype, "alpha": alpha,
            "causal": causal, "padded": padded, "q_scale": q_scale, "k_scale": k_scale, "train": train}


def _dense(name, B, H, q_len, k_len, D, dtype, alibi):
    return {"name": name, "kind": "dense", "B": B, "H": H, "q_len": q_len, "k_len": k_len, "D": D, "dtype": dtype, "alibi": alibi}


def listed():
    return [
        # the attention maps of a small model, one call per layer: latency counts
        _rows("rows_128x256_f32", 128, 256, "f32", 1.5, False),
        # the output layer of a language model in training: a vocabulary of odd size, single precision
        _rows("rows_2048x32001_f32_train", 2048, 32001, "f32", 1.5, True),
        # a large activation in half the bytes, forward and backward, where memory is the bound
        _rows("rows_16384x8192_bf16_train", 16384, 8192, "bf16", 1.5, True),
        # the smallest attention call: a short prompt in single precision
        _attention("prefill_1x8x128_d64_f32", 1, 8, 8, 128, 64, "f32", 1.5, True, False, 1.0, 1.0, False),
        # fine-tuning an encoder on padded batches of a few hundred tokens
        _attention("encoder_16x12x500_d64_bf16_train", 16, 12, 12, 500, 64, "bf16", 1.5, False, True, 1.0, 1.0, True),
        # one prompt of ordinary length through a layer with grouped K/V heads
        _attention("prefill_1x32x2048_d128_bf16", 1, 32, 8, 2048, 128, "bf16", 1.5, True, False, 1.0, 1.0, False),
        # training in single precision on padded batches
        _attention("train_2x8x1500_d64_f32", 2, 8, 8, 1500, 64, "f32", 1.5, True, True, 1.0, 1.0, True),
        # training where scores are flat (q scaled twice, as at the beginning of training): supports of hundreds of keys
        _attention("train_4x16x4096_d64_bf16_flat", 4, 16, 16, 4096, 64, "bf16", 1.5, True, False, 0.125, 1.0, True),
        # long documents through a block-mask layer: not causal, generic alpha, peaked scores
        _attention("encoder_2x16x16384_d64_bf16", 2, 16, 16, 16384, 64, "bf16", 1.333, False, False, 3.0, 3.0, False),
        # a large prefill of prompts of different lengths
        _attention("prefill_8x32x8192_d128_bf16", 8, 32, 8, 8192, 128, "bf16", 1.5, True, True, 1.0, 1.0, False),
        # a training step of the same layer
        _attention("train_8x32x8192_d128_bf16", 8, 32, 8, 8192, 128, "bf16", 1.5, True, True, 1.0, 1.0, True),
        # a decoding step of a batch against left-padded caches
        _dense("decode_16x16_k4096_d64_bf16", 16, 16, 1, 4096, 64, "bf16", True),
    ]


def _spread(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm, odd as often as not."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("rows", "rows", "attention", "attention", "attention", "dense"))
    if kind == "rows":
        cols = _spread(rng, 64, 65536)
        if rng.random() < 0.5:
            cols = max(64, cols // 64 * 64)
        rows = _spread(rng, 16, max(32, min(32768, (1 << 26) // cols)))
        case = _rows("", rows, cols, rng.choice(("f32", "bf16", "f16")), rng.choice((1.333, 1.5, 1.5, 2.0)), rng.random() < 0.5)
    elif kind == "dense":
        q_len = rng.choice((1, 1, 1, _spread(rng, 2, 16)))
        k_len = _spread(rng, 64, 8192)
        D = rng.choice((64, 128))
        B = _spread(rng, 1, 32)
        H = rng.choice((8, 16, 32))
        while B > 1 and B * H * k_len * (D + 4 * q_len) > (1 << 27):
            B //= 2
        case = _dense("", B, H, q_len, k_len, D, rng.choice(("f32", "bf16", "bf16", "f16")), rng.random() < 0.5)
    else:
        dtype = rng.choice(("bf16", "bf16", "f16", "f32"))
        causal = rng.random() < 0.6
        alpha = 1.5 if causal else rng.choice((1.333, 1.5, 2.0))
        Hkv = rng.choice((4, 8, 16))
        Hq = Hkv * rng.choice((1, 2, 4)) if causal else Hkv
        D = rng.choice((64, 128))
        padded = rng.random() < 0.5
        N = _spread(rng, 64, 16384)
        if not padded:
            N = 1 << (N.bit_length() - 1)
        q_scale = rng.choice((1.0, 1.0, 1.0, 3.0, 0.125))
        # a quarter of the largest listed case's score products, a sixtieth for single precision
        most = (1 << 31) if dtype != "f32" else (1 << 27)
        while Hq * N * N * D > 64 * most:
            N //= 2
        B = _spread(rng, 1, 16)
        while B > 1 and B * Hq * N * N * D > 64 * most:
            B //= 2
        case = _attention("", B, Hq, Hkv, N, D, dtype, alpha, causal, padded, q_scale, 1.0, rng.random() < 0.5)
    del case["name"]
    return case


def _lengths(case):
    """Valid lengths of a padded batch in ascending order: evenly spread over [n/4, n]."""
    n = case["N"] if case["kind"] == "attention" else case["k_len"]
    if case["kind"] == "attention" and not case["padded"]:
        return [n] * case["B"]
    B, lo = case["B"], max(1, n // 4)
    return [n - (n - lo) * i // max(1, B - 1) for i in range(B)][::-1]


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[case["dtype"]]

    def normal(shape, scale=1.0):
        return (torch.randn(shape, generator=g, device="cuda") * scale).to(dtype)

    state = {"case": case}
    if case["kind"] == "rows":
        shape = (case["rows"], case["cols"])
        state["x"] = normal(shape, 4.0).requires_grad_(case["train"])
        if case["train"]:
            state["dy"] = normal(shape)
        return state
    lens = torch.tensor(_lengths(case), dtype=torch.int32, device="cuda")
    lens = lens[torch.randperm(case["B"], generator=g, device="cuda")]
    if case["kind"] == "dense":
        B, H, D = case["B"], case["H"], case["D"]
        state["q"] = normal((B, H, case["q_len"], D))
        state["k"] = normal((B, H, case["k_len"], D))
        state["v"] = normal((B, H, case["k_len"], D))
        state["varlen"] = lens
        slopes = torch.tensor([2.0 ** (-8.0 * (h + 1) / H) for h in range(H)], device="cuda")
        state["slopes"] = slopes if case["alibi"] else None
        return state
    B, N, D = case["B"], case["N"], case["D"]
    state["q"] = normal((B, case["Hq"], N, D), case["q_scale"]).requires_grad_(case["train"])
    state["k"] = normal((B, case["Hkv"], N, D), case["k_scale"]).requires_grad_(case["train"])
    state["v"] = normal((B, case["Hkv"], N, D)).requires_grad_(case["train"])
    state["varlen"] = lens if case["padded"] else None
    if case["train"]:
        state["dout"] = normal((B, case["Hq"], N, D))
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "rows":
        y = A.triton_entmax(state["x"], alpha=case["alpha"])
        if not case["train"]:
            return y
        return [y.detach(), *torch.autograd.grad(y, (state["x"],), state["dy"])]
    q, k, v = state["q"], state["k"], state["v"]
    if case["kind"] == "dense":
        return slow_entmax_attention(q, k, v, alpha=1.5, varlen=state["varlen"], is_causal=True, padding="left",
                                     alibi_slopes=state["slopes"])
    out = A.adasplash(q, k, v, alpha=case["alpha"], is_causal=case["causal"], varlen=state["varlen"])
    if not case["train"]:
        return out
    return [out.detach(), *torch.autograd.grad(out, (q, k, v), state["dout"])]


def work(case):
    size = 4 if case["dtype"] == "f32" else 2
    if case["kind"] == "rows":
        n = case["rows"] * case["cols"]
        # maximum, threshold and power of every value; with the gradient two sums and a product more
        return {"bytes": n * size * (4 if case["train"] else 2), "flops": n * (8 if case["train"] else 4)}
    lens, D = _lengths(case), case["D"]
    if case["kind"] == "dense":
        q_rows, keys = case["B"] * case["H"] * case["q_len"], case["H"] * sum(lens)
        return {"bytes": size * D * (2 * q_rows + 2 * keys), "flops": 4 * D * keys * case["q_len"]}
    # two products of a forward pass, halved by a causal mask; five more in the gradients' (S, dP, dV, dK, dQ)
    flops = 4 * case["Hq"] * D * sum(n * n for n in lens) / (2 if case["causal"] else 1)
    q_elems, kv_elems = D * case["Hq"] * sum(lens), D * case["Hkv"] * sum(lens)
    padding = D * case["Hq"] * (case["B"] * case["N"] - sum(lens))  # zeros of the padded output rows
    if not case["train"]:
        return {"bytes": size * (2 * q_elems + 2 * kv_elems + padding), "flops": flops}
    padding_kv = D * case["Hkv"] * (case["B"] * case["N"] - sum(lens))
    return {"bytes": size * (4 * q_elems + 4 * kv_elems + 2 * padding + 2 * padding_kv), "flops": 3.5 * flops}


def tolerance(case):
    f32 = case["dtype"] == "f32"
    if case.get("train") and case["alpha"] == 2.0:
        # sparsemax's derivative is one on the support and zero off it: a value at the border, which rounding may put on either
        # side, changes its row's gradient at once
        return {"rel": 5e-3 if f32 else 2e-2, "max": 0.99}
    # 32-bit: sums of up to some ten thousand terms in any order, and thresholds solved to about 1e-6 of a probability of order
    # one; 16-bit: probabilities and their gradients are rounded to the type (2^-9 for bf16) before they weight rows, and the
    # results are rounded once more
    return {"rel": 2e-5 if f32 else 1e-2}
