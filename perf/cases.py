"""What this package's performance is measured on: attention calls as a model makes them, from the smallest configuration to the largest ones.

A case is one call of the triple-dot or of the dot-product-sum attention, for inference (`train` false: forward alone, no
graph) or for a training step (forward and backward; the five gradients come back beside the output).  Its keys:

    op      "tdp" (triple-dot product) or "dps" (dot-product sum)
    B H T D batch, heads, sequence length, head dimension
    dtype   "bf16", "fp16" or "fp32"
    window  tdp: k1_window and k2_window; dps: k_diff (0: no window)
    kk      tdp: kk_left and kk_right (0: no window)
    causal, convert (convert_to_float32), fused (five slices of one [B,T,5,H,D] projection instead of dense tensors), train
"""
import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "flash-3-way-attention_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _case(op, B, H, T, D, dtype, window=0, kk=0, causal=True, convert=False, fused=False, train=True):
    return {"op": op, "B": B, "H": H, "T": T, "D": D, "dtype": dtype, "window": window, "kk": kk, "causal": causal,
            "convert": convert, "fused": fused, "train": train}


def listed():
    named = {
        # the smallest configuration of the benchmark: one short prompt in fp32, where launches and the host count
        "tdp_infer_fp32_short": _case("tdp", 1, 2, 64, 32, "fp32", train=False),
        # a small model's training step
        "tdp_train_small": _case("tdp", 2, 4, 256, 64, "bf16"),
        # the headline configuration, as a training step
        "tdp_train_main": _case("tdp", 4, 8, 1024, 64, "bf16"),
        # the forward sweep at head dimension 128: a long sequence at inference
        "tdp_infer_long_d128": _case("tdp", 1, 16, 2048, 128, "bf16", train=False),
        # head dimension 128 trained straight from one fused projection, on a length that is no multiple of anything
        "tdp_train_d128_fused": _case("tdp", 2, 4, 777, 128, "bf16", fused=True),
        # the published windowed forward case
        "tdp_infer_window_fp16": _case("tdp", 2, 8, 2048, 64, "fp16", window=128, kk=32, train=False),
        # a training step under a wide sliding window
        "tdp_train_window": _case("tdp", 2, 4, 2048, 64, "bf16", window=512, kk=512),
        # full precision training at a ragged length (the type the reference's benchmark scripts use)
        "tdp_train_fp32": _case("tdp", 2, 4, 500, 64, "fp32"),
        # 16-bit tensors whose score operands keep their precision, small heads
        "tdp_train_convert_d32": _case("tdp", 2, 8, 512, 32, "fp16", convert=True),
        # dot-product sum at the headline shape, a training step
        "dps_train_main": _case("dps", 4, 8, 1024, 64, "bf16"),
        # the longest dot-product-sum configuration of the reference's benchmark
        "dps_train_long": _case("dps", 1, 8, 8192, 64, "bf16", window=2048),
        # dot-product sum in full precision at a ragged length
        "dps_train_fp32": _case("dps", 2, 8, 1000, 64, "fp32", window=128),
    }
    return [dict(c, name=n) for n, c in named.items()]


def _triples(c):
    """Valid (q, j, k) of one head: j, k <= q, q - j and q - k <= window, |j - k| <= kk (all of them without causal)."""
    T = c["T"]
    if not c["causal"]:
        return T ** 3
    w, kk = c["window"] or T, c["kk"] or T
    total = 0
    for q in range(T):
        n = min(q, w) + 1  # keys of either kind that the window leaves
        m = min(n - 1, kk)
        total += n + 2 * m * n - m * (m + 1)  # pairs of [0, n) x [0, n) at most kk apart
    return total


def _pairs(c):
    """Score products of the dot-product sum in its factorised form: (s, t) with t - s <= k_diff, and (t, q)."""
    T = c["T"]
    if not c["causal"]:
        return 2 * T * T
    w = min(c["window"] or T, T - 1)
    return (w + 1) * T - w * (w + 1) // 2 + T * (T + 1) // 2


def work(c):
    D, heads = c["D"], c["B"] * c["H"]
    element = 4 if c["dtype"] == "fp32" else 2
    forward = 4 * D * heads * (_triples(c) if c["op"] == "tdp" else _pairs(c))
    backward = (3.0 if c["op"] == "tdp" else 2.5) * forward
    # in: five tensors, for a training step dO too; out: the output, for a training step five gradients
    tensors = 12 if c["train"] else 6
    return {"bytes": tensors * heads * c["T"] * D * element, "flops": forward + (backward if c["train"] else 0)}


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """Any op, type, head dimension, mask and length of the listed ranges, no costlier than the largest listed case."""
    while True:
        op = rng.choice(["tdp", "tdp", "tdp", "dps", "dps"])
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
        D = rng.choice([32, 64, 64, 128]) if op == "tdp" else rng.choice([32, 64, 64])
        T = _log_uniform(rng, 64, 2048 if op == "tdp" else 8192)
        B, H = rng.choice([1, 2, 4]), rng.choice([2, 4, 8, 16])
        windowed, causal = rng.random() < 0.3, rng.random() < 0.9
        window = _log_uniform(rng, 16, 512 if op == "tdp" else 2048) if windowed and causal else 0
        kk = rng.choice([0, window, max(window // 4, 8)]) if window and op == "tdp" else 0
        convert = op == "tdp" and D < 128 and dtype != "fp32" and rng.random() < 0.2
        c = _case(op, B, H, T, D, dtype, window, kk, causal, convert, rng.random() < 0.25, rng.random() < 0.6)
        rate = 60e12 if dtype == "fp32" else 500e12  # roughly what a large case reaches
        if work(c)["flops"] / rate <= 15e-3 and B * H * T * D <= 1 << 25:
            return c


def prepare(c, seed):
    from flash_trittention.dot_product_sum.trittention_triton import TrittentionTriton
    from flash_trittention.triple_dot_product.flash_trittention import FlashTrittentionModule

    B, H, T, D, dtype = c["B"], c["H"], c["T"], c["D"], _DTYPES[c["dtype"]]
    g = torch.Generator(device="cuda").manual_seed(seed)
    if c["fused"]:
        x = torch.randn(B, T, 5, H, D, generator=g, device="cuda").to(dtype)
        inputs = [x[:, :, i].transpose(1, 2) for i in range(5)]
        grad = torch.randn(B, T, H, D, generator=g, device="cuda").to(dtype).transpose(1, 2)
    else:
        inputs = [torch.randn(B, H, T, D, generator=g, device="cuda").to(dtype) for _ in range(5)]
        grad = torch.randn(B, H, T, D, generator=g, device="cuda").to(dtype)
    if c["train"]:
        inputs = [t.detach().requires_grad_(True) for t in inputs]
    scale = 1 / math.sqrt(D)
    if c["op"] == "tdp":
        window, kk = c["window"] or None, c["kk"] or None
        module = FlashTrittentionModule(causal=c["causal"], softmax_scale=scale, k1_window=window, k2_window=window,
                                        kk_left=kk, kk_right=kk, convert_to_float32=c["convert"])
    else:
        module = TrittentionTriton(causal=c["causal"], softmax_scale=scale, k_diff=c["window"] or T,
                                   convert_to_float32=c["convert"])
    return {"module": module, "inputs": inputs, "grad": grad, "train": c["train"], "dps": c["op"] == "dps"}


def run(state):
    if not state["train"]:
        with torch.no_grad():
            return state["module"](*state["inputs"])
    out = state["module"](*state["inputs"])
    o = out[0] if state["dps"] else out
    return out, torch.autograd.grad(o, state["inputs"], state["grad"])


def tolerance(c):
    """Four times what the outputs differ by from the same call in fp64 (fp32 tensors) or in fp32 from the same rounded
    inputs (16-bit tensors), the worst output of the listed cases and of a score of drawn ones, 2-norm / single element:
    fp32 9e-7 / 4e-5; bf16 triple-dot 3e-3 / 0.18 (D = 32 under a window 5e-3), bf16 dot-product sum 4.5e-3 / 0.38; fp16 an
    eighth of bf16.  Without a causal mask every row averages over all keys and the gradients of D = 32 keep a fifth of
    that precision (1.5e-2 in bf16)."""
    rel, most = (4e-6, 2e-4) if c["dtype"] == "fp32" else (1.2e-2, 0.7) if c["op"] == "tdp" else (1.8e-2, 0.9)
    if c["op"] == "tdp" and c["window"]:
        rel *= 1.5
    if not c["causal"]:
        rel *= 5
    if c["dtype"] == "fp16":
        rel, most = rel / 8, most / 8
    return {"rel": min(rel, 0.03), "max": most}
