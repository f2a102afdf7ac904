"""The work a user of this package has it do, as cases that can be timed and compared.

Every case goes through the public entry points of ``rwkv_kernel.RWKVKernelOperator`` on the GPU:

    decode         one token per sequence, the state carried in fp32: ``op(..., return_state=True)``
    decode_fused   the same with the layer's group norm and gate in the output stage (``forward_gn_gate``)
    prefill        a prompt: T tokens per sequence from a state to a state
    prefill_fused  the same with group norm and gate
    train          forward and backward of the operator
    train_fused    forward and backward of operator, group norm and gate
    train_mix      forward and backward of the layer's input side (token shift and five low-rank mixers)

Sizes are the layer shapes of this repository's benchmark and tests (heads of 64 channels; 32 and 64 heads are
its two model layers) and lengths and batches around them.  Inputs have the benchmark's distributions:
r, k, v, gy ~ N(0,1), the raw decay w ~ U(-6,1), u ~ N(0,0.25).

The module is imported with the repository's root as the working folder.
"""
import math
import os
import sys

import torch

sys.path.insert(1, os.path.join(os.getcwd(), "star-rwkv6_amd"))
os.environ.setdefault("KERAS_BACKEND", "torch")

from rwkv_kernel import RWKVKernelOperator  # noqa: E402

N = 64                      # head size
MAX_T = 16384               # the operator's declared longest sequence
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _case(kind, B, T, H, dtype="bf16", R=0):
    return {"kind": kind, "B": B, "T": T, "H": H, "dtype": dtype, "R": R}


def listed():
    named = {
        # generation for one user: one token of one sequence, a layer of 2048 channels; latency alone
        "decode_one": _case("decode", 1, 1, 32),
        # generation for a full batch of 64 sequences, with the layer's output stage
        "decode_batch": _case("decode_fused", 64, 1, 32),
        # the prompt of one request, of no special length
        "prefill_one": _case("prefill", 1, 1337, 32),
        # the prompts of a full batch of requests
        "prefill_batch": _case("prefill_fused", 64, 512, 32),
        # a training step of the 2048-channel layer at its usual batch and length
        "train_layer": _case("train", 8, 1024, 32),
        # ... of the 4096-channel layer at four times the length: the largest case
        "train_large": _case("train", 4, 4096, 64),
        # fine-tuning on one long document per GPU
        "train_long": _case("train", 1, 8192, 32),
        # a batch cut to the longest of its texts, a layer of 2560 channels: nothing divides evenly
        "train_ragged": _case("train", 6, 999, 40),
        # full-precision training at the usual shape
        "train_f32": _case("train", 8, 1024, 32, dtype="f32"),
        # a small model's step in half precision (fp32 outputs and gradients)
        "train_small_f16": _case("train", 2, 200, 8, dtype="f16"),
        # operator with group norm and gate, as the model's training step calls it
        "train_fused": _case("train_fused", 8, 1024, 32),
        # the layer's input side in the model's training step, mixers of rank 32
        "train_mix": _case("train_mix", 8, 1024, 32, R=32),
    }
    return [dict(c, name=name) for name, c in named.items()]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode_fused", "prefill", "prefill_fused", "train", "train", "train", "train_fused", "train_mix"])
    H = rng.choice([8, 12, 16, 24, 32, 32, 40, 48, 64])
    if kind in ("decode", "decode_fused"):
        return _case(kind, _log_int(rng, 1, 256), 1, H, dtype=rng.choice(["bf16", "bf16", "f16", "f32"]) if kind == "decode" else "bf16")
    dtype = rng.choice(["bf16", "bf16", "f16", "f32"]) if kind == "train" else "bf16"
    T = _log_int(rng, 64, 8192)
    # largest: 2^26 elements per tensor (the 4096-channel layer) for bf16 tensors through the operator alone,
    # 2^24 (the 2048-channel layer at its usual shape) otherwise
    cap = 2 ** 26 if dtype == "bf16" and kind in ("prefill", "train") else 2 ** 24
    most = max(1, min(64, cap // (T * H * N)))
    while T * H * N > cap:
        T = T * 3 // 4
    return _case(kind, _log_int(rng, 1, most), T, H, dtype=dtype, R=rng.choice([32, 64]) if kind == "train_mix" else 0)


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    kind, B, T, H = case["kind"], case["B"], case["T"], case["H"]
    C, dt = H * N, DTYPES[case["dtype"]]
    out_dt = torch.float32 if dt == torch.float16 else dt

    def normal(*shape, std=1.0, dtype=dt):
        return (torch.randn(*shape, generator=g, device=dev) * std).to(dtype)

    state = {"kind": kind, "op": RWKVKernelOperator(N, MAX_T)}
    if kind == "train_mix":
        # x is the output of a layer norm in bf16, the parameters are kept in fp32 as in a mixed-precision step, with the
        # spread the model's initialisation gives them
        R = case["R"]
        f32 = torch.float32
        state["leaves"] = [normal(B, T, C), torch.rand(C, generator=g, device=dev), normal(5 * R, C, std=0.5 / C ** 0.5, dtype=f32),
                           normal(5, C, R, std=0.5 / R ** 0.5, dtype=f32), normal(5, C, std=0.3, dtype=f32)]
        state["gout"] = [normal(B, T, C) for _ in range(5)]
        for x in state["leaves"]:
            x.requires_grad_(True)
        return state
    r, k, v = (normal(B, T, C) for _ in range(3))
    w = (torch.rand(B, T, C, generator=g, device=dev) * 7.0 - 6.0).to(dt)
    leaves = [r, k, v, w, normal(H, N, std=0.5)]
    if kind.endswith("_fused"):
        gate = torch.nn.functional.silu(torch.randn(B, T, C, generator=g, device=dev)).to(dt)
        leaves += [gate, 1.0 + normal(H, N, std=0.2, dtype=torch.float32), normal(H, N, std=0.2, dtype=torch.float32)]
    state["leaves"] = leaves
    if kind.startswith("train"):
        state["gout"] = normal(B, T, C, dtype=out_dt)
        for x in leaves:
            x.requires_grad_(True)
    else:
        state["s0"] = normal(B, H, N, N, dtype=torch.float32)
    return state


def run(state):
    kind, op, leaves = state["kind"], state["op"], state["leaves"]
    if kind in ("decode", "prefill"):
        return op(*leaves, return_state=True, init_state=state["s0"])
    if kind in ("decode_fused", "prefill_fused"):
        return op.forward_gn_gate(*leaves, return_state=True, init_state=state["s0"])
    if kind == "train":
        y, _ = op(*leaves)
        return [y, *torch.autograd.grad(y, leaves, state["gout"])]
    if kind == "train_fused":
        out, _ = op.forward_gn_gate(*leaves)
        return [out, *torch.autograd.grad(out, leaves, state["gout"])]
    outs = op.shift_mix(*leaves)
    return [*outs, *torch.autograd.grad(outs, leaves, state["gout"])]


def work(case):
    kind, B, T, H = case["kind"], case["B"], case["T"], case["H"]
    C, es = H * N, 2 if case["dtype"] == "bf16" else 4
    n, es_in = B * T * C, 4 if case["dtype"] == "f32" else 2
    if kind == "train_mix":
        # x and five gradients in, five outputs and x's gradient out, the weights and their gradients; the products
        # with the two mixer matrices, their gradients by input and by weight
        R = case["R"]
        return {"bytes": 12 * n * 2 + 2 * (2 * 5 * R * C + 5 * C + C) * 4, "flops": 6 * 2 * B * T * C * 5 * R}
    # forward: per token and head the state times a vector, its decay and its rank-one update, 6 N^2
    flops, fused = 6 * n * N, kind.endswith("_fused")
    if kind.startswith("train"):
        # r, k, v, w and the arriving gradient in, the output and four gradients out (with the gate: it and its
        # gradient too); the state and the reverse state against three vectors each: 14 N^2 more
        return {"bytes": n * (4 * es_in + 6 * es) + (2 * n * es if fused else 0), "flops": flops + 14 * n * N}
    return {"bytes": n * (4 * es_in + es) + (n * es if fused else 0) + 2 * B * H * N * N * 4, "flops": flops}


def tolerance(case):
    # About four times the largest relative error of any output against float64 on the same inputs, measured:
    # f32 4.2e-6 (gw; the others 2e-7); f16 2.1e-4 (the gradients' own rounding); bf16 3.9e-3 for the operator and
    # 4.3e-3 for the input side.  Group norm divides by a head's spread, which magnifies the rounding of y where
    # that spread is small: 1.1e-2 on u's gradient.
    if case["dtype"] == "f32":
        return {"rel": 2e-5}
    if case["dtype"] == "f16":
        return {"rel": 1e-3}
    return {"rel": 4e-2 if case["kind"] == "train_fused" else 1.6e-2}
