"""What the performance of this package is measured on: listed cases and a generator of more.

Every case is one attention forward through a public entry point of `cuda_attn`, as a program calls
it: q, k and v are on the GPU, the output is a new tensor. Sizes are the package's own benchmark
configurations (cuda_attn/workloads.py), the shapes of its benchmark sweeps (bench/benchmark.py,
bench/sweep_tiles.py) and of its parity tests.
"""
from __future__ import annotations

import math
import os
import random
import sys

import torch

_PKG = os.path.join(os.getcwd(), "phantom-a100_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import cuda_attn  # noqa: E402

_DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_TILES = ((64, 32), (64, 64), (128, 32), (128, 64))


def _case(entry, dtype, b, h, n, d, causal=False, qk_scale=1.0, out_f32=False, br=0, bc=0, name=None):
    c = {"entry": entry, "dtype": dtype, "b": b, "h": h, "n": n, "d": d, "causal": causal,
         "qk_scale": qk_scale, "out_f32": out_f32, "br": br, "bc": bc}
    return c if name is None else {"name": name, **c}


def listed():
    return [
        # The smallest benchmark configuration: one slice of short rows, where launch latency and
        # the host path count.
        _case("fused_tc", "f16", 1, 42, 128, 64, out_f32=True, name="tc_f16_d64_42x128"),
        # An ordinary encoder layer: a batch of 1024-token rows.
        _case("fused_tc", "f16", 8, 16, 1024, 64, name="tc_f16_d64_8x16x1024"),
        # The headline configuration: the long rows of a large decoder's head dim.
        _case("fused_tc", "bf16", 4, 32, 4096, 128, name="tc_bf16_d128_4x32x4096"),
        # One long document whose softmax rows are sharply peaked (the running max moves).
        _case("fused_tc", "f16", 1, 16, 8192, 64, qk_scale=3.0, out_f32=True, name="tc_f16_d64_1x16x8192_peaked"),
        # A training or batched prefill step of a decoder: causal rows.
        _case("fused_tc", "bf16", 4, 32, 2048, 128, causal=True, name="tc_bf16_d128_causal_4x32x2048"),
        # The prefill of one prompt of an odd length: a small causal grid, ragged rows.
        _case("fused_tc", "bf16", 1, 32, 1030, 128, causal=True, name="tc_bf16_d128_causal_1x32x1030"),
        # The smallest fp32 configuration.
        _case("fused", "f32", 1, 42, 128, 64, name="fused_f32_42x128"),
        # fp32 inputs at the benchmark sweep's middle size (a model kept in fp32).
        _case("fused", "f32", 4, 16, 2048, 64, name="fused_f32_4x16x2048"),
        # fp16 storage with fp32 arithmetic, causal, at the sweep's ordinary size.
        _case("fused", "f16", 4, 16, 1024, 64, causal=True, name="fused_f16_causal_4x16x1024"),
        # The tuned kernel at its default tile (fused_db): what the tile sweep starts from.
        _case("fused_db", "f16", 4, 16, 1024, 64, br=64, bc=32, name="db_f16_4x16x1024"),
        # The unfused matrix-core path at the sweep's middle size (a 1 GiB score workspace).
        _case("tiled", "f16", 4, 16, 2048, 64, name="tiled_f16_4x16x2048"),
        # The plain three-pass path as the cross-check of a small layer: odd rows, a head dim that
        # only the unfused entry points take.
        _case("naive", "f32", 2, 8, 333, 80, name="naive_f32_d80_2x8x333"),
    ]


# Entry point -> (share of the draws, largest FLOPs of a drawn case: at most its listed one's).
_SHARES = {"fused_tc": (10, 1.0e12), "fused": (4, 6.0e10), "fused_tuned": (1, 1.7e10), "fused_db": (1, 1.7e10),
           "fused_vec": (1, 1.7e10), "tiled": (2, 6.0e10), "naive": (1, 1.5e9)}


def draw(rng: random.Random):
    entry = rng.choices(list(_SHARES), [s for s, _ in _SHARES.values()])[0]
    most = _SHARES[entry][1]
    dtype, d, qk_scale, out_f32, br, bc = "f16", 64, rng.choice([1.0, 1.0, 1.0, 3.0]), False, 0, 0
    if entry == "fused_tc":
        dtype, d = rng.choice(["f16", "bf16"]), rng.choice([64, 128])
        out_f32 = rng.random() < 0.2
    elif entry in ("fused", "tiled", "naive"):
        dtype = rng.choice(["f32", "f16"])
        if entry == "fused":
            out_f32 = dtype == "f16" and rng.random() < 0.2
        else:
            d = rng.choice([32, 40, 64, 64, 80, 96, 128])
    else:
        br, bc = rng.choice(_TILES) if entry == "fused_tuned" else (64, 32)
    causal = rng.random() < 0.5
    # Row length over its logarithm, half of them multiples of 64 and half as they fall; then a
    # number of heads that keeps the case within its entry point's largest, also over its logarithm.
    n_most = {"naive": 600, "tiled": 4096}.get(entry, 8192)
    n = int(math.exp(rng.uniform(math.log(48), math.log(n_most))))
    if rng.random() < 0.5:
        n = max(64, n // 64 * 64)
    bh_most = min(512.0, most / (4.0 * n * n * d), 2.0 ** 27 / (n * d))
    if entry in ("tiled", "naive"):
        bh_most = min(bh_most, 2.0 ** 29 / (n * n))   # a score workspace of at most 2 GiB
    heads = max(1, int(math.exp(rng.uniform(0.0, math.log(max(1.0, bh_most))))))
    b = rng.choice([x for x in (1, 1, 2, 4, 8) if x <= heads])
    return _case(entry, dtype, b, max(1, heads // b), n, d, causal, qk_scale, out_f32, br, bc)


def _inputs(case, seed):
    """q, k, v: N(0, 1) draws, q and k times qk_scale, cast to the case's dtype."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    shape = (case["b"], case["h"], case["n"], case["d"])
    out = []
    for i in range(3):
        x = torch.randn(shape, dtype=torch.float32, device="cuda", generator=g)
        out.append((x * case["qk_scale"] if i < 2 else x).to(_DTYPES[case["dtype"]]))
    return out


def prepare(case, seed):
    q, k, v = _inputs(case, seed)
    kwargs = {"causal": case["causal"]}
    if case["entry"] == "fused_tuned":
        kwargs.update(br=case["br"], bc=case["bc"])
    if case["out_f32"]:
        kwargs["out_dtype"] = torch.float32
    return {"fn": getattr(cuda_attn, case["entry"]), "q": q, "k": k, "v": v, "kwargs": kwargs}


def run(state):
    return state["fn"](state["q"], state["k"], state["v"], **state["kwargs"])


def work(case):
    """q, k and v read once, the output written once; 4 d operations per visible (query, key)."""
    bh, n, d = case["b"] * case["h"], case["n"], case["d"]
    isz = 4 if case["dtype"] == "f32" else 2
    osz = 4 if case["out_f32"] else isz
    pairs = n * (n + 1) // 2 if case["causal"] else n * n
    return {"bytes": (3 * isz + osz) * bh * n * d, "flops": 4 * bh * pairs * d}


def tolerance(case):
    """About four times what two correct forwards at the case's precision differ by.

    Against 64 bits, fp32 arithmetic is seen 2.8e-7 to 1.2e-6 off (sums in some order); an fp16
    output adds its rounding (2.0e-4 to 2.9e-4). The 16-bit matrix-core entry points also round
    every probability to the input dtype before P.V: 0.8e-4 to 2.9e-4 (fp16), 2.0e-3 to 2.3e-3 (bf16).
    """
    if case["entry"] in ("fused", "tiled", "naive"):
        if case["dtype"] == "f32" or case["out_f32"]:
            return {"rel": 4e-6, "max": 1e-4}
        return {"rel": 1e-3, "max": 1e-2}
    if case["dtype"] == "bf16":
        return {"rel": 1e-2, "max": 1e-1}
    return {"rel": 2e-3, "max": 2e-2}


def exact(case, seed):
    q, k, v = _inputs(case, seed)
    b, h, n, d = q.shape
    out = torch.empty((b * h, n, d), dtype=torch.float64, device="cuda")
    q, k, v = (t.view(b * h, n, d) for t in (q, k, v))
    keys = torch.arange(n, device="cuda")
    for i in range(b * h):
        ki, vi = k[i].double(), v[i].double()
        for r in range(0, n, 2048):
            s = (q[i, r:r + 2048].double() @ ki.t()) / math.sqrt(d)
            if case["causal"]:
                s.masked_fill_(keys[None, :] > keys[r:r + 2048, None], -math.inf)
            out[i, r:r + 2048] = torch.softmax(s, dim=-1) @ vi
    return out.view(b, h, n, d)
