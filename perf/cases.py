"""The work a program gives this library, as a list of cases that can be timed and compared.

Each case is one call of a public operator of the `beam` package on torch tensors:

    gemm    c = a @ b.T            beam.gemmrc
    splitk  c = a @ b.T            beam.gemmrc_splitk, tile and slice count left to the library
    ln      y = LayerNorm(a @ b.T) beam.gemmrc_ln
    nn      c = a @ b              beam.matmul, b stored [K, N]
    silu    c = a @ b.T, y = silu(x) in one call   beam.parallel_gemmrc_silu

`listed()` holds one representative of every range, `draw()` takes further cases out of the same ranges.
"""
import os
import sys

import torch  # before beam: both then use torch's HIP runtime

sys.path.insert(0, os.path.join(os.getcwd(), "general-nvgpu-testing_amd"))

from beam import _C  # noqa: E402

_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # one small layer: launch latency and the host's share of a call decide
        {"name": "gemm_512", "op": "gemm", "dtype": "fp16", "M": 512, "N": 512, "K": 512},
        # an ordinary layer, too small to fill the chip with large tiles
        {"name": "gemm_2048", "op": "gemm", "dtype": "bf16", "M": 2048, "N": 2048, "K": 2048},
        # the large square product that the benchmark quotes
        {"name": "gemm_8192", "op": "gemm", "dtype": "fp16", "M": 8192, "N": 8192, "K": 8192},
        # sizes that no tile divides, rows still 16-byte aligned
        {"name": "gemm_ragged", "op": "gemm", "dtype": "fp16", "M": 3000, "N": 5000, "K": 2000},
        # sizes as data sets have them: odd rows, columns and depth
        {"name": "gemm_odd", "op": "gemm", "dtype": "bf16", "M": 3001, "N": 5001, "K": 2001},
        # decoding: a few tokens through a wide projection, the weights are read once
        {"name": "gemm_decode", "op": "gemm", "dtype": "bf16", "M": 16, "N": 11008, "K": 4096},
        # a small output under a long sum
        {"name": "splitk_256", "op": "splitk", "dtype": "fp16", "M": 256, "N": 256, "K": 32768},
        # a short batch through a layer with LayerNorm, result waited for and checked (the default)
        {"name": "ln_small", "op": "ln", "dtype": "bf16", "M": 512, "N": 1024, "K": 1024, "check": True},
        # a full-size layer with LayerNorm inside a stream of other work
        {"name": "ln_4096", "op": "ln", "dtype": "fp16", "M": 4096, "N": 4096, "K": 4096, "check": False},
        # prefill: thousands of tokens through the same projection, weights stored [K, N]
        {"name": "nn_prefill", "op": "nn", "dtype": "bf16", "M": 4096, "N": 11008, "K": 4096},
        # a classifier's head: the number of classes is whatever it is
        {"name": "nn_head", "op": "nn", "dtype": "fp16", "M": 2048, "N": 1001, "K": 2000},
        # a layer that applies SiLU to another array on the way
        {"name": "silu_4096", "op": "silu", "dtype": "fp16", "M": 4096, "N": 4096, "K": 4096, "count": 1 << 24},
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], spread evenly over its logarithm."""
    v = lo * (hi / lo) ** rng.random()
    return max(step, min(hi, int(round(v / step)) * step))


_ODD_MOST = 2 * 3001 * 5001 * 2001  # flops of the largest drawn case whose rows are not 16-byte aligned


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "odd", "decode", "splitk", "ln", "ln", "nn", "nn_any", "silu"])
    dtype = rng.choice(["fp16", "bf16"])
    n_step = 8 if rng.random() < 0.7 else 1
    if kind == "gemm":
        return {"op": "gemm", "dtype": dtype, "M": _log(rng, 64, 8192), "N": _log(rng, 64, 8192, n_step), "K": _log(rng, 64, 8192, 8)}
    if kind == "odd":
        while True:
            M, N, K = (_log(rng, 33, 5001) for _ in range(3))
            if K % 8 and 2 * M * N * K <= _ODD_MOST:
                return {"op": "gemm", "dtype": dtype, "M": M, "N": N, "K": K}
    if kind == "decode":
        return {"op": "gemm", "dtype": dtype, "M": _log(rng, 1, 64), "N": _log(rng, 1024, 16384, 8), "K": _log(rng, 1024, 16384, 8)}
    if kind == "splitk":
        return {"op": "splitk", "dtype": dtype, "M": _log(rng, 16, 512), "N": _log(rng, 16, 512, n_step), "K": _log(rng, 4096, 65536, 8)}
    if kind == "ln":
        return {"op": "ln", "dtype": dtype, "M": _log(rng, 16, 8192), "N": _log(rng, 256, 8192, n_step), "K": _log(rng, 256, 8192, 8),
                "check": rng.random() < 0.5}
    if kind == "nn":
        return {"op": "nn", "dtype": dtype, "M": _log(rng, 16, 8192), "N": _log(rng, 64, 8192, 8), "K": _log(rng, 64, 8192, 8)}
    if kind == "nn_any":
        while True:
            M, N, K = (_log(rng, 33, 5001) for _ in range(3))
            if (N % 8 or K % 8) and 2 * M * N * K <= _ODD_MOST:
                return {"op": "nn", "dtype": dtype, "M": M, "N": N, "K": K}
    return {"op": "silu", "dtype": dtype, "M": _log(rng, 256, 8192), "N": _log(rng, 256, 8192, 8), "K": _log(rng, 256, 8192, 8),
            "count": _log(rng, 1 << 18, 1 << 26)}


def prepare(case, seed):
    """Activations ~ N(0, 1), weights ~ N(0, 1) / sqrt(K), LayerNorm's gamma ~ 1 + 0.1 N(0, 1) and beta ~ 0.1 N(0, 1)."""
    dtype = _DTYPES[case["dtype"]]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    M, N, K = case["M"], case["N"], case["K"]

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device="cuda", dtype=dtype)

    s = {"op": case["op"], "a": normal(M, K), "b": normal(K, N) if case["op"] == "nn" else normal(N, K)}
    s["b"] *= K ** -0.5
    s["c"] = torch.empty(M, N, device="cuda", dtype=dtype)
    if case["op"] == "ln":
        s["gamma"], s["beta"], s["check"] = 1 + 0.1 * normal(N), 0.1 * normal(N), case["check"]
    if case["op"] == "silu":
        s["x"] = normal(case["count"])
        s["y"] = torch.empty_like(s["x"])
    return s


def run(s):
    op = s["op"]
    if op == "gemm":
        _C.gemmrc(s["a"], s["b"], s["c"])
    elif op == "splitk":
        _C.gemmrc_splitk(s["a"], s["b"], s["c"])
    elif op == "ln":
        _C.gemmrc_ln(s["a"], s["b"], s["c"], s["gamma"], s["beta"], check=s["check"])
    elif op == "nn":
        _C.matmul(s["a"], s["b"], s["c"])
    else:
        _C.parallel_gemmrc_silu(s["a"], s["b"], s["c"], s["x"], s["y"])
        return s["c"], s["y"]
    return s["c"]


def work(case):
    M, N, K = case["M"], case["N"], case["K"]
    count = case.get("count", 0)
    vectors = 2 * N if case["op"] == "ln" else 0
    return {"bytes": 2 * (M * K + N * K + M * N + vectors + 2 * count), "flops": 2 * M * N * K}


def tolerance(case):
    """Four times the distance from the same product in 64 bits: 2.0e-4 in fp16, 1.6e-3 in bf16, the rounding of the
    16-bit result; the largest single difference is two units in its last place."""
    if case["dtype"] == "fp16":
        return {"rel": 8e-4, "max": 2e-3}
    return {"rel": 6.5e-3, "max": 1.6e-2}
