"""What a program does with this framework, as timed cases.

A case is one pass through the public entry points: ``hc.gfx950.gemm`` on
device tensors, the DSL's own call ``hc.simulator.launch(kernel, a, b, c)``,
the two products of a linear layer's backward, and the masked tile gather /
scatter.  Operands are float16 or bfloat16, sums and outputs float32.

``listed()`` are fixed cases, ``draw(rng)`` gives more of the same ranges
(sizes log-uniform, odd ones among them), ``prepare`` makes what a program
holds before the call (device tensors from the seed, and the output buffer it
reuses), ``run`` is the pass, ``exact`` the same result in 64 bits by plain
torch.
"""

from __future__ import annotations

import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "5_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import hc  # noqa: E402
import hc.gfx950 as g  # noqa: E402
from hc.gfx950 import kernels  # noqa: E402

DEV = "cuda"
_DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32, "int64": torch.int64}
_LAUNCH_KERNELS = {
    "float16": kernels.tiled_gfx950_mfma_matmul,
    "bfloat16": kernels.tiled_gfx950_mfma_matmul_bf16,
}
_MAX_FLOPS = 2 * 8192**3  # the largest listed product


def _gemm(name, m, n, k, dtype, dist):
    return {"name": name, "path": "gemm", "m": m, "n": n, "k": k, "dtype": dtype, "dist": dist}


def listed():
    return [
        # The smallest call: the reference example's CPU-runnable size, where
        # the launch and the host's share count.
        _gemm("small_128_f16", 128, 128, 128, "float16", "normal"),
        # The DSL's launch surface on device tensors at an ordinary small size:
        # binding and validation in Python, then the product.
        {"name": "launch_512_f16", "path": "launch", "m": 512, "n": 512, "k": 512, "dtype": "float16",
         "dist": "uniform"},
        # An ordinary square product, too small to fill the chip with the
        # largest tiles.
        _gemm("square_2048_bf16", 2048, 2048, 2048, "bfloat16", "uniform"),
        # The headline: a square, compute-bound product.
        _gemm("square_4096_f16", 4096, 4096, 4096, "float16", "uniform"),
        # The largest: several tiles per CU.
        _gemm("square_8192_bf16", 8192, 8192, 8192, "bfloat16", "weights"),
        # Masked tails in every extent, rows aligned to nothing but an element.
        _gemm("ragged_4095x3001x1027_f16", 4095, 3001, 1027, "float16", "uniform"),
        # Decoding: a few rows against a large weight, bound by reading it ...
        _gemm("decode_16x8192x8192_f16", 16, 8192, 8192, "float16", "layer"),
        # ... and a full decode batch, between the bandwidth and the matrix cores.
        _gemm("batch_128x8192x8192_bf16", 128, 8192, 8192, "bfloat16", "layer"),
        # Many rows onto a few columns (a router, a low-rank projection).
        _gemm("narrow_65536x8x4096_bf16", 65536, 8, 4096, "bfloat16", "layer"),
        # A small output over a long contraction (Gram matrices, weight
        # gradients of many tokens).
        _gemm("long_k_512x512x16384_f16", 512, 512, 16384, "float16", "normal"),
        # Backward of y = x @ w: dx = dy @ w^T and dw = x^T @ dy, with the
        # transposes as views, as an autograd function writes them.
        {"name": "backward_4096x2048x2048_bf16", "path": "backward", "m": 4096, "n": 2048, "k": 2048,
         "dtype": "bfloat16", "dist": "layer"},
        # Masked tiles of a ragged matrix, gathered and scattered into another.
        {"name": "tiles_64x64_of_4095x3001_f16", "path": "tiles", "m": 4095, "n": 3001, "th": 64, "tw": 64,
         "mask": False, "dtype": "float16"},
    ]


def _size(rng, lo, hi):
    """Log-uniform in [lo, hi]; one in three is left as it falls (often odd),
    the others are a multiple of 8, or of 64 where that large."""
    v = lo * (hi / lo) ** rng.random()
    kind = rng.randrange(3)
    unit = 1 if kind == 0 else (8 if kind == 1 or v < 256 else 64)
    return int(min(hi, max(lo, round(v / unit) * unit)))


def draw(rng):
    dtype = rng.choice(["float16", "bfloat16"])
    kind = rng.choice(["general", "general", "general", "launch", "decode", "batch", "narrow", "long_k", "backward",
                       "tiles"])
    dist = rng.choice(["uniform", "normal", "layer"])
    if kind == "launch":
        m, n, k = (_size(rng, 16, 1024) for _ in range(3))
        return {"path": "launch", "m": m, "n": n, "k": k, "dtype": dtype, "dist": dist}
    if kind == "tiles":
        return {"path": "tiles", "m": _size(rng, 256, 8192), "n": _size(rng, 256, 8192),
                "th": rng.choice([16, 32, 64, 128, 37]), "tw": rng.choice([16, 32, 64, 128, 37]),
                "mask": rng.random() < 0.5, "dtype": rng.choice(["float16", "bfloat16", "float32", "int64"])}
    if kind == "backward":
        return {"path": "backward", "m": _size(rng, 256, 8192), "n": _size(rng, 256, 4096),
                "k": _size(rng, 256, 4096), "dtype": dtype, "dist": "layer"}
    if kind == "general":
        m, n, k = (_size(rng, 65, 8192) for _ in range(3))
    elif kind == "decode":
        m, n, k = _size(rng, 1, 64), _size(rng, 1024, 16384), _size(rng, 1024, 16384)
    elif kind == "batch":
        m, n, k = _size(rng, 65, 512), _size(rng, 1024, 16384), _size(rng, 1024, 16384)
    elif kind == "narrow":
        m, n, k = _size(rng, 2048, 65536), _size(rng, 1, 64), _size(rng, 512, 16384)
        k = min(k, (1 << 28) // m)
    else:
        m, n, k = _size(rng, 65, 1024), _size(rng, 65, 1024), _size(rng, 4096, 65536)
    while 2 * m * n * k > _MAX_FLOPS:
        k = max(65, k // 2)
    return {"path": "gemm", "m": m, "n": n, "k": k, "dtype": dtype, "dist": dist}


def _values(gen, shape, dtype, kind):
    if kind == "uniform":
        x = torch.rand(shape, generator=gen, device=DEV) * 2 - 1
    else:
        x = torch.randn(shape, generator=gen, device=DEV)
        if kind == "weight":
            x *= 0.02
    return x.to(dtype)


def _operands(case, seed):
    """The tensors of a product: (a, b), or (x, w, dy) of a backward."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    dt = _DTYPES[case["dtype"]]
    m, n, k = case["m"], case["n"], case["k"]
    # "layer": activations N(0, 1) against weights N(0, 0.02^2); "weights":
    # both N(0, 0.02^2).
    a_kind = {"uniform": "uniform", "normal": "normal", "layer": "normal", "weights": "weight"}[case["dist"]]
    b_kind = {"uniform": "uniform", "normal": "normal", "layer": "weight", "weights": "weight"}[case["dist"]]
    a = _values(gen, (m, k), dt, a_kind)
    b = _values(gen, (k, n), dt, b_kind)
    if case["path"] != "backward":
        return a, b
    return a, b, _values(gen, (m, n), dt, "weight")


def _tile_source(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    dt = _DTYPES[case["dtype"]]
    m, n, th, tw = case["m"], case["n"], case["th"], case["tw"]
    if dt == torch.int64:
        src = torch.randint(-(1 << 40), 1 << 40, (m, n), generator=gen, device=DEV)
    else:
        src = _values(gen, (m, n), dt, "normal")
    # The grid of tiles that covers the matrix: the last row and column of
    # tiles reach past it.
    r = torch.arange(0, m, th, device=DEV)
    c = torch.arange(0, n, tw, device=DEV)
    origins = torch.cartesian_prod(r, c).to(torch.int64).contiguous()
    mask = None
    if case["mask"]:
        mask = torch.rand((origins.shape[0], th, tw), generator=gen, device=DEV) < 0.8
    return src, origins, mask


def prepare(case, seed):
    if case["path"] == "tiles":
        src, origins, mask = _tile_source(case, seed)
        return {"path": "tiles", "src": src, "origins": origins, "mask": mask, "shape": (case["th"], case["tw"]),
                "dst": torch.zeros_like(src)}
    ops = _operands(case, seed)
    if case["path"] == "backward":
        return {"path": "backward", "x": ops[0], "w": ops[1], "dy": ops[2]}
    out = torch.empty((case["m"], case["n"]), dtype=torch.float32, device=DEV)
    state = {"path": case["path"], "a": ops[0], "b": ops[1], "c": out}
    if case["path"] == "launch":
        state["kernel"] = _LAUNCH_KERNELS[case["dtype"]]
    return state


def run(state):
    path = state["path"]
    if path == "gemm":
        return g.gemm(state["a"], state["b"], out=state["c"])
    if path == "launch":
        hc.simulator.launch(state["kernel"], state["a"], state["b"], state["c"])
        return state["c"]
    if path == "backward":
        dx = g.gemm(state["dy"], state["w"].t())
        dw = g.gemm(state["x"].t(), state["dy"])
        return dx, dw
    tiles, active = g.tile_load(state["src"], state["origins"], state["shape"], mask=state["mask"])
    g.tile_store(state["dst"], state["origins"], tiles, mask=active)
    return tiles, active, state["dst"]


def work(case):
    m, n = case["m"], case["n"]
    if case["path"] == "tiles":
        size = _DTYPES[case["dtype"]].itemsize
        th, tw = case["th"], case["tw"]
        ntiles = -(-m // th) * -(-n // tw)
        elems = ntiles * th * tw
        # Gather: the matrix, the origins and the mask in, tiles and activity
        # out.  Scatter: tiles, activity and origins in, the matrix out.
        gather = size * m * n + 16 * ntiles + (elems if case["mask"] else 0) + (size + 1) * elems
        scatter = (size + 1) * elems + 16 * ntiles + size * m * n
        return {"bytes": gather + scatter, "flops": 0}
    k = case["k"]
    if case["path"] == "backward":
        # dx (m x k) = dy @ w^T, dw (k x n) = x^T @ dy; 16-bit in, 32-bit out.
        return {"bytes": 2 * m * n + 2 * k * n + 4 * m * k + 2 * m * k + 2 * m * n + 4 * k * n,
                "flops": 4 * m * n * k}
    return {"bytes": 2 * m * k + 2 * k * n + 4 * m * n, "flops": 2 * m * n * k}


def tolerance(case):
    if case["path"] == "tiles":
        return "exact"  # copies
    # 32-bit sums of exact products: only the order of the additions is free.
    # Measured against the same sums in 64 bits: 0.8e-7 (k = 128) to 5.7e-7
    # (k = 8192 in one run); two orders differ by about 1.4 times that, and
    # the worst of 10^8 elements by about six times the typical one.
    return {"rel": 4e-6, "max": 4e-5}


def exact(case, seed):
    if case["path"] == "tiles":
        return None
    ops = [t.double() for t in _operands(case, seed)]
    if case["path"] == "backward":
        x, w, dy = ops
        return torch.mm(dy, w.t().contiguous()), torch.mm(x.t().contiguous(), dy)
    return torch.mm(ops[0], ops[1])
