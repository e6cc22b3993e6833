"""The work this library is used for, as measurable cases.

A graph's plan (the SW32 format on the GPU) is built once and then multiplied with INT8 features over
and over: the SpMM cases. Fresh FP32 features are quantized and packed before each multiplication:
the layer and feature cases. Building the plan from a CSR is host work done once per graph, in
prepare(). Graph sizes and distributions follow the library's synthetic configurations (uniform,
community, banded and hub matrices) and its small test matrices; odd and ragged sizes are generic.

Matrices are drawn on the GPU from the seed, duplicates dropped, and go through make_canonical_csr
and convert_csr_to_sw32 as a user's matrix does.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import tcc_spmm_amd as T
from tcc_spmm_amd.device import (TorchDeviceMatrix, pack_features_int8x16,
                                 quantize_features_int8, quantize_pack_features_int8)

DEVICE = "cuda"


# --------------------------------------------------------------------------------------------------
# Cases


def listed() -> list[dict]:
    return [
        # The smallest call: one mini-batch's rows against a few thousand sources. Launch and host
        # time are everything.
        spmm("tiny_f128", "uniform", 300, 4000, 25, 128),
        # A small uniform graph that leaves most of the chip idle.
        spmm("uniform_4k_f128", "uniform", 4096, 4096, 16, 128),
        # A sampled mini-batch's layer: few rows, many more sources, fresh features of all of them.
        spmm("batch_10k_f128", "uniform", 10007, 100003, 25, 128, op="layer"),
        # One layer on a small citation-like graph with fresh features: quantize, pack, multiply.
        spmm("layer_20k_f256", "community", 20011, 20011, 12, 256, op="layer"),
        # An ordinary graph of about a hundred thousand nodes, row count not a multiple of 32.
        spmm("banded_100k_f128", "banded", 100003, 100003, 20, 128),
        # A medium power-law graph with communities, both widths; the wide one through the entry
        # point that takes no workspace (serving under graph capture).
        spmm("community_262k_f128", "community", 262144, 262144, 32, 128),
        spmm("community_262k_f256", "community", 262144, 262144, 32, 256, op="noalloc"),
        # A large product graph, both widths: the headline workload.
        spmm("banded_2m_f128", "banded", 2449029, 2449029, 51.5, 128),
        spmm("banded_2m_f256", "banded", 2449029, 2449029, 51.5, 256),
        # A skewed graph with hub rows, empty rows and a row count that is not a multiple of 32.
        spmm("hub_1m_f256", "hub", 1000003, 1000003, 20, 256),
        # New features for the large graph, in one pass, before a multiplication.
        dict(name="quantize_pack_2m_f128", op="quantize_pack", sources=2449029, features=128),
        # Raw input features of an odd width, quantized only (packing needs multiples of 16).
        dict(name="quantize_300k_f50", op="quantize", sources=300007, features=50),
    ]


def spmm(name, graph, rows, cols, degree, features, op="spmm") -> dict:
    return dict(name=name, op=op, graph=graph, rows=rows, cols=cols, degree=float(degree),
                features=features)


def _log_int(rng, lo, hi) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    """A multiplication most of the time: 200 to 2.4M rows, mean degree 4 to 64 (at most 100M
    entries), square or a mini-batch's rectangle. Else new features of 1K to 2.4M sources."""
    what = rng.random()
    if what < 0.2:
        op = rng.choice(("quantize", "quantize_pack", "features"))
        features = rng.choice((32, 64, 128, 256, 512)) if op != "quantize" else rng.randint(16, 600)
        return dict(op=op, sources=_log_int(rng, 1000, min(2449029, 600_000_000 // features)),
                    features=features)
    graph = rng.choice(("uniform", "community", "banded", "hub"))
    rows = _log_int(rng, 200, 2400000)
    cols = _log_int(rng, 2000, 100000) if graph == "uniform" and rng.random() < 0.5 else rows
    degree = math.exp(rng.uniform(math.log(4), math.log(64)))
    degree = round(min(degree, cols / 8, 100_000_000 / rows), 1)
    op = rng.choice(("spmm", "spmm", "spmm", "layer"))
    return dict(op=op, graph=graph, rows=rows, cols=cols, degree=degree,
                features=rng.choice((128, 256)))


# --------------------------------------------------------------------------------------------------
# Inputs


def _generator(seed: int) -> torch.Generator:
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _hubs(case) -> tuple[int, int]:
    """Hub rows and their degree: 64 rows of 15% of the columns at a million rows, fewer below."""
    return max(1, min(64, case["rows"] // 15625)), max(1, int(case["cols"] * 0.15))


def _degrees(case, g) -> torch.Tensor:
    """Row degrees: a Pareto tail scaled to the mean degree (power-law graphs), or constant."""
    rows, mean, graph = case["rows"], case["degree"], case["graph"]
    if graph == "uniform":
        return torch.full((rows,), int(mean), dtype=torch.int64, device=DEVICE)
    alpha, top = {"community": (2.1, 20000), "banded": (2.65, 17000), "hub": (1.8, 250000)}[graph]
    top = max(1, min(top, case["cols"] // 4))
    u = 1.0 - torch.rand(rows, dtype=torch.float64, device=DEVICE, generator=g)
    z = torch.floor(u.pow(-1.0 / (alpha - 1.0)))
    low, high = 1e-4, 1e6
    for _ in range(60):  # the scale at which the clipped degrees have the wanted mean
        k = math.sqrt(low * high)
        small = float((z * k).round().clamp(1, top).mean()) < mean
        low, high = (k, high) if small else (low, k)
    degrees = (z * math.sqrt(low * high)).round().clamp(1, top).to(torch.int64)
    if graph == "hub":
        degrees[torch.rand(rows, device=DEVICE, generator=g) < 0.05] = 0
        count, degree = _hubs(case)
        degrees[torch.randperm(rows, device=DEVICE, generator=g)[:count]] = degree
    return degrees


def _matrix(case, g):
    """(row offsets, columns, values) of the case's matrix, int64 and float32 tensors on the GPU."""
    rows, cols, graph = case["rows"], case["cols"], case["graph"]
    degrees = _degrees(case, g)
    row = torch.repeat_interleave(torch.arange(rows, device=DEVICE), degrees)
    n = row.numel()
    col = torch.randint(cols, (n,), device=DEVICE, generator=g)
    if graph == "community":  # 70% inside the row's block of 4,096 sources
        at = (row & ~4095) + (col & 4095)
        near = torch.rand(n, device=DEVICE, generator=g) < 0.7
        col = torch.where(near & (at < cols), at, col)
    elif graph == "banded":  # 60% at a log-uniform distance of up to 32,768 rows
        r = torch.rand(n, device=DEVICE, generator=g)
        far = torch.exp(torch.rand(n, device=DEVICE, generator=g) * math.log(32768.0)).floor_()
        at = row + torch.where(r < 0.3, far, -far).to(torch.int64)
        col = torch.where((r < 0.6) & (at >= 0) & (at < cols), at, col)
    key = torch.unique(row.mul_(cols).add_(col))
    del row, col
    row = torch.div(key, cols, rounding_mode="floor")
    col = key - row * cols
    counts = torch.bincount(row, minlength=rows)
    if graph in ("community", "banded"):  # symmetric normalisation of the adjacency matrix
        inv = counts.clamp(min=1).to(torch.float32).rsqrt()
        val = inv[row] * inv[col.clamp(max=rows - 1)]
    else:
        val = 2.0 * torch.rand(key.numel(), device=DEVICE, generator=g) - 1.0
        val = torch.where(val == 0, torch.ones_like(val), val)
    offsets = torch.zeros(rows + 1, dtype=torch.int64, device=DEVICE)
    torch.cumsum(counts, 0, out=offsets[1:])
    return offsets, col, val


def _features(sources, features, g, outliers=False) -> torch.Tensor:
    """N(0, 1) features; hub graphs have N(0, 4) ones with 1% of the rows a hundred times larger."""
    x = torch.randn((sources, features), device=DEVICE, generator=g)
    if outliers:
        large = torch.rand((sources, 1), device=DEVICE, generator=g) < 0.01
        x *= torch.where(large, 200.0, 2.0)
    return x


def _csr(case, matrix):
    offsets, col, val = matrix
    return T.make_canonical_csr(case["rows"], case["cols"],
                                offsets.to(torch.int32).cpu().numpy().view(np.uint32),
                                col.to(torch.int32).cpu().numpy().view(np.uint32),
                                val.cpu().numpy())


def prepare(case, seed):
    g = _generator(seed)
    op = case["op"]
    if "sources" in case:
        n, f = case["sources"], case["features"]
        return dict(op=op, x=_features(n, f, g),
                    q=torch.empty((n, f), dtype=torch.int8, device=DEVICE),
                    packed=torch.empty((n, f), dtype=torch.int8, device=DEVICE),
                    scale=torch.empty(n, device=DEVICE))
    rows, cols = case["rows"], case["cols"]
    csr = _csr(case, _matrix(case, g))
    f = case["features"]
    matrix = TorchDeviceMatrix(T.convert_csr_to_sw32(rows, cols, csr), f, device=DEVICE)
    x = _features(cols, f, g, outliers=case["graph"] == "hub")
    packed, scale = quantize_pack_features_int8(x)
    return dict(op=op, matrix=matrix, x=x if op == "layer" else None, packed=packed, scale=scale,
                y=torch.empty((rows, f), device=DEVICE))


# --------------------------------------------------------------------------------------------------
# One pass


def run(state):
    op = state["op"]
    if op == "spmm":
        return state["matrix"].spmm(state["packed"], state["scale"], state["y"])
    if op == "noalloc":
        return state["matrix"].spmm_noalloc(state["packed"], state["scale"], state["y"])
    if op == "layer":
        packed, scale = quantize_pack_features_int8(state["x"], state["packed"], state["scale"])
        return packed, scale, state["matrix"].spmm(packed, scale, state["y"])
    if op == "quantize":
        return quantize_features_int8(state["x"], state["q"], state["scale"])
    if op == "quantize_pack":
        return quantize_pack_features_int8(state["x"], state["packed"], state["scale"])
    q, scale = quantize_features_int8(state["x"], state["q"], state["scale"])
    return q, scale, pack_features_int8x16(q, state["packed"])


def work(case):
    """Bytes and operations of one pass: matrix entries (source and value) and row offsets, features,
    scales and results once each."""
    if "sources" in case:
        n, f = case["sources"], case["features"]
        return dict(bytes=n * (4 * f + f + 4) + (n * f if case["op"] == "features" else 0), flops=0)
    rows, cols = case["rows"], case["cols"]
    nnz = rows * case["degree"]
    if case["graph"] == "hub":
        nnz += math.prod(_hubs(case))
    f = case["features"]
    x = cols * (f + 4) + (cols * 4 * f if case["op"] == "layer" else 0)
    return dict(bytes=int(8 * nnz + 4 * rows + x + 4 * rows * f), flops=int(2 * nnz * f))


def tolerance(case):
    """Quantized bytes and scales are defined to the bit. Y is a sum of exact products in
    FP32: another order of the additions moves it by a few units in the last place."""
    if case["op"] in ("quantize", "quantize_pack", "features"):
        return "exact"
    # Sums in another order differ from these by rel 1e-7 to 7e-7 (hub rows of 150,000 terms the
    # most); single results near zero by more of the root mean square.
    return {"rel": 3e-6, "max": 1e-3, "differ": 0.0}


# --------------------------------------------------------------------------------------------------
# The same in 64 bits


def _scales(x: torch.Tensor) -> torch.Tensor:
    """Largest magnitude of each row / 127, by a true division (a scalar divisor is multiplied by
    its rounded reciprocal)."""
    top = x.abs().amax(1, keepdim=True)
    return top / torch.full_like(top, 127.0)


def _tf32(v: torch.Tensor) -> torch.Tensor:
    """FP32 rounded to TF32's ten explicit mantissa bits, ties away from zero."""
    return ((v.view(torch.int32) + 0x1000) & -0x2000).view(torch.float32)


def exact(case, seed):
    """Y = tf32(A) x tf32(dequantized X) with the products and sums in 64 bits; scales in 64 bits."""
    g = _generator(seed)
    if "sources" in case:
        x = _features(case["sources"], case["features"], g)
        scale = x.abs().amax(1).double() / 127.0
        return (None, scale, None) if case["op"] == "features" else (None, scale)
    offsets, col, val = _matrix(case, g)
    rows, f = case["rows"], case["features"]
    x = _features(case["cols"], f, g, outliers=case["graph"] == "hub")
    scale = _scales(x)
    x = _tf32((x / scale).round_().clamp_(-127, 127) * scale)
    val = _tf32(val)
    counts = offsets[1:] - offsets[:-1]
    row = torch.repeat_interleave(torch.arange(rows, device=DEVICE), counts)
    y = torch.zeros((rows, f), dtype=torch.float64, device=DEVICE)
    step = max(1, (1 << 28) // f)
    for at in range(0, col.numel(), step):
        part = slice(at, at + step)
        y.index_add_(0, row[part], x[col[part]].double() * val[part].double().unsqueeze(1))
    if case["op"] == "layer":
        return None, scale.view(-1).double(), y
    return y
