"""Cases that stand for what this library is used for: CSR SpMM, CSR-sampled SDDMM and the fused SDDMM -> SpMM, called
from Python on device tensors.

A case is one matrix (M x K, how its nonzeros lie), one dense width and one way of calling:
  call "prepared"  the lead path: dlspm_analyze and dlspm_advise once per matrix (dl.prepare), the output tensor kept;
  call "plain"     the drop-in call: no plan, no memory, a new output tensor each time.
rows "uniform"     every position with the same probability (random and magnitude pruning);
     "lognormal"   row lengths spread lognormally (sigma 0.6; magnitude-pruned layers with uneven rows);
     "topk"        the same number of nonzeros in every row (per-row top-k pruning);
     "window"      a band of `band` columns that moves with the row plus random columns (sparse attention).
"""
import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "dlspm-esimd_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)
import dlspm_hip as dl  # noqa: E402

_OPS = {"spmm": dl.OP_SPMM, "sddmm": dl.OP_SDDMM, "fused": dl.OP_FUSED}
_SIGMA = 0.6
_BLOCK = 1 << 26  # positions of a mask drawn at a time


def _case(op, M, K, width, density, rows, call, band=0):
    return {"op": op, "M": M, "K": K, "width": width, "density": density, "rows": rows, "band": band, "call": call}


def listed():
    return [
        # SpMM: weight matrix times activations.
        # A pruned attention projection at a short sequence: the smallest call, all latency (benchmark configuration 1).
        dict(_case("spmm", 512, 512, 128, 0.3, "uniform", "prepared"), name="spmm_projection_small"),
        # A feed-forward layer pruned to 90 % with uneven rows: the headline benchmark (configuration 2).
        dict(_case("spmm", 2048, 512, 256, 0.1, "lognormal", "prepared"), name="spmm_ffn_uneven_rows"),
        # Top-k pruned layer on a width between the powers of two (configuration 4).
        dict(_case("spmm", 2048, 512, 392, 0.2, "topk", "prepared"), name="spmm_ffn_topk_w392"),
        # A pruned convolution layer of ResNet-50 at a batch of images: few rows, a wide activation matrix.
        dict(_case("spmm", 256, 2304, 3136, 0.1, "uniform", "plain"), name="spmm_conv_wide"),
        # The benchmark grid, a square matrix at its lowest density and the largest matrix at its highest.
        dict(_case("spmm", 8192, 8192, 128, 0.1, "uniform", "prepared"), name="spmm_grid_square"),
        dict(_case("spmm", 32768, 8192, 128, 0.3, "uniform", "prepared"), name="spmm_grid_largest"),
        # SDDMM: sampled scores, and the gradient of a sparse weight's values.
        # The mask of configuration 3.
        dict(_case("sddmm", 2048, 2048, 128, 0.05, "uniform", "prepared"), name="sddmm_mask_2048"),
        # Odd sizes, uneven rows, a head dimension between the powers of two.
        dict(_case("sddmm", 3001, 4499, 80, 0.03, "lognormal", "prepared"), name="sddmm_ragged_d80"),
        # The benchmark grid at its narrow width, called as a drop-in.
        dict(_case("sddmm", 24576, 8192, 32, 0.2, "uniform", "plain"), name="sddmm_grid_narrow"),
        # Fused: one head of sparse attention.
        # Local window plus random columns (configuration 5).
        dict(_case("fused", 4096, 4096, 64, 48 / 4096, "window", "prepared", band=32), name="fused_window_4096"),
        # A long sequence with a wide window, called as a drop-in.
        dict(_case("fused", 16384, 16384, 128, 0.0, "window", "plain", band=128), name="fused_long_window"),
        # The benchmark grid: operands beyond one L2.
        dict(_case("fused", 8192, 8192, 128, 0.1, "uniform", "prepared"), name="fused_grid_square"),
    ]


_GRID_M = (1024, 3072, 4096, 2048, 6144, 8192, 12288, 16384, 24576, 32768)
_GRID_K = (1024, 2048, 4096, 8192)
_MOST = 32768 * 8192 * 0.3 * 128  # gathered floats of the largest listed case


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _log(rng, low, high):
    return round(math.exp(rng.uniform(math.log(low), math.log(high))), 5)


def _gathered(case):
    return (2 if case["op"] == "fused" else 1) * _nnz(case) * case["width"]


def draw(rng):
    while True:
        case = _draw(rng)
        if _gathered(case) <= _MOST:
            return case


def _draw(rng):
    kind = rng.choice(("layer", "conv", "grid", "attention"))
    call = rng.choice(("prepared", "plain"))
    if kind == "layer":  # pruned linear layers: sizes of any parity, 2 ... 50 % dense
        return _case(rng.choice(("spmm", "spmm", "sddmm")), _log_int(rng, 64, 4096), _log_int(rng, 64, 4096),
                     _log_int(rng, 16, 512), _log(rng, 0.02, 0.5), rng.choice(("uniform", "lognormal", "topk")), call)
    if kind == "conv":  # pruned convolutions: few output channels, many pixels
        M, K, N = _log_int(rng, 64, 2048), _log_int(rng, 64, 4608), 49 * _log_int(rng, 1, 256)
        return _case("spmm", M, K, N, _log(rng, 0.02, 0.5), rng.choice(("uniform", "lognormal")), call)
    if kind == "grid":  # the benchmark grid's matrices and densities, its widths and those between and above them
        op = rng.choice(("spmm", "sddmm", "fused"))
        return _case(op, rng.choice(_GRID_M) - rng.randrange(0, 64), rng.choice(_GRID_K) - rng.randrange(0, 64),
                     rng.choice((32, 128, _log_int(rng, 16, 256))), rng.choice((0.1, 0.2, 0.3)),
                     rng.choice(("uniform", "uniform", "lognormal")), call)
    # attention masks: windows with random columns, or random columns alone
    L, D = _log_int(rng, 1024, 16384), rng.choice((32, 64, 80, 96, 128, 256))
    rows = rng.choice(("window", "window", "uniform"))
    band = 2 * _log_int(rng, 8, 128) if rows == "window" else 0
    density = round((_log_int(rng, 8, 64) if rows == "window" else _log_int(rng, 16, 256)) / L, 6)
    return _case(rng.choice(("sddmm", "fused", "fused")), L, L, D, density, rows, call, band)


def _band(case):
    """First column and end of every row's band, as int64 tensors on the CPU (rows without a band: empty)."""
    M, K, half = case["M"], case["K"], case["band"] // 2
    i = torch.arange(M) * K // M
    return (i - half).clamp_(min=0), (i + half).clamp_(max=K)


def _structure(case, g):
    """row_offsets and col_indices (int32, columns ascending) on the GPU, _nnz(case) nonzeros in all."""
    M, K, dev = case["M"], case["K"], "cuda"
    first, end = (t.to(dev).unsqueeze(1) for t in _band(case))
    in_band = int((end - first).sum())
    wanted = _nnz(case) - in_band
    # a few more positions than wanted, of which some are then left out
    density = wanted / (M * K - in_band)
    share = torch.full((M, 1), density, device=dev)
    if case["rows"] == "lognormal":
        share *= torch.exp(_SIGMA * torch.randn((M, 1), device=dev, generator=g))
        for _ in range(6):
            share = (share * (density / share.mean())).clamp_(max=1.0)
    share *= 1.01 + 6.0 / math.sqrt(max(wanted, 1))
    positions = []
    step = max(1, _BLOCK // K)
    j = torch.arange(K, device=dev).unsqueeze(0)
    for r0 in range(0, M, step):
        r1 = min(M, r0 + step)
        u = torch.rand((r1 - r0, K), device=dev, generator=g)
        if case["rows"] == "topk":
            keep = torch.zeros((r1 - r0, K), dtype=torch.bool, device=dev)
            keep.scatter_(1, torch.topk(u, wanted // M, dim=1).indices, True)
        else:
            keep = u < share[r0:r1]
            if case["band"]:
                keep &= (j < first[r0:r1]) | (j >= end[r0:r1])
        positions.append(keep.view(-1).nonzero().view(-1) + r0 * K)
    position = torch.cat(positions)
    del positions, u, keep
    excess = position.numel() - wanted
    if excess > 0:
        stride = position.numel() // excess
        out = torch.arange(excess, device=dev) * stride + torch.randint(0, stride, (excess,), device=dev, generator=g)
        left = torch.ones(position.numel(), dtype=torch.bool, device=dev)
        left[out] = False
        position = position[left]
    if case["band"]:
        band = ((j >= first) & (j < end)).view(-1).nonzero().view(-1)
        position = torch.cat((position, band)).sort().values
    row_offsets = torch.searchsorted(position, torch.arange(M + 1, device=dev) * K).to(torch.int32)
    return row_offsets, (position % K).to(torch.int32)


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    M, K, width, op = case["M"], case["K"], case["width"], case["op"]
    row_offsets, col_indices = _structure(case, g)
    normal = lambda *shape: torch.randn(shape, device="cuda", generator=g)  # noqa: E731
    nnz = col_indices.numel()
    if op == "spmm":
        # weights, and activations behind a rectifier: half of them zero
        dense = (0.05 * normal(nnz), normal(K, width).clamp_(min=0.0))
    elif op == "sddmm":
        dense = (normal(M, width), normal(K, width))
    else:
        dense = (normal(M, width), normal(K, width), normal(K, width))
    state = {"op": op, "matrix": (row_offsets, col_indices), "dense": dense, "scale": 1.0 / math.sqrt(width), "plan": None, "out": None}
    if case["call"] == "prepared":
        state["plan"] = dl.prepare(row_offsets, col_indices, K, _OPS[op], width)
        state["out"] = torch.empty((nnz,) if op == "sddmm" else (M, width), device="cuda")
    return state


def run(state):
    matrix, dense, plan, out = state["matrix"], state["dense"], state["plan"], state["out"]
    if state["op"] == "spmm":
        return dl.spmm(*matrix, *dense, out=out, plan=plan)
    if state["op"] == "sddmm":
        return dl.sddmm(*matrix, *dense, out=out, plan=plan)
    return dl.fused(*matrix, *dense, state["scale"], out=out, plan=plan)


def _nnz(case):
    """Number of nonzeros: the same for every seed."""
    M, K = case["M"], case["K"]
    if case["rows"] == "topk":
        return M * max(1, int(case["density"] * K))
    first, end = _band(case)
    in_band = int((end - first).sum())
    return max(1, in_band + int(case["density"] * (M * K - in_band)))


def work(case):
    """Every operand read once, every result written once; a multiply and an add per nonzero and column."""
    M, K, width, nnz = case["M"], case["K"], case["width"], _nnz(case)
    if case["op"] == "spmm":
        return {"bytes": 4.0 * (M + 1) + 8.0 * nnz + 4.0 * (K + M) * width, "flops": 2.0 * nnz * width}
    if case["op"] == "sddmm":
        return {"bytes": 4.0 * (M + 1) + 8.0 * nnz + 4.0 * (K + M) * width, "flops": 2.0 * nnz * width}
    return {"bytes": 4.0 * (M + 1) + 4.0 * nnz + 4.0 * (2 * K + 2 * M) * width, "flops": 4.0 * nnz * width}


def tolerance(case):
    """Sums in 32-bit floats, in any order."""
    return {"rel": 1e-5}
