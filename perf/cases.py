"""The calls a user of the VCSR SpMM library makes, as measurable cases.

A case is a sparse matrix (one of four structures, with its size), the width O
of the dense operand and the way the product is called:

  overwrite   C = A*B over a built and uploaded format (`run_vcsr_spmm_gpu_ex`)
  accumulate  C zeroed, then C += A*B (`run_vcsr_spmm_gpu`, the reference
              harness's sequence)
  noalloc     C = A*B through the allocation-free entry point
              (`run_vcsr_spmm_gpu_noalloc`: serving loops, graph capture)
  csr         C = A*B on plain CSR arrays, no format build
              (`run_csr_wave_spmm_gpu`: a matrix that is used once or changes)
  first       everything a new matrix costs: CSR object, VCSR build, upload
              and one synchronous product

B and C are FP32 torch tensors on the GPU, handed to the library by address on
the null stream, which is torch's current stream.
"""
from __future__ import annotations

import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    name = "vcsr_spmm_amd"
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(
            name, os.path.join(_ROOT, "vcsr-spmm_amd", "__init__.py"))
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
        mod.load_library()
    return sys.modules[name]


# ------------------------------------------------------------------- cases
def listed():
    return [
        # The smallest call: a 4K x 4K matrix of 16 entries a row, 32 columns
        # (the repository's plumbing configuration).  Latency of one launch.
        dict(name="uniform-4k-o32", matrix="uniform", n=4096, row=16, block=1, O=32,
             call="overwrite"),
        # Banded FEM matrix, 3 unknowns a node, 64 entries a row: a few
        # vectors at once (block solvers), the headline width, a wide one.
        dict(name="banded-62k-o8", matrix="banded", n=62451, row=64, block=3, O=8,
             call="overwrite"),
        dict(name="banded-62k-o128", matrix="banded", n=62451, row=64, block=3, O=128,
             call="overwrite"),
        dict(name="banded-62k-o512", matrix="banded", n=62451, row=64, block=3, O=512,
             call="overwrite"),
        # 6 unknowns a node (shells) and a width that is not a multiple of 4.
        dict(name="banded6-30k-o50", matrix="banded", n=30000, row=60, block=6, O=50,
             call="overwrite"),
        # Circuit / graph matrix with power-law rows: narrow, the headline
        # width the way the reference's harness calls it, and an odd width
        # (class scores of a graph) from a serving loop.
        dict(name="powerlaw-322k-o8", matrix="powerlaw", n=321821, row=6, block=1, O=8,
             call="overwrite"),
        dict(name="powerlaw-322k-o128", matrix="powerlaw", n=321821, row=6, block=1, O=128,
             call="accumulate"),
        dict(name="powerlaw-100k-o47", matrix="powerlaw", n=100003, row=6, block=1, O=47,
             call="noalloc"),
        # The largest call: uniform random columns, B of 1 GB, no reuse.
        dict(name="uniform-1m-o256", matrix="uniform", n=1000000, row=16, block=1, O=256,
             call="overwrite"),
        # Dense 16 x 16 blocks at 5% (the matrix-core path).
        dict(name="blocks-16k-o512", matrix="blocks", n=16384, row=816, block=16, O=512,
             call="overwrite"),
        # A matrix used without a format build, power-law rows.
        dict(name="csr-powerlaw-100k-o64", matrix="powerlaw", n=100003, row=6, block=1, O=64,
             call="csr"),
        # A new matrix: build, upload and one product.
        dict(name="first-banded-20k-o32", matrix="banded", n=20001, row=64, block=3, O=32,
             call="first"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case: any structure, size, width (odd ones among them) and call."""
    matrix = rng.choice(["banded", "banded", "powerlaw", "powerlaw", "uniform", "blocks"])
    call = rng.choice(["overwrite", "overwrite", "overwrite", "accumulate", "noalloc", "csr",
                       "first"])
    if matrix == "banded":
        block = rng.choice([1, 2, 3, 3, 4, 6])
        n, row = _log_int(rng, 4000, 120000), rng.randint(18, 80)
    elif matrix == "powerlaw":
        block, n, row = 1, _log_int(rng, 10000, 400000), 6
    elif matrix == "uniform":
        block, n, row = 1, _log_int(rng, 4000, 1000000), rng.randint(4, 16)
    else:
        block, n = 16, 16 * _log_int(rng, 128, 1024)
        row = 16 * rng.randint(6, 51)
    if call == "noalloc" and matrix == "banded":
        call = "overwrite"  # long rows there can need more than its fixed scratch
    if call == "first":  # no dearer than the listed one
        n = min(n, max(16 * 128, 1280000 // row))
    width = _log_int(rng, 4, 512)
    if rng.random() < 0.25:  # widths are often powers of two
        width = 1 << rng.randint(2, 9)
    while n * row * width > 16000000 * 256 or n * width > 256000000:
        width = max(4, width // 2)
    if block > 1:
        n = n // block * block
    return dict(matrix=matrix, n=n, row=row, block=block, O=width, call=call)


# ---------------------------------------------------------------- matrices
# All structures are made on the GPU as sorted unique keys row * n + column.
def _degrees_powerlaw(n):
    """Zipf(2) row lengths at the quantiles of [0, 1), the longest n/18."""
    k = np.arange(1, max(2, n // 18) + 1, dtype=np.float64)
    cdf = np.cumsum(1.0 / k ** 2)
    cdf /= cdf[-1]
    return np.searchsorted(cdf, (np.arange(n) + 0.5) / n) + 1


def _blocks_per_row(case):
    """Blocks drawn in each block row of a banded matrix: 70% to 130% of the
    mean, evenly spread."""
    nb, mean = case["n"] // case["block"], case["row"] / case["block"]
    lo, hi = max(1, int(0.7 * mean)), max(2, int(1.3 * mean))
    return lo + np.arange(nb) % (hi - lo + 1)


def _half_band(case):
    return min(1000 // case["block"], case["n"] // case["block"] // 4)


def _matrix(case, gen, dev):
    n, b = case["n"], case["block"]

    def rand(m):
        return torch.rand(m, generator=gen, device=dev, dtype=torch.float64)

    def repeat(counts):
        counts = torch.as_tensor(counts, device=dev)
        return torch.repeat_interleave(torch.arange(len(counts), device=dev), counts)

    if case["matrix"] == "uniform":
        rows = torch.arange(n, device=dev).repeat_interleave(case["row"])
        keys = rows * n + (rand(rows.numel()) * n).long()
    elif case["matrix"] == "powerlaw":
        deg = torch.as_tensor(_degrees_powerlaw(n), device=dev)
        deg = deg[torch.randperm(n, generator=gen, device=dev)]
        rows = torch.repeat_interleave(torch.arange(n, device=dev), deg)
        near = (rows + (rand(rows.numel()) * 129).long() - 64).clamp_(0, n - 1)
        far = (rand(rows.numel()) * n).long()
        cols = torch.where(rand(rows.numel()) < 0.7, near, far)
        diag = torch.arange(n, device=dev)
        keys = torch.cat([rows * n + cols, diag * n + diag])
    else:
        nb = n // b
        if case["matrix"] == "banded":
            br = repeat(_blocks_per_row(case))
            w = _half_band(case)
            bc = br + (rand(br.numel()) * (2 * w + 1)).long() - w
            bc = torch.where(bc < 0, bc + 2 * w + 1, torch.where(bc >= nb, bc - 2 * w - 1, bc))
            diag = torch.arange(nb, device=dev)
            bk = torch.cat([br * nb + bc, diag * nb + diag])
        else:
            per = case["row"] // b
            order = rand(nb * nb).view(nb, nb).argsort(dim=1)[:, :per]
            bk = (torch.arange(nb, device=dev)[:, None] * nb + order).reshape(-1)
        bk = torch.unique(bk)
        i = torch.arange(b, device=dev)
        keys = (((bk // nb) * b)[:, None, None] + i[None, :, None]) * n \
            + ((bk % nb) * b)[:, None, None] + i[None, None, :]
    keys = torch.unique(keys.reshape(-1))
    rows, cols = keys // n, keys % n
    row_ptr = torch.zeros(n + 1, dtype=torch.int64, device=dev)
    row_ptr[1:] = torch.cumsum(torch.bincount(rows, minlength=n), 0)
    if case["matrix"] in ("banded", "blocks"):
        val = torch.randn(keys.numel(), generator=gen, device=dev)
    else:
        val = torch.rand(keys.numel(), generator=gen, device=dev) * 2 - 1
    return row_ptr.int(), cols.int(), val


def _inputs(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    row_ptr, col, val = _matrix(case, gen, dev)
    shape = (case["n"], case["O"])
    if case["matrix"] == "blocks":
        B = torch.randn(shape, generator=gen, device=dev)
    else:
        B = torch.rand(shape, generator=gen, device=dev) * 2 - 1
    return row_ptr, col, val, B


def _nnz(case):
    """Expected entries of the matrix (repeated draws of a column count once)."""
    n, b = case["n"], case["block"]
    if case["matrix"] == "uniform":
        return n * case["row"]
    if case["matrix"] == "powerlaw":
        d = _degrees_powerlaw(n)
        return float(np.sum(129 * (1 - np.exp(-0.7 * d / 129)) + 0.3 * d + 1 - np.minimum(1, d / 180)))
    if case["matrix"] == "banded":
        c, w = _blocks_per_row(case).astype(np.float64), 2 * _half_band(case) + 1
        return float(np.sum(1 + (w - 1) * (1 - (1 - 1 / w) ** c))) * b * b
    return (n // b) * (case["row"] // b) * b * b


# ------------------------------------------------------------------ passes
class _Buf:
    """A torch tensor as the library's device buffers are described."""

    def __init__(self, t):
        self.t = t
        self.ptr = ctypes.c_void_p(t.data_ptr())
        self.nbytes = t.numel() * t.element_size()
        self.dtype = np.int32 if t.dtype == torch.int32 else np.float32


def _format(vs, case, csr):
    if case["matrix"] == "blocks":
        return vs.csr_to_vcsr_tc(csr, 16)
    return vs.csr_to_vcsr_seg(csr, 4, 64)


def prepare(case, seed):
    vs = _package()
    row_ptr, col, val, B = _inputs(case, seed)
    C = torch.empty((case["n"], case["O"]), device=B.device)
    state = dict(vs=vs, case=case, B=_Buf(B), C=_Buf(C))
    if case["call"] == "csr":
        state["csr"] = (_Buf(row_ptr), _Buf(col), _Buf(val))
        return state
    host = tuple(t.cpu().numpy() for t in (row_ptr, col, val))
    if case["call"] == "first":
        state["host"] = host
        return state
    torch.cuda.synchronize()
    fmt = _format(vs, case, vs.Csr.from_arrays(case["n"], case["n"], *host))
    fmt.upload()
    state["fmt"] = fmt
    return state


def run(state):
    vs, case, B, C = state["vs"], state["case"], state["B"], state["C"]
    n, O, call = case["n"], case["O"], case["call"]
    if call == "overwrite":
        vs.run_vcsr_spmm_gpu_ex(state["fmt"], B, O, 64, C, accumulate=False)
    elif call == "accumulate":
        C.t.zero_()
        vs.run_vcsr_spmm_gpu(state["fmt"], B, O, 64, C)
    elif call == "noalloc":
        vs.run_vcsr_spmm_gpu_noalloc(state["fmt"], B, O, C)
    elif call == "csr":
        row_ptr, col, val = state["csr"]
        vs.run_csr_wave_spmm_gpu(n, n, row_ptr, col, val, B, O, C)
    else:
        fmt = _format(vs, case, vs.Csr.from_arrays(n, n, *state["host"]))
        fmt.upload()
        vs.run_vcsr_spmm_gpu_ex(fmt, B, O, 64, C, timed=True, accumulate=False)
    return C.t


def work(case):
    n, O, nnz = case["n"], case["O"], _nnz(case)
    return {"bytes": 4.0 * (n + 1) + 8.0 * nnz + 8.0 * n * O, "flops": 2.0 * nnz * O}


def tolerance(case):
    # FP32 sums in another order: the present paths are 7e-8 to 3e-7 of the
    # result's norm off the 64-bit one (rows of up to a few thousand entries),
    # 5e-7 where 816 terms of N(0,1) products are added in one chain.
    return {"rel": 2e-6 if case["matrix"] == "blocks" else 1.2e-6}


def exact(case, seed):
    row_ptr, col, val, B = _inputs(case, seed)
    n, O = case["n"], case["O"]
    out = torch.zeros((n, O), dtype=torch.float64, device=B.device)
    rows = torch.repeat_interleave(torch.arange(n, device=B.device), (row_ptr[1:] - row_ptr[:-1]).long())
    col, val, B = col.long(), val.double(), B.double()
    step = max(1, (1 << 28) // O)
    for a in range(0, col.numel(), step):
        e = min(col.numel(), a + step)
        out.index_add_(0, rows[a:e], B[col[a:e]] * val[a:e, None])
    return out
