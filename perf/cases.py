"""Timed cases of the grouped GEMM: what a program has it compute, through the PyTorch entry points.

A case is a dict of plain values; its problem shapes come from those values alone (numpy's frozen
RandomState streams), its operand values from the seed given to prepare().  Three entry points:

  plan     GroupedGemmPlan(...) once, run() per pass: fixed tensors refilled in place between passes
  once     run_grouped_gemm(...): prepare, upload, launch and wait in one call
  moe      MoeGroupedGemmPlan(...) once, run(counts) per pass: token counts that live on the GPU

Matrices are tightly packed (lda = k, ldb = ldc = ldd = n) in one pool per operand, each on a
256-byte boundary, so odd k or n gives rows that start on 2-byte boundaries.  The plan and once
cases return the whole D pool (the padding between matrices stays zero), the moe cases D.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from grouped_gemm_gpu_kernel_amd.api import KernelConfig, SortMode
from grouped_gemm_gpu_kernel_amd.torch_ops import GroupedGemmPlan, MoeGroupedGemmPlan, run_grouped_gemm

ALIGN = 256  # bytes between the starts of two matrices of a pool are a multiple of this

# Candidate sizes of the "small" set of many tiny problems.
SMALL_M = (16, 24, 32, 48, 64)
SMALL_N = (16, 32, 48, 64, 96)
SMALL_K = (16, 24, 32, 48, 64)


def _plan(name, shapes, count, lo, hi, klo, khi, config, values="uniform", c=True, entry="plan", matrix_cores=True,
          shape_seed=42):
    return {"name": name, "entry": entry, "shapes": shapes, "count": count, "lo": lo, "hi": hi, "klo": klo, "khi": khi,
            "config": config, "values": values, "c": c, "matrix_cores": matrix_cores, "shape_seed": shape_seed}


def _moe(name, experts, tokens, k, n, shape_seed=42):
    return {"name": name, "entry": "moe", "experts": experts, "tokens": tokens, "k": k, "n": n, "config": "128x64x32",
            "shape_seed": shape_seed}


def listed():
    return [
        # The smallest call: a handful of odd-sized problems, one launch, bound by its latency.
        _plan("tiny16", "uniform", 16, 1, 256, 1, 256, "128x64x32"),
        # Many tiny problems (batched small layers), with the default macro-tile.
        _plan("small256", "small", 256, 16, 96, 16, 64, "64x64x16"),
        # The mixed-size training or serving set the library is quoted on: 64 to 1024 rows and
        # columns, k to 2048, half of the sizes odd, C read.
        _plan("mixed512", "log", 512, 64, 1024, 64, 2048, "128x64x32"),
        # A batch of equal dense layers, no C.
        _plan("dense64", "equal", 64, 2048, 2048, 2048, 2048, "128x64x32", values="normal", c=False),
        # A few problems that each fill many compute units, ragged in every dimension, C read.
        _plan("ragged24", "log", 24, 300, 3000, 129, 4097, "64x128x32"),
        # One large GEMM through the grouped path.
        _plan("square8192", "equal", 1, 8192, 8192, 8192, 8192, "128x64x32", values="normal", c=False),
        # The largest: 5% large problems hidden among thousands of tiny ones.
        _plan("longtail4096", "longtail", 4096, 1, 4096, 1, 8192, "128x64x32"),
        # A mixture-of-experts layer in prefill: 16384 tokens, Zipf-like routing, some experts empty.
        _moe("moe64_prefill", 64, 16384, 4096, 14336),
        # The same layer in decode: a few tokens per expert, the weights are what is moved.
        _moe("moe64_decode", 64, 256, 4096, 14336),
        # A small expert layer: bound by the prepare and the launch rather than by the products.
        _moe("moe16_small", 16, 512, 1024, 2048),
        # A one-off call that pays for its own preparation, upload and wait.
        _plan("once64", "log", 64, 64, 512, 64, 1024, "128x64x32", entry="once"),
        # The path without matrix cores (use_tensor_cores off).
        _plan("fma256", "log", 256, 16, 256, 16, 256, "64x64x16", matrix_cores=False),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    config = rng.choice(("128x64x32", "64x64x16", "64x128x32"))
    seed = rng.randrange(1 << 30)
    kind = rng.choice(("plan", "plan", "mixed", "equal", "longtail", "moe", "moe", "once", "fma"))
    if kind == "plan":  # from a handful of small problems to a few ragged large ones
        lo = _log_int(rng, 8, 300)
        hi = _log_int(rng, 2 * lo, 10 * lo)
        klo = _log_int(rng, 8, 256)
        khi = _log_int(rng, 2 * klo, 16 * klo)
        case = _plan("", "log", _log_int(rng, 8, 64), lo, hi, klo, khi, config, c=rng.random() < 0.6, shape_seed=seed)
    elif kind == "mixed":
        lo = _log_int(rng, 16, 96)
        case = _plan("", "log", _log_int(rng, 128, 768), lo, lo * rng.randint(4, 12), lo, lo * rng.randint(8, 24),
                     config, c=rng.random() < 0.6, shape_seed=seed)
    elif kind == "equal":
        size = _log_int(rng, 500, 4096)
        k = _log_int(rng, 500, 4096)
        size -= size % rng.choice((1, 8, 64))
        k -= k % rng.choice((1, 8, 64))
        count = max(1, min(64, int(4e11 / (size * size * k))))
        case = _plan("", "equal", rng.randint(1, count), size, size, k, k, config, values="normal",
                     c=rng.random() < 0.3, shape_seed=seed)
    elif kind == "longtail":
        case = _plan("", "longtail", _log_int(rng, 64, 2048), 1, _log_int(rng, 1500, 4096), 1,
                     _log_int(rng, 2000, 8192), config, shape_seed=seed)
    elif kind == "moe":
        experts = _log_int(rng, 4, 128)
        k = 64 * _log_int(rng, 8, 64)
        n = 64 * _log_int(rng, 8, 224)
        if experts * k * n > 64 * 4096 * 14336:
            experts = max(4, 64 * 4096 * 14336 // (k * n))
        case = _moe("", experts, _log_int(rng, 64, 16384), k, n, shape_seed=seed)
        case["config"] = config
    elif kind == "once":
        case = _plan("", "log", _log_int(rng, 8, 256), 32, _log_int(rng, 64, 700), 32, _log_int(rng, 64, 1024), config,
                     c=rng.random() < 0.6, entry="once", shape_seed=seed)
    else:
        case = _plan("", "log", _log_int(rng, 32, 512), 16, _log_int(rng, 64, 400), 16, _log_int(rng, 64, 400), config,
                     c=rng.random() < 0.6, matrix_cores=False, shape_seed=seed)
    del case["name"]
    return case


# ---------------------------------------------------------------- shapes

def _log_uniform(rs, lo, hi, count):
    u = rs.uniform(math.log(lo), math.log(hi + 1), count)
    return np.clip(np.floor(np.exp(u)), lo, hi).astype(np.int64)


def _shapes(case):
    """(m, n, k, alpha, beta) of every problem of a plan or once case."""
    rs = np.random.RandomState(case["shape_seed"])
    count, lo, hi, klo, khi = case["count"], case["lo"], case["hi"], case["klo"], case["khi"]
    alpha, beta = np.ones(count), np.full(count, 0.5 if case["c"] else 0.0)
    if case["shapes"] == "equal":
        m = n = np.full(count, lo, np.int64)
        k = np.full(count, klo, np.int64)
    elif case["shapes"] == "uniform":
        m, n = rs.randint(lo, hi + 1, count), rs.randint(lo, hi + 1, count)
        k = rs.randint(klo, khi + 1, count)
    elif case["shapes"] == "small":
        m, n, k = rs.choice(SMALL_M, count), rs.choice(SMALL_N, count), rs.choice(SMALL_K, count)
    elif case["shapes"] == "log":
        m, n = _log_uniform(rs, lo, hi, count), _log_uniform(rs, lo, hi, count)
        k = _log_uniform(rs, klo, khi, count)
        alpha = rs.uniform(0.5, 2.0, count)
        if case["c"]:
            beta = rs.uniform(0.1, 1.0, count)
    elif case["shapes"] == "longtail":
        n_large = max(1, count // 20 + (1 if count == 4096 else 0))
        large = np.zeros(count, bool)
        large[rs.permutation(count)[:n_large]] = True
        m, n, k = rs.randint(1, 65, count), rs.randint(1, 65, count), rs.randint(1, 65, count)
        m[large] = rs.randint(1024, hi + 1, n_large)
        n[large] = rs.randint(1024, hi + 1, n_large)
        k[large] = rs.randint(1024, khi + 1, n_large)
        beta = np.ones(count) if case["c"] else beta
    else:
        raise ValueError(case["shapes"])
    return (m.astype(np.int64), n.astype(np.int64), k.astype(np.int64), [float(x) for x in alpha.astype(np.float32)],
            [float(x) for x in beta.astype(np.float32)])


def _counts(case):
    """Token counts of a moe case before the seed permutes the experts: Zipf(1.2) over the experts,
    the emptiest sixteenth of them emptied into the largest."""
    rs = np.random.RandomState(case["shape_seed"])
    experts = case["experts"]
    weights = np.arange(1, experts + 1, dtype=np.float64) ** -1.2
    counts = rs.multinomial(case["tokens"], weights / weights.sum()).astype(np.int64)
    order = np.argsort(counts, kind="stable")
    for e in order[:experts // 16]:
        counts[order[-1]] += counts[e]
        counts[e] = 0
    return counts


def _config(case):
    return KernelConfig.named(case["config"], use_tensor_cores=case.get("matrix_cores", True))


# ---------------------------------------------------------------- operands

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _f16(shape, g, values, k):
    """binary16 operands: uniform in [-1, 1), or normal with deviation 1 / sqrt(k)."""
    t = torch.empty(shape, dtype=torch.float16, device="cuda")
    if values == "normal":
        return t.normal_(0.0, 1.0 / math.sqrt(k), generator=g)
    return t.uniform_(-1.0, 1.0, generator=g)


def _pool(rows, cols, itemsize):
    """Element offsets of tightly packed matrices of a pool, and its size."""
    step = ALIGN // itemsize
    sizes = (rows * cols + step - 1) // step * step
    ends = np.cumsum(sizes)
    return ends - sizes, int(ends[-1])


def _views(pool, offsets, rows, cols):
    return [pool[int(o):int(o) + int(r * c)].view(int(r), int(c)) for o, r, c in zip(offsets, rows, cols)]


def _set_operands(case, seed):
    m, n, k, alpha, beta = _shapes(case)
    g = _generator(seed)
    a_off, a_size = _pool(m, k, 2)
    b_off, b_size = _pool(k, n, 2)
    d_off, d_size = _pool(m, n, 4)
    kmax = int(k.max())
    a = _views(_f16(a_size, g, case["values"], kmax), a_off, m, k)
    b = _views(_f16(b_size, g, case["values"], kmax), b_off, k, n)
    c = None
    if case["c"]:
        c = _views(torch.empty(d_size, dtype=torch.float32, device="cuda").uniform_(-1.0, 1.0, generator=g), d_off, m, n)
    return a, b, c, alpha, beta, (d_off, d_size, m, n)


def _moe_operands(case, seed):
    experts, k, n = case["experts"], case["k"], case["n"]
    g = _generator(seed)
    counts = np.random.RandomState(seed % (1 << 31)).permutation(_counts(case))
    a = torch.empty((case["tokens"], k), dtype=torch.float16, device="cuda").normal_(0.0, 1.0, generator=g)
    b = torch.empty((experts, k, n), dtype=torch.float16, device="cuda").normal_(0.0, 0.02, generator=g)
    return a, b, counts


def prepare(case, seed):
    if case["entry"] == "moe":
        a, b, counts = _moe_operands(case, seed)
        d = torch.zeros((case["tokens"], case["n"]), dtype=torch.float32, device="cuda")
        plan = MoeGroupedGemmPlan(a, b, d, config=_config(case))
        return {"entry": "moe", "plan": plan, "counts": torch.tensor(counts, dtype=torch.int32, device="cuda")}
    a, b, c, alpha, beta, (d_off, d_size, m, n) = _set_operands(case, seed)
    pool = torch.zeros(d_size, dtype=torch.float32, device="cuda")
    d = _views(pool, d_off, m, n)
    if case["entry"] == "once":
        return {"entry": "once", "args": (a, b, c, alpha, beta), "config": _config(case), "d": d, "pool": pool}
    plan = GroupedGemmPlan(a, b, c, d, alpha, beta, sort_mode=SortMode.kByTilesThenK, config=_config(case))
    return {"entry": "plan", "plan": plan, "pool": pool}


def run(state):
    if state["entry"] == "moe":
        return state["plan"].run(state["counts"])
    if state["entry"] == "once":
        a, b, c, alpha, beta = state["args"]
        run_grouped_gemm(a, b, c, alpha, beta, config=state["config"], out=state["d"])
        return state["pool"]
    state["plan"].run()
    return state["pool"]


def work(case):
    if case["entry"] == "moe":
        rows, experts = case["tokens"], int(np.count_nonzero(_counts(case)))
        k, n = case["k"], case["n"]
        return {"bytes": 2.0 * rows * k + 2.0 * experts * k * n + 4.0 * rows * n, "flops": 2.0 * rows * n * k}
    m, n, k, _, _ = (np.asarray(x, np.float64) for x in _shapes(case))
    return {"bytes": float(np.sum(2 * m * k + 2 * k * n + 4 * m * n * (2 if case["c"] else 1))),
            "flops": float(np.sum(2 * m * n * k))}


def tolerance(case):
    """binary16 products are exact in binary32; their binary32 sums over k differ with the order.
    Measured against 64 bits: 5e-8 (k to 64) to 5.7e-7 (k = 8192)."""
    return {"rel": 2.5e-6, "max": 1e-4}


def exact(case, seed):
    if case["entry"] == "moe":
        a, b, counts = _moe_operands(case, seed)
        out = torch.zeros((case["tokens"], case["n"]), dtype=torch.float64, device="cuda")
        row = 0
        for e, rows in enumerate(int(x) for x in counts):
            if rows:
                out[row:row + rows] = a[row:row + rows].double() @ b[e].double()
            row += rows
        return out
    a, b, c, alpha, beta, (d_off, d_size, m, n) = _set_operands(case, seed)
    pool = torch.zeros(d_size, dtype=torch.float64, device="cuda")
    for i, d in enumerate(_views(pool, d_off, m, n)):
        torch.mm(a[i].double(), b[i].double(), out=d)
        d *= alpha[i]
        if c is not None:
            d += beta[i] * c[i].double()
    return pool
