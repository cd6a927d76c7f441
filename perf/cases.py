"""The work that a program has this library do: calls of its public routines, over the sizes, modes and layouts in use.

A case is one call of one routine on data already where the routine takes it (device pointers, or host
arrays for the reference's C interface), with the scratch and descriptors that a program keeps.  Binary128
values are int64 tensors of shape (..., 2), their little-endian {lo, hi} words.  Outputs are those words, whole;
they are bytes, so no 64-bit value stands beside them.  Only the C interface's dot returns a double.
"""
import math
import random

import numpy as np
import torch

import qblas_amd as qb

ROW, COL = qb.ROW_MAJOR, qb.COL_MAJOR
LAYOUT = {"row": ROW, "col": COL}
T = 16  # chunks of the reference-order dot: the threads of the host that it stands in for
SIGN = -(2**63)


# ------------------------------------------------------------------------------------------------
# the cases
# ------------------------------------------------------------------------------------------------
def dot(mode, n, data, **more):
    return dict(op="dot", mode=mode, n=n, data=data, inc=1, host=False) | more


def gemv(mode, layout, m, n, data, alpha, beta, **more):
    return dict(op="gemv", mode=mode, layout=layout, m=m, n=n, pad=0, inc=1, data=data, alpha=alpha, beta=beta, host=False) | more


def gemm(mode, layout, m, n, k, data, alpha, beta, **more):
    return dict(op="gemm", mode=mode, layout=layout, m=m, n=n, k=k, pad=0, data=data, alpha=alpha, beta=beta) | more


def gemm_batch(mode, layout, count, lo, hi, shapes, data="uniform", **more):
    return dict(op="gemm_batch", mode=mode, layout=layout, count=count, lo=lo, hi=hi, shapes=shapes, data=data) | more


def gemv_batch(mode, layout, count, lo, hi, shapes, data="uniform", **more):
    return dict(op="gemv_batch", mode=mode, layout=layout, count=count, lo=lo, hi=hi, shapes=shapes, data=data) | more


def listed():
    return [
        # the smallest calls: a correctly rounded dot of a short vector inside an iteration; latency counts
        dot("exact", 1001, "uniform", name="dot exact 1001"),
        # the default mode's dot of a long vector resident on the GPU, in the order of a 16-thread host
        dot("reference", 1 << 20, "uniform", name="dot reference 2^20"),
        # the benchmark's memory-bound dot in double-double arithmetic
        dot("dd", 1 << 24, "uniform", name="dot dd 2^24"),
        # the README's call: row-major 1500 x 1500, alpha 1, beta 0, default mode, through the C interface on host arrays
        gemv("reference", "row", 1500, 1500, "uniform", 1.0, 0.0, host=True, name="host gemv reference 1500"),
        # the benchmark's memory-bound gemv, row-major, double-double
        gemv("dd", "row", 8192, 8192, "uniform", 1.5, -0.5, name="gemv dd row 8192"),
        # the same, column-major, correctly rounded
        gemv("exact", "col", 8192, 8192, "uniform", 1.5, -0.5, name="gemv exact col 8192"),
        # a column-major gemv in the default mode, ragged, on entries that were doubles before
        gemv("reference", "col", 2049, 777, "double", 1.0, 1.0, pad=3, name="gemv reference col ragged"),
        # the default mode's product of ordinary ragged matrices
        gemm("reference", "row", 500, 333, 700, "uniform", 1.5, -0.5, name="gemm reference ragged"),
        # a small product in the certified fast mode, accumulated into C, padded leading dimensions
        gemm("ozaki", "col", 150, 200, 333, "uniform", 1.5, -0.5, pad=5, name="gemm ozaki small"),
        # the benchmark's headline product
        gemm("ozaki", "row", 4096, 4096, 4096, "wide", 1.0, 0.0, name="gemm ozaki 4096"),
        # the benchmark's batch of uneven small products, each with its own alpha and beta
        gemm_batch("ozaki", "row", 4096, 8, 256, 7, name="gemm batch ozaki 4096"),
        # a batch of uneven small gemv problems in the default mode
        gemv_batch("reference", "row", 2048, 32, 1024, 8, name="gemv batch reference 2048"),
    ]


def spread(rng, lo, hi):
    """An integer of [lo, hi], even over its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    """One more case of the same ranges.  The reference order and double-double gemm have lower size limits: they cost more a step."""
    op = rng.choice(("dot", "dot", "gemv", "gemv", "gemv", "gemm", "gemm", "gemm", "gemm_batch", "gemv_batch"))
    layout = rng.choice(("row", "col"))
    data = rng.choice(("uniform", "uniform", "wide", "double"))
    alpha, beta = rng.choice(((1.0, 0.0), (1.5, -0.5), (1.0, 1.0), (-0.75, 0.25)))
    pad = rng.choice((0, 0, 1, 7))
    if op == "dot":
        mode = rng.choice(("reference", "exact", "dd"))
        return dot(mode, spread(rng, 100, 1 << (20 if mode == "reference" else 24)), data, inc=rng.choice((1, 1, 1, 2)),
                   host=rng.random() < 0.25)
    if op == "gemv":
        mode = rng.choice(("reference", "exact", "dd"))
        m, n = spread(rng, 16, 8192), spread(rng, 16, 8192)
        host = rng.random() < 0.2
        if host:
            m, n = min(m, 2048), min(n, 2048)
        return gemv(mode, layout, m, n, data, alpha, beta, pad=pad, inc=rng.choice((1, 1, 1, 2)), host=host)
    if op == "gemm":
        mode = rng.choice(("reference", "dd", "ozaki", "ozaki"))
        top = {"reference": 1024, "dd": 2048, "ozaki": 4096}[mode]
        m, n, k = (spread(rng, 16, top) for _ in range(3))
        if mode == "ozaki" and rng.random() < 0.15:
            data = "cancel"
            m, n, k = min(m, 1500), min(n, 1500), min(k, 3000)
        return gemm(mode, layout, m, n, k, data, alpha, beta, pad=pad)
    if op == "gemm_batch":
        mode = rng.choice(("reference", "dd", "ozaki", "ozaki"))
        hi = rng.randint(32, 256)
        return gemm_batch(mode, layout, spread(rng, 32, 512 if mode == "reference" else 4096), 8, hi, rng.randrange(1 << 20), data)
    mode = rng.choice(("reference", "exact", "dd"))
    return gemv_batch(mode, layout, spread(rng, 32, 2048), 32, rng.randint(64, 1024), rng.randrange(1 << 20), data)


# ------------------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------------------
def words(g, n, data, device):
    """n binary128 values: "uniform": uniform over [-1, 1) with all 113 significand bits in use; "double": the same with a
    double's 53; "wide": random sign, magnitude log-uniform over [2^-30, 2^30), all bits in use."""
    v = torch.empty((n, 2), dtype=torch.int64, device=device)
    v[:, 0] = torch.randint(SIGN, 2**63 - 1, (n,), generator=g, device=device, dtype=torch.int64)
    if data == "wide":
        e = torch.randint(16383 - 30, 16383 + 30, (n,), generator=g, device=device, dtype=torch.int64)
        r = torch.randint(SIGN, 2**63 - 1, (n,), generator=g, device=device, dtype=torch.int64)
        v[:, 1] = (r & SIGN) | (e << 48) | (r & (2**48 - 1))
        return v
    d = torch.rand(n, generator=g, device=device, dtype=torch.float64).mul_(2).sub_(1).view(torch.int64)
    f = d & (2**52 - 1)
    v[:, 1] = (d & SIGN) | ((((d >> 52) & 0x7FF) + (16383 - 1023)) << 48) | (f >> 4)
    v[:, 0] = (f << 60) | (0 if data == "double" else v[:, 0] & (2**60 - 1))
    return v


def to_double(v):
    """The values of binary128 words as doubles (truncated to 53 bits), for |v| well inside the double range."""
    lo, hi = v[:, 0], v[:, 1]
    d = (hi & SIGN) | ((((hi >> 48) & 0x7FFF) - (16383 - 1023)) << 52) | ((hi & (2**48 - 1)) << 4) | ((lo >> 60) & 15)
    return d.view(torch.float64)


def generator(seed, device):
    return torch.Generator(device=device).manual_seed(int(seed))


def cancelling(g, m, n, k, device):
    """A (m x k) and B^T (n x k): of every 8 products of a row and a column two large ones cancel, so the sums are small beside them."""
    a, b = words(g, m * k, "uniform", device).view(m, k, 2), words(g, n * k, "uniform", device).view(n, k, 2)
    if k < 2:
        return a, b
    last = k - 1 - (k - 2) % 8  # as many second members of a pair as first ones
    big = a[:, 0:last:8, :].clone()
    big[..., 1] += 66 << 48  # times 2^66, about 1e20
    a[:, 0:last:8, :] = big
    big[..., 1] ^= SIGN
    a[:, 1 : last + 1 : 8, :] = big
    b[:, 1 : last + 1 : 8, :] = b[:, 0:last:8, :]
    return a, b


def stored(v, rows, cols, layout, pad):
    """The matrix v (rows x cols) in a layout with `pad` unused elements after each row or column, and its leading dimension."""
    v = v.view(rows, cols, 2)
    v = v if layout == "row" else v.transpose(0, 1)
    if pad:
        w = torch.zeros((v.shape[0], v.shape[1] + pad, 2), dtype=torch.int64, device=v.device)
        w[:, : v.shape[1]] = v
        v = w
    return v.contiguous(), v.shape[1]


def sizes(case):
    """The problems' sizes of a batch: the case's own, whatever the values."""
    r = random.Random(case["shapes"])
    dims = 3 if case["op"] == "gemm_batch" else 2
    return [tuple(r.randint(case["lo"], case["hi"]) for _ in range(dims)) for _ in range(case["count"])]


def batch(case, g, r):
    """One buffer with all operands, and the descriptors on the GPU."""
    device, gemms, col = "cuda", case["op"] == "gemm_batch", case["layout"] == "col"
    dims = np.array(sizes(case), dtype=np.int64)
    m, n = dims[:, 0], dims[:, 1]
    parts = (m * dims[:, 2], dims[:, 2] * n) if gemms else (m * n, n)
    outs = m * n if gemms else m
    offsets = [np.cumsum(p) - p for p in parts]
    bufs = [words(g, int(p.sum()), case["data"], device) for p in parts]
    out = words(g, int(outs.sum()), case["data"], device)
    p = np.zeros(case["count"], dtype=qb.GEMM_PROBLEM if gemms else qb.GEMV_PROBLEM)
    p["m"], p["n"] = m, n
    at = [np.uint64(b.data_ptr()) + (o * 16).astype(np.uint64) for b, o in zip(bufs, offsets)]
    to = np.uint64(out.data_ptr()) + ((np.cumsum(outs) - outs) * 16).astype(np.uint64)
    if gemms:
        k = dims[:, 2]
        p["k"], p["A"], p["B"], p["C"] = k, at[0], at[1], to
        p["lda"], p["ldb"], p["ldc"] = (m, k, m) if col else (k, n, n)
    else:
        p["A"], p["x"], p["y"], p["incx"], p["incy"] = at[0], at[1], to, 1, 1
        p["lda"] = m if col else n
    for i in range(case["count"]):
        p["alpha"][i], p["beta"][i] = qb.from_double(r.uniform(-2, 2)), qb.from_double(r.uniform(-0.9, 0.9))
    return dict(bufs=bufs, out=out, problems=torch.from_numpy(p.view(np.uint8).copy()).to(device))


def prepare(case, seed):
    op, device = case["op"], "cpu" if case.get("host") else "cuda"
    g, state = generator(seed, device), dict(case=case)
    mode = qb.MODES[case["mode"]]
    if op == "dot":
        n, inc = case["n"], case["inc"]
        state |= dict(x=words(g, 1 + (n - 1) * inc, case["data"], device), y=words(g, 1 + (n - 1) * inc, case["data"], device),
                      out=torch.zeros(2, dtype=torch.int64, device=device))
    elif op == "gemv":
        m, n, inc = case["m"], case["n"], case["inc"]
        A, lda = stored(words(g, m * n, case["data"], device), m, n, case["layout"], case["pad"])
        state |= dict(A=A, lda=lda, x=words(g, 1 + (n - 1) * inc, case["data"], device), out=words(g, 1 + (m - 1) * inc, case["data"], device))
    elif op == "gemm":
        m, n, k, layout, pad = case["m"], case["n"], case["k"], case["layout"], case["pad"]
        if case["data"] == "cancel":
            a, b = cancelling(g, m, n, k, device)
            b = b.transpose(0, 1).contiguous()
            c = words(g, m * n, "uniform", device)
        else:
            a, b, c = (words(g, r * q, case["data"], device) for r, q in ((m, k), (k, n), (m, n)))
        (A, lda), (B, ldb), (C, ldc) = stored(a, m, k, layout, pad), stored(b, k, n, layout, pad), stored(c, m, n, layout, pad)
        state |= dict(A=A, lda=lda, B=B, ldb=ldb, out=C, ldc=ldc)
    else:
        state |= batch(case, g, random.Random(int(seed)))
    if device == "cpu":  # the C interface takes arrays, and a mode and a thread count that a program sets once
        qb.set_mode(mode)
        qb.set_num_threads(T)
        state |= {key: v.numpy().view(np.uint64) for key, v in state.items() if isinstance(v, torch.Tensor)}
    else:
        state["alpha"], state["beta"] = (qb.from_double(case.get(key, 0.0)) for key in ("alpha", "beta"))
    state["mode"] = mode
    return state


# ------------------------------------------------------------------------------------------------
# one pass
# ------------------------------------------------------------------------------------------------
def run(state):
    s, c = state, state["case"]
    op, out = c["op"], state["out"]
    if c.get("host"):
        if op == "dot":
            return qb.qdot(c["n"], s["x"], c["inc"], s["y"], c["inc"])
        qb.qgemv("R" if c["layout"] == "row" else "C", "N", c["m"], c["n"], c["alpha"], s["A"], s["lda"], s["x"], c["inc"], c["beta"], out,
                 c["inc"])
        return out.view(np.int64)
    stream = torch.cuda.current_stream().cuda_stream
    mode, layout = s["mode"], LAYOUT[c.get("layout", "row")]
    if op == "dot":
        qb.dev_dot(mode, c["n"], s["x"].data_ptr(), c["inc"], s["y"].data_ptr(), c["inc"], T, out.data_ptr(), stream)
    elif op == "gemv":
        qb.dev_gemv(mode, layout, c["m"], c["n"], s["alpha"], s["A"].data_ptr(), s["lda"], s["x"].data_ptr(), c["inc"], s["beta"],
                    out.data_ptr(), c["inc"], stream)
    elif op == "gemm":
        qb.dev_gemm(mode, layout, c["m"], c["n"], c["k"], s["alpha"], s["A"].data_ptr(), s["lda"], s["B"].data_ptr(), s["ldb"], s["beta"],
                    out.data_ptr(), s["ldc"], stream)
    elif op == "gemm_batch":
        qb.dev_gemm_batched(mode, layout, c["count"], s["problems"].data_ptr(), stream)
    else:
        qb.dev_gemv_batched(mode, layout, c["count"], s["problems"].data_ptr(), stream)
    return out


def exact(case, seed):
    """The host dot returns a double, which a 64-bit sum gives; every other output is binary128 words, which 64 bits do not hold."""
    if not (case["op"] == "dot" and case.get("host")):
        return None
    s = prepare(case, seed)
    x, y = (to_double(torch.from_numpy(s[key].view(np.int64))[:: case["inc"]]).numpy() for key in ("x", "y"))
    return float(math.fsum((x * y).tolist()))


def work(case):
    """Bytes: each operand read once, each result read (where beta is not 0) and written once.  Flops: binary128 operations, a
    multiplication and an addition for each product."""
    op = case["op"]
    if op == "dot":
        return dict(bytes=32.0 * case["n"] + 16, flops=2.0 * case["n"])
    probs = [tuple(case[key] for key in ("m", "n", "k") if key in case)] if op in ("gemv", "gemm") else sizes(case)
    outs = 32.0 if case.get("beta", 1.0) else 16.0
    total, flops = 0.0, 0.0
    for p in probs:
        m, n, k = p if len(p) == 3 else (p[0], 1, p[1])
        total += 16.0 * (m * k + k * n) + outs * m * n
        flops += 2.0 * m * n * k
    return dict(bytes=total, flops=flops)
