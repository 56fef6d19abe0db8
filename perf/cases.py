"""Performance cases of the single-rank local multiply: what a program that
uses this library has it do, through its public entry points.

A case is a dict of plain values with a "kind":
  gemm       C <- alpha op(A) op(B) + beta C on device-resident operands (Handle.dgemm)
  ozaki      the same product in split precision on the INT8 matrix cores (Handle.dgemm_ozaki)
  transform  the block copy / transpose of a ScaLAPACK reorder (Handle.block_transform)
  grouped    a batch of small uneven products replayed as a graph (Grouped.graph_run)
  layout     a product of matrices given as grids of device blocks (Handle.dgemm_layout)
  host       a product of pinned host operands (Handle.dgemm_host)
Matrices are column-major FP64; an r x c matrix with leading dimension ld is a
torch tensor of shape (c, ld).  Calls with beta != 0 update C in place, so such
a pass first copies the kept C0 over C with the library's own block copy.
"""
import math

import numpy as np
import torch

import cosma_amd as ca

_handle = None


def handle():
    """The one handle that a program keeps for all its calls."""
    global _handle
    if _handle is None:
        _handle = ca.Handle(0)
    return _handle


def gemm(name, ta, tb, m, n, k, beta=0.0, pad=0):
    return {"name": name, "kind": "gemm", "ta": ta, "tb": tb, "m": m, "n": n, "k": k, "alpha": 1.0, "beta": beta,
            "pad": pad}


def listed():
    return [
        # the smallest multiplies of a block-sparse or deeply split run: launch latency
        gemm("gemm_100", "N", "N", 100, 100, 100),
        # the miniapp's default problem through local_multiply
        gemm("gemm_2000", "N", "N", 2000, 2000, 2000),
        # odd extents and odd leading dimensions, as submatrices of a pdgemm have them
        gemm("gemm_ragged", "N", "T", 1537, 1021, 2999, pad=3),
        # tall-skinny A^T B, one k-panel of the 2048 x 2048 x 2^20 run
        gemm("gemm_tall", "T", "N", 2048, 2048, 65536),
        # the headline product: 16384^3, A^T B + C / 2
        gemm("gemm_16384", "T", "N", 16384, 16384, 16384, beta=0.5),
        # split precision at the size of its benchmark, uniform entries
        {"name": "ozaki_8192", "kind": "ozaki", "ta": "N", "tb": "N", "m": 8192, "n": 8192, "k": 8192, "phi": 0.0},
        # split precision at an ordinary, ragged size with entries of uneven magnitude
        {"name": "ozaki_3000", "kind": "ozaki", "ta": "T", "tb": "N", "m": 3000, "n": 2501, "k": 4100, "phi": 1.0},
        # pdgemm's transpose of an operand, odd extents and leading dimensions
        {"name": "transpose_odd", "kind": "transform", "op": "T", "rows": 8191, "cols": 12289, "beta": 0.0, "pad": 2},
        # pdgemm's last step: the product scaled into C (after a plain copy that restores C)
        {"name": "update", "kind": "transform", "op": "N", "rows": 16384, "cols": 8192, "beta": 0.5, "pad": 0},
        # 4096 uneven products, m, n, k log-uniform in [16, 512], one graph launch
        {"name": "grouped_4096", "kind": "grouped", "count": 4096, "lo": 16, "hi": 512, "dims": 5},
        # multiply_using_layout: 4000^3 from 256 x 256 blocks in device memory
        {"name": "layout_4000", "kind": "layout", "ta": "N", "tb": "N", "m": 4000, "n": 4000, "k": 4000,
         "block": 256},
        # local_multiply of operands in pinned host memory with the default tiles
        {"name": "host_8192", "kind": "host", "ta": "N", "tb": "N", "m": 8192, "n": 8192, "k": 8192},
    ]


def log_int(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the listed ones' ranges."""
    kind = rng.choice(["small", "medium", "medium", "tall", "large", "ozaki", "ozaki", "transform", "transform",
                       "grouped", "layout", "host"])
    ta, tb = rng.choice("NT"), rng.choice("NT")
    if kind in ("small", "medium", "tall", "large"):
        beta, pad = rng.choice([0.0, 0.5]), rng.choice([0, 0, 1, 2, 3])
        if kind == "small":
            m, n, k = (log_int(rng, 32, 512) for _ in range(3))
        elif kind == "medium":
            m, n, k = (log_int(rng, 512, 4096) for _ in range(3))
        elif kind == "tall":
            m, n, k = log_int(rng, 512, 4096), log_int(rng, 512, 4096), log_int(rng, 8192, 131072)
            ta, tb = "T", "N"
        else:
            m, n, k = (128 * log_int(rng, 32, 96) for _ in range(3))
        c = gemm("", ta, tb, m, n, k, beta, pad)
        del c["name"]
        return c
    if kind == "ozaki":
        m, n, k = (log_int(rng, 1024, 8192) for _ in range(3))
        return {"kind": kind, "ta": ta, "tb": tb, "m": m, "n": n, "k": k, "phi": rng.choice([0.0, 1.0, 4.0])}
    if kind == "transform":
        return {"kind": kind, "op": ta, "rows": log_int(rng, 256, 16384), "cols": log_int(rng, 256, 16384),
                "beta": rng.choice([0.0, 0.0, 0.5]), "pad": rng.choice([0, 1, 2])}
    if kind == "grouped":
        return {"kind": kind, "count": log_int(rng, 64, 4096), "lo": 16, "hi": log_int(rng, 128, 512),
                "dims": rng.randrange(1 << 30)}
    if kind == "layout":
        m, n, k = (log_int(rng, 1024, 6000) for _ in range(3))
        return {"kind": kind, "ta": ta, "tb": tb, "m": m, "n": n, "k": k, "block": log_int(rng, 128, 1024)}
    m, n, k = (log_int(rng, 1024, 8192) for _ in range(3))
    return {"kind": "host", "ta": ta, "tb": tb, "m": m, "n": n, "k": k}


# ------------------------------------------------------------------- inputs
def stored(case):
    """Stored extents (rows, cols) of A and B."""
    m, n, k = case["m"], case["n"], case["k"]
    return (m, k) if case["ta"] == "N" else (k, m), (k, n) if case["tb"] == "N" else (n, k)


def source(case, seed):
    """The seeded generator that every input of a case is drawn from, in order."""
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * seed + 17)
    return g


def uniform(g, rows, cols, pad=0):
    """A column-major rows x cols matrix of uniform [-1, 1) entries, leading dimension rows + pad."""
    return torch.rand((cols, rows + pad), dtype=torch.float64, device="cuda", generator=g) * 2 - 1


def lognormal(g, rows, cols, phi):
    """Entries (u - 1/2) exp(phi z): uniform for phi = 0, magnitudes spread over many binades for phi = 4."""
    x = torch.rand((cols, rows), dtype=torch.float64, device="cuda", generator=g) - 0.5
    if phi:
        x *= torch.exp(phi * torch.randn((cols, rows), dtype=torch.float64, device="cuda", generator=g))
    return x


def batch_dims(case):
    """m, n, k of every problem of a batch, log-uniform in [lo, hi]; the same for every seed."""
    rng = np.random.default_rng(case["dims"])
    lo, hi = case["lo"], case["hi"]
    return np.clip(np.rint(np.exp(rng.uniform(math.log(lo), math.log(hi), (case["count"], 3)))), lo, hi).astype(int)


def batch_inputs(case, seed):
    """Dims, packed A, packed B and the packed offsets of every problem's A, B, C."""
    d = batch_dims(case)
    g = source(case, seed)
    m, n, k = d[:, 0], d[:, 1], d[:, 2]
    offs = [np.concatenate([[0], np.cumsum(s)]) for s in (m * k, k * n, m * n)]
    A, B = (torch.rand(int(o[-1]), dtype=torch.float64, device="cuda", generator=g) * 2 - 1 for o in offs[:2])
    return d, A, B, offs


def grid_of(rows, cols, size):
    """(row, col, rows, cols, offset) of the blocks of a matrix packed block after block."""
    out, off = [], 0
    for c in range(0, cols, size):
        for r in range(0, rows, size):
            nr, nc = min(size, rows - r), min(size, cols - c)
            out.append((r, c, nr, nc, off))
            off += nr * nc
    return out


def pack(x, rows, cols, size):
    """The blocks of the column-major matrix x, one after the other, each contiguous."""
    out = torch.empty(rows * cols, dtype=torch.float64, device="cuda")
    for r, c, nr, nc, off in grid_of(rows, cols, size):
        out[off:off + nr * nc].view(nc, nr).copy_(x[c:c + nc, r:r + nr])
    return out


def block_list(t, rows, cols, size):
    return [(t.data_ptr() + 8 * off, nr, r, c, nr, nc) for r, c, nr, nc, off in grid_of(rows, cols, size)]


def gemm_inputs(case, seed):
    g = source(case, seed)
    (ar, ac), (br, bc) = stored(case)
    pad = case.get("pad", 0)
    A, B = uniform(g, ar, ac, pad), uniform(g, br, bc, pad)
    C0 = uniform(g, case["m"], case["n"], pad) if case.get("beta") else None
    return A, B, C0


def ozaki_inputs(case, seed):
    g = source(case, seed)
    (ar, ac), (br, bc) = stored(case)
    return lognormal(g, ar, ac, case["phi"]), lognormal(g, br, bc, case["phi"])


def transform_inputs(case, seed):
    g = source(case, seed)
    rows, cols, pad = case["rows"], case["cols"], case["pad"]
    src = uniform(g, rows, cols, pad) if case["op"] == "N" else uniform(g, cols, rows, pad)
    return src, uniform(g, rows, cols, pad) if case["beta"] else None


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "handle": handle()}
    if kind == "gemm":
        A, B, C0 = gemm_inputs(case, seed)
        C = torch.zeros((case["n"], case["m"] + case["pad"]), dtype=torch.float64, device="cuda")
        s.update(A=A, B=B, C=C, C0=C0)
    elif kind == "ozaki":
        A, B = ozaki_inputs(case, seed)
        s.update(A=A, B=B, C=torch.zeros((case["n"], case["m"]), dtype=torch.float64, device="cuda"))
    elif kind == "transform":
        src, dst0 = transform_inputs(case, seed)
        dst = torch.zeros((case["cols"], case["rows"] + case["pad"]), dtype=torch.float64, device="cuda")
        s.update(src=src, dst=dst, dst0=dst0)
    elif kind == "grouped":
        d, A, B, offs = batch_inputs(case, seed)
        C = torch.zeros(int(offs[2][-1]), dtype=torch.float64, device="cuda")
        problems = [("N", "N", int(m), int(n), int(k), 1.0, A.data_ptr() + 8 * int(offs[0][i]), int(m),
                     B.data_ptr() + 8 * int(offs[1][i]), int(k), 0.0, C.data_ptr() + 8 * int(offs[2][i]), int(m))
                    for i, (m, n, k) in enumerate(d)]
        plan = ca.Grouped(s["handle"], problems)
        plan.tune()
        s.update(A=A, B=B, C=C, plan=plan)
    elif kind == "layout":
        (ar, ac), (br, bc) = stored(case)
        A, B, _ = gemm_inputs(case, seed)
        size = case["block"]
        A, B = pack(A, ar, ac, size), pack(B, br, bc, size)
        C = torch.zeros(case["m"] * case["n"], dtype=torch.float64, device="cuda")
        s.update(A=A, B=B, C=C, a=block_list(A, ar, ac, size), b=block_list(B, br, bc, size),
                 c=block_list(C, case["m"], case["n"], size))
    else:
        A, B, _ = gemm_inputs(case, seed)
        for name, x in (("A", A), ("B", B)):
            s[name] = torch.empty(x.shape, dtype=torch.float64, pin_memory=True)
            s[name].copy_(x)
        s["C"] = torch.empty((case["n"], case["m"]), dtype=torch.float64, pin_memory=True)
    return s


# ---------------------------------------------------------------------- run
def run(s):
    case, h = s["case"], s["handle"]
    kind = case["kind"]
    if kind == "transform":
        (src, lds), (dst, ldd) = ca.colmajor(s["src"]), ca.colmajor(s["dst"])
        rows, cols = case["rows"], case["cols"]
        if s["dst0"] is not None:
            h.block_transform("N", rows, cols, 1.0, s["dst0"].data_ptr(), ldd, 0.0, dst, ldd)
        h.block_transform(case["op"], rows, cols, 1.0, src, lds, case["beta"], dst, ldd)
        return s["dst"]
    if kind == "grouped":
        s["plan"].graph_run()
        return s["C"]
    m, n, k = case["m"], case["n"], case["k"]
    if kind == "layout":
        h.dgemm_layout(case["ta"], case["tb"], m, n, k, 1.0, s["a"], s["b"], 0.0, s["c"])
        return s["C"]
    (a, lda), (b, ldb), (c, ldc) = ca.colmajor(s["A"]), ca.colmajor(s["B"]), ca.colmajor(s["C"])
    if kind == "gemm":
        if s["C0"] is not None:
            h.block_transform("N", m, n, 1.0, s["C0"].data_ptr(), ldc, 0.0, c, ldc)
        h.dgemm(case["ta"], case["tb"], m, n, k, case["alpha"], a, lda, b, ldb, case["beta"], c, ldc)
        return s["C"]
    if kind == "ozaki":
        info = h.dgemm_ozaki(case["ta"], case["tb"], m, n, k, 1.0, a, lda, b, ldb, 0.0, c, ldc)
        return {"c": s["C"], "count": info["count"], "bits": info["bits"]}
    h.dgemm_host(case["ta"], case["tb"], m, n, k, 1.0, a, lda, b, ldb, 0.0, c, ldc)
    return s["C"]


def work(case):
    kind = case["kind"]
    if kind == "transform":
        rows_cols = 8.0 * case["rows"] * case["cols"]
        return {"bytes": rows_cols * (5 if case["beta"] else 2), "flops": 0.0}
    if kind == "grouped":
        m, n, k = (batch_dims(case)[:, i].astype(float) for i in range(3))
        return {"bytes": float(8 * (m * k + k * n + m * n).sum()), "flops": float(2 * (m * n * k).sum())}
    m, n, k = float(case["m"]), float(case["n"]), float(case["k"])
    # beta != 0: C0 and C are read once more each and C is written twice
    return {"bytes": 8 * (m * k + k * n + m * n * (4 if case.get("beta") else 1)), "flops": 2 * m * n * k}


# -------------------------------------------------------------------- exact
def product(case, A, B):
    """op(A) op(B) of column-major operands as a column-major (n, m) tensor."""
    (ar, _), (br, _) = stored(case)
    A, B = A[:, :ar], B[:, :br]                       # (cols, rows): the transposes of the matrices
    left = B if case["tb"] == "N" else B.t()          # op(B)^T, n x k
    right = A if case["ta"] == "N" else A.t()         # op(A)^T, k x m
    return torch.mm(left, right)


def exact(case, seed):
    kind = case["kind"]
    if kind == "transform":
        src, dst0 = transform_inputs(case, seed)
        rows, cols = case["rows"], case["cols"]
        out = torch.zeros((cols, rows + case["pad"]), dtype=torch.float64, device="cuda")
        x = src[:, :rows] if case["op"] == "N" else src[:, :cols].t()
        out[:, :rows] = x if dst0 is None else x + case["beta"] * dst0[:, :rows]
        return out
    if kind == "grouped":
        d, A, B, offs = batch_inputs(case, seed)
        C = torch.zeros(int(offs[2][-1]), dtype=torch.float64, device="cuda")
        for i, (m, n, k) in enumerate(d.tolist()):
            a, b, c = (int(o[i]) for o in offs)
            C[c:c + m * n].view(n, m).copy_(torch.mm(B[b:b + k * n].view(n, k), A[a:a + m * k].view(k, m)))
        return C
    if kind == "ozaki":
        return {"c": product(case, *ozaki_inputs(case, seed)), "count": None, "bits": None}
    A, B, C0 = gemm_inputs(case, seed)
    X = product(case, A, B)
    if kind == "layout":
        return pack(X, case["m"], case["n"], case["block"])
    if kind == "host":
        return X.cpu()
    m, out = case["m"], torch.zeros((case["n"], case["m"] + case["pad"]), dtype=torch.float64, device="cuda")
    out[:, :m] = case["alpha"] * X + (case["beta"] * C0[:, :m] if C0 is not None else 0.0)
    return out
