"""The products this library is used for, as measurable cases.

Every case is one step of a program that keeps its operands on the GPU and
repeats a product: the B operand is rebuilt (or takes new values), then
``rt.tilespgemm`` runs symbolic, allocate and numeric.  The result is C's tile
structure and values where they are left on the device, except for the
"host" cases, whose program takes C back as a host CSR.

Kinds (sizes are the case's own):

laplace   C = A*A, 5-point 2D Laplacian of a g x g grid: the smallest product
          of a parity run or a coarse solver level, bound by launches.
random    C = A*B, rectangular with uniformly scattered columns and an
          independent B: unstructured graphs, sparse tiles, no locality.
stencil   C = A*A^T, 27-point stencil on a g^3 grid: the benchmark's product
          (normal equations, strength-of-connection matrices).
fem       C = A*A, block FEM with dense 4x4 node blocks, magnitudes over six
          decades, on the FP64 matrix cores.
split     the same in the split-BF16 precision.
bgrf      the driver's default layout: A in the BGRF order, C exported to the
          host and its rows restored, as a program does that hands C on.
banded    C = A*A of one banded problem per call.
batch     many banded problems in one block-diagonal call.
amg       Galerkin products R*(A*P) of several 7-point hierarchies in two
          block-diagonal calls (set-up phase of a multigrid solver).
values    A*P with an unchanged P structure and new P values from the host
          (time stepping): values-only B update and the product.
rmat      C = A*A of an R-MAT graph: hub rows, the longest rows and the
          largest C.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(_ROOT, "rtt-spgemm_amd") not in sys.path:
    sys.path.insert(0, os.path.join(_ROOT, "rtt-spgemm_amd"))

import rtt_amd as rt  # noqa: E402


def listed():
    return [
        # The benchmark's smallest configuration: 4096 rows, all latency.
        {"name": "laplace-64-aa", "kind": "laplace", "g": 64},
        # An unstructured rectangular product with ragged sizes.
        {"name": "random-20011x15013", "kind": "random", "m": 20011, "k": 15013, "n": 17017,
         "per_a": 8, "per_b": 6},
        # An ordinary normal-equations product, 262k rows.
        {"name": "stencil-64-aat", "kind": "stencil", "g": 64},
        # The headline product, 2.1M rows and 2.5e8 entries of C.
        {"name": "stencil-128-aat", "kind": "stencil", "g": 128},
        # The matrix-core path at the benchmark's size.
        {"name": "fem-500k-aa", "kind": "fem", "nodes": 500000},
        # Split precision, as the benchmark's comparison runs it.
        {"name": "fem-50k-split", "kind": "split", "nodes": 50000},
        # The driver's default flow end to end: BGRF layout, C on the host.
        {"name": "fem-20k-bgrf-host", "kind": "bgrf", "nodes": 20000},
        # One problem per call, the median problem of the banded batch.
        {"name": "banded-16k", "kind": "banded", "rows": 16000, "bandwidth": 32, "per_row": 17},
        # 64 such problems (log-normal sizes) in one call.
        {"name": "banded-batch-64", "kind": "batch", "problems": 64},
        # Eight AMG hierarchies in two calls, as in the benchmark.
        {"name": "amg-batch-8", "kind": "amg", "problems": 8, "g_lo": 32, "g_hi": 96},
        # New values on an unchanged structure, every step.
        {"name": "amg-values-64", "kind": "values", "g": 64},
        # Hub rows and wide rows: the second benchmark mode's family.
        {"name": "rmat-18-aa", "kind": "rmat", "scale": 18, "edge_factor": 16},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["laplace", "random", "stencil", "stencil", "fem", "fem", "split", "bgrf",
                       "banded", "batch", "amg", "values", "rmat"])
    if kind == "laplace":
        return {"kind": kind, "g": _log_int(rng, 9, 900)}
    if kind == "random":
        return {"kind": kind, "m": _log_int(rng, 500, 120000), "k": _log_int(rng, 500, 120000),
                "n": _log_int(rng, 500, 120000), "per_a": rng.randint(1, 16),
                "per_b": rng.randint(1, 16)}
    if kind == "stencil":
        return {"kind": kind, "g": _log_int(rng, 9, 127)}
    if kind == "fem":
        return {"kind": kind, "nodes": _log_int(rng, 700, 480000)}
    if kind == "split":
        return {"kind": kind, "nodes": _log_int(rng, 700, 100000)}
    if kind == "bgrf":
        return {"kind": kind, "nodes": _log_int(rng, 300, 30000)}
    if kind == "banded":
        return {"kind": kind, "rows": _log_int(rng, 1000, 200000),
                "bandwidth": rng.randint(8, 64), "per_row": rng.randint(5, 30)}
    if kind == "batch":
        return {"kind": kind, "problems": rng.randint(3, 63)}
    if kind == "amg":
        lo = rng.randint(12, 48)
        return {"kind": kind, "problems": rng.randint(1, 7), "g_lo": lo,
                "g_hi": lo + rng.randint(1, 48)}
    if kind == "values":
        return {"kind": kind, "g": _log_int(rng, 11, 97)}
    return {"kind": kind, "scale": rng.randint(9, 17), "edge_factor": rng.choice([6, 8, 12, 16])}


# ---- operands ------------------------------------------------------------------

# A case's structure is its own; the seed gives the values.
STRUCTURE = 20260101


def _uniform(n, seed, lo, hi):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    gen = torch.Generator(device=dev).manual_seed(seed)
    x = torch.rand(n, dtype=torch.float64, device=dev, generator=gen)
    return x.mul_(hi - lo).add_(lo).cpu().numpy()


def _with_values(a, seed):
    """The same matrix with values U[-1, 1] drawn from the seed."""
    return rt.CsrMatrix(a.m, a.n, a.rowptr, a.col, _uniform(a.nnz, seed, -1.0, 1.0))


def _fem(nodes, spatial, seed):
    """Block FEM with magnitudes 10^U[-3, 3] and random signs, as the generator draws them."""
    a = rt.gen_fem_blocks(nodes, 6, spatial, STRUCTURE)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    u = torch.from_numpy(_uniform(a.nnz, seed, -6.0, 6.0)).to(dev)
    sign = torch.where(u < 0, -1.0, 1.0).to(torch.float64)
    a.val = (sign * torch.pow(10.0, u.abs() - 3.0)).cpu().numpy()
    return a


def _batch_shapes(case):
    return rt.gen_banded_batch_shapes(case["problems"], seed=STRUCTURE)


def _amg_grids(case):
    return np.random.default_rng(STRUCTURE).integers(case["g_lo"], case["g_hi"] + 1,
                                                     case["problems"])


def _amg_parts(case, seed):
    gs = _amg_grids(case)
    A = [rt.gen_poisson7_jumps(int(g), 3.0, seed + p) for p, g in enumerate(gs)]
    P = [rt.gen_aggregation_prolongator(a, int(g)) for a, g in zip(A, gs)]
    R = [rt.csr_transpose(p) for p in P]
    return tuple(rt.block_diag(x, 8)[0] for x in (A, P, R))


def _square(case, seed):
    """A of the kinds that form A*A or A*A^T."""
    kind = case["kind"]
    if kind == "laplace":
        return rt.gen_laplace2d(case["g"], 0.1, seed)
    if kind == "stencil":
        return rt.gen_stencil27(case["g"], 0.5, 1.5, seed)
    if kind in ("fem", "split"):
        return _fem(case["nodes"], True, seed)
    if kind == "bgrf":
        return _fem(case["nodes"], False, seed)
    if kind == "banded":
        return _with_values(rt.gen_banded(case["rows"], case["bandwidth"], case["per_row"],
                                          STRUCTURE), seed)
    if kind == "batch":
        rows, bw, per = _batch_shapes(case)
        return _with_values(rt.block_diag([
            rt.gen_banded(int(r), int(b), int(p), STRUCTURE + i)
            for i, (r, b, p) in enumerate(zip(rows, bw, per))], 8)[0], seed)
    return _with_values(rt.gen_rmat(case["scale"], case["edge_factor"], seed=STRUCTURE), seed)


def _random_pair(case, seed):
    return (_with_values(rt.gen_random(case["m"], case["k"], case["per_a"], STRUCTURE), seed),
            _with_values(rt.gen_random(case["k"], case["n"], case["per_b"], STRUCTURE + 1),
                         seed + 1))


def _values_parts(case, seed):
    A = rt.gen_poisson7_jumps(case["g"], 3.0, seed)
    P = rt.gen_aggregation_prolongator(A, case["g"])
    return A, P, P.val * _uniform(P.nnz, seed, 0.5, 1.5)


def prepare(case, seed):
    if not rt.initialised():
        rt.init(0)
    kind = case["kind"]
    precision = "split-bf16" if kind == "split" else "fp64"
    s = {"kind": kind, "b": None, "aat": 1 if kind == "stencil" else 0,
         "sched": rt.schedule(materialize_output=kind == "bgrf", precision=precision)}
    if kind == "random":
        A, B = _random_pair(case, seed)
        s["a"], s["src"] = rt.prepare_identity_a(A), rt.upload_csr(B)
    elif kind == "values":
        A, P, s["new"] = _values_parts(case, seed)
        s["a"], s["src"] = rt.prepare_identity_a(A), rt.upload_csr(P)
        s["b"] = rt.rebuild_b_general(s["a"], s["src"])
    elif kind == "amg":
        A, P, R = _amg_parts(case, seed)
        s["a"], s["src"], s["r"] = rt.prepare_identity_a(A), rt.upload_csr(P), rt.prepare_identity_a(R)
        # A*P as the second product's operand, as the benchmark prepares it.
        tc, _ = rt.tilespgemm(s["a"], rt.rebuild_b_general(s["a"], s["src"]), rt.schedule())
        s["src2"], s["b2"] = rt.upload_csr(rt.tile2csr(tc)), None
    elif kind == "bgrf":
        s["a"] = rt.prepare_bgrf_a(_square(case, seed))
        s["rows"] = s["a"].row_new_to_old()
    else:
        s["a"] = rt.prepare_identity_a(_square(case, seed))
    return s


# ---- one step ------------------------------------------------------------------

class _Device:
    """Device memory of the library as torch sees foreign arrays.  A tensor made from it keeps
    it, and with it the handle that owns the memory."""

    def __init__(self, owner, ptr, n, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (int(n),), "typestr": typestr,
                                         "data": (int(ptr), False), "version": 2}


def _device_c(a):
    """C as the last product on `a` left it: every array, where it lies."""
    v = rt.DeviceC()
    if rt.load().rtt_last_c_view(a.handle, ctypes.byref(v)) != rt.RTT_OK:
        raise RuntimeError("no C on this handle")
    t, z, r = v.num_tiles, v.nnz, v.tilem
    out = {}
    for name, n, ts, dt in (("tile_ptr", r + 1, "<i8", torch.int64),
                            ("tile_col", t, "<i4", torch.int32),
                            ("tile_mask", t, "<i8", torch.int64),
                            ("tile_nnz", t + 1, "<i8", torch.int64),
                            ("tile_csr_ptr", 8 * t, "|u1", torch.uint8),
                            ("tile_csr_col", z, "|u1", torch.uint8),
                            ("tile_csr_val", z, "<f8", torch.float64)):
        out[name] = (torch.as_tensor(_Device(a, getattr(v, name), n, ts), device="cuda") if n
                     else torch.empty(0, dtype=dt, device="cuda"))
    return out


def run(s):
    kind = s["kind"]
    if kind == "values":
        s["src"].set_values(s["new"])
        rt.update_b_values(s["a"], s["src"], s["b"])
    elif kind in ("random", "amg"):
        s["b"] = rt.rebuild_b_general(s["a"], s["src"], s["b"])
    else:
        s["b"] = rt.rebuild_b(s["a"], s["aat"], s["b"])
    tc, _ = rt.tilespgemm(s["a"], s["b"], s["sched"])
    if kind == "bgrf":
        c = (rt.tile2csr_restore_rows(tc, s["rows"], len(s["rows"])) if s["rows"] is not None
             else rt.tile2csr(tc))
        return {"rowptr": c.rowptr, "col": c.col, "val": c.val}
    if kind == "amg":
        s["b2"] = rt.rebuild_b_general(s["r"], s["src2"], s["b2"])
        rt.tilespgemm(s["r"], s["b2"], s["sched"])
        return {"ap": _device_c(s["a"]), "rap": _device_c(s["r"])}
    return _device_c(s["a"])


# ---- work and exact values -------------------------------------------------------

def _banded_counts(rows, bandwidth, per_row):
    """(nnz, products, nnz of C) of a banded product, expected."""
    width = 2 * bandwidth + 1
    p = min(1.0, per_row / width)
    fill = sum(1.0 - math.exp(-p * p * (width - abs(d)))
               for d in range(-2 * bandwidth, 2 * bandwidth + 1))
    per = min(per_row, width) + 1 - p
    return rows * per, rows * per * per, rows * min(fill, 4 * bandwidth + 1)


def _counts(case):
    """[(nnz A, nnz B, products, nnz C, rows)] of the step's products."""
    kind = case["kind"]
    if kind == "laplace":
        g = case["g"]
        nnz = 5 * g * g - 4 * g
        return [(nnz, nnz, 25 * (g - 2) ** 2 + 64 * (g - 2) + 36, 13 * g * g - 20 * g + 4, g * g)]
    if kind == "stencil":
        g = case["g"]
        return [((3 * g - 2) ** 3, (3 * g - 2) ** 3, (9 * g - 10) ** 3, (5 * g - 6) ** 3, g ** 3)]
    if kind in ("fem", "split", "bgrf"):
        n = case["nodes"]
        return [(130.6 * n, 130.6 * n, 4360 * n, 411 * n, 4 * n)]
    if kind == "random":
        a, p = case["m"] * min(case["per_a"], case["k"]), min(case["per_b"], case["n"])
        fill = case["n"] * (1.0 - math.exp(-min(case["per_a"], case["k"]) * p / case["n"]))
        return [(a, case["k"] * p, a * p, case["m"] * fill, case["m"])]
    if kind == "banded":
        nnz, products, c = _banded_counts(case["rows"], case["bandwidth"], case["per_row"])
        return [(nnz, nnz, products, c, case["rows"])]
    if kind == "batch":
        shapes = zip(*(x.tolist() for x in _batch_shapes(case)))
        nnz, products, c, rows = (sum(x) for x in zip(*(
            (*_banded_counts(r, b, p), r) for r, b, p in shapes)))
        return [(nnz, nnz, products, c, rows)]
    if kind in ("amg", "values"):
        gs = ([case["g"]] if kind == "values" else
              _amg_grids(case))
        n = float(sum(int(g) ** 3 for g in gs))
        first = (6.9 * n, 3.85 * n, 26.5 * n, 9.4 * n, n)
        return [first] if kind == "values" else [first, (3.85 * n, 9.4 * n, 36.5 * n, 3.7 * n, n / 8)]
    f = case["edge_factor"] / 16.0
    n = 2.0 ** case["scale"]
    per = 14.3 * 1.017 ** (case["scale"] - 15) * f
    return [(per * n, per * n, 4466 * 1.36 ** (case["scale"] - 15) * f * f * n,
             1759 * 1.41 ** (case["scale"] - 15) * f ** 1.7 * n, n)]


def work(case):
    """Compressed operands read once and C written once (12 bytes an entry, 4 a row), and two
    operations a scalar product."""
    got = _counts(case)
    return {"bytes": float(sum(12 * (a + b + c) + 12 * r for a, b, _, c, r in got)),
            "flops": float(sum(2 * p for _, _, p, _, _ in got))}


MOST_PRODUCTS = 5e8   # beyond this the expansion below takes too long
BLOCK_PRODUCTS = 3e7


def _product(a, b, order):
    """Values of a * b in float64 by expanding every scalar product and summing
    the ones of an entry: entries in the order of 8x8 tiles (`order` "tiles":
    tile row, tile column, then row by row) or of a CSR ("rows")."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    arp, acol, aval = (torch.from_numpy(np.asarray(x)).to(dev) for x in (a.rowptr, a.col, a.val))
    brp, bcol, bval = (torch.from_numpy(np.asarray(x)).to(dev) for x in (b.rowptr, b.col, b.val))
    arp, brp, acol, bcol = arp.long(), brp.long(), acol.long(), bcol.long()
    arow = torch.repeat_interleave(torch.arange(a.m, device=dev), arp[1:] - arp[:-1])
    count = (brp[1:] - brp[:-1])[acol]
    before = torch.zeros(acol.numel() + 1, dtype=torch.long, device=dev)
    torch.cumsum(count, 0, out=before[1:])
    # Blocks of whole tile rows with about BLOCK_PRODUCTS products each.
    starts = arp[torch.clamp(torch.arange(0, a.m + 8, 8, device=dev), max=a.m)]
    cum = before[starts].cpu().numpy()
    edges, at = starts.cpu().numpy(), 0
    tiles = (b.n + 7) // 8
    vals, cols, rows = [], [], []
    while at < len(cum) - 1:
        to = max(at + 1, int(np.searchsorted(cum, cum[at] + BLOCK_PRODUCTS, side="right")) - 1)
        e0, e1, total = int(edges[at]), int(edges[to]), int(cum[to] - cum[at])
        at = to
        if not total:
            continue
        e = torch.repeat_interleave(torch.arange(e0, e1, device=dev), count[e0:e1])
        f = brp[acol[e]] + torch.arange(total, device=dev) - (before[e] - before[e0])
        i, j = arow[e], bcol[f]
        key = (i * b.n + j if order == "rows" else
               ((i // 8) * tiles + j // 8) * 64 + (i % 8) * 8 + j % 8)
        uniq, where = torch.unique(key, return_inverse=True)
        vals.append(torch.zeros(uniq.numel(), dtype=torch.float64, device=dev)
                    .index_add_(0, where, aval[e] * bval[f]))
        if order == "rows":
            rows.append(torch.div(uniq, b.n, rounding_mode="floor"))
            cols.append(uniq % b.n)
    val = torch.cat(vals) if vals else torch.zeros(0, dtype=torch.float64, device=dev)
    if order != "rows":
        return val
    row = torch.cat(rows) if rows else torch.zeros(0, dtype=torch.long, device=dev)
    col = torch.cat(cols) if cols else torch.zeros(0, dtype=torch.long, device=dev)
    ptr = np.zeros(a.m + 1, np.int64)
    ptr[1:] = torch.cumsum(torch.bincount(row, minlength=a.m), 0).cpu().numpy()
    return rt.CsrMatrix(a.m, b.n, ptr, col.cpu().numpy(), val.cpu().numpy())


def _transpose(a):
    order = np.argsort(a.col, kind="stable")
    rows = np.repeat(np.arange(a.m), np.diff(a.rowptr))
    ptr = np.zeros(a.n + 1, np.int64)
    ptr[1:] = np.cumsum(np.bincount(a.col, minlength=a.n))
    return rt.CsrMatrix(a.n, a.m, ptr, rows[order], a.val[order])


def _tiled(val):
    return {"tile_ptr": None, "tile_col": None, "tile_mask": None, "tile_nnz": None,
            "tile_csr_ptr": None, "tile_csr_col": None, "tile_csr_val": val}


def exact(case, seed):
    kind = case["kind"]
    if sum(p for _, _, p, _, _ in _counts(case)) > MOST_PRODUCTS:
        return None
    if kind == "amg":
        A, P, R = _amg_parts(case, seed)
        ap = _product(A, P, "rows")
        return {"ap": _tiled(_product(A, P, "tiles")), "rap": _tiled(_product(R, ap, "tiles"))}
    if kind == "values":
        A, P, new = _values_parts(case, seed)
        return _tiled(_product(A, rt.CsrMatrix(P.m, P.n, P.rowptr, P.col, new), "tiles"))
    if kind == "random":
        return _tiled(_product(*_random_pair(case, seed), "tiles"))
    A = _square(case, seed)
    if kind == "bgrf":
        c = _product(A, A, "rows")
        return {"rowptr": None, "col": None, "val": c.val}
    return _tiled(_product(A, _transpose(A) if kind == "stencil" else A, "tiles"))
