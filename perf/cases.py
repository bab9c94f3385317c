"""The workloads this framework's speed is judged on, each as one pass through
its public entry points.

``listed()`` holds twelve cases and ``draw(rng)`` makes more of the same
ranges.  A case is a plain dict: ``op`` says which entry points a pass calls,
``kind`` which matrix family it runs on, and the rest are sizes and options.

Matrix families (the generators of the benchmark's configurations, restated
on the GPU so that a case is made in a fraction of a second):

* ``uniform``: about ``degree`` random columns in every row;
* ``powerlaw``: heavy-tailed degrees (exponent 1.8, at most 4096 per row),
  random columns;
* ``band``: 16x16 blocks on 33 block diagonals, a block kept with probability
  0.6 and an entry of it with 0.7;
* ``blocks``: half of the 16-row windows hold four random 16x16 blocks at 50%
  fill, the rows of the other half ``degree`` random columns;
* ``graph``: heavy-tailed degrees (exponent 2, at most 8192), 70% of the edges
  inside communities of 4096 nodes, nodes relabelled at random.
"""

import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ascend-spmm_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import spmm_npu  # noqa: E402

DTYPE = {"fp16": torch.float16, "fp32": torch.float32}
BYTES = {"fp16": 2, "fp32": 4}


def listed():
    return [
        # A small operator inside a larger program (a mini-batch, one relation of
        # many): launches and host time count.  Rows no multiple of 16, torch's
        # own int64 CSR indices.
        dict(name="csr_small_fp16_i64", op="csr", kind="uniform", rows=1021, degree=8, width=48,
             dtype="fp16", index=64),
        # The fp32 anchor configuration: 16384 rows, 8 nonzeros each, 128 features.
        dict(name="csr_uniform_fp32", op="csr", kind="uniform", rows=16384, degree=8, width=128,
             dtype="fp32", index=32),
        # The headline configuration: power-law rows, 2M nonzeros, 128 features.
        dict(name="csr_powerlaw_fp16", op="csr", kind="powerlaw", rows=100000, degree=20, width=128,
             dtype="fp16", index=32),
        # A block-structured matrix converted whole to 16x1 blocks (csr_to_bcsr),
        # every window on the matrix cores.
        dict(name="bcsr_band_fp16", op="bcsr", kind="band", rows=65536, degree=0, width=256,
             dtype="fp16", index=32),
        # The same matrix through the cost-model split (preprocess), both engines.
        dict(name="mixed_band_fp16", op="mixed", kind="band", rows=65536, degree=0, width=128,
             dtype="fp16", index=32),
        # The half-blocked, half-scattered configuration at its two widths.
        dict(name="mixed_blocks_fp16_n64", op="mixed", kind="blocks", rows=200000, degree=4, width=64,
             dtype="fp16", index=32),
        dict(name="mixed_blocks_fp16_n512", op="mixed", kind="blocks", rows=200000, degree=4, width=512,
             dtype="fp16", index=32),
        # The recommended path (preprocess, then spmm_ascend_cube) on a power-law
        # matrix whose row count is no multiple of the window.
        dict(name="mixed_powerlaw_fp16", op="mixed", kind="powerlaw", rows=99991, degree=20, width=128,
             dtype="fp16", index=32),
        # One training step's sparse part on a fixed graph: pack, A x, restore,
        # and the gradient with respect to x through the packed transpose.
        dict(name="graph_train_fp32", op="graph", kind="graph", rows=131072, degree=30, width=256,
             dtype="fp32", index=32),
        # Getting a new matrix ready: the cost-model split of the headline matrix,
        dict(name="preprocess_powerlaw_fp16", op="preprocess", kind="powerlaw", rows=100000, degree=20, width=0,
             dtype="fp16", index=32),
        # the packed graph layout with its transpose, for training on a graph,
        dict(name="preprocess_graph_fp32", op="preprocess_graph", kind="graph", rows=262144, degree=30, width=0,
             dtype="fp32", index=32),
        # and the whole-matrix conversion to blocks.
        dict(name="to_bcsr_band_fp16", op="to_bcsr", kind="band", rows=65536, degree=0, width=0,
             dtype="fp16", index=32),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# Most multiply-adds (nonzeros times features) and nonzeros of a drawn case.
_MOST_MACS = {"csr": 1.0e9, "bcsr": 3.6e9, "mixed": 1.8e9, "graph": 0.9e9}
_MOST_NNZ = 7.0e6


def draw(rng):
    op = rng.choice(["csr", "csr", "bcsr", "mixed", "mixed", "graph", "preprocess", "preprocess_graph", "to_bcsr"])
    kind = {"csr": lambda: rng.choice(["uniform", "powerlaw"]),
            "bcsr": lambda: rng.choice(["band", "blocks"]),
            "mixed": lambda: rng.choice(["band", "blocks", "powerlaw"]),
            "graph": lambda: "graph",
            "preprocess": lambda: rng.choice(["powerlaw", "band", "blocks"]),
            "preprocess_graph": lambda: "graph",
            "to_bcsr": lambda: rng.choice(["band", "blocks"])}[op]()
    dtype = "fp32" if kind == "graph" else rng.choice(["fp16", "fp16", "fp32"])
    index = rng.choice([32, 32, 64])
    degree = {"uniform": _log_int(rng, 4, 40), "powerlaw": rng.randint(10, 24), "band": 0,
              "blocks": rng.randint(2, 8), "graph": rng.randint(12, 32)}[kind]
    rows = {"uniform": _log_int(rng, 700, 200000), "powerlaw": _log_int(rng, 8000, 120000),
            "band": _log_int(rng, 2000, 65536), "blocks": _log_int(rng, 8000, 200000),
            "graph": _log_int(rng, 16384, 262144 if op == "preprocess_graph" else 131072)}[kind]
    width = 0
    case = dict(op=op, kind=kind, rows=rows, degree=degree, width=width, dtype=dtype, index=index)
    nnz = _nominal(case)[0]
    while op.startswith("preprocess") and nnz > _MOST_NNZ:
        case["rows"] = rows = rows // 2 + 1
        nnz = _nominal(case)[0]
    if op in _MOST_MACS:
        most = min(512 if dtype == "fp16" else 256, _MOST_MACS[op] / nnz)
        width = max(16, min(512, _log_int(rng, 16, max(most, 17)) // 16 * 16))
        case["width"] = width
    return case


# ------------------------------------------------------------------ matrices

def _degrees(g, rows, exponent, most, total):
    """Heavy-tailed degrees in [1, most] whose sum is close to total."""
    u = torch.rand(rows, generator=g, device="cuda", dtype=torch.float64).clamp_min(1e-12)
    d = torch.floor(u.pow(-1.0 / (exponent - 1.0))).clamp(1, most)
    f = 1.0
    for _ in range(12):
        now = torch.round(d * f).clamp(1, most).sum().item()
        f *= total / now
    return torch.round(d * f).clamp(1, most).long()


def _random_columns(g, degrees, cols):
    rows = torch.repeat_interleave(torch.arange(degrees.numel(), device="cuda"), degrees)
    return rows, torch.randint(0, cols, (rows.numel(),), generator=g, device="cuda")


def _relabelling(g, n, whole):
    """A random permutation of [0, n): of everything, or inside groups of 16."""
    if whole:
        return torch.randperm(n, generator=g, device="cuda")
    i = torch.arange(n, device="cuda")
    return torch.argsort(i // 16 * 2.0 + torch.rand(n, generator=g, device="cuda", dtype=torch.float64))


def _matrix(case, seed):
    """Square CSR with distinct ascending columns per row: (crow, col, value).

    The layout operators' output sizes follow from the pattern.  So that they
    are the same for every seed, those cases draw one pattern per case and the
    seed relabels it: rows inside their 16-row windows, and columns by the same
    permutation, or (scattered columns, no transpose) by any.
    """
    n, kind = case["rows"], case["kind"]
    g, relabel = torch.Generator(device="cuda"), case["op"] not in ("csr", "bcsr", "graph")
    g.manual_seed(131 * n + case["degree"] if relabel else 1_000_003 * seed + 2027)
    if kind == "uniform":
        r, c = _random_columns(g, torch.full((n,), case["degree"], device="cuda"), n)
    elif kind == "powerlaw":
        r, c = _random_columns(g, _degrees(g, n, 1.8, min(4096, n // 2), n * case["degree"]), n)
    elif kind == "graph":
        d = _degrees(g, n, 2.0, min(8192, n // 2), n * case["degree"])
        r, c = _random_columns(g, d, n)
        near = torch.rand(r.numel(), generator=g, device="cuda") < 0.7
        c = torch.where(near, (r // 4096 * 4096 + c % 4096).clamp_max(n - 1), c)
        label = torch.randperm(n, generator=g, device="cuda")
        r, c = label[r], label[c]
    elif kind == "band":
        nb = (n + 15) // 16
        keep = torch.rand(nb, 1, 33, 1, generator=g, device="cuda") < 0.6
        hit = (torch.rand(nb, 16, 33, 16, generator=g, device="cuda") < 0.7) & keep
        b, i, d, j = torch.nonzero(hit, as_tuple=True)
        r, c = 16 * b + i, 16 * (b + d - 16) + j
        ok = (r < n) & (c >= 0) & (c < n)
        r, c = r[ok], c[ok]
    else:  # blocks
        nb = (n + 15) // 16
        order = torch.randperm(nb, generator=g, device="cuda")
        bw, sw = order[: nb // 2], order[nb // 2:]
        at = torch.randint(0, nb, (bw.numel(), 4), generator=g, device="cuda")
        hit = torch.rand(bw.numel(), 4, 16, 16, generator=g, device="cuda") < 0.5
        w, k, i, j = torch.nonzero(hit, as_tuple=True)
        r, c = 16 * bw[w] + i, 16 * at[w, k] + j
        rs = (16 * sw[:, None] + torch.arange(16, device="cuda")).reshape(-1).repeat_interleave(case["degree"])
        cs = torch.randint(0, n, (rs.numel(),), generator=g, device="cuda")
        r, c = torch.cat([r, rs]), torch.cat([c, cs])
        ok = (r < n) & (c < n)
        r, c = r[ok], c[ok]
    if relabel:
        g.manual_seed(1_000_003 * seed + 2027)
        rows = _relabelling(g, n, False)
        r, c = rows[r], (_relabelling(g, n, True) if kind in ("uniform", "powerlaw") else rows)[c]
    if kind != "band" or relabel:  # a fresh band comes in row order and distinct
        key = torch.unique(r * n + c)
        r, c = key // n, key % n
    crow = torch.zeros(n + 1, dtype=torch.long, device="cuda")
    crow[1:] = torch.cumsum(torch.bincount(r, minlength=n), 0)
    if kind == "graph":
        value = torch.rand(c.numel(), generator=g, device="cuda")
    else:
        value = 2.0 * torch.rand(c.numel(), generator=g, device="cuda") - 1.0
    index = torch.int32 if case["index"] == 32 else torch.int64
    return crow.to(index), c.to(index), value.to(DTYPE[case["dtype"]])


def _dense(case, seed, salt=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(1_000_003 * seed + 7919 + salt)
    return torch.randn(case["rows"], case["width"], generator=g, device="cuda").to(DTYPE[case["dtype"]])


# -------------------------------------------------------------------- a pass

_BLOCK_KEYS = ("crow_window_ptr", "unique_col_ids", "value")
_VECTOR_KEYS = ("vrow_window_ptr", "vcol_indices", "vvalue")


def prepare(case, seed):
    """What a program holds before the pass: the matrix in the layout the pass
    takes, the partition starts the operators' signatures ask for, the node
    features (and the gradient that arrives at the output)."""
    n, op = case["rows"], case["op"]
    crow, col, value = _matrix(case, seed)
    state = {"op": op, "n": n}
    if op in ("preprocess", "preprocess_graph", "to_bcsr"):
        state["csr"] = (crow, col, value)
    elif op == "csr":
        state["args"] = (crow, col, value, _dense(case, seed), spmm_npu.make_start(crow, 40).cuda())
    elif op == "bcsr":
        p = spmm_npu.csr_to_bcsr(crow, col, value, n, n, 16)
        state["args"] = tuple(p[k] for k in _BLOCK_KEYS) + (
            torch.zeros(n + 1, dtype=crow.dtype, device="cuda"), col[:0], value[:0], _dense(case, seed),
            spmm_npu.make_start(p["crow_window_ptr"], 20).cuda(), torch.zeros(40, dtype=torch.int32, device="cuda"))
    elif op == "mixed":
        p = spmm_npu.preprocess(crow, col, value, n, n)
        state["args"] = tuple(p[k] for k in _BLOCK_KEYS + _VECTOR_KEYS) + (
            _dense(case, seed), spmm_npu.make_start(p["crow_window_ptr"], 20).cuda(),
            spmm_npu.make_start(p["vrow_window_ptr"], 40).cuda())
        state["permutation"] = p["permutation"]
    else:  # graph
        prep = spmm_npu.preprocess(crow, col, value, n, n, graph_layout=True)
        state["graph"] = spmm_npu.PackedGraph(prep)
        state["x"] = _dense(case, seed).requires_grad_()
        state["grad"] = _dense(case, seed, salt=1)
    return state


def run(state):
    op, n = state["op"], state["n"]
    if op == "csr":
        return spmm_npu.spmm_csr(*state["args"])
    if op in ("bcsr", "mixed"):
        return spmm_npu.spmm_ascend_cube(*state["args"])
    if op == "graph":
        g = state["graph"]
        y = g.restore(g(g.pack(state["x"])))
        (dx,) = torch.autograd.grad(y, state["x"], state["grad"])
        return {"y": y.detach(), "dx": dx}
    if op == "to_bcsr":
        return spmm_npu.csr_to_bcsr(*state["csr"], n, n, 16)
    return spmm_npu.preprocess(*state["csr"], n, n, graph_layout=op == "preprocess_graph")


# ------------------------------------------------------- work and tolerances

def _nominal(case):
    """Expected (nonzeros, 16x1 blocks of the whole matrix)."""
    n, d = case["rows"], case["degree"]
    if case["kind"] == "band":
        windows = n / 16.0
        mean = 33.0 - 272.0 / max(windows, 33.0)  # block diagonals cut off at both ends
        return windows * mean * 0.6 * 0.7 * 256, windows * mean * 0.6 * 16
    if case["kind"] == "blocks":
        return n / 2.0 * (32 + d), n / 2.0 * (4.0 + d)
    return float(n) * d, float(n) * d


def work(case):
    """Each input read once and each output written once (4-byte indices:
    4 (M + 1) + (4 + s) nnz for the matrix, s N K and s N M for the dense
    operand and the result); 2 nnz N operations."""
    n, w, s, ix = case["rows"], case["width"], BYTES[case["dtype"]], case["index"] // 8
    nnz, blocks = _nominal(case)
    matrix = ix * (n + 1) + (ix + s) * nnz
    if case["op"] in ("csr", "bcsr", "mixed"):
        return {"bytes": matrix + 2.0 * s * w * n, "flops": 2.0 * nnz * w}
    if case["op"] == "graph":  # x and the gradient in, y and dx out; the matrix and its transpose
        return {"bytes": 2.0 * matrix + 4.0 * s * w * n, "flops": 4.0 * nnz * w}
    whole = (ix + 16 * s) * blocks
    if case["op"] == "to_bcsr":
        return {"bytes": matrix + whole + ix * n / 16.0, "flops": 0.0}
    # The cost model gives blocks / 295 = vector nonzeros / 505: of scattered
    # nonzeros (a block each) 295 / 800 become blocks.
    share = min(1.0, 295.0 * nnz / (505.0 * blocks + 295.0 * nnz))
    split = share * whole + (1.0 - share * blocks / nnz) * (ix + s) * nnz + ix * n + 16.0 * n
    if case["op"] == "preprocess":
        return {"bytes": matrix + split, "flops": 0.0}
    return {"bytes": matrix + 2.0 * split, "flops": 0.0}


def tolerance(case):
    """Layouts are integers and copied values: exact.  Products: about four
    times the distance from 64-bit sums measured on the listed cases (fp16:
    the one rounding of the result; fp32: the 32-bit sums)."""
    if case["op"] in ("preprocess", "preprocess_graph", "to_bcsr"):
        return "exact"
    return {"rel": 8e-4} if case["dtype"] == "fp16" else {"rel": 2e-6}


def _product(crow, col, value, x):
    """A x in 64 bits: products summed by row, a slice of nonzeros at a time."""
    rows = torch.repeat_interleave(torch.arange(crow.numel() - 1, device="cuda"), crow.long().diff())
    out = torch.zeros(crow.numel() - 1, x.size(1), dtype=torch.float64, device="cuda")
    x, value, col = x.double(), value.double(), col.long()
    step = max(1, 100_000_000 // x.size(1))
    for a in range(0, col.numel(), step):
        part = slice(a, a + step)
        out.index_add_(0, rows[part], value[part, None] * x[col[part]])
    return out


def exact(case, seed):
    op = case["op"]
    if op in ("preprocess", "preprocess_graph", "to_bcsr"):
        return None  # integers and copied values
    crow, col, value = _matrix(case, seed)
    x = _dense(case, seed)
    out = _product(crow, col, value, x)
    if op == "csr":
        return out
    n = case["rows"]
    if op == "bcsr":  # whole windows
        return torch.cat([out, out.new_zeros(-n % 16, out.size(1))])
    if op == "graph":
        rows = torch.repeat_interleave(torch.arange(n, device="cuda"), crow.long().diff())
        order = torch.argsort(col.long() * n + rows)
        tcrow = torch.zeros(n + 1, dtype=torch.long, device="cuda")
        tcrow[1:] = torch.cumsum(torch.bincount(col.long(), minlength=n), 0)
        return {"y": out, "dx": _product(tcrow, rows[order], value[order], _dense(case, seed, salt=1))}
    # mixed: the split's row order (-1: a padding row, zero)
    order = _packed_rows(crow, col, n)
    if order is None:
        return None
    return torch.where(order[:, None] >= 0, out[order.clamp_min(0)], out.new_zeros(()))


def _packed_rows(crow, col, n):
    """Original row of each packed row (-1: padding): the windows by density
    (nonzeros per block, ties in order), block windows 16 rows each, then the
    vector windows' own rows.  Only a last window of fewer than 16 rows needs
    the split's boundary; None when that window is the marginal one."""
    nwin = -(-n // 16)
    rows = torch.repeat_interleave(torch.arange(n, device="cuda"), crow.long().diff())
    nnz = torch.bincount(rows // 16, minlength=nwin)
    blocks = torch.bincount(torch.unique(rows // 16 * n + col.long()) // n, minlength=nwin)
    density = torch.where(blocks > 0, nnz.double() / blocks.clamp_min(1).double(), 0.0)
    windows = torch.sort(density, descending=True, stable=True)[1]
    packed = (16 * windows[:, None] + torch.arange(16, device="cuda")).reshape(-1)
    if n % 16 == 0:
        return packed
    after = torch.cumsum(blocks[windows], 0).double() / 295.0
    left = (nnz.sum() - torch.cumsum(nnz[windows], 0)).double() / 505.0
    reached = torch.nonzero(after >= left)
    boundary = int(reached[0]) if reached.numel() else -1
    at = int(torch.nonzero(windows == nwin - 1)[0])
    if at == boundary:
        return None
    return torch.where(packed < n, packed, -1) if at < boundary else packed[packed < n]
