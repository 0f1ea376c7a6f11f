"""Performance cases of the SpGEMM library: C = A . B in CSR on the GPU.

Every case is a product (or a batch of products) that programs built on
this library run, called through the package's public functions.  The
matrices follow the repository's own workloads (gpuspgemm_amd/generators.py:
uniform, power-law, 27-point stencil, batched instances), drawn here with
torch on the GPU so that new inputs take fractions of a second, plus two
generic ones of the same families: a stencil with several unknowns per grid
node and a denser power-law graph.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import gpuspgemm_amd as g

DEV = "cuda"
CHUNK = 1 << 25  # products expanded at once by the 64-bit product below


def listed() -> list[dict]:
    return [
        # a small linear-algebra call inside a larger program: latency and launches count
        {"name": "uniform_1k", "kind": "uniform", "m": 1024, "per_row": 8, "dtype": "f64"},
        # the small uniform workload of the tests and the benchmark, in single precision
        {"name": "uniform_4k_f32", "kind": "uniform", "m": 4096, "per_row": 8, "dtype": "f32"},
        # squaring a web-like graph of ordinary size (short rows, a few long ones)
        {"name": "powerlaw_50k", "kind": "powerlaw", "m": 50_000, "x_min": 1.2, "dtype": "f64"},
        # the headline workload: a million-row power-law matrix squared
        {"name": "powerlaw_1m", "kind": "powerlaw", "m": 1_000_000, "x_min": 1.2, "dtype": "f64"},
        # the same in single precision, as graph programs often run it
        {"name": "powerlaw_1m_f32", "kind": "powerlaw", "m": 1_000_000, "x_min": 1.2, "dtype": "f32"},
        # a coarse level of a multigrid set-up: the 27-point stencil on 32^3 points
        {"name": "stencil_32", "kind": "grid", "g": 32, "dof": 1, "dtype": "f64"},
        # a middle level on an odd grid, in single precision
        {"name": "stencil_61_f32", "kind": "grid", "g": 61, "dof": 1, "dtype": "f32"},
        # the finest level: the benchmark's 96^3 stencil squared
        {"name": "stencil_96", "kind": "grid", "g": 96, "dof": 1, "dtype": "f64"},
        # a finite-element matrix with three unknowns per node (81 entries a row, as in
        # structural mechanics): many products per entry of C
        {"name": "elastic_27", "kind": "grid", "g": 27, "dof": 3, "dtype": "f64"},
        # two-hop neighbourhoods of a denser graph: rows of C from tens to tens of thousands of entries
        {"name": "graph_100k", "kind": "powerlaw", "m": 100_000, "x_min": 8.0, "dtype": "f64"},
        # a product of two different rectangular matrices with ragged rows, a third of them skewed
        {"name": "pair_131k", "kind": "pair", "m": 131_071, "k": 70_001, "n": 99_991, "dtype": "f64"},
        # many independent products of uneven sizes in one call
        {"name": "batch_20", "kind": "batch", "count": 20, "lo": 1_000, "hi": 200_000, "dtype": "f64"},
    ]


def _log_uniform(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["uniform", "powerlaw", "powerlaw", "grid", "grid", "elastic", "graph", "pair", "batch"])
    dtype = rng.choice(["f64", "f64", "f32"])
    if kind == "uniform":
        return {"kind": "uniform", "m": _log_uniform(rng, 1_000, 300_000), "per_row": rng.randint(3, 24), "dtype": dtype}
    if kind == "powerlaw":
        return {"kind": "powerlaw", "m": _log_uniform(rng, 3_000, 1_000_000), "x_min": round(rng.uniform(1.0, 2.5), 2),
                "dtype": dtype}
    if kind == "grid":
        return {"kind": "grid", "g": _log_uniform(rng, 10, 96), "dof": 1, "dtype": dtype}
    if kind == "elastic":
        dof = rng.randint(2, 4)
        return {"kind": "grid", "g": _log_uniform(rng, 6, {2: 40, 3: 28, 4: 20}[dof]), "dof": dof, "dtype": dtype}
    if kind == "graph":
        return {"kind": "powerlaw", "m": _log_uniform(rng, 5_000, 120_000), "x_min": round(rng.uniform(4.0, 10.0), 2),
                "dtype": dtype}
    if kind == "pair":
        return {"kind": "pair", "m": _log_uniform(rng, 2_000, 200_000), "k": _log_uniform(rng, 2_000, 200_000),
                "n": _log_uniform(rng, 2_000, 200_000), "dtype": dtype}
    return {"kind": "batch", "count": rng.randint(2, 20), "lo": 1_000, "hi": _log_uniform(rng, 10_000, 200_000),
            "dtype": dtype}


# ---------------------------------------------------------------- inputs

# A case fixes the sizes of its matrices and where their entries lie, up to a cyclic renumbering of all indices; the
# seed draws the renumbering and the values.  So two seeds give different arrays of the same lengths, C's included.

def _generator(seed: int, stream: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed((seed * 1_000_003 + stream) & 0x7FFFFFFF)


def _rand(n: int, gen: torch.Generator) -> torch.Tensor:
    return torch.rand(n, generator=gen, device=DEV, dtype=torch.float64)


def _values(nnz: int, seed: int, stream: int) -> torch.Tensor:
    return _rand(nnz, _generator(seed + 1, stream)) * 2.0 - 1.0


def _csr(rows: torch.Tensor, cols: torch.Tensor, m: int, n: int, seed: int, stream: int):
    """(m, n, row pointers, columns, values) of the distinct entries, with row i renumbered to i + shift (mod m)
    and column j to j + shift (mod n), the shift being the seed's."""
    shift = seed * 104_729
    keys = torch.unique((rows + shift) % m * n + (cols + shift) % n)
    rows = torch.div(keys, n, rounding_mode="floor")
    rpt = torch.zeros(m + 1, dtype=torch.int64, device=DEV)
    rpt[1:] = torch.cumsum(torch.bincount(rows, minlength=m), 0)
    return m, n, rpt, keys - rows * n, _values(keys.numel(), seed, stream)


def _uniform(m: int, per_row: int, seed: int):
    rows = torch.arange(m, device=DEV).repeat_interleave(per_row)
    cols = (_rand(rows.numel(), _generator(0, 1)) * m).long()
    return _csr(rows, cols, m, m, seed, 1)


def _powerlaw(m: int, x_min: float, seed: int):
    """Pareto(2) row lengths up to 20000; 70 % of the columns within 64 of the diagonal, the others uniform."""
    gen = _generator(0, 2)
    u = 1.0 - _rand(m, gen)
    lengths = torch.ceil(x_min / torch.sqrt(u)).clamp_(max=min(20_000, m)).long()
    rows = torch.arange(m, device=DEV).repeat_interleave(lengths)
    local = _rand(rows.numel(), gen) < 0.7
    lo, hi = (rows - 64).clamp_(min=0), (rows + 64).clamp_(max=m - 1)
    near = lo + (_rand(rows.numel(), gen) * (hi - lo + 1)).long()
    far = (_rand(rows.numel(), gen) * m).long()
    return _csr(rows, torch.where(local, near, far), m, m, seed, 2)


def _grid(side: int, dof: int, seed: int):
    """27-point stencil on side^3 nodes with dof unknowns per node (dense dof x dof blocks)."""
    r = torch.arange(side ** 3, device=DEV)
    x, y, z = r % side, torch.div(r, side, rounding_mode="floor") % side, torch.div(r, side * side, rounding_mode="floor")
    cols, valid = [], []
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                valid.append((x + dx >= 0) & (x + dx < side) & (y + dy >= 0) & (y + dy < side)
                             & (z + dz >= 0) & (z + dz < side))
                cols.append(r + (dz * side + dy) * side + dx)
    cols, valid = torch.stack(cols, 1), torch.stack(valid, 1)
    if dof > 1:  # node row -> dof rows; node column -> dof columns
        cols = (cols[:, :, None] * dof + torch.arange(dof, device=DEV)).reshape(cols.shape[0], -1)
        valid = valid.repeat_interleave(dof, 1)
        cols, valid = cols.repeat_interleave(dof, 0), valid.repeat_interleave(dof, 0)
    m = side ** 3 * dof
    rpt = torch.zeros(m + 1, dtype=torch.int64, device=DEV)
    rpt[1:] = torch.cumsum(valid.sum(1), 0)
    col = cols[valid]
    rows = torch.arange(m, device=DEV).repeat_interleave(rpt[1:] - rpt[:-1])
    val = torch.where(col == rows, 26.0, -1.0).double() + 1e-3 * _values(col.numel(), seed, 3)
    return m, m, rpt, col, val


def _ragged(m: int, n: int, seed: int, stream: int):
    """Geometric(1/6) row lengths; a third of the rows with columns skewed as by R-MAT (a=.57, b=c=.19)."""
    gen = _generator(0, stream)
    u = 1.0 - _rand(m, gen)
    lengths = torch.ceil(torch.log(u) / math.log(5.0 / 6.0)).clamp_(1, n).long()
    rows = torch.arange(m, device=DEV).repeat_interleave(lengths)
    skewed = (_rand(m, gen) < 1.0 / 3.0)[rows]
    uni = (_rand(rows.numel(), gen) * n).long()
    rmat = torch.zeros_like(rows)
    for _ in range(max(1, math.ceil(math.log2(n)))):
        rmat = rmat * 2 + (_rand(rows.numel(), gen) < 0.24).long()
    return _csr(rows, torch.where(skewed & (rmat < n), rmat, uni), m, n, seed, stream)


def _operands(case: dict, seed: int) -> list[tuple]:
    """The (A, B) pairs of a case, each matrix a tuple (m, n, rpt, col, val) of 64-bit torch tensors whose
    values are those that the case's type holds; A is B where the case squares a matrix."""
    kind = case["kind"]
    if kind == "uniform":
        A = _uniform(case["m"], case["per_row"], seed)
        pairs = [(A, A)]
    elif kind == "powerlaw":
        A = _powerlaw(case["m"], case["x_min"], seed)
        pairs = [(A, A)]
    elif kind == "grid":
        A = _grid(case["g"], case["dof"], seed)
        pairs = [(A, A)]
    elif kind == "pair":
        pairs = [(_ragged(case["m"], case["k"], seed, 4), _ragged(case["k"], case["n"], seed, 5))]
    else:
        # sizes spread evenly over their logarithm
        pairs = []
        for i in range(case["count"]):
            at = (i + 0.5) / case["count"]
            m = int(round(case["lo"] ** (1 - at) * case["hi"] ** at))
            pairs.append((_ragged(m, m, seed, 10 + 2 * i), _ragged(m, m, seed, 11 + 2 * i)))
        # in no order of size
        pairs = pairs[::2] + pairs[1::2][::-1]

    def narrow(M):
        return M if case["dtype"] == "f64" else (*M[:4], M[4].float().double())
    out = []
    for A, B in pairs:
        nA = narrow(A)
        out.append((nA, nA if B is A else narrow(B)))
    return out


def _upload(M: tuple, dtype: str) -> g.DeviceCSR:
    m, n, rpt, col, val = M
    value = np.float64 if dtype == "f64" else np.float32
    return g.HostCSR(m, n, rpt.int().cpu().numpy(), col.int().cpu().numpy(), val.cpu().numpy().astype(value)).to_device()


def prepare(case: dict, seed: int) -> dict:
    dev = []
    for A, B in _operands(case, seed):
        dA = _upload(A, case["dtype"])
        dev.append((dA, dA if B is A else _upload(B, case["dtype"])))
    torch.cuda.empty_cache()
    return {"batch": case["kind"] == "batch", "A": [a for a, _ in dev], "B": [b for _, b in dev]}


# ---------------------------------------------------------------- the call

class _Array:
    """An array of a device matrix for torch, keeping the matrix alive (no copy)."""

    def __init__(self, owner: g.DeviceCSR, ptr: int, n: int, typestr: str):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": typestr, "data": (ptr, False), "strides": None,
                                         "version": 2}


def _views(C: g.DeviceCSR) -> dict:
    v = "<f8" if C.dtype == np.float64 else "<f4"
    return {"rpt": torch.as_tensor(_Array(C, C.raw.rpt, C.m + 1, "<i4"), device=DEV),
            "col": torch.as_tensor(_Array(C, C.raw.col, C.nnz, "<i4"), device=DEV),
            "val": torch.as_tensor(_Array(C, C.raw.val, C.nnz, v), device=DEV)}


def run(state: dict):
    if state["batch"]:
        return [_views(C) for C in g.proposal_batched(state["A"], state["B"])]
    return _views(g.proposal(state["A"][0], state["B"][0]))


# ---------------------------------------------------------------- what a pass cannot do without

def _expand(A: tuple, B: tuple, r0: int, r1: int):
    """Keys row * n + column and values of the products of A's rows [r0, r1)."""
    _, n, brpt, bcol, bval = B
    e0, e1 = int(A[2][r0]), int(A[2][r1])
    col = A[3][e0:e1]
    rows = torch.arange(r0, r1, device=DEV).repeat_interleave(A[2][r0 + 1:r1 + 1] - A[2][r0:r1])
    length = brpt[col + 1] - brpt[col]
    entry = torch.arange(e1 - e0, device=DEV).repeat_interleave(length)
    first = torch.cumsum(length, 0) - length
    at = torch.arange(entry.numel(), device=DEV) - first[entry] + brpt[col][entry]
    return rows[entry] * n + bcol[at], A[4][e0:e1][entry] * bval[at]


def _row_cuts(A: tuple, B: tuple) -> tuple[list[int], int]:
    """Row ranges of about CHUNK products each, and the number of products."""
    length = B[2][A[3] + 1] - B[2][A[3]]
    upto = torch.zeros(length.numel() + 1, dtype=torch.int64, device=DEV)
    upto[1:] = torch.cumsum(length, 0)
    upto = upto[A[2]]  # products before each row
    total = int(upto[-1])
    marks = torch.arange(0, max(total, 1), CHUNK, device=DEV)
    inner = torch.searchsorted(upto, marks).clamp_(max=A[0]).tolist()
    return sorted({0, *inner, A[0]}), total


def _product(A: tuple, B: tuple, values: bool) -> dict:
    cuts, total = _row_cuts(A, B)
    counts, cols, vals = [], [], []
    nnz = 0
    for r0, r1 in zip(cuts[:-1], cuts[1:]):
        key, prod = _expand(A, B, r0, r1)
        if not values:
            nnz += torch.unique(key).numel()
            continue
        uniq, back = torch.unique(key, return_inverse=True)
        row = torch.div(uniq, B[1], rounding_mode="floor")
        counts.append(torch.bincount(row - r0, minlength=r1 - r0))
        cols.append((uniq - row * B[1]).int())
        vals.append(torch.zeros(uniq.numel(), dtype=torch.float64, device=DEV).index_add_(0, back, prod))
    if not values:
        return {"nip": total, "nnz": nnz}
    rpt = torch.zeros(A[0] + 1, dtype=torch.int64, device=DEV)
    rpt[1:] = torch.cumsum(torch.cat(counts), 0)
    return {"rpt": rpt.int(), "col": torch.cat(cols), "val": torch.cat(vals)}


def exact(case: dict, seed: int):
    out = [_product(A, B, True) for A, B in _operands(case, seed)]
    return out if case["kind"] == "batch" else out[0]


def work(case: dict) -> dict:
    """Operands read once, C written once; a multiply and an add per intermediate product."""
    value = 8 if case["dtype"] == "f64" else 4
    if case["kind"] == "grid":  # closed forms: 3, 5 and 9 points per axis, less the faces
        s, d = case["g"], case["dof"]
        m = s ** 3 * d
        sizes = [(m, d * d * (3 * s - 2) ** 3), (m, d * d * (5 * s - 6) ** 3)]
        nip = d ** 3 * (9 * s - 10) ** 3
    else:
        sizes, nip = [], 0
        for A, B in _operands(case, 0):
            sizes += [(M[0], M[3].numel()) for M in ((A,) if B is A else (A, B))]
            c = _product(A, B, False)
            sizes.append((A[0], c["nnz"]))
            nip += c["nip"]
        torch.cuda.empty_cache()
    return {"bytes": sum(4 * (m + 1) + (4 + value) * nnz for m, nnz in sizes), "flops": 2 * nip}


def tolerance(case: dict) -> dict:
    # The structure is exact; the order in which a sum's products are added is not fixed.
    return {"rel": 1e-15} if case["dtype"] == "f64" else {"rel": 5e-7}
