"""What is timed of this framework, and the inputs it is timed on.

The cases are the calls that a user of the adaptive SpMSpV engine makes: one
product with a sparse x through the learned selector (small, ordinary and
large, from a hundredth of a percent of the columns to all of them), dense
products with and without the CSR5 copy, the sort-based column product on a
rectangular matrix, the set-up of a new matrix on a handle, and the drivers
built on the product (BFS, multi-source BFS, PageRank, a batch of vectors).

Matrices and vectors are made on the GPU with torch from the seed; the
library gets their device pointers, as its C interface takes them.
"""
import ctypes
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "spmspv-adaptive_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import spmspv_amd as sa  # noqa: E402

DEV = "cuda"


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one short product on a small uniform matrix (16 rows per column, 655
        # keys): an inner step of an iterative method, latency alone
        {"name": "auto_uniform64k", "op": "auto", "kind": "uniform", "n": 65536, "per": 16, "keys": 655},
        # an ordinary frontier on a power-law graph, a thousandth of its columns
        {"name": "auto_rmat20_0.1pct", "op": "auto", "kind": "rmat", "scale": 20, "per": 16, "keys": 1049},
        # a tenth of the columns: the middle of the density range
        {"name": "auto_rmat20_10pct", "op": "auto", "kind": "rmat", "scale": 20, "per": 16, "keys": 104858},
        # one percent of the columns of a large graph
        {"name": "auto_rmat22_1pct", "op": "auto", "kind": "rmat", "scale": 22, "per": 16, "keys": 41943},
        # the sort-based column product by name, on a rectangular matrix with
        # sizes that are no multiple of anything (least squares, bipartite graphs)
        {"name": "sort_rect", "op": "sort", "kind": "random", "m": 700001, "n": 300007, "per": 24, "keys": 60001},
        # a dense x on a power-law graph with the CSR5 copy: y = A x in an eigensolver
        {"name": "spmv_csr5_rmat20", "op": "spmv", "kind": "rmat", "scale": 20, "per": 16, "csr5": True},
        # a dense x on a banded matrix (a discretised operator) in the default format
        {"name": "spmv_banded", "op": "spmv", "kind": "banded", "n": 1000003, "per": 27, "csr5": False},
        # a new matrix on a handle that exists: both formats are built, one product on each
        {"name": "setup_rmat19", "op": "setup", "kind": "rmat", "scale": 19, "per": 16, "keys": 5243},
        # BFS of one source on a large graph, the kernel chosen per level
        {"name": "bfs_rmat22", "op": "bfs", "kind": "rmat", "scale": 22, "per": 16},
        # 64 BFSs at once (landmark distances, betweenness samples)
        {"name": "bfs64_rmat18", "op": "bfs_multi", "kind": "rmat", "scale": 18, "per": 16, "sources": 64},
        # PageRank by residual pushes: x goes from dense to a few entries
        {"name": "pagerank_rmat18", "op": "pagerank", "kind": "rmat", "scale": 18, "per": 16},
        # a batch of vectors of mixed densities against one matrix
        {"name": "batch48_rmat20", "op": "batched", "kind": "rmat", "scale": 20, "per": 16, "vectors": 48},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """A case of the listed ones' ranges: any operation, any matrix kind it
    takes, sizes over their logarithm, densities from 1e-4 to 1."""
    op = rng.choice(["auto", "auto", "auto", "sort", "spmv", "spmv", "setup", "bfs", "bfs_multi", "pagerank", "batched"])
    c = {"op": op}
    kinds = {"auto": ["rmat", "uniform", "random", "banded"], "sort": ["random", "rmat", "uniform"],
             "spmv": ["rmat", "banded", "random"], "setup": ["rmat", "random", "banded"], "bfs": ["rmat", "uniform"],
             "bfs_multi": ["rmat", "uniform"], "pagerank": ["rmat"], "batched": ["rmat", "uniform"]}[op]
    c["kind"] = rng.choice(kinds)
    top = {"setup": 19, "bfs_multi": 18, "pagerank": 18, "batched": 19}.get(op, 21)
    c["per"] = _log(rng, 4, 28)
    if c["kind"] == "rmat":
        c["per"] = _log(rng, 8, 16)
        c["scale"] = rng.randint(15, top)
        n = 1 << c["scale"]
    else:
        n = c["n"] = _log(rng, 1 << 15, (1 << top) // 2) | rng.randint(0, 1)
        if c["kind"] == "random":
            c["m"] = _log(rng, max(1 << 14, n // 3), 3 * n)
    if op in ("auto", "sort", "setup"):
        dense = {"auto": 1.0, "sort": 0.25, "setup": 0.1}[op]
        c["keys"] = max(1, int(n * 10 ** rng.uniform(-4, 0) * dense))
    if op == "spmv":
        c["csr5"] = rng.random() < 0.5
    if op == "bfs_multi":
        c["sources"] = rng.choice([7, 33, 64])
    if op == "batched":
        c["vectors"] = rng.randint(5, 48)
    return c


# ------------------------------------------------------------------ the inputs
class Array:
    """A torch tensor's device memory as the binding takes it (`.ptr`)."""

    def __init__(self, t):
        self.t = t
        self.ptr = ctypes.c_void_p(t.data_ptr())
        self.count = t.numel()


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _shape(case):
    if case["kind"] == "rmat":
        return 1 << case["scale"], 1 << case["scale"]
    return case.get("m", case["n"]), case["n"]


def _matrix(case, seed):
    """CSR (row_ptr, col, val) on the GPU, int32 / int32 / float32; columns
    ascending and distinct in every row, values in (0, 1]."""
    m, n = _shape(case)
    g = _gen(seed)
    kind, per = case["kind"], case["per"]
    if kind == "rmat":  # a, b, c, d = .57, .19, .19, .05; symmetrised, no self loops
        scale = case["scale"]
        i = torch.zeros(per << scale, dtype=torch.int64, device=DEV)
        j = torch.zeros_like(i)
        for _ in range(scale):
            u = torch.rand(i.numel(), device=DEV, generator=g)
            i.mul_(2).add_(u >= 0.76)
            j.mul_(2).add_(((u >= 0.57) & (u < 0.76)) | (u >= 0.95))
        del u
        keep = i != j
        i, j = i[keep], j[keep]
        key = torch.cat([i * n + j, j * n + i])
        del i, j, keep
    elif kind == "banded":  # `per` diagonals around the main one
        off = torch.arange(per, device=DEV) - per // 2
        i = torch.arange(n, device=DEV).repeat_interleave(per)
        j = i + off.repeat(n)
        keep = (j >= 0) & (j < n)
        key = (i * n + j)[keep]
    elif kind == "uniform":  # `per` rows at random in every column
        j = torch.arange(n, device=DEV).repeat_interleave(per)
        key = torch.randint(m, (n * per,), device=DEV, generator=g) * n + j
    else:  # "random": uneven rows (about `per` each, a few empty, some ten times as long)
        deg = (per * torch.rand(m, device=DEV, generator=g).mul_(-1).add_(1).log_().neg_()).to(torch.int64)
        i = torch.arange(m, device=DEV).repeat_interleave(deg)
        key = i * n + torch.randint(n, (i.numel(),), device=DEV, generator=g)
    key = torch.unique_consecutive(torch.sort(key).values)
    row = key // n
    col = (key - row * n).to(torch.int32)
    rp = torch.zeros(m + 1, dtype=torch.int32, device=DEV)
    rp[1:] = torch.cumsum(torch.bincount(row, minlength=m), 0).to(torch.int32)
    val = 1 - torch.rand(col.numel(), device=DEV, generator=g)
    return rp, col, val


def _vector(n, k, g):
    """k distinct keys of [0, n), ascending, and values in [-1, 1)."""
    key = torch.randperm(n, device=DEV, generator=g)[:k].sort().values.to(torch.int32)
    return key, torch.rand(k, device=DEV, generator=g).mul_(2).sub_(1)


class State:
    """A matrix, its handle set up as a program sets it up once (CSR in, CSC
    built, buffers reserved, the trained selectors loaded), x and y."""

    def __init__(self, case, seed):
        self.case = case
        self.m, self.n = _shape(case)
        self.csr = _matrix(case, seed)
        rp, col, val = self.csr
        self.nnz = col.numel()
        self.arrays = [Array(t) for t in self.csr]
        self.g = _gen(seed + 1)
        A = self.A = sa.SpmspvHandle(self.m, self.n, self.nnz)
        A.InputCSR(self.nnz, *self.arrays)
        A.ToCSC()
        A.allocPreBuffer()
        A.selector_set_weights(np.load(os.path.join(PKG, "selector_weights.npy")))
        A.bfs_selector_set_weights(np.load(os.path.join(PKG, "bfs_selector_weights.npy")))

    def out(self, count, dtype):
        return Array(torch.zeros(count, dtype=dtype, device=DEV))

    def sparse_x(self, k):
        self.key, self.val = (Array(t) for t in _vector(self.n, k, self.g))
        self.yk, self.yv = self.out(self.m, torch.int32), self.out(self.m, torch.float32)


def prepare(case, seed):
    s = State(case, seed)
    A, op = s.A, case["op"]
    if op in ("auto", "batched", "pagerank") and case["kind"] == "rmat":
        # what a program that tuned the handle for its graphs has set: CSR5 row
        # tiles and the products for which the bucket kernel is taken
        A.set_spmv_type(1)
        A.csr5_preprocess()
        A.set_bucket_range(s.nnz // 80, s.nnz // 5)
    if op in ("auto", "sort", "setup"):
        s.sparse_x(case["keys"])
    if op in ("spmv", "setup"):
        A.set_spmv_type(1 if op == "setup" or case["csr5"] else 0)
        if op == "spmv" and case["csr5"]:
            A.csr5_preprocess()
        s.x = Array(torch.rand(s.n, device=DEV, generator=s.g).mul_(2).sub_(1))
        s.y = s.out(s.m, torch.float32)
    if op in ("bfs", "bfs_multi"):
        deg = torch.diff(s.csr[0])
        some = torch.nonzero(deg > 0).reshape(-1)
        pick = torch.randint(some.numel(), (case.get("sources", 1),), device=DEV, generator=s.g)
        s.sources = some[pick].to(torch.int32).cpu().numpy()
        s.levels = s.out(s.n * s.sources.size, torch.int32)
    if op == "pagerank":
        s.rank = s.out(s.n, torch.float32)
    if op == "batched":
        off, keys, vals, room = [0], [], [], [0]
        for d in np.geomspace(2e-4, 0.2, case["vectors"]):
            k, v = _vector(s.n, max(1, int(d * s.n)), s.g)
            keys.append(k)
            vals.append(v)
            off.append(off[-1] + k.numel())
            room.append(room[-1] + s.m)
        s.vptr = Array(torch.tensor(off, dtype=torch.int32, device=DEV))
        s.vkey, s.vval = Array(torch.cat(keys)), Array(torch.cat(vals))
        s.yoff = Array(torch.tensor(room, dtype=torch.int64, device=DEV))
        s.yk, s.yv = s.out(room[-1], torch.int32), s.out(room[-1], torch.float32)
        s.ynnz = s.out(case["vectors"], torch.int32)
    return s


# ------------------------------------------------------------------ one pass
def _sparse_y(s, count):
    """The count and the arrays it counts in, as the caller holds them (room
    for m entries, zero past the count)."""
    return {"count": count, "key": s.yk.t, "val": s.yv.t}


def run(s):
    A, op = s.A, s.case["op"]
    if op == "auto":
        A.set_sparse_x(s.key, s.val, s.key.count)
        return _sparse_y(s, A.run_auto(y_key=s.yk, y_val=s.yv)[0])
    if op == "sort":
        A.set_sparse_x(s.key, s.val, s.key.count)
        return _sparse_y(s, A.run(sa.K_COL_LB_SORT, y_key=s.yk, y_val=s.yv))
    if op == "spmv":
        A.set_vector_type(sa.SPMSPV_VEC_DENSE)
        A.set_x(s.x)
        A.run(sa.K_SPMV_LB, y_dense=s.y, want_nnz=False)
        return s.y.t
    if op == "setup":
        A.InputCSR(s.nnz, *s.arrays)
        A.ToCSC()
        A.csr5_preprocess()
        A.set_vector_type(sa.SPMSPV_VEC_DENSE)
        A.set_x(s.x)
        A.run(sa.K_SPMV_LB, y_dense=s.y, want_nnz=False)
        A.set_sparse_x(s.key, s.val, s.key.count)
        return {"dense": s.y.t, **_sparse_y(s, A.run(sa.K_COL_LB_SORT, y_key=s.yk, y_val=s.yv))}
    if op == "bfs":
        A.bfs(int(s.sources[0]), s.levels, use_graphs=1)
        return s.levels.t
    if op == "bfs_multi":
        A.bfs_multi(s.sources, s.levels)
        return s.levels.t
    if op == "pagerank":
        A.pagerank(s.rank, damping=0.85, eps=1e-4, max_iter=500)
        return s.rank.t
    A.run_batched(s.vptr, s.vkey, s.vval, s.yoff, s.yk, s.yv, s.ynnz)
    return {"count": s.ynnz.t, "key": s.yk.t, "val": s.yv.t}


# ------------------------------------------------------------------ what it cannot do without
def _products(case, nnz, n):
    """Expected nonzeros under x and rows they touch."""
    b = nnz * case["keys"] / n
    m = _shape(case)[0]
    return b, m * (1 - (1 - 1 / m) ** b)


def work(case):
    m, n = _shape(case)
    nnz = {"rmat": 1.9, "random": 0.97 * m / n, "banded": 1.0, "uniform": 1.0}[case["kind"]] * case["per"] * n
    op = case["op"]
    row = 4 * (m + 1) + 8 * nnz  # the whole matrix once
    if op in ("auto", "sort"):
        b, y = _products(case, nnz, n)
        return {"bytes": 16 * case["keys"] + 8 * b + 8 * y, "flops": 2 * b}
    if op == "spmv":
        return {"bytes": row + 4 * n + 4 * m, "flops": 2 * nnz}
    if op == "setup":  # read the CSR, write the CSC and the CSR5 copy, then the products
        b, y = _products(case, nnz, n)
        return {"bytes": row + (8 * nnz + 4 * n) + 8 * nnz + (row + 4 * n + 4 * m) + 8 * b + 8 * y, "flops": 2 * nnz + 2 * b}
    if op == "bfs":  # every row index once, levels written
        return {"bytes": 4 * nnz + 8 * n, "flops": nnz}
    if op == "bfs_multi":  # one 64-bit word read per edge, levels written
        return {"bytes": 4 * nnz + 4 * n * (case["sources"] + 1), "flops": nnz}
    if op == "pagerank":  # about 30 whole products' worth of pushes
        return {"bytes": 30 * (8 * nnz + 16 * n), "flops": 60 * nnz}
    k = n * np.geomspace(2e-4, 0.2, case["vectors"])
    b = nnz / n * k
    return {"bytes": float((16 * k + 8 * b + 8 * m * (1 - np.exp(-b / m))).sum()), "flops": float(2 * b.sum())}


# ------------------------------------------------------------------ in 64 bits
def _product64(s, key, val):
    """Count, keys and values of A x in 64 bits (the rows with an entry under
    x's keys), padded with zeros to m."""
    rp, col, a = s.csr
    x = torch.zeros(s.n, dtype=torch.float64, device=DEV)
    hit = torch.zeros(s.n, dtype=torch.bool, device=DEV)
    x[key.long()] = val.double()
    hit[key.long()] = True
    at = torch.nonzero(hit[col]).reshape(-1)
    row = torch.searchsorted(rp[1:], at.to(torch.int32), right=True)
    y = torch.zeros(s.m, dtype=torch.float64, device=DEV).index_add_(0, row, a[at].double() * x[col[at]])
    support = torch.zeros(s.m, dtype=torch.bool, device=DEV)
    support[row] = True
    k = torch.nonzero(support).reshape(-1)
    pad = s.m - k.numel()
    return {"count": k.numel(), "key": torch.nn.functional.pad(k.to(torch.int32), (0, pad)),
            "val": torch.nn.functional.pad(y[k], (0, pad))}


def _dense64(s, x):
    rp, col, a = s.csr
    row = torch.arange(s.m, device=DEV).repeat_interleave(torch.diff(rp).long())
    return torch.zeros(s.m, dtype=torch.float64, device=DEV).index_add_(0, row, a.double() * x.double()[col])


def _pagerank64(s, damping, eps, max_iter):
    """The residual pushes in 64 bits: every vertex over the threshold gives
    its residual to its column's rows, until none is over it."""
    rp, col, a = s.csr
    n = s.n
    a = a.double()
    row = torch.arange(n, device=DEV).repeat_interleave(torch.diff(rp).long())
    w = torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, col.long(), a)
    r = torch.full((n,), (1 - damping) / n, dtype=torch.float64, device=DEV)
    p = torch.zeros_like(r)
    active = torch.ones(n, dtype=torch.bool, device=DEV)
    for _ in range(max_iter):
        take = torch.where(active, r, torch.zeros_like(r))
        p += take
        r -= take
        x = torch.where(w > 0, take / w.clamp_min(1e-300), torch.zeros_like(take))
        r.index_add_(0, row, damping * a * x[col.long()])
        active = r > eps * (1 - damping) / n
        if not bool(active.any()):
            break
    return p + r


def exact(case, seed):
    s = prepare(case, seed)
    op = case["op"]
    if op in ("auto", "sort"):
        return _product64(s, s.key.t, s.val.t)
    if op == "spmv":
        return _dense64(s, s.x.t)
    if op == "setup":
        return {"dense": _dense64(s, s.x.t), **_product64(s, s.key.t, s.val.t)}
    if op == "pagerank":
        return _pagerank64(s, 0.85, 1e-4, 500)
    if op == "batched":
        at = s.vptr.t.tolist()
        y = [_product64(s, s.vkey.t[b:e], s.vval.t[b:e]) for b, e in zip(at, at[1:])]
        return {"count": torch.tensor([v["count"] for v in y], dtype=torch.int32, device=DEV),
                "key": torch.cat([v["key"] for v in y]), "val": torch.cat([v["val"] for v in y])}
    return None  # levels are whole numbers
