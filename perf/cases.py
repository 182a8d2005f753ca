"""What a user of this package has it do, as measurable cases.

Every case is one call path of the public interface on a matrix family that
the repository's benchmark, tests and workload generators use: banded
unsymmetric matrices (the original test scale and below), 2D 5-point and 3D
7-point grids in nested-dissection, natural or computed order with a few
one-directional extra entries, or symmetrized.  Outputs are whole: the sorted
L and U rows, per-row fills, supernodes and totals, on the host, where every
caller of this interface takes them.

A case fixes its base pattern.  The seed adds entries (one per 16 rows) that
elimination fills in any event: every pattern of a case has the same L and U,
so its outputs keep their sizes, with other per-row fills and totals.

The path of a case:
  oneshot     symbfact(A): plan, upload, execute, fetch, release (a program
              that factors each pattern once)
  plan        Plan(A) kept; a pass is execute() + fetch()
  batch       Plan([A, ...]) kept; a pass is execute() + fetch() of them all
  handoff     Plan(A) kept; execute() + fetch_supernodal(), the input of a
              supernodal numeric phase, + fetch() for its counts and rows
  serve       Server kept; submit() of every request, then wait() for each
"""
import math

import numpy as np

import gsofa_amd as g
from gsofa_amd import _lib

ND_LEAF = 64  # leaf size of the geometric nested dissection (gsofa_amd/configs.py)


def listed():
    return [
        # the smallest request of a stream: a 16 x 16 grid, all latency
        {"name": "oneshot_grid2d_nd_16", "path": "oneshot", "family": "grid2d", "side": 16},
        # the smallest benchmark workload: 64 x 64 grid in natural order
        {"name": "oneshot_grid2d_natural_64", "path": "oneshot", "family": "grid2d", "side": 64, "order": "natural"},
        # a structural matrix of BCSSTK18's size and row length, symmetric
        {"name": "plan_band_sym_11948", "path": "plan", "family": "band", "n": 11948, "band": 120, "lam": 6.0,
         "sym": True},
        # a 3D model at the size where one call is all of a user's wait, odd side
        {"name": "oneshot_grid3d_nd_33", "path": "oneshot", "family": "grid3d", "side": 33},
        # an input that came without an ordering: nested dissection by this
        # library, supernodes capped as SuperLU_DIST callers do
        {"name": "plan_grid2d_reordered_181", "path": "plan", "family": "grid2d", "side": 181, "order": "order_nd",
         "max_supernode_size": 32},
        # fill counts alone (choosing an ordering): no L/U is built
        {"name": "counts_band_100003", "path": "plan", "family": "band", "n": 100003, "band": 256, "lam": 8.0,
         "counts_only": True},
        # the structure handed to a numeric phase, by columns and supernodes
        {"name": "handoff_grid3d_nd_27", "path": "handoff", "family": "grid3d", "side": 27},
        # one GPU's share of four (the reference's N_GPU), label-correcting mode
        {"name": "share_grid3d_nd_21", "path": "plan", "family": "grid3d", "side": 21, "n_virtual_gpu": 4,
         "virtual_gpu_id": 1},
        # the 3D nested-dissection workload
        {"name": "plan_grid3d_nd_48", "path": "plan", "family": "grid3d", "side": 48},
        # many small matrices in one plan
        {"name": "batch_grid2d_nd_128", "path": "batch", "family": "mix2d", "count": 128, "lo": 16, "hi": 256},
        # a request stream: 2D and 3D grids submitted to a running server
        {"name": "serve_mix_8", "path": "serve", "family": "mix3d", "count": 8, "lo": 16, "hi": 48},
        # the original test scale, the largest
        {"name": "plan_band_659033", "path": "plan", "family": "band", "n": 659033, "band": 256, "lam": 8.0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["oneshot", "plan", "counts", "handoff", "share", "batch", "serve"])
    if kind == "batch":
        return {"path": "batch", "family": "mix2d", "count": _log_int(rng, 2, 160), "lo": 16,
                "hi": rng.randint(64, 256)}
    if kind == "serve":
        return {"path": "serve", "family": "mix3d", "count": rng.randint(3, 8), "lo": 16, "hi": rng.randint(20, 48)}
    c = {"path": "plan" if kind in ("counts", "share") else kind}
    small = kind in ("share", "handoff")
    fam = rng.choice(["band", "grid2d", "grid3d"])
    c["family"] = fam
    if fam == "band":
        top = {"oneshot": 200000, "plan": 400000, "counts": 400000, "handoff": 60000, "share": 20000}[kind]
        c["n"] = _log_int(rng, 1000, top)
        c["band"] = rng.randint(40, 256)
        c["lam"] = round(rng.uniform(4.0, 8.0), 2)
        c["sym"] = rng.random() < 0.3
        if c["sym"]:
            c["lam"] = round(c["lam"] / 2, 2)
    elif fam == "grid2d":
        c["order"] = rng.choice(["nd", "nd", "natural", "order_nd"])
        c["side"] = _log_int(rng, 16, (60 if small else 110) if c["order"] == "natural" else (128 if small else 256))
        c["sym"] = rng.random() < 0.3
    else:
        c["side"] = _log_int(rng, 10, {"share": 24, "handoff": 32}.get(kind, 46))
        c["sym"] = rng.random() < 0.3
    if kind == "counts":
        c["counts_only"] = True
    elif kind == "share":
        c["n_virtual_gpu"] = rng.randint(2, 8)
        c["virtual_gpu_id"] = rng.randrange(c["n_virtual_gpu"])
    elif rng.random() < 0.3:
        c["max_supernode_size"] = rng.choice([8, 32, 128])
    return c


def _pattern(n, rows, cols):
    """The matrix of these entries (0-based, any order, duplicates dropped)."""
    key = np.unique(rows.astype(np.int64) * n + cols)
    end = np.cumsum(np.bincount(key // n, minlength=n))
    return g.CsrMatrix(n, np.concatenate([[0], end[:-1]]), end, key % n)


def _row_index(A):
    return np.repeat(np.arange(A.n, dtype=np.int64), A.colend - A.colbeg)


def _coupled(A, seed, sym):
    """A with up to n / 16 entries (i, j) more, i -> k -> j in A with k below
    both: each is in struct(L + U) of A, which therefore stays as it is."""
    rng = np.random.default_rng(seed)
    rows, cols = _row_index(A), A.csr.astype(np.int64)
    below = np.flatnonzero(cols < rows)
    if below.size == 0:
        return A
    e = rng.choice(below, A.n // 16 + 1)
    i, k = rows[e], cols[e]
    beg, end = A.colbeg[k].astype(np.int64), A.colend[k].astype(np.int64)
    j = cols[beg + rng.integers(0, 1 << 30, i.size) % (end - beg)]
    ok = (j > k) & (j != i)
    i, j = i[ok], j[ok]
    more = [np.concatenate([rows, i]), np.concatenate([cols, j])]
    if sym:
        more = [np.concatenate([more[0], j]), np.concatenate([more[1], i])]
    return _pattern(A.n, *more)


def _grid(side, dims, order, pattern_seed):
    return g.gen_grid(side, side, side if dims == 3 else 1, nd_leaf=ND_LEAF if order == "nd" else 0,
                      extra_prob=0.05, extra_dist=2 if dims == 3 else 3, seed=pattern_seed)


def _matrix(case, seed):
    fam, sym = case["family"], bool(case.get("sym"))
    if fam == "band":
        A = g.gen_band(case["n"], case["band"], case["lam"], 3)
    else:
        order = case.get("order", "nd")
        A = _grid(case["side"], 3 if fam == "grid3d" else 2, order, 2)
        if order == "order_nd":
            A = g.permute(A, g.order_nd(A))
    if sym:
        r = _row_index(A)
        A = _pattern(A.n, np.concatenate([r, A.csr]), np.concatenate([A.csr, r]))
    return _coupled(A, seed, sym)


def _matrices(case, seed):
    L = _lib.lib()
    out = []
    for i in range(case["count"]):
        if case["family"] == "mix2d" or i % 2 == 0:
            side = int(L.gsofa_gen_side_loguniform(4, i, case["lo"], max(case["hi"], 128)))
            A = _grid(side, 2, "nd", 4000012 + i)
        else:
            A = _grid(int(L.gsofa_gen_uniform_int(5, 3, i, case["lo"], case["hi"])), 3, "nd", 5000015 + i)
        out.append(_coupled(A, seed * 1000003 + i, False))
    return out


def _options(case):
    keys = ("counts_only", "max_supernode_size", "n_virtual_gpu", "virtual_gpu_id")
    return {k: case[k] for k in keys if k in case}


def prepare(case, seed):
    path = case["path"]
    if path == "serve":
        return {"path": path, "server": g.Server(mem_gb=48.0, max_inflight=4, max_batch=64),
                "mats": _matrices(case, seed)}
    if path == "batch":
        mats = _matrices(case, seed)
        return {"path": path, "plan": g.Plan(mats)}
    A = _matrix(case, seed)
    if path == "oneshot":
        return {"path": path, "A": A, "options": _options(case)}
    return {"path": path, "plan": g.Plan(A, **_options(case))}


def _out(r):
    d = {"totals": np.array([r.fill_count, r.te_alg, r.reach, r.n_super], np.int64)}
    for k in ("row_fill", "row_te", "row_reach", "L_rowptr", "L_col", "U_rowptr", "U_col", "super_start", "supno"):
        v = getattr(r, k)
        if v is not None:
            d[k] = v
    return d


def run(state):
    path = state["path"]
    if path == "oneshot":
        return _out(g.symbfact(state["A"], **state["options"]))
    if path == "serve":
        srv = state["server"]
        tickets = [srv.submit(A) for A in state["mats"]]
        return [_out(srv.wait(t)[0]) for t in tickets]
    plan = state["plan"]
    plan.execute()
    if path == "handoff":
        h, out = plan.fetch_supernodal(), _out(plan.fetch())
        out.update((k, getattr(h, k)) for k in ("xsup", "xsub", "sub", "xlcol", "lrow", "xucol", "urow"))
        return out
    return _out(plan.fetch())


def _bound(A):
    """(nnz(L), nnz(U)) at most: exact for symmetric patterns."""
    import ctypes as C
    f, lb, ub = C.c_uint64(), C.c_uint64(), C.c_uint64()
    m = A.to_c()
    if _lib.lib().gsofa_fill_bound(C.byref(m), None, C.byref(f), C.byref(lb), C.byref(ub)) != 0:
        raise ValueError("gsofa_fill_bound failed")
    return lb.value, ub.value


def work(case):
    """Bytes of one pass: the pattern read once, every output written once.
    No floating-point work."""
    mats = _matrices(case, 1) if case["path"] in ("batch", "serve") else [_matrix(case, 1)]
    total = 0
    for A in mats:
        total += 4 * (A.n + 1) + 4 * A.nnz
        if case.get("counts_only"):
            total += 8 * A.n
            continue
        lb, ub = _bound(A)
        cols = 4 * (lb + ub) // case.get("n_virtual_gpu", 1)
        if case["path"] == "handoff":  # by columns too
            cols *= 2
        # row pointers of L and U, row fills, supernode ids and starts
        total += cols + 16 * (A.n + 1) + 8 * A.n + 8 * A.n
    return {"bytes": int(total), "flops": 0}
