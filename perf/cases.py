"""What this framework's users run, as measurable cases: one symbolic factorisation (or one set of
them) through a public entry point, over seeded synthetic patterns of the shapes the framework is
used on. torch is imported first so that the engine and torch share one HIP runtime."""
import ctypes as C
import math

import numpy as np
import torch

import gsofatpds_amd as g

# Totals a caller reads from a result (the timing and the path a source took are not results).
TOTALS = ("fill_count", "nnz_F", "nnz_L", "nnz_U", "edge_checks", "reach", "supernodes", "supernodes_counted")
# Entries per row of a pattern, for work(): the stencil's points (or the mean degree), the diagonal.
POINTS = {"grid2d": 9, "grid2d5": 5, "grid3d": 7, "er": 7, "sym2d": 9, "sym3d": 7}


def listed():
    return [
        # The smallest call: a coarse-level or subdomain matrix in natural order, through the entry
        # that allocates nothing (loops that may be captured). Launches and latency are the cost.
        {"name": "noalloc_natural_1024", "entry": "noalloc", "family": "grid2d5", "n": 1024, "natural": True},
        # The same entry in a serving loop near its middle size: a 3-D subdomain, ordered by the caller.
        {"name": "noalloc_grid3d_21952", "entry": "noalloc", "family": "grid3d", "n": 21952, "natural": False},
        # The small workload of the benchmark: a 64 x 64 five-point grid in natural order.
        {"name": "plan_natural_4096", "entry": "plan", "family": "grid2d5", "n": 4096, "natural": True},
        # A structurally symmetric matrix of the size of the reference's own input (one traversal
        # serves both triangles).
        {"name": "plan_sym_11948", "entry": "plan", "family": "sym3d", "n": 11948, "natural": False},
        # An odd, ragged 2-D size in nested-dissection order: the everyday mid-size solve.
        {"name": "plan_grid2d_49729", "entry": "plan", "family": "grid2d", "n": 49729, "natural": False},
        # The 3-D workload of the benchmark: large separators, long lists.
        {"name": "plan_grid3d_110592", "entry": "plan", "family": "grid3d", "n": 110592, "natural": False},
        # The benchmark's reference shape.
        {"name": "plan_grid2d_659033", "entry": "plan", "family": "grid2d", "n": 659033, "natural": False},
        # The largest: a 2-D problem whose vertex bitmap no longer fits a compute unit's LDS.
        {"name": "plan_grid2d_1500625", "entry": "plan", "family": "grid2d", "n": 1500625, "natural": False},
        # An unstructured (circuit-like) pattern in reverse Cuthill-McKee order.
        {"name": "plan_er_20011", "entry": "plan", "family": "er", "n": 20011, "natural": False},
        # The explicit L and U structure, fetched by the numeric phase that follows.
        {"name": "structure_grid2d_40401", "entry": "structure", "family": "grid2d", "n": 40401, "natural": False},
        # Many matrices of uneven size in one captured launch.
        {"name": "batch_24", "entry": "batch", "family": "mix", "n": 50000, "count": 24},
        # A burst of requests to the server, host preparation included.
        {"name": "serve_24", "entry": "serve", "family": "mix", "n": 50000, "count": 24},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    entry = rng.choice(("noalloc", "plan", "plan", "plan", "structure", "batch", "serve"))
    if entry == "noalloc":
        family = rng.choice(("grid2d", "grid2d5", "grid3d"))
        natural = rng.random() < 0.25
        return {"entry": entry, "family": family, "n": _log(rng, 600, 4096 if natural else 40000), "natural": natural}
    if entry == "plan":
        family = rng.choice(("grid2d", "grid2d", "grid2d5", "grid3d", "sym2d", "sym3d", "er"))
        hi = {"grid2d": 1500000, "grid2d5": 1200000, "grid3d": 110000, "sym2d": 400000, "sym3d": 60000, "er": 40000}
        natural = family in ("grid2d5", "sym3d") and rng.random() < 0.25
        return {"entry": entry, "family": family, "n": _log(rng, 2000, 6000 if natural else hi[family]),
                "natural": natural}
    if entry == "structure":
        return {"entry": entry, "family": rng.choice(("grid2d", "grid2d5", "sym2d")), "n": _log(rng, 3000, 60000),
                "natural": False}
    return {"entry": entry, "family": "mix", "n": _log(rng, 6000, 60000), "count": rng.randint(6, 28)}


def _symmetric(p):
    """The pattern with only those entries kept whose transpose is there too."""
    rows = np.repeat(np.arange(p.n, dtype=np.int64), p.end - p.beg)
    cols = p.adj.astype(np.int64)
    keep = np.isin(rows * p.n + cols, cols * p.n + rows, assume_unique=True)
    ptr = np.zeros(p.n + 1, np.int64)
    np.cumsum(np.bincount(rows[keep], minlength=p.n), out=ptr[1:])
    return g.Pattern.from_rowptr(ptr, p.adj[keep])


def _pattern(family, n, natural, seed):
    """A seeded pattern of n rows; stencils are truncated row-major to n, as the benchmark's are."""
    seed = (0x5EED * 1000003 + seed * 7919 + n) & 0x7FFFFFFFFFFF
    if family == "er":
        return g.generate(kind=g.GEN_ERDOS_RENYI, n_keep=n, order=g.ORDER_RCM, drop_side=g.DROP_ANY, drop_ppm=100000,
                          avg_degree_x100=600, seed=seed)
    order = g.ORDER_NATURAL if natural else g.ORDER_ND
    three = family in ("grid3d", "sym3d")
    w = math.ceil(round(n ** (1 / 3), 9)) if three else math.ceil(math.sqrt(n))
    # the entries that make a pattern unsymmetric: dropped below the diagonal (2-D), above it (3-D),
    # on both sides in natural order; symmetric patterns drop pairs
    sym = family.startswith("sym")
    side = g.DROP_ANY if natural or sym else g.DROP_UPPER if three else g.DROP_LOWER
    p = g.generate(kind=g.GEN_STENCIL, dims=3 if three else 2, points=POINTS[family], nx=w, ny=w, nz=w if three else 1,
                   n_keep=n, order=order, nd_leaf=64, drop_side=side,
                   drop_ppm=200000 if natural else 150000 if three else 30000 if sym else 100000,
                   extra_every=8 if family == "grid2d" and not natural else 0, seed=seed)
    return _symmetric(p) if sym else p


def _members(case):
    """Sizes and families of a set's members: log-uniform sizes up to the case's, half of them
    stencils (2-D and 3-D), half unstructured. They depend on the case alone; the entries on the seed."""
    count, hi, lo = case["count"], case["n"], 1500
    for k in range(count):
        u = ((k * 0.6180339887 + 0.37 * count) % 1.0)
        yield ("grid2d", "er", "grid3d", "er")[k % 4], int(round(math.exp(math.log(lo) + u * (math.log(hi) - math.log(lo)))))


def prepare(case, seed):
    entry = case["entry"]
    if entry in ("batch", "serve"):
        pats = [_pattern(f, n, False, seed * 64 + k) for k, (f, n) in enumerate(_members(case))]
        # a batch, or a running server, is kept by the program that uses it
        kept = g.Batch(pats) if entry == "batch" else g.Server(slots=4)
        return {"entry": entry, "patterns": pats, "kept": kept}
    p = _pattern(case["family"], case["n"], case["natural"], seed)
    if entry == "noalloc":
        ptr = np.concatenate([p.beg, p.end[-1:]]).astype(np.int32)
        return {"entry": entry, "n": p.n, "rowptr": torch.from_numpy(ptr).cuda(), "adj": torch.from_numpy(p.adj).cuda(),
                "nzu": torch.zeros(p.n, dtype=torch.int32, device="cuda"),
                "flags": torch.zeros(p.n, dtype=torch.uint8, device="cuda"),
                "totals": torch.zeros(len(g.NOALLOC_TOTALS), dtype=torch.int64, device="cuda")}
    state = {"entry": entry, "kept": g.Plan(p, structure=1 if entry == "structure" else 0).stage_timing(False)}
    if entry == "structure":
        # buffers of the numeric phase, kept from call to call; entries past the structure's stay -1
        cap = _triangle_cap(p.n)
        state["structure"] = {"u_rowptr": np.zeros(p.n + 1, np.int64), "u_col": np.full(cap, -1, np.int32),
                              "l_colptr": np.zeros(p.n + 1, np.int64), "l_row": np.full(cap, -1, np.int32)}
    return state


def _triangle_cap(n):
    """More entries than one triangle of a 2-D nested-dissection structure has (about 3 n log2(n))."""
    return int(5 * n * math.log2(n))


def _fetch_structure(plan, out):
    """The structure into the caller's buffers, as a program over the C interface takes it."""
    lib, nu, nl = g.lib(), C.c_int64(), C.c_int64()
    rc = lib.gsofa_structure_size(plan._h, C.byref(nu), C.byref(nl))
    if rc == g.OK and max(nu.value, nl.value) > len(out["u_col"]):
        raise MemoryError("the structure is larger than its buffers")
    i32, i64 = C.POINTER(C.c_int32), C.POINTER(C.c_int64)
    if rc == g.OK:
        rc = lib.gsofa_structure_get(plan._h, out["u_rowptr"].ctypes.data_as(i64), out["u_col"].ctypes.data_as(i32),
                                     out["l_colptr"].ctypes.data_as(i64), out["l_row"].ctypes.data_as(i32))
    if rc != g.OK:
        raise g.GsofaError(rc, lib.gsofa_last_error().decode(errors="replace"))
    return out


def _totals(r):
    return np.array([getattr(r, k) for k in TOTALS], np.int64)


def run(state):
    entry = state["entry"]
    if entry == "noalloc":
        # enqueued on torch's current (default) stream; the outputs stay on the device
        g.run_noalloc(state["n"], state["adj"].numel(), state["rowptr"].data_ptr(), state["adj"].data_ptr(),
                      state["nzu"].data_ptr(), state["flags"].data_ptr(), state["totals"].data_ptr())
        return {"nzu": state["nzu"], "flags": state["flags"], "totals": state["totals"]}
    kept = state["kept"]
    if entry == "plan":
        kept.run()
        return {"totals": _totals(kept.result()), "nzu": kept.nzu(), "flags": kept.supernode_flags()}
    if entry == "structure":
        kept.run()
        return {"totals": _totals(kept.result()), "flags": kept.supernode_flags(),
                **_fetch_structure(kept, state["structure"])}
    count = len(state["patterns"])
    if entry == "batch":
        kept.run()
        return {"totals": np.stack([_totals(kept.result(i)) for i in range(count)]),
                "nzu": np.concatenate([kept.nzu(i) for i in range(count)]),
                "flags": np.concatenate([kept.supernode_flags(i) for i in range(count)])}
    ids = [kept.submit(p) for p in state["patterns"]]
    totals = np.stack([_totals(kept.wait(i)) for i in ids])
    # the server keeps a request's totals and the digests of its counts and flags
    infos = [kept.info(i) for i in ids]
    for i in ids:
        kept.release(i)
    return {"totals": totals,
            "digests": np.array([[x["nzu_digest"], x["supernode_digest"]] for x in infos], np.uint64).view(np.int64)}


def _per_matrix(family, n, structure):
    nnz = n * POINTS[family] * 0.94
    out = 5.0 * n + 8 * len(TOTALS)  # upper counts, supernode flags, totals
    if structure:  # both triangles: about 6 n log2(n) entries in 2-D nested dissection, their offsets
        out += 16.0 * n + 4.0 * 6 * n * math.log2(n)
    return 4.0 * (n + 1) + 4.0 * nnz + out


def work(case):
    if case["entry"] in ("batch", "serve"):
        total = sum(_per_matrix(f, n, False) for f, n in _members(case))
    else:
        total = _per_matrix(case["family"], case["n"], case["entry"] == "structure")
    return {"bytes": total, "flops": 0}


def exact(case, seed):
    """Every output is a whole number or a byte: nothing is rounded."""
    return None
