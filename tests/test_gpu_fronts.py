"""Fronts (elimination subtrees as bit matrices) at the edges of their sizes, against the oracle and
against runs without fronts (pre_escalate=-1)."""
import numpy as np
import pytest

import gsofatpds_amd as g
import oracle

pytestmark = pytest.mark.gpu


def nested(leaf, seps, arms, tops, reach, drop, seed, symmetric=False, rows=9000):
    """A tree of separators over blocks of `leaf` rows, numbered in postorder: level k joins `arms` of
    level k - 1 by seps[k] rows, until there are `rows`; a row of a leaf block holds up to `reach` rows
    above its block. Every block is connected by its chain i - i + 1."""
    rng = np.random.default_rng(seed)
    levels, per = len(seps), leaf
    for s in seps:
        per = per * arms + s
    trees = max(1, -(-rows // per))
    blocks = []  # (first row, rows, level), postorder

    def build(level, at):
        for _ in range(arms if level else 0):
            at = build(level - 1, at)
        size = seps[level - 1] if level else leaf
        blocks.append((at, size, level))
        return at + size

    at = 0
    for _ in range(trees):
        at = build(levels, at)
    n = at + tops
    a = set()

    def pair(i, j):
        keep = rng.random(2) >= drop
        if symmetric:
            keep[:] = keep.any()
        if keep[0]:
            a.add((i, j))
        if keep[1]:
            a.add((j, i))

    for k, (lo, size, level) in enumerate(blocks):
        end = lo + size
        above = [b for b in blocks[k + 1:] if b[2] > level]
        parents = []  # the separators above it, outermost last
        want = level + 1
        for b in above:
            if b[2] == want:
                parents.append(b)
                want += 1
        up = np.concatenate([np.arange(b[0], b[0] + b[1]) for b in parents] + [np.arange(n - tops, n)])
        for i in range(lo, end):
            if i + 1 < end:
                a.add((i, i + 1))
                a.add((i + 1, i))
            for j in rng.integers(lo, end, 2):
                if int(j) != i:
                    pair(i, int(j))
            if up.size:
                for j in rng.choice(up, min(up.size, 1 + int(rng.integers(0, reach))), replace=False):
                    pair(i, int(j))
        if parents:  # the block hangs on its separator
            a.add((end - 1, parents[0][0]))
            a.add((parents[0][0], end - 1))
    for i in range(n):
        a.add((i, i))
    for i in range(n - tops, n - 1):
        a.add((i, i + 1))
        a.add((i + 1, i))
    e = np.array(sorted(a), np.int64)
    ptr = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(e[:, 0], minlength=n), out=ptr[1:])
    return g.Pattern.from_rowptr(ptr, e[:, 1].astype(np.int32))


CASES = {
    # level 0: a lane per row
    "leaf_8": lambda: nested(24, [8], 3, 20, 2, 0.2, 1),
    "leaf_63": lambda: nested(63, [], 1, 40, 2, 0.2, 2),
    "leaf_64": lambda: nested(64, [], 1, 40, 2, 0.2, 3),
    "leaf_65": lambda: nested(65, [], 1, 40, 2, 0.2, 4),
    "leaf_surface_128": lambda: nested(40, [], 1, 128, 20, 0.1, 5),
    "leaf_surface_129": lambda: nested(40, [], 1, 129, 20, 0.1, 6),
    "leaf_surface_300": lambda: nested(60, [], 1, 300, 24, 0.1, 7),  # none fits: runs without
    # levels 1 and 2: 32 pivots to a block, 256 and 512 nodes
    "separators_of_1": lambda: nested(50, [1, 1, 1], 2, 30, 3, 0.2, 8),
    "separators_of_32": lambda: nested(50, [32, 32], 2, 60, 6, 0.2, 9),
    "separators_of_33": lambda: nested(50, [33, 65], 3, 60, 6, 0.2, 10),
    "wide_nodes": lambda: nested(48, [100, 120], 2, 90, 12, 0.2, 11),
    "over_256_nodes": lambda: nested(48, [130, 260], 2, 90, 12, 0.2, 12, rows=16000),
    "long_rows": lambda: nested(60, [60, 60], 2, 200, 40, 0.15, 13),
    "symmetric": lambda: nested(50, [40, 60], 2, 90, 6, 0.2, 14, symmetric=True),
    "large": lambda: nested(60, [30, 40, 60, 90], 2, 150, 5, 0.2, 15, rows=30000),
}


def results(plan):
    plan.run()
    r = plan.result()
    return ((r.fill_count, r.nnz_F, r.nnz_L, r.nnz_U, r.edge_checks, r.reach, r.supernodes_counted),
            g.fnv1a_array(plan.nzu()), g.fnv1a_array(plan.supernode_flags()))


@pytest.mark.parametrize("case", sorted(CASES))
def test_fronts_at_their_edges(case):
    p = CASES[case]()
    print(f"[fronts] {case} n={p.n} nnz={p.nnz}", flush=True)
    o = oracle.symbfact(p, chunk=128, structure=False)
    for structure in (0, 1):
        with g.Plan(p, structure=structure) as plan:
            got = [results(plan) for _ in range(2)]
            lists = oracle.structure_digests(*plan.structure()) if structure else None
            assert np.array_equal(plan.nzu(), o["nzu"])
            assert np.array_equal(plan.supernode_flags(), o["sup_flag"])
        t = got[0][0]
        assert (t[0], t[1], t[4], t[5], t[6]) == (o["fill"], o["nnz_F"], o["W"], o["R"], o["nsup"])
        with g.Plan(p, structure=structure, pre_escalate=-1) as plan:
            want = results(plan)
            if structure:
                assert lists == oracle.structure_digests(*plan.structure())
        assert got == [want, want]


def test_level_2_of_a_large_grid():
    """Enough rows for every level, too many for the oracle: against runs without fronts."""
    for dims, w, ppm in ((2, 420, 100000), (3, 44, 150000), (2, 420, 0)):
        p = g.generate(kind=g.GEN_STENCIL, dims=dims, points=9 if dims == 2 else 7, nx=w, ny=w,
                       nz=w if dims == 3 else 1, order=g.ORDER_ND, nd_leaf=64,
                       drop_side=g.DROP_LOWER if dims == 2 else g.DROP_UPPER, drop_ppm=ppm, seed=w)
        print(f"[fronts] grid n={p.n} nnz={p.nnz}", flush=True)
        with g.Plan(p) as plan:
            got = results(plan)
        with g.Plan(p, pre_escalate=-1) as plan:
            assert got == results(plan)
