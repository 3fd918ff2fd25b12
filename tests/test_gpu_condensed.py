"""GPU parity of the workgroup path on condensed graphs (small finished subtrees contracted), against
the oracle where it is cheap and against runs without the elimination tree (pre_escalate=-1), which
keep every vertex."""
import sys

import numpy as np
import pytest

import gsofatpds_amd as g
import oracle

pytestmark = pytest.mark.gpu

TOTALS = ("fill_count", "nnz_F", "nnz_L", "nnz_U", "edge_checks", "reach", "supernodes_counted")


def grid(dims, points, w, n=0, side=g.DROP_LOWER, ppm=100000, seed=1, extra=0):
    return g.generate(kind=g.GEN_STENCIL, dims=dims, points=points, nx=w, ny=w, nz=w if dims == 3 else 1, n_keep=n,
                      order=g.ORDER_ND, nd_leaf=64, drop_side=side, drop_ppm=ppm, extra_every=extra, seed=seed)


def with_duplicates(p):
    rows = [list(p.adj[p.beg[v]:p.end[v]]) for v in range(p.n)]
    for v in range(0, p.n, 5):
        rows[v] += rows[v][-2:] + rows[v][:1]
    for v in range(0, p.n, 11):  # no diagonal
        rows[v] = [c for c in rows[v] if c != v]
    ptr = np.zeros(p.n + 1, np.int64)
    ptr[1:] = np.cumsum([len(r) for r in rows])
    return g.Pattern.from_rowptr(ptr, np.concatenate([np.array(r, np.int32) for r in rows]))


def relabelled(p):
    """The same matrix with the rows of the upper half interleaved: subtrees are no row ranges."""
    perm = np.arange(p.n, dtype=np.int32)
    perm[: p.n // 2 // 2 * 2] = np.arange(p.n // 2 // 2 * 2).reshape(2, -1).T.reshape(-1).argsort().astype(np.int32)
    return g.permute(p, None, perm)


CASES = {
    "2d_9pt_odd": lambda: (grid(2, 9, 101, n=10007, extra=8), {}),
    "2d_9pt_drops_everywhere": lambda: (grid(2, 9, 96, side=g.DROP_ANY, ppm=150000, seed=2), {}),
    "2d_5pt_many_drops": lambda: (grid(2, 5, 120, ppm=400000, seed=3), {}),
    "3d_7pt": lambda: (grid(3, 7, 21, side=g.DROP_UPPER, ppm=150000, seed=4), {}),
    "3d_27pt_long_rows": lambda: (grid(3, 27, 18, side=g.DROP_ANY, ppm=60000, seed=5), {}),
    "2d_mirrored": lambda: (grid(2, 9, 90, ppm=0, seed=6), {}),
    "2d_mirrored_both_directions": lambda: (grid(2, 9, 90, ppm=0, seed=6), {"symmetric": -1}),
    "duplicates": lambda: (with_duplicates(grid(2, 9, 80, seed=7)), {}),
    "interleaved": lambda: (relabelled(grid(2, 9, 80, seed=8)), {}),
    "block_1": lambda: (grid(2, 9, 70, seed=9), {"chain_block": 1}),
    "block_100_threads_512": lambda: (grid(2, 9, 110, seed=10), {"chain_block": 100, "heavy_threads": 512}),
    "small_queues": lambda: (grid(2, 9, 100, seed=11), {"queue_capacity": 64}),
    "uncut": lambda: (grid(2, 9, 100, seed=12), {"split_blocks": -1}),
}


def facts(plan, structure):
    r = plan.result()
    out = [tuple(getattr(r, k) for k in TOTALS), g.fnv1a_array(plan.nzu()), g.fnv1a_array(plan.supernode_flags())]
    if structure:
        out.append(oracle.structure_digests(*plan.structure()))
    return out


@pytest.mark.parametrize("case", sorted(CASES))
@pytest.mark.parametrize("chunk", [128, 1000])
def test_condensed_equals_oracle_and_uncondensed(case, chunk):
    p, opt = CASES[case]()
    print(f"[condensed] {case} n={p.n} nnz={p.nnz} S={chunk} {opt}", flush=True)
    o = oracle.symbfact(p, chunk=chunk, structure=False)
    for structure in (0, 1):
        with g.Plan(p, chunk_size=chunk, structure=structure, **opt) as plan:
            got = []
            for _ in range(3):  # every run builds the graph anew
                got.append(facts(plan.run(), structure))
            r = plan.result()
            assert (r.fill_count, r.nnz_F, r.edge_checks, r.reach, r.supernodes_counted) == (
                o["fill"], o["nnz_F"], o["W"], o["R"], o["nsup"])
            assert np.array_equal(plan.nzu(), o["nzu"])
            assert np.array_equal(plan.supernode_flags(), o["sup_flag"])
        with g.Plan(p, chunk_size=chunk, structure=structure, pre_escalate=-1, **opt) as plan:
            want = facts(plan.run(), structure)
        assert all(x == want for x in got)
        sys.stdout.flush()


def test_condensed_members_in_a_batch_graph():
    """Condensed, mirrored, unstructured and tiny members in one captured graph, replayed."""
    pats = [grid(2, 9, 60 + 17 * k, seed=20 + k) for k in range(3)]
    pats.append(grid(3, 7, 17, side=g.DROP_UPPER, seed=30))
    pats.append(grid(2, 9, 75, ppm=0, seed=31))
    pats.append(g.generate(kind=g.GEN_ERDOS_RENYI, n_keep=3001, order=g.ORDER_RCM, drop_ppm=100000, seed=32))
    pats.append(grid(2, 5, 9, seed=33))
    want = []
    for p in pats:
        with g.Plan(p, pre_escalate=-1) as plan:
            want.append(facts(plan.run(), False))
    b = g.Batch(pats)
    try:
        for rep in range(3):
            print(f"[condensed batch] replay {rep}", flush=True)
            b.run().sync()
            got = []
            for i in range(len(pats)):
                r = b.result(i)
                got.append([tuple(getattr(r, k) for k in TOTALS), g.fnv1a_array(b.nzu(i)),
                            g.fnv1a_array(b.supernode_flags(i))])
            assert got == want
            g.device_synchronize()
    finally:
        b.close()
