"""Checkpoints of unstructured patterns' workgroup path, against the oracle: sizes around the smallest
that has them and around their spacing, sparse patterns (checkpoints outside the large strongly connected
part) and dense ones, item lengths from one row to more than the spacing, bitmaps in HBM."""
import numpy as np
import pytest

import gsofatpds_amd as g
import oracle

pytestmark = pytest.mark.gpu

PATTERNS = [  # rows, average degree x 100, order, entries dropped (ppm)
    (511, 600, g.ORDER_RCM, 100000),
    (512, 600, g.ORDER_RCM, 100000),
    (545, 900, g.ORDER_NATURAL, 0),
    (2113, 250, g.ORDER_NATURAL, 300000),
    (4097, 600, g.ORDER_RCM, 100000),
    (6001, 350, g.ORDER_NATURAL, 100000),
]


@pytest.mark.parametrize("n,degree,order,drop", PATTERNS)
@pytest.mark.parametrize("structure", [0, 1])
def test_checkpoints_equal_the_oracle(n, degree, order, drop, structure):
    p = g.generate(kind=g.GEN_ERDOS_RENYI, n_keep=n, order=order, drop_side=g.DROP_ANY, drop_ppm=drop,
                   avg_degree_x100=degree, seed=n)
    o = oracle.symbfact(p, chunk=128, structure=bool(structure))
    for opt in ({}, {"chain_block": 1}, {"chain_block": 200}, {"heavy_threads": 512}, {"bitmap_in_hbm": 1},
                {"pair_directions": -1}):
        print(f"[checkpoints] n={n} nnz={p.nnz} {opt}", flush=True)
        with g.Plan(p, structure=structure, pair_directions=opt.get("pair_directions", 1),
                    **{k: v for k, v in opt.items() if k != "pair_directions"}) as plan:
            for _ in range(2):  # every run makes its checkpoints anew
                plan.run()
                r = plan.result()
                assert (r.fill_count, r.nnz_F, r.edge_checks, r.reach, r.supernodes_counted) == (
                    o["fill"], o["nnz_F"], o["W"], o["R"], o["nsup"])
            assert np.array_equal(plan.nzu(), o["nzu"])
            assert np.array_equal(plan.supernode_flags(), o["sup_flag"])
            if structure:
                up, ui, lp, li = plan.structure()
                want = oracle.split_structure(n, o["F_rowptr"], o["F_cols"])
                assert all(np.array_equal(a, b) for a, b in zip((up, ui, lp, li), want))


@pytest.mark.parametrize("n", [600, 3001])
def test_checkpoints_of_mirrored_patterns(n):
    """An unstructured symmetric pattern: one direction, whose bitmaps serve for both."""
    p = g.generate(kind=g.GEN_ERDOS_RENYI, n_keep=n, order=g.ORDER_RCM, drop_side=g.DROP_ANY, drop_ppm=100000, seed=n)
    rows = np.repeat(np.arange(n, dtype=np.int64), p.end - p.beg)
    both = np.unique(np.concatenate([rows * n + p.adj, p.adj.astype(np.int64) * n + rows]))
    ptr = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(both // n, minlength=n), out=ptr[1:])
    p = g.Pattern.from_rowptr(ptr, (both % n).astype(np.int32))
    o = oracle.symbfact(p, chunk=128, structure=False)
    for opt in ({}, {"chain_block": 1}, {"symmetric": -1}, {"bitmap_in_hbm": 1}):
        print(f"[checkpoints] mirrored n={n} nnz={p.nnz} {opt}", flush=True)
        with g.Plan(p, pair_directions=1, **opt) as plan:
            plan.run()
            r = plan.result()
            assert (r.fill_count, r.nnz_F, r.edge_checks, r.reach, r.supernodes_counted) == (
                o["fill"], o["nnz_F"], o["W"], o["R"], o["nsup"])
            assert np.array_equal(plan.nzu(), o["nzu"])
            assert np.array_equal(plan.supernode_flags(), o["sup_flag"])
