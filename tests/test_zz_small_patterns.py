"""Small patterns, whose input, layout and queue are made by one workgroup each, around the sizes where
that ends (4,096 rows, 16 entries a row on average, 4,096 block slots), against plans on the wave and
workgroup paths' general set-up (two matrices in a set) and the oracle."""
import numpy as np
import pytest

import gsofatpds_amd as g
import oracle
from test_zz_no_alloc import prepared, run_noalloc

pytestmark = pytest.mark.gpu


def pattern(n, degree, seed):
    rng = np.random.default_rng(seed)
    k = n * degree
    e = np.unique(rng.integers(0, n, k) * n + np.minimum(n - 1, np.abs(rng.normal(0, 60, k).astype(np.int64) + rng.integers(0, n, k))))
    long_row = np.arange(0, n, max(1, n // 40)) + (n // 2) * n  # more entries than a row has slots
    diag = np.arange(0, n, 3) * (n + 1)
    e = np.unique(np.concatenate([e, long_row, diag]))
    ptr = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(e // n, minlength=n), out=ptr[1:])
    return g.Pattern.from_rowptr(ptr, (e % n).astype(np.int32))


@pytest.mark.parametrize("n,degree", [(1, 1), (2, 1), (63, 3), (1023, 2), (1025, 3), (200, 15), (200, 17), (4095, 2), (4096, 3),
                                      (4097, 2)])
def test_small_patterns_equal_the_oracle(n, degree):
    p = pattern(n, degree, n + degree)
    print(f"[small] n={n} nnz={p.nnz}", flush=True)
    o = oracle.symbfact(p, chunk=128, structure=False)
    want = (o["fill"], o["nnz_F"], o["W"], o["R"], o["nsup"])
    for opt in ({}, {"chain_block": 1}, {"pair_directions": 1, "chain_block": 2}):
        with g.Plan(p, **opt) as plan:
            plan.run()
            r = plan.result()
            assert (r.fill_count, r.nnz_F, r.edge_checks, r.reach, r.supernodes_counted) == want
            assert np.array_equal(plan.nzu(), o["nzu"])
            assert np.array_equal(plan.supernode_flags(), o["sup_flag"])
    b = g.Batch([p, p])
    try:
        b.run().sync()
        r = b.result(1)
        assert (r.fill_count, r.nnz_F, r.edge_checks, r.reach, r.supernodes_counted) == want
    finally:
        b.close()
    rowptr, adj = prepared(p)
    nzu, flags, t = run_noalloc(rowptr, adj)
    assert np.array_equal(nzu, o["nzu"]) and np.array_equal(flags, o["sup_flag"])


@pytest.mark.parametrize("n", [5, 1025, 4096, 4097])
def test_small_patterns_that_break_the_row_rule(n):
    """The last row's last entry out of range, or a row out of order: flagged, and nothing counted."""
    rowptr, adj = prepared(pattern(n, 2, 7))
    for spoil in ("range", "order", "start", "end"):
        a, p = adj.copy(), rowptr.copy()
        if spoil == "range":
            a[-1] = n
        elif spoil == "order":
            v = int(np.argmax(np.diff(p) > 1))
            a[p[v]], a[p[v] + 1] = a[p[v] + 1], a[p[v]]
        elif spoil == "start":
            p[0] = 1
        else:
            p[-1] -= 1
        nzu, flags, t = run_noalloc(p, a)
        assert t["input_error"] == 1 and t["fill_count"] == 0 and not nzu.any(), spoil
