"""Totals of the allocation-free entry against the oracle, where its route changes: one workgroup's set-up
(4,096 rows, 16 entries a row on average), one workgroup's queue (4,096 block slots), checkpoints (paired,
512 rows on, and off again where the scratch has no room for them)."""
import numpy as np
import pytest

import gsofatpds_amd as g
import oracle
from test_zz_no_alloc import prepared, run_noalloc
from test_zz_small_patterns import pattern

pytestmark = pytest.mark.gpu

OPTIONS = ({}, {"chain_block": 1}, {"chain_block": 2, "pair_directions": 1}, {"pair_directions": 1},
           {"chain_block": 1, "pair_directions": 1, "n_processes": 3})


def unstructured(n):
    return g.generate(kind=g.GEN_ERDOS_RENYI, n_keep=n, order=g.ORDER_RCM, drop_side=g.DROP_ANY, drop_ppm=100000,
                      avg_degree_x100=500, seed=n)


CASES = {f"{n}x{k}": (lambda n=n, k=k: pattern(n, k, n + k))
         for n, k in ((1, 1), (2, 1), (64, 3), (511, 4), (512, 4), (513, 4), (250, 15), (250, 17), (1024, 2), (2047, 2),
                      (2049, 2), (4095, 2), (4096, 2), (4097, 2))}
CASES.update({f"unstructured_{n}": (lambda n=n: unstructured(n)) for n in (511, 512, 4096, 4097, 12007)})


@pytest.mark.parametrize("case", sorted(CASES))
def test_totals_equal_the_oracle(case):
    rowptr, adj = prepared(CASES[case]())
    p = g.Pattern.from_rowptr(rowptr, adj)
    o = oracle.symbfact(p, chunk=128, structure=False)
    for opt in OPTIONS:
        print(f"[noalloc] {case} n={p.n} nnz={p.nnz} {opt}", flush=True)
        for _ in range(2):  # the scratch as the first call left it
            nzu, flags, t = run_noalloc(rowptr, adj, **opt)
            assert t["input_error"] == 0
            assert (t["fill_count"], t["nnz_F"], t["edge_checks"], t["reach"], t["supernodes_counted"]) == (
                o["fill"], o["nnz_F"], o["W"], o["R"], o["nsup"])
            assert t["supernodes"] == o["nsup"] + opt.get("n_processes", 1)
            assert t["nnz_U"] == int(o["nzu"].sum()) and t["nnz_L"] + t["nnz_U"] + p.n == o["nnz_F"]
            assert np.array_equal(nzu, o["nzu"]) and np.array_equal(flags, o["sup_flag"])


@pytest.mark.parametrize("n", [45000, 65536])
def test_paired_runs_at_the_scratch_limit(n):
    """The spill regions take what the scratch has: no room for checkpoints, the same results."""
    rowptr, adj = prepared(unstructured(n))
    p = g.Pattern.from_rowptr(rowptr, adj)
    with g.Plan(p, pair_directions=1) as plan:
        plan.run()
        r, nzu, flags = plan.result(), plan.nzu(), plan.supernode_flags()
    got = run_noalloc(rowptr, adj, pair_directions=1)
    assert np.array_equal(got[0], nzu) and np.array_equal(got[1], flags)
    for k in ("fill_count", "nnz_F", "nnz_L", "nnz_U", "edge_checks", "reach", "supernodes"):
        assert got[2][k] == getattr(r, k), k
