"""The largest frontier queues that the workgroup path's LDS holds, given by the caller: accepted and
correct with the window rows of as many directions as the matrices' items run."""
import numpy as np
import pytest

import gsofatpds_amd as g
import oracle

pytestmark = pytest.mark.gpu

RESERVE, WINDOW = 3072, 65 * 16 * 4  # bytes of static LDS set aside, and of one direction's window rows


def unstructured(n, symmetric):
    p = g.generate(kind=g.GEN_ERDOS_RENYI, n_keep=n, order=g.ORDER_RCM, drop_side=g.DROP_ANY, drop_ppm=100000, seed=n)
    if not symmetric:
        return p
    rows = np.repeat(np.arange(n, dtype=np.int64), p.end - p.beg)
    both = np.unique(np.concatenate([rows * n + p.adj, p.adj.astype(np.int64) * n + rows]))
    ptr = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(both // n, minlength=n), out=ptr[1:])
    return g.Pattern.from_rowptr(ptr, (both % n).astype(np.int32))


@pytest.mark.parametrize("symmetric", [0, -1])
@pytest.mark.parametrize("below", [0, 64, 519, 520, 600])
def test_largest_queues_of_mirrored_unstructured_patterns(symmetric, below):
    n = 5000
    p = unstructured(n, True)
    directions = 1 if symmetric == 0 else 2  # traversed from A alone, or in paired items
    room = g.device_query()["lds_per_block"] - RESERVE - (n + 31) // 32 * 4 - directions * WINDOW
    queue = room // 8 - below
    o = oracle.symbfact(p, chunk=128, structure=False)
    with g.Plan(p, pair_directions=1, symmetric=symmetric, queue_capacity=queue) as plan:
        assert plan.config()["queue_capacity"] == queue
        for _ in range(2):
            plan.run()
            r = plan.result()
            assert (r.fill_count, r.nnz_F, r.edge_checks, r.reach, r.supernodes_counted) == (
                o["fill"], o["nnz_F"], o["W"], o["R"], o["nsup"])
        assert np.array_equal(plan.nzu(), o["nzu"])
        assert np.array_equal(plan.supernode_flags(), o["sup_flag"])


@pytest.mark.parametrize("symmetric", [0, -1])
def test_one_more_entry_is_refused(symmetric):
    n = 5000
    p = unstructured(n, True)
    room = g.device_query()["lds_per_block"] - RESERVE - (n + 31) // 32 * 4 - (1 if symmetric == 0 else 2) * WINDOW
    with pytest.raises(g.GsofaError) as e:
        g.Plan(p, pair_directions=1, symmetric=symmetric, queue_capacity=room // 8 + 1)
    assert e.value.code == g.ERR_CAPACITY
