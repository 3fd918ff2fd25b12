"""Supernode flags of rows that run on condensed graphs, with duplicate entries, against the oracle.

Duplicates of an upper entry raise nzU of their row alone, so nzU can fall by one from row to row over
rows that are not one another's ancestors: only then does a flag depend on a bit of the column's window
behind rows of other subtrees, and behind the list nodes that these bring to the condensed graph."""
import numpy as np
import pytest

import gsofatpds_amd as g
import oracle

pytestmark = pytest.mark.gpu


def behind_lists(units, top_u=49, tail=127):
    """21 dense blocks of 64 rows, a path of 70 rows that ends in s, `units` subtrees of 8 rows (entries
    above the diagonal only: nothing of them is contracted, and each brings up to 8 list nodes), and r,
    which holds s, 8 * units + 1 rows above it. Row s has as many duplicates of r as make nzU fall by one
    on every row from s to r. The tail's rows are what all of these hold."""
    s = 21 * 64 + 69
    r = s + 8 * units + 1
    n = r + 1 + tail
    rows = [{i} for i in range(n)]
    for b in range(21):
        for i in range(64 * b, 64 * b + 64):
            rows[i].update(range(64 * b, 64 * b + 64))
    for i in range(s - 69, s):
        rows[i].add(i + 1)
        rows[i + 1].add(i)
    for i in range(s + 1, r):
        end = (i - s) % 8 == 0  # its unit's last row
        rows[i].update(range(r, r + top_u + r - i - (0 if end else 1)))
        if not end:
            rows[i].add(i + 1)
    rows[s].update(range(r, r + 1 + top_u))
    rows[r].update(range(r + 1, r + 1 + top_u))
    rows[r].add(s)
    lists = [sorted(x) for x in rows]
    lists[s] += [r] * (r - s - 1)
    ptr = np.zeros(n + 1, np.int64)
    np.cumsum([len(x) for x in lists], out=ptr[1:])
    return g.Pattern.from_rowptr(ptr, np.concatenate(lists).astype(np.int32)), s, r


def check(p, chunk, structure=0):
    o = oracle.symbfact(p, chunk=chunk, structure=False)
    with g.Plan(p, chunk_size=chunk, structure=structure) as plan:
        for _ in range(2):
            plan.run()
            t = plan.result()
            assert np.array_equal(plan.nzu(), o["nzu"])
            assert np.array_equal(plan.supernode_flags(), o["sup_flag"])
            assert (t.fill_count, t.nnz_F, t.edge_checks, t.reach) == (o["fill"], o["nnz_F"], o["W"], o["R"])
            assert t.supernodes_counted == o["nsup"]
    return o


@pytest.mark.parametrize("units", [1, 6, 8, 9, 10])
@pytest.mark.parametrize("structure", [0, 1])
def test_window_behind_list_nodes(units, structure):
    p, s, r = behind_lists(units)
    print(f"[windows] {units} units, n={p.n} s={s} r={r}", flush=True)
    o = check(p, 128, structure)
    assert np.all(np.diff(o["nzu"][s:r + 1]) == -1)  # every row from s to r is consulted
    assert o["sup_flag"][r] == 0 and o["sup_flag"][s] == 1


@pytest.mark.parametrize("chunk", [128, 200, 47])
def test_duplicates_on_condensed_grids(chunk):
    p = g.generate(kind=g.GEN_STENCIL, dims=2, points=9, nx=111, ny=109, order=g.ORDER_ND, nd_leaf=64,
                   drop_side=g.DROP_LOWER, drop_ppm=100000, seed=chunk)
    rng = np.random.default_rng(chunk)
    lists = []
    for v in range(p.n):
        row = p.adj[p.beg[v]:p.end[v]]
        more = rng.choice(row, int(rng.integers(0, 6)))
        lists.append(rng.permutation(np.concatenate([row, more])))
    ptr = np.zeros(p.n + 1, np.int64)
    np.cumsum([len(x) for x in lists], out=ptr[1:])
    check(g.Pattern.from_rowptr(ptr, np.concatenate(lists)), chunk)
