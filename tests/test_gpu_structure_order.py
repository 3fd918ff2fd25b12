"""The explicit structure's lists come sorted from the device: at the edges of the sort's sizes (a wave's
64 to 1,024 entries, a workgroup's bitmap in LDS and, beyond 1,048,576 rows, in HBM)."""
import numpy as np
import pytest

import gsofatpds_amd as g

pytestmark = pytest.mark.gpu

LENGTHS = (1, 2, 3, 63, 64, 65, 127, 128, 129, 256, 257, 511, 512, 513, 1023, 1024, 1025, 1500, 4097)


@pytest.mark.parametrize("n", [9001, 1048576, 1048577, 1200007])
@pytest.mark.parametrize("transposed", [False, True])
def test_lists_of_every_length_are_sorted(n, transposed):
    """Rows 2k and 2k + 1 of an otherwise diagonal matrix: the second holds the first, so its U list is
    the union of both rows; in rows spread over the matrix, the last ones near its end."""
    rng = np.random.default_rng(n)
    at = np.linspace(0, n - 5000, len(LENGTHS)).astype(np.int64) // 2 * 2
    rows, cols, want = [np.arange(n)], [np.arange(n)], {}
    for v, length in zip(at.tolist(), LENGTHS):
        # no column is one of the rows: nothing else is reached
        free = np.setdiff1d(np.arange(v + 2, n), np.concatenate([at, at + 1]))
        u = np.unique(np.concatenate([rng.choice(free, length, replace=False), [n - 1][: length - 1]]))[-length:]
        a, b = u[::2], u[1::2]
        for r, c in ((v, a), (v + 1, b), (v + 1, [v])):
            rows.append(np.full(len(c), r))
            cols.append(np.asarray(c, np.int64))
        want[v], want[v + 1] = a, u
    r, c = np.concatenate(rows).astype(np.int64), np.concatenate(cols).astype(np.int64)
    if transposed:
        r, c = c, r
    order = np.lexsort((c, r))
    ptr = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(r, minlength=n), out=ptr[1:])
    print(f"[structure order] n={n} transposed={transposed}", flush=True)
    with g.Plan(g.Pattern.from_rowptr(ptr, c[order].astype(np.int32)), structure=1) as plan:
        plan.run()
        for _ in range(2):  # reading leaves the lists as they are
            up, ui, lp, li = plan.structure()
            if transposed:
                up, ui, lp, li = lp, li, up, ui
            assert up[-1] == len(ui) == sum(len(x) for x in want.values())
            for v, x in want.items():
                assert np.array_equal(ui[up[v]:up[v + 1]], x), v
            assert np.array_equal(np.flatnonzero(np.diff(lp)), at) and np.array_equal(li, at + 1)
