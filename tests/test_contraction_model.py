"""The contraction that the workgroup path's condensed graph rests on, as a host model on small random
matrices: for a row c, S(c) = {c} + (R_c of A, R_c of A^T) becomes one node with the edges U_c and the
vertices of R_c outside S(c), and every source outside c's elimination subtree keeps its U list, its
|R| and the sum of the degrees of R."""
import numpy as np
import pytest


def reach(adj, weight, s):
    """Nodes below s that s reaches through nodes below s, and all above that they or s hold."""
    seen, up, stack = set(), set(), [s]
    while stack:
        for x in adj[stack.pop()]:
            if x > s:
                up.add(x)
            elif x < s and x not in seen:
                seen.add(x)
                stack.append(x)
    return seen, up, sum(weight[v][0] for v in seen), sum(weight[v][1] for v in seen)


def tree(rows):
    n = len(rows)
    parent, anc = [-1] * n, [-1] * n
    for i in range(n):
        for j in sorted({j for j in range(i) if j in rows[i] or i in rows[j]}):
            while anc[j] not in (-1, i):
                anc[j], j = i, anc[j]
            if anc[j] == -1:
                anc[j] = parent[j] = i
    sub = [{v} for v in range(n)]
    for v in range(n):
        if parent[v] >= 0:
            sub[parent[v]] |= sub[v]
    return sub


@pytest.mark.parametrize("seed", range(60))
def test_contracted_subtrees_keep_every_other_row(seed):
    rng = np.random.default_rng(seed)
    n = int(rng.integers(2, 40))
    density, sym = rng.choice([0.03, 0.08, 0.2, 0.5]), rng.choice([0.0, 0.5, 1.0])
    upper = np.triu(rng.random((n, n)) < density, 1)
    lower = np.where(rng.random((n, n)) < sym, upper.T, np.tril(rng.random((n, n)) < density, -1))
    a = upper | lower
    rows = [[set(np.flatnonzero(m[i]).tolist()) for i in range(n)] for m in (a, a.T)]
    sub = tree(rows[0])
    degrees = [(len(rows[0][v]), 1) for v in range(n)]
    want = [[reach(r, degrees, s) for s in range(n)] for r in rows]
    # several disjoint subtrees, and then one above them
    graph, weight, done, alive = [[set(x) for x in r] for r in rows], list(degrees), set(), set(range(n))
    for c in sorted(rng.choice(n, min(n, 6), replace=False).tolist()):
        if c in done:
            continue
        got = [reach(graph[d], weight, c) for d in (0, 1)]
        assert all(got[d][1:] == want[d][c][1:] for d in (0, 1))
        s = (got[0][0] & got[1][0]) | {c}
        weight[c] = (sum(weight[v][0] for v in s), sum(weight[v][1] for v in s))
        for d in (0, 1):
            graph[d][c] = got[d][1] | (got[d][0] - s)
            for v in alive - s:
                if graph[d][v] & s:
                    graph[d][v] = (graph[d][v] - s) | {c}
        alive -= s - {c}
        done |= sub[c]
        for v in sorted(set(range(n)) - done):
            for d in (0, 1):
                assert reach(graph[d], weight, v)[1:] == want[d][v][1:]
