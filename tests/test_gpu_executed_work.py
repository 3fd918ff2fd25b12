"""Executed work of plans that run by fronts and condensed graphs: what its counts can be at most, and
their sums."""
import pytest

import gsofatpds_amd as g

pytestmark = pytest.mark.gpu


def grid(dims, w, side, ppm, seed=5):
    return g.generate(kind=g.GEN_STENCIL, dims=dims, points=9 if dims == 2 else 7, nx=w, ny=w, nz=w if dims == 3 else 1,
                      order=g.ORDER_ND, nd_leaf=64, drop_side=side, drop_ppm=ppm, seed=seed)


CASES = {"grid2d": lambda: grid(2, 143, g.DROP_LOWER, 100000), "grid3d": lambda: grid(3, 24, g.DROP_UPPER, 150000),
         "mirrored": lambda: grid(2, 120, g.DROP_ANY, 0), "wide": lambda: grid(3, 40, g.DROP_UPPER, 150000)}


@pytest.mark.parametrize("structure", [0, 1])
@pytest.mark.parametrize("case", sorted(CASES))
def test_counts_of_condensed_runs(case, structure):
    p = CASES[case]()
    with g.Plan(p, structure=structure) as plan:
        f = plan.fronts()
        for _ in range(2):
            plan.run()
            r, w = plan.result(), plan.executed_work()
        print(f"[work] {case} n={p.n} {f} heavy_sources={r.heavy_sources} {w}", flush=True)
        assert f["units"] > 0 and 0 < f["nodes"] < 0.7 * p.n
        # a node that is expanded is a source, or was inspected by its traversal before
        assert r.heavy_sources <= w["heavy_rows"] <= r.heavy_sources + w["heavy_edges"]
        # every row of either direction (of one, mirrored) is finished once, and every entry written once
        rows, entries = (p.n, r.nnz_U) if case == "mirrored" else (2 * p.n, r.nnz_L + r.nnz_U)
        assert w["light_rows"] + r.heavy_sources == rows
        assert w["light_out"] + w["heavy_out"] == entries


def test_a_plan_without_fronts_says_so():
    p = g.generate_workload(g.WL_GRID2D_4096)
    with g.Plan(p) as plan:
        assert plan.fronts() == {"units": 0, "nodes": 0}
        plan.run()
        w = plan.executed_work()
        assert w["light_rows"] > 0 and w["light_edges"] > 0
