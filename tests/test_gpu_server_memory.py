"""The server's device memory: what its slots keep between groups is within the budget and reported, and
costs no request its admission."""
import re
import time

import numpy as np
import pytest

import gsofatpds_amd as g

pytestmark = pytest.mark.gpu


def footprint(p, **opt):
    """A request's footprint, from the rejection by a server whose budget is one byte."""
    srv = g.Server(slots=1, hbm_budget_bytes=1)
    try:
        with pytest.raises(g.GsofaError) as e:
            srv.wait(srv.submit(p, **opt), 10.0)
        assert e.value.code == g.ERR_REJECTED
        return int(re.search(r"footprint (\d+) B", str(e.value)).group(1))
    finally:
        srv.stop()


def pattern(n, seed=1):
    w = int(np.ceil(np.sqrt(n)))
    return g.generate(kind=g.GEN_STENCIL, dims=2, points=9, nx=w, ny=w, n_keep=n, order=g.ORDER_ND, seed=seed)


def idle(srv):
    t_end = time.time() + 30
    while srv.stats()["running"] and time.time() < t_end:
        time.sleep(0.001)
    return srv.stats()


def test_memory_kept_between_groups_is_within_the_budget():
    small, big = pattern(3000), pattern(60000)
    with g.Plan(big) as plan:
        plan.run()
        want = plan.result().as_dict()
    need = footprint(big)
    for budget in (need, need + need // 16, 4 * need):
        srv = g.Server(slots=3, hbm_budget_bytes=budget)
        try:
            seen = []
            for _ in range(2):
                for _ in range(4):  # the slots' memory grows to what their groups ask for
                    srv.wait(srv.submit(small), 60.0)
                    seen.append(srv.stats()["hbm_in_use"])
                kept = idle(srv)["hbm_in_use"]
                rid = srv.submit(big)
                seen.append(srv.stats()["hbm_in_use"])
                r = srv.wait(rid, 60.0).as_dict()
                assert all(r[k] == want[k] for k in ("fill_count", "nnz_F", "edge_checks", "reach", "supernodes"))
                seen.append(srv.stats()["hbm_in_use"])
                print(f"[memory] budget {budget} kept {kept} seen up to {max(seen)}", flush=True)
                assert 0 < kept <= budget // 8
            # (a finished group is charged until its slot is free again)
            assert max(seen) <= budget
        finally:
            srv.stop()


def estimate(p, paired, cus):
    """What admission charged a request before unstructured matrices had checkpoints."""
    n, blocks, bw = p.n, (p.n + 3) // 4, (p.n + 31) // 32
    region = 4 * n + 6 * bw if paired else 3 * n + bw
    return (12 * (n + 1) + 8 * p.nnz + 128 * n + 28 * n + 3 * n + 8 * blocks + 16 * n + 20 * blocks + 4 * n + 16 +
            4 * (4 * cus + 32) * region + (1 << 20))


def unstructured(n, seed=1):
    return g.generate(kind=g.GEN_ERDOS_RENYI, n_keep=n, order=g.ORDER_RCM, drop_side=g.DROP_ANY, drop_ppm=100000,
                      avg_degree_x100=600, seed=seed)


@pytest.mark.parametrize("n", [1, 60, 511, 512, 5003, 40000])
@pytest.mark.parametrize("pair", [0, 1])
def test_a_request_needs_no_larger_budget_than_it_did(n, pair):
    p = unstructured(n) if n > 1 else g.Pattern.from_dense(np.ones((1, 1), bool))
    need = footprint(p, pair_directions=pair)
    assert need <= estimate(p, pair == 1, g.device_query()["cus"])
    srv = g.Server(slots=1, hbm_budget_bytes=need)
    try:
        got = srv.wait(srv.submit(p, pair_directions=pair), 60.0)
    finally:
        srv.stop()
    with g.Plan(p, pair_directions=pair) as plan:
        plan.run()
        want = plan.result()
    assert (got.fill_count, got.nnz_F, got.edge_checks) == (want.fill_count, want.nnz_F, want.edge_checks)
