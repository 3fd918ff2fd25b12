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
