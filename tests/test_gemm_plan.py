"""The launch plans, from the library's own planner (zest_gemm_plan, host arithmetic): what a launch's plan has to
satisfy for the kernels, over a sweep of sizes. CPU only."""
from __future__ import annotations

import numpy as np
import pytest


@pytest.mark.parametrize("kind", [-2, -1, 0, 2])
def test_plans_fit_their_launch(zest, kind):
    rng = np.random.default_rng(17 + kind)
    for _ in range(400):
        M = int(np.exp(rng.uniform(0, np.log(5000))))
        K = int(np.exp(rng.uniform(np.log(8), np.log(70000)))) // 8 * 8
        n = int(rng.integers(1, 5)) if kind == -1 else 1
        ns = [int(np.exp(rng.uniform(0, np.log(40000)))) for _ in range(n)]
        if kind >= 0:
            ns = [max(1, ns[0] // 64) * 64]
        p, nk = zest.gemm_plan(M, ns, K, kind), (K + 63) // 64
        cols = [(ns[0] + 127) // 128 * 128] if kind >= 0 else ns
        tiles = -(-M // p["tile_rows"]) * sum(-(-c // p["tile_cols"]) for c in cols)
        assert p["tiles"] == tiles and 0 < p["whole_tiles"] <= tiles, (M, ns, K, p)
        # every split and K-group has steps, equal ones where there are K-groups
        assert p["splits"] * p["k_groups"] <= nk
        assert p["k_groups"] == 1 or nk % (p["splits"] * p["k_groups"]) == 0
        # 160-column tiles read only rows that every packed weight holds
        assert p["tile_cols"] != 160 or all(c % 160 == 0 for c in ns)
        if p["whole_tiles"] < tiles:
            assert kind < 0 and p["splits"] == 1 and p["whole_tiles"] % 8 == 0 and p["tile_rows"] == 256
        want = tiles * p["splits"] * p["tile_rows"] * p["tile_cols"] * 4 if p["splits"] > 1 else 0
        assert p["workspace"] == want < 2 ** 31
        if kind == -2:
            q = zest.gemm_plan(M, ns, K, -1)
            assert (p["splits"], p["k_groups"]) == (q["splits"], q["k_groups"])  # the same sums, bit for bit
        if kind >= 0:
            q = zest.gemm_plan(M, ns, K, -1)
            assert (p["splits"], p["k_groups"]) == (q["splits"], q["k_groups"])


def test_plan_arguments(zest):
    for bad in [dict(m=0, ns=[8], k=8), dict(m=1, ns=[0], k=8), dict(m=1, ns=[8], k=7), dict(m=1, ns=[8], k=8, cus=0),
                dict(m=1, ns=[8] * 5, k=8), dict(m=1, ns=[8, 8], k=8, kind=2), dict(m=1, ns=[8], k=8, kind=9)]:
        with pytest.raises(RuntimeError):
            zest.gemm_plan(**bad)
