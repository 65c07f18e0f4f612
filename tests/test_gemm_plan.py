"""The launch plans, from the library's own planner (zest_gemm_plan, host arithmetic): what a launch's plan has to
satisfy for the kernels, over a sweep of sizes. CPU only."""
from __future__ import annotations

import numpy as np
import pytest
from gemm_plans import FUSED, PLAIN, RESIDUAL, plan_name


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


@pytest.mark.parametrize("kind,cases", [(-1, PLAIN), (-2, RESIDUAL), (2, FUSED)])
def test_labelled_cases_take_their_plans(zest, kind, cases):
    for M, ns, K, shape, splits in cases:
        ns = [2 * ns] if kind >= 0 else ns
        assert plan_name(zest, M, ns, K, kind) == (shape, splits), (M, ns, K)


def test_labelled_cases_cover_what_the_planner_takes(zest):
    # every (shape, split or not) that each kind of launch takes over a wide sweep of sizes has a labelled case
    rng = np.random.default_rng(3)
    for kind, cases in ((-1, PLAIN), (-2, RESIDUAL), (2, FUSED)):
        have = {(shape, splits > 1) for *_, shape, splits in cases}
        seen = set()
        for _ in range(6000):
            M, K = int(np.exp(rng.uniform(np.log(32), np.log(4200)))), int(np.exp(rng.uniform(np.log(200), np.log(30000)))) // 8 * 8
            ns = [max(1, int(np.exp(rng.uniform(np.log(64), np.log(20000)))) // 160) * 160]
            if kind == -1 and rng.random() < 0.4:
                ns.append(ns[0] // 480 * 160 + 160)
            if kind >= 0:
                ns = [max(1, ns[0] // 64) * 64]
            shape, splits = plan_name(zest, M, ns, K, kind)
            seen.add((shape, splits > 1))
        assert seen <= have, (kind, seen - have)


def test_mixed_launch_of_a_part_round(zest):
    # q, k and v of the hidden-2560 layer at 2048 tokens: a round and a half of 256x128 tiles runs the half as halves
    # (60.8 us, whole tiles 63.7, as timed when the two were last told apart)
    assert plan_name(zest, 2048, [4096, 1024, 1024], 2560) == ("mixed", 1)


def test_no_alloc_workspace_bound(zest):
    # plans fit the static array of zest_gemm_group_noalloc for every K up to 32768, and for weights of whole 160-row
    # tiles at any K; others may outgrow it as 256x128 tiles, where the best plan that fits takes a twentieth longer
    rng, most, over = np.random.default_rng(11), 64 << 20, 0
    for _ in range(4000):
        M = int(np.exp(rng.uniform(0, np.log(4200))))
        K = int(np.exp(rng.uniform(np.log(1000), np.log(120000)))) // 8 * 8
        N = int(np.exp(rng.uniform(np.log(64), np.log(17000)))) // 160 * 160 + (160 if rng.random() < 0.5 else 96)
        p = zest.gemm_plan(M, [N], K)
        if p["workspace"] > most:
            over += 1
            assert K > 32768 and p["tile_rows"] == 256 and N % 160, (M, N, K, p)
    assert over < 100
    assert zest.gemm_plan(2048, [2816], 65536)["workspace"] > most      # what the entry point refuses
    for N in (2432, 2560, 2688):
        assert zest.gemm_plan(2048, [N], 65536)["workspace"] <= most
