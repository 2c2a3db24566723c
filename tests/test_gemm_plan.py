"""The tile GEMM's choice of tile and K ranges (vkllm_hip_gemm_plan, host arithmetic): the GPU tests' products reach every
tile, whole and with K split, for one matrix and for the SwiGLU's two; and the scratch is never exceeded.
"""
import random

import pytest
import test_gemm_gpu as G


@pytest.fixture(scope="module")
def plan(vk):
    return vk.gemm_plan


def test_every_tile_is_tested_whole_and_split(plan):
    rng = random.Random(3)
    tiles = set()
    for _ in range(20000):
        M, N, K = (int(2 ** rng.uniform(a, b)) for a, b in ((1, 12), (5, 15), (0, 8)))
        tiles.add(plan(M, 32 * max(1, N // 32), 64 * K)[:2])
    tested = {(p[:2], p[2] > 1, epi == G.SWIGLU) for *_, epi, _, p in G.PLANNED}
    assert tiles == {t for t, _, _ in tested}
    assert tested == {(t, split, dual) for t in tiles for split in (False, True) for dual in (False, True)}


def test_plans_fit_the_scratch(plan):
    rng = random.Random(4)
    for _ in range(5000):
        M, N, K = rng.randint(1, 2100), 8 * rng.randint(1, 4000), 64 * rng.randint(1, 220)
        work = rng.choice([0, 1 << 16, 1 << 20, 16 << 20])
        splits = plan(M, N, K, work)[2]
        assert 1 <= splits <= 8 and (splits == 1 or splits * M * N <= work)
        assert splits == 1 or K // splits >= 192  # 256 of K a range, less what the ranges' rounding to 64 moves


@pytest.mark.parametrize("M,N", [(640, 8192), (1024, 8192), (2048, 4096), (4096, 2048), (4096, 16384)])
def test_short_rows(plan, M, N):
    """Products of short rows are their workgroups' starts and epilogues: up to K 192 two workgroups of 128 x 128 a CU (on
    one large tile a CU 2048 x 4096 x 64 takes 8.3 us instead of 7.3); up to K 512 not 256 x 128, which ran at 10.7 or at
    17 us (2048 x 4096 x 256) from one run to the next."""
    for K in (64, 128, 192):
        assert plan(M, N, K) == (128, 128, 1)
    for K in (256, 320, 512):
        assert plan(M, N, K)[:2] != (256, 128)


def test_fallback_products_have_no_tile(plan):
    assert plan(77, 1000, 1000) == (0, 0, 0) and plan(2, 8, (1 << 22) + 64) == (0, 0, 0)
