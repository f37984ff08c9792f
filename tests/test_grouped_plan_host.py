"""sp_moe_grouped_plan: which kernel a grouped expert product takes (host code, no GPU)."""
import pytest

ROWS, NARROW, TILES_64, TILES_128, WIDE, RING = 0, 1, 2, 3, 4, 16


def plan(gated, pairs, n, k, experts, row_div=0, a_stride=None):
    from scratchpad_amd import _native
    return _native.load().sp_moe_grouped_plan(gated, row_div, pairs, n, k, experts, k if a_stride is None else a_stride)


@pytest.mark.parametrize("experts, n, k", [(32, 1024, 2048), (8, 1536, 1024), (64, 1408, 4096)])
def test_gated_products_of_many_rows_keep_the_wide_kernel(experts, n, k):
    assert plan(1, 320 * experts, n, k, experts) >= RING and plan(0, 2000 * experts, n, k, experts) >= RING
    for mean in (321, 512, 2000):
        assert plan(1, mean * experts, n, k, experts) == WIDE


def test_products_that_the_ring_does_not_take():
    """K no multiple of 64, rows or weights past 32-bit offsets"""
    for gated in (0, 1):
        assert [plan(gated, mean * 8, 512, 1056, 8) for mean in (10, 11, 56, 57, 320, 321)] == [ROWS, TILES_64, TILES_64, TILES_128, TILES_128, WIDE]
        assert plan(gated, 100 * 8, 512, 1024, 8, a_stride=1 << 22) == TILES_128 and plan(gated, 100 * 8, 512, 1024, 8, 4, 1 << 22) >= RING
        assert plan(gated, 100 * 2, 1 << 20, 2048, 2) == TILES_128
    assert plan(0, 64, 512, 40, 8) == plan(0, 0, 512, 64, 8) == plan(0, 64, 512, 64, 8, -1) == plan(0, 64, 512, 64, 8, a_stride=32) == -1


def test_the_compared_sizes_take_every_ring_tile():
    """test_gpu_grouped_product's: each of the ten tiles, plain and gated, with more steps of K than its ring holds; and what they are compared with
    is the rows kernel"""
    from tests.test_gpu_grouped_product import RING as sizes, rows_kernel_share
    taken = [[plan(gated, E * mean, N >> gated, K, E, 2) for E, mean, N, K in sizes] for gated in (0, 1)]
    for gated in (0, 1):
        # (a ring holds at most 4 steps of 64, the second tile's 3 of 128)
        deep = {p for p, (_, _, _, K) in zip(taken[gated], sizes) if p >= RING and K > (384 if p == RING + 1 else 256)}
        assert deep == set(range(RING, RING + 10))
    for E, mean, N, K in sizes:
        assert rows_kernel_share(E, N, K) >= 16
