"""Slices of K that the linear layers' plans make: whole steps of 64 elements, and never fewer than the four that the tile for rows far apart loads ahead."""
import random

import mdx


def test_slices_have_four_steps_and_more():
    L, rng = mdx._lib.lib(), random.Random(3)
    seen = set()
    for _ in range(20000):
        rows, k = rng.randint(1, 128), 256 * rng.randint(1, 40)
        n = 64 * (rng.randint(1, 64) if rng.random() < 0.7 else rng.randint(64, 4000))
        s = L.mdx_decode_linear_splits(rows, n, k)
        assert s > 0 and k % (64 * s) == 0 and k // 64 // s >= 4, (rows, n, k, s)
        seen.add(s)
        rows, k = rng.randint(1, 1536), 128 * rng.randint(2, 80)
        s = L.mdx_linear_splits(rows, n, k)
        assert s <= 0 or (k % (64 * s) == 0 and k // 64 // s >= 4), (rows, n, k, s)
    assert len(seen) > 4


def test_small_tiles_keep_slices_of_four_steps():
    """Few rows and columns fill few CUs: K is cut down to the four steps that the smaller depth of the small tiles takes."""
    L = mdx._lib.lib()
    for rows, n, k, slices in ((32, 512, 512, 2), (8, 1024, 1024, 4), (32, 1024, 2048, 8), (64, 512, 1024, 4), (16, 2048, 2048, 8), (128, 512, 512, 2), (32, 2048, 2048, 4)):
        assert L.mdx_decode_linear_splits(rows, n, k) == slices, (rows, n, k)
        assert L.mdx_linear_splits(rows, n, k) == slices, (rows, n, k)


def test_second_rounds_of_small_tiles_are_not_taken_for_free():
    """480 tiles of 32 x 64 would be two rounds on 256 CUs: two slices of K in larger tiles, which are one."""
    assert mdx._lib.lib().mdx_linear_splits(160, 6144, 2048) == 2


def test_division_by_one_multiplication():
    """What the tiles' places are computed by: the factor that divisor() of mdx_common.h chooses gives the quotient for every number up to its bound."""
    for d in [2, 3, 5, 6, 7, 24, 48, 64, 96, 192, 594, 1187, 3561, 65535]:
        factor = ((1 << 32) + d - 1) // d
        n_max = ((1 << 32) - 1) // d
        edges = {0, 1, d - 1, d, d + 1, n_max} | {m * d + e for m in (1, 2, 1000, n_max // d) for e in (-1, 0, 1)}
        assert all(n * factor >> 32 == n // d for n in edges if 0 <= n <= n_max)
