"""The rule that picks the group-scaled (W4A8) GEMM's tile (csrc/gemm.hip: GROUP_TILES, tile_us, dispatch8), restated with the
constants read from the source, against measured times of the tiles that fit at each shape: the pick is within 4% of the
fastest one (MI355X, us, k-interleaved activations)."""
import os
import re

import pytest

SOURCE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "comfyui-rdna2-attention_amd", "csrc", "gemm.hip")
CUS = 256


def group_tiles():
    with open(SOURCE) as f:
        source = f.read()
    body = re.search(r"GROUP_TILES\[\] = \{(.*?)\n\};", source, re.S).group(1)
    tiles = [tuple(float(v.rstrip("f")) for v in row.split(",")) for row in re.findall(r"\{([^{}]*)\}", body)]
    assert len(tiles) == 5
    return tiles, int(re.search(r"#define GROUP_WIDE_K (\d+)", source).group(1))


def fits(tile, stages, K):
    """launch_gemm8's LDS check: the stages (or the output tile), then bn halves per 128 values of k; the scale block is static."""
    bm, bn, resident = (int(v) for v in tile[:3])
    dynamic = max(stages * (bm * 128 + bn * 64), bm * (bn * 2 + 16)) + bn * (K // 128) * 2
    return dynamic <= 160 * 1024 // resident - (bn * 4 + max(256, bn * 2) + bm * 4)


def tile_us(tile, M, N, K):
    bm, bn, resident, fixed, s0, s1, s2 = tile
    tiles, whole, slices = -(-M // int(bm)) * -(-N // int(bn)), CUS * int(resident), K // 128

    def slice_us(n):
        busy = n / CUS
        return s2 * (0.7 + 0.15 * busy) if n > CUS else s0 + (s1 - s0) * max(0.0, 2 * busy - 1)

    us = tiles // whole * (fixed + slices * slice_us(whole))
    return us + (fixed + slices * slice_us(tiles % whole) if tiles % whole else 0.0)


def pick(M, N, K):
    tiles, wide_k = group_tiles()
    order = sorted(range(5), key=lambda i: tile_us(tiles[i], M, N, K))
    return next(i for i in order if (i < 4 or K > wide_k) and fits(tiles[i], (3, 3, 3, 4, 3)[i], K))


# Tiles in the table's order: 128 x 128 (two per CU), 128 x 256, 64 x 128, 64 x 64, 128 x 128 (one per CU).
MEASURED = [
    (4096, 12288, 3072, {0: 192.5, 1: 204.0, 2: 218.7, 3: 259.5, 4: 214.2}),
    (4096, 3072, 12288, {1: 219.0, 2: 207.4, 3: 278.2, 4: 249.9}),
    (531, 1920, 14080, {1: 107.1, 2: 47.5, 3: 49.3, 4: 80.7}),
    (4096, 3072, 16384, {3: 360.4, 4: 322.8}),
    (4096, 12288, 16384, {3: 1410.1, 4: 1326.7}),
    (1101, 3072, 16384, {3: 113.3, 4: 99.1}),
    (512, 3072, 16384, {3: 56.3, 4: 92.5}),
    (2359, 3584, 16256, {3: 269.6, 4: 299.3}),
    (4096, 3072, 24576, {3: 525.6, 4: 478.4}),
    (300, 384, 20480, {3: 51.1, 4: 113.6}),
    (2901, 7040, 19968, {3: 716.3, 4: 662.2}),
    (300, 384, 32768, {4: 184.8}),
]


@pytest.mark.parametrize("M,N,K,us", MEASURED, ids=lambda v: str(v) if isinstance(v, int) else "us")
def test_group_scaled_pick_is_among_the_fastest(M, N, K, us):
    tiles, _ = group_tiles()
    assert {i for i in range(5) if fits(tiles[i], (3, 3, 3, 4, 3)[i], K)} >= set(us)
    assert us[pick(M, N, K)] <= 1.04 * min(us.values())


def test_wide_k_is_where_the_wider_tiles_stop_fitting():
    tiles, wide_k = group_tiles()
    assert all(fits(tiles[i], 3, wide_k) and not fits(tiles[i], 3, wide_k + 128) for i in (1, 2))
    assert fits(tiles[3], 4, 32000) and not fits(tiles[3], 4, 32128) and fits(tiles[4], 3, 44416)
