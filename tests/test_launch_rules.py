"""The sizes of the GPU tests reach every tile that a launch can choose (CPU only: the tables and the rules are read from
the sources, so that other figures there do not leave a tile without a test)."""
import math
import re
from pathlib import Path

import pytest

from tests import test_gpu_experts_small, test_gpu_gemm, test_gpu_linear_tiled

CSRC = Path(__file__).resolve().parent.parent / "llaminar_amd" / "csrc"
CUS = 256


def over(a, b):
    return -(-a // b)


def sizes(test):
    """The parameters of the test's mark that holds the sizes."""
    return next(m.args[1] for m in test.pytestmark if m.name == "parametrize" and m.args[0].startswith("M,"))


# ---- linear layers of many rows (linear_tiled.hip: expected) -------------------------------------------

LINEAR = (CSRC / "seq" / "linear_tiled.hip").read_text()
TILES = {kind: [tuple(map(float, t)) for t in re.findall(r"\{(\d+), (\d+), (\d+), (\d+), ([\d.]+)f, ([\d.]+)f, ([\d.]+)f, wide_launch<%s," % kind, LINEAR)]
         for kind in ("bf16", "float")}


def linear_tile(kind, M, N, K, batch=1, group_rows=None):
    def expected(tile):
        height, width, groups, resident, alone, full, start = tile
        rows = over(M, height) * batch
        if group_rows is not None:
            rows = max(min(batch, group_rows), group_rows / height + 0.5 * min(batch, group_rows))
        tiles, slots = rows * over(N, width), CUS * resident
        return math.ceil(tiles / slots) * (over(K // 64, groups) * (alone + (full - alone) * min(1.0, tiles / slots)) + start)
    return min(range(len(TILES[kind])), key=lambda i: expected(TILES[kind][i]))


def test_the_tables_are_read():
    assert len(TILES["bf16"]) == LINEAR.count("wide_launch<bf16,") >= 2 and len(TILES["float"]) == LINEAR.count("wide_launch<float,") >= 2


@pytest.mark.parametrize("kind", ["bf16", "float"])
def test_every_tile_of_linear_layers_has_sizes(kind):
    every = set(range(len(TILES[kind])))
    assert {linear_tile(kind, *s) for s in test_gpu_linear_tiled.SHAPES} == every
    ragged = [s for s in test_gpu_linear_tiled.SHAPES
              if s[0] % TILES[kind][linear_tile(kind, *s)][0] and s[1] % TILES[kind][linear_tile(kind, *s)][1]]
    assert {linear_tile(kind, *s) for s in ragged} == every, "rows and columns short of a tile"
    if kind == "float":
        assert {linear_tile(kind, *s) for s in test_gpu_linear_tiled.WHOLE} == every


@pytest.mark.parametrize("kind", ["bf16", "float"])
def test_every_tile_of_grouped_layers_has_sizes(kind):
    chosen = set()
    for M, experts, top, ff, K, _ in sizes(test_gpu_experts_small.test_rows_grouped_by_expert):
        chosen |= {linear_tile(kind, M, n, k, experts, M * top) for n, k in ((ff, K), (K, ff))}
    assert chosen == set(range(len(TILES[kind])))


# ---- prompt GEMM (gemm.hip: gemm_split_choice) -----------------------------------------------------------

GEMM = (CSRC / "gemm.hip").read_text()
SPLIT = [tuple(map(float, t)) for t in
         re.findall(r"\{(\d), (\d), (\d), ([\d.]+), ([\d.]+)\}", re.search(r"SPLIT\[\] = \{(.*)\};", GEMM).group(1))]


def gemm_choice(M, N, K):
    SB, alone, two = K // 256, 0.9 if M <= 32 else 2.0 if M <= 64 else 2.75, 1.7 if M <= 32 else 2.75 if M <= 64 else 4.5
    tiles = over(N, 64) * over(M, 32 if M <= 32 else 64 if M <= 64 else 128)
    rest = tiles % (2 * CUS)
    undivided = SB * (tiles // (2 * CUS) * two + (0.0 if rest == 0 else alone if rest <= CUS else two))
    best, choice = undivided, -1
    for i, (mt, rn, ks, step, fixed) in enumerate(SPLIT):
        rounds = over(over(N, 32 * int(rn)) * over(M, 32 * int(mt)), CUS)
        us = rounds * (over(SB, int(ks)) * step + fixed)
        if us < best and us < (0.85 if rounds > 1 else 0.95) * undivided:
            best, choice = us, i
    return choice


def test_every_kernel_of_the_prompt_gemm_has_sizes():
    assert len(SPLIT) == GEMM.count("case") - GEMM.count("case LLAM") == 5
    products = sizes(test_gpu_gemm.test_random_shapes) + sizes(test_gpu_gemm.test_a_walk_dealt_to_wavefronts)
    sums = [s[:3] for s in sizes(test_gpu_gemm.test_block_sums_of_the_gemm_kernel)] + sizes(test_gpu_gemm.test_a_walk_dealt_to_wavefronts)
    for shapes in (products, sums):
        assert {gemm_choice(*s) for s in shapes} == {-1, 0, 1, 2, 3, 4}
        undivided = [M for M, N, K in shapes if gemm_choice(M, N, K) == -1]
        assert {0 if M <= 32 else 1 if M <= 64 else 2 for M in undivided} == {0, 1, 2}, "a tile of 32, 64 or 128 tokens"
        assert any(M % 64 for M in undivided if 32 < M <= 64)
