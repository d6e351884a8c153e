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


def triples(text):
    return [tuple(map(float, t)) for t in re.findall(r"\{([\d.]+), ([\d.]+), ([\d.]+)\}", text)]


TABLE = re.search(r"SPLIT\[\] = \{(.*?)\}\};", GEMM, re.S).group(1) + "}"
SPLIT = list(zip([tuple(map(int, t)) for t in re.findall(r"\{(\d), (\d), (\d), \{", TABLE)], triples(TABLE)))
START, WHOLE_START = map(float, re.search(r"SPLIT_START = ([\d.]+), WHOLE_START = ([\d.]+)", GEMM).groups())
WHOLE = triples(re.search(r"WHOLE\[\] = \{(.*?)\}\}\};", GEMM, re.S).group(1) + "}")


def gemm_choice(fmt, M, N, K):
    """fmt: 0, 1, 2 for Q4_K, Q6_K, IQ3_S."""
    SB, kind = K // 256, 0 if M <= 32 else 1 if M <= 64 else 2
    full, last, alone = (t[fmt] for t in WHOLE[3 * kind:3 * kind + 3])
    tiles = over(N, 64) * over(M, (32, 64, 128)[kind])
    before = (tiles - 1) // (2 * CUS)
    rest = tiles - before * 2 * CUS
    light = rest == 2 * CUS and (M <= 32 or (M > 64 and SB <= 4))
    end = alone if rest <= CUS else full if light else last
    best, choice = 0.97 * (WHOLE_START + SB * (before * full + end)), -1
    for i, ((mt, rn, ks), step) in enumerate(SPLIT):
        groups = over(N, 32 * rn) * over(M, 32 * mt)
        left = groups % CUS
        rounds = 1.0 if groups <= CUS else groups // CUS + (0.6 + 0.4 * left / CUS if left else 0.0)
        us = rounds * (over(SB, ks) * step[fmt] + START)
        if us < best:
            best, choice = us, i
    return choice


def test_the_prompt_gemm_takes_the_fastest_kernel_of_each_measured_size():
    """The tables of measured times beside the rule: within 3 % of the fastest (two sizes of a table are that close)."""
    names = ["Q4_K", "Q6_K", "IQ3_S"]
    rows = re.findall(r"//   (\d+) x (\d+) x (\d+), (\w+) +([\d. ]+)\n", GEMM)
    assert len(rows) == 16
    for M, N, K, fmt, times in rows:
        times = [float(t) for t in times.split()]
        assert len(times) == 8
        assert times[1 + gemm_choice(names.index(fmt), int(M), int(N), int(K))] <= 1.03 * min(times), (M, N, K, fmt)
    number = r"([\d.]+), ([\d.]+), ([\d.]+)"
    full = re.findall(rf"(\d+) x (\d+) x (\d+) +{number} (->|:) {number} \((\d)\)", GEMM)
    assert len(full) == 8
    for M, N, K, *rest in full:
        M, N, K, entry = int(M), int(N), int(K), int(rest[7])
        assert over(N, 64) * over(M, 32 if M <= 32 else 64 if M <= 64 else 128) % (2 * CUS) == 0
        whole, other = [float(t) for t in rest[:3]], [float(t) for t in rest[4:7]]
        for fmt in range(3):
            assert gemm_choice(fmt, M, N, K) == (entry if rest[3] == "->" else -1)
            assert (other if rest[3] == "->" else whole)[fmt] <= 1.01 * (whole if rest[3] == "->" else other)[fmt]


def test_every_kernel_of_the_prompt_gemm_has_sizes():
    assert len(SPLIT) == GEMM.count("case") - GEMM.count("case LLAM") == 7 and len(WHOLE) == 9
    dealt = sizes(test_gpu_gemm.test_a_walk_dealt_to_wavefronts) + sizes(test_gpu_gemm.test_tiles_of_dealt_walks)
    products = sizes(test_gpu_gemm.test_random_shapes) + dealt
    sums = [s[:3] for s in sizes(test_gpu_gemm.test_block_sums_of_the_gemm_kernel)] + dealt
    for fmt in range(3):
        for shapes in (products, sums):
            chosen = {s: gemm_choice(fmt, *s) for s in shapes}
            assert set(chosen.values()) == set(range(-1, len(SPLIT)))
            for i, ((mt, rn, ks), _) in enumerate(SPLIT):
                own = [s for s in shapes if chosen[s] == i]
                assert any(M % (32 * mt) for M, N, K in own) and any(N % (32 * rn) for M, N, K in own), (fmt, SPLIT[i])
                assert ks == 1 or any(K // 256 % ks for M, N, K in own), (fmt, SPLIT[i])
            undivided = [M for M, N, K in shapes if chosen[M, N, K] == -1]
            assert {0 if M <= 32 else 1 if M <= 64 else 2 for M in undivided} == {0, 1, 2}, "a tile of 32, 64 or 128 tokens"
            assert any(M % 64 for M in undivided if 32 < M <= 64)
