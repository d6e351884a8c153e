"""The sizes of the GPU tests reach every tile that a launch can choose (CPU only: the tables and the rules are read from
the sources, so that other figures there do not leave a tile without a test)."""
import math
import re
from pathlib import Path

import numpy as np
import pytest

from oracle.binding import FMT_IQ3_S, FMT_Q4_K, FMT_Q6_K
from tests import fake_hip, test_gpu_bosirax, test_gpu_experts_small, test_gpu_gemm, test_gpu_linear_tiled

CSRC = Path(__file__).resolve().parent.parent / "llaminar_amd" / "csrc"
CUS = 256
FORMATS = [FMT_Q4_K, FMT_Q6_K, FMT_IQ3_S]


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


# ---- prompt GEMM (gemm.hip: gemm_plan): what the library launches --------------------------------------------

GEMM = (CSRC / "gemm.hip").read_text()
TILES_OF_WALKS = [tuple(map(int, t)) for t in re.findall(r"\{(\d), (\d), (\d), \{", re.search(r"SPLIT\[\] = \{(.*?)\}\}; //", GEMM, re.S).group(1))]
WHOLE = -1   # gemm_kernel, as the tables beside the rule have it
LAUNCHES = """
lib = ctypes.CDLL({library!r})
p, i = ctypes.c_void_p(1 << 20), ctypes.c_int
def launches(ok):
    assert ok
    return [l[1:] for l in log() if l[0] == "launch"]
answer([[launches(lib.llam_ql_gemm(ctypes.c_uint8(fmt), p, p, p, i(M), i(N), i(K), i(N), i(0), None)),
         launches(lib.llam_ql_gemm_block_sums(ctypes.c_uint8(fmt), p, p, p, i(M), i(N), i(K), i(row0), i(rows or N), i(0), None))]
        for fmt, M, N, K, row0, rows in {calls}])
"""


def gemm_launches(tmp_path, calls):
    """(format, M, N, K, first row, rows of the sums; 0: all) -> the launches of the product and of its block sums, each
    (tile or tokens, grid), as the library makes them."""
    def read(kernel, *numbers):
        if tile := re.search(r"gemm_split_kernel\w+TraitsELi(\d)ELi(\d)ELi(\d)ELb[01]ELb([01])E", kernel):
            return tuple(map(int, tile.groups())), tuple(map(int, numbers[:2]))
        return int(re.search(r"gemm_kernel\w+TraitsELb[01]ELi(\d+)E", kernel).group(1)), tuple(map(int, numbers[:2]))
    answer = fake_hip.run(tmp_path, LAUNCHES.format(library=str(CSRC.parent / "lib" / "libllaminar_ql.so"), calls=calls))
    return [tuple([read(*launch) for launch in side] for side in call) for call in answer]


def test_block_sums_run_on_the_launches_of_the_product(tmp_path):
    shapes = [(324, 5397, 1792), (196, 16697, 2304), (77, 17381, 4864), (338, 14686, 2560), (40, 8192, 5120), (130, 257, 256), (9, 70, 768)]
    calls = [(fmt, *s, 0, 0) for fmt in FORMATS for s in shapes]
    cut = 0
    for call, (product, sums) in zip(calls, gemm_launches(tmp_path, calls)):
        assert product == sums, call
        cut += len(product) == 2
    assert cut >= 9
    # a window on both sides of the seam at row 16384, and one on either: the workgroups that meet it
    calls = [(FORMATS[0], 196, 16697, 2304, *w) for w in ((16300, 100), (16000, 384), (16384, 64))]
    (_, both), (_, below), (_, above) = gemm_launches(tmp_path, calls)
    assert [t[:3] for t, _ in both] == [(4, 4, 1), (1, 1, 4)] and [g for _, g in both] == [(1, 2), (1, 7)]
    assert [t[:3] for t, _ in below] == [(4, 4, 1)] and below[0][1] == (3, 2)
    assert [t[:3] for t, _ in above] == [(1, 1, 4)] and above[0][1] == (2, 7)


def gemm_parts(tmp_path, calls):
    """(format, M, N, K) -> [(entry of SPLIT or WHOLE, launched tile or tokens, rows of W before it, its rows)], first launch first."""
    out = []
    for (_, M, N, K), (product, _) in zip(calls, gemm_launches(tmp_path, [(*c, 0, 1) for c in calls])):
        entries = [TILES_OF_WALKS.index(t[:3]) if isinstance(t, tuple) else WHOLE for t, _ in product]
        heights = [32 * t[0] if isinstance(t, tuple) else t for t, _ in product]
        widths = [32 * t[1] if isinstance(t, tuple) else 64 for t, _ in product]
        assert [g[1] for _, g in product] == [over(M, h) for h in heights]
        if len(product) == 1:
            assert product[0][1][0] == over(N, widths[0])
            out.append([(entries[0], product[0][0], 0, N)])
        else:
            # (the first launch has whole tiles, of rows that are a multiple of 64)
            first = [f for f in range(64, N, 64) if over(f, widths[0]) == product[0][1][0] and over(N - f, widths[1]) == product[1][1][0]]
            assert first
            out.append([(entries[0], product[0][0], 0, first[-1]), (entries[1], product[1][0], first[-1], N - first[-1])])
    return out


def test_the_prompt_gemm_takes_the_fastest_kernel_of_each_measured_size(tmp_path):
    """The tables of measured times beside the rule: within 3 % of the fastest (two sizes of a table are that close)."""
    names = ["Q4_K", "Q6_K", "IQ3_S"]
    rows = re.findall(r"//   (\d+) x (\d+) x (\d+), (\w+) +([\d. ]+)\n", GEMM)
    assert len(rows) == 16
    plans = gemm_parts(tmp_path, [(FORMATS[names.index(fmt)], int(M), int(N), int(K)) for M, N, K, fmt, _ in rows])
    for (M, N, K, fmt, times), parts in zip(rows, plans):
        times = [float(t) for t in times.split()]
        assert len(times) == 1 + len(TILES_OF_WALKS)
        if len(parts) == 1:
            assert times[1 + parts[0][0]] <= 1.03 * min(times), (M, N, K, fmt)
    number = r"([\d.]+), ([\d.]+), ([\d.]+)"
    full = re.findall(rf"(\d+) x (\d+) x (\d+) +{number} (->|:) {number} \((\d)\)", GEMM)
    assert len(full) == 8
    plans = iter(gemm_parts(tmp_path, [(fmt, int(M), int(N), int(K)) for M, N, K, *_ in full for fmt in FORMATS]))
    for M, N, K, *rest in full:
        M, N, K, entry = int(M), int(N), int(K), int(rest[7])
        assert over(N, 64) * over(M, 32 if M <= 32 else 64 if M <= 64 else 128) % (2 * CUS) == 0
        whole, other = [float(t) for t in rest[:3]], [float(t) for t in rest[4:7]]
        for fmt in range(3):
            assert [p[0] for p in next(plans)] == [entry if rest[3] == "->" else WHOLE]
            assert (other if rest[3] == "->" else whole)[fmt] <= 1.01 * (whole if rest[3] == "->" else other)[fmt]


def entries_of(tmp_path, fmt, shapes):
    return {p[0] for parts in gemm_parts(tmp_path, [(fmt, *s) for s in shapes]) for p in parts}


@pytest.mark.parametrize("fmt", FORMATS)
def test_every_kernel_of_the_prompt_gemm_has_sizes(fmt, tmp_path):
    assert len(TILES_OF_WALKS) == GEMM.count("case") - GEMM.count("case LLAM") == 8
    walks = set(range(len(TILES_OF_WALKS)))
    dealt = sizes(test_gpu_gemm.test_a_walk_dealt_to_wavefronts) + sizes(test_gpu_gemm.test_tiles_of_dealt_walks)
    products = sizes(test_gpu_gemm.test_random_shapes) + dealt
    sums = [s[:3] for s in sizes(test_gpu_gemm.test_block_sums_of_the_gemm_kernel)] + dealt
    for shapes in (products, sums):
        plans = dict(zip(shapes, gemm_parts(tmp_path, [(fmt, *s) for s in shapes])))
        alone = {s: parts[0] for s, parts in plans.items() if len(parts) == 1}
        assert {p[0] for p in alone.values()} == walks | {WHOLE}
        for i, (mt, rn, ks) in enumerate(TILES_OF_WALKS):
            own = [s for s, p in alone.items() if p[0] == i]
            assert any(M % (32 * mt) for M, N, K in own) and any(N % (32 * rn) for M, N, K in own), TILES_OF_WALKS[i]
            assert ks == 1 or any(K // 256 % ks for M, N, K in own), TILES_OF_WALKS[i]
        undivided = [M for (M, N, K), p in alone.items() if p[0] == WHOLE]
        assert {alone[s][1] for s in alone if alone[s][0] == WHOLE} == {32, 64, 128}
        assert any(M % 64 for M in undivided if 32 < M <= 64)
        # (Q4_K walks of 32 x 64: weights by way of LDS for one token tile, straight into registers for several)
        ways = {p[1][3] for p in alone.values() if p[0] == 1}
        assert ways == ({0, 1} if fmt == FMT_Q4_K else {1})
    # scales that are not finite: every walk has a second one
    for test in (test_gpu_gemm.test_dealt_walks_at_the_ends_of_the_scales, test_gpu_gemm.test_an_infinite_scale_leaves_other_tokens_and_rows_alone):
        assert entries_of(tmp_path, fmt, sizes(test)) >= walks


@pytest.mark.parametrize("fmt", FORMATS)
def test_launches_in_two_have_sizes(fmt, tmp_path):
    """The seam of every size is where the GPU test looks, and each format has first and second launches of the tiles that it uses."""
    cut = sizes(test_gpu_gemm.test_rows_in_two_launches)
    firsts, rests = set(), set()
    for (M, N, K, seams), parts in zip(cut, gemm_parts(tmp_path, [(fmt, *s[:3]) for s in cut])):
        assert seams[FORMATS.index(fmt)] == (parts[1][2] if len(parts) == 2 else 0), (M, N, K)
        if len(parts) == 2:
            firsts.add(parts[0][0])
            rests.add(parts[1][0])
    random, calls = np.random.default_rng(1), []
    while len(calls) < 1500:
        N, K = int(np.exp(random.uniform(np.log(1000), np.log(25600)))), 256 * int(np.exp(random.uniform(np.log(4), np.log(100))))
        M = int(np.exp(random.uniform(np.log(9), np.log(max(10, min(2048, 512 * 25600 * 5120 // (N * K)))))))
        calls.append((fmt, M, N, K))
    count = {}
    for parts in gemm_parts(tmp_path, calls):
        if len(parts) == 2:
            for key in (("first", parts[0][0]), ("rest", parts[1][0])):
                count[key] = count.get(key, 0) + 1
    used = {key for key, n in count.items() if n >= 3}
    assert len(used) >= 5 and used <= {("first", f) for f in firsts} | {("rest", r) for r in rests}


# ---- grouping of pairs by expert (moe.hip) ----------------------------------------------------------------

@pytest.mark.parametrize("experts", [1, 1528, 1529, 1536, 1537, 2048])
def test_grouping_asks_for_the_lds_that_it_takes(experts, tmp_path):
    """Two counts a word and wavefront beside the arrays of 2048 experts: more than 64 KiB has to be asked for before the launch."""
    fixed = (2 * 2048 + 1 + 3 * 16) * 4
    calls = fake_hip.run(tmp_path, f"""
lib, p, i = ctypes.CDLL({str(CSRC.parent / "lib" / "libllaminar_ql.so")!r}), ctypes.c_void_p(1 << 20), ctypes.c_int
assert lib.llam_ql_moe_group(p, i(999), i(1), i({experts}), p, i(0), None)
answer(log())
""")
    dynamic = int(calls[-1][-1])
    assert calls[-1][0] == "launch" and "moe_group_kernel" in calls[-1][1] and dynamic == 16 * over(experts, 2) * 4
    granted = max([int(c[2]) for c in calls if c[0] == "lds"], default=64 * 1024 - fixed)
    assert dynamic <= granted


# ---- graphs of decoding steps (sequence_model.cpp) ----------------------------------------------------------

DECODE = """
from llaminar_amd import sequence
from llaminar_amd.models import kogilix
from tests import sequence_models as sm
cfg = sm.config(sm.mlstm(mlp=sm.dense()))
model = sequence.SequenceModel(kogilix.weights(cfg, sm.random_weights(cfg)), 4, 512, 64, "float32")
log()
def decode(steps, times=1):
    for _ in range(times):
        model.decode([0, 1], [3, 3], [1, 2], steps)
    calls = log()
    return [sum(c[0] == what for c in calls) for what in ("instantiate", "replay", "launch")], [int(c[1]) for c in calls if c[0] == "replay"]
"""


def test_a_graph_of_several_steps_is_made_where_it_is_replayed(tmp_path):
    """128 steps of a shape in calls of one and three: single steps, before and after; then a call of six replays a graph of four."""
    ones, threes, six = fake_hip.run(tmp_path, DECODE + "answer([decode(1, 130), decode(3, 50), decode(6)])")
    assert ones[0][:2] == [0, 0] and ones[0][2] % 130 == 0
    step = ones[0][2] // 130
    assert threes[0] == [1, 3 * 50 - 1, step] and set(threes[1]) == {step}
    assert six[0] == [1, 3, 0] and six[1] == [4 * step, step, step]


def test_decoding_goes_on_where_a_graph_of_several_steps_cannot_be_made(tmp_path):
    long, after, error = fake_hip.run(tmp_path, DECODE + """
first = decode(2)
fake.fake_hip_largest_graph(2 * first[1][0])
answer([decode(8, 16), decode(8, 3), model._error()])
""")
    assert long[0] == [0, 8 * 16, 0] and after[0] == [0, 8 * 3, 0] and len(set(long[1] + after[1])) == 1
    assert error == ""


# ---- linear layers cut along K (linear_tiled.hip: linear_plan): what the library launches --------------------

SLICED = """
from llaminar_amd import sequence as sq
lib = sq.load()
p = 1 << 20
def launches(M, N, K, dtype, bytes, scratch=p):
    a = sq.LinearArgs(d_a=p, d_w=p, d_y=p, M=M, N=N, K=K, lda=K, ldy=N, batch=1)
    assert lib.llam_seq_linear_within(ctypes.byref(a), scratch, bytes, dtype, 0, None)
    return [l[1:] for l in log() if l[0] == "launch"]
def need(M, N, K, dtype):
    return lib.llam_seq_linear_scratch_bytes(M, N, K, dtype, 0)
"""
WIDE = re.compile(r"linear_wide_kernelI(DF16b|f)((?:Li\d+E)+)Lb([01])E")


def sliced(launched):
    """(type and tile, pieces) of a layer's launches, None where nothing is cut."""
    kind, tile, split = WIDE.search(launched[0][0]).groups()
    assert (split == "1") == (len(launched) == 2)
    if split == "0":
        return None
    return (kind, tuple(map(int, re.findall(r"\d+", tile)))[:6]), int(launched[0][1])


def test_every_tile_that_is_cut_has_sizes(tmp_path):
    chosen = fake_hip.run(tmp_path, SLICED + f"""
answer([launches(M, N, K, dtype, need(M, N, K, dtype)) for dtype in (0, 1) for M, N, K in {test_gpu_linear_tiled.SPLIT}])""")
    cuts = [c for c in map(sliced, chosen) if c]
    for kind, name in (("DF16b", "bf16"), ("f", "float")):
        every = {tuple(map(int, re.findall(r"\d+", t)))[:6] for t in re.findall(r"split_launch<%s, ([\d, ]+)>\}" % name, LINEAR)}
        assert {t for (k, t), _ in cuts if k == kind} == every and len(every) >= 4


def test_a_layer_stays_within_its_scratch(tmp_path):
    """What is asked for serves every number of rows up to the most, none is written past it, and without any nothing is cut."""
    rng = np.random.default_rng(5)
    layers = [(int(rng.integers(17, 2100)), 16 * int(2 ** rng.uniform(0, 11)), 64 * int(2 ** rng.uniform(0, 9)), int(rng.integers(2))) for _ in range(60)]
    found = fake_hip.run(tmp_path, SLICED + f"""
rows = lambda most: sorted({{17, 64, 65, 129, 257, most // 2, most - 1, most}} & set(range(17, most + 1)))
answer([[need(most, N, K, dtype), need(most, N, K, dtype) // 2,
         [[launches(M, N, K, dtype, size) for M in rows(most)] for size in (need(most, N, K, dtype), 1 << 40, need(most, N, K, dtype) // 2, 0)],
         [launches(M, N, K, dtype, 1 << 40, None) for M in rows(most)]] for most, N, K, dtype in {layers}])""")
    cut = 0
    for (most, N, K, dtype), (need, half, (enough, plenty, little, none), null) in zip(layers, found):
        assert enough == plenty and none == null and all(sliced(l) is None for l in none) and need <= 192 << 20
        rows = sorted({17, 64, 65, 129, 257, most // 2, most - 1, most} & set(range(17, most + 1)))
        for launched, limit in ((enough, need), (little, half)):
            for M, l in zip(rows, launched):
                if sliced(l):
                    cut += 1
                    (_, (height, width, *_)), pieces = sliced(l)
                    whole = over(M, height) * over(N, width) // CUS * CUS
                    rest = over(M, height) * over(N, width) - whole
                    slices = (pieces - whole) // rest
                    assert pieces == whole + rest * slices and 2 <= slices <= 8 and slices <= K // 64
                    assert rest * slices * height * width * 4 <= limit
    assert cut > 50


def test_some_rows_get_a_tile_of_as_many_groups(tmp_path):
    """llam_seq_linear_rows: a tile whose sums are of the same turns as those of the tile for all rows; few rows in a small one.  What is
    no part of the layer, and layers of few rows, are refused."""
    layers = [(M, N, K, batch, dtype) for dtype in (0, 1) for M, N, K, batch in
              [(*s, 1) for s in test_gpu_linear_tiled.SHAPES] + [(601, 512, 128, 16), (2049, 128, 512, 16), (1025, 512, 128, 64)]]
    found = fake_hip.run(tmp_path, SLICED + f"""
def rows(M, N, K, batch, dtype, *stretches):
    a = sq.LinearArgs(d_a=p, d_w=p, d_y=p, M=M, N=N, K=K, lda=K * batch, ldy=N * batch, batch=batch, a_stride=K, w_stride=N * K, y_stride=N)
    first, n = ((ctypes.c_int32 * len(stretches))(*(s[i] for s in stretches)) for i in (0, 1))
    ok = lib.llam_seq_linear_rows(ctypes.byref(a), len(stretches), first, n, dtype, 0, None)
    return [ok] + [l[1:] for l in log() if l[0] == "launch"]
answer([[[rows(*l, *s) for s in ([(0, l[0])], [(l[0] // 2, 1)], [(0, 2), (5, 7), (13, 4)], [])] for l in {layers}],
        [rows(40, 64, 128, 1, 0, *s)[0] for s in ([(-1, 5)], [(0, 41)], [(40, 1)], [(2, 0)], [(3, 2), (4, 1)], [(3, 2), (0, 1)], [(3, 2), (5, 35)])],
        rows(40, 64, 128, 1, 0, *[(i, 1) for i in range(0, 40, 2)]), rows(16, 64, 128, 1, 0, (0, 16))[0]])""")
    for (M, N, K, batch, dtype), (whole, *some, none) in zip(layers, found[0]):
        assert none == [True]
        (height, width, _, _, groups, *_), = [tuple(map(int, re.findall(r"\d+", WIDE.search(whole[1][0]).group(2))))]
        assert [int(v) for v in whole[1][1:4]] == [over(M, height) * over(N, width), batch, 1]
        for (ok, launch), stretches in zip(some, (1, 3)):
            tile = tuple(map(int, re.findall(r"\d+", WIDE.search(launch[0]).group(2))))
            assert ok and tile[4] == groups and tile[0] <= height and [int(v) for v in launch[1:4]] == [over(N, tile[1]), batch, stretches]
    assert found[1] == [False] * 6 + [True] and found[3] is False
    assert [int(l[3]) for l in found[2][1:]] == [8, 8, 4]


# ---- order of the workgroups of attention (grouped_attention.hip: attention_run) -------------------------------

def test_long_walks_are_dealt_in_rounds(tmp_path):
    """The shapes of the GPU test have more workgroups than compute units, whose walks are long enough for the order of rounds."""
    found = fake_hip.run(tmp_path, f"""
from llaminar_amd import sequence as sq
lib, p = sq.load(), 1 << 20
def launches(heads, groups, dim, ntok, pos, n, dtype):
    a = sq.AttentionArgs(heads, groups, dim, dim, -(-(pos + ntok) // 128) * 128, 0, 1.0, p, p)
    e = sq.Entries(p, p, p, p)
    assert lib.llam_seq_attention(ctypes.byref(a), p, ctypes.byref(e), 0, n, ntok, pos + ntok, p, heads * dim, p, 1 << 40, dtype, 0, None), lib.llam_ql_last_error()
    return [int(v) for v in next(l for l in log() if l[0] == "launch" and "16attention_kernel" in l[1])[2:5]]
answer([[launches(*case, dtype) for dtype in (0, 1)] for case in {test_gpu_bosirax.LONG_WALKS}])""")
    long = int(re.search(r"ATT_LONG = (\d+);", (CSRC / "seq" / "grouped_attention.hip").read_text()).group(1))
    rests = set()
    for (_, _, _, ntok, pos, _), (bf16, f32) in zip(test_gpu_bosirax.LONG_WALKS, found):
        assert (pos + ntok) / bf16[1] >= long and math.prod(bf16) > CUS and math.prod(f32) > CUS
        rests.add(math.prod(bf16) % CUS)
    assert 0 in rests and len(rests) > 2


# ---- latent portions with keys and values of every head (sequence_model.cpp: latent_expands) -----------------

LATENT = """
from llaminar_amd import sequence
from llaminar_amd.models import kogilix
from tests import sequence_models as sm, test_gpu_sequence as tg
def steps(layer, dtype, cap, rows, *portions):
    cfg = sm.config(layer, width=64)
    model = sequence.SequenceModel(kogilix.weights(cfg, sm.random_weights(cfg)), 6, cap, rows, dtype)
    bytes, got = model.device_bytes(), []
    for p in portions:
        log()
        model.forward([(b, at, [1] * n) for b, (at, n) in enumerate(p)], [])
        got.append([next((k for k in ("transpose_tiles", "latent_attention", "16attention") if k in l[1]), "") for l in log() if l[0] == "launch"])
    model.close()
    return bytes, got
layer = lambda name: tg.EXPANDED[name]
"""


def test_latent_portions_are_expanded_where_it_gains(tmp_path):
    """By a portion's own size, whatever lies beside it; never where the heads are no size of the attention kernels, or for few tokens."""
    single, bf16, wide, far, small = fake_hip.run(tmp_path, LATENT + """
answer([steps(layer("heads of 64"), "float32", 1024, 1024, [(0, 60)], [(0, 400)], [(0, 60), (0, 400), (0, 1), (0, 300), (0, 30)], [(1000, 1)], [(900, 20)]),
        steps(layer("heads of 64"), "bfloat16", 1024, 1024, [(0, 300)], [(0, 700)], [(300, 500)]),
        steps(layer("heads of 192"), "bfloat16", 1024, 1024, [(0, 700)]),
        steps(layer("heads of 64"), "float32", 40000, 1024, [(0, 900)], [(39000, 900)]),
        steps(layer("heads of 64"), "float32", 1024, 64, [(0, 64)])])""")
    count = lambda launches: [launches.count(k) for k in ("transpose_tiles", "latent_attention", "16attention")]  # noqa: E731
    assert [count(l) for l in single[1]] == [[0, 1, 0], [1, 0, 1], [2, 3, 2], [0, 1, 0], [0, 1, 0]]
    assert [count(l)[0] for l in bf16[1]] == [0, 1, 1]
    assert [count(l)[0] for l in wide[1]] == [0]
    # (the keys and values of 40,000 positions would be more than the scratch that is kept for them at most)
    assert [count(l)[0] for l in far[1]] == [1, 0] and far[0] - single[0] < (320 << 20) + 6 * 39000 * 400 * 4
    assert [count(l)[0] for l in small[1]] == [0] and small[0] < single[0]


def test_one_head_is_expanded_without_slices(tmp_path):
    """The keys and values of a layer of one head are plain products, which must not be cut along K: what is left there would overwrite them."""
    found = fake_hip.run(tmp_path, LATENT.replace("got.append(", "got.append([l[1] for l in log(False) if l[0] == 'launch']); (lambda _: None)(") + """
answer([steps(layer("one head"), dtype, 1600, 1600, [(0, 1600)], [(90, 1510)])[1] for dtype in ("float32", "bfloat16")])""")
    for launched in sum(found, []):
        first, = [i for i, name in enumerate(launched) if "transpose_tiles" in name]
        last = next(i for i, name in enumerate(launched) if "16attention" in name)
        products = launched[first + 1:last]
        assert len(products) == 2 and all(WIDE.search(name).group(3) == "0" for name in products), products


def test_the_line_of_expanded_portions(tmp_path):
    """Portions that were measured on both sides (sequence_model.cpp: latent_gains), by heads and type: tokens and positions before them."""
    sides = [(16, "bfloat16", [(600, 0), (1024, 0), (400, 1920), (256, 7680)], [(512, 0), (128, 1920), (128, 7680)]),
             (64, "bfloat16", [(400, 0), (600, 0)], [(300, 0), (128, 1920)]),
             (16, "float32", [(200, 0), (251, 0), (64, 512), (48, 1920), (128, 1920), (64, 7680)], [(100, 0), (187, 0), (48, 512), (17, 1920), (32, 7680)]),
             (40, "float32", [(130, 0), (64, 512), (64, 1920)], [(100, 0), (17, 512), (32, 1920)])]
    found = fake_hip.run(tmp_path, LATENT + f"""
answer([[["transpose_tiles" in got for got in steps(sm.latent(heads=heads, dim=128, vdim=128, q_rank=64, kv_rank=512), dtype, 8000, 1100,
                                                    *[[(at, n)] for n, at in side])[1]] for side in (gains, stays)] for heads, dtype, gains, stays in {sides}])""")
    for (gains, stays), (_, _, a, b) in zip(found, sides):
        assert gains == [True] * len(a) and stays == [False] * len(b)


def test_latent_products_are_of_the_rows_that_stay(tmp_path):
    """Beside portions that are expanded, W_uk and W_uv meet the others' rows alone, in one launch;
    where portions of both kinds take turns, those that stay go first."""
    found = fake_hip.run(tmp_path, LATENT.replace("[next((", "[l[1:5] if l[3] == '40' and 'linear_' in l[1] else next((") + """
answer(steps(layer("heads of 64"), "float32", 1024, 1600, [(0, 400)], [(0, 400), (500, 1)], [(0, 60), (0, 400), (500, 1), (0, 450), (0, 30), (7, 1)],
             [(0, 60), (0, 400), (0, 30), (0, 450), (7, 1), (0, 350)], [(0, 60), (0, 400), (0, 30), (0, 450), (7, 1), (0, 20)])[1])""")
    assert found[4].index("transpose_tiles") > max(i for i, l in enumerate(found[4]) if l == "latent_attention")
    for launches, rows, expanded in zip(found, ([], [1], [60, 1, 31], [60, 30, 1], [111]), (1, 1, 2, 3, 2)):
        products = [l for l in launches if isinstance(l, list)]
        assert len(products) == 2 * (len(rows) > 0) + 2 * expanded
        for (name, x, _, z), N in zip(products, [384, 64] * (len(rows) > 0)):
            height, width = map(int, re.findall(r"\d+", WIDE.search(name).group(2))[:2])
            assert int(x) == over(max(rows), height) * over(N, width) and height <= 128 and int(z) == len(rows)
