"""P3 on the GPU: prefill GEMM (int8 MFMA, per-block fp32 rescale) through the
C-ABI against the oracle, and against the decode GEMV whose per-block integer
pipeline is separately pinned bit-exact."""
import numpy as np
import pytest

from llaminar_amd import synth
from oracle.binding import FMT_IQ3_S, FMT_Q4_K, FMT_Q6_K
from tests.helpers import FMTS, TOL, rel_err, sync, upload_q8, upload_weights

pytestmark = pytest.mark.gpu

GOLD = {FMT_Q4_K: "q4k", FMT_Q6_K: "q6k", FMT_IQ3_S: "iq3s"}


@pytest.mark.parametrize("fmt", list(FMTS.values()), ids=list(FMTS))
def test_golden_fixture(capi, dev, golden, fmt):
    name = GOLD[fmt]
    W = golden[f"{name}_w"]
    N, K = W.shape[0], W.shape[1] * 256
    wd = upload_weights(capi, dev, fmt, W)
    qd = upload_q8(dev, golden["act_q8"])
    for M in (1, 4, 5):
        y = capi.gemm(fmt, wd, qd, M, N, K)
        sync()
        assert rel_err(y.cpu().numpy(), golden[f"{name}_c_avx512_m{M}"]) <= TOL[fmt] * 1e-2


@pytest.mark.parametrize("fmt", list(FMTS.values()), ids=list(FMTS))
@pytest.mark.parametrize("M,N,K", [(1, 128, 256), (17, 100, 512), (128, 128, 1024), (130, 257, 768), (300, 64, 2048),
                                   # launches of few tokens run tiles of 32 tokens: one, two (the second
                                   # holds one token) and three rows of tiles, then the first 128-token launch
                                   (32, 200, 1024), (33, 130, 5120), (96, 64, 2048), (97, 64, 2048),
                                   # 33 to 64 tokens whose walk one workgroup keeps: a tile of 64, full and not, rows
                                   # of one row tile and of many
                                   (64, 130, 1024), (40, 130, 512), (33, 20480, 2048), (57, 65, 256),
                                   # and more, in tiles of 128
                                   (130, 257, 256), (255, 100, 512)])
def test_random_shapes(capi, dev, oracle, fmt, M, N, K):
    W = synth.weights_numpy(fmt, N, K, 7 + M + N)
    q8 = oracle.quantize(synth.activations_numpy(M, K, 9 + K))
    wd = upload_weights(capi, dev, fmt, W)
    qd = upload_q8(dev, q8)
    y = capi.gemm(fmt, wd, qd, M, N, K)
    sync()
    C = oracle.gemm(fmt, W, K, q8)
    assert rel_err(y.cpu().numpy(), C) <= TOL[fmt] * 1e-2


@pytest.mark.parametrize("fmt", list(FMTS.values()), ids=list(FMTS))
def test_gemm_rows_equal_gemv(capi, dev, oracle, fmt):
    """Integer parity by transitivity: the GEMV's block sums are bit-exact, and every GEMM
    row must reproduce the GEMV output of that row to fp32 re-association accuracy."""
    M, N, K = 8, 384, 5120
    W = synth.weights_numpy(fmt, N, K, 71)
    q8 = oracle.quantize(synth.activations_numpy(M, K, 72))
    wd = upload_weights(capi, dev, fmt, W)
    qd = upload_q8(dev, q8)
    yg = capi.gemm(fmt, wd, qd, M, N, K)
    yv = capi.gemv(fmt, wd, qd, M, N, K)
    sync()
    assert rel_err(yg.cpu().numpy(), yv.cpu().numpy()) <= 2e-6


@pytest.mark.parametrize("fmt", list(FMTS.values()), ids=list(FMTS))
@pytest.mark.parametrize("M,N,K,r0,nr", [(1, 128, 256, 0, 128), (17, 100, 512, 37, 63), (130, 257, 768, 190, 67),
                                         (300, 200, 2048, 60, 70), (40, 130, 1280, 60, 70), (96, 70, 512, 0, 70),
                                         (64, 130, 1024, 60, 70), (40, 130, 512, 1, 129), (57, 65, 256, 64, 1),
                                         (130, 257, 256, 190, 67), (255, 100, 512, 37, 63)])
def test_block_sums_of_the_gemm_kernel(capi, dev, oracle, fmt, M, N, K, r0, nr):
    """The matrix unit's per-block results of llam_ql_gemm's own kernels (block-sum variants, chosen by the same rule) are
    the reference's int32 sums bit for bit: ragged tiles, windows that start and end inside a 64-row tile, token tails,
    tiles of 32, 64 and 128 tokens that one workgroup walks, and walks dealt to wavefronts."""
    W = synth.weights_numpy(fmt, N, K, 70 + M + N)
    q8 = oracle.quantize(synth.activations_numpy(M, K, 90 + K))
    wd = upload_weights(capi, dev, fmt, W)
    qd = upload_q8(dev, q8)
    s = capi.gemm_block_sums(fmt, wd, qd, M, N, K, r0, nr)
    sync()
    _, sums = oracle.gemm(fmt, W, K, q8, n0=r0, n1=r0 + nr, want_sums=True)
    assert np.array_equal(s.cpu().numpy(), sums)


@pytest.mark.parametrize("fmt", list(FMTS.values()), ids=list(FMTS))
@pytest.mark.parametrize("M,N,K", [
    (12, 97, 8960), (33, 31, 2304),    # to 8: 35 and 9 super-blocks, rows short of a tile
    (65, 97, 768), (40, 8161, 5120),   # to 4, 32 tokens: less than a step; the last row tile of one row
    (129, 3999, 1536),                 # to 2, 32 tokens: the last token tile of one token
    (129, 3999, 2816),                 # to 4, 64 tokens: 11 super-blocks
    (190, 9985, 1280),                 # to 2, 64 tokens: half a step left over, the last row tile of one row
])
def test_a_walk_dealt_to_wavefronts(capi, dev, oracle, fmt, M, N, K):
    """Tiles whose super-blocks are dealt to several wavefronts: rows, tokens and super-blocks left over.  Every element
    written and near the oracle's, the block sums of a window that starts inside a tile bit for bit, and the same bits
    again.  The tolerance is the one of the undivided walk: the parts are sums of the same products."""
    import torch

    W = synth.weights_numpy(fmt, N, K, 11 + M + N)
    q8 = oracle.quantize(synth.activations_numpy(M, K, 13 + K))
    wd = upload_weights(capi, dev, fmt, W)
    qd = upload_q8(dev, q8)
    y, again = (torch.full((M, N), float("nan"), device=dev) for _ in range(2))
    capi.gemm(fmt, wd, qd, M, N, K, out=y)
    capi.gemm(fmt, wd, qd, M, N, K, out=again)
    r0 = max(0, N - 75)
    s = capi.gemm_block_sums(fmt, wd, qd, M, N, K, r0, N - r0)
    sync()
    assert torch.equal(y, again)
    got = y.cpu().numpy()
    C = oracle.gemm(fmt, W, K, q8)
    assert rel_err(got, C) <= TOL[fmt] * 1e-2
    assert np.abs(got - C).max() <= 1e-4 * np.abs(C).max()
    _, sums = oracle.gemm(fmt, W, K, q8, n0=r0, n1=N, want_sums=True)
    assert np.array_equal(s.cpu().numpy(), sums)


@pytest.mark.parametrize("fmt", list(FMTS.values()), ids=list(FMTS))
@pytest.mark.parametrize("M,N,K", [
    (9, 33, 1792), (31, 4095, 2304),        # tiles of 32 x 32: super-blocks left over
    (20, 12001, 4864), (31, 8161, 1280), (33, 4100, 2816),  # 32 x 64
    (63, 8161, 2048), (33, 8161, 4864),     # 64 x 32
    (129, 4999, 1536), (129, 4999, 2816),   # 64 x 64: the last token tile of one token, a super-block left over
    (64, 20001, 1024), (33, 24997, 1280),   # 64 x 128
    (66, 4259, 768),                        # 32 x 64, several token tiles
    (67, 8573, 1280),                       # 96 x 64: the last token tile of three tokens less, rows and a super-block left over
    (324, 5397, 1792),                      # 128 x 64
    (97, 9799, 4352), (193, 8000, 2560), (257, 8129, 2304),  # (others by format)
    (128, 24997, 1280),                     # 128 x 128
    (255, 24997, 1280),                     # and short of a tile both ways
    (512, 8192, 1280),                      # one whole round of them
])
def test_tiles_of_dealt_walks(capi, dev, oracle, fmt, M, N, K):
    """Every tile whose half super-blocks are dealt to wavefronts, with rows, tokens and super-blocks left over: each element
    written once and the same bits again, near the oracle's on the first and last rows of W, their block sums bit for bit.
    The tolerance is that of the undivided walk: the parts are sums of the same products."""
    import torch

    W = synth.weights_numpy(fmt, N, K, 17 + M + N)
    q8 = oracle.quantize(synth.activations_numpy(M, K, 19 + K))
    wd = upload_weights(capi, dev, fmt, W)
    qd = upload_q8(dev, q8)
    y, again = (torch.full((M, N + 4), float("nan"), device=dev) for _ in range(2))
    for out in (y, again):
        capi.gemm(fmt, wd, qd, M, N, K, out=out[:, :N])
    sync()
    assert torch.equal(y[:, :N], again[:, :N]) and bool(torch.isnan(y[:, N:]).all())
    got, n = y.cpu().numpy(), min(N, 96)
    for r0 in (0, N - n):
        s = capi.gemm_block_sums(fmt, wd, qd, M, N, K, r0, n)
        sync()
        C, sums = oracle.gemm(fmt, W, K, q8, n0=r0, n1=r0 + n, want_sums=True)
        part = got[:, r0:r0 + n]
        assert rel_err(part, C) <= TOL[fmt] * 1e-2
        assert np.abs(part - C).max() <= 1e-4 * np.abs(C).max()
        assert np.array_equal(s.cpu().numpy(), sums)


@pytest.mark.parametrize("fmt", list(FMTS.values()), ids=list(FMTS))
@pytest.mark.parametrize("M,N,K,seams", [  # seams: where the second launch of Q4_K, Q6_K and IQ3_S begins (0: there is none)
    (193, 17159, 1024, (16384, 16384, 16384)),
    (65, 18660, 3840, (16384, 16384, 16384)),
    (193, 19075, 1536, (16384, 16384, 16384)),
    (250, 8191, 4096, (0, 0, 0)),
    (196, 16697, 2304, (16384, 16384, 16384)),
    (262, 11930, 2560, (0, 6528, 6528)),
    (205, 18287, 2304, (16384, 16384, 16384)),
    (198, 19661, 2304, (16384, 16384, 16384)),
    (222, 18644, 2304, (16384, 16384, 16384)),
    (77, 17381, 4864, (16384, 16384, 16384)),
    (132, 11388, 2816, (10880, 0, 0)),
    (100, 10226, 8192, (8192, 8192, 8192)),
    (338, 14686, 2560, (10880, 10880, 10880)),
    (68, 16623, 2048, (16384, 16384, 16384)),
    (145, 10902, 2816, (8192, 8192, 0)),
    (97, 16407, 4096, (16384, 16384, 16384)),
    (30, 18305, 6144, (16384, 0, 0)),
    (16, 21409, 4352, (0, 16384, 0)),
    (193, 23864, 2560, (0, 16384, 16384)),
    (294, 17404, 2560, (0, 10880, 10880)),
    (407, 20506, 1792, (16384, 0, 0)),
    (194, 17837, 1792, (16384, 16384, 16384)),
])
def test_rows_in_two_launches(capi, dev, oracle, fmt, M, N, K, seams):
    """Rows whose tiles fill whole rounds and the rest as a launch of its own (and some sizes that one launch does): every element
    written, those on both sides of the seam and the last ones near the oracle's, the same bits again, and the block sums of
    windows that lie on both sides of the seam bit for bit."""
    import torch

    W = synth.weights_numpy(fmt, N, K, 31 + M)
    q8 = oracle.quantize(synth.activations_numpy(M, K, 37 + K))
    wd, qd = upload_weights(capi, dev, fmt, W), upload_q8(dev, q8)
    y, again = (torch.full((M, N + 3), float("nan"), device=dev) for _ in range(2))
    for out in (y, again):
        capi.gemm(fmt, wd, qd, M, N, K, out=out[:, :N])
    sync()
    assert torch.equal(y[:, :N], again[:, :N]) and bool(torch.isnan(y[:, N:]).all()) and not bool(torch.isnan(y[:, :N]).any())
    got = y.cpu().numpy()
    for r0 in (min(max(0, seams[list(FMTS.values()).index(fmt)] - 48), N - 96), N - 96):
        C, sums = oracle.gemm(fmt, W, K, q8, n0=r0, n1=r0 + 96, want_sums=True)
        assert rel_err(got[:, r0:r0 + 96], C) <= TOL[fmt] * 1e-2
        assert np.abs(got[:, r0:r0 + 96] - C).max() <= 1e-4 * np.abs(C).max()
        s = capi.gemm_block_sums(fmt, wd, qd, M, N, K, r0, 96)
        sync()
        assert np.array_equal(s.cpu().numpy(), sums)


@pytest.mark.parametrize("fmt", list(FMTS.values()), ids=list(FMTS))
@pytest.mark.parametrize("M,N,K", [(116, 14367, 1536), (992, 4800, 6400), (256, 8192, 8192), (232, 16587, 13312), (252, 4642, 24576)])
def test_dealt_walks_round_no_coarser_than_four_sums(capi, dev, oracle, fmt, M, N, K):
    """The distance from 64 bits.  A rounding of a 32-bit number is off by 0.425 x 2^-24 of it in the root mean square (evenly spread
    over a unit in the last place, significands by their logarithm).  A walk of B blocks in P sums, each block rounded once at the size
    of the sum by then, is B / 2P roundings at the size of the result, and half as many again where the minima of a pair of blocks
    are another summand; a block's own product and the last additions are few more.
    So four sums give sqrt(B / 8 + 6) roundings (with minima 1.5 B / 8), and a tenth is left for the sample."""
    W = synth.weights_numpy(fmt, N, K, 41 + M)
    q8 = oracle.quantize(synth.activations_numpy(M, K, 43 + K))
    y = capi.gemm(fmt, upload_weights(capi, dev, fmt, W), upload_q8(dev, q8), M, N, K)
    sync()
    n0, n, blocks = 64, 48, K // 32
    _, sums = oracle.gemm(fmt, W, K, q8, n0=n0, n1=n0 + n, want_sums=True)
    scales, minima = np.empty((n, blocks)), np.empty((n, blocks))
    for r in range(n):
        for sb in range(K // 256):
            _, d, m = oracle.subblocks(fmt, W[n0 + r, sb])
            scales[r, 8 * sb:8 * sb + 8], minima[r, 8 * sb:8 * sb + 8] = d.view(np.float16), m.view(np.float16)
    heads = q8.reshape(M, blocks, 36)
    a = heads[:, :, :2].copy().view(np.float16)[:, :, 0].astype(np.float64)
    a_sum = heads[:, :, 2:4].copy().view(np.int16)[:, :, 0] * a
    exact = np.einsum("mnb,nb,mb->mn", sums.astype(np.float64), scales, a, optimize=True)
    if fmt == FMT_Q4_K:
        exact += a_sum @ minima.T
    got = y.cpu().numpy()[:, n0:n0 + n].astype(np.float64)
    assert np.linalg.norm(got - exact) / np.linalg.norm(exact) <= 1.1 * 0.425 * 2.0 ** -24 * np.sqrt((1.5 if fmt == FMT_Q4_K else 1.0) * blocks / 8 + 6)


@pytest.mark.parametrize("fmt", list(FMTS.values()), ids=list(FMTS))
@pytest.mark.parametrize("M,N,K", [(40, 1000, 2304), (129, 4999, 1536), (97, 9799, 1536), (255, 24997, 512), (66, 4259, 768), (20, 12001, 1280),
                                   (35, 4155, 768), (33, 24997, 1280), (67, 8573, 1280), (129, 11253, 768), (324, 5397, 1792)])
def test_dealt_walks_at_the_ends_of_the_scales(capi, dev, oracle, fmt, M, N, K):
    """Scales that are not finite, and scales that are fp16's smallest: an infinite or undefined scale of one Q8_1 block makes
    exactly that token's outputs what the sums as such are (infinite, or not a number), weights' scales below fp16's normal
    range and tokens' scales of one unit are multiplied as they are.  The tolerance is that of every walk."""
    import torch

    W = synth.weights_numpy(fmt, N, K, 23 + M)
    at = {FMT_Q4_K: 0, FMT_Q6_K: 208}.get(fmt, 0)
    blocks = W.reshape(N, K // 256, -1)
    blocks[5::7, :, at:at + 2] = np.frombuffer(np.float16(3e-6).tobytes(), np.uint8)
    q8 = oracle.quantize(synth.activations_numpy(M, K, 29 + K))
    heads = q8.reshape(M, K // 32, 36)
    special = {0: np.float16(np.inf), 7: np.float16(np.nan), M - 1: np.float16(-np.inf), 3: np.float16(6e-8)}
    for m, d in special.items():
        heads[m, (5 * m) % (K // 32), :2] = np.frombuffer(d.tobytes(), np.uint8)
    wd = upload_weights(capi, dev, fmt, W)
    y = capi.gemm(fmt, wd, upload_q8(dev, q8), M, N, K)
    sync()
    got, n = y.cpu().numpy(), min(N, 96)
    for r0 in (0, N - n):
        C, sums = oracle.gemm(fmt, W, K, q8, n0=r0, n1=r0 + n, want_sums=True)
        if fmt != FMT_Q4_K:
            # (the oracle adds minima of zero times an infinite scale, which these formats do not have)
            for m in (0, M - 1):
                with np.errstate(invalid="ignore"):
                    C[m] = sums[m, :, (5 * m) % (K // 32)] * np.float32(special[m])
        part = got[:, r0:r0 + n]
        assert np.array_equal(np.isnan(part), np.isnan(C)) and np.array_equal(np.isposinf(part), np.isposinf(C))
        assert np.array_equal(np.isneginf(part), np.isneginf(C))
        whole = np.isfinite(C).all(1)
        assert rel_err(part[whole], C[whole]) <= TOL[fmt] * 1e-2
        assert whole.sum() == M - 3


@pytest.mark.parametrize("fmt", list(FMTS.values()), ids=list(FMTS))
@pytest.mark.parametrize("M,N,K", [(31, 4095, 2304), (20, 12001, 4864), (40, 1000, 2304), (129, 4999, 1536), (33, 24997, 1280),
                                   (199, 5120, 1536), (255, 24997, 1280), (256, 8192, 2048), (66, 4259, 768), (35, 4155, 768), (324, 5397, 1792)])
def test_an_infinite_scale_leaves_other_tokens_and_rows_alone(capi, dev, oracle, fmt, M, N, K):
    """An infinity in one token and one in one row of W: every other element has the bits that it has without them."""
    import torch

    W = synth.weights_numpy(fmt, N, K, 51 + M)
    q8 = oracle.quantize(synth.activations_numpy(M, K, 53 + K))
    plain = capi.gemm(fmt, upload_weights(capi, dev, fmt, W), upload_q8(dev, q8), M, N, K)
    infinite = np.frombuffer(np.float16(np.inf).tobytes(), np.uint8)
    token, row, at = M // 2, N // 2, {FMT_Q4_K: 0, FMT_Q6_K: 208}.get(fmt, 0)
    q8.reshape(M, K // 32, 36)[token, 3, :2] = infinite
    W.reshape(N, K // 256, -1)[row, 1, at:at + 2] = infinite
    odd = capi.gemm(fmt, upload_weights(capi, dev, fmt, W), upload_q8(dev, q8), M, N, K)
    sync()
    others = torch.ones(M, N, dtype=torch.bool, device=dev)
    others[token], others[:, row] = False, False
    assert torch.equal(plain[others], odd[others])
    assert not bool(torch.isfinite(odd[token]).any()) and not bool(torch.isfinite(odd[:, row]).all())


def test_block_sums_at_their_limits(capi, dev, oracle):
    """Q6_K rows and activations whose every product is the largest there is, 127 and -128 both ways: sums of 32 of them."""
    M, N, K, fmt = 33, 4096, 512, FMT_Q6_K
    W = synth.weights_numpy(fmt, N, K, 5)
    W.reshape(N, -1, 210)[:, :, :192] = np.where(np.arange(N)[:, None, None] % 2, 255, 0)   # all bits: q = 31; none: -32
    W.reshape(N, -1, 210)[:, :, 192:208] = 127
    x = np.where(np.arange(M)[:, None] % 2, 1.0, -1.0) * np.ones((M, K), np.float32)
    q8 = oracle.quantize(x.astype(np.float32))
    wd = upload_weights(capi, dev, fmt, W)
    qd = upload_q8(dev, q8)
    s = capi.gemm_block_sums(fmt, wd, qd, M, N, K, 0, 64)
    y = capi.gemm(fmt, wd, qd, M, N, K)
    sync()
    C, sums = oracle.gemm(fmt, W, K, q8, n0=0, n1=64, want_sums=True)
    assert np.abs(sums).max() >= 32 * 120 * 127
    assert np.array_equal(s.cpu().numpy(), sums)
    assert rel_err(y.cpu().numpy()[:, :64], C) <= TOL[fmt] * 1e-2


@pytest.mark.parametrize("fmt", list(FMTS.values()), ids=list(FMTS))
def test_more_tiles_than_the_chip_holds(capi, dev, oracle, fmt):
    """More tiles than the chip holds at once, with a sparsely filled last round of workgroups
    (580 tiles of 128 x 64 on 512 workgroup slots), ragged in both directions (130 tokens: the
    second token tile holds two; 18550 rows: the last row tile holds 54): every output element
    written exactly once and equal to the oracle's."""
    import torch

    M, N, K = 130, 18550, 512
    W = synth.weights_numpy(fmt, N, K, 4242)
    q8 = oracle.quantize(synth.activations_numpy(M, K, 4243))
    wd = upload_weights(capi, dev, fmt, W)
    qd = upload_q8(dev, q8)
    y = torch.full((M, N), float("nan"), device=dev)
    capi.gemm(fmt, wd, qd, M, N, K, out=y)
    sync()
    got = y.cpu().numpy()
    assert np.isfinite(got).all()
    C = oracle.gemm(fmt, W, K, q8)
    assert rel_err(got, C) <= TOL[fmt] * 1e-2
    # the worst single element, too: a misplaced tile would hide in a norm
    assert np.abs(got - C).max() <= 1e-4 * np.abs(C).max()
    y2 = torch.full((M, N), float("nan"), device=dev)
    capi.gemm(fmt, wd, qd, M, N, K, out=y2)
    sync()
    assert torch.equal(y, y2)


def test_prefill_config_full_size(capi, dev, oracle):
    """Config 3: M=512, K=5120, N=25600, Q4_K.  Oracle on a window of weight rows for all
    512 tokens; determinism over the whole output."""
    import torch

    M, N, K = 512, 25600, 5120
    fmt = FMT_Q4_K
    wd = synth.weights_torch(fmt, N, K, 31337, dev)
    x = synth.activations_numpy(M, K, 5)
    xd = torch.from_numpy(x).to(dev)
    qd = capi.quantize_q8_1(xd)
    y = capi.gemm(fmt, wd, qd, M, N, K)
    y2 = capi.gemm(fmt, wd, qd, M, N, K)
    sync()
    assert torch.equal(y, y2)
    q8 = oracle.quantize(x)
    assert np.array_equal(qd.cpu().numpy().reshape(q8.shape), q8)
    Wh = wd.cpu().numpy()
    for n0 in (0, 12800 - 32, N - 64):
        C, sums = oracle.gemm(fmt, Wh, K, q8, n0=n0, n1=n0 + 64, want_sums=True)
        assert rel_err(y.cpu().numpy()[:, n0:n0 + 64], C) <= TOL[fmt] * 1e-2
        s = capi.gemm_block_sums(fmt, wd, qd, M, N, K, n0, 64)
        sync()
        assert np.array_equal(s.cpu().numpy(), sums), f"block sums of rows from {n0}"
    assert np.isfinite(y.cpu().numpy()).all()


def test_epilogue_alpha_beta_bias(capi, dev, oracle):
    import torch

    rng = np.random.default_rng(4)
    C = rng.standard_normal((5, 96)).astype(np.float32)
    T = rng.standard_normal((5, 96)).astype(np.float32)
    b = rng.standard_normal(96).astype(np.float32)
    for alpha, beta, bias in ((1.0, 0.0, None), (0.5, 2.0, b), (2.0, 1.0, None)):
        cd = torch.from_numpy(C.copy()).to(dev)
        capi.epilogue(cd, torch.from_numpy(T).to(dev), None if bias is None else torch.from_numpy(bias).to(dev),
                      alpha, beta)
        sync()
        want = oracle.epilogue(C, T, alpha, beta, bias)
        assert np.allclose(cd.cpu().numpy(), want, rtol=1e-6, atol=1e-6)
    # beta == 0 must overwrite NaNs, like the reference's zero-fill
    cd = torch.full((5, 96), float("nan"), device=dev)
    capi.epilogue(cd, torch.from_numpy(T).to(dev), None, 1.0, 0.0)
    sync()
    assert np.array_equal(cd.cpu().numpy(), T)


def test_empty_and_errors(capi, dev):
    import torch

    lib = capi.load()
    w = torch.zeros(4096, dtype=torch.uint8, device=dev)
    y = torch.zeros(64, device=dev)
    assert lib.llam_ql_gemm(FMT_Q4_K, w.data_ptr(), w.data_ptr(), y.data_ptr(), 0, 4, 256, 4, 0, None)
    assert not lib.llam_ql_gemm(FMT_Q4_K, w.data_ptr(), w.data_ptr(), y.data_ptr(), 2, 4, 255, 4, 0, None)
