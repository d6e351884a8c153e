"""Linear layers of up to 16 rows against sums in 64 bits: half and whole tiles at the edges of their rule, the fused norm."""
import ctypes

import pytest

from llaminar_amd import sequence as sq
from tests.test_gpu_linear_tiled import tiles

pytestmark = pytest.mark.gpu

F32, BF16 = sq.F32, sq.BF16

# half tiles: one to eight rows, one tile, the most tiles (128), K of one step, of fewer steps than wavefronts, of an odd
# number of steps a wavefront, 65 tiles and K of 4096; whole tiles on the other side: nine rows, 129 and 256 tiles, K of
# 2048 (bf16); walks of half a round of steps, of one round and of one and a part, four wavefronts with rounds of 4, 5, 7
# and 8 steps
SHAPES = [(1, 16, 64), (8, 16, 4096), (8, 2048, 128), (7, 2064, 1088), (3, 2048, 10304), (8, 4080, 4160), (9, 2048, 4096),
          (8, 4096, 4096), (5, 4096, 4032), (6, 1040, 4096), (8, 2048, 5120), (4, 1024, 2112), (8, 48, 2048), (16, 48, 8256), (12, 4112, 1024), (16, 80, 2048),
          (9, 48, 2112), (9, 48, 960), (12, 2064, 576)]


# a fused norm takes up to 8192 values: all of them in one row and in sixteen, half and whole tiles
NORMED = [(1, 16, 64), (1, 2048, 5120), (2, 1040, 4096), (3, 80, 2112), (7, 2064, 1088), (1, 32, 8192), (2, 80, 4096), (3, 32, 2688), (4, 2048, 2048), (5, 4112, 1600), (16, 32, 512)]


@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("M,N,K,norm", [(*s, False) for s in SHAPES] + [(*s, True) for s in NORMED])
def test_few_rows(dev, M, N, K, norm, dtype):
    import torch

    torch.manual_seed(M + N + K)
    a = torch.randn(M, K + 64, device=dev)[:, :K]
    w = torch.randn(N, K, device=dev).bfloat16()
    scale, real = torch.rand(K, device=dev) + 0.5, K - 3
    y = torch.full((M + 1, N + 4), 5.0, device=dev)
    h = torch.zeros(M, K, device=dev, dtype=torch.float32 if dtype == F32 else torch.bfloat16)
    given = a if norm or dtype == F32 else torch.nn.functional.pad(a.bfloat16(), (0, 64))[:, :K]
    laid = tiles(w)
    args = sq.LinearArgs(d_a=given.data_ptr(), d_w=laid.data_ptr(), d_y=y.data_ptr(), M=M, N=N, K=K, lda=K + 64, ldy=N + 4, out=sq.OUT_F32, batch=1)
    if norm:
        args.d_norm, args.d_h_out, args.k_real, args.eps = scale.data_ptr(), h.data_ptr(), real, 1e-5
    assert sq.load().llam_seq_linear(ctypes.byref(args), dtype, 0, torch.cuda.current_stream().cuda_stream), sq.load().llam_ql_last_error()
    torch.cuda.synchronize()
    x = given.double()
    if norm:
        x = x / torch.sqrt((x * x).sum(1, keepdim=True) / real + 1e-5) * scale.double()
        # the sum of squares: off by K 2^-24 of itself at most, its root by half of that; then three products and a rounding to T
        # (bf16: 8 significant bits, so half a unit of the last is 2^-8 of the value at most)
        relative = K * 2.0 ** -25 + 6 * 2.0 ** -24 + (2.0 ** -8 if dtype == BF16 else 0.0)
        assert ((h.double() - x).abs() <= relative * x.abs()).all()
        x = h.double()
    # K products in 32 bits, in any order: each addition is off by 2^-23 of a partial sum at most
    bound = (K + 1) * 2.0 ** -23 * (x.abs() @ w.double().abs().T)
    assert ((y[:M, :N].double() - x @ w.double().T).abs() <= bound).all()
    assert (y[M:] == 5.0).all() and (y[:, N:] == 5.0).all(), "written past the output"


def test_a_normed_value_beyond_32_bits(dev):
    """An infinite normed value of a row of fp32, which is cut in pieces: infinite sums in that row, none in the other."""
    import torch

    torch.manual_seed(0)
    a, w = torch.randn(2, 2048, device=dev), torch.randn(64, 2048, device=dev).bfloat16()
    scale = torch.ones(2048, device=dev)
    a[0, 5], a[1, 5], scale[5] = 10.0, 0.0, 3e38
    y, laid = torch.zeros(2, 64, device=dev), tiles(w)
    args = sq.LinearArgs(d_a=a.data_ptr(), d_w=laid.data_ptr(), d_y=y.data_ptr(), M=2, N=64, K=2048, lda=2048, ldy=64, out=sq.OUT_F32, batch=1)
    args.d_norm, args.k_real, args.eps = scale.data_ptr(), 2048, 1e-5
    assert sq.load().llam_seq_linear(ctypes.byref(args), F32, 0, torch.cuda.current_stream().cuda_stream), sq.load().llam_ql_last_error()
    torch.cuda.synchronize()
    assert (w[:, 5] != 0).all()
    assert torch.equal(y[0], torch.sign(w[:, 5].float()) * float("inf")) and torch.isfinite(y[1]).all()


@pytest.mark.parametrize("pair", [False, True])
@pytest.mark.parametrize("M,N,K", [(1, 16, 8192), (3, 2064, 2688), (8, 4112, 1024), (16, 48, 512)])
def test_normed_values_and_weights_beyond_the_pieces(dev, M, N, K, pair):
    """Normed rows of fp32 are cut in pieces: infinite weights, and values down to the smallest bf16, are multiplied whole."""
    import torch

    torch.manual_seed(M)
    a, w = torch.randn(M, K, device=dev), torch.randn(N, K, device=dev).bfloat16()
    laid, lib, stream = tiles(w), sq.load(), torch.cuda.current_stream().cuda_stream
    infinite = w.clone()
    infinite[3, 5], infinite[N - 1, K - 1], infinite[9, 0], infinite[9, 9] = float("inf"), float("-inf"), float("inf"), float("-inf")
    a[0, 5], a[:, 0] = 0.0, 1.5
    laid_infinite = tiles(infinite)

    def run(weights, scale):
        y, h = torch.zeros(2, M, N, device=dev), torch.zeros(M, K, device=dev)
        args = [sq.LinearArgs(d_a=a.data_ptr(), d_w=weights.data_ptr(), d_y=y[i].data_ptr(), M=M, N=N, K=K, lda=K, ldy=N, out=sq.OUT_F32, batch=1,
                              d_norm=scale.data_ptr(), k_real=K, eps=1e-5) for i in range(2)]
        args[0].d_h_out = h.data_ptr()
        if pair:
            assert lib.llam_seq_linear_pair(ctypes.byref(args[0]), ctypes.byref(args[1]), F32, 0, stream), lib.llam_ql_last_error()
        else:
            assert lib.llam_seq_linear(ctypes.byref(args[0]), F32, 0, stream), lib.llam_ql_last_error()
        torch.cuda.synchronize()
        if pair:
            assert torch.equal(y[0].view(torch.int32), y[1].view(torch.int32))
        return y[0], h.double()

    y, h = run(laid_infinite, torch.ones(K, device=dev))
    want = (h @ infinite.double().T).float()
    assert torch.isnan(want[0, 3])
    for kind in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(kind(y), kind(want))
    plain = [n for n in range(N) if n not in (3, 9, N - 1)]
    bound = (K + 1) * 2.0 ** -23 * (h.abs() @ w.double().abs().T)
    assert ((y[:, plain].double() - h @ w[plain].double().T).abs() <= bound[:, plain]).all()
    for size in (1e-30, 1e-36, 1.2e-39):
        for kept in (1, K):   # single values and whole rows
            scale = torch.zeros(K, device=dev)
            scale[:kept] = size
            y, h = run(laid, scale)
            # and each product and sum may be rounded to a multiple of the smallest value, 2^-149
            bound = (K + 1) * 2.0 ** -23 * (h.abs() @ w.double().abs().T) + K * 2.0 ** -149
            assert (h != 0).any() and ((y.double() - h @ w.double().T).abs() <= bound).all()
