"""Linear layers of many rows against sums in 64 bits: every tile of the rule at its edges, strides, batches, outputs."""
import ctypes

import pytest

from llaminar_amd import sequence as sq

pytestmark = pytest.mark.gpu

F32, BF16 = sq.F32, sq.BF16


def tiles(w):
    n, k = w.shape
    return w.reshape(n // 16, 16, k // 32, 4, 8).permute(0, 2, 3, 1, 4).contiguous()


def run(torch, a, w, y, dtype, out=sq.OUT_F32, N=None, K=None, batch=1, strides=(0, 0, 0), bias=None):
    M = y.shape[-2] if y.dim() == 3 else y.shape[0]
    args = sq.LinearArgs(d_a=a.data_ptr(), d_w=w.data_ptr(), d_y=y.data_ptr(), M=M, N=N, K=K, lda=a.stride(-2), ldy=y.stride(-2), out=out,
                         batch=batch, a_stride=strides[0], w_stride=strides[1], y_stride=strides[2], limit=7.0)
    if bias is not None:
        args.d_bias = bias.data_ptr()
    ok = sq.load().llam_seq_linear(ctypes.byref(args), dtype, 0, torch.cuda.current_stream().cuda_stream)
    assert ok, sq.load().llam_ql_last_error()
    torch.cuda.synchronize()


def close(torch, y, a, w, K, extra=0.0):
    """Sums of K products in 32 bits, in any order: each addition is off by 2^-23 of a partial sum at most."""
    a, w = a.double(), w.double()
    bound = (K + 1) * 2.0 ** -23 * (a.abs() @ w.abs().T)
    want = a @ w.T
    assert ((y.double() - want).abs() <= bound + extra * want.abs()).all()
    return want


# rows x columns x K: a single row more than the row-at-a-time kernel takes, edges of every tile, K of one and of an
# odd number of turns, and each tile with rows and columns left over (test_launch_rules.py)
SHAPES = [(17, 16, 64), (31, 48, 192), (33, 80, 320), (64, 64, 128), (65, 272, 704), (100, 6160, 2048), (127, 144, 64),
          (129, 256, 2048), (255, 528, 192), (257, 1040, 128), (300, 6160, 512), (522, 2048, 2112), (300, 16384, 192),
          (1000, 8208, 64), (2048, 2048, 192), (2048, 4112, 128), (2048, 15440, 64),
          (1000, 6160, 192), (2000, 3088, 320), (300, 8208, 192), (2000, 2064, 192), (520, 2064, 2112)]


@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_sums(dev, M, N, K, dtype):
    import torch

    torch.manual_seed(M + N)
    a = torch.randn(M, K + 64, device=dev)[:, :K]
    a = a if dtype == F32 else torch.nn.functional.pad(a.bfloat16(), (0, 64))[:, :K]
    w = torch.randn(N, K, device=dev).bfloat16()
    y = torch.full((M + 1, N + 4), 5.0, device=dev)
    run(torch, a, tiles(w), y[:M, :N], dtype, N=N, K=K)
    close(torch, y[:M, :N], a, w, K)
    assert (y[M:] == 5.0).all() and (y[:, N:] == 5.0).all(), "written past the output"


@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("out", [sq.OUT_ADD, sq.OUT_ELEM, sq.OUT_GATED, sq.OUT_RELU2, sq.OUT_GATED_CLAMP])
@pytest.mark.parametrize("M,N,K", [(40, 96, 192), (300, 2080, 128), (2048, 4128, 64), (1000, 6176, 192)])
def test_outputs(dev, M, N, K, out, dtype):
    import torch

    torch.manual_seed(out)
    a, w = torch.randn(M, K, device=dev), (torch.randn(N, K, device=dev) * K ** -0.5).bfloat16()
    a = a if dtype == F32 else a.bfloat16()
    gated = out in (sq.OUT_GATED, sq.OUT_GATED_CLAMP)
    kind = torch.float32 if dtype == F32 or out == sq.OUT_ADD else torch.bfloat16
    y = torch.randn(M, N // 2 if gated else N, device=dev).to(kind)
    before = y.double()
    run(torch, a, tiles(w), y, dtype, out, N, K)
    z = a.double() @ w.double().T
    if gated:
        pair = z.reshape(M, N // 32, 2, 16)
        gate, up = pair[:, :, 0].reshape(M, -1), pair[:, :, 1].reshape(M, -1)
        if out == sq.OUT_GATED:
            want = torch.nn.functional.gelu(gate, approximate="tanh") * up
        else:
            g, u = gate.clamp(max=7.0), up.clamp(-7.0, 7.0)
            want = g * torch.sigmoid(1.702 * g) * (u + 1.0)
    else:
        want = {sq.OUT_ADD: before + z, sq.OUT_ELEM: z, sq.OUT_RELU2: torch.relu(z) ** 2}[out]
    # rounding of the result, and sums of unit size (error below 2^-23 K) through an activation of slope below 20
    off = (y.double() - want).abs()
    assert (off <= (2.0 ** -8 if kind == torch.bfloat16 else 2.0 ** -20) * want.abs() + 20 * K * 2.0 ** -23).all()


@pytest.mark.parametrize("dtype", [BF16, F32])
def test_batches_and_strides(dev, dtype):
    import torch

    B, M, N, K = 5, 70, 48, 128
    a = torch.randn(M, B, K, device=dev)
    a = a if dtype == F32 else a.bfloat16()
    w = torch.randn(B, N, K, device=dev).bfloat16()
    y = torch.zeros(M, B, N, device=dev)
    t = torch.stack([tiles(w[b]) for b in range(B)])
    run(torch, a.permute(1, 0, 2), t, y.permute(1, 0, 2), dtype, N=N, K=K, batch=B, strides=(K, N * K, N))
    for b in range(B):
        close(torch, y[:, b], a[:, b], w[b], K)


@pytest.mark.parametrize("M", [20, 300, 2048])
def test_values_at_the_ends_of_the_range(dev, M):
    """32-bit rows are multiplied in three pieces: infinities, numbers that are none and the largest and the small
    ones come out as a product of the whole value gives them."""
    import torch

    N, K = 2048 if M == 2048 else 64, 256
    torch.manual_seed(1)
    a = torch.randn(M, K, device=dev)
    a[3, 5], a[M - 1, 255], a[9, 100], a[11, 0], a[11, 1] = float("inf"), float("-inf"), float("nan"), 3.4e38, -3.4e38
    a[12] *= 1e-30
    a[13] = 0.0
    w = torch.randn(N, K, device=dev).bfloat16()
    y = torch.zeros(M, N, device=dev)
    run(torch, a, tiles(w), y, F32, N=N, K=K)
    want = (a.double() @ w.double().T).float()
    rows = [m for m in range(M) if m != 11]   # (whose sums overflow or not by the order)
    for kind in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(kind(y[rows]), kind(want[rows]))
    plain = [m for m in range(M) if m not in (3, 9, 11, M - 1)]
    close(torch, y[plain], a[plain], w, K)
    assert (y[13] == 0.0).all()


# the smallest shapes of each tile of 32-bit rows
WHOLE = [(20, 64, 256), (300, 6160, 512), (257, 4112, 64), (1000, 6160, 192)]


@pytest.mark.parametrize("M,N,K", WHOLE)
def test_infinite_weights_of_32_bit_rows(dev, M, N, K):
    """Most pieces of a value are zero, and zero times infinity is not a number: such sums are those of the whole values."""
    import torch

    torch.manual_seed(M)
    a, w = torch.randn(M, K, device=dev).bfloat16().float(), torch.randn(N, K, device=dev).bfloat16()
    w[3, 5], w[N - 1, K - 1], w[N // 2, 0], w[N // 2, 9] = float("inf"), float("-inf"), float("inf"), float("-inf")
    a[2, 5], a[M - 1, 7] = 0.0, float("inf")
    y = torch.zeros(M, N, device=dev)
    run(torch, a, tiles(w), y, F32, N=N, K=K)
    want = (a.double() @ w.double().T).float()
    assert torch.isposinf(want[:, 3]).any() and torch.isnan(want[2, 3])
    for kind in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(kind(y), kind(want))
    plain = [n for n in range(N) if n not in (3, N // 2, N - 1)]
    close(torch, y[:M - 1][:, plain], a[:M - 1], w[plain], K)


@pytest.mark.parametrize("M,N,K", WHOLE)
def test_small_values_of_32_bit_rows(dev, M, N, K):
    """Rows down to values of the size of the smallest bf16, whole ones and single values: no bits lost below it."""
    import torch

    torch.manual_seed(M)
    a, w = torch.randn(M, K, device=dev), torch.randn(N, K, device=dev).bfloat16()
    a[::6], a[3::6] = 0.0, 0.0
    a[::6, 0], a[3::6, K - 1] = 1.2345678, -1.9876543
    a = (a.double() * 10.0 ** -(20 + torch.arange(M, device=dev) % 20).double().unsqueeze(1)).float()
    y = torch.zeros(M, N, device=dev)
    run(torch, a, tiles(w), y, F32, N=N, K=K)
    want = a.double() @ w.double().T
    # as in close(), and each product and sum may be rounded to a multiple of the smallest value, 2^-149
    bound = (K + 1) * 2.0 ** -23 * (a.double().abs() @ w.double().abs().T) + K * 2.0 ** -149
    # (a sum that the pieces make zero is taken at its word: of each value less than 2^-133 may be missing)
    bound[y == 0.0] = K * 2.0 ** -133 * float(w.abs().max())
    assert ((y.double() - want).abs() <= bound).all() and (y != 0.0).double().mean() > 0.99


@pytest.mark.parametrize("out", [sq.OUT_ELEM, sq.OUT_GATED, sq.OUT_RELU2])
@pytest.mark.parametrize("M,N,K", SHAPES[:6] + [(300, 2080, 128), (2000, 3104, 64), (520, 2080, 2112)])
def test_rows_that_start_at_eight_bytes(dev, M, N, K, out):
    """bf16 results whose rows lie 8 bytes off 16: the same values as of aligned rows, and nothing past them."""
    import torch

    N = max(32, N // 32 * 32) if out == sq.OUT_GATED else N
    columns = N // 2 if out == sq.OUT_GATED else N
    torch.manual_seed(M)
    a, t = torch.randn(M, K, device=dev).bfloat16(), tiles((torch.randn(N, K, device=dev) * K ** -0.5).bfloat16())
    aligned, y = torch.full((M, columns + 8), 5.0, device=dev).bfloat16(), torch.full((M + 1, columns + 4), 5.0, device=dev).bfloat16()
    run(torch, a, t, aligned[:, :columns], BF16, out, N, K)
    run(torch, a, t, y[:M, :columns], BF16, out, N, K)
    assert torch.equal(y[:M, :columns], aligned[:, :columns])
    assert (y[M:] == 5.0).all() and (y[:, columns:] == 5.0).all() and (aligned[:, columns:] == 5.0).all()


@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("M,N,K,batch", [(*s, 1) for s in SHAPES] + [(70, 48, 128, 5), (601, 512, 128, 16), (2049, 128, 512, 16)])
def test_some_rows_of_a_layer(dev, M, N, K, batch, dtype):
    """The bits that the rows have among all, whatever tile they get by themselves; the others are neither read nor written."""
    import torch

    torch.manual_seed(M + N)
    kind, out = (torch.float32, sq.OUT_F32) if dtype == F32 or batch == 1 else (torch.bfloat16, sq.OUT_ELEM)
    a = torch.randn(M, batch * K, device=dev).to(torch.float32 if dtype == F32 else torch.bfloat16)
    t = torch.stack([tiles((torch.randn(N, K, device=dev) * K ** -0.5).bfloat16()) for _ in range(batch)])
    all_rows, y = torch.zeros(M, batch * N + 4, device=dev, dtype=kind), torch.empty(M, batch * N + 4, device=dev, dtype=kind)
    args = sq.LinearArgs(d_w=t.data_ptr(), M=M, N=N, K=K, lda=batch * K, ldy=batch * N + 4, out=out, batch=batch, a_stride=K, w_stride=N * K,
                         y_stride=N)
    args.d_a, args.d_y = a.data_ptr(), all_rows.data_ptr()
    lib, stream = sq.load(), torch.cuda.current_stream().cuda_stream
    assert lib.llam_seq_linear(ctypes.byref(args), dtype, 0, stream), lib.llam_ql_last_error()
    for stretches in [[(0, 1)], [(M - 1, 1)], [(1, M - 1)], [(0, M // 2), (M - 7, 7)], [(0, M)], [], [(i, 1) for i in range(0, 17, 2)],
                      [(0, 3), (3, M // 3), (M // 2, M // 4), (M - 1, 1)]]:
        only, others = torch.full_like(a, float("nan")), torch.ones(M, dtype=torch.bool, device=dev)
        for first, n in stretches:
            only[first:first + n] = a[first:first + n]
            others[first:first + n] = False
        args.d_a, args.d_y = only.data_ptr(), y.fill_(5.0).data_ptr()
        first, n = ((ctypes.c_int32 * len(stretches))(*(s[i] for s in stretches)) for i in (0, 1))
        assert lib.llam_seq_linear_rows(ctypes.byref(args), len(stretches), first, n, dtype, 0, stream), lib.llam_ql_last_error()
        torch.cuda.synchronize()
        assert torch.equal(y[~others, :batch * N], all_rows[~others, :batch * N]), stretches
        assert (y[others] == 5.0).all() and (y[:, batch * N:] == 5.0).all()


# ---- tiles cut along K (llam_seq_linear_within) ------------------------------------------------------------

# every tile that is cut, with and without whole ones beside it, slices of unequal length (test_launch_rules.py)
SPLIT = [(17, 48, 2112), (33, 80, 1024), (65, 2064, 8256), (257, 2064, 8256), (1000, 16400, 512), (700, 6160, 8256), (2048, 4112, 2112),
         (65, 2064, 1024), (2048, 272, 4160), (2048, 1280, 8256), (1500, 6160, 512), (200, 4112, 4160)]


def run_within(torch, a, w, y, dtype, out=sq.OUT_F32, N=None, K=None, bias=None, short=0):
    """The layer with the scratch that it asks for, `short` bytes less; what lies behind the scratch stays as it is."""
    M = y.shape[0]
    need = sq.load().llam_seq_linear_scratch_bytes(M, N, K, dtype, 0)
    scratch = torch.full((need + 4096,), 171, dtype=torch.uint8, device=y.device)
    args = sq.LinearArgs(d_a=a.data_ptr(), d_w=w.data_ptr(), d_y=y.data_ptr(), M=M, N=N, K=K, lda=a.stride(-2), ldy=y.stride(-2), out=out,
                         batch=1, limit=7.0, d_bias=0 if bias is None else bias.data_ptr())
    ok = sq.load().llam_seq_linear_within(ctypes.byref(args), scratch.data_ptr(), need - short, dtype, 0, torch.cuda.current_stream().cuda_stream)
    assert ok, sq.load().llam_ql_last_error()
    torch.cuda.synchronize()
    assert (scratch[need - short:] == 171).all(), "written past the scratch"
    return need


@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("M,N,K", SPLIT)
def test_slices_of_k(dev, M, N, K, dtype):
    import torch

    torch.manual_seed(M + N)
    a = torch.randn(M, K, device=dev)
    a = a if dtype == F32 else a.bfloat16()
    w, bias = torch.randn(N, K, device=dev).bfloat16(), torch.randn(N, device=dev)
    y = torch.full((M + 1, N + 4), 5.0, device=dev)
    run_within(torch, a, tiles(w), y[:M, :N], dtype, N=N, K=K)
    close(torch, y[:M, :N], a, w, K)
    assert (y[M:] == 5.0).all() and (y[:, N:] == 5.0).all(), "written past the output"
    again = torch.empty(M, N, device=dev)
    run_within(torch, a, tiles(w), again, dtype, N=N, K=K)
    assert torch.equal(again, y[:M, :N])
    run_within(torch, a, tiles(w), again, dtype, N=N, K=K, bias=bias)
    assert torch.equal(again, y[:M, :N] + bias)
    run_within(torch, a, tiles(w), again, dtype, N=N, K=K, short=16)   # (fewer slices, or none)
    close(torch, again, a, w, K)


@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("out", [sq.OUT_ADD, sq.OUT_ELEM, sq.OUT_GATED, sq.OUT_RELU2, sq.OUT_GATED_CLAMP])
@pytest.mark.parametrize("M,N,K", [(40, 96, 2112), (300, 2080, 4160), (700, 6176, 4160)])
def test_outputs_of_slices(dev, M, N, K, out, dtype):
    """The same values as without scratch: sums of unit size differ by their rounding, 2^-23 K, through slopes below 20."""
    import torch

    torch.manual_seed(out)
    a, w = torch.randn(M, K, device=dev), tiles((torch.randn(N, K, device=dev) * K ** -0.5).bfloat16())
    a = a if dtype == F32 else a.bfloat16()
    kind = torch.float32 if dtype == F32 or out == sq.OUT_ADD else torch.bfloat16
    y = torch.randn(M, N // 2 if out in (sq.OUT_GATED, sq.OUT_GATED_CLAMP) else N, device=dev).to(kind)
    want = y.clone()
    run(torch, a, w, want, dtype, out, N, K)
    run_within(torch, a, w, y, dtype, out, N, K)
    off = (y.double() - want.double()).abs()
    assert (off <= (2.0 ** -8 if kind == torch.bfloat16 else 2.0 ** -20) * want.double().abs() + 20 * K * 2.0 ** -23).all()


@pytest.mark.parametrize("M,N,K", [(20, 64, 2048), (65, 2064, 1024), (200, 4112, 4160)])
def test_infinite_and_small_values_in_slices(dev, M, N, K):
    """32-bit rows in three pieces: what the pieces do not carry is multiplied once more, slice by slice."""
    import torch

    torch.manual_seed(M)
    a, w = torch.randn(M, K, device=dev).bfloat16().float(), torch.randn(N, K, device=dev).bfloat16()
    w[3, 5], w[N - 1, K - 1], w[N // 2, 0], w[N // 2, K - 9] = float("inf"), float("-inf"), float("inf"), float("-inf")
    a[2, 5], a[M - 1, 7] = 0.0, float("inf")
    a[5] = 0.0
    a[5, 3], a[5, K - 2] = 1.2345678e-33, -2.3e-34
    y = torch.zeros(M, N, device=dev)
    assert run_within(torch, a, tiles(w), y, F32, N=N, K=K) > 0
    want = (a.double() @ w.double().T).float()
    assert torch.isposinf(want[:, 3]).any() and torch.isnan(want[2, 3])
    for kind in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(kind(y), kind(want))
    plain = [n for n in range(N) if n not in (3, N // 2, N - 1)]
    close(torch, y[:M - 1][:, plain], a[:M - 1], w[plain], K)
