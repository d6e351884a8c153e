"""Routed experts.  Of 2 to 16 rows: the rows that share an expert are multiplied together, and each is what it is alone.
Of more: rows grouped by expert, against sums in 64 bits."""
import ctypes

import pytest

from llaminar_amd import sequence as sq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [sq.BF16, sq.F32])
@pytest.mark.parametrize("M,experts,top,ff,shared", [(2, 2, 2, 64, 0), (3, 1, 1, 192, 64), (8, 6, 4, 128, 320), (15, 64, 6, 64, 64),
                                                     (16, 70, 64, 64, 0), (16, 3, 1, 320, 128)])
def test_rows_together_are_rows_alone(dev, M, experts, top, ff, shared, dtype):
    """Bit for bit: the columns of a matrix product do not meet."""
    import torch

    K, T = 320, torch.float32 if dtype == sq.F32 else torch.bfloat16
    torch.manual_seed(M + experts)
    up, down = (torch.randn(experts * ff * K, device=dev).bfloat16() for _ in range(2))
    both = torch.randn(2, max(shared, 1) * K, device=dev).bfloat16()
    logits, h = torch.randn(M, experts + 16, device=dev), torch.randn(M, K, device=dev).to(T)
    base = torch.randn(M, K + 4, device=dev)
    lib, stream = sq.load(), torch.cuda.current_stream().cuda_stream

    def run(rows):
        x, n = base[rows].clone(), len(rows)
        z, r = logits[rows].clone(), h[rows].clone()
        size = lib.llam_seq_experts_scratch_bytes(n, experts, top, ff, shared, K)
        scratch = torch.full((size,), 255, dtype=torch.uint8, device=dev)
        a = sq.ExpertsArgs(d_logits=z.data_ptr(), ldz=experts + 16, d_up=up.data_ptr(), d_down=down.data_ptr(), up_stride=ff * K, down_stride=ff * K,
                           experts=experts, top=top, ff=ff, shared_ff=shared, K=K, N=K, d_h=r.data_ptr(), d_x=x.data_ptr(), ldx=K + 4)
        if shared:
            a.d_shared_up, a.d_shared_down = both[0].data_ptr(), both[1].data_ptr()
        assert lib.llam_seq_experts(ctypes.byref(a), n, scratch.data_ptr(), size, dtype, 0, stream), lib.llam_ql_last_error()
        torch.cuda.synchronize()
        return x

    together = run(list(range(M)))
    alone = torch.cat([run([m]) for m in range(M)])
    assert torch.isfinite(together).all() and not torch.equal(together, base)
    assert torch.equal(together, alone)


# rows, experts, of a row, widths of an expert, the shared one and the model: one list and two, halves of tiles and (more than 8 rows
# of a wide model) whole ones; fewer k-steps than wavefronts, a remainder of them, more
@pytest.mark.parametrize("dtype", [sq.BF16, sq.F32])
@pytest.mark.parametrize("M,experts,top,ff,shared,K", [(1, 6, 4, 64, 64, 128), (8, 40, 3, 576, 0, 192), (9, 5, 5, 64, 1216, 128), (9, 30, 2, 640, 64, 4160),
                                                       (16, 1024, 4, 64, 0, 4096), (16, 300, 64, 64, 64, 192), (13, 2, 1, 192, 0, 4160)])
def test_few_rows_against_64_bits(dev, M, experts, top, ff, shared, K, dtype):
    few_rows_against_64_bits(dev, M, experts, top, ff, shared, K, dtype)


# lists of some hundred experts, whose uses are more than the 48 KB of LDS that a launch has without asking, up to the most there can be; several
# windows of 64 experts, with the shared one first; lists of one row, two and four, of eight rows each of experts of one step, of nine
@pytest.mark.parametrize("dtype", [sq.BF16, sq.F32])
@pytest.mark.parametrize("M,experts,top,ff,shared,K", [(16, 448, 28, 64, 0, 4096), (16, 1024, 64, 64, 64, 4096), (8, 600, 64, 64, 128, 4096), (16, 600, 64, 64, 704, 2048),
                                                       (3, 9, 2, 128, 64, 1024), (5, 9, 3, 576, 0, 1024), (11, 40, 7, 64, 0, 512), (16, 70, 5, 576, 576, 256)])
def test_long_lists_and_short_ones(dev, M, experts, top, ff, shared, K, dtype):
    few_rows_against_64_bits(dev, M, experts, top, ff, shared, K, dtype)


@pytest.mark.parametrize("dtype", [sq.BF16, sq.F32])
@pytest.mark.parametrize("M,K", [(4, 192), (8, 2048), (9, 4160), (16, 2048)])
def test_rows_beside_rows_that_are_not_finite(dev, M, K, dtype):
    """Rows of infinities and of no numbers that chose the same experts: every other row has the bits that it has beside finite ones."""
    import torch

    lib, experts, top, ff, shared = sq.load(), 5, 3, 192, 64
    T = torch.float32 if dtype == sq.F32 else torch.bfloat16
    torch.manual_seed(M)
    laid = [(torch.randn(n, device=dev) * k ** -0.5).bfloat16() for n, k in ((experts * ff * K, K), (experts * K * ff, ff), (shared * K, K), (K * shared, shared))]
    logits, h, x = torch.randn(M, 16, device=dev), torch.randn(M, K, device=dev).to(T), torch.randn(M, K, device=dev)
    logits[:, 1] = 9.0
    size = lib.llam_seq_experts_scratch_bytes(M, experts, top, ff, shared, K)
    bad, got = [1, M - 1], []
    for value in (None, float("inf"), float("nan")):
        rows, y = h.clone(), x.clone()
        if value is not None:
            rows[bad[0], 0], rows[bad[1], 3] = value, -value
        scratch = torch.full((size,), 255, dtype=torch.uint8, device=dev)
        a = sq.ExpertsArgs(d_logits=logits.data_ptr(), ldz=16, d_up=laid[0].data_ptr(), d_down=laid[1].data_ptr(), up_stride=ff * K, down_stride=ff * K,
                           experts=experts, top=top, ff=ff, shared_ff=shared, K=K, N=K, d_h=rows.data_ptr(), d_x=y.data_ptr(), ldx=K,
                           d_shared_up=laid[2].data_ptr(), d_shared_down=laid[3].data_ptr())
        assert lib.llam_seq_experts(ctypes.byref(a), M, scratch.data_ptr(), size, dtype, 0, torch.cuda.current_stream().cuda_stream), lib.llam_ql_last_error()
        torch.cuda.synchronize()
        got.append(y)
    good = [m for m in range(M) if m not in bad]
    for y in got[1:]:
        assert torch.equal(y[good], got[0][good]) and torch.isfinite(y[good]).all()
    assert not torch.isfinite(got[1][bad]).any()  # (of sums that are no numbers max(z, 0) is 0)


def few_rows_against_64_bits(dev, M, experts, top, ff, shared, K, dtype):
    import torch

    T = torch.float32 if dtype == sq.F32 else torch.bfloat16
    torch.manual_seed(M + experts)
    tiled = lambda w: w.reshape(w.shape[0], w.shape[1] // 16, 16, w.shape[2] // 32, 4, 8).permute(0, 1, 3, 4, 2, 5).contiguous()  # noqa: E731
    matrix = lambda n, rows, k: (torch.randn(n, rows, k, device=dev) * k ** -0.5).bfloat16()  # noqa: E731
    up, down = matrix(experts, ff, K), matrix(experts, K, ff)
    both = [matrix(1, max(shared, 64), K), matrix(1, K, max(shared, 64))]
    logits, h, x = torch.randn(M, experts + 16, device=dev), torch.randn(M, K, device=dev).to(T), torch.randn(M, K, device=dev)
    want = x.double()
    weights, ids = logits[:, :experts].double().topk(top, 1)
    weights = torch.softmax(weights, 1)

    def part(m, u, d):
        return d.double() @ torch.relu(u.double() @ h[m].double()).square().to(T).double()

    for m in range(M):
        for j in range(top):
            want[m] += weights[m, j] * part(m, up[ids[m, j]], down[ids[m, j]])
        if shared:
            want[m] += torch.sigmoid(logits[m, experts].double()) * part(m, both[0][0], both[1][0])
    lib, laid = sq.load(), [tiled(w) for w in (up, down, *both)]
    size = lib.llam_seq_experts_scratch_bytes(M, experts, top, ff, shared, K)
    scratch = torch.full((size + 64,), 255, dtype=torch.uint8, device=dev)
    a = sq.ExpertsArgs(d_logits=logits.data_ptr(), ldz=experts + 16, d_up=laid[0].data_ptr(), d_down=laid[1].data_ptr(), up_stride=ff * K,
                       down_stride=ff * K, experts=experts, top=top, ff=ff, shared_ff=shared, K=K, N=K, d_h=h.data_ptr(), d_x=x.data_ptr(), ldx=K)
    if shared:
        a.d_shared_up, a.d_shared_down = laid[2].data_ptr(), laid[3].data_ptr()
    assert lib.llam_seq_experts(ctypes.byref(a), M, scratch.data_ptr(), size, dtype, 0, torch.cuda.current_stream().cuda_stream), lib.llam_ql_last_error()
    torch.cuda.synchronize()
    assert (scratch[size:] == 255).all()
    # fp32: sums of up to K products, 2^-24 each.  bf16: the square of a sum whose rounding may fall to the other side, 2^-8 of few of the ff values
    assert (x.double() - want).norm() / (want.norm()) < (2e-6 if dtype == sq.F32 else 2e-3)


# rows, experts, of a row, width of an expert, of the model, slope of the logits: few rows; more than 64 experts, evenly and
# mostly the first ones chosen, many without a row; groups of several tiles with a last one of few rows, of all rows; each tile
# (test_launch_rules.py)
@pytest.mark.parametrize("dtype", [sq.BF16, sq.F32])
@pytest.mark.parametrize("M,experts,top,ff,K,slope", [(17, 8, 2, 64, 320, 0.0), (40, 130, 3, 192, 256, 0.0), (300, 150, 4, 192, 128, 0.2),
                                                      (300, 64, 6, 320, 192, 0.0), (700, 3, 2, 320, 128, 0.5), (260, 5, 1, 64, 64, 9.0),
                                                      (500, 40, 3, 2048, 64, 0.1), (400, 20, 3, 64, 1088, 0.0),
                                                      (200, 12, 2, 2688, 64, 0.2), (1200, 2, 2, 2368, 64, 0.0), (700, 4, 2, 1024, 1088, 0.5),
                                                      (1500, 3, 3, 4096, 64, 0.0)])
def test_rows_grouped_by_expert(dev, M, experts, top, ff, K, slope, dtype):
    import torch

    T = torch.float32 if dtype == sq.F32 else torch.bfloat16
    torch.manual_seed(M + experts)
    up, down = torch.randn(experts, ff, K, device=dev) * K ** -0.5, torch.randn(experts, K, ff, device=dev) * ff ** -0.5
    up, down = up.bfloat16(), down.bfloat16()
    lay = lambda w: w.reshape(experts, w.shape[1] // 16, 16, w.shape[2] // 32, 4, 8).permute(0, 1, 3, 4, 2, 5).contiguous()
    up_laid, down_laid = lay(up), lay(down)
    logits = torch.randn(M, experts + 16, device=dev)
    logits[:, :experts] -= slope * torch.arange(experts, device=dev)
    h, base = torch.randn(M, K, device=dev).to(T), torch.randn(M, K, device=dev)
    x, lib = base.clone(), sq.load()
    size = lib.llam_seq_experts_scratch_bytes(M, experts, top, ff, 0, K)
    scratch = torch.full((size,), 255, dtype=torch.uint8, device=dev)
    a = sq.ExpertsArgs(d_logits=logits.data_ptr(), ldz=experts + 16, d_up=up_laid.data_ptr(), d_down=down_laid.data_ptr(), up_stride=ff * K,
                       down_stride=ff * K, experts=experts, top=top, ff=ff, K=K, N=K, d_h=h.data_ptr(), d_x=x.data_ptr(), ldx=K)
    assert lib.llam_seq_experts(ctypes.byref(a), M, scratch.data_ptr(), size, dtype, 0, torch.cuda.current_stream().cuda_stream), lib.llam_ql_last_error()
    torch.cuda.synchronize()
    chosen, ids = logits[:, :experts].double().topk(top, 1)
    weights = torch.softmax(chosen, 1)
    want, bound, unit = base.double(), 2.0 ** -21 * base.double().abs(), 2.0 ** -23
    for e in range(experts):
        rows, at = (ids == e).nonzero(as_tuple=True)
        if not len(rows):
            continue
        u, d, r = up[e].double(), down[e].double(), h[rows].double()
        s = r @ u.T
        off = (K + 1) * unit * (r.abs() @ u.abs().T)            # sums of K products in 32 bits, in any order
        act = torch.relu(s) ** 2
        off = 2 * s.abs() * off + off ** 2 + (2.0 ** -8 if dtype == sq.BF16 else unit) * act   # squared, rounded to T
        w = weights[rows, at].unsqueeze(1)
        want.index_add_(0, rows, w * (act @ d.T))
        bound.index_add_(0, rows, 1.01 * w * ((off + (ff + 16) * unit * act) @ d.abs().T))   # (16: the weight and the sum of choices)
    assert ((x.double() - want).abs() <= bound).all()
