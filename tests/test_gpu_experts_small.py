"""Routed experts of 2 to 16 rows: the rows that share an expert are multiplied together, and each is what it is alone."""
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
