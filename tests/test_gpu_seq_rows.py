"""Row operators of sequence models by themselves: at the edges of what a thread, a workgroup or a wavefront holds."""

import numpy as np
import pytest

from llaminar_amd import sequence

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch(dev):
    import torch

    return torch


@pytest.fixture(scope="module")
def lib(torch):
    return sequence.load()


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("K", [8, 1032, 2048, 2056, 6144, 6152])
def test_norm_of_short_and_long_rows(torch, lib, dev, K, dtype):
    """Rows that a workgroup holds in registers (up to 2048 and 6144 columns) and longer ones; one norm or two; rows in any order."""
    M, ldx, real, eps = 5, K + 4, K - 3, 1e-3
    rng = np.random.default_rng(K)
    x, norms = rng.standard_normal((M, ldx)).astype(np.float32), rng.standard_normal((2, K)).astype(np.float32)
    order = rng.permutation(M).astype(np.int32)
    kind = torch.float32 if dtype == sequence.F32 else torch.bfloat16
    xd, nd, od = (torch.from_numpy(v).to(dev) for v in (x, norms, order))
    y = torch.zeros((3, M, K), dtype=kind, device=dev)
    assert lib.llam_seq_rmsnorm(xd.data_ptr(), ldx, od.data_ptr(), nd[0].data_ptr(), eps, real, y[0].data_ptr(), M, K, dtype, 0, None)
    assert lib.llam_seq_rmsnorm_pair(xd.data_ptr(), ldx, nd[0].data_ptr(), nd[1].data_ptr(), eps, real, y[1].data_ptr(), y[2].data_ptr(), M, K,
                                     dtype, 0, None)
    torch.cuda.synchronize()
    got = y.float().cpu().numpy().astype(np.float64)
    inv = 1 / np.sqrt((x[:, :K].astype(np.float64) ** 2).sum(1, keepdims=True) / real + eps)
    for n, (rows, norm) in enumerate(((order, norms[0]), (slice(None), norms[0]), (slice(None), norms[1]))):
        want = (x[:, :K] * inv * norm)[rows]
        # the sum: 32-bit additions, up to 24 in a thread and 9 above it; root, reciprocal, two products; then the type's rounding
        bound = np.abs(want) * (40 * 2.0 ** -24 + (2.0 ** -8 if dtype != sequence.F32 else 0))
        assert (np.abs(got[n] - want) <= bound + 1e-30).all(), n
