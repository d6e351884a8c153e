"""Row operators of sequence models by themselves: at the edges of what a thread, a workgroup or a wavefront holds."""
import ctypes

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


@pytest.mark.parametrize("M,top,experts", [(17, 1, 3), (500, 2, 7), (1820, 9, 40), (1821, 9, 40), (4000, 9, 40)])
def test_experts_of_many_tokens(torch, lib, dev, M, top, experts):
    """(token, choice) pairs by their expert: up to 16384 of them are held at once, more are not."""
    W = 64
    rng = np.random.default_rng(M)
    h, z = rng.standard_normal((M, W)).astype(np.float32), rng.standard_normal((M, experts)).astype(np.float32)
    up, down = (torch.from_numpy(rng.standard_normal((experts, W, W)).astype(np.float32) / 8).bfloat16() for _ in range(2))
    tiles = [torch.from_numpy(np.stack([sequence.tiled(m) for m in w.view(torch.uint16).numpy()]).view(np.int16)).to(dev) for w in (up, down)]
    hd, zd, x = torch.from_numpy(h).to(dev), torch.from_numpy(z).to(dev), torch.zeros((M, W), device=dev)
    a = sequence.ExpertsArgs()
    a.d_logits, a.ldz, a.d_up, a.d_down, a.up_stride, a.down_stride = zd.data_ptr(), experts, tiles[0].data_ptr(), tiles[1].data_ptr(), W * W, W * W
    a.experts, a.top, a.ff, a.shared_ff, a.K, a.N, a.d_h, a.d_x, a.ldx = experts, top, W, 0, W, W, hd.data_ptr(), x.data_ptr(), W
    size = lib.llam_seq_experts_scratch_bytes(M, experts, top, W, 0, W)
    scratch = torch.zeros(size, dtype=torch.uint8, device=dev)
    assert lib.llam_seq_experts(ctypes.byref(a), M, scratch.data_ptr(), size, sequence.F32, 0, None), lib.llam_ql_last_error()
    torch.cuda.synchronize()
    chosen = np.argsort(-z, axis=1, kind="stable")[:, :top]
    w = np.exp(np.take_along_axis(z, chosen, 1).astype(np.float64))
    w /= w.sum(1, keepdims=True)
    u, d = up.double().numpy(), down.double().numpy()
    want, size = np.zeros((M, W)), np.zeros((M, W))
    for e in range(experts):
        t, c = np.nonzero(chosen == e)
        y = np.maximum(h[t].astype(np.float64) @ u[e].T, 0) ** 2
        want[t] += w[t, c][:, None] * (y @ d[e].T)
        size[t] += w[t, c][:, None] * ((np.abs(h[t]) @ np.abs(u[e]).T) ** 2 @ np.abs(d[e]).T)
    # two products of 64 terms, the first squared, and a sum of the choices, all in 32 bits
    assert (np.abs(x.cpu().numpy() - want) <= size * (3 * 64 + top + 16) * 2.0 ** -24).all()


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("rank,tokens,length", [(64, 1, 129), (64, 1, 1024), (64, 1, 1025), (512, 1, 1024), (512, 70, 100), (128, 40, 511),
                                                (128, 40, 513), (576, 300, 330), (192, 1, 2000)])
def test_latent_attention_merged_from_stretches(torch, lib, dev, rank, tokens, length, dtype):
    """Two to sixteen stretches of a sequence: up to eight are merged by a wavefront a row, more by a workgroup."""
    heads = 16
    rng = np.random.default_rng(length)
    kind = torch.float32 if dtype == sequence.F32 else torch.bfloat16
    q, cache = (torch.from_numpy(rng.standard_normal(s).astype(np.float32)).to(kind) for s in ((tokens * heads, rank), (2, length, rank)))
    qd, cd, out = q.to(dev), cache.to(dev), torch.zeros((tokens * heads, rank), dtype=kind, device=dev)
    where = [torch.tensor([v], dtype=torch.int32, device=dev) for v in (0, tokens, 1, length - tokens)]
    e = sequence.Entries(*(t.data_ptr() for t in where))
    floats = lib.llam_seq_latent_scratch_floats(tokens, 2, heads, rank, length)
    scratch = torch.full((floats,), float("nan"), device=dev)
    scale = rank ** -0.5
    assert lib.llam_seq_latent_attention(qd.data_ptr(), cd.data_ptr(), ctypes.byref(e), 0, 1, tokens, length, heads, rank, length, scale,
                                         out.data_ptr(), scratch.data_ptr(), floats, dtype, 0, None), lib.llam_ql_last_error()
    torch.cuda.synchronize()
    k = cache[1].double().numpy()
    s = q.double().numpy().reshape(tokens, heads, rank) @ k.T * scale
    hidden = np.arange(length)[None, None] > (length - tokens + np.arange(tokens))[:, None, None]
    s = np.where(hidden, -np.inf, s)
    p = np.exp(s - s.max(-1, keepdims=True))
    want = (p / p.sum(-1, keepdims=True) @ k).reshape(tokens * heads, rank)
    # scores: `rank` products of size 0.64 scale added in 32 bits, the exponential's argument rounded; a weight's relative error is twice that;
    # bf16: weights in two pieces of 8 bits, the result rounded
    wrong = 2 * (0.64 * rank * scale * 32 + 8) * 2.0 ** -24 + (2.0 ** -16 if dtype != sequence.F32 else 0)
    bound = wrong * np.abs(k).max() + (np.abs(want) * 2.0 ** -8 if dtype != sequence.F32 else 0)
    assert (np.abs(out.float().cpu().numpy() - want) <= bound).all()


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("heads,kv,dim,vdim,rot,chunk,append", [(4, 2, 64, 64, 0, 0, True), (16, 1, 128, 128, 128, 0, True), (12, 4, 128, 64, 50, 100, True),
                                                                (6, 6, 256, 128, 254, 128, True), (34, 2, 64, 128, 64, 0, True),
                                                                (8, 2, 128, 256, 32, 0, False), (5, 1, 64, 64, 64, 60, False)])
def test_a_decoded_token_is_turned_by_its_attention(torch, lib, dev, heads, kv, dim, vdim, rot, chunk, append, dtype):
    """One launch or rotary_kernel before it: outputs and caches the same bits, at the edges of tiles, stretches and the ring."""
    n, ring = 6, 256
    positions = [0, 127, 128, 255, 200, 31] if not chunk else [0, 127, 128, 255, 256, 700]
    kind = torch.float32 if dtype == sequence.F32 else torch.bfloat16
    columns = heads * dim + kv * (dim + vdim)
    torch.manual_seed(heads)
    proj, turns = torch.randn(n, columns + 4, device=dev), torch.rand(max(rot // 2, 1), dtype=torch.float64, device=dev)
    caches = [torch.randn(n, kv, ring, d, device=dev).to(kind) for d in (dim, vdim)]
    slot = torch.tensor([3, 0, 5, 1, 2, 4], dtype=torch.int32, device=dev)
    pos, row, one = (torch.tensor(v, dtype=torch.int32, device=dev) for v in (positions, list(range(n)), [1] * n))
    e = sequence.Entries(row.data_ptr(), one.data_ptr(), slot.data_ptr(), pos.data_ptr())
    floats = lib.llam_seq_attention_scratch_floats(vdim)
    got = []
    for together in (False, True):
        k, v = (c.clone() for c in caches)
        q, o = torch.zeros(n, heads * dim, dtype=kind, device=dev), torch.zeros(n, heads * vdim, dtype=kind, device=dev)
        scratch = torch.full((floats,), float("nan"), device=dev)
        a = sequence.AttentionArgs(heads, kv, dim, vdim, ring, chunk, dim ** -0.5, k.data_ptr(), v.data_ptr())
        end = (max(positions) + 1, o.data_ptr(), heads * vdim, scratch.data_ptr(), floats, dtype, 0, None)
        if together:
            assert lib.llam_seq_attention_decode(ctypes.byref(a), proj.data_ptr(), columns + 4, append, turns.data_ptr(), rot, ctypes.byref(e),
                                                 slot.data_ptr(), pos.data_ptr(), n, end[0], q.data_ptr(), *end[1:]), lib.llam_ql_last_error()
        else:
            assert lib.llam_seq_rotary(ctypes.byref(a), proj.data_ptr(), columns + 4, append, turns.data_ptr(), rot, slot.data_ptr(), pos.data_ptr(),
                                       q.data_ptr(), n, dtype, 0, None)
            assert lib.llam_seq_attention(ctypes.byref(a), q.data_ptr(), ctypes.byref(e), 0, n, 1, *end), lib.llam_ql_last_error()
        torch.cuda.synchronize()
        got.append((o, k, v))
    assert torch.isfinite(got[0][0].float()).all()
    assert all(torch.equal(x, y) for x, y in zip(*got))
