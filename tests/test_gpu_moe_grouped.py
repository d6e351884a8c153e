"""Grouped expert launches of larger batches (int8 matrix unit) against the per-slot launches, and the device-side
sort of their (token, slot) pairs at the ends of its range."""
import numpy as np
import pytest

from llaminar_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi(dev):
    from llaminar_amd import capi

    capi.load()
    return capi


# format, hidden, inter, routed experts, tokens, routed slots: tiles of 16 and 32 pairs; experts of one pair and
# of all tokens; rows of 1, 2, 3, 4, 8 and 16 super-blocks (of the longest in Q4_K, 32 pairs find no room)
CASES = [("iq3_s", 2048, 512, 64, 61, 8), ("iq3_s", 768, 256, 40, 73, 5), ("q4_k", 1024, 768, 16, 100, 4),
         ("q6_k", 512, 1024, 8, 150, 2), ("q4_k", 4096, 256, 4, 300, 1), ("iq3_s", 256, 4096, 3, 220, 2),
         ("q6_k", 2048, 512, 100, 64, 8), ("q4_k", 2048, 512, 32, 60, 8), ("q4_k", 256, 256, 1, 431, 1)]


@pytest.mark.parametrize("name,hidden,inter,routed,T,k", CASES)
def test_grouped_batches_against_slots(capi, dev, name, hidden, inter, routed, T, k):
    import torch

    fmt, E, S = capi.FORMATS[name], routed + 1, k + 1
    mats = [[capi.prepare_weights(fmt, synth.weights_torch(fmt, n, kk, 7 * e + j, dev), n, kk)
             for j, (n, kk) in enumerate(((inter, hidden), (inter, hidden), (hidden, inter)))] for e in range(min(E, 9))]
    table = capi.expert_table([mats[e % len(mats)] for e in range(E)], dev)
    if E > 3:
        table.view(torch.int64).view(E, 3)[2] = 0   # expert 2 lives elsewhere
    rng = np.random.default_rng(T)
    ids = np.stack([rng.permutation(max(routed, k))[:k] % routed for _ in range(T)]).astype(np.int32)
    ids = np.concatenate([ids, np.full((T, 1), routed, np.int32)], axis=1)   # the always-on expert: all tokens
    ids[5, 0], ids[7, :] = 9999, -1                                          # out of range; a token without experts
    idd = torch.from_numpy(ids).to(dev)
    w = torch.from_numpy(rng.random((T, S)).astype(np.float32)).to(dev)
    q8 = capi.quantize_q8_1(torch.from_numpy(synth.activations_numpy(T, hidden, 4) / hidden ** 0.5).to(dev))
    gate, up = (torch.full((T * S, inter), 3.0, device=dev) for _ in range(2))
    assert capi.load().llam_ql_moe_gate_up(fmt, table.data_ptr(), E, idd.data_ptr(), q8.data_ptr(), gate.data_ptr(), up.data_ptr(),
                                           T, S, hidden, inter, 0, None)
    group = capi.moe_group(idd, E)
    gate_g, up_g = (torch.full((T * S, inter), 3.0, device=dev) for _ in range(2))
    capi.moe_gate_up_grouped(fmt, table, E, group, q8, T, S, hidden, inter, gate=gate_g, up=up_g)
    torch.cuda.synchronize()

    def close(a, b, K):
        # sums of K / 32 exact block products, in another order for some row lengths: an addition is off by 2^-24 of a partial sum, which
        # is at most a few times the spread of the results
        assert torch.isfinite(a).all()
        if K // 256 in (2, 4, 8, 16):   # the blocks of such rows are added in the same order: the same bits
            assert torch.equal(a, b)
        assert float((a - b).abs().max()) <= (K // 32) * 2.0 ** -22 * float(b.abs().max())

    close(gate_g, gate, hidden)
    close(up_g, up, hidden)
    q8a = capi.swiglu_quantize(gate, up)
    pairs, base = torch.full((T * S, hidden), float("nan"), device=dev), torch.randn(T, hidden, device=dev)
    for accumulate in (False, True):
        out, out_g = base.clone(), base.clone()
        capi.moe_down(fmt, table, E, idd, w, q8a, out, T, S, hidden, inter, accumulate=accumulate)
        capi.moe_down_grouped(fmt, table, E, group, idd, w, q8a, pairs, out_g, T, S, hidden, inter, accumulate=accumulate)
        torch.cuda.synchronize()
        close(out_g, out, inter)
        assert torch.equal(out_g[7], base[7] if accumulate else torch.zeros_like(base[7]))


@pytest.mark.parametrize("T,S,E", [(1, 1, 1), (455, 9, 257), (4096, 1, 2048), (1, 4096, 3), (1024, 1, 2047), (63, 1, 64), (65, 1, 1), (999, 1, 1531)])
def test_pairs_sorted_by_expert(capi, dev, T, S, E):
    import torch

    ids = np.random.default_rng(E).integers(-2, E + 2, size=(T, S)).astype(np.int32)
    P = T * S
    g = capi.moe_group(torch.from_numpy(ids).to(dev), E)
    torch.cuda.synchronize()
    w = g.cpu().numpy().view(np.int32)
    flat = ids.reshape(-1)
    valid = np.flatnonzero((flat >= 0) & (flat < E))
    order = valid[np.argsort(flat[valid], kind="stable")]
    experts, begins = np.unique(flat[order], return_index=True)
    assert (int(w[0]), int(w[1])) == (len(experts), len(valid))
    assert np.array_equal(w[4:4 + len(experts)], experts)
    assert np.array_equal(w[4 + P:4 + P + len(experts) + 1], np.append(begins, len(valid)))
    assert np.array_equal(w[5 + 2 * P:5 + 2 * P + len(valid)], order)


@pytest.mark.parametrize("T,S,E", [(5, 3, 4), (64, 9, 257), (455, 9, 257), (4096, 1, 2048), (2, 2000, 3), (1023, 4, 1)])
def test_chunks_of_an_experts_pairs(capi, dev, T, S, E):
    """The units of work: every expert's run of pairs in stretches of two or four, in order."""
    import torch

    ids = np.random.default_rng(T).integers(-1, E + 1, size=(T, S)).astype(np.int32)
    P = T * S
    g = capi.moe_group(torch.from_numpy(ids).to(dev), E)
    torch.cuda.synchronize()
    w = g.cpu().numpy().view(np.int32)
    size = 4 if P >= 512 else 2
    counts = np.bincount(ids[(ids >= 0) & (ids < E)], minlength=E)
    want, begin = [], 0
    for e, n in enumerate(counts):
        want += [(e, begin + j, min(size, n - j)) for j in range(0, n, size)]
        begin += n
    assert (int(w[2]), int(w[3])) == (len(want), size)
    at = 5 + 3 * P
    got = np.stack([w[at + k * P:at + k * P + len(want)] for k in range(3)], 1)
    assert np.array_equal(got, np.array(want, np.int32).reshape(-1, 3))


@pytest.mark.parametrize("S,hidden,accumulate", [(1, 256, False), (10, 1280, False), (11, 256, True), (63, 1024, False), (70, 1280, True)])
def test_weighted_sums_of_a_tokens_slots(capi, dev, S, hidden, accumulate):
    """One to many slots, some without an expert (what lies in their rows is not a number), a token without any: the live slots one
    after the other, products and sums rounded to 32 bits, the same bits."""
    import torch

    T, E, inter, fmt = 7, 5, 256, capi.FORMATS["q4_k"]
    mats = [tuple(capi.prepare_weights(fmt, synth.weights_torch(fmt, n, k, 3 * e + j, dev), n, k)
                  for j, (n, k) in enumerate(((inter, hidden), (inter, hidden), (hidden, inter)))) for e in range(E)]
    table = capi.expert_table(mats, dev)
    table.view(torch.int64).view(E, 3)[3] = 0   # expert 3 lives elsewhere
    rng = np.random.default_rng(S)
    ids = rng.integers(-1, E + 1, size=(T, S)).astype(np.int32)
    ids[4] = -1
    idd, w = torch.from_numpy(ids).to(dev), torch.from_numpy(rng.standard_normal((T, S)).astype(np.float32)).to(dev)
    act = capi.quantize_q8_1(torch.from_numpy(synth.activations_numpy(T * S, inter, 9)).to(dev))
    pairs, base = torch.full((T * S, hidden), float("nan"), device=dev), torch.randn(T, hidden, device=dev)
    out = base.clone()
    capi.moe_down_grouped(fmt, table, E, capi.moe_group(idd, E), idd, w, act, pairs, out, T, S, hidden, inter, accumulate=accumulate)
    torch.cuda.synchronize()
    rows, weights, start = pairs.cpu().numpy().reshape(T, S, hidden), w.cpu().numpy(), base.cpu().numpy()
    for t in range(T):
        y = start[t] if accumulate else None
        for s in range(S):
            if 0 <= ids[t, s] < E and ids[t, s] != 3:
                v = weights[t, s] * rows[t, s]
                y = v if y is None else y + v
        assert np.array_equal(out[t].cpu().numpy(), np.zeros(hidden, np.float32) if y is None else y), t
