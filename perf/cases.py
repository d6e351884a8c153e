"""The work that a user has this package do, as cases that can be timed and checked.

Six kinds of pass, each through the public entry points:

  gemv      one projection of a decode step, fp32 rows in and out (capi.gemv_f32)
  gemm      one projection of a prompt: quantise the rows, multiply (capi.quantize_q8_1, capi.gemm)
  moe       the routed feed-forward of some tokens (capi.moe_*), per slot or grouped by expert
  dense     one greedy step of the quantized dense decoder (decoder.DenseDecoder), as a replayed graph
  prompt    a prompt through a sequence model (engine.Engine.feed), the logits of its last token
  serve     several prompts at once, a burst of greedy decoding, the logits after it (SequenceModel)

``listed`` holds the sizes of this repository's benchmark and ragged ones beside them; ``draw`` takes any
sizes of the same ranges.
"""
import math
import re
from pathlib import Path

import torch

from llaminar_amd import capi, synth
from llaminar_amd import sequence as sq
from llaminar_amd.decoder import DenseDecoder, Shape
from llaminar_amd.engine import Engine

DEVICE = "cuda:0"
FORMATS = capi.FORMATS
BLOCK_BYTES = {"q4_k": 144, "q6_k": 210, "iq3_s": 110}
VOCAB = 32768
TOP = 8  # routed experts of a token in the "moe" cases; one more is always on

# Sizes of the sequence models by family and width (those of bench.py --workload sequence).
SEQUENCE = {
    2048: dict(ff=8192, moe=(64, 6, 1408, 2816), latent=(16, 128, 128, 768, 512), memory=(4, 256, 512),
               attention=(16, 4, 128, 128), delta=(16, 8, 128, 128)),
    5120: dict(ff=25600, moe=(64, 6, 1536, 3072), latent=(64, 128, 128, 1536, 512), memory=(8, 256, 512),
               attention=(40, 8, 128, 128), delta=(40, 20, 128, 128)),
}
DENSE = {2048: dict(hidden=2048, n_heads=32, n_kv=4, ffn=8192), 5120: dict(hidden=5120, n_heads=64, n_kv=8, ffn=25600)}
EPS = 1e-5


def listed():
    return [
        # decoding one sequence: the gate or up projection of a 27B/32B-class decoder layer, the smallest call
        dict(name="gemv_q4_k_1x25600x5120", kind="gemv", fmt="q4_k", M=1, N=25600, K=5120),
        # a prompt of 512 tokens through that projection
        dict(name="gemm_q4_k_512x25600x5120", kind="gemm", fmt="q4_k", M=512, N=25600, K=5120),
        # a ragged prompt through the down projection: long rows, few of them
        dict(name="gemm_q6_k_199x5120x25600", kind="gemm", fmt="q6_k", M=199, N=5120, K=25600),
        # a short prompt, or drafted tokens being checked, in the smallest format
        dict(name="gemm_iq3_s_40x8192x5120", kind="gemm", fmt="iq3_s", M=40, N=8192, K=5120),
        # decoding one token through 256 small experts: latency and launches
        dict(name="moe_iq3_s_1", kind="moe", fmt="iq3_s", tokens=1, hidden=2048, inter=512, experts=256),
        # a ragged prompt through them
        dict(name="moe_iq3_s_333", kind="moe", fmt="iq3_s", tokens=333, hidden=2048, inter=512, experts=256),
        # a decode step of the dense model at a filled cache, alone and for eight sequences at once
        dict(name="dense_1_ctx4096", kind="dense", width=5120, layers=4, batch=1, context=4096),
        dict(name="dense_8_ctx4096", kind="dense", width=5120, layers=4, batch=8, context=4096),
        # prompts as they are fed: one portion of 2048 tokens; the second is the largest call
        dict(name="prompt_kogilix_2048_w2048", kind="prompt", family="kogilix", width=2048, dtype="bfloat16", tokens=2048, portion=2048),
        dict(name="prompt_bosirax_2048_w5120", kind="prompt", family="bosirax", width=5120, dtype="bfloat16", tokens=2048, portion=2048),
        # serving: ragged prompts in one step, then greedy decoding; the second in 32-bit
        dict(name="serve_kogilix_8_w2048", kind="serve", family="kogilix", width=2048, dtype="bfloat16", batch=8, prompt=251, steps=32),
        dict(name="serve_bosirax_3_w2048_f32", kind="serve", family="bosirax", width=2048, dtype="float32", batch=3, prompt=187, steps=16),
    ]


def _log_int(rng, low, high):
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(("gemv", "gemm", "gemm", "moe", "moe", "dense", "prompt", "prompt", "serve"))
    fmt = rng.choice(sorted(FORMATS))
    if kind == "gemv":
        return dict(kind=kind, fmt=fmt, M=rng.randint(1, 8), N=_log_int(rng, 1000, 32768), K=256 * _log_int(rng, 4, 100))
    if kind == "gemm":
        N, K = _log_int(rng, 1000, 25600), 256 * _log_int(rng, 4, 100)
        return dict(kind=kind, fmt=fmt, M=_log_int(rng, 9, max(9, min(2048, 512 * 25600 * 5120 // (N * K)))), N=N, K=K)
    if kind == "moe":
        return dict(kind=kind, fmt=fmt, tokens=_log_int(rng, 1, 512), hidden=rng.choice((1024, 2048, 4096)),
                    inter=rng.choice((512, 768, 1024)), experts=rng.choice((64, 128, 256)))
    if kind == "dense":
        return dict(kind=kind, width=rng.choice(sorted(DENSE)), layers=rng.randint(1, 4), batch=rng.randint(1, 8),
                    context=_log_int(rng, 33, 8192))
    family, dtype = rng.choice(("bosirax", "kogilix")), rng.choice(("bfloat16", "bfloat16", "float32"))
    if kind == "prompt":
        width = 2048 if dtype == "float32" else rng.choice((2048, 5120))
        return dict(kind=kind, family=family, width=width, dtype=dtype, tokens=_log_int(rng, 17, 2048 if dtype == "bfloat16" else 500),
                    portion=rng.choice((512, 2048)))
    return dict(kind=kind, family=family, width=2048, dtype=dtype, batch=rng.randint(1, 8), prompt=_log_int(rng, 9, 251),
                steps=rng.randint(4, 32) if dtype == "bfloat16" else rng.randint(2, 8))


def _generator(seed, device=DEVICE):
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    return g


# ---- quantized matrices -----------------------------------------------------------------------------

def _blocks(fmt, n, k, g):
    """Raw super-blocks of an [n, k] matrix: every packed byte uniform, the fp16 scales uniform in [0.001, 0.02)."""
    w = torch.randint(0, 256, (n * (k // 256), BLOCK_BYTES[fmt]), dtype=torch.uint8, device=DEVICE, generator=g)
    for at in {"q4_k": (0, 2), "q6_k": (208,), "iq3_s": (0,)}[fmt]:
        d = torch.rand(w.shape[0], device=DEVICE, generator=g) * 0.019 + 0.001
        w[:, at:at + 2] = d.to(torch.float16).view(torch.uint8).reshape(-1, 2)
    return w.reshape(-1)


def _half(w, at):
    return w[:, at:at + 2].contiguous().view(torch.float16).double()


def _to_half(x):
    """To fp16 as the weight packer rounds: nearest for ordinary results, towards zero below them."""
    small = x.abs() < 2.0 ** -14
    return torch.where(small, torch.trunc(x * 2.0 ** 24) * 2.0 ** -24, x.to(torch.float16).to(x.dtype))


def _over(x, y):
    """x / y, rounded once (torch multiplies by the reciprocal of a plain number)."""
    return x / torch.full_like(x, y)


def _decode(fmt, raw, n, k):
    """[n, k] weights as the block products see them: (integers [n, k/32, 32], scales, minima [n, k/32]), in 64 bits."""
    w = raw.reshape(-1, BLOCK_BYTES[fmt])
    t = w.shape[0]
    if fmt == "q4_k":
        s = w[:, 4:16].int()
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).float()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).float()
        q = w[:, 16:].reshape(t, 4, 1, 32)
        ints = torch.cat([q & 15, q >> 4], 2).double()
        scales = _to_half(_half(w, 0).float() * sc).double()
        minima = _to_half(-_half(w, 2).float() * mn).double()
    elif fmt == "q6_k":
        ql, qh = w[:, :128].reshape(t, 2, 2, 32).int(), w[:, 128:192].reshape(t, 2, 1, 32).int()
        low = torch.stack([ql[:, :, 0] & 15, ql[:, :, 1] & 15, ql[:, :, 0] >> 4, ql[:, :, 1] >> 4], 2)
        shift = torch.tensor([0, 2, 4, 6], device=w.device).reshape(1, 1, 4, 1)
        q = (low | (((qh >> shift) & 3) << 4)) - 32
        sub = w[:, 192:208].view(torch.int8).reshape(t, 8, 2).float()
        top = sub.abs().amax(2, keepdim=True)
        f = torch.where(top > 0, torch.round(sub * 127.0 * 256.0 / (top * 32.0).clamp(min=1.0)), torch.zeros_like(sub)).int()
        product = q.reshape(t, 8, 2, 16) * f.reshape(t, 8, 2, 1) + 128
        wrapped = ((product + 32768) & 65535) - 32768
        ints = (((wrapped >> 8) + 128 & 255) - 128).reshape(t, 8, 32).double()
        scales = _to_half(_over(_half(w, 208).float() * top[:, :, 0] * 32.0, 127.0)).double()
        minima = torch.zeros_like(scales)
    else:
        text = (Path(__file__).resolve().parent.parent / "include" / "llaminar_amd" / "iq3s_grid.h").read_text()
        book = torch.tensor([int(v, 16) for v in re.findall(r"0x([0-9a-f]{8})u", text)[:512]], device=w.device)
        index = w[:, 2:66].reshape(t, 8, 8).long()
        bit = torch.arange(8, device=w.device)
        index = index | (((w[:, 66:74].reshape(t, 8, 1).long() >> bit) & 1) << 8)
        magnitude = ((book[index].unsqueeze(-1) >> (8 * torch.arange(4, device=w.device))) & 255).reshape(t, 8, 32).float()
        sign = ((w[:, 74:106].reshape(t, 8, 4, 1).int() >> bit) & 1).reshape(t, 8, 32)
        nib = torch.stack([w[:, 106:110] & 15, w[:, 106:110] >> 4], 2).reshape(t, 8).float()
        db = _half(w, 0).float() * (1.0 + 2.0 * nib)
        v = magnitude * (1.0 - 2.0 * sign) * db.unsqueeze(-1)
        scale = _over(v.abs().amax(2), 127.0)
        ints = torch.round(v * (1.0 / scale).unsqueeze(-1)).double()
        scales, minima = _to_half(scale).double(), torch.zeros_like(db).double()
    return ints.reshape(n, k // 32, 32), scales.reshape(n, k // 32), minima.reshape(n, k // 32)


def _quantised(x):
    """Rows as their Q8_1 blocks stand for them: (values [m, k], scale * sum [m, k/32]), in 64 bits."""
    b = x.float().reshape(x.shape[0], -1, 32)
    d = _over(b.abs().amax(2, keepdim=True), 127.0)
    q = torch.where(d > 0, torch.round(b * (1.0 / d)), torch.zeros_like(b)).clamp(-128, 127).double()
    d = d.to(torch.float16).double()
    return (q * d).reshape(x.shape), (q.sum(2) * d[:, :, 0])


def _product(fmt, raw, n, k, x):
    """Quantised rows times a quantised matrix, in 64 bits, some rows of the matrix at a time."""
    a, sums = _quantised(x)
    out, step, per = [], max(1, (1 << 26) // k), k // 256 * BLOCK_BYTES[fmt]
    for at in range(0, n, step):
        rows = min(step, n - at)
        ints, scales, minima = _decode(fmt, raw[at * per:(at + rows) * per], rows, k)
        out.append(a @ (ints * scales.unsqueeze(-1)).reshape(rows, k).T + sums @ minima.T)
    return torch.cat(out, 1)


def _silu(z):
    return z * torch.sigmoid(z)


# ---- gemv, gemm --------------------------------------------------------------------------------------

def _linear_inputs(case, seed):
    g = _generator(seed)
    return _blocks(case["fmt"], case["N"], case["K"], g), torch.randn(case["M"], case["K"], device=DEVICE, generator=g)


def _prepare_linear(case, seed):
    M, N, K, fmt = case["M"], case["N"], case["K"], FORMATS[case["fmt"]]
    raw, x = _linear_inputs(case, seed)
    return dict(case=case, fmt=fmt, w=capi.prepare_weights(fmt, raw, N, K), x=x, y=torch.empty(M, N, device=DEVICE),
                q8=torch.empty(M * (K // 32) * 36, dtype=torch.uint8, device=DEVICE))


def _run_gemv(s):
    c = s["case"]
    return capi.gemv_f32(s["fmt"], s["w"], s["x"], c["M"], c["N"], c["K"], out=s["y"], q8_scratch=s["q8"])


def _run_gemm(s):
    c = s["case"]
    capi.quantize_q8_1(s["x"], out=s["q8"])
    return capi.gemm(s["fmt"], s["w"], s["q8"], c["M"], c["N"], c["K"], out=s["y"])


# ---- moe ----------------------------------------------------------------------------------------------

def _moe_inputs(case, seed):
    g = _generator(seed)
    H, I, fmt = case["hidden"], case["inter"], case["fmt"]
    experts = [[_blocks(fmt, n, k, g) for n, k in ((I, H), (I, H), (H, I))] for _ in range(case["experts"] + 1)]
    # hidden rows as a norm leaves them for weights of this spread: gate and up of the size of one
    x = torch.randn(case["tokens"], H, device=DEVICE, generator=g) / (2.8 * H ** 0.5)
    logits = torch.randn(case["tokens"], case["experts"], device=DEVICE, generator=g)
    return experts, x, logits


def _prepare_moe(case, seed):
    T, H, I, E, fmt = case["tokens"], case["hidden"], case["inter"], case["experts"], FORMATS[case["fmt"]]
    experts, x, logits = _moe_inputs(case, seed)
    keep = [tuple(capi.prepare_weights(fmt, raw, n, k) for raw, (n, k) in zip(e, ((I, H), (I, H), (H, I)))) for e in experts]
    S = TOP + 1  # the last slot of every token is the expert that is always on
    empty = dict(dtype=torch.uint8, device=DEVICE)
    return dict(case=case, fmt=fmt, keep=keep, table=capi.expert_table(keep, DEVICE), x=x, logits=logits,
                ids=torch.full((T, S), E, dtype=torch.int32, device=DEVICE), weights=torch.ones(T, S, device=DEVICE),
                q8=torch.empty(T * (H // 32) * 36, **empty), q8_act=torch.empty(T * S * (I // 32) * 36, **empty),
                gate=torch.empty(T * S, I, device=DEVICE), up=torch.empty(T * S, I, device=DEVICE),
                group=torch.empty(int(capi.load().llam_ql_moe_group_bytes(T, S)), **empty),
                pairs=torch.empty(T * S, H, device=DEVICE), out=torch.empty(T, H, device=DEVICE))


def _run_moe(s):
    c, fmt, table, ids, weights = s["case"], s["fmt"], s["table"], s["ids"], s["weights"]
    T, H, I, E, S = c["tokens"], c["hidden"], c["inter"], c["experts"] + 1, TOP + 1
    if T * S < 432:  # from here on grouping by expert pays (bench.py)
        capi.moe_route_gate_up_swiglu(fmt, table, E, s["logits"], TOP, s["x"], ids, weights, I, q8_out=s["q8_act"],
                                      q8_hidden=s["q8"], scratch=(s["gate"], s["up"]))
        capi.moe_down(fmt, table, E, ids, weights, s["q8_act"], s["out"], T, S, H, I)
    else:
        capi.moe_route_quantize(s["logits"], TOP, s["x"], s["q8"], ids=ids, weights=weights)
        capi.moe_group(ids, E, group=s["group"])
        capi.moe_gate_up_grouped(fmt, table, E, s["group"], s["q8"], T, S, H, I, gate=s["gate"], up=s["up"])
        act = capi.swiglu_quantize(s["gate"], s["up"])
        capi.moe_down_grouped(fmt, table, E, s["group"], ids, weights, act, s["pairs"], s["out"], T, S, H, I)
    return s["out"], ids, weights


def _exact_moe(case, seed):
    T, H, I, fmt = case["tokens"], case["hidden"], case["inter"], case["fmt"]
    experts, x, logits = _moe_inputs(case, seed)
    p = torch.softmax(logits.double(), 1)
    weights, ids = p.topk(TOP, 1)
    weights = torch.cat([weights / weights.sum(1, keepdim=True), torch.ones(T, 1, device=DEVICE, dtype=torch.float64)], 1)
    ids = torch.cat([ids, torch.full((T, 1), case["experts"], device=DEVICE)], 1)
    out = torch.zeros(T, H, dtype=torch.float64, device=DEVICE)
    for e, (gate, up, down) in enumerate(experts):
        token, slot = (ids == e).nonzero(as_tuple=True)
        if len(token):
            act = _silu(_product(fmt, gate, I, H, x[token])) * _product(fmt, up, I, H, x[token])
            out.index_add_(0, token, _product(fmt, down, H, I, act) * weights[token, slot].unsqueeze(1))
    return out, None, weights


# ---- dense decoder --------------------------------------------------------------------------------------

def _dense_shape(case):
    return Shape(n_layers=case["layers"], vocab=VOCAB, **DENSE[case["width"]])


def _dense_state(case, seed):
    """Newest tokens and, per layer, the keys and values of the positions before them (position-major)."""
    s, B = _dense_shape(case), case["batch"]
    cap = -(-(case["context"] + 1) // 32) * 32
    g = _generator(seed + 7919)
    caches = [tuple(torch.randn(B, s.n_kv, cap, s.head_dim, device=DEVICE, generator=g).to(torch.float16) for _ in range(2))
              for _ in range(s.n_layers)]
    ids = torch.randint(0, s.vocab, (B,), generator=_generator(seed, "cpu")).numpy()
    return cap, caches, ids


def _prepare_dense(case, seed):
    shape, B = _dense_shape(case), case["batch"]
    cap, caches, ids = _dense_state(case, seed)
    dec = DenseDecoder(shape, B, cap, torch.device(DEVICE), seed=seed)
    for n, (k, v) in enumerate(caches):
        dec.buffer("kcache", n).copy_(capi.kcache_tiled(k))
        dec.buffer("vcache", n).copy_(capi.vcache_tiled(v))
    pos = [case["context"] - 1] * B
    dec.set_state(ids, pos)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        dec.step(stream)
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            dec.step(stream)
    torch.cuda.synchronize()
    logits, chosen = dec.buffer("logits"), dec.buffer("ids")
    logits.owner = chosen.owner = dec  # whose memory it is
    return dict(dec=dec, graph=graph, ids=ids, pos=pos, logits=logits, chosen=chosen)


def _run_dense(s):
    # (a sampler of the user's own sets the tokens; the step is the captured one)
    s["dec"].set_state(s["ids"], s["pos"])
    s["graph"].replay()
    return s["logits"], s["chosen"]


def _exact_dense(case, seed):
    shape, B = _dense_shape(case), case["batch"]
    cap, caches, ids = _dense_state(case, seed)
    dec = DenseDecoder(shape, B, cap, torch.device(DEVICE), seed=seed, keep_raw=True, batch_planes=False)
    raw, H, D, p = dec.raw, shape.hidden, shape.head_dim, case["context"] - 1
    G = shape.n_heads // shape.n_kv

    def norm(x, name):
        return x / torch.sqrt((x * x).mean(1, keepdim=True) + shape.rms_eps) * raw[name].double()

    def rotate(x):
        angle = p * float(shape.rope_theta) ** (-torch.arange(0, D, 2, dtype=torch.float64, device=DEVICE) / D)
        u, v = x[..., :D // 2], x[..., D // 2:]
        return torch.cat([u * angle.cos() - v * angle.sin(), v * angle.cos() + u * angle.sin()], -1)

    per = H // 256 * 144
    rows = torch.cat([raw["embed"][i * per:(i + 1) * per] for i in ids.tolist()]).reshape(-1, 144)
    s = rows[:, 4:16].int()
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
    q = rows[:, 16:].reshape(-1, 4, 1, 32)
    x = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
    x = (x * (_half(rows, 0) * sc).unsqueeze(-1) - (_half(rows, 2) * mn).unsqueeze(-1)).reshape(B, H)
    names = {name: ("q4_k" if fmt == FORMATS["q4_k"] else "q6_k", n, k) for name, n, k, fmt in shape.projections()}
    for n, (keys, values) in enumerate(caches):
        def project(name, a):
            fmt, rows, columns = names[name]
            return _product(fmt, raw[f"{n}.{name}"], rows, columns, a)

        h = norm(x, f"{n}.attn_norm")
        heads = rotate(project("wq", h).reshape(B, shape.n_kv, G, D))
        k, v = keys[:, :, :p + 1].double(), values[:, :, :p + 1].double()
        k[:, :, p] = rotate(project("wk", h).reshape(B, shape.n_kv, D)).to(torch.float16).double()
        v[:, :, p] = project("wv", h).reshape(B, shape.n_kv, D).to(torch.float16).double()
        weights = torch.softmax(heads @ k.transpose(2, 3).contiguous() * D ** -0.5, -1)
        x = x + project("wo", (weights @ v).reshape(B, -1))
        h = norm(x, f"{n}.ffn_norm")
        x = x + project("wdown", _silu(project("wgate", h)) * project("wup", h))
    return _product("q6_k", raw["lm_head"], shape.vocab, H, norm(x, "final_norm")), None


# ---- sequence models ------------------------------------------------------------------------------------

def _layers(family, width):
    z = SEQUENCE[width]

    def kogilix(mixer, ffn, kv_from=-1):
        w = sq.Layer(mixer=mixer, kv_from=kv_from, ffn=ffn)
        if mixer == sq.MIXER_LATENT_ATTENTION:
            w.heads, w.dim, w.vdim, w.q_rank, w.kv_rank = z["latent"]
        else:
            w.heads, w.dim, w.vdim = z["memory"]
        if ffn == sq.FFN_GATED:
            w.ff = z["ff"]
        else:
            w.experts, w.top, w.ff, w.shared_ff = z["moe"]
        return w

    def bosirax(mixer, kv_from=-1):
        w = sq.Layer(mixer=mixer, kv_from=kv_from, parallel=1, ffn=sq.FFN_GATED_CLAMP, ff=z["ff"], limit=7.0)
        w.heads, w.kv_heads, w.dim, w.vdim = z["attention" if mixer == sq.MIXER_ATTENTION else "delta"]
        w.chunk, w.taps = 8192, 4
        return w

    if family == "kogilix":
        return [kogilix(sq.MIXER_MATRIX_MEMORY, sq.FFN_GATED), kogilix(sq.MIXER_LATENT_ATTENTION, sq.FFN_EXPERTS),
                kogilix(sq.MIXER_MATRIX_MEMORY, sq.FFN_EXPERTS), kogilix(sq.MIXER_LATENT_ATTENTION, sq.FFN_GATED, kv_from=1)]
    return [bosirax(sq.MIXER_DELTA), bosirax(sq.MIXER_ATTENTION), bosirax(sq.MIXER_ATTENTION, kv_from=1), bosirax(sq.MIXER_DELTA)]


BUCKETS = 100003


def _tensors(model):
    return {t.data_ptr(): t for t in model.keep}


def _tiles(w, n, k):
    """[n, k] matrix -> the order of its matrix-unit tiles."""
    return w.reshape(n // 16, 16, k // 32, 4, 8).permute(0, 2, 3, 1, 4).reshape(-1)


def _untiled(t, n, k):
    return t.reshape(-1, n // 16, k // 32, 4, 16, 8).permute(0, 1, 4, 2, 3, 5).reshape(-1, n, k)


def _next_token(token):
    """The token that the head prefers after `token`: its row is that token's embedding, as sure as a trained model
    is of most tokens, so that greedy choices do not hang on the last bit of a sum."""
    return (token * 12345 + 6789) % VOCAB


def _model(case, seed, slots, cap, max_rows):
    layers = _layers(case["family"], case["width"])
    model = synth.sequence_model_torch(layers, case["width"], VOCAB, torch.device(DEVICE), slots=slots, cap=cap, max_rows=max_rows,
                                       dtype=case["dtype"], eps=EPS, seed=seed, pairs=BUCKETS if case["family"] == "bosirax" else 0)
    at = next(n for n, t in enumerate(model.keep) if t.shape == (VOCAB, case["width"]))
    embed, head = model.keep[at], model.keep[at + 1]   # made one after the other
    # (12345 and the vocabulary share no factor: every token is preferred after exactly one)
    # Experts: every token belongs to `top` of them, and its embedding points at their rows of the router, so that
    # the choice, too, is as clear as a trained router's.
    g = _generator(seed + 15485863)
    tensors = _tensors(model)
    for w in layers:
        if w.ffn == sq.FFN_EXPERTS:
            router = torch.randn(sq.pad_to(w.experts + 1, 16), case["width"], device=DEVICE, generator=g) * case["width"] ** -0.5
            router = router.to(torch.bfloat16)
            tensors[w.w_router].copy_(_tiles(router, *router.shape))
            own = torch.rand(VOCAB, w.experts, device=DEVICE, generator=g).topk(w.top, 1).indices
            embed += (12.0 * router[own].float().sum(1)).to(torch.bfloat16)
    rows = torch.empty_like(embed)
    rows[_next_token(torch.arange(VOCAB, device=DEVICE))] = embed
    head.copy_(_tiles(rows, VOCAB, case["width"]))
    torch.cuda.synchronize()
    return layers, model, embed, rows


def _prompts(case, seed):
    """Token lists, ragged: each prompt of a batch is a little shorter than the one before."""
    g = _generator(seed + 104729, "cpu")
    if case["kind"] == "prompt":
        lengths = [case["tokens"]]
    else:
        lengths = [max(2, case["prompt"] - 13 * b) for b in range(case["batch"])]
    return [torch.randint(0, VOCAB, (n,), generator=g).tolist() for n in lengths]


def _prepare_prompt(case, seed):
    prompts = _prompts(case, seed)
    _, model, _, _ = _model(case, seed, 1, case["tokens"], case["portion"])
    return dict(model=model, engine=Engine(model), prompt=prompts[0])


def _run_prompt(s):
    engine, prompt = s["engine"], s["prompt"]
    logits = engine.feed([("prompt", prompt, [len(prompt) - 1])])[0][0]
    engine.release("prompt")
    return logits


def _prepare_serve(case, seed):
    prompts = _prompts(case, seed)
    rows = sum(len(p) for p in prompts)
    _, model, _, _ = _model(case, seed, len(prompts), max(len(p) for p in prompts) + case["steps"] + 1, rows)
    return dict(model=model, prompts=prompts, steps=case["steps"])


def _run_serve(s):
    model, prompts, steps = s["model"], s["prompts"], s["steps"]
    slots, ends, at = list(range(len(prompts))), [], -1
    for p in prompts:
        at += len(p)
        ends.append(at)
    first = model.forward([(b, 0, p) for b, p in enumerate(prompts)], ends)
    chosen = [int(t) for t in first.argmax(1)]
    tokens = model.decode(slots, [len(p) for p in prompts], chosen, steps)
    last = model.forward([(b, len(p) + steps, [int(tokens[-1, b])]) for b, p in enumerate(prompts)], slots)
    return first, tokens, last


def _plain(case, seed, sequences, wanted):
    """Logits of the wanted places of some sequences, from the equations, in 64 bits; None where it would take long."""
    width = case["width"]
    longest = max(len(s) for s in sequences)
    layers, model, embed, head = _model(case, seed, 1, longest, longest)
    at, P, dev = _tensors(model), sq.P, DEVICE
    f64 = dict(dtype=torch.float64, device=dev)

    def matrices(pointer, n, k):
        return _untiled(at[pointer], sq.pad_to(n, 16), P(k))

    def times(x, pointer, n, k, w=None):
        """x W^T of an [n, k] matrix, some of its rows at a time."""
        w = matrices(pointer, n, k)[0] if w is None else w
        step = max(1, (1 << 27) // k)
        return torch.cat([x @ w[r:min(n, r + step)].double().T for r in range(0, n, step)], 1)

    def rms(x):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)

    def per_sequence(f, *arrays):
        out, row = [], 0
        for s in sequences:
            out.append(f(*[a[row:row + len(s)] for a in arrays]))
            row += len(s)
        return torch.cat(out)

    def attend(q, k, v, scale):  # [T, heads, .], one head at a time
        T = q.shape[0]
        mask = torch.full((T, T), -math.inf, **f64).triu(1)
        per = q.shape[1] // k.shape[1]
        return torch.stack([torch.softmax(q[:, h] @ k[:, h // per].T * scale + mask, 1) @ v[:, h // per] for h in range(q.shape[1])], 1)

    def latent(w, x):
        H, d, vd, qr, r = w.heads, w.dim, w.vdim, w.q_rank, w.kv_rank
        own = w.kv_from < 0
        y = times(rms(x), w.w_in, qr + (r if own else 0), width)
        if own:
            caches.append(rms(y[:, qr:]))
        c = caches[-1]
        q = times(rms(y[:, :qr]), w.w_uq, H * d, qr).reshape(-1, H, d)
        uk, uv = matrices(w.w_uk_t, r, d).double(), matrices(w.w_uv, vd, r).double()
        k = torch.stack([c @ uk[h] for h in range(H)], 1)
        v = torch.stack([c @ uv[h].T for h in range(H)], 1)
        return per_sequence(lambda *a: attend(*a, w.scale), q, k, v).reshape(len(x), -1)

    def memory(w, x):
        H, d, vd = w.heads, w.dim, w.vdim
        y = times(rms(x), w.w_in, 2 * H * (d + vd) + 2 * H, width)
        q, k, v, g, i, f = torch.split(y, [H * d, H * d, H * vd, H * vd, H, H], 1)
        q, k, v = q.reshape(-1, H, d) * d ** -0.5, k.reshape(-1, H, d), v.reshape(-1, H, vd)
        cap = w.gate_cap
        i = cap * torch.tanh((i + 2.0) / cap)
        f = torch.nn.functional.logsigmoid(cap * torch.tanh((f + 2.0) / cap))

        def walk(q, k, v, i, f):
            S, n, m = torch.zeros(H, d, vd, **f64), torch.zeros(H, d, **f64), torch.zeros(H, **f64)
            out = []
            for t in range(len(q)):
                new = torch.maximum(f[t] + m, i[t])
                keep, take = torch.exp(f[t] + m - new).reshape(H, 1), torch.exp(i[t] - new).reshape(H, 1) * k[t]
                S = S * keep.unsqueeze(2) + take.unsqueeze(2) * v[t].unsqueeze(1)
                n, m = n * keep + take, new
                out.append((q[t].unsqueeze(1) @ S)[:, 0] / (torch.maximum((n * q[t]).sum(1).abs(), torch.exp(-m)) + 1e-6).unsqueeze(1))
            return torch.stack(out)

        o = per_sequence(walk, q, k, v, i, f)
        return rms(o).reshape(len(x), -1) * torch.sigmoid(g)

    def grouped(w, x):
        H, G, d, vd = w.heads, w.kv_heads, w.dim, w.vdim
        own = w.kv_from < 0
        y = times(rms(x), w.w_in, H * d + (G * (d + vd) if own else 0), width)
        angle = positions.unsqueeze(1) * 10000.0 ** (-torch.arange(0, d, 2, **f64) / d)
        c, s = angle.cos().unsqueeze(1), angle.sin().unsqueeze(1)

        def rotate(z):
            u, v = z[..., :d // 2], z[..., d // 2:]
            return torch.cat([u * c - v * s, v * c + u * s], -1)

        if own:
            caches.append((rotate(y[:, H * d:(H + G) * d].reshape(-1, G, d)), y[:, (H + G) * d:].reshape(-1, G, vd)))
        k, v = caches[-1]
        return per_sequence(lambda *a: attend(*a, w.scale), rotate(y[:, :H * d].reshape(-1, H, d)), k, v).reshape(len(x), -1)

    def delta(w, x):
        H, G, d, vd, taps = w.heads, w.kv_heads, w.dim, w.vdim, w.taps
        y = times(rms(x), w.w_in, 2 * G * d + 2 * H * vd + 2 * H, width)
        conv, z, b, a = torch.split(y, [2 * G * d + H * vd, H * vd, H, H], 1)

        def convolve(z):
            back = torch.cat([torch.zeros(taps - 1, z.shape[1], **f64), z])
            return _silu(sum(0.5 * back[j:j + len(z)] for j in range(taps)))

        q, k, v = torch.split(per_sequence(convolve, conv), [G * d, G * d, H * vd], 1)
        unit = lambda u: u / torch.sqrt((u * u).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
        q = (unit(q.reshape(-1, G, d)) * d ** -0.5).repeat_interleave(H // G, 1)
        k, v = unit(k.reshape(-1, G, d)).repeat_interleave(H // G, 1), v.reshape(-1, H, vd)
        beta, decay = torch.sigmoid(b), torch.exp(-math.exp(-2.0) * torch.nn.functional.softplus(a - 1.0))

        def walk(q, k, v, decay, beta):
            S, out = torch.zeros(H, d, vd, **f64), []
            for t in range(len(q)):
                S = S * decay[t].reshape(H, 1, 1)
                u = beta[t].unsqueeze(1) * (v[t] - (k[t].unsqueeze(1) @ S)[:, 0])
                S = S + k[t].unsqueeze(2) * u.unsqueeze(1)
                out.append((q[t].unsqueeze(1) @ S)[:, 0])
            return torch.stack(out)

        return rms(per_sequence(walk, q, k, v, decay, beta)).reshape(len(x), -1) * _silu(z)

    def gate_up(w, x):
        y = matrices(w.w_up, 2 * w.ff, width)[0].reshape(w.ff // 16, 2, 16, width)
        return [times(rms(x), None, w.ff, width, y[:, n].reshape(w.ff, width)) for n in (0, 1)]

    def feed_forward(w, x):
        if w.ffn == sq.FFN_GATED:
            gate, up = gate_up(w, x)
            return times(torch.nn.functional.gelu(gate, approximate="tanh") * up, w.w_down, width, w.ff)
        h = rms(x)
        z = times(h, w.w_router, w.experts + 1, width)
        top, ids = z[:, :w.experts].topk(w.top, 1)
        weights = torch.softmax(top, 1)
        relu2 = lambda u: torch.relu(u) ** 2  # noqa: E731
        y = torch.sigmoid(z[:, w.experts:]) * times(relu2(times(h, w.w_shared_up, w.shared_ff, width)), w.w_shared_down, width, w.shared_ff)
        up, down = matrices(w.w_up, w.ff, width), matrices(w.w_down, width, w.ff)
        for e in range(w.experts):
            token, slot = (ids == e).nonzero(as_tuple=True)
            if len(token):
                a = relu2(h[token] @ up[e].double().T) @ down[e].double().T
                y.index_add_(0, token, a * weights[token, slot].unsqueeze(1))
        return y

    positions = torch.cat([torch.arange(len(s), **f64) for s in sequences])
    ids = torch.tensor([t for s in sequences for t in s], device=dev)
    x = embed[ids].double()
    if case["family"] == "bosirax":
        table = next(t for t in model.keep if t.shape == (BUCKETS + 1, width))
        pair = (torch.cat([ids[:1], ids[:-1]]) * 40503 + ids * 19) % BUCKETS
        x = x + table[torch.where(positions == 0, torch.full_like(pair, BUCKETS), pair)].double()
    caches = []
    mixers = {sq.MIXER_LATENT_ATTENTION: latent, sq.MIXER_MATRIX_MEMORY: memory, sq.MIXER_ATTENTION: grouped, sq.MIXER_DELTA: delta}
    for w in layers:
        y = mixers[w.mixer](w, x)
        if w.parallel:
            gate, up = gate_up(w, x)
            gate, up = gate.clamp(max=w.limit), up.clamp(-w.limit, w.limit)
            y = torch.cat([y, gate * torch.sigmoid(1.702 * gate) * (up + 1.0)], 1)
            x = x + times(y, w.w_out, width, y.shape[1])
        else:
            x = x + times(y, w.w_out, width, y.shape[1])
            x = x + feed_forward(w, x)
    model.close()
    rows, row = [], 0
    for s, places in zip(sequences, wanted):
        rows += [row + p for p in places]
        row += len(s)
    return rms(x[rows]) @ head.double().T


def _exact_prompt(case, seed):
    prompt = _prompts(case, seed)[0]
    return _plain(case, seed, [prompt], [[len(prompt) - 1]])[0]


def _exact_serve(case, seed):
    # every choice is the token that the head prefers after the one before
    sequences, wanted = [], []
    for p in _prompts(case, seed):
        s = list(p)
        for _ in range(case["steps"] + 1):
            s.append(_next_token(s[-1]))
        sequences.append(s)
        wanted.append([len(p) - 1, len(s) - 1])
    logits = _plain(case, seed, sequences, wanted)
    return logits[0::2], None, logits[1::2]


def _layer_work(w, width, rows):
    """(bytes of weights read once for `rows` tokens of a step, products of one token)."""
    if w.mixer == sq.MIXER_LATENT_ATTENTION:
        n = width * (w.q_rank + (w.kv_rank if w.kv_from < 0 else 0)) + w.heads * (w.dim * w.q_rank + (w.dim + w.vdim) * w.kv_rank + w.vdim * width)
    elif w.mixer == sq.MIXER_ATTENTION:
        n = width * (w.heads * (w.dim + w.vdim) + (w.kv_heads * (w.dim + w.vdim) if w.kv_from < 0 else 0))
    elif w.mixer == sq.MIXER_DELTA:
        n = width * (2 * w.kv_heads * w.dim + 3 * w.heads * w.vdim + 2 * w.heads)
    else:
        n = width * (2 * w.heads * w.dim + 3 * w.heads * w.vdim + 2 * w.heads)
    read = n
    if w.ffn == sq.FFN_EXPERTS:
        each, shared = 2 * width * w.ff, 2 * width * w.shared_ff + width * (w.experts + 1)
        n += w.top * each + shared
        read += w.experts * (1.0 - (1.0 - w.top / w.experts) ** rows) * each + shared
    else:
        n += 3 * width * w.ff
        read += 3 * width * w.ff
    return 2 * read, n


def _token_work(w, length):
    """(bytes, operations) of one token's mixing at the given length of its sequence."""
    if w.mixer == sq.MIXER_LATENT_ATTENTION:
        return 2 * length * w.kv_rank, 4 * length * w.heads * w.kv_rank
    if w.mixer == sq.MIXER_ATTENTION:
        return 2 * length * w.kv_heads * (w.dim + w.vdim), 2 * length * w.heads * (w.dim + w.vdim)
    return 8 * w.heads * w.dim * w.vdim, 6 * w.heads * w.dim * w.vdim


def _sequence_work(case):
    layers, width, prompts = _layers(case["family"], case["width"]), case["width"], _prompts(case, 0)
    lengths = [len(p) for p in prompts]
    portions = [sum(lengths)] if case["kind"] == "serve" else [min(case["portion"], lengths[0] - at) for at in range(0, lengths[0], case["portion"])]
    head = VOCAB * width
    nbytes, flops = 2 * head + 4 * VOCAB * len(lengths), 2 * head * len(lengths)
    for w in layers:
        for rows in portions:
            read, n = _layer_work(w, width, rows)
            nbytes += read
            flops += 2 * n * rows
        for length in lengths:  # a portion's mixing: its cache or state once, every token's sums
            nbytes += _token_work(w, length)[0]
            flops += length * _token_work(w, length / 2)[1]
    if case["kind"] == "serve":
        B, steps = len(lengths), case["steps"] + 1
        for w in layers:
            read, n = _layer_work(w, width, B)
            nbytes += steps * read
            flops += 2 * n * B * steps
            for length in lengths:
                b, f = _token_work(w, length + steps / 2)
                nbytes += steps * b
                flops += steps * f
        nbytes += steps * 2 * head + 4 * VOCAB * B
        flops += 2 * head * B * steps
    return dict(bytes=nbytes, flops=flops)


# ---- what is asked of this file -----------------------------------------------------------------------

def prepare(case, seed):
    return {"gemv": _prepare_linear, "gemm": _prepare_linear, "moe": _prepare_moe, "dense": _prepare_dense, "prompt": _prepare_prompt,
            "serve": _prepare_serve}[case["kind"]](case, seed) | {"kind": case["kind"]}


def run(state):
    return {"gemv": _run_gemv, "gemm": _run_gemm, "moe": _run_moe, "dense": _run_dense, "prompt": _run_prompt,
            "serve": _run_serve}[state["kind"]](state)


def exact(case, seed):
    if case["kind"] in ("gemv", "gemm"):
        raw, x = _linear_inputs(case, seed)
        return _product(case["fmt"], raw, case["N"], case["K"], x)
    return {"moe": _exact_moe, "dense": _exact_dense, "prompt": _exact_prompt, "serve": _exact_serve}[case["kind"]](case, seed)


def work(case):
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        M, N, K = case["M"], case["N"], case["K"]
        return dict(bytes=N * (K // 256) * BLOCK_BYTES[case["fmt"]] + 4 * M * (K + N), flops=2 * M * N * K)
    if kind == "moe":
        T, H, I, E = case["tokens"], case["hidden"], case["inter"], case["experts"]
        touched = 1 + E * (1.0 - (1.0 - TOP / E) ** T)
        per = 3 * I * (H // 256) * BLOCK_BYTES[case["fmt"]]
        return dict(bytes=touched * per + 4 * T * (2 * H + E), flops=2 * T * (TOP + 1) * 3 * I * H)
    if kind == "dense":
        s, B, ctx = _dense_shape(case), case["batch"], case["context"]
        per = {FORMATS["q4_k"]: 144, FORMATS["q6_k"]: 210}
        mats = [(n, k, f) for _, n, k, f in s.projections()] * s.n_layers + [(s.vocab, s.hidden, FORMATS["q6_k"])]
        kv = s.n_layers * B * 2 * s.n_kv * ctx * s.head_dim
        return dict(bytes=sum(n * (k // 256) * per[f] for n, k, f in mats) + 2 * kv + 4 * B * s.vocab,
                    flops=2 * B * sum(n * k for n, k, _ in mats) + 2 * kv * s.n_heads // s.n_kv)
    return _sequence_work(case)


def tolerance(case):
    # (about four times what the paths differ from 64-bit sums)
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        return {"rel": 2e-6}  # 32-bit sums of exact block products
    if kind == "moe":
        return {"rel": 3e-4, "max": 0.05, "differ": 0.001}  # an activation may round to the next of 255 values
    if kind == "dense":
        return {"rel": 2e-2, "max": 0.2, "differ": 0.01}    # the same, and all that follows from it through the layers
    if case["dtype"] == "float32":
        return {"rel": 2e-5, "differ": 0.01}
    return {"rel": 1.2e-2, "max": 0.1, "differ": 0.01}
