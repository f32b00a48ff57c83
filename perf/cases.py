"""What a user of this library has it do, as cases that can be timed and checked.

Every case goes through the public entry points (qwanto_amd.abi): the
synchronous host-pointer ABI that qwnrun drives, the device-pointer
extensions, and the resident decoder.  A case is a dict of plain values:

kind "gemm"     one projection over the host ABI (ctx.gemm): int8 tokens with
                their scales for the quantized formats, fp32 tokens for F16 and
                BF16 rows or where the device quantizes.
kind "mlp"      the MLP block of one decoded token, device pointers: RMSNorm +
                gate/up + SwiGLU in one launch, the down projection in a second.
kind "head"     the LM head of one decoded token, device pointers: final
                RMSNorm, logits, greedy id.
kind "kv"       a Q8 KV cache, device pointers: attention of one query token
                over the cached tokens; with fill, the cache is emptied and the
                whole prompt's K/V appended first.
kind "decode"   the resident decoder: position kept at `past` cached tokens,
                then `steps` forward steps, the logits of each.
kind "prefill"  the resident decoder emptied, then a whole prompt; the logits
                after its last token.
kind "verify"   the resident decoder at `past` cached tokens: a block of draft
                tokens, the logits after each, then back to `past`.

Models are random, with the value ranges of real checkpoints: block scales
and codes of normally distributed weights, attention logits spread enough for
the softmax to choose, norm weights around one, a few large activations.
"""
import math

import numpy as np
import torch

from qwanto_amd import abi

DEV = "cuda:0"


# ---- the cases ------------------------------------------------------------------

# Layer shapes of the two models the repository's benchmark decodes.
QWEN2_1P5B = dict(hidden=1536, inter=8960, heads=12, kv_heads=2, head_dim=128)
QWEN3_4B = dict(hidden=2560, inter=9728, heads=32, kv_heads=8, head_dim=128)
VOCAB = 151936


def listed():
    return [
        # the smallest call of the drop-in host: the key or value projection
        # of one token; all latency (launches, synchronisation, pinned copies)
        dict(name="host_kv_projection_q4_0", kind="gemm", dtype="q4_0", rows=256, cols=1536, batch=1, f32=False),
        # a prompt through the drop-in host's batched GEMM: many tokens, large
        # output rows back to the host
        dict(name="host_gate_77_tokens_hvsq2", kind="gemm", dtype="hvsq2", rows=9728, cols=2560, batch=77, f32=False),
        # the MLP of one decoded token, the two largest weight reads of a layer
        dict(name="mlp_token_hvsq2", kind="mlp", dtype="hvsq2", hidden=2560, inter=9728),
        # the LM head of one decoded token: the largest single weight read
        dict(name="head_token_f16", kind="head", dtype="f16", rows=VOCAB, cols=1536),
        # a short prompt's cache built and read once
        dict(name="kv_fill_333_tokens", kind="kv", heads=12, kv_heads=2, head_dim=128, tokens=333, fill=True),
        # decode attention over an ordinary and over a long context
        dict(name="attention_4096_tokens", kind="kv", heads=32, kv_heads=8, head_dim=128, tokens=4096, fill=False),
        dict(name="attention_32768_tokens", kind="kv", heads=32, kv_heads=8, head_dim=128, tokens=32768, fill=False),
        # greedy decode of the whole 1.5B-shaped model at a short context
        dict(name="decode_q4_0", kind="decode", dtype="q4_0", layers=28, vocab=VOCAB, max_ctx=512, past=40, steps=8,
             qk_norm=False, **QWEN2_1P5B),
        # decode steps deep into a long chat: the layers that read a long cache
        dict(name="decode_long_hvsq2", kind="decode", dtype="hvsq2", layers=2, vocab=32768, max_ctx=4096, past=3001,
             steps=4, qk_norm=True, **QWEN3_4B),
        # a long prompt (a document, a chat history) into a decoder with room to answer
        dict(name="prefill_1003_tokens_q4_0", kind="prefill", dtype="q4_0", layers=2, vocab=32768, max_ctx=2048,
             tokens=1003, qk_norm=False, **QWEN2_1P5B),
        # an ordinary prompt at a short context
        dict(name="prefill_333_tokens_hvsq2", kind="prefill", dtype="hvsq2", layers=2, vocab=32768, max_ctx=512,
             tokens=333, qk_norm=True, **QWEN3_4B),
        # speculative decoding: eight drafted tokens checked by the whole model
        dict(name="verify_8_tokens_q4_0", kind="verify", dtype="q4_0", layers=28, vocab=VOCAB, max_ctx=512, past=203,
             draft=8, qk_norm=False, **QWEN2_1P5B),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges the listed ones stand for: every dtype,
    projection sizes from a small model's to a 4B model's (odd ones in the host
    ABI, which takes any), 1 to 160 tokens a call, contexts of 1 to 32768
    tokens, head dims 64 and 128, prompts of 2 to 1200 tokens."""
    kind = rng.choice(["gemm", "gemm", "mlp", "head", "kv", "kv", "decode", "prefill", "prefill", "verify"])
    quant = rng.choice(["q4_0", "hvsq2"])
    if kind == "gemm":
        dtype = rng.choice(["q4_0", "hvsq2", "q4_0", "hvsq2", "f16", "bf16"])
        narrow = dtype in ("f16", "bf16")
        cols = _log_int(rng, 200, 9728)
        if rng.random() < 0.5:
            cols = max(256, cols // 256 * 256)
        return dict(kind=kind, dtype=dtype, rows=_log_int(rng, 100, 9728), cols=cols,
                    batch=rng.choice([1, _log_int(rng, 2, 16), _log_int(rng, 2, 160)]) if not narrow else
                    _log_int(rng, 1, 16), f32=narrow or rng.random() < 0.3)
    if kind == "mlp":
        return dict(kind=kind, dtype=quant, hidden=32 * rng.randint(8, 96), inter=32 * _log_int(rng, 16, 320))
    if kind == "head":
        return dict(kind=kind, dtype=rng.choice(["f16", "bf16"]), rows=_log_int(rng, 1000, VOCAB),
                    cols=32 * rng.randint(8, 80))
    if kind == "kv":
        kv = rng.choice([1, 2, 4, 8])
        return dict(kind=kind, heads=kv * rng.choice([1, 2, 4, 6, 8]), kv_heads=kv, head_dim=rng.choice([64, 128, 128]),
                    tokens=_log_int(rng, 1, 32768), fill=rng.random() < 0.2)
    kv = rng.choice([1, 2, 4, 8])
    hd = rng.choice([64, 128, 128])
    cfg = dict(kind=kind, dtype=quant, layers=rng.randint(1, 3), vocab=_log_int(rng, 1000, 32768),
               qk_norm=rng.random() < 0.5, hidden=256 * rng.randint(1, 10), inter=256 * _log_int(rng, 2, 38),
               heads=kv * rng.choice([1, 2, 4, 6]), kv_heads=kv, head_dim=hd)
    long = rng.random() < 0.5
    cfg["max_ctx"] = rng.choice([2048, 4096]) if long else rng.choice([512, 1024])
    if kind == "prefill":
        cfg["tokens"] = _log_int(rng, 2, 1200 if long else 500)
        # no dearer than the largest listed prompt
        while work(cfg)["flops"] > 3.8e11:
            cfg["tokens"] -= 16
    elif kind == "decode":
        cfg.update(past=_log_int(rng, 1, 2000 if long else 500), steps=rng.randint(1, 4))
    else:
        cfg.update(past=_log_int(rng, 1, 1500 if long else 480), draft=rng.randint(2, 16))
    return cfg


# ---- inputs ---------------------------------------------------------------------


def _gen(seed, salt):
    return torch.Generator(device=DEV).manual_seed(seed * 1000003 + salt)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)


def _activations(g, tokens, cols):
    """Normal activations with a few columns that are large in every token."""
    big = torch.where(torch.rand(cols, generator=g, device=DEV) < 0.005, 8.0, 1.0)
    return _normal(g, tokens, cols) * big


def _weights(g, dtype, rows, cols, std):
    """One matrix as its on-disk bytes ([rows][bytes per row] uint8, on the GPU)."""
    if dtype in ("f16", "bf16"):
        w = _normal(g, rows, cols) * std
        return w.to(torch.float16 if dtype == "f16" else torch.bfloat16).view(torch.uint8).reshape(rows, cols * 2)
    if dtype == "q4_0":
        # [fp16 d][16 bytes, element j and 16 + j ...]: codes of normal weights, d ~ the block's maximum / 8
        nb = (cols + 31) // 32
        out = torch.empty(rows, nb, 18, device=DEV, dtype=torch.uint8)
        d = (std * (0.26 + 0.04 * _normal(g, rows, nb))).abs().to(torch.float16)
        out[:, :, :2] = d.reshape(rows, nb, 1).view(torch.uint8)
        lo = (torch.randn(rows, nb, 16, generator=g, device=DEV, dtype=torch.float16) * 3.5 + 8.0).round_().clamp_(0, 15)
        hi = (torch.randn(rows, nb, 16, generator=g, device=DEV, dtype=torch.float16) * 3.5 + 8.0).round_().clamp_(0, 15)
        out[:, :, 2:] = lo.to(torch.uint8) | (hi.to(torch.uint8) << 4)
        return out.reshape(rows, nb * 18)
    # HyperVSQ-2: [fp16 d][fp16 m][4 bytes of octant multipliers][2][64 bytes of 2-bit codes]
    nb = (cols + 255) // 256
    out = torch.zeros(rows, nb, 74, device=DEV, dtype=torch.uint8)
    d = (std * (1.6 + 0.2 * _normal(g, rows, nb))).abs().to(torch.float16)
    m = (std * 0.05 * _normal(g, rows, nb)).to(torch.float16)
    out[:, :, 0:2] = d.reshape(rows, nb, 1).view(torch.uint8)
    out[:, :, 2:4] = m.reshape(rows, nb, 1).view(torch.uint8)
    s = torch.randint(3, 9, (rows, nb, 4, 2), generator=g, device=DEV, dtype=torch.uint8)
    out[:, :, 4:8] = s[..., 0] | (s[..., 1] << 4)
    c = torch.zeros(rows, nb, 64, device=DEV, dtype=torch.uint8)
    for i in range(4):
        # codes 0..3 (weights -1..2 in steps) with a mean of 1: zero-mean weights
        r = torch.rand(rows, nb, 64, generator=g, device=DEV, dtype=torch.float16)
        c |= ((r > 0.31).to(torch.uint8) + (r > 0.75).to(torch.uint8) + (r > 0.94).to(torch.uint8)) << (2 * i)
    out[:, :, 10:] = c
    return out.reshape(rows, nb * 74)


def _dense(raw, dtype, cols):
    """The weights those bytes stand for, float64 [rows][cols]."""
    rows = raw.shape[0]
    if dtype in ("f16", "bf16"):
        return raw.reshape(rows, cols, 2).view(torch.float16 if dtype == "f16" else torch.bfloat16).reshape(rows, cols).double()
    if dtype == "q4_0":
        b = raw.reshape(rows, -1, 18)
        d = b[:, :, :2].contiguous().view(torch.float16).double()
        byte = b[:, :, 2:]
        # element 2j is the low nibble of byte j, 2j + 1 the high one
        code = torch.stack((byte & 15, byte >> 4), dim=-1).reshape(rows, -1, 32)
        return ((code.double() - 8.0) * d).reshape(rows, -1)[:, :cols]
    b = raw.reshape(rows, -1, 74)
    d = b[:, :, 0:2].contiguous().view(torch.float16).double()
    m = b[:, :, 2:4].contiguous().view(torch.float16).double()
    s = torch.stack((b[:, :, 4:8] & 15, b[:, :, 4:8] >> 4), dim=-1).reshape(rows, -1, 8, 1).double()
    byte = b[:, :, 10:]
    code = torch.stack([(byte >> (2 * i)) & 3 for i in range(4)], dim=-1).reshape(rows, -1, 8, 32).double()
    w = (d / 8.0).unsqueeze(-1) * s * (code - 1.0) + m.unsqueeze(-1)
    return w.reshape(rows, -1)[:, :cols]


def _quantize(x):
    """The per-token int8 activations of fp32 x [tokens][cols], as the formats
    define them: (int8 values as float32, scales)."""
    x = x.float()
    amax = x.abs().amax(dim=1, keepdim=True)
    scale = torch.where(amax > 0, amax / torch.full_like(amax, 127.0), torch.ones_like(amax))
    return (x * (1.0 / scale)).clamp(-127.0, 127.0).round(), scale


def _q8_cache(x):
    """K or V [tokens][channels] as the Q8 cache holds it, in float64 (64-channel groups)."""
    t, c = x.shape
    pad = (-c) % 64
    g = torch.nn.functional.pad(x.float(), (0, pad)).reshape(t, -1, 64)
    amax = g.abs().amax(dim=2, keepdim=True)
    scale = torch.where(amax > 0, amax / torch.full_like(amax, 127.0), torch.ones_like(amax))
    q = (g / scale).clamp(-127.0, 127.0).round()
    return (q.double() * scale.double()).reshape(t, -1)[:, :c]


def _proj64(x, w):
    """y of the quantized projection with dense float64 weights w: x fp32 quantized per token."""
    q, s = _quantize(x)
    return (q.double() @ w.t()) * s.double()


class _State:
    """A context with its tensors, caches or decoder; closed with the state."""

    def __init__(self):
        self.ctx = abi.Context(abi.load(), device=0)
        self.dec = None

    def __del__(self):
        try:
            if self.dec is not None:
                self.dec.close()
            self.ctx.close()
        except Exception:
            pass


def _gemm_inputs(case, seed):
    g = _gen(seed, 1)
    raw = _weights(g, case["dtype"], case["rows"], case["cols"], 0.02)
    return raw, _activations(g, case["batch"], case["cols"])


def _mlp_inputs(case, seed):
    g = _gen(seed, 2)
    d, i = case["hidden"], case["inter"]
    ws = [_weights(g, case["dtype"], *shape, 0.02) for shape in ((i, d), (i, d), (d, i))]
    return ws, _activations(g, 1, d)[0].contiguous(), 1.0 + 0.2 * _normal(g, d)


def _head_inputs(case, seed):
    g = _gen(seed, 3)
    return (_weights(g, case["dtype"], case["rows"], case["cols"], 0.02), _activations(g, 1, case["cols"])[0].contiguous(),
            1.0 + 0.2 * _normal(g, case["cols"]))


def _kv_inputs(case, seed):
    g = _gen(seed, 4)
    t, c = case["tokens"], case["kv_heads"] * case["head_dim"]
    scale = 0.5 + 1.5 * torch.rand(c, generator=g, device=DEV)
    return _normal(g, t, c) * scale, _normal(g, t, c) * scale.flip(0), 1.5 * _normal(g, case["heads"] * case["head_dim"])


# sigma of each projection's weights: q and k large enough that the softmax
# chooses among the tokens, the others as in a trained model
STD = {"q": 0.035, "k": 0.035, "v": 0.03, "o": 0.03, "gate": 0.03, "up": 0.03, "down": 0.02}


def _model_shapes(case):
    d, i = case["hidden"], case["inter"]
    q, kv = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
    return {"q": (q, d), "k": (kv, d), "v": (kv, d), "o": (d, q), "gate": (i, d), "up": (i, d), "down": (d, i)}


def _model_layer(case, seed, layer):
    """One layer's raw matrices and norm weights (the same for prepare and exact)."""
    g = _gen(seed, 100 + layer)
    shapes = _model_shapes(case)
    # narrower inputs than 1536 get larger weights, so every width has outputs of one size
    raw = {p: _weights(g, case["dtype"], *shapes[p], STD[p] * math.sqrt(1536.0 / (shapes[p][1] if p != "down" else
                                                                                  shapes[p][1] / 5.8)))
           for p in shapes}
    d = case["hidden"]
    vec = {"input_norm": 1.0 + 0.2 * _normal(g, d), "post_norm": 1.0 + 0.2 * _normal(g, d)}
    if case["qk_norm"]:
        for n in ("q_norm", "k_norm"):
            vec[n] = 1.2 + 0.2 * _normal(g, case["head_dim"])
    return raw, vec


def _model_ends(case, seed):
    """The embedding (also the LM head), the final norm and the token ids."""
    g = _gen(seed, 99)
    # rows of several times what the layers add together: a value that a
    # rounding moves in one layer stays a small part of the logits
    embed = (6.0 * math.sqrt(case["layers"]) * _normal(g, case["vocab"], case["hidden"])).to(torch.float16)
    final = 1.0 + 0.2 * _normal(g, case["hidden"])
    n = case.get("past", 0) + case.get("steps", 0) + case.get("draft", 0) + case.get("tokens", 0)
    ids = torch.randint(0, case["vocab"], (n,), generator=g, device=DEV, dtype=torch.int32)
    return embed, final, ids


ROPE_THETA, EPS = 1.0e6, 1.0e-6


def _decoder(state, case, seed):
    layers = []
    for l in range(case["layers"]):
        raw, vec = _model_layer(case, seed, l)
        layers.append({**{p: w.reshape(-1).cpu().numpy() for p, w in raw.items()},
                       **{n: v.cpu().numpy() for n, v in vec.items()}})
    embed, final, ids = _model_ends(case, seed)
    cfg = dict(hidden=case["hidden"], intermediate=case["inter"], layers=case["layers"], heads=case["heads"],
               kv_heads=case["kv_heads"], head_dim=case["head_dim"], vocab=case["vocab"], max_ctx=case["max_ctx"],
               rope_theta=ROPE_THETA, rms_eps=EPS)
    model = {"cfg": cfg, "dtype": case["dtype"], "layers": layers, "embed": embed.cpu().numpy(),
             "final_norm": final.cpu().numpy()}
    state.dec = abi.ResidentDecoder(state.ctx, model)
    state.ids = ids.cpu().numpy()


def prepare(case, seed):
    st = _State()
    st.case, kind = case, case["kind"]
    if kind == "gemm":
        raw, x = _gemm_inputs(case, seed)
        data = raw.cpu().numpy()
        if case["dtype"] == "f16":
            data = data.view(np.float16)
        elif case["dtype"] == "bf16":
            data = data.view(np.uint16)
        st.h = st.ctx.upload(data, case["dtype"], case["rows"], case["cols"])
        if case["f32"]:
            st.x, st.scales = x.cpu().numpy(), None
        else:
            q, s = _quantize(x)
            st.x, st.scales = q.to(torch.int8).cpu().numpy(), s.reshape(-1).cpu().numpy()
    elif kind == "mlp":
        ws, st.x, st.norm = _mlp_inputs(case, seed)
        d, i = case["hidden"], case["inter"]
        hs = [st.ctx.upload(w.cpu().numpy(), case["dtype"], *shape) for w, shape in zip(ws, ((i, d), (i, d), (d, i)))]
        st.h = torch.empty(i, device=DEV)
        st.y = torch.empty(d, device=DEV)
        spare = torch.empty(i, device=DEV)
        st.reqs = [st.ctx.gemv_group_request(hs[:2], [st.h.data_ptr(), spare.data_ptr()], "rmsnorm", "swiglu",
                                             x_ptr=st.x.data_ptr(), norm_ptr=st.norm.data_ptr(), eps=EPS),
                   st.ctx.gemv_group_request(hs[2:], [st.y.data_ptr()], "f32", "store", x_ptr=st.h.data_ptr())]
        st.keep = (hs, spare)
    elif kind == "head":
        raw, st.x, st.norm = _head_inputs(case, seed)
        h = st.ctx.upload(raw.cpu().numpy(), case["dtype"], case["rows"], case["cols"])
        st.logits = torch.empty(case["rows"], device=DEV)
        st.best = torch.zeros(1, device=DEV, dtype=torch.int32)
        args = dict(input_mode="rmsnorm", output_mode="argmax", x_ptr=st.x.data_ptr(), norm_ptr=st.norm.data_ptr(), eps=EPS)
        probe, keep = st.ctx.gemv_group_request([h], [st.logits.data_ptr()], partials_ptr=16, **args)
        st.parts = st.ctx.gemv_group_partials(probe)
        st.partials = torch.zeros(st.parts, device=DEV, dtype=torch.int64)
        st.req = st.ctx.gemv_group_request([h], [st.logits.data_ptr()], partials_ptr=st.partials.data_ptr(), **args)
    elif kind == "kv":
        st.k, st.v, st.q = _kv_inputs(case, seed)
        st.cache = st.ctx.kv_create(case["tokens"], case["kv_heads"], case["head_dim"])
        st.ctx.kv_append_device(st.cache, st.k.data_ptr(), st.v.data_ptr(), case["tokens"])
        st.out = torch.empty(case["heads"] * case["head_dim"], device=DEV)
        need = st.ctx.attention_workspace_bytes(st.cache, case["heads"], case["tokens"] - 1)
        st.work = torch.empty(max(need, 16), device=DEV, dtype=torch.uint8)
        if not case["fill"]:
            torch.cuda.synchronize()
            st.k = st.v = None
    else:
        _decoder(st, case, seed)
        if "past" in case:
            st.dec.prefill(st.ids[:case["past"]], logits=False)
    torch.cuda.synchronize()
    return st


# ---- one pass -------------------------------------------------------------------


def run(st):
    case, ctx = st.case, st.ctx
    kind = case["kind"]
    if kind == "gemm":
        if st.scales is None:
            return ctx.gemm(st.h, st.x, case["rows"], case["cols"])
        if case["batch"] == 1:
            return ctx.gemm(st.h, st.x, case["rows"], case["cols"], scale=float(st.scales[0]), gemv=True)
        return ctx.gemm(st.h, st.x, case["rows"], case["cols"], scales=st.scales)
    if kind == "mlp":
        for req, _ in st.reqs:
            ctx.gemv_group_device(req)
        return st.h, st.y
    if kind == "head":
        ctx.gemv_group_device(st.req[0])
        ctx.argmax_device(st.partials.data_ptr(), st.parts, st.best.data_ptr())
        return st.logits, st.best
    if kind == "kv":
        n = case["tokens"]
        if case["fill"]:
            ctx.kv_reset(st.cache)
            ctx.kv_append_device(st.cache, st.k.data_ptr(), st.v.data_ptr(), n)
        ctx.kv_attention_device(st.cache, st.q.data_ptr(), st.out.data_ptr(), case["heads"], n - 1,
                                1.0 / math.sqrt(case["head_dim"]), st.work.data_ptr())
        return st.out
    dec = st.dec
    if kind == "prefill":
        dec.reset()
        return dec.prefill(st.ids)[0]
    past = case["past"]
    if kind == "decode":
        dec.truncate(past)
        return [dec.forward(int(t))[0] for t in st.ids[past:]]
    logits, _ = dec.verify(st.ids[past:])
    dec.truncate(past)
    return logits


# ---- work and tolerance ---------------------------------------------------------


def _row_bytes(dtype, cols):
    return {"q4_0": (cols + 31) // 32 * 18, "hvsq2": (cols + 255) // 256 * 74}.get(dtype, 2 * cols)


def work(case):
    kind = case["kind"]
    if kind == "gemm":
        n, k, m = case["rows"], case["cols"], case["batch"]
        return {"bytes": n * _row_bytes(case["dtype"], k) + m * k * (4 if case["f32"] else 1) + m * n * 4,
                "flops": 2 * m * n * k}
    if kind == "mlp":
        d, i = case["hidden"], case["inter"]
        return {"bytes": 2 * i * _row_bytes(case["dtype"], d) + d * _row_bytes(case["dtype"], i) + 4 * (3 * d + 2 * i),
                "flops": 6 * d * i}
    if kind == "head":
        return {"bytes": case["rows"] * (2 * case["cols"] + 4) + 8 * case["cols"], "flops": 2 * case["rows"] * case["cols"]}
    if kind == "kv":
        t, c, q = case["tokens"], case["kv_heads"] * case["head_dim"], case["heads"] * case["head_dim"]
        cache = 2 * t * (c + 4 * ((c + 63) // 64))
        return {"bytes": cache * (2 if case["fill"] else 1) + (8 * t * c if case["fill"] else 0) + 8 * q, "flops": 4 * t * q}
    shapes = _model_shapes(case)
    params = sum(n * k for n, k in shapes.values()) * case["layers"]
    weights = sum(n * _row_bytes(case["dtype"], k) for n, k in shapes.values()) * case["layers"]
    head = case["vocab"] * case["hidden"]
    q, c = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
    token = 2 * (c + 4 * ((c + 63) // 64)) * case["layers"]  # cache bytes of one token
    if kind == "prefill":
        t = case["tokens"]
        return {"bytes": weights + 2 * head + t * (token + 2 * case["hidden"]) + 4 * case["vocab"],
                "flops": 2 * t * params + 2 * head + 2 * t * t * q * case["layers"]}
    past, new = case["past"], case.get("steps", case.get("draft"))
    rounds = new if kind == "decode" else 1  # times the weights and the cache have to be read
    return {"bytes": rounds * (weights + 2 * head + past * token) + new * (token + 4 * case["vocab"]),
            "flops": new * (2 * params + 2 * head + 4 * past * q * case["layers"])}


def tolerance(case):
    """About four times the distance between two runs of the path whose fp32
    sums are ordered differently, or between it and the 64-bit result."""
    kind = case["kind"]
    if kind in ("gemm", "head"):
        # exact products (integer block sums), fp32 sums: 5e-8 seen for the
        # quantized rows, 2e-7 for F16 and BF16 ones
        return {"rel": 1e-6, "max": 8e-6}
    if kind == "kv":
        return {"rel": 2.5e-6, "max": 2e-5}  # 5.6e-7 and 3.4e-6 seen
    if kind == "mlp":
        # 2e-7 seen, and now and then one normalized value at a rounding
        # boundary that moves one int8 step (up to 0.2 of the values' rms)
        w = math.sqrt(min(case["hidden"], case["inter"]))
        return {"rel": 0.4 / w, "max": 2.0 / w}
    # Whole layers: values at rounding boundaries of the int8 activations and
    # cache entries move one step, and move others in what follows: 3e-3 to
    # 7e-3 seen for one to 28 layers, the largest differences 5x that
    return {"rel": 2.5e-2, "max": 0.12}


# ---- the same in 64 bits ----------------------------------------------------------


def _rms64(x, w):
    x = x.double()
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + EPS) * w.double()


def _attend64(q, k, v, heads, kv_heads, scale, first):
    """Causal attention in float64: q [new][heads][D] at positions first.., k/v [all][kv_heads][D]."""
    out = torch.empty_like(q)
    pos = torch.arange(k.shape[0], device=q.device)
    mask = pos[None, :] > (first + torch.arange(q.shape[0], device=q.device))[:, None]
    for h in range(heads):
        j = h * kv_heads // heads
        s = (q[:, h] @ k[:, j].t()) * scale
        out[:, h] = torch.softmax(s.masked_fill(mask, -math.inf), dim=1) @ v[:, j]
    return out


def _decoder64(case, seed):
    """The logits [tokens][vocab] after every token a pass feeds, in float64."""
    embed, final, ids = _model_ends(case, seed)
    t, h, j, dim = ids.numel(), case["heads"], case["kv_heads"], case["head_dim"]
    x = embed[ids.long()].double()
    half = dim // 2
    # the rotation angles are fp32 by definition
    inv = torch.from_numpy(np.power(np.float32(ROPE_THETA), (-2.0 * np.arange(half, dtype=np.float32) / np.float32(dim)))
                           .astype(np.float32)).to(DEV)
    ang = (torch.arange(t, device=DEV, dtype=torch.float32)[:, None] * inv[None, :]).double()
    cos, sin = ang.cos()[:, None, :], ang.sin()[:, None, :]

    def rope(z):
        a, b = z[..., :half], z[..., half:]
        return torch.cat((a * cos - b * sin, a * sin + b * cos), dim=-1)

    for l in range(case["layers"]):
        raw, vec = _model_layer(case, seed, l)
        shapes = _model_shapes(case)

        def proj(p, z):
            return _proj64(z, _dense(raw[p], case["dtype"], shapes[p][1]))

        n = _rms64(x, vec["input_norm"])
        q, k, v = proj("q", n).reshape(t, h, dim), proj("k", n).reshape(t, j, dim), proj("v", n)
        if case["qk_norm"]:
            q, k = _rms64(q, vec["q_norm"]), _rms64(k, vec["k_norm"])
        q, k = rope(q), rope(k).reshape(t, j * dim)
        k, v = _q8_cache(k).reshape(t, j, dim), _q8_cache(v).reshape(t, j, dim)
        a = _attend64(q, k, v, h, j, 1.0 / math.sqrt(dim), 0)
        x = x + proj("o", a.reshape(t, h * dim))
        n = _rms64(x, vec["post_norm"])
        g = proj("gate", n)
        x = x + proj("down", g / (1.0 + torch.exp(-g)) * proj("up", n))
    new = case.get("steps", case.get("draft", 1))
    z = _rms64(x[-new:], final)
    # the head in slices: the embedding in float64 is large
    return torch.cat([z @ e.double().t() for e in embed.split(16384)], dim=1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemm":
        raw, x = _gemm_inputs(case, seed)
        w = _dense(raw, case["dtype"], case["cols"])
        return _proj64(x, w) if case["dtype"] in ("q4_0", "hvsq2") else x.double() @ w.t()
    if kind == "mlp":
        ws, x, norm = _mlp_inputs(case, seed)
        w = [_dense(r, case["dtype"], c) for r, c in zip(ws, (case["hidden"], case["hidden"], case["inter"]))]
        n = _rms64(x[None, :], norm)
        g, u = _proj64(n, w[0]), _proj64(n, w[1])
        h = g / (1.0 + torch.exp(-g)) * u
        return h[0], _proj64(h, w[2])[0]
    if kind == "head":
        raw, x, norm = _head_inputs(case, seed)
        n = _rms64(x[None, :], norm)
        y = torch.cat([n @ _dense(r, case["dtype"], case["cols"]).t() for r in raw.split(16384)], dim=1)[0]
        return y, None
    if kind == "kv":
        k, v, q = _kv_inputs(case, seed)
        t, j, d = case["tokens"], case["kv_heads"], case["head_dim"]
        k, v = _q8_cache(k).reshape(t, j, d), _q8_cache(v).reshape(t, j, d)
        return _attend64(q.double().reshape(1, case["heads"], d), k, v, case["heads"], j, 1.0 / math.sqrt(d), t - 1).reshape(-1)
    logits = _decoder64(case, seed)
    if kind == "prefill":
        return logits[-1]
    return list(logits) if kind == "decode" else logits
