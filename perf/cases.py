"""The calls that programs make of this library, as cases for timing and comparison.

A case is a dict of plain values; `kind` says which part of the library it calls:

  moe        moe_ffn_forward (DeviceMoE.forward) on `layers` MoE layers, one call each, of `tokens` tokens: a
             decode step of 1 to 32 sequences (captured in a HIP graph, as a serving loop does), or a prefill
             chunk (eager calls). `zipf`: a router bias that sends most tokens to few experts.
  attention  one decode step's attention over a contiguous KV store: per layer the new token's keys and values
             are appended and every query head attends the whole context (device positions, one HIP graph).
  model      one greedy decode step of a whole model (vireo_model_step_pos): `layers` blocks of attention over
             `context` tokens and an MoE FFN, the LM head and the argmax (one HIP graph).
  matvec     gguf_matmul (qmatvec_async) of one input with `count` matrices of `rows` x `cols`, the projections
             of a dense block (one HIP graph).

Every state has weights of its own, made on the GPU from the seed, and a step runs over several layers, so that
weights come from HBM as they do in a model. A state is warmed up by one pass over inputs of its own: a program
that serves has its experts pinned (and a captured graph, where it uses one) before the call that is timed.
"""
import ctypes as C
import math

import torch

from vireo_amd import _lib
from vireo_amd import kv as KV
from vireo_amd import model as MD
from vireo_amd import moe as M
from vireo_amd import workloads as W

DEV = "cuda"
GRAPH_TOKENS = 32  # calls of up to this many tokens are decode steps, replayed from a HIP graph
ROPE_BASE = 1000000.0
ATTN_TYPES = (W.Q4_K, W.Q4_K, W.Q6_K, W.Q4_K)  # wq, wk, wv, wo of the whole model
ATTN_SIGMA = 0.05  # their standard deviation (DeviceModel)
MODEL_HEADS = (32, 4, 128)  # query heads, kv heads, head size of the whole model
BLOCK_TOKENS = 32  # tokens per KV block


def listed():
    return [
        # one sequence decoding: a token through consecutive MoE layers of Qwen3-30B-A3B, the benchmark's headline
        {"name": "decode-1-qwen3-q4", "kind": "moe", "shape": "qwen3-30b-a3b-q4_k_m", "tokens": 1, "layers": 8,
         "zipf": False},
        # a few sequences decoding together
        {"name": "decode-4-olmoe-q4", "kind": "moe", "shape": "olmoe-q4_k_m", "tokens": 4, "layers": 4, "zipf": False},
        # a serving batch on the 8-bit model, an odd number of sequences
        {"name": "decode-23-olmoe-q8", "kind": "moe", "shape": "olmoe-q8_0", "tokens": 23, "layers": 2, "zipf": False},
        # a full serving batch on the 4-bit model
        {"name": "decode-32-qwen3-q4", "kind": "moe", "shape": "qwen3-30b-a3b-q4_k_m", "tokens": 32, "layers": 2,
         "zipf": False},
        # a short prompt, ragged against every tile
        {"name": "prefill-101-qwen3-q4", "kind": "moe", "shape": "qwen3-30b-a3b-q4_k_m", "tokens": 101, "layers": 1,
         "zipf": False},
        # a prefill chunk of the size schedulers use beside decode
        {"name": "prefill-512-olmoe-q4", "kind": "moe", "shape": "olmoe-q4_k_m", "tokens": 512, "layers": 1,
         "zipf": False},
        # the benchmark's prefill: 2048 tokens, skewed routing, 8-bit experts
        {"name": "prefill-2048-qwen3-q8-zipf", "kind": "moe", "shape": "qwen3-30b-a3b-q8_0", "tokens": 2048,
         "layers": 1, "zipf": True},
        # a long prompt on the 4-bit model: the largest call
        {"name": "prefill-4093-qwen3-q4", "kind": "moe", "shape": "qwen3-30b-a3b-q4_k_m", "tokens": 4093, "layers": 1,
         "zipf": False},
        # attention of a decode step at the benchmark's context
        {"name": "attention-4096", "kind": "attention", "heads": 32, "kv_heads": 4, "head_size": 128, "context": 4096,
         "layers": 8},
        # a long conversation
        {"name": "attention-30001", "kind": "attention", "heads": 32, "kv_heads": 4, "head_size": 128,
         "context": 30001, "layers": 4},
        # a whole decode step: attention, MoE, LM head
        {"name": "model-8-context-1000", "kind": "model", "shape": "qwen3-30b-a3b-q4_k_m", "layers": 8,
         "context": 1000, "vocab": 151936},
        # the projections of a dense block
        {"name": "matvec-q6k-4096", "kind": "matvec", "type": "Q6_K", "cols": 4096, "rows": 4099, "count": 8},
    ]


def _log_int(rng, lo, hi):
    return min(hi, int(lo * (hi / lo) ** rng.random() + 0.5))


def draw(rng):
    kind = rng.choice(["moe"] * 7 + ["attention", "model", "matvec"])
    if kind == "moe":
        tokens = _log_int(rng, 1, 4000)
        return {"kind": "moe", "shape": rng.choice(sorted(W.SHAPES)), "tokens": tokens,
                "layers": 8 if tokens == 1 else 4 if tokens <= 8 else 2 if tokens <= 64 else 1,
                "zipf": tokens > 64 and rng.random() < 0.4}
    if kind == "attention":
        heads, kv_heads = rng.choice([(32, 4), (16, 16), (32, 8), (8, 2)])
        context = _log_int(rng, 60, 30000)
        return {"kind": "attention", "heads": heads, "kv_heads": kv_heads, "head_size": rng.choice([64, 128]),
                "context": context, "layers": 8 if context * kv_heads < 40000 else 2}
    if kind == "model":
        return {"kind": "model", "shape": rng.choice(["olmoe-q4_k_m", "qwen3-30b-a3b-q4_k_m", "olmoe-q8_0"]),
                "layers": rng.randint(2, 8), "context": _log_int(rng, 30, 4000), "vocab": rng.choice([50304, 151936])}
    return {"kind": "matvec", "type": rng.choice(sorted(W.TYPE_NAMES.values())), "cols": 256 * rng.randint(1, 32),
            "rows": _log_int(rng, 100, 12000), "count": 8}


def _gen(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed((seed * 1000003 + salt) % (1 << 62))
    return g


def _type_id(name):
    return next(t for t, n in W.TYPE_NAMES.items() if n == name)


def _graph(step):
    """`step` captured in a HIP graph (after the pass that warmed it up)."""
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        step(s)
    return g


# ---- moe ----------------------------------------------------------------------------------------------------------

def _moe_inputs(case, seed):
    shape, T, L = W.SHAPES[case["shape"]], case["tokens"], case["layers"]
    bias = W.zipf_bias(shape.E, 1.1, seed % 1000) if case["zipf"] else None
    moe = M.DeviceMoE(shape, L, seed=seed, logit_bias=bias, device=DEV)
    # the residual stream and its RMSNorm, per layer
    x = torch.randn((L, T, shape.d), generator=_gen(seed, 1), device=DEV)
    hb = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + W.EPS)
    return moe, x, hb


def _moe_prepare(case, seed):
    moe, x, hb = _moe_inputs(case, seed)
    shape, T, L = moe.shape, case["tokens"], case["layers"]
    idx = torch.empty((L, T, shape.k), dtype=torch.int32, device=DEV)
    w = torch.empty((L, T, shape.k), dtype=torch.float32, device=DEV)
    st = {"moe": moe, "x": x, "hb": hb, "idx": idx, "w": w, "layers": L}

    def step(x, hb, stream=None):
        h = M._stream_handle(stream)
        for l in range(L):
            _lib.check(moe.lib.moe_ffn_forward(C.byref(moe.model), l, M._ptr(x[l]), M._ptr(hb[l]), T, M._ptr(idx[l]),
                                               M._ptr(w[l]), h), "moe_ffn_forward")

    other = torch.randn(hb.shape, generator=_gen(seed, 2), device=DEV)
    step(torch.zeros_like(x), other)
    torch.cuda.synchronize()
    st["graph"] = _graph(lambda s: step(x, hb, s)) if T <= GRAPH_TOKENS else None
    st["step"] = step
    return st


def _moe_run(st):
    if st["graph"] is not None:
        st["graph"].replay()
    else:
        st["step"](st["x"], st["hb"])
    return {"x": st["x"], "idx": st["idx"], "w": st["w"]}


def _routing_f32(R, hb, bias, k):
    """The reference's selection: in-order fp32 sums, softmax, the k most probable, the lower id first on a tie."""
    acc = torch.zeros((hb.shape[0], R.shape[0]), dtype=torch.float32, device=hb.device)
    hc, Rc = hb.t().contiguous(), R.t().contiguous()
    for i in range(hb.shape[1]):
        acc = acc + hc[i][:, None] * Rc[i][None, :]
    if bias is not None:
        acc = acc + bias
    e = torch.exp(acc - acc.max(1, keepdim=True).values)
    return torch.sort(e / e.sum(1, keepdim=True), dim=1, descending=True, stable=True).indices[:, :k]


def _moe_layer_64(moe, layer, x, hb):
    """x + moe(hb) and the weights of one layer in 64 bits; x and hb [tokens x d] (any float type)."""
    shape = moe.shape
    R = moe.routers[layer]
    idx = _routing_f32(R, hb.float(), moe.bias, shape.k)
    logits = hb.double() @ R.double().t()
    if moe.bias is not None:
        logits = logits + moe.bias.double()
    w = torch.softmax(logits, 1).gather(1, idx)
    if shape.renorm:
        w = w / w.sum(1, keepdim=True)
    gs, us, ds = moe.slices
    base, E = layer * moe.layer_bytes, shape.E
    out, h64 = x.double().clone(), hb.double()
    for e in range(E):
        t, j = (idx == e).nonzero(as_tuple=True)
        if t.numel() == 0:
            continue
        g = _dequant(shape.gate_type, moe.buf[base + e * gs:base + (e + 1) * gs], shape.d)
        u = _dequant(shape.up_type, moe.buf[base + E * gs + e * us:base + E * gs + (e + 1) * us], shape.d)
        o = base + E * (gs + us)
        dn = _dequant(shape.down_type, moe.buf[o + e * ds:o + (e + 1) * ds], shape.fe)
        a = h64[t] @ g.t()
        y = (a * torch.sigmoid(a) * (h64[t] @ u.t())) @ dn.t()
        out.index_add_(0, t, y * w[t, j][:, None])
    return out, w


def _moe_exact(case, seed):
    moe, x, hb = _moe_inputs(case, seed)
    outs = [_moe_layer_64(moe, l, x[l], hb[l]) for l in range(case["layers"])]
    moe.close()
    return {"x": torch.stack([o[0] for o in outs]), "idx": None, "w": torch.stack([o[1] for o in outs])}


def _distinct(case, shape):
    """Experts that `tokens` tokens are expected to reach."""
    if case["zipf"]:
        p = [r ** -1.1 for r in range(1, shape.E + 1)]
        p = [min(1.0, shape.k * v / sum(p)) for v in p]
    else:
        p = [shape.k / shape.E] * shape.E
    return sum(1 - (1 - v) ** case["tokens"] for v in p)


def _moe_work(case):
    s, T, L = W.SHAPES[case["shape"]], case["tokens"], case["layers"]
    bytes_ = s.E * s.d * 4 + _distinct(case, s) * s.expert_bytes() + 3 * T * s.d * 4 + T * s.k * 8
    return {"bytes": L * bytes_, "flops": L * T * (s.k * 6 * s.d * s.fe + 2 * s.E * s.d)}


# ---- attention ----------------------------------------------------------------------------------------------------

def _kv_rows(seed, layers, kv_heads, hd, context):
    """Keys and values [context + 1 x layers * kv_heads x head size]: the context and the step's own token."""
    n = layers * kv_heads
    return tuple(torch.randn((context + 1, n, hd), generator=_gen(seed, salt), device=DEV) for salt in (11, 12))


def _kv_fill(store, k, v, tokens):
    """Append the first `tokens` tokens of every row, up to 16 rows a call."""
    n, s, lib = k.shape[1], MD._stream(), _lib.load()
    step = k.stride(0) * 4
    for r in range(0, n, 16):
        m, ka, va = min(16, n - r), k.data_ptr() + r * k.shape[2] * 4, v.data_ptr() + r * k.shape[2] * 4
        for t in range(tokens):
            rc = lib.vireo_kv_append_n(store.h, r, m, t, ka + t * step, va + t * step, s)
            if rc:
                _lib.check(rc, "vireo_kv_append_n")


def _attention_prepare(case, seed):
    L, H, KVH, hd, ctx = case["layers"], case["heads"], case["kv_heads"], case["head_size"], case["context"]
    k, v = _kv_rows(seed, L, KVH, hd, ctx)
    store = KV.DeviceKV(L * KVH, hd, BLOCK_TOKENS, dense=True, max_tokens=ctx + 64)
    _kv_fill(store, k, v, ctx)
    st = {"kv": store, "pos": torch.full((1,), ctx, dtype=torch.int32, device=DEV),
          "q": torch.randn((L, H, hd), generator=_gen(seed, 13), device=DEV),
          "out": torch.empty((L, H, hd), device=DEV), "k": k[ctx].clone(), "v": v[ctx].clone()}
    del k, v

    def step(stream=None):
        for l in range(L):
            rows = slice(l * KVH, (l + 1) * KVH)
            store.append_pos(l * KVH, st["pos"], st["k"][rows], st["v"][rows], stream=stream)
            store.attend_gqa_pos(l * KVH, H, KVH, st["pos"], st["q"][l], st["out"][l], stream=stream)

    step()
    torch.cuda.synchronize()
    st["out"].zero_()
    st["graph"] = _graph(step)
    return st


def _attention_run(st):
    st["graph"].replay()
    return st["out"]


def _attend_64(q, k, v):
    """q [heads x hd], k and v [context x kv heads x hd] -> [heads x hd], in 64 bits."""
    KVH, hd = k.shape[1], k.shape[2]
    qq = q.double().reshape(KVH, -1, hd)
    kk, vv = (a.double().permute(1, 0, 2).contiguous() for a in (k, v))
    p = torch.softmax(torch.matmul(qq, kk.transpose(1, 2).contiguous()) / math.sqrt(hd), dim=-1)
    return torch.matmul(p, vv).reshape(-1, hd)


def _attention_exact(case, seed):
    L, H, KVH, hd, ctx = case["layers"], case["heads"], case["kv_heads"], case["head_size"], case["context"]
    k, v = _kv_rows(seed, L, KVH, hd, ctx)
    q = torch.randn((L, H, hd), generator=_gen(seed, 13), device=DEV)
    rows = [slice(l * KVH, (l + 1) * KVH) for l in range(L)]
    return torch.stack([_attend_64(q[l], k[:, rows[l]], v[:, rows[l]]) for l in range(L)])


def _attention_work(case):
    L, H, KVH, hd, n = case["layers"], case["heads"], case["kv_heads"], case["head_size"], case["context"] + 1
    return {"bytes": L * (n * KVH * hd * 8 + 2 * H * hd * 4), "flops": L * 4 * H * hd * n}


# ---- model --------------------------------------------------------------------------------------------------------

def _model_inputs(case, seed):
    H, KVH, hd = MODEL_HEADS
    L, ctx = case["layers"], case["context"]
    m = MD.DeviceModel(W.SHAPES[case["shape"]], L, H, KVH, hd, vocab=case["vocab"], max_pos=ctx + 64, seed=seed,
                       attn_types=ATTN_TYPES, block_tokens=BLOCK_TOKENS, rope_base=ROPE_BASE, contiguous=True)
    k, v = _kv_rows(seed, L, KVH, hd, ctx)
    return m, k, v, (seed * 7919 + 17) % case["vocab"]


def _model_prepare(case, seed):
    m, k, v, token = _model_inputs(case, seed)
    ctx = case["context"]
    _kv_fill(m.kv, k, v, ctx)

    def step(stream=None):  # every pass decodes the same token at the same position
        m.pos.fill_(ctx)
        m.token.fill_(token)
        m.step_pos(stream=stream)

    step()
    torch.cuda.synchronize()
    return {"m": m, "graph": _graph(step)}


def _model_run(st):
    st["graph"].replay()
    return {"logits": st["m"].logits, "x": st["m"].x}


def _model_exact(case, seed):
    m, k, v, token = _model_inputs(case, seed)
    H, KVH, hd = MODEL_HEADS
    L, ctx, moe = case["layers"], case["context"], m.stack.moe
    d = moe.shape.d
    lm_rb = W.row_bytes(W.Q8_0, d)
    norm = lambda a: a * torch.rsqrt((a * a).mean(-1, keepdim=True) + W.EPS)  # noqa: E731 (unit weights)
    ang = ctx * ROPE_BASE ** (-2.0 * torch.arange(hd // 2, dtype=torch.float64, device=DEV) / hd)
    cos, sin = torch.cos(ang), torch.sin(ang)

    def rope(a):
        lo, hi = a[..., :hd // 2], a[..., hd // 2:]
        return torch.cat([lo * cos - hi * sin, lo * sin + hi * cos], dim=-1)

    base = m.wbuf.data_ptr()

    def matrix(l, i, n, rows):
        at = m._mats[4 * l + i].data - base
        return _dequant(ATTN_TYPES[i], m.wbuf[at:at + W.row_bytes(ATTN_TYPES[i], n) * rows], n)

    x = _dequant(W.Q8_0, m.stack.lm[token * lm_rb:(token + 1) * lm_rb], d)[0]
    for l in range(L):
        xb = norm(x)
        q, kn, vn = (matrix(l, i, d, hd * n) @ xb for i, n in ((0, H), (1, KVH), (2, KVH)))
        q, kn = rope(norm(q.reshape(H, hd))), rope(norm(kn.reshape(KVH, hd)))
        rows = slice(l * KVH, (l + 1) * KVH)
        kk = torch.cat([k[:ctx, rows].double(), kn[None]])
        vv = torch.cat([v[:ctx, rows].double(), vn.reshape(1, KVH, hd)])
        x = x + matrix(l, 3, H * hd, d) @ _attend_64(q, kk, vv).reshape(-1)
        x = _moe_layer_64(moe, l, x[None], norm(x)[None])[0][0]
    xb = norm(x)
    logits = torch.cat([_dequant(W.Q8_0, m.stack.lm[r * lm_rb:min(r + 16384, case["vocab"]) * lm_rb], d) @ xb
                        for r in range(0, case["vocab"], 16384)])
    m.close()
    return {"logits": logits, "x": x}


def _model_work(case):
    H, KVH, hd = MODEL_HEADS
    s, L, V = W.SHAPES[case["shape"]], case["layers"], case["vocab"]
    dims = [(s.d, H * hd), (s.d, KVH * hd), (s.d, KVH * hd), (H * hd, s.d)]
    attn = sum(W.row_bytes(t, n) * r for t, (n, r) in zip(ATTN_TYPES, dims))
    kv = KVH * (case["context"] + 1) * hd * 8
    layer = attn + kv + s.E * s.d * 4 + s.k * s.expert_bytes()
    flops = 2 * sum(n * r for n, r in dims) + 4 * H * hd * (case["context"] + 1) + s.k * 6 * s.d * s.fe + 2 * s.E * s.d
    return {"bytes": L * layer + V * (W.row_bytes(W.Q8_0, s.d) + 4), "flops": L * flops + 2 * V * s.d}


# ---- matvec -------------------------------------------------------------------------------------------------------

def _matvec_inputs(case, seed):
    typ, n, d, cnt = _type_id(case["type"]), case["cols"], case["rows"], case["count"]
    per = (W.row_bytes(typ, n) * d + 255) // 256 * 256
    w = torch.empty(per * cnt, dtype=torch.uint8, device=DEV)
    for i in range(cnt):
        if typ in (W.F32, W.F16):
            v = torch.randn(n * d, generator=_gen(seed, 21 + i), device=DEV) * W.WEIGHT_SIGMA
            b = (v.half() if typ == W.F16 else v).view(torch.uint8)
            w[i * per:i * per + b.numel()] = b
        else:
            _lib.check(_lib.load().vireo_synth_matrix_dev(typ, C.c_void_p(w.data_ptr() + i * per), n, 0, d, seed,
                                                          W.stream_id(i, W.KIND_GATE), W.WEIGHT_SIGMA,
                                                          M._stream_handle()), "vireo_synth_matrix_dev")
    return typ, w.view(cnt, per), torch.randn(n, generator=_gen(seed, 20), device=DEV)


def _matvec_prepare(case, seed):
    typ, w, x = _matvec_inputs(case, seed)
    y = torch.zeros((case["count"], case["rows"]), device=DEV)

    def step(stream=None):
        for i in range(case["count"]):
            M.qmatvec(y[i], x, w[i], typ, case["cols"], case["rows"], stream=stream)

    step()
    torch.cuda.synchronize()
    return {"w": w, "x": x, "y": y, "graph": _graph(step)}


def _matvec_run(st):
    st["graph"].replay()
    return st["y"]


def _matvec_exact(case, seed):
    typ, w, x = _matvec_inputs(case, seed)
    nb = W.row_bytes(typ, case["cols"]) * case["rows"]
    return torch.stack([_dequant(typ, w[i, :nb], case["cols"]) @ x.double() for i in range(case["count"])])


def _matvec_work(case):
    typ, n, d, cnt = _type_id(case["type"]), case["cols"], case["rows"], case["count"]
    return {"bytes": cnt * (W.row_bytes(typ, n) * d + 4 * d) + 4 * n, "flops": cnt * 2 * n * d}


# ---- the GGUF formats in 64 bits ----------------------------------------------------------------------------------

def _dequant(typ, raw, n):
    """The rows of n weights in the bytes `raw` (uint8, on the device), as float64 [rows x n]."""
    be, bb = W.BLOCK[typ]
    raw = raw.contiguous()
    if typ == W.F32:
        return raw.view(torch.float32).reshape(-1, n).double()
    if typ == W.F16:
        return raw.view(torch.float16).reshape(-1, n).double()
    b = raw.reshape(-1, bb)

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()  # [blocks x 1]

    if typ == W.Q8_0:
        y = half(0) * b[:, 2:34].contiguous().view(torch.int8).double()
    elif typ == W.Q5_0:
        bits = (b[:, 2:6, None].int() >> torch.arange(8, device=b.device)) & 1  # bit j of the 32: weight j
        qs = b[:, 6:22].int()
        q = torch.cat([qs & 15, qs >> 4], 1) | (bits.reshape(-1, 32) << 4)
        y = half(0) * (q - 16).double()
    elif typ == W.Q4_K:
        s = b[:, 4:16].int()
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        qs = b[:, 16:144].int().reshape(-1, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
        y = (half(0) * sc)[:, :, None] * q - (half(2) * mn)[:, :, None]
    elif typ == W.Q6_K:
        ql, qh = b[:, :128].int().reshape(-1, 2, 2, 32), b[:, 128:192].int().reshape(-1, 2, 32)
        q = torch.stack([(ql[:, :, g & 1] >> (4 * (g >> 1))) & 15 | (((qh >> (2 * g)) & 3) << 4) for g in range(4)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double() * half(208)
        y = (q - 32).double().reshape(-1, 16, 16) * sc[:, :, None]
    else:
        raise ValueError(typ)
    return y.reshape(-1, n)


# ---- by kind ------------------------------------------------------------------------------------------------------

_KINDS = {"moe": (_moe_prepare, _moe_run, _moe_exact, _moe_work),
          "attention": (_attention_prepare, _attention_run, _attention_exact, _attention_work),
          "model": (_model_prepare, _model_run, _model_exact, _model_work),
          "matvec": (_matvec_prepare, _matvec_run, _matvec_exact, _matvec_work)}


def prepare(case, seed):
    _lib.check(_lib.load().vireo_hip_init(0), "vireo_hip_init")
    return dict(_KINDS[case["kind"]][0](case, seed), kind=case["kind"])


def run(state):
    return _KINDS[state["kind"]][1](state)


def exact(case, seed):
    return _KINDS[case["kind"]][2](case, seed)


def work(case):
    return _KINDS[case["kind"]][3](case)


def tolerance(case):
    """About four times the largest relative error against exact() that the library shows on these cases: of the
    output of a decode batch on split 16-bit operands (2.8e-7), of a prefill through bf16 GEMMs (5.4e-4, in the
    residual stream it is added to), of the attention (4.5e-7), of a whole step (2e-5: the rotation angles are 32-bit
    numbers) and of a matvec (2.5e-7)."""
    if case["kind"] == "moe":
        return {"rel": 2e-3 if case["tokens"] >= 64 else 1.2e-6}
    return {"rel": {"attention": 2e-6, "model": 1e-4, "matvec": 1e-6}[case["kind"]]}
