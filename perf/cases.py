"""The work this framework is measured on, through its public entry points.

A case is a dict of plain values; ``kind`` picks the path:

  moe_decode   one token through the MoE block of every layer of a model
               (MoEBlock.forward, one call per layer)
  moe_prefill  T tokens at once through one layer's MoE block (MoEBlock.prefill)
  attention    decode attention of one query over a KV cache
               (DenseOps.attention_decode)
  head         final norm, lm_head and greedy token (DenseOps.rmsnorm,
               matvec_bf16, argmax)
  decoder      a whole call: reset, the prompt in one batch, then one step per
               given token (Decoder.prefill_device, step_device), with the
               logits of the prompt's last token and of every step

Inputs are made on the GPU from the seed alone.  Expert weights have the form
a converter writes (uniform nibbles, group bias about -7.5 scales, so that the
weights are centred with a variance of about 1 / columns); routers are bf16
N(0, 0.02), activations N(0, 1), dense weights N(0, 1 / columns).
"""
from __future__ import annotations

import math

import torch

from m1moe_amd._lib import DecShape
from m1moe_amd import _lib
from m1moe_amd.decoder import Decoder, DenseOps
from m1moe_amd.engine import HIPContext, MoEBlock, expert_bytes, expert_offsets, make_shape
from m1moe_amd.synth import zipf_logit_bias

DEV = "cuda"
EPS = 1e-5

# the two model widths of the repository's own configurations
OLMOE = dict(hidden=2048, experts=64, top_k=8, inter=1024, group=64, norm=False)
MIXTRAL = dict(hidden=4096, experts=8, top_k=2, inter=14336, group=64, norm=True)
# their attention, vocabulary and RoPE
OLMOE_DEC = dict(vocab=50304, heads=16, kv_heads=16, head_dim=128, qk_norm=True, theta=10000.0)
MIXTRAL_DEC = dict(vocab=32000, heads=32, kv_heads=8, head_dim=128, qk_norm=False, theta=1e6)


# ---- the cases ------------------------------------------------------------------------


def listed():
    return [
        # the smallest call: a small model's single layer, f32 activations, groups of 32
        dict(name="decode_small", kind="moe_decode", hidden=256, experts=16, top_k=4, inter=128,
             group=32, norm=True, layers=1, x="f32"),
        # one token through all 16 MoE layers of an OLMoE-1B-7B-shaped model
        dict(name="decode_olmoe", kind="moe_decode", **OLMOE, layers=16, x="bf16"),
        # one token through four Mixtral-8x7B-shaped MoE layers, f32 activations
        dict(name="decode_mixtral", kind="moe_decode", **MIXTRAL, layers=4, x="f32"),
        # a chat turn's worth of new tokens, an odd number of them
        dict(name="prefill_olmoe_37", kind="moe_prefill", **OLMOE, T=37, zipf=0.0, x="f32"),
        # the benchmark's prefill: 512 tokens, skewed expert loads
        dict(name="prefill_olmoe_512", kind="moe_prefill", **OLMOE, T=512, zipf=1.1, x="bf16"),
        # a long prompt through one Mixtral-shaped layer, ragged
        dict(name="prefill_mixtral_1000", kind="moe_prefill", **MIXTRAL, T=1000, zipf=0.0,
             x="f32"),
        # decode attention early in a conversation (multi-head, OLMoE shape)
        dict(name="attention_short", kind="attention", heads=16, kv_heads=16, head_dim=128,
             seq=200),
        # decode attention late in one (grouped heads, Mixtral shape)
        dict(name="attention_long", kind="attention", heads=32, kv_heads=8, head_dim=128,
             seq=5003),
        # the end of every step: final norm, lm_head, greedy token
        dict(name="head_olmoe", kind="head", hidden=2048, vocab=50304),
        # a whole turn of the OLMoE-shaped model: 128-token prompt, 16 steps
        dict(name="turn_olmoe", kind="decoder", **OLMOE, **OLMOE_DEC, layers=16, T=128, steps=16),
        # a ragged prompt through four of its layers
        dict(name="prompt_olmoe_333", kind="decoder", **OLMOE, **OLMOE_DEC, layers=4, T=333,
             steps=1),
        # the benchmark's 2048-token context through two Mixtral-shaped layers
        dict(name="prompt_mixtral_2048", kind="decoder", **MIXTRAL, **MIXTRAL_DEC, layers=2,
             T=2048, steps=2),
    ]


def _pad4(n):
    """Row length in 4-byte words of an output whose rows the library takes one
    by one (16-byte aligned)."""
    return (n + 3) // 4 * 4


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _moe_shape(rng):
    """One of the two model widths, or a generic one within the library's limits."""
    pick = rng.random()
    if pick < 0.35:
        return dict(OLMOE)
    if pick < 0.6:
        return dict(MIXTRAL)
    group = rng.choice([32, 64, 128])
    step = max(64, group)
    hidden = step * _log_int(rng, 2, 4096 // step)
    inter = step * _log_int(rng, 1, 4096 // step)
    experts = _log_int(rng, 4, 64)
    return dict(hidden=hidden, experts=experts, top_k=rng.randint(1, min(8, experts)),
                inter=inter, group=group, norm=rng.random() < 0.5)


def draw(rng):
    kind = rng.choice(["moe_decode", "moe_decode", "moe_prefill", "moe_prefill", "attention",
                       "head", "decoder", "decoder"])
    if kind == "moe_decode":
        s = _moe_shape(rng)
        return dict(kind=kind, **s, layers=rng.randint(1, 4), x=rng.choice(["f32", "bf16"]))
    if kind == "moe_prefill":
        s = _moe_shape(rng)
        return dict(kind=kind, **s, T=_log_int(rng, 2, 1000), zipf=rng.choice([0.0, 1.1]),
                    x=rng.choice(["f32", "bf16"]))
    if kind == "attention":
        heads, kv = rng.choice([(16, 16), (32, 8), (32, 32), (8, 1), (24, 8)])
        return dict(kind=kind, heads=heads, kv_heads=kv, head_dim=rng.choice([64, 128, 128, 256]),
                    seq=_log_int(rng, 16, 8192))
    if kind == "head":
        return dict(kind=kind, hidden=64 * _log_int(rng, 4, 64), vocab=_log_int(rng, 1000, 64000))
    if rng.random() < 0.5:
        return dict(kind=kind, **OLMOE, **OLMOE_DEC, layers=rng.randint(1, 4),
                    T=_log_int(rng, 2, 2000), steps=rng.randint(0, 8))
    if rng.random() < 0.6:
        return dict(kind=kind, **MIXTRAL, **MIXTRAL_DEC, layers=rng.randint(1, 2),
                    T=_log_int(rng, 2, 1900), steps=rng.randint(0, 4))
    group = rng.choice([32, 64])
    kv = rng.choice([1, 2, 4])
    return dict(kind=kind, hidden=64 * _log_int(rng, 2, 32), experts=_log_int(rng, 4, 32),
                top_k=rng.randint(1, 4), inter=64 * _log_int(rng, 1, 32), group=group,
                norm=rng.random() < 0.5, vocab=_log_int(rng, 300, 20000), heads=kv * rng.choice([1, 2, 4]),
                kv_heads=kv, head_dim=rng.choice([64, 128]), qk_norm=rng.random() < 0.5,
                theta=10000.0, layers=rng.randint(1, 3), T=_log_int(rng, 2, 1000),
                steps=rng.randint(0, 8))


# ---- inputs ---------------------------------------------------------------------------


def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1000003 + stream)
    return g


def _normal(shape, seed, stream, sigma=1.0, dtype=torch.float32):
    return (torch.randn(shape, generator=_gen(seed, stream), device=DEV) * sigma).to(dtype)


def _shape(c, layers):
    return make_shape(c["hidden"], c["experts"], c["top_k"], c["inter"], c["group"], layers,
                      c["norm"])


def _projections(c):
    """(rows, columns, offsets of W, S and B) of gate, up and down in an expert block."""
    off = expert_offsets(_shape(c, 1))
    h, i = c["hidden"], c["inter"]
    return [(i, h, *off[0:3]), (i, h, *off[3:6]), (h, i, *off[6:9])]


def _image(c, seed, layer):
    """One layer's expert blocks in the on-disk layout: uint8 [experts, block bytes]."""
    n = expert_bytes(_shape(c, 1))
    g = _gen(seed, 100 + layer)
    img = torch.randint(0, 256, (c["experts"], n), dtype=torch.uint8, generator=g, device=DEV)
    for rows, cols, _, s_off, b_off in _projections(c):
        m = rows * cols // c["group"]
        u = torch.rand((c["experts"], m), generator=g, device=DEV)
        s = ((0.75 + 0.5 * u) / (4.6 * math.sqrt(cols))).to(torch.bfloat16)
        z = torch.randn((c["experts"], m), generator=g, device=DEV)
        b = (-7.5 * s.float() * (1 + 0.05 * z)).to(torch.bfloat16)
        img[:, s_off:s_off + 2 * m] = s.view(torch.uint8)
        img[:, b_off:b_off + 2 * m] = b.view(torch.uint8)
    return img


def _router(c, seed, layer):
    return _normal((c["experts"], c["hidden"]), seed, 300 + layer, 0.02, torch.bfloat16)


def _host_bits(t):
    """bf16 tensor -> host uint16 array of its bits."""
    return t.contiguous().view(torch.int16).cpu().numpy().view("uint16")


def _context(c, seed, layers):
    ctx = HIPContext(_shape(c, layers))
    for layer in range(layers):
        ctx.upload_layer_experts(layer, _image(c, seed, layer).cpu().numpy().reshape(-1))
        ctx.upload_router(layer, _host_bits(_router(c, seed, layer)))
        if c.get("zipf"):
            ctx.set_logit_bias(layer, zipf_logit_bias(c["experts"], c["zipf"]))
    return ctx


def _x_dtype(c):
    return torch.bfloat16 if c["x"] == "bf16" else torch.float32


def _moe_inputs(c, seed):
    """Activations and residuals, one row per layer (decode) or per token (prefill)."""
    n = c["layers"] if c["kind"] == "moe_decode" else c["T"]
    return (_normal((n, c["hidden"]), seed, 1, 1.0, _x_dtype(c)),
            _normal((n, c["hidden"]), seed, 2))


def _attention_inputs(c, seed):
    kvd = c["kv_heads"] * c["head_dim"]
    return (_normal((c["heads"], c["head_dim"]), seed, 1), _normal((c["seq"], kvd), seed, 2),
            _normal((c["seq"], kvd), seed, 3))


def _head_inputs(c, seed):
    h = c["hidden"]
    return (_normal((h,), seed, 1), (1 + _normal((h,), seed, 2, 0.1)).to(torch.bfloat16),
            _normal((c["vocab"], h), seed, 3, 1 / math.sqrt(h), torch.bfloat16))


def _dense(c, seed, which, layer):
    """Dense tensor `which` of the decoder, bf16."""
    h, hd = c["hidden"], c["head_dim"]
    qd, kvd = c["heads"] * hd, c["kv_heads"] * hd
    dims = {_lib.W_EMBED: (c["vocab"], h), _lib.W_LM_HEAD: (c["vocab"], h),
            _lib.W_FINAL_NORM: (h,), _lib.W_IN_NORM: (h,), _lib.W_POST_NORM: (h,),
            _lib.W_Q: (qd, h), _lib.W_K: (kvd, h), _lib.W_V: (kvd, h), _lib.W_O: (h, qd),
            _lib.W_Q_NORM: (hd,), _lib.W_K_NORM: (hd,)}[which]
    stream = 1000 + 20 * layer + which
    if len(dims) == 1:
        return (1 + _normal(dims, seed, stream, 0.1)).to(torch.bfloat16)
    sigma = 1.0 if which == _lib.W_EMBED else 1 / math.sqrt(dims[1])
    return _normal(dims, seed, stream, sigma, torch.bfloat16)


def _tokens(c, seed):
    return torch.randint(0, c["vocab"], (c["T"] + c["steps"],), dtype=torch.int32,
                         generator=_gen(seed, 4), device=DEV)


def prepare(case, seed):
    c = case
    if c["kind"] in ("moe_decode", "moe_prefill"):
        layers = c["layers"] if c["kind"] == "moe_decode" else 1
        ctx = _context(c, seed, layers)
        x, res = _moe_inputs(c, seed)
        n = x.shape[0]
        out = torch.empty_like(res)
        k = _pad4(c["top_k"]) if c["kind"] == "moe_decode" else c["top_k"]
        idx = torch.empty((n, k), dtype=torch.int32, device=DEV)
        w = torch.empty((n, k), dtype=torch.float32, device=DEV)
        state = dict(block=MoEBlock(ctx), tensors=(x, res, out, idx, w), dtype=c["x"])
    elif c["kind"] == "attention":
        ctx = HIPContext(make_shape(64, 1, 1, 64))  # the building blocks need a context's stream
        q, k, v = _attention_inputs(c, seed)
        state = dict(ops=DenseOps(ctx), tensors=(q, k, v, torch.empty_like(q)))
    elif c["kind"] == "head":
        ctx = HIPContext(make_shape(64, 1, 1, 64))
        x, nw, w = _head_inputs(c, seed)
        state = dict(ops=DenseOps(ctx), tensors=(
            x, nw, w, torch.empty_like(x),
            torch.empty((c["vocab"],), dtype=torch.float32, device=DEV),
            torch.empty((1,), dtype=torch.int32, device=DEV)))
    else:
        ctx = _context(c, seed, c["layers"])
        dec = Decoder(ctx, DecShape(c["vocab"], c["heads"], c["kv_heads"], c["head_dim"],
                                    c["T"] + c["steps"], 1 if c["qk_norm"] else 0, c["theta"], EPS))
        dec.upload_all(lambda which, layer: _host_bits(_dense(c, seed, which, layer)))
        logits = torch.empty((1 + c["steps"], _pad4(c["vocab"])), dtype=torch.float32, device=DEV)
        next_token = torch.empty((1,), dtype=torch.int32, device=DEV)
        state = dict(decoder=dec, tensors=(_tokens(c, seed), logits, next_token))
    state.update(case=c, ctx=ctx)
    torch.cuda.synchronize()  # the inputs are on torch's stream, the calls on the library's
    return state


# ---- one pass -------------------------------------------------------------------------


def run(state):
    c, t = state["case"], state["tensors"]
    if c["kind"] == "moe_decode":
        x, res, out, idx, w = t
        forward, dtype = state["block"].forward, state["dtype"]
        xs, rs, ks = x.stride(0) * x.element_size(), 4 * c["hidden"], 4 * idx.stride(0)
        xp, rp, op, ip, wp = (a.data_ptr() for a in t)
        for layer in range(c["layers"]):
            forward(layer, xp + layer * xs, dtype, rp + layer * rs, op + layer * rs,
                    ip + layer * ks, wp + layer * ks)
        return out, idx[:, :c["top_k"]], w[:, :c["top_k"]]
    if c["kind"] == "moe_prefill":
        x, res, out, idx, w = t
        state["block"].prefill(0, c["T"], x.data_ptr(), state["dtype"], res.data_ptr(),
                               out.data_ptr(), idx.data_ptr(), w.data_ptr())
        return out, idx, w
    if c["kind"] == "attention":
        q, k, v, out = t
        state["ops"].attention_decode(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                                      c["heads"], c["kv_heads"], c["head_dim"], c["seq"])
        return out
    if c["kind"] == "head":
        x, nw, w, xn, logits, idx = t
        ops = state["ops"]
        ops.rmsnorm(x.data_ptr(), nw.data_ptr(), xn.data_ptr(), c["hidden"], EPS)
        ops.matvec_bf16(w.data_ptr(), xn.data_ptr(), None, logits.data_ptr(), c["vocab"],
                        c["hidden"])
        ops.argmax(logits.data_ptr(), c["vocab"], idx.data_ptr())
        return logits, idx
    tokens, logits, next_token = t
    dec = state["decoder"]
    tp, lp, row = tokens.data_ptr(), logits.data_ptr(), 4 * logits.stride(0)
    dec.reset()
    dec.prefill_device(tp, c["T"], next_token.data_ptr(), lp)
    for i in range(c["steps"]):
        dec.step_device(tp + 4 * (c["T"] + i), next_token.data_ptr(), lp + (1 + i) * row)
    return logits[:, :c["vocab"]]


# ---- what a pass cannot do without ----------------------------------------------------


def _moe_work(c, T, x_bytes):
    """Bytes and operations of one layer's MoE block for T tokens."""
    h, k = c["hidden"], c["top_k"]
    block = 3 * h * c["inter"] * (0.5 + 4.0 / c["group"])
    experts = min(c["experts"], T * k)
    return (experts * block + 2 * c["experts"] * h + T * h * (x_bytes + 8),
            T * (6.0 * h * c["inter"] * k + 2.0 * h * c["experts"]))


def work(case):
    c = case
    if c["kind"] == "moe_decode":
        b, f = _moe_work(c, 1, 2 if c["x"] == "bf16" else 4)
        return {"bytes": c["layers"] * b, "flops": c["layers"] * f}
    if c["kind"] == "moe_prefill":
        b, f = _moe_work(c, c["T"], 2 if c["x"] == "bf16" else 4)
        return {"bytes": b, "flops": f}
    if c["kind"] == "attention":
        qd, kvd = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
        return {"bytes": 8.0 * c["seq"] * kvd + 8.0 * qd, "flops": 4.0 * c["seq"] * qd}
    if c["kind"] == "head":
        h, v = c["hidden"], c["vocab"]
        return {"bytes": 2.0 * v * h + 4.0 * v + 6.0 * h, "flops": 2.0 * v * h}
    h, qd, kvd = c["hidden"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    layer_w = h * (2.0 * qd + 2.0 * kvd)
    total_b = total_f = 0.0
    for first, T in [(0, c["T"])] + [(c["T"] + i, 1) for i in range(c["steps"])]:
        b, f = _moe_work(c, T, 0)
        pairs = T * first + T * (T + 1) / 2.0
        total_b += c["layers"] * (b - 8.0 * T * h + 2 * layer_w + 8.0 * (first + T) * kvd)
        total_f += c["layers"] * (f + 2.0 * T * layer_w + 4.0 * pairs * qd)
        total_b += 2.0 * c["vocab"] * h + 4.0 * c["vocab"] + 2.0 * T * h
        total_f += 2.0 * c["vocab"] * h
    return {"bytes": total_b, "flops": total_f}


# ---- tolerances -----------------------------------------------------------------------


def tolerance(case):
    c = case
    if c["kind"] in ("attention", "head"):
        # f32 sums in another order (2e-7 off 64 bits; expf within an ulp or two)
        return {"rel": 2e-6}
    if c["kind"] == "moe_decode":
        # f32 sums of exact products, the inputs and SwiGLU products with 22 bits and
        # the group sums cancelling against the bias term (2e-6 .. 2e-5 off 64 bits)
        return {"rel": 8e-5}
    # the prefill multiplies f16 expert weights and f16 SwiGLU products (2^-11 each):
    # one layer 4e-5 .. 1.6e-4 off 64 bits, a whole call 3e-5 .. 9e-4
    return {"rel": 1e-3} if c["kind"] == "moe_prefill" else {"rel": 4e-3}


# ---- the same in 64 bits --------------------------------------------------------------


def _weights64(c, block):
    """gate, up and down of one expert block in f64."""
    found = []
    for rows, cols, w_off, s_off, b_off in _projections(c):
        m = rows * cols // c["group"]
        packed = block[w_off:w_off + rows * cols // 2]
        nib = torch.stack((packed & 15, packed >> 4), 1).reshape(m, c["group"]).double()
        s = block[s_off:s_off + 2 * m].clone().view(torch.bfloat16).double()
        b = block[b_off:b_off + 2 * m].clone().view(torch.bfloat16).double()
        found.append((nib * s[:, None] + b[:, None]).reshape(rows, cols))
    return found


def _moe64(c, seed, layer, x, res, img=None):
    """(out, experts, weights) of the MoE block for the rows of x."""
    img = _image(c, seed, layer) if img is None else img
    logits = x @ _router(c, seed, layer).double().t().contiguous()
    if c.get("zipf"):
        logits = logits + torch.from_numpy(zipf_logit_bias(c["experts"], c["zipf"])).to(DEV).double()
    idx = torch.sort(logits, dim=1, descending=True, stable=True)[1][:, :c["top_k"]]
    w = torch.softmax(logits, 1).gather(1, idx)
    if c["norm"]:
        w = w / w.sum(1, keepdim=True)
    out = res.clone()
    for e in torch.unique(idx).tolist():
        gate, up, down = (m.t().contiguous() for m in _weights64(c, img[e]))
        tok, slot = torch.nonzero(idx == e, as_tuple=True)
        g = x[tok] @ gate
        y = (g * torch.sigmoid(g) * (x[tok] @ up)) @ down
        out.index_add_(0, tok, y * w[tok, slot][:, None])
    return out, idx, w


def _rms64(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x, theta):
    """x [n, heads, head_dim] at positions 0 .. n - 1; the angles as the model
    defines them, in f32."""
    n, _, hd = x.shape
    d = torch.arange(hd // 2, device=DEV, dtype=torch.float64)
    freq = (1.0 / theta ** (2 * d / hd)).float()
    ang = (torch.arange(n, device=DEV).float()[:, None] * freq[None, :]).double()[:, None, :]
    a, b = x[..., :hd // 2], x[..., hd // 2:]
    return torch.cat((a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos()), -1)


def _causal64(q, k, v):
    """One head's causal attention: q, k, v [n, head_dim]."""
    n = q.shape[0]
    s = (q @ k.t().contiguous()) / math.sqrt(q.shape[1])
    s = s.masked_fill(torch.ones((n, n), dtype=torch.bool, device=DEV).triu(1), -math.inf)
    return torch.softmax(s, 1) @ v


def _decoder64(c, seed):
    def weight(which, layer=0):
        return _dense(c, seed, which, layer)

    def project(x, which, layer):
        return x @ weight(which, layer).double().t().contiguous()

    hd = c["head_dim"]
    x = weight(_lib.W_EMBED)[_tokens(c, seed).long()].double()
    n = x.shape[0]
    for layer in range(c["layers"]):
        xn = _rms64(x, weight(_lib.W_IN_NORM, layer))
        q = project(xn, _lib.W_Q, layer).reshape(n, c["heads"], hd)
        k = project(xn, _lib.W_K, layer).reshape(n, c["kv_heads"], hd)
        v = project(xn, _lib.W_V, layer).reshape(n, c["kv_heads"], hd)
        if c["qk_norm"]:
            q, k = _rms64(q, weight(_lib.W_Q_NORM, layer)), _rms64(k, weight(_lib.W_K_NORM, layer))
        q, k = _rope64(q, c["theta"]), _rope64(k, c["theta"])
        share = c["heads"] // c["kv_heads"]
        att = torch.cat([_causal64(q[:, i], k[:, i // share], v[:, i // share])
                         for i in range(c["heads"])], 1)
        x = x + project(att, _lib.W_O, layer)
        x = _moe64(c, seed, layer, _rms64(x, weight(_lib.W_POST_NORM, layer)), x)[0]
    x = _rms64(x[c["T"] - 1:], weight(_lib.W_FINAL_NORM))
    return project(x, _lib.W_LM_HEAD, 0)


def exact(case, seed):
    c = case
    if c["kind"] == "moe_decode":
        x, res = (a.double() for a in _moe_inputs(c, seed))
        rows = [_moe64(c, seed, i, x[i:i + 1], res[i:i + 1]) for i in range(c["layers"])]
        out, idx, w = (torch.cat(p) for p in zip(*rows))
        return out, idx.int(), w
    if c["kind"] == "moe_prefill":
        x, res = (a.double() for a in _moe_inputs(c, seed))
        out, idx, w = _moe64(c, seed, 0, x, res)
        return out, idx.int(), w
    if c["kind"] == "attention":
        q, k, v = (a.double() for a in _attention_inputs(c, seed))
        hd, share, found = c["head_dim"], c["heads"] // c["kv_heads"], []
        for i in range(c["heads"]):
            at = slice((i // share) * hd, (i // share + 1) * hd)
            p = torch.softmax((k[:, at].contiguous() @ q[i]) / math.sqrt(hd), 0)
            found.append(p @ v[:, at].contiguous())
        return torch.stack(found)
    if c["kind"] == "head":
        x, nw, w = (a.double() for a in _head_inputs(c, seed))
        logits = w @ _rms64(x, nw)
        return logits, logits.argmax().reshape(1).int()
    return _decoder64(c, seed)
