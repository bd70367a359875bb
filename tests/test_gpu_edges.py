"""Edge sizes of the dense kernels' tiles, loops and dispatch rules on the GPU,
against the CPU oracle."""
import numpy as np
import pytest

import m1moe_amd as m
from m1moe_amd.decoder import DenseOps
from oracle import oracle as orc

from cases import rel_l2, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops_ctx():
    ctx = m.HIPContext(m.make_shape(128, 8, 2, 64, 64))
    yield ctx, DenseOps(ctx)
    ctx.close()


def bf16(a):
    from m1moe_amd.synth import f32_to_bf16
    return f32_to_bf16(np.asarray(a, np.float32))


@pytest.mark.parametrize("n", [2, 3, 5, 4095, 4097, 32768, 32769, 65539])
@pytest.mark.parametrize("where", ["first", "last", "tie", "nan0"])
def test_argmax_edges(ops_ctx, n, where):
    """The largest value in the first or last element (a group of four or the
    tail after it), tied across the passes, and the NaN rule; exact."""
    ctx, ops = ops_ctx
    x = np.random.default_rng(n).normal(0, 1, n).astype(np.float32)
    if where == "tie":
        x[[n // 2, n - 1]] = 20.0
    else:
        x[0 if where == "first" else n - 1] = 20.0
    if where == "nan0":
        x[0] = np.nan
    dx, di = ctx.to_device(x), ctx.alloc(16)
    say(f"argmax n={n} {where}")
    ops.argmax(dx, n, di)
    ctx.sync()
    assert int(di.download(np.int32, 1)[0]) == orc.argmax(x)
    dx.free()
    di.free()


@pytest.mark.parametrize("n", [4, 64, 4092, 4096, 4100, 8192, 8196])
def test_rmsnorm_edges(ops_ctx, n):
    """Both sides of the register form's limits (8192 elements, multiples of
    four): f32 sums of at most 8196 squares, well inside 1e-6."""
    ctx, ops = ops_ctx
    rng = np.random.default_rng(n)
    x, w = rng.normal(0, 2, n).astype(np.float32), bf16(rng.normal(1, 0.1, n))
    dx, dw, dout = ctx.to_device(x), ctx.to_device(w), ctx.alloc(4 * n)
    say(f"rmsnorm n={n}")
    ops.rmsnorm(dx, dw, dout, n, 1e-5)
    ctx.sync()
    assert rel_l2(dout.download(np.float32), orc.rmsnorm(x, w, 1e-5)) < 1e-6
    for b in (dx, dw, dout):
        b.free()


# ---- router -----------------------------------------------------------------------------


@pytest.mark.parametrize("T", [1, 3, 127, 128, 129, 255, 256, 257, 511, 513])
@pytest.mark.parametrize("name", ["tiny", "tiny_renorm"])
def test_router_tokens_per_wave(name, T):
    """Both sides of every tokens-per-wave rule (8 and 16 experts, one workgroup
    row): logits bit for bit as the oracle's (f64 sums rounded once), top-K
    exact, weights to a few f32 roundings."""
    from cases import make_case
    from m1moe_amd import synth
    from m1moe_amd.engine import MoEBlock
    c = make_case(name, seed=71)
    try:
        E, K = c.shape.num_experts, c.shape.top_k
        x = c.x_bf16(T)
        dx = c.ctx.to_device(x)
        di, dw, dl = c.ctx.alloc(4 * T * K), c.ctx.alloc(4 * T * K), c.ctx.alloc(4 * T * E)
        say(f"router {name} T={T}")
        MoEBlock(c.ctx).router_topk(0, T, dx, "bf16", di, dw, dl)
        c.ctx.sync()
        idx, w = di.download(np.int32).reshape(T, K), dw.download(np.float32).reshape(T, K)
        logits = dl.download(np.float32).reshape(T, E)
        want = (synth.bf16_to_f32(x).astype(np.float64) @
                synth.bf16_to_f32(c.routers[0]).astype(np.float64).T).astype(np.float32)
        assert np.array_equal(logits, want)
        order = np.argsort(-want, axis=1, kind="stable")[:, :K]
        assert np.array_equal(idx, order)
        p = np.exp(want.astype(np.float64) - want.max(1, keepdims=True))
        p = np.take_along_axis(p / p.sum(1, keepdims=True), order, 1)
        if c.shape.norm_topk_prob:
            p /= p.sum(1, keepdims=True)
        assert np.abs(w - p).max() < 1e-6
    finally:
        c.close()


# ---- decode attention -------------------------------------------------------------------


@pytest.mark.parametrize("nh,nkv,hd,sl", [
    # 64 groups on 256 CUs: four workgroups each, chunks of 64 (one batch per wave),
    # 65 .. 96 or 80 (one larger batch) and above (two batches in flight; at head_dim 64
    # 385 .. 512 positions are one workgroup's)
    (64, 64, 64, 256), (64, 64, 64, 257), (64, 64, 64, 384), (64, 64, 64, 385), (64, 64, 64, 513),
    (64, 64, 128, 255), (64, 64, 128, 320), (64, 64, 128, 321), (64, 64, 256, 256),
    (64, 64, 256, 259), (64, 8, 64, 2049), (64, 8, 128, 130), (64, 8, 128, 8191),
    # one position past a chunk, past a wave's batch; more groups than CUs
    (32, 8, 128, 65), (32, 8, 128, 17), (24, 8, 64, 9), (300, 300, 64, 333), (2, 2, 256, 2),
    # eight heads per group: half a batch per wave, a whole one, the larger one
    (8, 1, 128, 1), (8, 1, 128, 32), (8, 1, 128, 33), (64, 8, 128, 2049), (64, 8, 128, 2560),
    (8, 1, 256, 31), (8, 1, 256, 33), (8, 1, 256, 64), (16, 2, 256, 129),
    # one workgroup per group up to 256, 320, 512 positions; more groups than CUs: one up to
    # 256, chunks in the light forms, then of at least 256
    (100, 100, 64, 512), (100, 100, 64, 513), (86, 86, 128, 320), (86, 86, 128, 321), (70, 70, 128, 257),
    (128, 64, 128, 256), (260, 260, 64, 256), (260, 260, 64, 257), (260, 260, 64, 3073), (260, 260, 128, 1281)])
def test_attention_decode_chunk_edges(ops_ctx, nh, nkv, hd, sl):
    """f32 sums of at most 8191 terms against the oracle's f64: 1e-6 (2e-7
    seen), for lengths around every batch and chunk rule; the last V row is
    large, so a position read twice or left out shows."""
    ctx, ops = ops_ctx
    rng = np.random.default_rng(nh * 7 + sl)
    kvd = nkv * hd
    q = rng.normal(0, 1, nh * hd).astype(np.float32)
    kc = rng.normal(0, 1, (sl, kvd)).astype(np.float32)
    vc = rng.normal(0, 1, (sl, kvd)).astype(np.float32)
    vc[-1] *= 100
    dq, dk, dv, dout = ctx.to_device(q), ctx.to_device(kc), ctx.to_device(vc), ctx.alloc(4 * nh * hd)
    say(f"attention nh={nh} nkv={nkv} hd={hd} seq={sl}")
    ops.attention_decode(dq, dk, dv, dout, nh, nkv, hd, sl)
    ctx.sync()
    assert rel_l2(dout.download(np.float32), orc.attention(q, kc, vc, nh, nkv, hd, sl)) < 1e-6
    for b in (dq, dk, dv, dout):
        b.free()


# queries of few bits in one dimension: with keys of 10 bits every dot product is
# exact in f32; at head_dim 64 the scores are 300 to 500 exponents of two
_LARGE_Q = (1920.0, 2176.0, 2304.0)


@pytest.mark.parametrize("nh,nkv,hd,sl", [
    (2, 1, 64, 300), (8, 1, 64, 700), (4, 1, 128, 300), (16, 16, 64, 1000), (8, 1, 256, 700),   # merged in the launch
    (8, 1, 256, 130), (300, 300, 64, 333)])                    # by each group's last workgroup
def test_attention_decode_merges_large_scores(ops_ctx, nh, nkv, hd, sl):
    """Large scores that differ from chunk to chunk by up to 12 exponents of two,
    their dot products exact in f32: what is left is the rounding of the
    exponents (12 x 2^-24 x ln 2), the hardware exp2 (one ulp), the f32 numerators
    and their sums, 5e-7 in all.  Scores or maxima rounded at their own size
    (2^-25 of 400) are off by several 1e-6."""
    ctx, ops = ops_ctx
    rng = np.random.default_rng(nh + sl)
    q = np.zeros((nh, hd), np.float32)
    q[:, 5] = np.array(_LARGE_Q)[np.arange(nh) % 3]
    n = q[:, 5].astype(np.float64) / np.sqrt(hd) * np.log2(np.e)
    p = np.arange(sl)
    kc = rng.normal(0, 1, (sl, nkv, hd)).astype(np.float32)    # (the other dims of q are 0)
    kc[:, :, 5] = (1 - (p * 7 % 16 + 3 * (p // 64) % 16) / 1024)[:, None]
    vc = rng.normal(0, 1, (sl, nkv, hd)).astype(np.float32)
    e = n[:, None] * kc[:, 0, 5].astype(np.float64)
    w = np.exp2(e - e.max(1, keepdims=True))
    w /= w.sum(1, keepdims=True)
    want = np.stack([w[i] @ vc[:, i * nkv // nh].astype(np.float64) for i in range(nh)])
    dq, dk, dv, dout = ctx.to_device(q), ctx.to_device(kc), ctx.to_device(vc), ctx.alloc(4 * nh * hd)
    say(f"attention large scores nh={nh} nkv={nkv} hd={hd} seq={sl}")
    ops.attention_decode(dq, dk, dv, dout, nh, nkv, hd, sl)
    ctx.sync()
    rel = rel_l2(dout.download(np.float32).reshape(nh, hd), want)
    say(f"rel L2 {rel:.2e}")
    assert rel < 5e-7
    for b in (dq, dk, dv, dout):
        b.free()


def test_decoder_step_merges_large_scores():
    """The same through a decoder step, 5 chunks (merged by o_proj while it
    stages its input) and 10 (in the attention launch): embeddings of +-1 and
    eps 0 make the projections' input exactly +-1, a RoPE base of 1e30 leaves the
    last pair of a head unrotated, zeroed experts leave the residual.  Bound: the
    attention's 5e-7 and the f32 sums of v, o_proj, norm and lm_head."""
    from test_gpu_decoder import Pair, _zero_experts
    from m1moe_amd import _lib, synth
    from m1moe_amd.synth import bf16_to_f32
    wl = synth.DecoderWorkload("wide", synth.CONFIGS["tiny"], 1, 300, 2, 1, 64, 1e30, False, 8, 8,
                               rms_eps=0.0)
    p = Pair(wl, seed=64, max_seq=700)
    try:
        _zero_experts(p)
        h, hd, D = 128, 64, 31
        rng = np.random.default_rng(64)
        emb = rng.choice([-1.0, 1.0], (wl.vocab, h))
        emb[:, :4] = 1
        emb[:, 4:10] = 1 - 2 * (np.arange(wl.vocab)[:, None] >> np.arange(6) & 1)
        wq, wk = np.zeros((2 * hd, h)), np.zeros((hd, h))
        wq[[D, hd + D], 0] = _LARGE_Q[1:]
        wk[D, 3] = 1 - 2.0 ** -4
        wk[D, 4:10] = 2.0 ** -np.arange(10, 4, -1)   # (keys of 10 bits)
        ones, val = np.ones(h), {}
        for which, a in ((_lib.W_EMBED, emb), (_lib.W_IN_NORM, ones), (_lib.W_POST_NORM, ones),
                         (_lib.W_FINAL_NORM, ones), (_lib.W_Q, wq), (_lib.W_K, wk),
                         (_lib.W_V, rng.normal(0, 1, (hd, h))), (_lib.W_O, rng.normal(0, 0.1, (h, 2 * hd))),
                         (_lib.W_LM_HEAD, rng.normal(0, 0.1, (wl.vocab, h)))):
            p.dec.upload(which, 0, bf16(a))
            val[which] = bf16_to_f32(bf16(a)).astype(np.float64)
        toks = np.array([i * 7 % 16 + 3 * (i // 64) % 16 + 64 * (i % 4) for i in range(640)], np.int32)
        for n in (300, 620):
            p.dec.reset()
            p.dec.prefill(toks[:n - 1])
            say(f"step {n}")
            _, got = p.dec.forward(int(toks[n - 1]), return_logits=True)
            x = val[_lib.W_EMBED][toks[:n]]
            k, v = x @ val[_lib.W_K].T, x @ val[_lib.W_V].T
            q = (val[_lib.W_Q] @ x[-1]).reshape(2, hd)
            e = q @ k.T / 8 * np.log2(np.e)
            w = np.exp2(e - e.max(1, keepdims=True))
            att = (w / w.sum(1, keepdims=True)) @ v
            y = x[-1] + val[_lib.W_O] @ att.reshape(-1)
            rel = rel_l2(got, val[_lib.W_LM_HEAD] @ (y / np.sqrt((y * y).mean())))
            say(f"rel L2 {rel:.2e}")
            assert rel < 1e-6
    finally:
        p.close()


def test_decoder_steps_in_a_long_cache():
    """A cache of 5000 positions shared by 16 workgroups per head: the chunk
    grows with the position (64 up to 1024 positions, then more), the
    deferred, the synchronous and the single-chunk forms in turn."""
    from test_gpu_decoder import Pair, _zero_experts
    from m1moe_amd import synth
    wl = synth.DecoderWorkload("longcache", synth.CONFIGS["tiny_renorm"], 1, 300, 16, 16, 64,
                               1e4, True, 8, 8)
    p = Pair(wl, seed=63, max_seq=5000)
    try:
        _zero_experts(p)
        toks = synth.prompt_tokens(wl, 7, 1100)
        off = 0
        for n, steps in ((60, 8), (190, 4), (800, 3), (20, 3)):
            _prefill_matches(p, toks[off:], (n,))
            off += n
            for t in toks[off:off + steps]:
                say(f"step at position {off}")
                _, g_lg = p.dec.forward(int(t), return_logits=True)
                _, w_lg = p.orc.step(int(t))
                assert rel_l2(g_lg, w_lg) < 1e-5
            off += steps
    finally:
        p.close()


@pytest.mark.parametrize("hd", [64, 128, 256])
def test_decoder_steps_eight_heads_per_group(hd):
    """Steps of 8 q heads over one kv head at the first positions, around the end
    of half a wave's batch, of a batch and of a chunk, and over several chunks."""
    from test_gpu_decoder import Pair, _zero_experts
    from m1moe_amd import synth
    wl = synth.DecoderWorkload("eight", synth.CONFIGS["tiny_renorm"], 1, 300, 8, 1, hd, 1e4, True, 8, 8)
    p = Pair(wl, seed=65, max_seq=300)
    try:
        _zero_experts(p)
        toks = synth.prompt_tokens(wl, 9, 300)
        at = 0
        for stop, steps in ((3, 2), (31, 3), (63, 3), (128, 2), (255, 3)):
            say(f"prefill {at} .. {stop}, then {steps} steps")
            p.dec.prefill(toks[at:stop])
            for t in toks[at:stop]:
                p.orc.step(int(t))
            for t in toks[stop:stop + steps]:
                _, g_lg = p.dec.forward(int(t), return_logits=True)
                _, w_lg = p.orc.step(int(t))
                assert rel_l2(g_lg, w_lg) < 1e-5
            at = stop + steps
    finally:
        p.close()


@pytest.mark.parametrize("heads,kv,hd,steps", [(24, 24, 64, (2, 62, 126, 254, 256, 258)), (32, 16, 128, (126, 128)),
                                               (32, 32, 128, (255, 256))])
def test_decoder_steps_around_one_workgroup(heads, kv, hd, steps):
    """Steps of a long cache around the positions up to which one workgroup takes
    all of a group (256; 128 with 16 groups of two), with the early and the shared
    forms on both sides."""
    from test_gpu_decoder import Pair, _zero_experts
    from m1moe_amd import synth
    wl = synth.DecoderWorkload("one", synth.CONFIGS["tiny"], 1, 300, heads, kv, hd, 1e4, True, 8, 8)
    p = Pair(wl, seed=66, max_seq=4000)
    try:
        _zero_experts(p)
        toks = synth.prompt_tokens(wl, 10, 300)
        at = 0
        for stop in steps:
            say(f"{heads}/{kv}/{hd}: step at {stop}")
            if stop > at:
                p.dec.prefill(toks[at:stop])
            for t in toks[at:stop]:
                p.orc.step(int(t))
            _, g_lg = p.dec.forward(int(toks[stop]), return_logits=True)
            _, w_lg = p.orc.step(int(toks[stop]))
            assert rel_l2(g_lg, w_lg) < 1e-5
            at = stop + 1
    finally:
        p.close()


# ---- prefill attention ------------------------------------------------------------------


def _prefill_matches(p, toks, Ts):
    """The prompts' last logits against the oracle's token-by-token run: with
    the MoE block zeroed every operation is an f32 sum, held to 1e-5 as the
    other dense prefill tests hold it."""
    off = 0
    for T in Ts:
        say(f"prefill T={T} at position {off}")
        _, g_lg = p.dec.prefill(toks[off:off + T], return_logits=True)
        for t in toks[off:off + T]:
            _, w_lg = p.orc.step(int(t))
        off += T
        assert np.all(np.isfinite(g_lg))
        rel = rel_l2(g_lg, w_lg)
        assert rel < 1e-5, f"T={T}: rel L2 {rel:.2e}"


@pytest.mark.parametrize("heads,kv,hd,Ts", [(2, 1, 64, (31,)), (2, 1, 64, (32, 1, 32)),
                                            (3, 3, 64, (33, 95)), (8, 2, 128, (129,)),
                                            (16, 4, 128, (64, 3, 127)), (24, 8, 64, (40,))])
def test_prefill_attention_tile_edges(heads, kv, hd, Ts):
    """32-query tiles and 32-key blocks one short of, at and past their edges,
    behind an earlier context too, heads in and not in multiples of 8; two
    layers, so that every query's output reaches the last logits."""
    from test_gpu_decoder import Pair, _zero_experts
    from m1moe_amd import synth
    wl = synth.DecoderWorkload("edges", synth.CONFIGS["tiny_renorm"], 2, 300, heads, kv, hd,
                               1e4, True, 8, 8)
    p = Pair(wl, seed=61, max_seq=sum(Ts))
    try:
        _zero_experts(p)
        _prefill_matches(p, synth.prompt_tokens(wl, 3, sum(Ts)), Ts)
    finally:
        p.close()


@pytest.mark.parametrize("heads,kv,qk_norm,Ts", [(2, 1, True, (17, 33)), (4, 4, False, (1, 16, 31)),
                                                 (3, 1, True, (50,))])
def test_prefill_head_dim_256(heads, kv, qk_norm, Ts):
    """RoPE rows with two pairs per lane and the SIMD attention's outputs in pairs,
    16-query tiles one short of, at and past their edge, behind an earlier
    context; two layers, so that every query's output reaches the last logits."""
    from test_gpu_decoder import Pair, _zero_experts
    from m1moe_amd import synth
    wl = synth.DecoderWorkload("hd256", synth.CONFIGS["tiny_renorm"], 2, 300, heads, kv, 256, 1e4, qk_norm, 8, 8)
    p = Pair(wl, seed=68, max_seq=sum(Ts))
    try:
        _zero_experts(p)
        _prefill_matches(p, synth.prompt_tokens(wl, 6, sum(Ts)), Ts)
    finally:
        p.close()


@pytest.mark.parametrize("hidden", [4096, 4160, 8192])
def test_prefill_row_norms_of_wide_rows(hidden):
    """Both sides of the row norms' register forms (4096, 8192 values a row)."""
    from test_gpu_decoder import Pair, _zero_experts
    from m1moe_amd import synth
    moe = synth.Workload("wide", dict(hidden=hidden, num_experts=2, top_k=1, intermediate=64, group_size=64,
                                      norm_topk_prob=False))
    wl = synth.DecoderWorkload("wide_rows", moe, 1, 300, 2, 1, 64, 1e4, True, 8, 8)
    p = Pair(wl, seed=69, max_seq=12)
    try:
        _zero_experts(p)
        _prefill_matches(p, synth.prompt_tokens(wl, 7, 12), (5, 7))
    finally:
        p.close()


def test_prefill_large_gemm_tile_over_three_segments():
    """1100 x 6144 x 512: nine rows of 24 tiles of 128 x 256 over q, k and v, the
    last one ragged; K and V of every token reach the last logits."""
    from test_gpu_decoder import Pair, _zero_experts
    from m1moe_amd import synth
    moe = synth.Workload("qkv", dict(hidden=512, num_experts=2, top_k=1, intermediate=64, group_size=64,
                                     norm_topk_prob=False))
    wl = synth.DecoderWorkload("segments", moe, 1, 300, 16, 16, 128, 1e4, True, 8, 8)
    p = Pair(wl, seed=70, max_seq=1100)
    try:
        _zero_experts(p)
        _prefill_matches(p, synth.prompt_tokens(wl, 8, 1100), (1100,))
    finally:
        p.close()


def test_prefill_large_gemm_tile_ragged_with_residual():
    """o_proj of 1700 x 4096 x 4096 (14 x 16 tiles of 128 x 256, the last row
    ragged) with the residual and the row norm, against the same prompt in
    pieces of 400 (64 x 128 tiles): f32 sums in another order, 1e-5.  Two layers, so
    that every row reaches the last logits through the second layer's K and V."""
    from m1moe_amd import synth
    from m1moe_amd.decoder import Decoder
    wl = synth.DECODERS["cfg4"]
    shape = synth.Workload("wide", dict(hidden=4096, num_experts=2, top_k=1, intermediate=64, group_size=64,
                                        norm_topk_prob=False)).shape(2)
    ctx = m.HIPContext(shape)
    try:
        for l in range(2):
            ctx.upload_layer_experts(l, np.zeros_like(synth.layer_image(shape, 71, l)))
            ctx.upload_router(l, synth.router(shape, 71, l))
        dec = Decoder(ctx, wl.dec_shape(1700))
        dec.upload_all(lambda which, l: synth.dense_weight(wl, 71, which, l))
        toks = synth.prompt_tokens(wl, 11, 1700)
        say("1700 tokens at once")
        _, whole = dec.prefill(toks, return_logits=True)
        dec.reset()
        for at in range(0, 1700, 400):
            say(f"tokens from {at}")
            _, pieces = dec.prefill(toks[at:at + 400], return_logits=True)
        assert np.all(np.isfinite(whole)) and rel_l2(whole, pieces) < 1e-5
        dec.close()
    finally:
        ctx.close()


def test_prefill_past_the_cache_reads_its_own_queries():
    """Tokens past the cache's end are reported; their logits come from this
    call's projections, not from what an earlier prompt left in the scratch
    (hidden 512: the q/k/v GEMM leaves split partials, summed by the RoPE rows)."""
    import m1moe_amd as m
    from test_gpu_decoder import Pair, _zero_experts
    from m1moe_amd import synth
    moe = synth.Workload("wide", dict(hidden=512, num_experts=4, top_k=1, intermediate=64, group_size=64,
                                      norm_topk_prob=False))
    wl = synth.DecoderWorkload("past", moe, 1, 300, 8, 2, 64, 1e4, True, 8, 8)
    p = Pair(wl, seed=67, max_seq=16)
    try:
        _zero_experts(p)
        found = []
        for seed in (1, 2):
            p.dec.prefill(synth.prompt_tokens(wl, seed, 16))
            p.dec.reset()
            p.dec.prefill(synth.prompt_tokens(wl, 3, 4))
            toks, lg, nx = p.ctx.to_device(synth.prompt_tokens(wl, 4, 16)), p.ctx.alloc(4 * 300), p.ctx.alloc(16)
            say(f"16 tokens at position 4 of 16, after prompt {seed}")
            p.dec.prefill_device(toks, 16, nx, lg)
            with pytest.raises(m.M1MoEError):
                p.ctx.sync()
            found.append(lg.download(np.float32, 300).copy())
            p.dec.reset()
        assert np.all(np.isfinite(found[0])) and np.array_equal(*found)
    finally:
        p.close()


def test_prefill_attention_keys_past_the_split():
    """A K value of 3.397e38 rounds to infinity in bf16 (its parts would add up
    to NaN): the wave's blocks are multiplied on f32 MFMA instead.  eps 0 and
    an embedding of ones make the projections' input exactly 1; queries of
    2e-38 keep the scores below 1."""
    from test_gpu_decoder import Pair, _zero_experts
    from m1moe_amd import _lib, synth
    wl = synth.DecoderWorkload("huge", synth.CONFIGS["tiny"], 1, 300, 2, 1, 64, 1e4, False, 8, 8,
                               rms_eps=0.0)
    p = Pair(wl, seed=62, max_seq=48)
    try:
        _zero_experts(p)
        h, kvd, qd = 128, 64, 128
        wq, wk = np.zeros((qd, h), np.float32), np.zeros((kvd, h), np.float32)
        wq[[0, 64], 0] = 2e-38
        wk[0, 0], wk[0, 1] = 3.3895e38, 8e35
        new = {(_lib.W_EMBED, "embed"): np.ones((wl.vocab, h)), (_lib.W_IN_NORM, "in_norm"): np.ones(h),
               (_lib.W_Q, "q"): wq, (_lib.W_K, "k"): wk}
        for (which, name), a in new.items():
            bits = bf16(a)
            p.dec.upload(which, 0, bits)
            if which in _lib.W_PER_LAYER:
                p.orc.t[name][0] = bits
            else:
                p.orc.t[name] = bits
        _prefill_matches(p, synth.prompt_tokens(wl, 5, 45), (40, 5))
        assert float(np.abs(p.orc.kc).max()) > 3.396e38
    finally:
        p.close()
