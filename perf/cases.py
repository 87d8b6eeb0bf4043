"""The work this library is run for, as cases to time: decode of one token, verification of a few tokens, prefill blocks and the
output head of the model the library serves (hidden 2816, 128 int4 experts of 704 with top-8 routing, a shared expert of 2112,
sliding-window layers of 16 query heads on 8 kv heads of 256 and every sixth layer global with 16 on 2 of 512, vocabulary 262144).

A case is a dict with a "kind":

  step    the routed-experts block of one token through `layers` layers, call by call (tf_moe_decode_step)
  token   one token from its id through `layers` whole decoder layers to fp16 logits, replayed from a HIP graph recorded at set-up,
          with `context` tokens already in the KV caches
  head    what follows the last layer: `mode` greedy (the fused argmax head) or sampled (logits, softcap + softmax, top-64 / top-p)
  verify  `tokens` rows through router, 8-of-128 experts and reduce in one call (speculative decoding checks 2 to 32 rows at once)
  block   a prefill block of `tokens` rows at position `start` through one whole layer, sliding-window or global
  attend  the attention of a prefill block alone, at positions where it outweighs the rest of the layer

Weights, caches and inputs are synthetic: uniform codes with zero-mean affine groups, routers whose logits have a standard deviation
of about one, token rows that share a common direction (which is what makes some experts popular: about 10 of 128 experts take half
of the pairs).  Each pass reads more than the last-level cache holds, or three states in turn do, as in a model of 30 layers.
"""
from __future__ import annotations

import ctypes as C
import importlib
import math

import numpy as np
import torch

tfk = importlib.import_module("turbo-fieldfare_amd")

D, F_MOE, F_SHARED, E, TOPK, VOCAB = 2816, 704, 2112, 128, 8, 262144
EPS = 1e-6
WINDOW, RING = 1024, 1152
# (head_dim, query heads, kv heads, window or 0, RoPE base, rotated pairs)
SLIDING = dict(hd=256, nq=16, nkv=8, window=WINDOW, theta=1e4, pairs=128)
GLOBAL = dict(hd=512, nq=16, nkv=2, window=0, theta=1e6, pairs=64)


# ---- the cases ---------------------------------------------------------------------------------------------------------------
def listed():
    return [
        # the headline loop: batch-1 routed experts, launched call by call; latency and launches count
        dict(name="step_6_layers", kind="step", layers=6, scales="bf16"),
        # generation: the whole model, a conversation of ordinary length
        dict(name="token_30_layers", kind="token", layers=30, context=1899, scales="bf16"),
        # generation deep into a long context: the global layer reads 32 K rows; fp16 scales
        dict(name="token_6_layers_long", kind="token", layers=6, context=32767, scales="fp16"),
        # the two output heads: greedy decoding and sampling
        dict(name="head_greedy", kind="head", mode="greedy", vocab=VOCAB, scales="bf16"),
        dict(name="head_sampled", kind="head", mode="sampled", vocab=VOCAB, scales="bf16"),
        # speculative decoding: a short and an ordinary draft
        dict(name="verify_3", kind="verify", tokens=3, scales="bf16"),
        dict(name="verify_16", kind="verify", tokens=16, scales="bf16"),
        # the ragged last block of a prompt, 8-bit shared expert
        dict(name="block_53", kind="block", tokens=53, start=1152, attention="sliding", shared_bits=8, scales="bf16"),
        # the block size the reference prefills with
        dict(name="block_128", kind="block", tokens=128, start=3968, attention="sliding", shared_bits=4, scales="bf16"),
        # larger blocks: a global layer with fp16 scales, and the throughput size
        dict(name="block_500_global", kind="block", tokens=500, start=1500, attention="global", shared_bits=4, scales="fp16"),
        dict(name="block_2048", kind="block", tokens=2048, start=0, attention="sliding", shared_bits=4, scales="bf16"),
        # long prompts: a block's global attention over 32 K keys
        dict(name="attend_128_at_32k", kind="attend", tokens=128, start=32640, attention="global"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("step", "token", "head", "verify", "block", "block", "attend"))
    scales = rng.choice(("bf16", "fp16"))
    if kind == "step":
        return dict(kind=kind, layers=rng.randint(5, 30), scales=scales)
    if kind == "token":
        return dict(kind=kind, layers=rng.randint(2, 24), context=_log_int(rng, 1, 32767), scales=scales)
    if kind == "head":
        return dict(kind=kind, mode=rng.choice(("greedy", "sampled")), vocab=_log_int(rng, 32768, VOCAB), scales=scales)
    if kind == "verify":
        return dict(kind=kind, tokens=rng.randint(2, 32), scales=scales)
    attention = rng.choice(("sliding", "global"))
    if kind == "block":
        most_tokens, most_start = (1024, 2048) if attention == "global" else (2048, 4096)
        return dict(kind=kind, tokens=_log_int(rng, 33, most_tokens), start=rng.choice((0, _log_int(rng, 16, most_start))), attention=attention,
                    shared_bits=rng.choice((4, 4, 8)), scales=scales)
    return dict(kind=kind, tokens=rng.randint(32, 160), start=_log_int(rng, 2000, 24000), attention=attention)


# ---- synthetic weights -------------------------------------------------------------------------------------------------------
def _generator(seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed * 1000003 + 17)
    return gen


def _codes(gen, nbytes):
    """nbytes of uniform random bits."""
    return torch.randint(-(1 << 31), 1 << 31, ((nbytes + 3) // 4,), dtype=torch.int32, device="cuda", generator=gen).view(torch.uint8)[:nbytes]


def _dtype(scales):
    return torch.float16 if scales == "fp16" else torch.bfloat16


def _affine(gen, shape, bits, scales, lo=None, hi=None):
    """Scales and biases that make uniform `bits`-bit codes weights of mean about zero."""
    lo, hi = (lo, hi) if lo is not None else ((0.005, 0.02) if bits == 4 else (0.0003, 0.0012))
    s = (torch.rand(shape, device="cuda", generator=gen) * (hi - lo) + lo).to(_dtype(scales))
    b = s.float() * (-7.5 if bits == 4 else -127.5) + (torch.rand(shape, device="cuda", generator=gen) - 0.5) * 0.02
    return s, b.to(_dtype(scales))


def _matrix(gen, rows, cols, bits=4, scales="bf16", lo=None, hi=None):
    W = _codes(gen, rows * cols * bits // 8).view(rows, cols * bits // 8)
    return (W, *_affine(gen, (rows, cols // 64), bits, scales, lo, hi))


def _norm(gen, n, lo=0.9, hi=1.1, signed=False):
    w = torch.rand(n, device="cuda", generator=gen) * (hi - lo) + lo
    if signed:
        w = w * (torch.randint(0, 2, (n,), device="cuda", generator=gen) * 2 - 1)
    return w.to(torch.bfloat16)


def _expert_layout():
    """Byte offsets of gate W,S,B, up W,S,B, down W,S,B in one expert's blob, and the blob's stride."""
    offsets, at = [], 0
    for rows, cols in ((F_MOE, D), (F_MOE, D), (D, F_MOE)):
        for nbytes in (rows * cols // 2, rows * (cols // 64) * 2, rows * (cols // 64) * 2):
            offsets.append(at)
            at += nbytes
    return offsets, (at + 16383) // 16384 * 16384


OFFSETS, STRIDE = _expert_layout()


def _experts(gen, scales):
    """One layer's router and its pool of resident experts."""
    pool = _codes(gen, E * STRIDE).view(E, STRIDE)
    for p, (rows, cols) in enumerate(((F_MOE, D), (F_MOE, D), (D, F_MOE))):
        n = rows * (cols // 64)
        for j, t in enumerate(_affine(gen, (E, n), 4, scales)):
            at = OFFSETS[3 * p + 1 + j]
            pool[:, at:at + 2 * n] = t.view(torch.uint8).view(E, 2 * n)
    W, S, B = _matrix(gen, E, D, 8, "bf16", 0.008, 0.03)
    eff = (torch.rand(D, device="cuda", generator=gen) + 0.5).div(D ** 0.5).to(torch.bfloat16)
    gain = (torch.rand(E, device="cuda", generator=gen) * 0.8 + 0.6).to(torch.bfloat16)
    return dict(pool=pool, W=W, S=S, B=B, eff=eff, gain=gain)


def _layer(gen, geo, scales, shared_bits=4):
    """One whole decoder layer's weights."""
    q, kv = geo["nq"] * geo["hd"], geo["nkv"] * geo["hd"]
    w = dict(q=_matrix(gen, q, D, 4, scales), k=_matrix(gen, kv, D, 4, scales), v=_matrix(gen, kv, D, 4, scales), o=_matrix(gen, D, q, 4, scales),
             gate=_matrix(gen, F_SHARED, D, shared_bits, scales), up=_matrix(gen, F_SHARED, D, shared_bits, scales),
             down=_matrix(gen, D, F_SHARED, shared_bits, scales))
    for name in ("input_norm", "pre_ffn", "pre_ffn2"):
        w[name] = _norm(gen, D)
    for name in ("post_attn", "post_ffn1", "post_ffn2", "post_ffn"):      # what a branch adds to the residual stream is small
        w[name] = _norm(gen, D, 0.05, 0.07, signed=True)
    w["q_norm"], w["k_norm"] = _norm(gen, geo["hd"]), _norm(gen, geo["hd"])
    w["experts"] = _experts(gen, scales)
    w["projections"] = [tfk.projection(*w[n], r, c) for n, r, c in (("gate", F_SHARED, D), ("up", F_SHARED, D), ("down", D, F_SHARED))]
    return w


def _rows(gen, tokens):
    """Token rows of unit variance with a common direction."""
    common = torch.randn((1, D), device="cuda", generator=gen)
    return ((torch.randn((tokens, D), device="cuda", generator=gen) + common) / 2 ** 0.5).to(torch.float16)


def _half(gen, *shape):
    return torch.randn(shape, device="cuda", generator=gen).to(torch.float16)


def _zeros(*shape, dtype=torch.float16):
    return torch.zeros(shape, dtype=dtype, device="cuda")


def _abc(m):
    return [m[0].data_ptr(), 0, m[1].data_ptr(), 0, m[2].data_ptr(), 0]


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _scale_code(case):
    return tfk.TF_FP16 if case["scales"] == "fp16" else tfk.TF_BF16


# ---- preparation and passes, kind by kind ------------------------------------------------------------------------------------
def prepare(case, seed):
    gen = _generator(seed)
    state = dict(case=case, ctx=tfk.Context(0), off=tfk.ExpertOffsets(*OFFSETS))
    state.update(_KINDS[case["kind"]][0](case, gen, state))
    return state


def run(state):
    return _KINDS[state["case"]["kind"]][1](state)


def _prepare_step(case, gen, state):
    n = case["layers"]
    return dict(layers=[_experts(gen, case["scales"]) for _ in range(n)], x=_rows(gen, n), residual=_half(gen, n, D), acts=_zeros(TOPK * F_MOE),
                y=_zeros(n, D), idx=_zeros(n, TOPK, dtype=torch.int32), wts=_zeros(n, TOPK), code=_scale_code(case))


def _run_step(s):
    k = s["ctx"]
    x, y, residual, idx, wts = (s[n].data_ptr() for n in ("x", "y", "residual", "idx", "wts"))
    acts, off, code, stream, step = s["acts"].data_ptr(), C.byref(s["off"]), s["code"], _stream(), k.lib.tf_moe_decode_step
    for i, e in enumerate(s["layers"]):
        row = i * D * 2
        k.check(step(k.handle, stream, *_abc((e["W"], e["S"], e["B"])), x + row, e["eff"].data_ptr(), 0, e["gain"].data_ptr(), 0,
                     e["pool"].data_ptr(), STRIDE, E, off, x + row, acts, residual + row, y + row, idx + i * TOPK * 4, wts + i * TOPK * 2,
                     D, F_MOE, TOPK, code))
    return dict(y=s["y"], experts=s["idx"], weights=s["wts"])


def _prepare_token(case, gen, state):
    geos = [GLOBAL if i % 6 == 5 else SLIDING for i in range(case["layers"])]
    layers, position = [], case["context"]
    for geo in geos:
        w = _layer(gen, geo, case["scales"])
        rows = RING if geo["window"] else position + 1                    # a ring for the window, all positions for a global layer
        w["k_cache"], w["v_cache"] = _half(gen, rows, geo["nkv"], geo["hd"]), _half(gen, rows, geo["nkv"], geo["hd"])
        layers.append(w)
    s = dict(geos=geos, layers=layers, table=_matrix(gen, VOCAB, D), final_norm=_norm(gen, D), logits=_zeros(VOCAB), hidden=_zeros(D),
             hidden_alt=_zeros(D), q=_zeros(16 * 512), attn=_zeros(16 * 512), o=_zeros(D), dense_x=_zeros(D), routed_x=_zeros(D), router_x=_zeros(D),
             shared=_zeros(D), h2=_zeros(D), zero=_zeros(D), sg=_zeros(F_SHARED), su=_zeros(F_SHARED), sa=_zeros(F_SHARED), acts=_zeros(TOPK * F_MOE),
             idx=_zeros(TOPK, dtype=torch.int32), wts=_zeros(TOPK), token=int(torch.randint(0, VOCAB, (1,), device="cuda", generator=gen)))
    state = dict(state, **s)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _token_calls(state, position)
        side.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"], stream=side):
            _token_calls(state, position)
    torch.cuda.current_stream().wait_stream(side)
    s["new_rows"] = [(w["k_cache"][position % RING if g["window"] else position], w["v_cache"][position % RING if g["window"] else position])
                     for g, w in zip(geos, layers)]
    return s


def _token_calls(s, position):
    """One token: embedding row, the layers (eight launches each), final norm and logits; nothing on the host in between."""
    k, code, st = s["ctx"], _scale_code(s["case"]), _stream()
    lib, h = k.lib, k.handle
    p = lambda name: s[name].data_ptr()
    k.check(lib.tf_embed_lookup_int4(h, st, *_abc(s["table"]), p("hidden"), 0, s["token"], D, D ** 0.5, VOCAB))
    before = None
    for geo, w in zip(s["geos"], s["layers"]):
        hd, nq, nkv = geo["hd"], geo["nq"], geo["nkv"]
        ptr = lambda name: w[name].data_ptr()
        row = (position % RING if geo["window"] else position) * nkv * hd * 2
        qkv = _abc(w["q"]) + _abc(w["k"]) + _abc(w["v"])
        out = (p("q"), 0, ptr("k_cache"), row, ptr("v_cache"), row, nq * hd, nkv * hd, D, code)
        if before is None:
            k.check(lib.tf_fused_norm_qkv_gemv(h, st, ptr("input_norm"), 0, EPS, *qkv, p("hidden"), *out))
        else:
            k.check(lib.tf_fused_layer_tail_norm_qkv_gemv(h, st, p("h2"), p("shared"), p("hidden_alt"), p("hidden"), before["post_ffn1"].data_ptr(), 0,
                                                          before["post_ffn2"].data_ptr(), 0, before["post_ffn"].data_ptr(), 0, EPS, 1.0,
                                                          ptr("input_norm"), 0, EPS, *qkv, *out))
        k.check(lib.tf_fused_qkv_epilogue(h, st, p("q"), 0, ptr("k_cache"), row, ptr("v_cache"), row, ptr("q_norm"), 0, ptr("k_norm"), 0, hd, nq, nkv,
                                          position, geo["theta"], geo["pairs"], EPS))
        if geo["window"]:
            k.check(lib.tf_attention_swa(h, st, p("q"), 0, ptr("k_cache"), 0, ptr("v_cache"), 0, p("attn"), 0, hd, nq, nkv, position + 1, WINDOW,
                                         hd ** -0.5, RING))
        else:
            k.check(lib.tf_attention_full(h, st, p("q"), 0, ptr("k_cache"), 0, ptr("v_cache"), 0, p("attn"), 0, hd, nq, nkv, position + 1, hd ** -0.5))
        k.check(lib.tf_dequant_int4_gemv(h, st, *_abc(w["o"]), p("attn"), 0, p("o"), 0, D, nq * hd, code, tfk.TF_FP16))
        e = w["experts"]
        gate, up, down = w["projections"]
        k.check(lib.tf_moe_decode_step_shared_post_attn(
            h, st, p("hidden"), p("o"), p("hidden_alt"), ptr("post_attn"), 0, ptr("pre_ffn"), 0, ptr("pre_ffn2"), 0, EPS,
            *_abc((e["W"], e["S"], e["B"])), p("router_x"), e["eff"].data_ptr(), 0, e["gain"].data_ptr(), 0, e["pool"].data_ptr(), STRIDE, E,
            C.byref(s["off"]), p("routed_x"), p("acts"), p("zero"), p("h2"), p("idx"), p("wts"), D, F_MOE, TOPK, code, p("dense_x"), C.byref(gate),
            C.byref(up), C.byref(down), p("shared"), p("sg"), p("su"), p("sa")))
        before = w
    k.check(lib.tf_fused_layer_tail_shared_norm(h, st, p("h2"), p("shared"), p("hidden_alt"), before["post_ffn1"].data_ptr(), 0,
                                                before["post_ffn2"].data_ptr(), 0, before["post_ffn"].data_ptr(), 0, D, EPS, 1.0))
    k.check(lib.tf_lm_head_logits_int4(h, st, p("hidden_alt"), 0, p("final_norm"), 0, *_abc(s["table"]), p("logits"), 0, D, VOCAB, EPS, tfk.TF_BF16,
                                       tfk.TF_FP16))


def _run_token(s):
    s["graph"].replay()
    return dict(logits=s["logits"], hidden=s["hidden_alt"], rows=s["new_rows"][-2:])


def _prepare_head(case, gen, state):
    v = case["vocab"]
    return dict(hidden=_rows(gen, 1), norm=_norm(gen, D), table=_matrix(gen, v, D, 4, case["scales"], 0.003, 0.012), logits=_zeros(v), probs=_zeros(v),
                token=_zeros(1, dtype=torch.int32), code=_scale_code(case))


def _run_head(s):
    k, v, st = s["ctx"], s["case"]["vocab"], _stream()
    if s["case"]["mode"] == "greedy":
        k.lm_head_greedy(s["hidden"], s["norm"], *s["table"], s["token"], D, v, EPS, s["code"])
        return dict(token=s["token"])
    k.lm_head_logits(s["hidden"], s["norm"], *s["table"], s["logits"], D, v, EPS, s["code"], tfk.TF_FP16)
    k.check(k.lib.tf_logit_softcap_softmax(k.handle, st, s["logits"].data_ptr(), s["probs"].data_ptr(), v, 30.0, tfk.TF_FP16))
    k.check(k.lib.tf_sample_topk64(k.handle, st, s["probs"].data_ptr(), s["token"].data_ptr(), v, 0.8, 0.95, 1234567))
    return dict(logits=s["logits"], probs=s["probs"], token=s["token"])


def _prepare_verify(case, gen, state):
    t = case["tokens"]
    return dict(experts=_experts(gen, case["scales"]), x=_rows(gen, t), idx=_zeros(t, TOPK, dtype=torch.int32), wts=_zeros(t, TOPK),
                acts=_zeros(t * TOPK * F_MOE), partials=_zeros(t, TOPK, D), h2=_zeros(t, D), code=_scale_code(case))


def _run_verify(s):
    k, e, t, x = s["ctx"], s["experts"], s["case"]["tokens"], s["x"].data_ptr()
    k.check(k.lib.tf_prefill_routed_moe_few_tokens(
        k.handle, _stream(), *_abc((e["W"], e["S"], e["B"])), x, 0, e["eff"].data_ptr(), 0, e["gain"].data_ptr(), 0, s["idx"].data_ptr(), 0,
        s["wts"].data_ptr(), 0, t, E, D, TOPK, D, x, 0, D, e["pool"].data_ptr(), STRIDE, C.byref(s["off"]), s["acts"].data_ptr(),
        s["partials"].data_ptr(), s["h2"].data_ptr(), 0, F_MOE, s["code"]))
    return dict(h2=s["h2"], partials=s["partials"], experts=s["idx"], weights=s["wts"])


def _attention_params(geo, tokens, start):
    q, kv = geo["nq"] * geo["hd"], geo["nkv"] * geo["hd"]
    return tfk.PrefillAttentionParams(start, tokens, geo["hd"], geo["nq"], geo["nkv"], start + tokens, geo["window"], kv, q, q, geo["hd"] ** -0.5)


def _geometry(case):
    return GLOBAL if case["attention"] == "global" else SLIDING


def _prepare_block(case, gen, state):
    t, start, geo = case["tokens"], case["start"], _geometry(case)
    state["ctx"].reserve(max_block_tokens=t, max_attention_block_tokens=t)
    n, q = t * TOPK, geo["nq"] * geo["hd"]
    cap = E + n // 64 + 1
    i32 = dict(dtype=torch.int32)
    return dict(geo=geo, w=_layer(gen, geo, case["scales"], case["shared_bits"]), hidden_in=_rows(gen, t), hidden=_zeros(t, D), x_norm=_zeros(t, D),
                q=_zeros(t, q), attn=_zeros(t, q), o=_zeros(t, D), dense_x=_zeros(t, D), routed_x=_zeros(t, D), router_x=_zeros(t, D), shared=_zeros(t, D),
                h1=_zeros(t, D), h2=_zeros(t, D), k_cache=_half(gen, start + t, geo["nkv"], geo["hd"]), v_cache=_half(gen, start + t, geo["nkv"], geo["hd"]),
                idx=_zeros(t, TOPK, **i32), wts=_zeros(t, TOPK), pairs=_zeros(n * 4, **i32), offsets=_zeros(E, **i32), counts=_zeros(E, **i32),
                chunks=_zeros(cap * 3, **i32), chunk_count=_zeros(1, **i32), cap=cap, acts=_zeros(n * F_MOE), partials=_zeros(n * D),
                row_scratch=[_zeros(F_SHARED) for _ in range(3)], params=_attention_params(geo, t, start), code=_scale_code(case))


def _run_block(s):
    k, w, geo, case, code, st = s["ctx"], s["w"], s["geo"], s["case"], s["code"], _stream()
    lib, h, t, start = k.lib, k.handle, s["case"]["tokens"], s["case"]["start"]
    hd, nq, nkv = geo["hd"], geo["nq"], geo["nkv"]
    q_width, kv_width = nq * hd, nkv * hd
    at = start * kv_width * 2
    p = lambda name: s[name].data_ptr()
    ptr = lambda name: w[name].data_ptr()
    s["hidden"].copy_(s["hidden_in"])           # the residual stream, as the layer before left it
    k.check(lib.tf_prefill_rmsnorm_bf16w_block(h, st, p("hidden"), 0, ptr("input_norm"), 0, p("x_norm"), 0, t, D, EPS))
    for name, out, offset, rows in (("q", "q", 0, q_width), ("k", "k_cache", at, kv_width), ("v", "v_cache", at, kv_width)):
        k.check(lib.tf_int4_qmm(h, st, *_abc(w[name]), p("x_norm"), 0, p(out), offset, t, rows, D, code))
    k.check(lib.tf_prefill_qkv_epilogue_block(h, st, p("q"), 0, p("k_cache"), at, p("v_cache"), at, ptr("q_norm"), 0, ptr("k_norm"), 0, start, t, hd, nq, nkv,
                                              q_width, kv_width, geo["theta"], geo["pairs"], EPS))
    k.check(lib.tf_prefill_attention_causal(h, st, p("q"), 0, p("k_cache"), 0, p("v_cache"), 0, p("attn"), 0, C.byref(s["params"]), 0))
    k.check(lib.tf_int4_qmm(h, st, *_abc(w["o"]), p("attn"), 0, p("o"), 0, t, D, q_width, code))
    k.check(lib.tf_prefill_post_attn_setup_block(h, st, p("hidden"), 0, p("o"), 0, p("dense_x"), 0, p("routed_x"), 0, p("router_x"), 0, ptr("post_attn"), 0,
                                                 ptr("pre_ffn"), 0, ptr("pre_ffn2"), 0, t, D, D, D, D, D, D, EPS))
    e = w["experts"]
    k.check(lib.tf_prefill_router_group_block(h, st, *_abc((e["W"], e["S"], e["B"])), p("router_x"), 0, e["eff"].data_ptr(), 0, e["gain"].data_ptr(), 0,
                                              p("idx"), 0, p("wts"), 0, t, E, D, TOPK, D, p("pairs"), p("offsets"), p("counts"), p("chunks"), p("chunk_count")))
    gate, up, down = w["projections"]
    scratch = [v for b in s["row_scratch"] for v in (b.data_ptr(), 0, F_SHARED * 2)]
    k.check(lib.tf_prefill_grouped_routed_moe_resident_shared(
        h, st, p("routed_x"), 0, D, p("pairs"), p("chunks"), p("chunk_count"), s["cap"], t * TOPK, e["pool"].data_ptr(), STRIDE, E, C.byref(s["off"]),
        p("acts"), p("partials"), D, F_MOE, TOPK, code, p("dense_x"), 0, p("shared"), 0, C.byref(gate), C.byref(up), C.byref(down), *scratch,
        t, F_SHARED, D, D, case["shared_bits"]))
    k.check(lib.tf_prefill_moe_reduce_token_major(h, st, p("partials"), 0, p("wts"), 0, p("h2"), 0, t, TOPK, D))
    k.check(lib.tf_prefill_rmsnorm_bf16w_block(h, st, p("shared"), 0, ptr("post_ffn1"), 0, p("h1"), 0, t, D, EPS))
    k.check(lib.tf_prefill_layer_tail_block(h, st, p("h2"), 0, p("h1"), 0, p("hidden"), 0, ptr("post_ffn2"), 0, ptr("post_ffn"), 0, t, D, D, D, D, EPS, 1.0))
    return dict(hidden=s["hidden"], k=s["k_cache"][start:], v=s["v_cache"][start:])


def _prepare_attend(case, gen, state):
    t, start, geo = case["tokens"], case["start"], _geometry(case)
    state["ctx"].reserve(max_attention_block_tokens=t)
    rows = start + t
    return dict(q=_half(gen, t, geo["nq"], geo["hd"]), k=_half(gen, rows, geo["nkv"], geo["hd"]), v=_half(gen, rows, geo["nkv"], geo["hd"]),
                out=_zeros(t, geo["nq"], geo["hd"]), params=_attention_params(geo, t, start))


def _run_attend(s):
    k = s["ctx"]
    k.check(k.lib.tf_prefill_attention_causal(k.handle, _stream(), s["q"].data_ptr(), 0, s["k"].data_ptr(), 0, s["v"].data_ptr(), 0, s["out"].data_ptr(), 0,
                                              C.byref(s["params"]), 0))
    return s["out"]


_KINDS = {"step": (_prepare_step, _run_step), "token": (_prepare_token, _run_token), "head": (_prepare_head, _run_head),
          "verify": (_prepare_verify, _run_verify), "block": (_prepare_block, _run_block), "attend": (_prepare_attend, _run_attend)}


# ---- what a pass cannot do without -------------------------------------------------------------------------------------------
def _matrix_bytes(rows, cols, bits=4):
    return rows * cols * bits // 8 + 2 * rows * (cols // 64) * 2


EXPERT_BYTES = 3 * _matrix_bytes(F_MOE, D)
ROUTER_BYTES = _matrix_bytes(E, D, 8) + D * 2 + E * 2


def _experts_in_use(tokens):
    """Experts that `tokens` rows with a common direction choose between them, averaged over a few routers."""
    rng = np.random.default_rng(7)
    seen = []
    for _ in range(8):
        logits = rng.standard_normal(E) + rng.standard_normal((tokens, E))
        seen.append(len(np.unique(np.argpartition(-logits, TOPK, axis=1)[:, :TOPK])))
    return float(np.mean(seen))


def _keys_seen(geo, tokens, start):
    return sum(min(start + i + 1, geo["window"] or start + i + 1) for i in range(tokens))


def _key_rows(geo, tokens, start):
    return min(start + tokens, (geo["window"] + tokens - 1) if geo["window"] else start + tokens)


def _layer_bytes(geo, tokens, start, shared_bits):
    """Weights of one layer once, the rows of its caches that the tokens see, the residual stream in and out."""
    q, kv = geo["nq"] * geo["hd"], geo["nkv"] * geo["hd"]
    weights = _matrix_bytes(q + 2 * kv, D) + _matrix_bytes(D, q) + 3 * _matrix_bytes(F_SHARED, D, shared_bits) + ROUTER_BYTES + _experts_in_use(tokens) * EXPERT_BYTES
    return weights + 2 * _key_rows(geo, tokens, start) * kv * 2 + 2 * tokens * D * 2 + 7 * D * 2


def _layer_flops(geo, tokens, start):
    q, kv = geo["nq"] * geo["hd"], geo["nkv"] * geo["hd"]
    per_token = 2 * D * (2 * q + 2 * kv) + 2 * 3 * D * F_SHARED + 2 * 3 * D * F_MOE * TOPK + 2 * D * E
    return tokens * per_token + 4 * _keys_seen(geo, tokens, start) * q


def work(case):
    kind = case["kind"]
    if kind == "step":
        per = TOPK * EXPERT_BYTES + ROUTER_BYTES + 3 * D * 2 + TOPK * 6
        return dict(bytes=case["layers"] * per, flops=case["layers"] * 2 * (3 * D * F_MOE * TOPK + D * E))
    if kind == "token":
        nbytes, flops = _matrix_bytes(VOCAB, D) + VOCAB * 2, 2 * D * VOCAB
        for i in range(case["layers"]):
            geo = GLOBAL if i % 6 == 5 else SLIDING
            nbytes += _layer_bytes(geo, 1, case["context"], 4)
            flops += _layer_flops(geo, 1, case["context"])
        return dict(bytes=nbytes, flops=flops)
    if kind == "head":
        v = case["vocab"]
        return dict(bytes=_matrix_bytes(v, D) + 2 * D * 2 + 4 + (v * 2 * 2 if case["mode"] == "sampled" else 0), flops=2 * v * D)
    if kind == "verify":
        t = case["tokens"]
        return dict(bytes=_experts_in_use(t) * EXPERT_BYTES + ROUTER_BYTES + t * (2 * D * 2 + TOPK * (D * 2 + 6)), flops=t * 2 * (3 * D * F_MOE * TOPK + D * E))
    t, start, geo = case["tokens"], case["start"], _geometry(case)
    if kind == "block":
        extra = t * (2 * geo["nkv"] * geo["hd"] * 2 + 2 * D * 2)      # the cache rows, the two experts' outputs
        return dict(bytes=_layer_bytes(geo, t, start, case["shared_bits"]) + extra, flops=_layer_flops(geo, t, start))
    q, kv = geo["nq"] * geo["hd"], geo["nkv"] * geo["hd"]
    return dict(bytes=2 * t * q * 2 + 2 * _key_rows(geo, t, start) * kv * 2, flops=4 * _keys_seen(geo, t, start) * q)


# About four times the distance of each path from the same computation in 64-bit floating point without intermediate rounding
# (2-norm / largest): step 3.8e-4 / 1.3e-3, verify 4.2e-4 / 1.8e-3, attend 2.9e-4 / 1.2e-3, sampled head 2.1e-3 / 3.7e-3.  A whole layer
# is 4e-4 / 2.9e-3 away, and up to 6e-4 / 0.1 where a row of a block whose eighth and ninth router logits nearly tie takes another
# expert; 30 layers of one token 1.6e-3 / 8e-3, and such a tie in an early layer adds about 0.5e-2 to everything after it.
_TOLERANCE = {"step": dict(rel=1.5e-3, max=5e-3, differ=0.01), "token": dict(rel=0.02, max=0.4), "verify": dict(rel=1.7e-3, max=7e-3, differ=0.01),
              "block": dict(rel=2.5e-3, max=0.4), "attend": dict(rel=1.2e-3, max=5e-3)}


def tolerance(case):
    if case["kind"] == "head":
        return "exact" if case["mode"] == "greedy" else dict(rel=8e-3, max=0.015, differ=0.01)
    return _TOLERANCE[case["kind"]]
