"""The measured work of this library: what an inference engine has it do, case by case.

A case is a dict of plain values; its "kind" names the call (or the chain of
calls) and the rest are sizes, types and options:

  engine   EngineContext.forward: one layer's decode step, host arrays in and out
  step     gqa_f16_step: decode with the prologue fused, over a batch of sequences
  verify   gqa_f16_varlen: several query rows per sequence (speculative verify)
  prefill  prefill_f16 / lfm3_prefill_f16: causal attention of prompts
  proj     quantize_q8_K + gqa_qkv_fused or matmul_prequant: the projections
  block    a whole attention layer over a prompt: quantize, fused Q/K/V,
           prologue, attention, quantize, output projection

Head shapes, contexts and batch sizes are those of bench.py and the tests:
16q/8kv and 32q/8kv of head_dim 64, 16q/4kv of head_dim 128 with the output
gate, sliding windows of 256 in rings of 264 slots, 2048-wide projections.
"""
import math

import numpy as np
import torch

import laii_amd as la

EPS = 1e-5
BASE_FULL, BASE_WINDOW = 1e6, 1e4
Q4_0, Q8_0, Q4_K, Q5_K, Q6_K, IQ4_XS = 2, 8, 12, 13, 14, 23
BLOCK_BYTES = {Q4_0: 144, Q8_0: 272, Q4_K: 144, Q5_K: 176, Q6_K: 210, IQ4_XS: 136}  # of 256 weights
GRID = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]   # IQ4_NL values


def listed():
    d64, d128 = dict(nq=32, nkv=8, hd=64), dict(nq=16, nkv=4, hd=128)
    return [
        # one chat user on a CPU engine that hands its attention to the GPU: a
        # layer call per token, arrays in host memory
        dict(name="engine_b1_32q8kv_pos4607", kind="engine", pos=4607, rows=1, window=0, gate=False, **d64),
        # the smallest device-resident call: one user, a short context
        dict(name="step_b1_16q8kv_ctx1024", kind="step", n_seq=1, ctx=1024, ragged=False, window=0, gate=False,
             table=False, nq=16, nkv=8, hd=64),
        # a serving batch of users at different lengths
        dict(name="step_b64_32q8kv_ctx8192_ragged", kind="step", n_seq=64, ctx=8192, ragged=True, window=0,
             gate=False, table=False, **d64),
        # long documents: the full-attention layers of a gated model
        dict(name="step_b32_d128_ctx32768_gate", kind="step", n_seq=32, ctx=32768, ragged=False, window=0, gate=True,
             table=False, **d128),
        # the same batch in its sliding-window layers: little data, many short rows
        dict(name="step_b32_d128_window256_gate", kind="step", n_seq=32, ctx=1001, ragged=True, window=256, gate=True,
             table=False, **d128),
        # speculative decoding: eight drafted tokens per user checked at once
        dict(name="verify_b16_rows8_32q8kv_ctx4096", kind="verify", n_seq=16, rows=8, ctx=4096, ragged=False,
             window=0, gate=False, **d64),
        # prompts: full pages, an odd length continuing a cached prefix, and a window layer
        dict(name="prefill_b4_n4096_32q8kv", kind="prefill", n_seq=4, n_tok=4096, pos=0, window=0, gate=False, **d64),
        dict(name="prefill_b2_n3001_d128_gate_pos517", kind="prefill", n_seq=2, n_tok=3001, pos=517, window=0,
             gate=True, **d128),
        dict(name="prefill_b4_n4096_d128_window256", kind="prefill", n_seq=4, n_tok=4096, pos=0, window=256,
             gate=True, **d128),
        # the output projection of one token: the smallest projection
        dict(name="proj_wo_q4k_1token", kind="proj", t0=Q4_K, t1=0, t2=0, r0=2048, r1=0, r2=0, n_cols=2048, tokens=1),
        # Q/K/V of a 64-user decode step, weights in Q8_0
        dict(name="proj_qkv_q8_0_64tokens", kind="proj", t0=Q8_0, t1=Q8_0, t2=Q8_0, r0=2048, r1=512, r2=512,
             n_cols=2048, tokens=64),
        # a prompt through a whole attention layer, weights in the usual 4-bit mix (V in Q6_K)
        dict(name="block_n2000_q4k_q6k", kind="block", t0=Q4_K, t1=Q4_K, t2=Q6_K, t3=Q4_K, n_tok=2000, pos=0, nq=32,
             nkv=8, hd=64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["engine", "step", "step", "verify", "prefill", "prefill", "proj", "proj", "proj", "block"])
    small, wide, gated = dict(nq=16, nkv=8, hd=64), dict(nq=32, nkv=8, hd=64), dict(nq=16, nkv=4, hd=128)
    if kind == "engine":
        shape = rng.choice([small, wide, gated])
        window = rng.choice([0, 256]) if shape is gated else 0
        return dict(kind=kind, pos=_log(rng, 16, 8000), rows=rng.choice([1, 1, 1, 2, 4, 7, 8]), window=window,
                    gate=shape is gated, **shape)
    if kind == "step":
        shape = rng.choice([small, wide, wide, gated, gated])
        n_seq = _log(rng, 1, 64)
        window = rng.choice([0, 256]) if shape is gated else 0
        ctx = _log(rng, 64, min(32768, 1048576 // n_seq))
        return dict(kind=kind, n_seq=n_seq, ctx=ctx, ragged=rng.random() < 0.7, window=window, gate=shape is gated,
                    table=shape is not gated and rng.random() < 0.3, **shape)
    if kind == "verify":
        shape = rng.choice([small, wide, wide, gated])
        n_seq = _log(rng, 1, 32)
        window = rng.choice([0, 256]) if shape is gated else 0
        return dict(kind=kind, n_seq=n_seq, rows=rng.randint(2, 8), ctx=_log(rng, 128, 8192), ragged=rng.random() < 0.7,
                    window=window, gate=shape is gated, **shape)
    if kind == "prefill":
        shape = rng.choice([wide, gated])
        window = rng.choice([0, 256]) if shape is gated else 0
        n_seq = rng.randint(1, 4)
        n_tok = _log(rng, 16, 4096)
        pos = rng.choice([0, 0, rng.randint(1, 1500)]) if n_tok < 2500 else 0
        return dict(kind=kind, n_seq=n_seq, n_tok=n_tok, pos=pos, window=window, gate=shape is gated, **shape)
    if kind == "proj":
        t = rng.choice(sorted(BLOCK_BYTES))
        n_cols = rng.choice([1024, 1536, 2048, 2048, 2304])
        tokens = _log(rng, 1, 2000)
        if rng.random() < 0.5:
            return dict(kind=kind, t0=t, t1=0, t2=0, r0=rng.choice([512, 1024, 2048, 2048, 1000]), r1=0, r2=0,
                        n_cols=n_cols, tokens=tokens)
        return dict(kind=kind, t0=t, t1=t, t2=rng.choice([t, Q6_K]), r0=2048, r1=512, r2=512, n_cols=n_cols,
                    tokens=tokens)
    t = rng.choice([Q4_K, Q4_K, Q5_K, Q8_0])
    return dict(kind="block", t0=t, t1=t, t2=Q6_K if t == Q4_K else t, t3=t, n_tok=_log(rng, 16, 2000),
                pos=rng.choice([0, rng.randint(1, 500)]), nq=32, nkv=8, hd=64)


# ---- inputs ------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _cache(g, slots, nkv, hd):
    """fp16 cache rows, 0.5 * N(0, 1) as keys and values are after their norms."""
    return (torch.randn((slots, nkv, hd), generator=g, device="cuda", dtype=torch.float16) * 0.5)


def _norm_w(g, hd):
    return 1.0 + 0.05 * _randn(g, hd)


def _rope(case, rows):
    """RoPE table (device) of `rows` positions as the engine builds it."""
    hd = case["hd"]
    if case.get("table"):
        c, s = la.rope_table_lfm2(rows, hd, BASE_FULL)
    elif hd == 128:
        base, dim = (BASE_WINDOW, hd) if case["window"] else (BASE_FULL, hd)
        c, s = la.rope_lut_lfm3(rows, hd, dim, base)
    else:
        c, s = la.rope_lut_lfm2(rows, hd, BASE_FULL)
    return torch.from_numpy(c).cuda(), torch.from_numpy(s).cuda()


def _contexts(case, seed):
    """Keys of each sequence before the rows of this call: uniform from a
    sixteenth of the longest, which one sequence has.  The seed orders them;
    their sum, and with it the work, is the case's."""
    n, ctx = case["n_seq"], case["ctx"]
    if not case["ragged"]:
        return np.full(n, ctx, np.int64)
    c = np.random.default_rng(n * 65537 + ctx).integers(max(1, ctx // 16), ctx + 1, size=n)
    c[0] = ctx
    return np.random.default_rng(seed).permutation(c)


def _half_bytes(g, n, lo, hi):
    v = (torch.rand(n, generator=g, device="cuda") * (hi - lo) + lo).to(torch.float16)
    return v.view(torch.uint8).reshape(n, 2)


def _weights(g, qtype, n_rows, n_cols):
    """Packed rows of a weight type: random quants, scales that give weights of
    about 0.05 with a mean near zero."""
    nb = n_cols // 256
    n = n_rows * nb
    w = torch.randint(0, 256, (n, BLOCK_BYTES[qtype]), generator=g, device="cuda", dtype=torch.uint8)
    if qtype in (Q4_K, Q5_K):
        step = 1.0 if qtype == Q4_K else 0.5
        w[:, 0:2] = _half_bytes(g, n, 1e-4 * step, 3e-4 * step)
        w[:, 2:4] = _half_bytes(g, n, 7.5e-4, 2.2e-3)
    elif qtype == Q6_K:
        w[:, 192:208] = torch.randint(-64, 64, (n, 16), generator=g, device="cuda", dtype=torch.int8).view(torch.uint8)
        w[:, 208:210] = _half_bytes(g, n, 5e-5, 1.5e-4)
    elif qtype == IQ4_XS:
        w[:, 0:2] = _half_bytes(g, n, 2e-5, 8e-5)
    else:
        b = w.reshape(n * 8, -1)
        b[:, 0:2] = _half_bytes(g, n * 8, 5e-3, 1.5e-2) if qtype == Q4_0 else _half_bytes(g, n * 8, 3e-4, 9e-4)
    return w.reshape(n_rows, -1)


def _mats(case):
    return [(case["t%d" % i], case["r%d" % i]) for i in range(3) if case["r%d" % i]]


def prepare(case, seed):
    kind, g = case["kind"], _gen(seed)
    st = dict(case=dict(case), stream=torch.cuda.current_stream().cuda_stream)
    if kind == "proj":
        n, cols = case["tokens"], case["n_cols"]
        st["x"] = _randn(g, n, cols)
        st["xq"] = torch.zeros((n, cols // 256 * 292), device="cuda", dtype=torch.uint8)
        st["w"] = [_weights(g, t, r, cols) for t, r in _mats(case)]
        st["out"] = [torch.zeros((n, r), device="cuda") for _, r in _mats(case)]
        return st
    nq, nkv, hd = case["nq"], case["nkv"], case["hd"]
    if kind == "engine":
        B, pos, win = case["rows"], case["pos"], case["window"]
        rng = np.random.default_rng(seed)
        lfm3 = hd == 128
        ctx = la.EngineContext(1, nq, nkv, hd, pos + B, EPS, rope_base=BASE_FULL, lfm3=lfm3, sliding_window=win,
                               swa_cap=win + 8 if win else 0, layer_is_swa=[1] if win else None,
                               rope_base_swa=BASE_WINDOW, rope_dim=hd if lfm3 else 0)
        st["qw"], st["kw"] = ((1 + 0.05 * rng.standard_normal(hd)).astype(np.float32) for _ in range(2))
        ctx.set_norms(0, st["qw"], st["kw"])
        slots = min(pos, win + 8) if win else pos
        st["kc"], st["vc"] = ((0.5 * rng.standard_normal((slots, nkv * hd), np.float32)).astype(np.float16)
                              for _ in range(2))
        ctx.kv_import(0, 0, st["kc"].view(np.uint16), st["vc"].view(np.uint16))
        st["q"] = rng.standard_normal((B, nq, hd), np.float32)
        st["k"], st["v"] = (rng.standard_normal((B, nkv, hd), np.float32) for _ in range(2))
        st["gate"] = rng.standard_normal((B, nq), np.float32) if case["gate"] else None
        st["ctx"] = ctx
        return st
    if kind in ("step", "verify"):
        n, win, rows = case["n_seq"], case["window"], case.get("rows", 1)
        before = _contexts(case, seed)
        if kind == "step":
            before = before - 1  # the context counts the new token
        slots = np.full(n, win + 8) if win else before + rows
        first = np.concatenate([[0], np.cumsum(slots)])
        st["k"], st["v"] = (_cache(g, int(first[-1]), nkv, hd) for _ in range(2))
        st["slots"], st["first"], st["before"] = slots, first, before
        row = nkv * hd * 2
        table = lambda t: torch.from_numpy(t.data_ptr() + first[:-1].astype(np.int64) * row).cuda()  # noqa: E731
        st["kt"], st["vt"] = table(st["k"]), table(st["v"])
        st["pos"] = torch.from_numpy(before.astype(np.int32)).cuda()
        st["q"] = _randn(g, n, rows, nq, hd)
        st["gate"] = _randn(g, n, rows, nq) if case["gate"] else None
        st["out"] = torch.zeros((n, rows, nq, hd), device="cuda")
        longest = int(before.max()) + rows
        st["hint"] = min(win + rows - 1, longest) if win else longest
        if kind == "step":
            st["kn"], st["vn"] = (_randn(g, n, rows, nkv, hd) for _ in range(2))
            st["qw"], st["kw"] = _norm_w(g, hd), _norm_w(g, hd)
            st["cos"], st["sin"] = _rope(case, longest)
        return st
    n_seq, n_tok, pos = case.get("n_seq", 1), case["n_tok"], case["pos"]
    if kind == "prefill":
        win = case["window"]
        st["kv0"] = max(0, pos + 1 - win) if win else 0
        rows = pos + n_tok - st["kv0"]
        st["q"] = (0.5 * _randn(g, n_seq, n_tok, nq, hd)).half().float()
        st["k"], st["v"] = (_cache(g, n_seq * rows, nkv, hd).reshape(n_seq, rows, nkv, hd) for _ in range(2))
        st["gate"] = _randn(g, n_seq, n_tok, nq) if case["gate"] else None
        st["out"] = torch.zeros((n_seq, n_tok, nq, hd), device="cuda")
        return st
    # block
    cols = nq * hd
    st["x"] = _randn(g, n_tok, cols)
    st["xq"] = torch.zeros((n_tok, cols // 256 * 292), device="cuda", dtype=torch.uint8)
    sizes = [nq * hd, nkv * hd, nkv * hd, cols]
    st["w"] = [_weights(g, case["t%d" % i], r, cols) for i, r in enumerate(sizes)]
    st["qkv"] = [torch.zeros((n_tok, r), device="cuda") for r in sizes[:3]]
    st["k"], st["v"] = (_cache(g, pos + n_tok, nkv, hd) for _ in range(2))
    st["k_before"], st["v_before"] = st["k"][:pos].clone(), st["v"][:pos].clone()
    st["kt"], st["vt"] = (torch.tensor([t.data_ptr()], device="cuda") for t in (st["k"], st["v"]))
    st["pos"] = torch.tensor([pos], device="cuda", dtype=torch.int32)
    st["qw"], st["kw"] = _norm_w(g, hd), _norm_w(g, hd)
    st["cos"], st["sin"] = _rope(case, pos + n_tok)
    st["attn"] = torch.zeros((n_tok, cols), device="cuda")
    st["aq"] = torch.zeros_like(st["xq"])
    st["out"] = torch.zeros((n_tok, cols), device="cuda")
    return st


# ---- one pass ----------------------------------------------------------------------

def _a(t):
    return None if t is None else t.data_ptr()


def run(st):
    c, s = st["case"], st["stream"]
    kind = c["kind"]
    if kind == "engine":
        return st["ctx"].forward(0, c["pos"], st["q"], st["k"], st["v"], st["gate"])
    if kind == "proj":
        n, cols = c["tokens"], c["n_cols"]
        la.quantize_q8_K(_a(st["x"]), _a(st["xq"]), n, cols, s)
        if len(st["w"]) == 1:
            la.matmul_prequant(_a(st["out"][0]), _a(st["w"][0]), c["t0"], c["r0"], cols, _a(st["xq"]), n, s)
        else:
            la.gqa_qkv_fused([_a(o) for o in st["out"]], [_a(w) for w in st["w"]], [c["t0"], c["t1"], c["t2"]],
                             [c["r0"], c["r1"], c["r2"]], cols, _a(st["xq"]), n, s)
        return [st["xq"], st["out"]]
    nq, nkv, hd = c["nq"], c["nkv"], c["hd"]
    if kind == "step":
        win = c["window"]
        la.gqa_f16_step(_a(st["q"]), _a(st["kn"]), _a(st["vn"]), _a(st["gate"]), True, _a(st["kt"]), _a(st["vt"]),
                        _a(st["pos"]), _a(st["out"]), c["n_seq"], 1, st["hint"], nq, nkv, hd, _a(st["qw"]),
                        _a(st["kw"]), EPS, _a(st["cos"]), _a(st["sin"]), win, win + 8 if win else 0, None, s,
                        la.PROLOGUE_TABLE if c["table"] else la.PROLOGUE_FAST)
        return [st["out"], st["k"], st["v"]]
    if kind == "verify":
        win = c["window"]
        la.gqa_f16_varlen(_a(st["q"]), _a(st["gate"]), True, _a(st["kt"]), _a(st["vt"]), _a(st["pos"]), _a(st["out"]),
                          c["n_seq"], c["rows"], st["hint"], nq, nkv, hd, win, win + 8 if win else 0, None, s)
        return st["out"]
    if kind == "prefill":
        stride = st["k"].stride(0)
        if hd == 64:
            la.prefill_f16(_a(st["q"]), _a(st["k"]), _a(st["v"]), _a(st["out"]), c["n_seq"], c["n_tok"], c["pos"],
                           stride, nq, nkv, hd, None, s)
        else:
            la.lfm3_prefill_f16(_a(st["q"]), _a(st["k"]), _a(st["v"]), _a(st["gate"]), True, _a(st["out"]), c["n_seq"],
                                c["n_tok"], c["pos"], st["kv0"], stride, c["window"], nq, nkv, hd, None, s)
        return st["out"]
    n, cols = c["n_tok"], nq * hd
    q, k, v = st["qkv"]
    la.quantize_q8_K(_a(st["x"]), _a(st["xq"]), n, cols, s)
    la.gqa_qkv_fused([_a(q), _a(k), _a(v)], [_a(w) for w in st["w"][:3]], [c["t0"], c["t1"], c["t2"]],
                     [nq * hd, nkv * hd, nkv * hd], cols, _a(st["xq"]), n, s)
    la.qkv_prologue(_a(q), _a(k), _a(v), _a(st["kt"]), _a(st["vt"]), _a(st["pos"]), 1, n, nq, nkv, hd, _a(st["qw"]),
                    _a(st["kw"]), EPS, _a(st["cos"]), _a(st["sin"]), 0, 0, s)
    la.prefill_f16(_a(q), _a(st["k"]), _a(st["v"]), _a(st["attn"]), 1, n, c["pos"], (c["pos"] + n) * nkv * hd, nq, nkv,
                   hd, None, s)
    la.quantize_q8_K(_a(st["attn"]), _a(st["aq"]), n, cols, s)
    la.matmul_prequant(_a(st["out"]), _a(st["w"][3]), c["t3"], cols, cols, _a(st["aq"]), n, s)
    return [st["out"], st["k"], st["v"]]


# ---- what a pass cannot do without ---------------------------------------------------

def _proj_work(types_rows, cols, n):
    b = n * cols * 4 + 2 * n * (cols // 256) * 292
    f = 0
    for t, r in types_rows:
        b += r * (cols // 256) * BLOCK_BYTES[t] + n * r * 4
        f += 2 * n * r * cols
    return b, f


def _prefill_flops(n_seq, n_tok, pos, window, nq, hd):
    p = np.arange(pos, pos + n_tok, dtype=np.int64) + 1
    keys = int((np.minimum(p, window) if window else p).sum())
    return 4 * hd * nq * n_seq * keys


def work(case):
    kind = case["kind"]
    if kind == "proj":
        b, f = _proj_work(_mats(case), case["n_cols"], case["tokens"])
        return dict(bytes=b, flops=f)
    nq, nkv, hd = case["nq"], case["nkv"], case["hd"]
    if kind in ("engine", "step", "verify"):
        rows, win = case.get("rows", 1), case["window"]
        n = case.get("n_seq", 1)
        if kind == "engine":
            before = np.array([case["pos"]])
        else:
            before = _contexts(case, 0) - (1 if kind == "step" else 0)
        union = np.minimum(before + rows, win + rows - 1) if win else before + rows
        p = before[:, None] + np.arange(rows)[None] + 1
        keys = int((np.minimum(p, win) if win else p).sum())
        new = 0 if kind == "verify" else n * rows * nkv * hd * 2 * (4 + 2)  # raw rows in, fp16 rows out
        b = int(union.sum()) * nkv * hd * 4 + n * rows * nq * hd * 8 + new
        return dict(bytes=b, flops=4 * hd * nq * keys)
    if kind == "prefill":
        n_seq, n_tok, pos, win = case["n_seq"], case["n_tok"], case["pos"], case["window"]
        kv0 = max(0, pos + 1 - win) if win else 0
        b = n_seq * (n_tok * nq * hd * 8 + (pos + n_tok - kv0) * nkv * hd * 4)
        return dict(bytes=b, flops=_prefill_flops(n_seq, n_tok, pos, win, nq, hd))
    n, pos, cols = case["n_tok"], case["pos"], nq * hd
    sizes = [nq * hd, nkv * hd, nkv * hd, cols]
    b = n * cols * 8 + (pos + 2 * n) * nkv * hd * 4
    f = _prefill_flops(1, n, pos, 0, nq, hd)
    for i, r in enumerate(sizes):
        b += r * (cols // 256) * BLOCK_BYTES[case["t%d" % i]]
        f += 2 * n * r * cols
    return dict(bytes=b, flops=f)


def tolerance(case):
    """About four times the distance from the 64-bit values: fp32 sums over
    exact products (projections) and over scores of ~fp32 accuracy (decode, up
    to 16 query rows per KV head), probabilities in fp16 beyond that, queries in
    fp16 too in prefill.  A block requantizes its attention to 8 bits."""
    kind = case["kind"]
    if kind in ("engine", "step", "verify"):
        few = case.get("rows", 1) * (case["nq"] // case["nkv"]) <= 16
        return dict(rel=6e-6, max=1e-3) if few else dict(rel=1e-3, max=2e-2)
    if kind == "prefill":
        return dict(rel=1e-3, max=2e-2)
    if kind == "proj":
        return dict(rel=4e-7, max=4e-6)
    return dict(rel=8e-3, max=5e-2)


# ---- the same in 64 bits, in plain torch ---------------------------------------------

def _norm_rope64(x, w, cos, sin):
    """RMS norm and rotation of pairs (i, i + hd/2); x [..., heads, hd], cos and sin [..., 1, hd/2]."""
    x = x.double()
    x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()
    lo, hi = x.chunk(2, -1)
    c, s = cos.double(), sin.double()
    return torch.cat([lo * c - hi * s, hi * c + lo * s], -1)


def _attend64(q, k, v, first, window, gate=None):
    """q [rows, nq, hd] at positions first.., keys [n, nkv, hd] at positions n0 = first + rows - n ..: causal, windowed."""
    rows, nq, hd = q.shape
    n, nkv, _ = k.shape
    mul = nq // nkv
    p = torch.arange(rows, device=q.device)[:, None] + (n - rows)
    t = torch.arange(n, device=q.device)[None]
    hide = t > p
    if window:
        hide = hide | (t <= p - window)
    out = torch.empty((rows, nq, hd), dtype=torch.float64, device=q.device)
    for j in range(nkv):
        kj, vj = k[:, j].double().t().contiguous(), v[:, j].double()
        for h in range(j * mul, (j + 1) * mul):
            s = (q[:, h].double() @ kj) / math.sqrt(hd)
            out[:, h] = torch.softmax(s.masked_fill(hide, -math.inf), -1) @ vj
    if gate is not None:
        out = out * torch.sigmoid(gate.double())[..., None]
    return out


def _attend_few64(q, k, v, window, gate):
    """_attend64 for few rows: all query heads of a KV head in one product."""
    rows, nq, hd = q.shape
    n, nkv, _ = k.shape
    mul = nq // nkv
    p = torch.arange(rows, device=q.device).repeat_interleave(mul)[:, None] + (n - rows)
    t = torch.arange(n, device=q.device)[None]
    hide = t > p
    if window:
        hide = hide | (t <= p - window)
    out = torch.empty((rows, nq, hd), dtype=torch.float64, device=q.device)
    for j in range(nkv):
        qj = q[:, j * mul:(j + 1) * mul].double().reshape(rows * mul, hd)
        s = (qj @ k[:, j].double().t().contiguous()) / math.sqrt(hd)
        o = torch.softmax(s.masked_fill(hide, -math.inf), -1) @ v[:, j].double()
        out[:, j * mul:(j + 1) * mul] = o.reshape(rows, mul, hd)
    if gate is not None:
        out = out * torch.sigmoid(gate.double())[..., None]
    return out


def _half64(x):
    """An fp64 value as an fp16 cache holds it."""
    return x.float().half().double()


def _scale_min(sc, j):
    if j < 4:
        return sc[:, j] & 63, sc[:, j + 4] & 63
    return (sc[:, j + 4] & 15) | ((sc[:, j - 4] >> 6) << 4), (sc[:, j + 4] >> 4) | ((sc[:, j] >> 6) << 4)


def _halves(b):
    return b.contiguous().view(torch.float16).double()


def _dequant64(w, qtype, n_cols):
    n_rows = w.shape[0]
    blk = w.reshape(-1, BLOCK_BYTES[qtype])
    i = blk.int()
    parts = []
    if qtype in (Q4_K, Q5_K):
        d, dm = _halves(blk[:, 0:2]), _halves(blk[:, 2:4])
        qs = i[:, 16:] if qtype == Q4_K else i[:, 48:]
        for j in range(8):
            sc, m = _scale_min(i[:, 4:16], j)
            q = (qs[:, 32 * (j // 2):32 * (j // 2) + 32] >> (4 * (j % 2))) & 15
            if qtype == Q5_K:
                q = q + 16 * ((i[:, 16:48] >> j) & 1)
            parts.append(d * sc[:, None] * q - dm * m[:, None])
    elif qtype == Q6_K:
        d = _halves(blk[:, 208:210])
        sc = blk[:, 192:208].contiguous().view(torch.int8).double()
        for h in range(2):
            ql, qh = i[:, 64 * h:64 * h + 64], i[:, 128 + 32 * h:160 + 32 * h]
            for k in range(4):
                low = (ql[:, 32 * (k % 2):32 * (k % 2) + 32] >> (4 * (k // 2))) & 15
                u = (low | (((qh >> (2 * k)) & 3) << 4)) - 32
                s = sc[:, 8 * h + 2 * k:8 * h + 2 * k + 2].repeat_interleave(16, 1)
                parts.append(d * s * u)
    elif qtype == IQ4_XS:
        d, grid = _halves(blk[:, 0:2]), torch.tensor(GRID, device=w.device, dtype=torch.float64)
        sh = i[:, 2] | (i[:, 3] << 8)
        for j in range(8):
            ls = (((i[:, 4 + j // 2] >> (4 * (j % 2))) & 15) | (((sh >> (2 * j)) & 3) << 4)) - 32
            q = i[:, 8 + 16 * j:24 + 16 * j]
            parts.append((d[:, 0] * ls)[:, None] * grid[torch.cat([q & 15, q >> 4], 1).long()])
    elif qtype == Q4_0:
        b = blk.reshape(-1, 18)
        q = b[:, 2:].int()
        parts.append(_halves(b[:, 0:2]) * (torch.cat([q & 15, q >> 4], 1) - 8))
    else:
        b = blk.reshape(-1, 34)
        parts.append(_halves(b[:, 0:2]) * b[:, 2:].contiguous().view(torch.int8).double())
    return torch.cat(parts, 1).reshape(n_rows, n_cols)


def _activations64(x):
    """The values that Q8_K blocks of x hold: d * q, d = max / 127, q = round(x * 127 / max)."""
    b = x.float().reshape(x.shape[0], -1, 256)
    top = b.abs().amax(-1, keepdim=True)
    safe = torch.where(top > 0, top, torch.ones_like(top))
    q = torch.round(b * (torch.full_like(safe, 127.0) / safe)).clamp(-128, 127)
    return ((top / torch.full_like(top, 127.0)).double() * q.double()).reshape(x.shape)


def exact(case, seed):
    kind, st = case["kind"], prepare(case, seed)
    if kind == "proj":
        x = _activations64(st["x"])
        outs = [x @ _dequant64(w, t, case["n_cols"]).t().contiguous() for w, (t, _) in zip(st["w"], _mats(case))]
        return [None, outs]
    nq, nkv, hd = case["nq"], case["nkv"], case["hd"]
    if kind == "engine":
        B, pos, win = case["rows"], case["pos"], case["window"]
        cos, sin = (t[pos:pos + B, None] for t in _rope(dict(case), pos + B))
        dev = {k: torch.from_numpy(st[k]).cuda() for k in ("q", "k", "v", "qw", "kw")}
        q = _norm_rope64(dev["q"], dev["qw"], cos, sin)
        k = _half64(_norm_rope64(dev["k"], dev["kw"], cos, sin))
        old = np.arange(max(0, pos + 1 - win) if win else 0, pos)
        at = old % (win + 8) if win else old
        kc, vc = (torch.from_numpy(st[n][at]).cuda().reshape(-1, nkv, hd).double() for n in ("kc", "vc"))
        gate = None if st["gate"] is None else torch.from_numpy(st["gate"]).cuda()
        o = _attend_few64(q, torch.cat([kc, k]), torch.cat([vc, _half64(dev["v"].double())]), win, gate)
        st["ctx"].close()
        return o.reshape(-1).cpu().numpy()
    if kind in ("step", "verify"):
        win, rows = case["window"], case.get("rows", 1)
        out = torch.empty(st["out"].shape, dtype=torch.float64, device="cuda")
        kept = [st["k"].double(), st["v"].double()] if kind == "step" else [st["k"], st["v"]]
        for s in range(case["n_seq"]):
            p, at = int(st["before"][s]), int(st["first"][s])
            q = st["q"][s].double()
            if kind == "step":
                cos, sin = st["cos"][p:p + 1, None], st["sin"][p:p + 1, None]
                q = _norm_rope64(q, st["qw"], cos, sin)
                slot = at + (p % (win + 8) if win else p)
                kept[0][slot] = _half64(_norm_rope64(st["kn"][s], st["kw"], cos, sin)[0])
                kept[1][slot] = _half64(st["vn"][s, 0].double())
            old = np.arange(max(0, p + 1 - win) if win else 0, p + rows)
            if win:
                at = torch.from_numpy(at + old % (win + 8)).cuda()
                k, v = kept[0][at], kept[1][at]
            else:
                k, v = (t[at:at + p + rows] for t in kept)
            out[s] = _attend_few64(q, k, v, win, None if st["gate"] is None else st["gate"][s])
        return [out] + kept if kind == "step" else out
    if kind == "prefill":
        gate = st["gate"]
        return torch.stack([_attend64(st["q"][s], st["k"][s], st["v"][s], case["pos"], case["window"],
                                      None if gate is None else gate[s]) for s in range(case["n_seq"])])
    n, pos, cols = case["n_tok"], case["pos"], nq * hd
    x = _activations64(st["x"])
    q, k, v = (x @ _dequant64(w, case["t%d" % i], cols).t().contiguous() for i, w in enumerate(st["w"][:3]))
    cos, sin = st["cos"][pos:, None], st["sin"][pos:, None]
    q = _norm_rope64(q.reshape(n, nq, hd), st["qw"], cos, sin)
    k = torch.cat([st["k_before"].double(), _half64(_norm_rope64(k.reshape(n, nkv, hd), st["kw"], cos, sin))])
    v = torch.cat([st["v_before"].double(), _half64(v.reshape(n, nkv, hd))])
    a = _activations64(_attend64(q, k, v, pos, 0).reshape(n, cols))
    return [a @ _dequant64(st["w"][3], case["t3"], cols).t().contiguous(), k, v]
