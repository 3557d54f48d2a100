"""Performance cases of the exact integer engine: what a program that serves these models has it do.

A case is a dict of plain values; its "kind" names the path:
  decode          GraphDecoder steps of B sequences over a filled KV cache (one HIP graph replay a step)
  prefill         TModel.forward of one prompt, logits of its last row
  attend          one decode attention layer: q|k|v epilogue, RoPE, cache write and integer attention
  attend_prefill  one prefill attention layer from the cache
  linear          one packed group-128 linear over R activation rows
  dropin          the seven linears of a decoder layer (or one N x K linear) through the op exact::gemv on row-major
                  tensors, one HIP graph
  sample          integer sampling of one token a row from a step's logits
prepare() makes what a program holds before the call (weights, cache, plans, warmed up), run() is one call, and exact()
restates the integer program in plain torch int64 / float64 arithmetic (every float64 sum stays below 2^53).
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "exact-llm_amd"))
from exact_amd import ops, synth  # noqa: E402
from exact_amd.model import DeviceWeights, GraphDecoder, TModel  # noqa: E402
from exact_amd.tables import DeviceTables  # noqa: E402

DEV = "cuda"
I16, I32, I64, F64 = torch.int16, torch.int32, torch.int64, torch.float64
ONE = 1 << 16   # Q16
SMALL, BASE, LARGE, MOE = "qwen2.5-0.5b", "qwen2.5-7b", "qwen2.5-14b", "qwen1.5-moe-a2.7b"


# ----------------------------------------------------------------------------- the cases
def listed():
    return [
        # one user of the smallest model, short chat turn: launches and latency bound every step
        dict(name="decode_small", kind="decode", model=SMALL, layers=24, B=1, n0=16, Smax=512, steps=8),
        # the headline: batch-1 decode of the 7B shape after a short prompt
        dict(name="decode_7b", kind="decode", model=BASE, layers=28, B=1, n0=16, Smax=512, steps=4),
        # batch-1 decode of the mixture-of-experts shape after its 256-token prompt
        dict(name="decode_moe", kind="decode", model=MOE, layers=8, B=1, n0=256, Smax=512, steps=4),
        # a serving batch deep in its context: eight sequences of different lengths up to 1793 positions
        dict(name="decode_batch_long", kind="decode", model=BASE, layers=8, B=8, n0=1793, Smax=2048, steps=2),
        # a short question: more rows than a GEMV takes, far fewer than a GEMM tile likes
        dict(name="prefill_short", kind="prefill", model=BASE, layers=8, T=41, Smax=512, graph=False),
        # a long document, odd length
        dict(name="prefill_long", kind="prefill", model=BASE, layers=8, T=1537, Smax=2048, graph=False),
        # a prompt of the mixture-of-experts shape, captured as a graph as a server of fixed prompt buckets does
        dict(name="prefill_moe", kind="prefill", model=MOE, layers=4, T=253, Smax=512, graph=True),
        # decode attention of one sequence near the end of the longest cache the engine takes
        dict(name="attend_long", kind="attend", H=28, KV=4, hd=128, R=1, n0=6001, Smax=8192),
        # the prefill attention benchmark: one 7B layer at 2048 tokens
        dict(name="attend_prefill", kind="attend_prefill", H=28, KV=4, hd=128, R=2048, p0=0),
        # the prefill GEMM benchmark: gate|up rows of the 7B shape, int8 activations
        dict(name="linear_prefill", kind="linear", R=2048, N=18944, K=3584, abits=7),
        # programs written against the reference's own op and tensors: a 7B decoder layer's calls
        dict(name="dropin_layer", kind="dropin", model=BASE),
        # the sampler of a batch-8 step over the full vocabulary
        dict(name="sample_batch", kind="sample", R=8, V=152064, temp=0.8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


HEADS = [(14, 2, 64), (28, 4, 128), (40, 8, 128), (16, 16, 128)]


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "attend", "attend_prefill", "linear", "linear", "dropin",
                       "sample"])
    if kind == "decode":
        n0 = _log_int(rng, 1, 4000)
        return dict(kind=kind, model=rng.choice([SMALL, BASE, LARGE, MOE]), layers=rng.randint(2, 6), B=_log_int(rng, 1, 8),
                    n0=n0, Smax=n0 + rng.randint(4, 260), steps=rng.randint(1, 3))
    if kind == "prefill":
        T = _log_int(rng, 2, 1537)
        return dict(kind=kind, model=rng.choice([SMALL, BASE, LARGE, MOE]), layers=rng.randint(1, 3), T=T,
                    Smax=T + rng.randint(1, 500), graph=rng.random() < 0.5)
    if kind == "attend":
        H, KV, hd = rng.choice(HEADS)
        n0 = _log_int(rng, 1, 8000)
        return dict(kind=kind, H=H, KV=KV, hd=hd, R=_log_int(rng, 1, 8), n0=n0, Smax=n0 + rng.randint(1, 190))
    if kind == "attend_prefill":
        H, KV, hd = rng.choice(HEADS[:3])
        R = _log_int(rng, 96, 1700)
        return dict(kind=kind, H=H, KV=KV, hd=hd, R=R, p0=rng.choice([0, 0, rng.randint(1, 300)]))
    if kind == "linear":
        N = rng.choice([18944, 13824, 4608, 5120, 2816, rng.randint(65, 9000)])
        return dict(kind=kind, R=_log_int(rng, 1, 2048), N=N, K=128 * _log_int(rng, 7, 40), abits=rng.choice([7, 15]))
    if kind == "dropin":
        return dict(kind=kind, model="", N=_log_int(rng, 64, 19000), K=128 * _log_int(rng, 1, 148))
    return dict(kind=kind, R=_log_int(rng, 1, 8), V=_log_int(rng, 1000, 152064), temp=round(rng.uniform(0.3, 1.5), 3))


# ----------------------------------------------------------------------------- prepare and run
def _gen(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1000003 + salt)
    return g


def _q16(g, shape, std):
    return (torch.randn(shape, generator=g, device=DEV) * (std * ONE)).round().to(I64)


def _tokens(seed, n, V):
    r = random.Random(seed)
    return [r.randrange(V) for _ in range(n)]


def _lens(case):
    """cached positions of each decode row: the sequences of a batch are of different lengths"""
    return [max(1, case["n0"] - (case["n0"] // 23) * r) for r in range(case.get("B", case.get("R")))]


def _fill_cache(layer, seed, li, lens, kstd):
    """keys (quantised per head row, as the engine stores them) and values of the first lens[b] positions of slot b"""
    kq, sk, v = layer
    B, KV, _, hd = kq.shape
    g = _gen(seed, 7 + li)
    for b in range(B):
        k = _q16(g, (KV, lens[b], hd), kstd)
        q, s = _qrow(k, 15)
        kq[b, :, :lens[b]] = q.to(I16)
        sk[b, :, :lens[b]] = s[..., 0].to(I32)
        v[b, :, :lens[b]] = _q16(g, (KV, lens[b], hd), 1.0)


MODEL_KSTD = 8.0   # key spread of the filled model caches: the synthetic models' queries are of spread 0.2
ATT_KSTD = 2.0     # ... and of the attention layer alone, whose queries are of spread 1


def _attend_inputs(case, seed):
    H, KV, hd, R, Smax = case["H"], case["KV"], case["hd"], case["R"], case["Smax"]
    g, nq = _gen(seed, 1), (H + 2 * KV) * hd
    std = torch.cat([torch.full((H * hd,), 1.0), torch.full((KV * hd,), ATT_KSTD), torch.full((KV * hd,), 1.0)]).to(DEV)
    s = torch.randint(6, 11, (R,), generator=g, device=DEV, dtype=I32)
    y = torch.randn((R, nq), generator=g, device=DEV).double() * std * ONE
    t = (y * torch.exp2(28.0 - s.double())[:, None]).round().to(I64)
    b = _q16(g, (nq,), 0.15)
    cache = (torch.zeros((R, KV, Smax, hd), dtype=I16, device=DEV), torch.zeros((R, KV, Smax), dtype=I32, device=DEV),
             torch.zeros((R, KV, Smax, hd), dtype=I64, device=DEV))
    _fill_cache(cache, seed, 0, _lens(case), ATT_KSTD)
    return t, s, b, cache


def _attend_prefill_inputs(case, seed):
    H, KV, hd, R, n = case["H"], case["KV"], case["hd"], case["R"], case["R"] + case["p0"]
    g = _gen(seed, 2)
    cache = (torch.zeros((1, KV, n, hd), dtype=I16, device=DEV), torch.zeros((1, KV, n), dtype=I32, device=DEV),
             torch.zeros((1, KV, n, hd), dtype=I64, device=DEV))
    _fill_cache(cache, seed, 0, [n], ATT_KSTD)
    q, s = _qrow(_q16(g, (R, H, hd), 1.0), 15)
    return q.to(I16).contiguous(), s[..., 0].to(I32).contiguous(), cache


def _linear_inputs(case, seed):
    """int8 weights of a clipped N(0, 40^2), (K, N); int16 scales (K / 128, N); activation rows"""
    g, lim = _gen(seed, 3), (1 << case["abits"]) - 1
    w = (torch.randn((case["K"], case["N"]), generator=g, device=DEV) * 40).round().clamp(-127, 127).to(torch.int8)
    m = torch.randint(synth.M_LO, synth.M_HI, (case["K"] // 128, case["N"]), generator=g, device=DEV, dtype=I16)
    x = torch.randint(-lim, lim + 1, (case["R"], case["K"]), generator=g, device=DEV, dtype=torch.int8 if lim < 128 else I16)
    return w, m, x


def _dropin_shapes(case):
    """(N, K, which calls share an activation row) of the case's calls"""
    if not case["model"]:
        return [(case["N"], case["K"], 0)]
    c = synth.CONFIGS[case["model"]]
    att, kv = c.H * c.hd, c.KV * c.hd
    return [(att, c.D, 0), (kv, c.D, 0), (kv, c.D, 0), (c.D, att, 1), (c.I, c.D, 2), (c.I, c.D, 2), (c.D, c.I, 3)]


def _dropin_inputs(case, seed):
    g, shapes, lins, rows = _gen(seed, 4), _dropin_shapes(case), [], {}
    for N, K, i in shapes:
        w = (torch.randn((N, K), generator=g, device=DEV) * 40).round().clamp(-127, 127).to(torch.int8)
        M = torch.randint(synth.M_LO, synth.M_HI, (N, K // 128), generator=g, device=DEV, dtype=I64)
        lins.append((w, M))
        if i not in rows:
            rows[i] = (torch.randn(K, generator=g, device=DEV) * 8000).round().clamp(-32767, 32767).to(I16)
    return [rows[i] for _, _, i in shapes], lins


def _sample_inputs(case, seed):
    return _q16(_gen(seed, 5), (case["R"], case["V"]), 3.0), torch.arange(case["R"], dtype=I32, device=DEV) * 17 + 3


def prepare(case, seed):
    k = case["kind"]
    if k in ("decode", "prefill"):
        cfg = synth.CONFIGS[case["model"]]
        B = case.get("B", 1)
        tm = TModel(DeviceWeights.synthetic(cfg, seed, DEV, layers=case["layers"]), Smax=case["Smax"], batch=B)
        cache = tm.new_cache()
        if k == "prefill":
            st = dict(case, tm=tm, cache=cache, ids=_tokens(seed, case["T"], cfg.V))
            tm.forward(st["ids"], cache, last_only=True, graph=case["graph"])   # a server's warm-up (and capture)
            return st
        lens = _lens(case)
        for li, layer in enumerate(cache.layers):
            _fill_cache(layer, seed, li, lens, MODEL_KSTD)
        cache.n = list(lens)
        gd = GraphDecoder(tm, cache, B)
        toks = _tokens(seed, B, cfg.V)
        gd.load(toks)
        gd.capture()
        return dict(case, gd=gd, cache=cache, lens=lens, toks=toks)
    if k == "attend":
        t, s, b, cache = _attend_inputs(case, seed)
        R, H, hd = case["R"], case["H"], case["hd"]
        return dict(case, t=t, s=s, b=b, cache=cache, tab=DeviceTables(DEV, case["Smax"], hd, 1e6),
                    slot=torch.arange(R, dtype=I32, device=DEV), pos=torch.tensor(_lens(case), dtype=I32, device=DEV),
                    out=torch.zeros((R, H * hd), dtype=I64, device=DEV),
                    obits=torch.zeros((R, H * ops.ATT_SPLIT_MAX), dtype=I32, device=DEV))
    if k == "attend_prefill":
        qq, sq, cache = _attend_prefill_inputs(case, seed)
        R, H, hd, n = case["R"], case["H"], case["hd"], case["R"] + case["p0"]
        return dict(case, qq=qq, sq=sq, cache=cache, tab=DeviceTables(DEV, n, hd, 1e6),
                    pos=torch.arange(case["p0"], n, dtype=I32, device=DEV),
                    out=torch.zeros((R, H * hd), dtype=I64, device=DEV), obits=torch.zeros((R, H), dtype=I32, device=DEV),
                    ws=ops.prefill_workspace(R, H, case["KV"], hd, n, DEV))
    if k == "linear":
        w, m, x = _linear_inputs(case, seed)
        wp, mp = ops.pack_linear(w, m)
        lin = ops.PackedLinear(wp, mp, case["N"], case["K"])
        out = torch.zeros((case["R"], case["N"]), dtype=I64, device=DEV)
        ops.linear_t(x, case["abits"], lin, out)   # the linear's cached column term is made on its first call
        return dict(case, x=x, lin=lin, out=out)
    if k == "dropin":
        xs, lins = _dropin_inputs(case, seed)
        calls = lambda: [torch.ops.exact.gemv(x, w, M) for x, (w, M) in zip(xs, lins)]
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            calls()
        torch.cuda.current_stream().wait_stream(side)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            outs = calls()
        return dict(case, xs=xs, lins=lins, graph=g, outs=outs)
    lg, step = _sample_inputs(case, seed)
    return dict(case, lg=lg, step=step, seed=seed, tnum=ops.temp_num(case["temp"]), tab=DeviceTables(DEV, 1, 64, 1e6),
                ids=torch.zeros(case["R"], dtype=I32, device=DEV))


def run(st):
    k = st["kind"]
    if k == "decode":
        gd, cache = st["gd"], st["cache"]
        cache.n = list(st["lens"])
        gd.load(st["toks"])
        ids = []
        for _ in range(st["steps"]):
            lg, nid = gd.step()
            ids.append(nid.clone())
        return dict(logits=lg, ids=ids, cache=cache.layers[-1])
    if k == "prefill":
        cache = st["cache"]
        cache.n = [0]
        lg = st["tm"].forward(st["ids"], cache, last_only=True, graph=st["graph"])
        return dict(logits=lg, cache=cache.layers[-1])
    if k == "attend":
        tab = st["tab"]
        ops.attention_qkv(st["t"], st["s"], st["b"], tab.cos, tab.sin, st["slot"], st["pos"], st["cache"], tab.exp, st["out"],
                          st["H"], st["KV"], st["hd"], tab.inv, st["obits"], obn=ops.ATT_SPLIT_MAX)
        return dict(out=st["out"], cache=st["cache"])
    if k == "attend_prefill":
        tab = st["tab"]
        ops.attention_prefill(st["qq"], st["sq"], st["cache"], 0, st["pos"], st["R"] + st["p0"], tab.exp, st["out"], st["H"],
                              st["KV"], st["hd"], tab.inv, st["ws"], st["obits"])
        return dict(out=st["out"], obits=st["obits"])
    if k == "linear":
        return ops.linear_t(st["x"], st["abits"], st["lin"], st["out"])
    if k == "dropin":
        st["graph"].replay()
        return st["outs"]
    return ops.sample(st["lg"], st["seed"], st["step"], st["tnum"], st["tab"].exp, st["ids"])


# ----------------------------------------------------------------------------- work and tolerance
def _lin_bytes(N, K):
    return N * K + N * (K // 128) * 2


def _model_work(case):
    """bytes and integer operations of the model's linears and attention for the rows of one pass"""
    c, nl = synth.CONFIGS[case["model"]], case["layers"]
    rows = case["B"] if case["kind"] == "decode" else case["T"]
    att, kv = c.H * c.hd, c.KV * c.hd
    shapes = [(att + 2 * kv, c.D), (c.D, att)]
    flops = sum(2 * rows * N * K for N, K in shapes)
    nbytes = sum(_lin_bytes(N, K) for N, K in shapes)
    if c.moe:
        pairs = rows * c.topk
        # experts that rows * topk independent choices reach
        e = c.NE * (1 - (1 - c.topk / c.NE) ** rows)
        for N, K in ((c.NE + 1, c.D), (2 * c.SI, c.D), (c.D, c.SI)):
            nbytes, flops = nbytes + _lin_bytes(N, K), flops + 2 * rows * N * K
        for N, K in ((2 * c.MI, c.D), (c.D, c.MI)):
            nbytes, flops = nbytes + e * _lin_bytes(N, K), flops + 2 * pairs * N * K
    else:
        for N, K in ((2 * c.I, c.D), (c.D, c.I)):
            nbytes, flops = nbytes + _lin_bytes(N, K), flops + 2 * rows * N * K
    keys = sum(n + 1 for n in _lens(case)) if case["kind"] == "decode" else case["T"]
    pairs = keys if case["kind"] == "decode" else case["T"] * (case["T"] + 1) // 2
    nbytes += keys * c.KV * (c.hd * 10 + 4)
    flops += 4 * pairs * c.H * c.hd
    hr = case["B"] if case["kind"] == "decode" else 1
    return nl * nbytes + _lin_bytes(c.V, c.D) + 8 * hr * c.V, nl * flops + 2 * hr * c.V * c.D


def work(case):
    k = case["kind"]
    if k in ("decode", "prefill"):
        nbytes, flops = _model_work(case)
        n = case.get("steps", 1)
        return dict(bytes=n * nbytes, flops=n * flops)
    if k in ("attend", "attend_prefill"):
        H, KV, hd, R = case["H"], case["KV"], case["hd"], case["R"]
        if k == "attend":
            keys = pairs = sum(n + 1 for n in _lens(case))
            rows = R * (H + 2 * KV) * hd * 8 + R * H * hd * 8
        else:
            keys, pairs = R + case["p0"], R * case["p0"] + R * (R + 1) // 2
            rows = R * H * hd * 10
        return dict(bytes=keys * KV * (hd * 10 + 4) + rows, flops=4 * pairs * H * hd)
    if k == "linear":
        R, N, K = case["R"], case["N"], case["K"]
        return dict(bytes=_lin_bytes(N, K) + R * K * (1 if case["abits"] == 7 else 2) + 8 * R * N, flops=2 * R * N * K)
    if k == "dropin":
        n = _dropin_shapes(case)
        return dict(bytes=sum(N * K + N * (K // 128) * 8 + 8 * N + 2 * K for N, K, _ in n), flops=sum(2 * N * K for N, K, _ in n))
    return dict(bytes=8 * case["R"] * case["V"], flops=20 * case["R"] * case["V"])


def tolerance(case):
    return "exact"   # an integer program: every output is the same bits on every conforming device


# ----------------------------------------------------------------------------- the program in plain torch
M64 = (1 << 64) - 1


def _s64(x):
    x &= M64
    return x - (1 << 64) if x >> 63 else x


def _mix64(z):
    z &= M64
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & M64
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & M64
    return z ^ (z >> 31)


def _key(seed, name):
    h = 0xCBF29CE484222325
    for b in name.encode():
        h = ((h ^ b) * 0x100000001B3) & M64
    return _mix64((seed * 0x9E3779B97F4A7C15) ^ h)


def _u32(key, idx):
    """the 32-bit uniform of SplitMix64 counter idx, as int64"""
    lsr = lambda a, n: (a >> n) & ((1 << (64 - n)) - 1)
    z = (idx + 1) * _s64(0x9E3779B97F4A7C15) + _s64(key)
    z = (z ^ lsr(z, 30)) * _s64(0xBF58476D1CE4E5B9)
    z = (z ^ lsr(z, 27)) * _s64(0x94D049BB133111EB)
    return lsr(z ^ lsr(z, 31), 32)


def _vector(key, n, lo, hi):
    return lo + ((_u32(key, torch.arange(n, device=DEV)) * (hi - lo)) >> 32)


def _weights(key, n, K):
    """W (len(n), K) of a synthetic matrix's output rows n: clipped N(0, 40^2)"""
    thr = [min(int(round(0.5 * math.erfc(-(j - 126.5) / 40.0 / math.sqrt(2.0)) * 2 ** 32)), 2 ** 32 - 1) for j in range(254)]
    u = _u32(key, n[:, None] * K + torch.arange(K, device=DEV)[None])
    return torch.searchsorted(torch.tensor(thr, device=DEV), u, right=True) - 127


def _scales(key, n, K):
    """M (len(n), K / 128)"""
    G = K // 128
    u = _u32(key, n[:, None] * G + torch.arange(G, device=DEV)[None])
    return synth.M_LO + ((u * (synth.M_HI - synth.M_LO)) >> 32)


def _shr(a, n):
    n = torch.as_tensor(n, device=a.device, dtype=I64)
    r, left = n.clamp(min=0), (-n).clamp(min=0)
    half = torch.where(r > 0, torch.ones_like(r) << (r - 1).clamp(min=0), torch.zeros_like(r))
    return ((a + half) >> r) << left


def _bitlen(m):
    return torch.where(m > 0, torch.frexp(m.double())[1].to(I64), torch.zeros_like(m))


def _qrow(x, bits):
    s = (_bitlen(x.abs().amax(-1, keepdim=True)) - bits).clamp(min=0)
    lim = (1 << bits) - 1
    return _shr(x, s).clamp(-lim, lim), s


def _irms(x, g):
    k = (_bitlen(x.abs().amax(-1, keepdim=True)) - 24).clamp(min=0)
    xs = _shr(x, k)
    ms = (xs * xs).sum(-1, keepdim=True) // x.shape[-1] + 1
    r = ms.double().sqrt().to(I64)
    r = torch.where(r * r > ms, r - 1, r)
    r = torch.where((r + 1) * (r + 1) <= ms, r + 1, r).clamp(min=1)
    return _shr(torch.div(x << 16, r << k, rounding_mode="floor") * g, 16)


EXP = [round(math.exp(-i / 256) * (1 << 24)) for i in range(256 * 40 + 2)]


def _softmax(sc, valid=None):
    """Q20 probabilities of the valid entries of each row"""
    T = torch.tensor(EXP, device=DEV)
    if valid is not None:
        sc = torch.where(valid, sc, torch.full_like(sc, -(1 << 60)))
    d = sc.amax(-1, keepdim=True) - sc
    i = (d >> 8).clamp(max=len(EXP) - 2)
    e = T[i] - _shr((T[i] - T[i + 1]) * (d & 255), 8)
    e = torch.where(d < (40 << 16), e, torch.zeros_like(e))
    if valid is not None:
        e = torch.where(valid, e, torch.zeros_like(e))
    return (e << 20) // e.sum(-1, keepdim=True)


def _lut16(x, fn, top):
    T = torch.tensor([round(fn((i - 4096) / 256) * ONE) for i in range(32 * 256 + 2)], device=DEV)
    t = (x + (16 << 16)).clamp(0, (32 << 16) - 1)
    a, b = T[t >> 8], T[(t >> 8) + 1]
    y = a + _shr((b - a) * (t & 255), 8)
    y = torch.where(x >= (16 << 16), x if top is None else torch.full_like(x, top), y)
    return torch.where(x < -(16 << 16), torch.zeros_like(x), y)


def _silu(x):
    return _lut16(x, lambda v: v / (1 + math.exp(-v)), None)


def _sig(x):
    return _lut16(x, lambda v: 1 / (1 + math.exp(-v)), ONE)


def _group_dot(xq, W, M):
    """sum_g (xq_g . W_g) M_g: xq (R, K), W (N, K), M (N, K / 128)"""
    t = torch.zeros((xq.shape[0], W.shape[0]), dtype=I64, device=DEV)
    x, w = xq.double(), W.double()
    for g in range(xq.shape[1] // 128):
        t += (x[:, 128 * g:128 * g + 128] @ w[:, 128 * g:128 * g + 128].T).to(I64) * M[:, g].to(I64)[None]
    return t


def _linear(seed, name, N, K, xq, s, bias=False):
    """shr(t, 28 - s) + b of the named synthetic linear"""
    out = []
    for n0 in range(0, N, 16384):
        n = torch.arange(n0, min(N, n0 + 16384), device=DEV)
        out.append(_group_dot(xq, _weights(_key(seed, name + ".w"), n, K), _scales(_key(seed, name + ".m"), n, K)))
    y = _shr(torch.cat(out, 1), 28 - s)
    return y + _vector(_key(seed, name + ".b"), N, *synth.BIAS) if bias else y


def _rope(y, pos, hd, theta=1e6):
    """y (R, heads, hd) at positions pos (R,)"""
    ang = pos.cpu().numpy().astype(np.float64)[:, None] * (1.0 / theta ** (np.arange(0, hd, 2, dtype=np.float64) / hd))[None]
    ang = np.concatenate([ang, ang], -1)
    cos, sin = (torch.tensor(np.rint(f(ang) * ONE).astype(np.int64), device=DEV)[:, None] for f in (np.cos, np.sin))
    rot = torch.cat([-y[..., hd // 2:], y[..., :hd // 2]], -1)
    return _shr(y * cos + rot * sin, 16)


def _attention(qq, sq, kq, sk, v, last):
    """rows qq (R, H, hd), sq (R, H) over one sequence's kq (KV, S, hd), sk (KV, S), v (KV, S, hd), keys 0..last[r]"""
    R, H, hd = qq.shape
    KV, S = kq.shape[:2]
    inv = int(round(ONE / math.sqrt(hd)))
    valid = torch.arange(S, device=DEV)[None] <= last[:, None]
    out = torch.empty((R, H, hd), dtype=I64, device=DEV)
    for h in range(H):
        kh = h // (H // KV)
        dot = (qq[:, h].double() @ kq[kh].double().T).to(I64)
        p = _softmax(_shr(dot * inv, 32 - sq[:, h].to(I64)[:, None] - sk[kh].to(I64)[None]), valid)
        out[:, h] = _shr((p.double() @ v[kh].double()).to(I64), 20)
    return out.reshape(R, H * hd)


def _qkv(y, H, KV, hd, pos):
    """y (R, (H + 2 KV) hd): quantised queries and keys with their shifts, and values"""
    R = y.shape[0]
    q, k, v = (t.reshape(R, -1, hd) for t in y.split([H * hd, KV * hd, KV * hd], 1))
    qq, sq = _qrow(_rope(q, pos, hd), 15)
    kq, sk = _qrow(_rope(k, pos, hd), 15)
    return qq, sq[..., 0], kq, sk[..., 0], v


def _moe(c, seed, li, xq, s):
    """the experts' weighted sum and the gated shared expert of the quantised rows xq"""
    def mlp(pre, g, u, d, I, xq, s):
        h = _shr(_silu(_linear(seed, pre + g, I, c.D, xq, s)) * _linear(seed, pre + u, I, c.D, xq, s), 16)
        return _linear(seed, pre + d, c.D, I, *_qrow(h, 15))

    p = _softmax(_linear(seed, f"L{li}.router", c.NE, c.D, xq, s))
    sel = torch.sort(p, dim=1, descending=True, stable=True)[1][:, :c.topk]
    out = torch.zeros((xq.shape[0], c.D), dtype=I64, device=DEV)
    for e in range(c.NE):
        r = torch.nonzero((sel == e).any(1))[:, 0]
        if len(r):
            out[r] += _shr(p[r, e][:, None] * mlp(f"L{li}.e{e}.", "gate", "up", "down", c.MI, xq[r], s[r]), 20)
    gate = _sig(_linear(seed, f"L{li}.sgate", 1, c.D, xq, s))
    return out + _shr(gate * mlp(f"L{li}.", "sg", "su", "sd", c.SI, xq, s), 16)


def _forward(c, nl, seed, ids, slot, pos, caches):
    """hidden rows of tokens ids at (slot, pos); the keys and values go into caches"""
    n = torch.tensor(ids, device=DEV)
    a = _weights(_key(seed, "emb.w"), n, c.D) * _scales(_key(seed, "emb.m"), n, c.D).repeat_interleave(128, 1)
    q, rem = a >> 12, a & 4095
    x = q + ((rem > 2048) | ((rem == 2048) & ((q & 1) == 1))).to(I64)
    for li in range(nl):
        gain = lambda name: _vector(_key(seed, f"L{li}.{name}"), c.D, *synth.GAIN)
        xq, s = _qrow(_irms(x, gain("g1")), 15)
        y = torch.cat([_linear(seed, f"L{li}.{p}", h * c.hd, c.D, xq, s, True) for p, h in (("q", c.H), ("k", c.KV), ("v", c.KV))], 1)
        qq, sq, kq, sk, v = _qkv(y, c.H, c.KV, c.hd, pos)
        ck, cs, cv = caches[li]
        ck[slot, :, pos], cs[slot, :, pos], cv[slot, :, pos] = kq.to(I16), sk.to(I32), v
        att = torch.cat([_attention(qq[slot == b], sq[slot == b], *(t[b][:, :int(pos[slot == b].max()) + 1] for t in caches[li]),
                                    pos[slot == b]) for b in sorted(set(slot.tolist()))])
        x = x + _linear(seed, f"L{li}.o", c.D, c.H * c.hd, *_qrow(att, 15))
        xq, s = _qrow(_irms(x, gain("g2")), 15)
        if c.moe:
            x = x + _moe(c, seed, li, xq, s)
            continue
        h = _shr(_silu(_linear(seed, f"L{li}.gate", c.I, c.D, xq, s)) * _linear(seed, f"L{li}.up", c.I, c.D, xq, s), 16)
        x = x + _linear(seed, f"L{li}.down", c.D, c.I, *_qrow(h, 15))
    return x


def _logits(c, seed, x):
    xq, s = _qrow(_irms(x, _vector(_key(seed, "gf"), c.D, *synth.GAIN)), 15)
    return _linear(seed, "emb" if c.tie else "head", c.V, c.D, xq, s)


def _exact_model(case, seed):
    c, nl, Smax = synth.CONFIGS[case["model"]], case["layers"], case["Smax"]
    B = case.get("B", 1)
    caches = [(torch.zeros((B, c.KV, Smax, c.hd), dtype=I16, device=DEV), torch.zeros((B, c.KV, Smax), dtype=I32, device=DEV),
               torch.zeros((B, c.KV, Smax, c.hd), dtype=I64, device=DEV)) for _ in range(nl)]
    if case["kind"] == "prefill":
        T = case["T"]
        x = _forward(c, nl, seed, _tokens(seed, T, c.V), torch.zeros(T, dtype=I64, device=DEV), torch.arange(T, device=DEV), caches)
        return dict(logits=_logits(c, seed, x[-1:]), cache=caches[-1])
    for li, layer in enumerate(caches):
        _fill_cache(layer, seed, li, _lens(case), MODEL_KSTD)
    toks, ids, pos = _tokens(seed, B, c.V), [], torch.tensor(_lens(case), device=DEV)
    for _ in range(case["steps"]):
        lg = _logits(c, seed, _forward(c, nl, seed, toks, torch.arange(B, device=DEV), pos, caches))
        nid = torch.tensor([int(torch.nonzero(r == r.max())[0, 0]) for r in lg], dtype=I32, device=DEV)
        ids.append(nid)
        toks, pos = nid.tolist(), pos + 1
    return dict(logits=lg, ids=ids, cache=caches[-1])


def exact(case, seed):
    k = case["kind"]
    if k in ("decode", "prefill"):
        return _exact_model(case, seed)
    if k == "attend":
        t, s, b, cache = _attend_inputs(case, seed)
        H, KV, hd = case["H"], case["KV"], case["hd"]
        pos = torch.tensor(_lens(case), device=DEV)
        qq, sq, kq, sk, v = _qkv(_shr(t, 28 - s.to(I64)[:, None]) + b, H, KV, hd, pos)
        r = torch.arange(case["R"], device=DEV)
        cache[0][r, :, pos], cache[1][r, :, pos], cache[2][r, :, pos] = kq.to(I16), sk.to(I32), v
        out = [_attention(qq[i:i + 1], sq[i:i + 1], *(c[i][:, :int(pos[i]) + 1] for c in cache), pos[i:i + 1]) for i in range(case["R"])]
        return dict(out=torch.cat(out), cache=cache)
    if k == "attend_prefill":
        qq, sq, cache = _attend_prefill_inputs(case, seed)
        out = _attention(qq, sq, *(c[0] for c in cache), torch.arange(case["p0"], case["p0"] + case["R"], device=DEV))
        return dict(out=out, obits=_bitlen(out.reshape(case["R"], case["H"], -1).abs().amax(-1)).to(I32))
    if k == "linear":
        w, m, x = _linear_inputs(case, seed)
        return _group_dot(x, w.T, m.T)
    if k == "dropin":
        xs, lins = _dropin_inputs(case, seed)
        return [_group_dot(x[None], w, M)[0] for x, (w, M) in zip(xs, lins)]
    lg, step = _sample_inputs(case, seed)
    cum = _softmax(_shr(lg * int(round(ONE / case["temp"])), 16)).cumsum(1)
    u = [(_mix64(seed + (s + 1) * 0x9E3779B97F4A7C15)) >> 44 for s in step.tolist()]
    target = (torch.tensor(u, device=DEV)[:, None] * cum[:, -1:]) >> 20
    return torch.searchsorted(cum, target, right=True)[:, 0].to(I32)
