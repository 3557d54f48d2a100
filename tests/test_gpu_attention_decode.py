"""Decode attention split over the keys (exact_attention_decode) against the two launches exact_qkv_rope_cache +
exact_attention, which the oracle pins: every output, cache entry and bit length equal."""
import numpy as np
import pytest
import torch

import exact_oracle as O
from exact_amd import ops, synth
from exact_amd.tables import exp_t, host_tables

pytestmark = pytest.mark.gpu
DEV = "cuda"
I8, I16, I32, I64 = torch.int8, torch.int16, torch.int32, torch.int64


def dev(a, dt):
    return torch.tensor(np.ascontiguousarray(a), dtype=dt, device=DEV)


def compare(H, KV, hd, Smax, pos, seed, vmag=29, table=None, obn=4, bias=True):
    """both paths on random caches (int16 keys over their whole range) with the rows at pos, in permuted slots"""
    rng = np.random.default_rng(seed)
    R, N = len(pos), (H + 2 * KV) * hd
    B = R + 1
    kq = rng.integers(-32767, 32768, (B, KV, Smax, hd))
    sk = rng.integers(0, 4, (B, KV, Smax))
    v = rng.integers(-(1 << vmag), 1 << vmag, (B, KV, Smax, hd))
    t = dev(rng.integers(-(1 << 44), 1 << 44, (R, N)), I64)
    s = dev(rng.integers(0, 12, R), I32)
    b = dev(rng.integers(-(1 << 20), 1 << 20, N), I64) if bias else None
    slot, pos = dev(rng.permutation(B)[:R], I32), dev(pos, I32)
    tabs = host_tables(Smax, hd, 1e6)
    cos, sin, expt = dev(tabs["cos"], I64), dev(tabs["sin"], I64), dev(exp_t() if table is None else table, I32)
    c_a = (dev(kq, I16), dev(sk, I32), dev(v, I64))
    c_b = tuple(x.clone() for x in c_a)
    qq, sq = torch.empty((R, H * hd), dtype=I16, device=DEV), torch.empty((R, H), dtype=I32, device=DEV)
    out_a, out_b = (torch.full((R, H * hd), x, dtype=I64, device=DEV) for x in (-7, -9))
    ob_a, ob_b = torch.full((R, H), -1, dtype=I32, device=DEV), torch.full((R, H, obn), -2, dtype=I32, device=DEV)
    inv, t0 = O.inv_sqrt_hd(hd), t.clone()
    ops.qkv_rope_cache(t, s, b, cos, sin, slot, pos, c_a, qq, sq, H, KV, hd)
    ops.attention(qq, sq, c_a, slot, pos, expt, out_a, H, KV, hd, inv, ob_a)
    work = ops.attention_work(R, H, KV, hd, Smax, DEV).fill_(0x5A)   # holds anything on entry
    ops._lib.call("exact_attention_decode", *(ops._ptr(x) for x in (t, s, b, cos, sin, slot, pos, *c_b, expt, out_b, ob_b)), obn,
                  ops._ptr(work), work.numel(), R, H, KV, hd, Smax, inv, ops._stream())
    assert torch.equal(out_b, out_a)
    assert torch.equal(ob_b.max(-1)[0], ob_a)
    assert all(torch.equal(x, y) for x, y in zip(c_b, c_a))
    assert torch.equal(t, t0)
    return out_a


# chunks of 128 keys: the first and last position of one, of the cache, and a cache of no whole chunks
@pytest.mark.parametrize("H,KV,hd,Smax,pos", [
    (7, 1, 128, 400, [0, 1, 127, 128, 129, 255, 256, 399]), (14, 2, 64, 129, [128, 127, 0]), (8, 1, 128, 1000, [999, 640]),
    (8, 1, 64, 300, [299, 3]), (10, 2, 128, 640, [639, 511, 512]), (4, 1, 128, 200, [130]), (4, 2, 64, 257, [256, 100]),
    (3, 3, 128, 300, [299, 127, 0]), (2, 2, 64, 8192, [8191, 8064]), (7, 1, 128, 8192, [8191])])
@pytest.mark.parametrize("obn", [1, 4])
def test_split_matches_two_launches(H, KV, hd, Smax, pos, obn):
    compare(H, KV, hd, Smax, pos, H * Smax + hd, obn=obn, bias=obn == 4)


def test_split_extreme_values_and_tables():
    """values of more than 31 bits take 64-bit products; a table with negative entries gives p outside [0, 2^31), a table of
    zeros gives 0"""
    compare(7, 1, 128, 300, [299, 130], 3, vmag=62)
    T = exp_t().copy()
    T[1:40] = -T[1:40] // 3
    compare(7, 1, 128, 300, [299, 130], 4, table=T)
    T = exp_t().copy()
    T[2:] = -(T[0] // 300)
    compare(4, 1, 64, 600, [599, 290], 5, table=T, vmag=40)
    assert not compare(4, 2, 128, 200, [199], 6, table=np.zeros_like(exp_t())).any()


@pytest.mark.parametrize("hd,obn", [(64, 4), (128, 1)])
def test_split_positions_outside_the_cache_give_zeros(hd, obn):
    """rows at positions -1 and Smax, on either path: outputs and bit lengths 0, the cache as it was"""
    H, KV, Smax = 4, 2, 256
    rng = np.random.default_rng(hd)
    d = lambda lo, hi, sh, dt: dev(rng.integers(lo, hi, sh), dt)
    kv = (d(-32767, 32768, (2, KV, Smax, hd), I16), d(0, 4, (2, KV, Smax), I32), d(-(1 << 29), 1 << 29, (2, KV, Smax, hd), I64))
    t, s = d(-(1 << 44), 1 << 44, (2, (H + 2 * KV) * hd), I64), d(0, 12, 2, I32)
    tabs = host_tables(Smax, hd, 1e6)
    cos, sin, expt = dev(tabs["cos"], I64), dev(tabs["sin"], I64), dev(exp_t(), I32)
    slot, pos, inv = dev([0, 1], I32), dev([-1, Smax], I32), O.inv_sqrt_hd(hd)
    work = ops.attention_work(2, H, KV, hd, Smax, DEV).fill_(0x5A)

    def one_launch(cache, out, ob):
        ops.attention_qkv(t, s, None, cos, sin, slot, pos, cache, expt, out, H, KV, hd, inv, ob, obn=obn, keys=1)

    def split(cache, out, ob):
        ops._lib.call("exact_attention_decode", *(ops._ptr(x) for x in (t, s, None, cos, sin, slot, pos, *cache, expt, out, ob)),
                      obn, ops._ptr(work), work.numel(), 2, H, KV, hd, Smax, inv, ops._stream())

    for path in (one_launch, split):
        cache = tuple(x.clone() for x in kv)
        out, ob = torch.full((2, H * hd), -1, dtype=I64, device=DEV), torch.full((2, H, obn), -1, dtype=I32, device=DEV)
        path(cache, out, ob)
        assert not out.any() and not ob.any(), path.__name__
        assert all(torch.equal(x, y) for x, y in zip(cache, kv)), path.__name__


@pytest.mark.parametrize("B", [1, 3])
def test_graph_decode_crosses_into_the_split(B, monkeypatch):
    """Steps over the position from which attention is split (their graphs differ) give the same tokens and logits as the
    one-launch attention throughout."""
    from exact_amd.model import DeviceWeights, GraphDecoder, TModel
    cfg = synth.CONFIGS["tiny-hd128"]
    got = []
    for work in (50 * 128, 1 << 30):
        monkeypatch.setattr(ops, "ATT_SHORT_CACHE", 0)
        monkeypatch.setattr(ops, "ATT_KEYS_WORK", work)
        tm = TModel(DeviceWeights.synthetic(cfg, 3, DEV), Smax=96, batch=B)
        cache = tm.new_cache()
        for b in range(B):
            tm.forward([(7 * i + b) % cfg.V for i in range(47 - b)], cache, last_only=True, slot=b)
        gd = GraphDecoder(tm, cache, B)
        gd.load([5 + b for b in range(B)])
        gd.capture()
        assert len(gd.graphs) == (2 if work < 1 << 30 else 1)
        rows = []
        for _ in range(8):
            lg, ids = gd.step()
            rows.append((lg.clone(), ids.clone()))
        got.append(rows)
        lg, _ = tm.decode_rows(rows[-1][1].tolist(), cache)   # eager, past the line
        rows.append((lg, lg))
    for (a, i), (b, j) in zip(*got):
        assert torch.equal(a, b) and torch.equal(i, j)


def test_grouped_batch_attention_of_eight_heads():
    """One KV head of eight query heads over a cache of 193 to 256 positions in several rounds of blocks"""
    rng = np.random.default_rng(8)
    R, H, KV, hd, Smax = 40, 8, 1, 128, 224
    d = lambda lo, hi, sh, dt: dev(rng.integers(lo, hi, sh), dt)
    t, s = d(-(1 << 44), 1 << 44, (R, (H + 2 * KV) * hd), I64), d(0, 12, R, I32)
    c_a = (d(-32767, 32768, (R, KV, Smax, hd), I16), d(0, 4, (R, KV, Smax), I32), d(-(1 << 29), 1 << 29, (R, KV, Smax, hd), I64))
    c_b = tuple(x.clone() for x in c_a)
    slot, pos = torch.arange(R, dtype=I32, device=DEV), d(0, Smax, R, I32)
    tabs = host_tables(Smax, hd, 1e6)
    cos, sin, expt = dev(tabs["cos"], I64), dev(tabs["sin"], I64), dev(exp_t(), I32)
    qq, sq = torch.empty((R, H * hd), dtype=I16, device=DEV), torch.empty((R, H), dtype=I32, device=DEV)
    out_a, out_b = torch.zeros((R, H * hd), dtype=I64, device=DEV), torch.ones((R, H * hd), dtype=I64, device=DEV)
    inv = O.inv_sqrt_hd(hd)
    ops.qkv_rope_cache(t, s, None, cos, sin, slot, pos, c_a, qq, sq, H, KV, hd)
    ops.attention(qq, sq, c_a, slot, pos, expt, out_a, H, KV, hd, inv)
    ops.attention_qkv(t, s, None, cos, sin, slot, pos, c_b, expt, out_b, H, KV, hd, inv, obn=4, keys=1)
    assert torch.equal(out_a, out_b) and all(torch.equal(x, y) for x, y in zip(c_a, c_b))


def test_captured_again_for_another_cache_over_the_line(monkeypatch):
    """A decoder captured below the position from which attention is split, then again with another cache above it: every
    later step, short positions among them, reads and writes that cache, and short positions keep the one launch"""
    from exact_amd.model import DeviceWeights, GraphDecoder, TModel
    monkeypatch.setattr(ops, "ATT_SHORT_CACHE", 0)
    monkeypatch.setattr(ops, "ATT_KEYS_WORK", 50 * 128)
    cfg = synth.CONFIGS["tiny-hd128"]
    tm = TModel(DeviceWeights.synthetic(cfg, 3, DEV), Smax=96)
    prompt = lambda n: [(11 * i + 3) % cfg.V for i in range(n)]
    want, ref = [], tm.new_cache()
    for n in (60, 20):
        ref.n[0] = 0
        tm.forward(prompt(n), ref, last_only=True)
        want.append([x.clone() for x in tm.decode_rows([5], ref)])
    first, cache = tm.new_cache(), tm.new_cache()
    tm.forward(prompt(12), first, last_only=True)
    gd = GraphDecoder(tm, first, 1)
    gd.load([5])
    gd.capture()
    old = [[x.clone() for x in layer] for layer in first.layers]
    gd.cache = cache
    for i, n in enumerate((60, 20)):
        cache.n[0] = 0
        tm.forward(prompt(n), cache, last_only=True)
        gd.load([5])
        if i == 0:
            gd.capture()
        assert gd._split() == (n == 60) and set(gd.graphs) == {(False, 0), (True, 0)}
        assert all(torch.equal(x, y) for x, y in zip(gd.step(), want[i])), n
    assert all(torch.equal(x, y) for a, b in zip(old, first.layers) for x, y in zip(a, b))
    assert all(torch.equal(x[:, :, :21], y[:, :, :21]) for a, b in zip(cache.layers, ref.layers) for x, y in zip(a, b))


def test_cache_longer_than_the_model(monkeypatch):
    """A cache made for more positions than the model's own: the split's workspace goes by the cache, before and after one of
    the model's length has been used"""
    from exact_amd.model import Cache, DeviceWeights, GraphDecoder, TModel
    monkeypatch.setattr(ops, "ATT_SHORT_CACHE", 0)
    monkeypatch.setattr(ops, "ATT_KEYS_WORK", 50 * 128)
    monkeypatch.setattr(ops, "ATT_EAGER_KEYS", {False: (50, 50), True: (50, 50)})
    cfg = synth.CONFIGS["tiny-hd128"]
    tm = TModel(DeviceWeights.synthetic(cfg, 3, DEV), Smax=96)
    prompt = [(11 * i + 3) % cfg.V for i in range(60)]
    got, kept = [], []
    for Smax in (96, 700, 96, 300):
        cache = Cache(cfg, 1, Smax, tm.dev, cfg.NL)
        tm.forward(prompt, cache, last_only=True)
        rows = [[x.clone() for x in tm.decode_rows([5], cache)]]
        cache.n[0] = 60
        gd = GraphDecoder(tm, cache, 1)
        gd.load([5])
        gd.capture()
        assert gd._split()
        rows.append([x.clone() for x in gd.step()])
        got.append(rows)
        kept.append((gd, cache))
    for gd, cache in kept:   # the captured steps still hold their own buffers
        cache.n[0] = 60
        gd.load([5])
        got.append([[x.clone() for x in gd.step()]])
    assert set(tm.workspace(1).att_work) == {96, 300, 700}
    assert all(torch.equal(x, y) for rows in got for r in rows for x, y in zip(r, got[0][0]))


@pytest.mark.parametrize("H,KV,hd", [(7, 1, 128), (4, 4, 64)])
def test_caches_off_16_bytes_stay_in_one_launch(H, KV, hd):
    """keys and values that start 8 bytes past a 16-byte boundary, at positions from which an aligned cache is split"""
    R, Smax = 2, 1700
    rng = np.random.default_rng(hd)
    d = lambda lo, hi, sh, dt: dev(rng.integers(lo, hi, sh), dt)
    t, s = d(-(1 << 44), 1 << 44, (R, (H + 2 * KV) * hd), I64), d(0, 12, R, I32)
    kv = (d(-32767, 32768, (R, KV, Smax, hd), I16), d(0, 4, (R, KV, Smax), I32), d(-(1 << 29), 1 << 29, (R, KV, Smax, hd), I64))
    slot, pos = dev([1, 0], I32), dev([1650, 900], I32)
    tabs = host_tables(Smax, hd, 1e6)
    cos, sin, expt = dev(tabs["cos"], I64), dev(tabs["sin"], I64), dev(exp_t(), I32)

    def off(x, n):   # a copy n elements past an aligned address
        y = torch.empty(x.numel() + n, dtype=x.dtype, device=DEV)[n:].view(x.shape)
        return y.copy_(x)

    got = []
    for nk, nv in ((0, 0), (4, 0), (0, 1), (4, 1)):
        cache = (off(kv[0], nk), kv[1].clone(), off(kv[2], nv))
        assert (cache[0].data_ptr() % 16, cache[2].data_ptr() % 16) == (2 * nk, 8 * nv)
        out, ob = torch.full((R, H * hd), -9, dtype=I64, device=DEV), torch.full((R, H, 4), -2, dtype=I32, device=DEV)
        ops.attention_qkv(t, s, None, cos, sin, slot, pos, cache, expt, out, H, KV, hd, O.inv_sqrt_hd(hd), ob, obn=4, keys=1651)
        got.append((out, ob.max(-1)[0], *cache))
    assert 1651 >= ops.attention_keys_from(R, H, KV, hd, Smax)
    assert all(torch.equal(x, y) for g in got[1:] for x, y in zip(g, got[0]))


@pytest.mark.parametrize("H,KV,hd", [(4, 1, 128), (5, 1, 128), (14, 2, 128), (8, 1, 128), (8, 2, 64), (7, 1, 64)])
@pytest.mark.parametrize("blocks", [257, 512, 513])
@pytest.mark.parametrize("Smax,obn", [(193, 4), (256, 1)])
def test_batch_attention_around_the_grouped_kernels_line(H, KV, hd, blocks, Smax, obn):
    """Rows in one more (row, head) block than the CUs hold, and in as many as, and more than, from which a block takes a whole
    group: equal to the two launches"""
    R = -(-blocks // H) if blocks != 512 else 512 // H
    rng = np.random.default_rng(R + hd)
    d = lambda lo, hi, sh, dt: dev(rng.integers(lo, hi, sh), dt)
    t, s = d(-(1 << 44), 1 << 44, (R, (H + 2 * KV) * hd), I64), d(0, 12, R, I32)
    c_a = (d(-32767, 32768, (R, KV, Smax, hd), I16), d(0, 4, (R, KV, Smax), I32), d(-(1 << 29), 1 << 29, (R, KV, Smax, hd), I64))
    c_b = tuple(x.clone() for x in c_a)
    slot, pos = dev(rng.permutation(R), I32), d(0, Smax, R, I32)
    pos[0], pos[1] = 0, Smax - 1
    tabs = host_tables(Smax, hd, 1e6)
    cos, sin, expt = dev(tabs["cos"], I64), dev(tabs["sin"], I64), dev(exp_t(), I32)
    qq, sq = torch.empty((R, H * hd), dtype=I16, device=DEV), torch.empty((R, H), dtype=I32, device=DEV)
    out_a, out_b = (torch.full((R, H * hd), x, dtype=I64, device=DEV) for x in (-7, -9))
    ob_a, ob_b = torch.full((R, H), -1, dtype=I32, device=DEV), torch.full((R, H, obn), -2, dtype=I32, device=DEV)
    inv = O.inv_sqrt_hd(hd)
    ops.qkv_rope_cache(t, s, None, cos, sin, slot, pos, c_a, qq, sq, H, KV, hd)
    ops.attention(qq, sq, c_a, slot, pos, expt, out_a, H, KV, hd, inv, ob_a)
    ops.attention_qkv(t, s, None, cos, sin, slot, pos, c_b, expt, out_b, H, KV, hd, inv, ob_b, obn=obn, keys=1)
    assert torch.equal(out_a, out_b) and torch.equal(ob_b.max(-1)[0], ob_a)
    assert all(torch.equal(x, y) for x, y in zip(c_a, c_b))
