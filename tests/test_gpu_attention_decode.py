"""Batched decode attention of a KV head with eight query heads, against the two launches exact_qkv_rope_cache +
exact_attention, which the oracle pins."""
import numpy as np
import pytest
import torch

import exact_oracle as O
from exact_amd import ops
from exact_amd.tables import exp_t, host_tables

pytestmark = pytest.mark.gpu
DEV = "cuda"
I16, I32, I64 = torch.int16, torch.int32, torch.int64


def dev(a, dt):
    return torch.tensor(np.ascontiguousarray(a), dtype=dt, device=DEV)


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
    ops.attention_qkv(t, s, None, cos, sin, slot, pos, c_b, expt, out_b, H, KV, hd, inv, obn=4)
    assert torch.equal(out_a, out_b) and all(torch.equal(x, y) for x, y in zip(c_a, c_b))
