"""Device integer sampler and receipts against the oracle (sample_int / generate / verify, exact_llm.py:243-276)."""
import numpy as np
import pytest
import torch

import exact_oracle as O
import helpers
from exact_amd import _lib, ops, synth
from exact_amd.model import DeviceWeights, TModel, generate, verify
from exact_amd.tables import exp_t

pytestmark = pytest.mark.gpu
DEV = "cuda"
I32, I64 = torch.int32, torch.int64


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


@pytest.mark.parametrize("R,V,temp", [(3, 152064, 1.0), (2, 1000, 0.7), (4, 7, 2.0), (1, 1, 1.0), (2, 5000, 0.05)])
def test_sample_matches_oracle(R, V, temp):
    rng = np.random.default_rng(V + R)
    lg = rng.integers(-(8 << 16), 8 << 16, (R, V))
    if V > 10:
        lg[0, :] = 12345                                # uniform row
        lg[1, V // 3] = 40 << 16                        # one dominant logit: most p are 0
    seed = 0x1234_5678_9ABC_DEF0
    steps = rng.integers(0, 1000, R).astype(np.int32)
    tnum = ops.temp_num(temp)
    ids, pd = torch.zeros(R, dtype=I32, device=DEV), torch.zeros((R, V), dtype=I64, device=DEV)
    ops.sample(torch.tensor(lg, device=DEV), seed, torch.tensor(steps, device=DEV), tnum,
               torch.tensor(exp_t(), dtype=I32, device=DEV), ids, pd)
    got, gp = host(ids), host(pd)
    for r in range(R):
        tok, p = O.sample_int(lg[r], seed, int(steps[r]), tnum)
        assert np.array_equal(gp[r], p), r
        assert got[r] == tok, (r, got[r], tok)


def test_generate_receipt_matches_oracle_and_verifies():
    cfg = synth.CONFIGS["tiny"]
    om = helpers.oracle_model(cfg, 5, T=64)
    tm = TModel(DeviceWeights.synthetic(cfg, 5, DEV), Smax=64)
    prompt = helpers.prompt(8, 7, cfg.V)
    rec, greedy = generate(tm, prompt, 12, seed=99, temp=0.8)
    orec, ogreedy, _ = O.generate(om, prompt, 12, seed=99, temp=0.8)
    assert rec["tokens"] == orec["tokens"] and rec["chain"] == orec["chain"] and greedy == ogreedy
    assert any(a != b for a, b in zip(rec["tokens"], greedy))       # it really samples
    assert verify(tm, rec) == (True, None)
    bad = dict(rec, tokens=list(rec["tokens"]))
    bad["tokens"][5] = (bad["tokens"][5] + 1) % cfg.V
    assert verify(tm, bad) == (False, 5)
    # the host checks each step one step behind the device: the first and last positions and the chain itself
    for pos in (0, 11):
        bad = dict(rec, tokens=list(rec["tokens"]))
        bad["tokens"][pos] = (bad["tokens"][pos] + 1) % cfg.V
        assert verify(tm, bad) == (False, pos)
    assert verify(tm, dict(rec, chain="0" * 16)) == (False, "chain")


@pytest.mark.parametrize("n", [1, 2])
def test_short_generations_match_oracle(n):
    """one token (no decode step) and two (one captured step) through the pipelined receipt path"""
    cfg = synth.CONFIGS["tiny"]
    om = helpers.oracle_model(cfg, 6, T=32)
    tm = TModel(DeviceWeights.synthetic(cfg, 6, DEV), Smax=32)
    prompt = helpers.prompt(3, 5, cfg.V)
    rec, greedy = generate(tm, prompt, n, seed=7, temp=0.9)
    orec, ogreedy, _ = O.generate(om, prompt, n, seed=7, temp=0.9)
    assert rec["tokens"] == orec["tokens"] and rec["chain"] == orec["chain"] and greedy == ogreedy
    assert verify(tm, rec) == (True, None)


@pytest.mark.parametrize("R,V", [(1, 1), (3, 63), (2, 1023), (2, 1024), (3, 1025), (1, 6143), (2, 6144), (9, 6145), (1, 152064)])
@pytest.mark.parametrize("temp", [0.05, 1.0])
def test_split_rows_match_oracle(R, V, temp):
    """exact_sample_split at the edges of its chunks, and where ops.sample changes to it; ids over the steps' own array"""
    rng = np.random.default_rng(V * 7 + R)
    lg = rng.integers(-(6 << 16), 6 << 16, (R, V))
    lg[0, -1] = 9 << 16                                 # the last logit of a row is likely drawn
    lgd, seed, tnum = torch.tensor(lg, device=DEV), 77, ops.temp_num(temp)
    ids = torch.arange(R, dtype=I32, device=DEV) * 5 + 2
    pd = torch.zeros((R, V), dtype=I64, device=DEV)
    expt = torch.tensor(exp_t(), dtype=I32, device=DEV)
    nb = _lib.load().exact_sample_workspace(R, V)
    work = torch.full((nb,), 0x55, dtype=torch.int8, device=DEV)
    p = lambda t: t.data_ptr()
    _lib.call("exact_sample_split", p(lgd), R, V, seed, p(ids), tnum, p(expt), p(ids), p(pd), p(work), nb,
              torch.cuda.current_stream().cuda_stream)
    other = torch.zeros(R, dtype=I32, device=DEV)
    ops.sample(lgd, seed, torch.arange(R, dtype=I32, device=DEV) * 5 + 2, tnum, expt, other)
    got, gp = host(ids), host(pd)
    for r in range(R):
        tok, pr = O.sample_int(lg[r], seed, 5 * r + 2, tnum)
        assert np.array_equal(gp[r], pr), r
        assert got[r] == tok == int(other[r]), (r, got[r], tok)


def test_split_rows_of_a_table_with_negative_entries_match_the_one_block_kernel():
    """prefix sums that decrease: both entry points count the sums up to the target alike"""
    V, R, seed, tnum = 5000, 3, 11, ops.temp_num(1.0)
    rng = np.random.default_rng(4)
    tab = np.array(exp_t(), dtype=np.int64)
    tab[700:1500] = -(tab[700:1500] // 3)
    expt = torch.tensor(tab, dtype=I32, device=DEV)
    lg = torch.tensor(rng.integers(-(3 << 16), 3 << 16, (R, V)), device=DEV)
    step = torch.arange(R, dtype=I32, device=DEV)
    out = []
    for lim in (V + 1, 1):
        ids, pd = torch.zeros(R, dtype=I32, device=DEV), torch.zeros((R, V), dtype=I64, device=DEV)
        old, ops.SAMPLE_SPLIT_FROM = ops.SAMPLE_SPLIT_FROM, lim
        try:
            ops.sample(lg, seed, step, tnum, expt, ids, pd)
        finally:
            ops.SAMPLE_SPLIT_FROM = old
        out.append((host(ids), host(pd)))
    assert (out[0][1] < 0).any()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("table", ["zeros", "zero sum"])
def test_split_rows_of_no_exponential_match_the_one_block_kernel(table):
    """a softmax denominator of 0, from a table of zeros and from entries that cancel: every p is 0 and so is every prefix
    sum, so that the token is V"""
    V, R, seed, tnum = 5000, 3, 11, ops.temp_num(1.0)
    tab = np.zeros_like(np.array(exp_t(), dtype=np.int64))
    lg = torch.zeros((R, V), dtype=I64, device=DEV)
    if table == "zero sum":   # 2000 logits each of 1000 and of -1000, 1 below the maximum, and 1000 of 0, 2 below it
        tab[0], tab[256:258] = 1000, -1000
        lg[:, ::2] = -(1 << 16)
        lg[:, ::5] = -(2 << 16)
    expt = torch.tensor(tab, dtype=I32, device=DEV)
    step = torch.arange(R, dtype=I32, device=DEV)
    for lim in (V + 1, 1):
        ids, pd = torch.zeros(R, dtype=I32, device=DEV), torch.full((R, V), 7, dtype=I64, device=DEV)
        old, ops.SAMPLE_SPLIT_FROM = ops.SAMPLE_SPLIT_FROM, lim
        try:
            ops.sample(lg, seed, step, tnum, expt, ids, pd)
        finally:
            ops.SAMPLE_SPLIT_FROM = old
        assert (host(ids) == V).all() and not host(pd).any(), lim


@pytest.mark.parametrize("R,rows", [(7, 3), (6, 2), (5, 1), (4, 9)])
@pytest.mark.parametrize("with_p", [False, True])
def test_split_rows_in_groups_match_one_block_a_row(R, rows, with_p, monkeypatch):
    """calls whose workspace is bounded to so many rows (a last group of fewer among them), ids over the steps' own array"""
    V, seed, tnum = 9000, 21, ops.temp_num(0.8)
    rng = np.random.default_rng(R)
    lg = torch.tensor(rng.integers(-(4 << 16), 4 << 16, (R, V)), device=DEV)
    expt = torch.tensor(exp_t(), dtype=I32, device=DEV)
    monkeypatch.setattr(ops, "SAMPLE_WORK_BYTES", _lib.load().exact_sample_workspace(rows, V) + 5)
    got = []
    for lim in (V + 1, V):
        monkeypatch.setattr(ops, "SAMPLE_SPLIT_FROM", lim)
        ids = torch.arange(R, dtype=I32, device=DEV) * 3 + 1
        pd = torch.full((R, V), -1, dtype=I64, device=DEV) if with_p else None
        torch.cuda.synchronize()
        ops.sample(lg, seed, ids, tnum, expt, ids, pd)
        got.append((host(ids), host(pd) if with_p else None))
    assert np.array_equal(got[0][0], got[1][0]) and (not with_p or np.array_equal(got[0][1], got[1][1]))


def test_many_split_rows_keep_the_workspace_bounded():
    """the memory that a call takes beside its logits"""
    R, V = 600, 152064
    lg = torch.zeros((R, V), dtype=I64, device=DEV)
    step, ids = torch.arange(R, dtype=I32, device=DEV), torch.zeros(R, dtype=I32, device=DEV)
    expt = torch.tensor(exp_t(), dtype=I32, device=DEV)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    ops.sample(lg, 3, step, ops.temp_num(1.0), expt, ids)
    assert torch.cuda.max_memory_allocated() - before <= ops.SAMPLE_WORK_BYTES + (2 << 20)
    got = host(ids)
    assert ((0 <= got) & (got < V)).all() and len(set(got.tolist())) > R // 2   # equal logits: tokens over the whole row


@pytest.mark.parametrize("V", [100, 9000, 20000])
def test_no_rows_are_refused(V):
    z = lambda *sh, dt=I32: torch.zeros(sh, dtype=dt, device=DEV)
    with pytest.raises(ops.ExactError, match="bad argument"):
        ops.sample(z(0, V, dt=I64), 1, z(0), ops.temp_num(1.0), torch.tensor(exp_t(), dtype=I32, device=DEV), z(0))
