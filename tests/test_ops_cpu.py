"""CPU checks of host-side dispatch rules in exact_amd.ops."""
import os

import pytest

from exact_amd import _lib


@pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH), reason="library not built")
def test_norm_gemv_one_block_per_cu_reads_the_kernel_split():
    """The model fuses the attention norm into the q|k|v GEMV only where exact_gemv_g128_norm_acc runs one 8-wave block
    per CU: rows wider than 1024 whose group-split tasks (ceil(N / 64) row blocks x min(G, ceil(4096 / row blocks)))
    fit one round of 8-wave blocks, or do with the split capped at 8 CUs / row blocks when that is at least 8. The
    split is the library's own query (no launch, no GPU needed with an explicit CU count); a device with fewer CUs
    gets fewer one-round shapes."""
    from exact_amd import ops
    assert ops.norm_gemv_one_block_per_cu(4608, 3584, cus=256)          # 7B q|k|v: 72 x 28 = 2016 tasks, 252 blocks
    assert ops.norm_gemv_one_block_per_cu(4608, 3584, cus=240)          # ... 240 CUs: split capped at 26 (1872 tasks)
    assert ops.norm_gemv_one_block_per_cu(7168, 5120, cus=256)          # 14B q|k|v: 112 x 37 tasks, capped at 112 x 18
    assert not ops.norm_gemv_one_block_per_cu(7168, 5120, cus=96)       # ... a cap of 6 parts: 4-wave blocks
    assert not ops.norm_gemv_one_block_per_cu(37888, 3584, cus=256)     # 7B gate|up: 592 row blocks, cap 3
    assert ops.norm_gemv_one_block_per_cu(300, 6144, cus=256)           # 5 x 48 = 240 tasks
    assert ops.norm_gemv_one_block_per_cu(6144, 2048, cus=256)          # MoE q|k|v: 96 x 16 = 1536 tasks, 192 blocks
    assert not ops.norm_gemv_one_block_per_cu(4608, 1024, cus=256)      # rows of 1024 and less keep 4-wave blocks
    assert not ops.norm_gemv_one_block_per_cu(1152, 896, cus=256)       # (the 0.5B's 896)
    assert ops.norm_gemv_one_block_per_cu(4608, 3584, R=2, cus=256)
    assert not ops.norm_gemv_one_block_per_cu(4608, 3584, R=3, cus=256)      # the launch takes at most 2 rows
    assert _lib.load().exact_gemv_g128_norm_acc_blockwaves(1, 4608, 100, 256) == 0   # K % 128: refused


def test_swiglu_gemm_refuses_wide_scales_and_biases():
    """gemm_swiglu_qrow hands the kernel the low scale plane and no bias, so a linear with either more is refused (before any
    buffer is looked at), and gemm_swiglu_supported says so"""
    import torch
    from exact_amd import ops
    wp, mp = torch.zeros(4 * 2 * 8192, dtype=torch.int8), torch.ones(4 * 2 * 64, dtype=torch.int16)
    for kw in (dict(mh=torch.ones_like(mp)), dict(bias=torch.zeros(256, dtype=torch.int64))):
        lin = ops.PackedLinear(wp, mp, 256, 256, **kw)
        assert not ops.gemm_swiglu_supported(512, lin)
        with pytest.raises(_lib.ExactError, match="wide scales or a bias"):
            ops.gemm_swiglu_qrow(None, lin, torch.zeros(512, dtype=torch.int32), None, None, None, None, None)


# us a layer in a graph, (heads, KV heads, hd), rows, cache length, position: one launch (two where rows x heads pass 256 and the
# cache 256 positions) and split over the keys
ATT_TIMES = [((16, 16, 128), 8, 4096, 384, 27.7, 72.6), ((16, 16, 128), 8, 8192, 512, 34.6, 78.1),
             ((16, 16, 128), 16, 4096, 1024, 74.2, 138.1), ((40, 8, 128), 8, 4096, 256, 30.6, 53.0),
             ((40, 8, 128), 16, 4096, 640, 71.9, 95.3), ((28, 4, 128), 8, 8192, 512, 26.6, 37.7),
             ((28, 4, 128), 1, 8192, 300, 15.7, 17.1), ((14, 2, 64), 8, 8192, 768, 18.2, 22.3),
             ((28, 4, 128), 1, 8192, 640, 25.4, 17.5), ((28, 4, 128), 8, 1024, 512, 26.7, 21.4),
             ((28, 4, 128), 8, 4096, 1024, 47.2, 36.6), ((40, 8, 128), 8, 1024, 320, 34.1, 25.6),
             ((40, 8, 128), 16, 2048, 768, 83.5, 58.8), ((16, 16, 128), 1, 4096, 640, 26.3, 18.5),
             ((16, 16, 128), 8, 1024, 768, 47.0, 39.5), ((14, 2, 64), 1, 4096, 1024, 21.5, 13.9)]


@pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH), reason="library not built")
@pytest.mark.parametrize("heads,R,Smax,pos,one,split", ATT_TIMES)
def test_attention_split_line_against_measured_times(heads, R, Smax, pos, one, split):
    """the faster of the two paths, at times measured well off the line: caches much longer than their positions too"""
    from exact_amd import ops
    assert (pos + 1 >= ops.attention_keys_from(R, *heads, Smax)) == (split < one)


# us a pass of 8 layers and the head launched by the host, (heads, KV heads, hd), MB a layer, rows, position (of 2048)
ATT_EAGER_TIMES = [((14, 2, 64), 15, 1, 1000, 597, 671), ((14, 2, 64), 15, 1, 1500, 599, 664), ((14, 2, 64), 15, 8, 1500, 836, 901),
                   ((16, 16, 128), 52, 1, 768, 1076, 1149), ((16, 16, 128), 52, 8, 768, 1518, 1578),
                   ((28, 4, 128), 233, 1, 200, 737, 786), ((28, 4, 128), 233, 1, 768, 866, 786),
                   ((28, 4, 128), 233, 8, 384, 1034, 1074), ((28, 4, 128), 233, 8, 1000, 1238, 1088)]


@pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH), reason="library not built")
@pytest.mark.parametrize("heads,MB,R,pos,one,split", ATT_EAGER_TIMES)
def test_attention_split_line_of_eager_passes_against_measured_times(heads, MB, R, pos, one, split):
    """a pass that the host's launches bound keeps the one launch a layer"""
    from exact_amd import ops
    assert (pos + 1 >= ops.attention_eager_keys_from(R, *heads, 2048, MB * 10**6)) == (split < one)


# us a call in a graph averaged over the positions of a cache, (heads, KV heads, hd), rows, cache length: one launch and split
ATT_MEANS = [((28, 4, 128), 1, 520, 14.6, 16.4), ((28, 4, 128), 1, 1024, 22.3, 17.8), ((28, 4, 128), 8, 520, 14.4, 18.6),
             ((28, 4, 128), 8, 4096, 88.2, 40.0), ((14, 2, 64), 8, 1024, 13.8, 14.9), ((14, 2, 64), 8, 4096, 48.1, 22.2),
             ((16, 16, 128), 8, 1024, 33.5, 35.9), ((16, 16, 128), 16, 4096, 138.4, 169.3), ((16, 16, 128), 2, 4096, 114.7, 29.6),
             ((40, 8, 128), 8, 1024, 58.7, 26.2)]


@pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH), reason="library not built")
@pytest.mark.parametrize("heads,R,Smax,one,split", ATT_MEANS)
def test_attention_without_known_positions_takes_the_faster_path_on_average(heads, R, Smax, one, split):
    """attention_qkv without keys: rows anywhere in the cache"""
    from exact_amd import ops
    assert (ops.known_keys(None, Smax) >= ops.attention_keys_from(R, *heads, Smax)) == (split < one)
    assert ops.known_keys(Smax + 9, Smax) == Smax and ops.known_keys(7, Smax) == 7
