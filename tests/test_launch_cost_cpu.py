"""What the chunk chooser takes a launch to cost follows the tiles that the launch has: their width, and those of the inputs' type."""
import numpy as np
import pytest
import torch

from chatlearn_amd import ops
from chatlearn_amd.fused import _launch_cost

V = 151936
BF16, FP32 = torch.bfloat16, torch.float32


def _forward_only(T, H, dtype):
    return _launch_cost([(0, T)], np.zeros(T + 1, dtype=np.int64), H, V, dtype)       # no row carries a gradient


@pytest.mark.parametrize("dtype", [BF16, FP32])
@pytest.mark.parametrize("T", [100, 256, 260, 588, 900, 1100, 3000, 16384])
def test_forward_counts_its_blocks_at_their_width(T, dtype):
    n_tb, n_split, tps, width, time = ops.lmhead_forward_tile_plan(T, 4096, V, dtype)
    assert n_tb == -(-T // width) and 128 <= width <= 256 and n_split * tps >= 594
    assert width / 256 <= time <= 1 and (time == 1) == (width == 256)
    assert _forward_only(T, 4096, dtype) == pytest.approx(-(-(n_tb * n_split) // 256) * tps * 4096 * time)
    if dtype == BF16:
        assert ops.lmhead_forward_launch_plan(T, V) == (n_tb, n_split, tps)
    else:
        assert width == 256


def test_widths_of_the_forward():
    assert [ops.lmhead_forward_tile_plan(T, 4096, V, BF16)[3] for T in (100, 128, 260, 588, 1100, 16384)] == [128, 128, 160, 224, 224, 256]


# (tokens, H, V) measured at every width, us per forward for blocks of (256, 224, 192, 160, 128): a narrower block costs more than its
# share of the products, so wide blocks that nearly fill the CUs, or their rounds, stay
TIMES = [((512, 4096, 32000), (102.0, 135.9, 125.2, 119.3, 109.5)), ((512, 7168, 32000), (173.8, 264.2, 233.4, 211.9, 210.8)),
         ((256, 7168, 50257), (175.6, 259.2, 241.9, 225.7, 223.0)), ((768, 4096, 50257), (250.6, 290.6, 272.2, 253.4, 287.4)),
         ((1400, 4096, 102400), (875.4, 918.5, 912.6, 912.2, 989.5)), ((600, 4096, 151936), (642.9, 585.3, 693.8, 623.0, 674.7)),
         ((300, 4096, 151936), (451.1, 402.1, 374.5, 341.0, 411.4)), ((384, 2048, 129280), (200.1, 183.3, 171.6, 207.4, 196.1)),
         ((512, 1024, 32000), (40.1, 51.6, 46.7, 42.5, 38.2)), ((160, 512, 151936), (55.4, 49.6, 46.0, 42.4, 49.0))]


@pytest.mark.parametrize("size,us", TIMES)
def test_the_width_that_was_fastest_is_taken(size, us):
    width = ops.lmhead_forward_tile_plan(*size, BF16)[3]
    assert us[(256 - width) // 32] <= 1.04 * min(us)


def test_narrow_blocks_are_cheaper_than_wide_ones():
    for few, more in ((128, 256), (260, 512), (588, 768), (1100, 1280)):
        assert _forward_only(few, 4096, BF16) < 0.97 * _forward_only(more, 4096, BF16)
        assert _forward_only(few, 4096, FP32) == pytest.approx(_forward_only(more, 4096, FP32))


@pytest.mark.parametrize("rows,H,dtype", [(128, 4096, BF16), (320, 2048, BF16), (1600, 7168, BF16), (1600, 7168, FP32), (12700, 4096, BF16)])
def test_dhidden_counts_its_row_tiles_at_their_width(rows, H, dtype):
    bulk, ks, width, time = ops.dhidden_tile_plan(rows, H, V, dtype)
    assert width / 256 <= time <= 1 and (time == 1) == (width == 256)
    n_walk, bulk_vt, ks_w = ops.dweight_launch_plan(rows, H, V, dtype)
    n_ht = -(-H // 256)
    dw = ((bulk_vt // n_walk) * rows + -(-((594 - bulk_vt) * n_ht * ks_w) // 256) * (rows / ks_w) if bulk_vt
          else (-(-594 // n_walk) if n_walk else -(-(594 * n_ht) // 256)) * rows)
    want = -(-(bulk * n_ht) // 256) * V + -(-(-(-(rows - 256 * bulk) // width) * n_ht * ks) // 256) * (V / ks) * time
    cum = np.arange(rows + 1)
    assert _launch_cost([(0, rows)], cum, H, V, dtype) - _forward_only(rows, H, dtype) - dw == pytest.approx(want)


@pytest.mark.parametrize("dtype,share", [(BF16, 0.15), (FP32, 0.015)])
def test_another_chunk_reads_dw_again(dtype, share):
    """The traffic costs the same time in either type, counted in products that take fp32 ten times as long."""
    one = _launch_cost([(0, 1024)], None, 4096, V, dtype)
    two = _launch_cost([(0, 1024), (1024, 2048)], None, 4096, V, dtype)
    assert two - 2 * one == pytest.approx(share * 594 * 16 / 256 * 2048)


# (rows, H, V) measured at every height, us of dhidden and the d(logits) pass for row tiles of (256, 192, 128)
HEIGHTS = [((640, 7168, 129280), (1007, 1248, 1312)), ((600, 4096, 32000), (214, 166, 255)), ((1100, 2048, 32000), (154, 198, 165)),
           ((320, 4096, 151936), (455, 405, 546)), ((128, 4096, 151936), (263, 262, 260)), ((384, 2048, 102400), (189, 175, 203)),
           ((190, 1024, 65536), (66, 58, 51)), ((1600, 7168, 102400), (2016, 1898, 2517)), ((830, 1024, 151936), (299, 315, 341))]


@pytest.mark.parametrize("size,us", HEIGHTS)
def test_the_height_that_was_fastest_is_taken(size, us):
    bulk, _, height, _ = ops.dhidden_tile_plan(*size, BF16)
    assert bulk == 0 and us[(256 - height) // 64] <= 1.03 * min(us)
