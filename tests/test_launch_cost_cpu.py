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


def _factor(width):
    """A tile's time against one of 256 rows: its share of the products, 2 % more per 32 rows less."""
    return width / 256 * (1 + 0.02 * (256 - width) / 32)


@pytest.mark.parametrize("dtype", [BF16, FP32])
@pytest.mark.parametrize("T", [100, 256, 260, 588, 900, 1100, 3000, 16384])
def test_forward_counts_its_blocks_at_their_width(T, dtype):
    n_tb, n_split, tps, width = ops.lmhead_forward_tile_plan(T, V, dtype)
    assert n_tb == -(-T // width) and 128 <= width <= 256 and n_split * tps >= 594
    assert _forward_only(T, 4096, dtype) == pytest.approx(-(-(n_tb * n_split) // 256) * tps * 4096 * _factor(width))
    if dtype == BF16:
        assert ops.lmhead_forward_launch_plan(T, V) == (n_tb, n_split, tps)
    else:
        assert width == 256


def test_widths_of_the_forward():
    assert [ops.lmhead_forward_tile_plan(T, V, BF16)[3] for T in (100, 128, 260, 588, 1100, 16384)] == [128, 128, 160, 224, 224, 256]


def test_narrow_blocks_are_cheaper_than_wide_ones():
    for few, more in ((128, 256), (260, 512), (588, 768), (1100, 1280)):
        assert _forward_only(few, 4096, BF16) < 0.97 * _forward_only(more, 4096, BF16)
        assert _forward_only(few, 4096, FP32) == pytest.approx(_forward_only(more, 4096, FP32))


@pytest.mark.parametrize("rows,H,dtype", [(128, 4096, BF16), (320, 2048, BF16), (1600, 7168, BF16), (1600, 7168, FP32), (12700, 4096, BF16)])
def test_dhidden_counts_its_row_tiles_at_their_width(rows, H, dtype):
    bulk, ks, width = ops.dhidden_tile_plan(rows, H, V, dtype)
    n_walk, bulk_vt, ks_w = ops.dweight_launch_plan(rows, H, V, dtype)
    n_ht = -(-H // 256)
    dw = ((bulk_vt // n_walk) * rows + -(-((594 - bulk_vt) * n_ht * ks_w) // 256) * (rows / ks_w) if bulk_vt
          else (-(-594 // n_walk) if n_walk else -(-(594 * n_ht) // 256)) * rows)
    want = -(-(bulk * n_ht) // 256) * V + -(-(-(-(rows - 256 * bulk) // width) * n_ht * ks) // 256) * (V / ks) * _factor(width)
    cum = np.arange(rows + 1)
    assert _launch_cost([(0, rows)], cum, H, V, dtype) - _forward_only(rows, H, dtype) - dw == pytest.approx(want)


@pytest.mark.parametrize("dtype,share", [(BF16, 0.15), (FP32, 0.015)])
def test_another_chunk_reads_dw_again(dtype, share):
    """The traffic costs the same time in either type, counted in products that take fp32 ten times as long."""
    one = _launch_cost([(0, 1024)], None, 4096, V, dtype)
    two = _launch_cost([(0, 1024), (1024, 2048)], None, 4096, V, dtype)
    assert two - 2 * one == pytest.approx(share * 594 * 16 / 256 * 2048)
