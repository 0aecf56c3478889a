"""The backward's scratch memory is the sum of what its launches read and write, and nothing for a W^T that is never formed."""
import pytest
import torch

from chatlearn_amd import _lib, ops

GIB = 1 << 30


def _up(x, to):
    return (x + to - 1) // to * to


def _expected(rows, H, V, dtype, keeps_logits, keeps_operands):
    es = 2 if dtype == torch.bfloat16 else 4
    ldv, ldt = _up(V, 64), _up(rows, 64)
    bulk, ks = ops.dhidden_launch_plan(rows, H, V, dtype)
    partials = [ks * (rows - 256 * bulk) * H * 4 if ks > 1 else 0]
    if not keeps_operands:
        n_walk, bulk, ks = ops.dweight_launch_plan(rows, H, V, dtype)
        partials.append(ks * (V - 256 * bulk) * H * 4 if bulk and ks > 1 else 0)
    return (0 if keeps_operands else _up(_up(H, 256) * ldt * es, 256)) + (0 if keeps_logits else _up(ldt * ldv * es, 256)) + _up(max(partials), 256)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,V", [(1024, 32003), (4096, 151936), (7168, 129280)])
@pytest.mark.parametrize("rows", [1, 256, 384, 385, 400, 1458, 12126, 25000])
def test_regions_add_up(lib, rows, H, V, dtype):
    dt = _lib.BF16 if dtype == torch.bfloat16 else _lib.F32
    for flags in range(8):
        have = lib.clgrpo_lmhead_bwd_workspace_bytes(rows, H, V, dt, 0, flags)
        assert have == _expected(rows, H, V, dtype, flags & 1, flags & 4), flags


def test_more_rows_are_recomputed_in_one_chunk(lib):
    """25000 rows of H = 4096 over 151936 entries: 7.3 GB, within the 8 GiB that a backward takes by default."""
    need = lib.clgrpo_lmhead_bwd_workspace_bytes(25000, 4096, 151936, _lib.BF16, 0, 0)
    assert need < ops.DEFAULT_BWD_WORKSPACE_BYTES
    step = lib.clgrpo_head_step_workspace_bytes(25000, 25000, 4096, 151936, 4, _lib.BF16, 0, ops.DEFAULT_BWD_WORKSPACE_BYTES)
    assert need <= step < need + 16 * 25000 * 64 + (1 << 20)
