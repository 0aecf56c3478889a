"""Scratch sizes against the launches that have to fit them (host arithmetic only)."""
import random

import pytest

from chatlearn_amd import _lib


def test_forward_scratch_covers_every_shorter_launch(lib):
    """Fewer token blocks get more vocabulary splits: scratch memory that a caller sized for T tokens has to hold the
    records of any launch of up to T tokens (whole and nearly whole blocks are where splits x tokens peaks)."""
    plan = (_lib.i32 * 3)()
    for V in (700, 33000, 129280, 151936):
        sizes = sorted({t for b in range(1, 72) for t in (256 * b - 255, 256 * b - 1, 256 * b)})
        have = [lib.clgrpo_lmhead_fwd_workspace_bytes(t, 4096, V, _lib.BF16) for t in sizes]
        assert have == sorted(have)
        for t, bytes_ in zip(sizes, have):
            for cus in (64, 256, 304):
                assert lib.clgrpo_lmhead_fwd_launch_plan(t, V, cus, plan) == 0
                assert plan[1] * t * 16 <= bytes_


@pytest.mark.parametrize("flags", range(8))
def test_step_scratch_covers_both_forwards(lib, flags):
    """A step whose forward leaves masked rows out runs it on n_live rows in the scratch planned for T."""
    r = random.Random(flags)
    up = lambda x: (x + 255) // 256 * 256
    for _ in range(1500):
        T, H, V = r.randint(1, 16384), r.choice([1024, 2048, 4096, 7168]), r.choice([33000, 70000, 129280, 151936])
        live = max(1, int(T * r.uniform(0.5, 1.0)))
        total = lib.clgrpo_head_step_workspace_bytes(T, live, H, V, 4, _lib.BF16, flags, 8 << 30)
        share = total - up(lib.clgrpo_policy_loss_workspace_bytes(T, 4)) - up(4 * T)
        for n in (T, live):
            assert share >= lib.clgrpo_lmhead_fwd_workspace_bytes(n, H, V, _lib.BF16), (T, live, H, V)
