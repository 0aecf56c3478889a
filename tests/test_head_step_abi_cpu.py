"""clgrpo_head_step refuses what would make one of its stages write or read outside a buffer before any stage is enqueued."""
import ctypes as C

import pytest

from chatlearn_amd import _lib

EINVAL, ESHAPE, ENULL = -1, -3, -4


def _args(**change):
    a = _lib.HeadStepArgs()
    for name in ("hidden", "weight", "labels", "old_logprob", "ref_logprob", "advantages", "cu_seqlens", "loss_mask", "row_order",
                 "logprob", "entropy", "lse", "g_logprob", "loss", "kl", "sums", "flags", "dhidden", "dweight", "workspace",
                 "saved_logits", "kept_dzt", "kept_hidt"):
        setattr(a, name, 1 << 20)                     # never read: every call below is refused
    a.T, a.n_live, a.H, a.V, a.B, a.dtype, a.stages, a.inv_temperature = 700, 513, 128, 1000, 2, _lib.BF16, 7, 1.0
    a.workspace_bytes, a.ld_saved, a.saved_rows, a.kept_ld, a.kept_k = 1 << 40, 1024, 768, 640, 64
    for name, value in change.items():
        setattr(a, name, value)
    return a


@pytest.mark.parametrize("change,code,text", [
    ({"saved_rows": 767}, ESHAPE, "saved_rows"),
    ({"saved_rows": 512, "stages": 1}, ESHAPE, "saved_rows"),
    ({"saved_logits": None, "kept_dzt": None}, ESHAPE, "need kept logits"),
    ({"saved_logits": None, "row_order": None, "n_live": 700}, ESHAPE, "need kept logits"),
    ({"kept_k": 128}, ESHAPE, "do not fit"),
    ({"kept_k": 32}, ESHAPE, "do not fit"),
    ({"kept_k": -64}, ESHAPE, "do not fit"),
    ({"kept_hidt": None}, ENULL, "kept_hidt"),
    ({"kept_dzt": None, "dhidden": None, "dweight": None}, ENULL, "dhidden"),
    ({"forward_live_only": 1, "entropy": None}, ENULL, "entropy"),
    ({"forward_live_only": 1, "n_live": 0, "lse": None}, ENULL, "lse"),
    ({"sums": None, "chunk": 1}, ENULL, "sums"),
    ({"flags": None, "chunk": 1}, ENULL, "flags"),
    ({"cu_seqlens": None}, ENULL, "cu_seqlens"),
    ({"chunk": -1}, EINVAL, "chunk"),
])
def test_refused_before_any_launch(lib, change, code, text):
    a = _args(**change)
    assert lib.clgrpo_head_step(C.byref(a), None) == code
    assert text in lib.clgrpo_last_error_string().decode()
