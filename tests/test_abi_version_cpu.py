"""The major part of the C ABI's version stands for the layouts that a caller may have built in: args structs and buffers."""
import ctypes as C
import os
import re

from chatlearn_amd import _lib

HEADER = open(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "clgrpo.h")).read()

# major version -> element (row, k) of saved_logits, as the header states it (E = 128 / sizeof(dtype))
SAVED_LOGITS = {
    3: "(((row / 256) * (ld_saved / E) + k / E) * 256 + row % 256) * E + k % E",
    4: "(((row / E) * (ld_saved / E) + k / E) * E + row % E) * E + k % E",
}
# and the sizes of the structs that hold or describe such buffers
SIZES = {4: {"LmheadFwdArgs": 136, "LmheadBwdArgs": 168, "HeadStepArgs": 392, "DweightArgs": 88}}


def test_a_changed_layout_has_a_new_major_version(lib):
    major = int(re.search(r"#define CLGRPO_VERSION (\d+)", HEADER).group(1)) // 100
    fwd = HEADER[HEADER.index("void* saved_logits;"):HEADER.index("} clgrpo_lmhead_fwd_args;")]
    formula = re.search(r"element \(row, k\) at\s+(.*?),\s+E = 128", fwd, flags=re.S).group(1)
    assert " ".join(formula.split()) == SAVED_LOGITS[major]
    assert {name: C.sizeof(getattr(_lib, name)) for name in SIZES[major]} == SIZES[major]
    assert lib.clgrpo_version() // 100 == major
