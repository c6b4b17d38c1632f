"""Shared arrays that kernels address four or more elements at a time say so in their declaration: dynamic shared memory
begins where a kernel's static shared variables end, at a multiple of what its declaration asks for."""
import os
import re

from conftest import ROOT

CSRC = os.path.join(ROOT, "da_transformer_amd", "csrc")


def test_dynamic_shared_memory_of_wide_accesses_is_aligned():
    """The chunked sweeps and the fused softmax kernels (arrays named lds_raw) store vectors of sixteen bytes and copy
    sixteen bytes a lane into them, the walk back stores vectors into its stages (WalkStage, at the beginning of lds_a and lds_walk);
    float[] alone promises four.  Declarations of one name are one symbol, so all of them have to say it."""
    seen = {"lds_raw": 0, "lds_a": 0, "lds_walk": 0}
    for name in sorted(os.listdir(CSRC)):
        text = open(os.path.join(CSRC, name)).read()
        for decl, array in re.findall(r"(extern\s+__shared__[^;]*?\b(\w+)\[\])", text):
            if array in seen:
                assert "__align__(16)" in decl, f"{name}: {decl}"
                seen[array] += 1
        # vectors and stages reach dynamic shared memory through those names only
        for array in re.findall(r"(?:x[248]|WalkStage) \*>\((?:&)?(lds_\w+)", text):
            assert array in seen, f"{name}: {array}"
    assert seen == {"lds_raw": 3, "lds_a": 2, "lds_walk": 1}
