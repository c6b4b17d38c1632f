"""Shared arrays that kernels address four or more elements at a time say so in their declaration: dynamic shared memory
begins where a kernel's static shared variables end, at a multiple of what its declaration asks for."""
import os
import re

from conftest import ROOT

CSRC = os.path.join(ROOT, "da_transformer_amd", "csrc")


def test_dynamic_shared_memory_of_wide_accesses_is_aligned():
    """The chunked sweeps and the fused softmax kernels (arrays named lds_raw) store vectors of sixteen bytes and copy
    sixteen bytes a lane into them; float[] alone promises four."""
    seen = 0
    for name in sorted(os.listdir(CSRC)):
        text = open(os.path.join(CSRC, name)).read()
        for decl in re.findall(r"extern\s+__shared__[^;]*\blds_raw\[\]", text):
            assert "__align__(16)" in decl, f"{name}: {decl}"
            seen += 1
        # vectors reach dynamic shared memory through that name only
        assert not re.findall(r"x[248] \*>\(lds_(?!raw\b)\w+", text), name
    assert seen == 3
