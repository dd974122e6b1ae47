"""Rules of the HIP sources that no run on a GPU shows."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pikv_amd", "csrc")


@pytest.mark.parametrize("path", sorted(glob.glob(os.path.join(CSRC, "*.h*"))), ids=os.path.basename)
def test_wave_barriers_are_fenced(path):
    """__builtin_amdgcn_wave_barrier orders no memory: where lanes of a wavefront exchange data through LDS it stands
    between a release and an acquire fence of wavefront scope."""
    with open(path) as f:
        code = re.sub(r"//[^\n]*", "", f.read())
    statements = [re.sub(r"\s+", "", s) for s in re.split(r"[;{}]", code)]
    statements = [s for s in statements if s]
    for i, s in enumerate(statements):
        if s == "__builtin_amdgcn_wave_barrier()":
            assert statements[i - 1] == '__builtin_amdgcn_fence(__ATOMIC_RELEASE,"wavefront")', path
            assert statements[i + 1] == '__builtin_amdgcn_fence(__ATOMIC_ACQUIRE,"wavefront")', path
