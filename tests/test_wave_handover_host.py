"""Values that lanes of a wave hand to one another through LDS: written, released, and acquired behind the wave's barrier.  With the acquire missing, the
compiler may read in front of the barrier, which no result shows until it does."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "xfastertransformer_amd", "csrc")
FENCE = r'__builtin_amdgcn_fence\(__ATOMIC_%s, "wavefront"\);'
WHOLE = re.compile(FENCE % "RELEASE" + r"\s*__builtin_amdgcn_wave_barrier\(\);\s*" + FENCE % "ACQUIRE")


def test_every_wave_barrier_releases_and_acquires():
    found = 0
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(CSRC, "*.hip"))):
        with open(path) as f:
            text = f.read()
        barriers, whole = len(re.findall(r"__builtin_amdgcn_wave_barrier\(\)", text)), len(WHOLE.findall(text))
        assert barriers == whole, f"{os.path.basename(path)}: {barriers - whole} of {barriers} wave barriers without both fences"
        found += barriers
    assert found >= 4
