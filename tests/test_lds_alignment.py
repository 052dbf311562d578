"""LDS arrays that kernels read in vectors of 16 bytes say so: a char or byte array's own
alignment is 1, and where the compiler then puts it is its choice."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "intent-attention-kernel_amd", "csrc")


def test_byte_arrays_in_the_lds_are_aligned():
    seen = 0
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(CSRC, "*.hip"))):
        for line in open(path):
            if re.search(r"__shared__[^;(]*(\(\([^)]*\)\))?[^;]*\b(char|uint8_t|unsigned char)\s+\w+\s*\[", line):
                seen += 1
                assert "aligned(16)" in line or "alignas(16)" in line, (os.path.basename(path), line.strip())
    assert seen >= 2
