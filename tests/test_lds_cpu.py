"""Dynamic LDS, into which the kernels lay values of 8 and 16 bytes, starts behind whatever static LDS a kernel has: its declaration has to
say how it is aligned."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "library_amd", "csrc")


def test_dynamic_lds_is_aligned():
    found = []
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h*"))):
        with open(path) as f:
            found += [(os.path.basename(path), d.strip()) for d in re.findall(r"extern\s+__shared__[^;]*;", f.read())]
    assert found
    for name, declaration in found:
        align = re.search(r"(?:__align__|alignas)\((\d+)\)", declaration)
        assert align and int(align.group(1)) >= 16, f"{name}: {declaration}"
