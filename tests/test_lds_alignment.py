"""Dynamic LDS starts behind a kernel's static LDS, on the boundary that its declaration asks for: a buffer that is read in 16-byte
vectors has to ask for 16 bytes."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fgms_amd", "csrc")
SOURCES = sorted(os.path.basename(f) for f in glob.glob(os.path.join(CSRC, "*.h*")) if "extern __shared__" in open(f).read())


@pytest.mark.parametrize("source", SOURCES)
def test_declared_for_sixteen_bytes(source):
    declared = re.findall(r"extern __shared__ ([^;]*);", open(os.path.join(CSRC, source)).read())
    assert declared
    for d in declared:
        assert d.startswith("int4v ") or "__align__(16)" in d, d
