"""The dW pass of shared K16 records (csrc/gl_record.hip) transposes X through LDS between the lanes of a
wave.  In the compiler's IR every change from writes to reads of that buffer, and back, has a
wavefront fence between: without one the accesses of different lanes are unordered and may be moved
past each other."""
import re
import subprocess
from pathlib import Path

import pytest

from granulelayer_amd import build


def fence_gaps(ir):
    """(kernel, line) of LDS accesses of rec_bwd_w_kernel that follow one of the other kind in their basic block
    with no wavefront fence between; and the number of LDS stores seen."""
    gaps, stores, kernel, last = [], 0, None, None
    for n, line in enumerate(ir.splitlines()):
        m = re.match(r"define .*@(\S+?)\(", line)
        if m:
            kernel = m.group(1) if "rec_bwd_w_kernel" in m.group(1) else None
        if kernel is None:
            continue
        if re.match(r"\d+:|[\w.]+:", line) or 'fence syncscope("wavefront")' in line:  # a new block, a fence
            last = None
        kind = None
        if "addrspace(3)" in line:
            kind = "store" if re.match(r"\s+store ", line) else "load" if re.search(r"= load ", line) else None
        if kind:
            stores += kind == "store"
            if last and last != kind:
                gaps.append((kernel, n))
            last = kind
    return gaps, stores


def test_lds_transpose_is_fenced(tmp_path):
    if not Path(build.HIPCC).exists():
        pytest.skip("no hipcc")
    out = tmp_path / "gl_record.ll"
    subprocess.run([build.HIPCC, *build.FLAGS, "--cuda-device-only", "-S", "-emit-llvm", str(build.CSRC / "gl_record.hip"),
                    "-o", str(out)], check=True, capture_output=True)
    gaps, stores = fence_gaps(out.read_text())
    assert stores >= 2 * 8 * 4  # two activations, 8 records, 4 row stores each: the kernel was found
    assert gaps == []
