"""The many-row product's first x tile, in the assembly of the kernels as they are built: the copies
that fill it and the other first requests may be issued in any order, so nothing less than a wait for
all of them may stand between the last one and the first barrier."""

from __future__ import annotations

import os
import re
import subprocess

import pytest

SOURCE = """
#include "dspark_qmm_wide.h"
template __global__ void dspark::wide::wide_kernel<8, %(mt)d, %(nt)d>(dspark::wide::Args);
template __global__ void dspark::wide::wide_kernel<4, %(mt)d, %(nt)d>(dspark::wide::Args);
"""


@pytest.mark.parametrize("mt,nt", [(2, 4), (4, 2), (8, 4)])   # three groups ahead, and one
def test_first_barrier_waits_for_every_copy(tmp_path, mt, nt):
    import build

    src, out = tmp_path / "k.hip", tmp_path / "k.s"
    src.write_text(SOURCE % {"mt": mt, "nt": nt})
    subprocess.run([build.hipcc(), *build.HIPCC_FLAGS, "--cuda-device-only", "-S", str(src), "-o", str(out)], check=True,
                   capture_output=True)
    bodies = re.split(r"^_ZN6dspark4wide11wide_kernel\w+:", out.read_text(), flags=re.M)[1:]
    assert len(bodies) == 2
    ahead, copies = (1 if mt * nt >= 24 else 3), (mt + 1) // 2
    for body in bodies:
        events = re.findall(r"global_load_lds_|s_barrier|;;#ASMSTART\s+s_waitcnt vmcnt\(0\)\s", body)
        first = events[:ahead * copies + 1]
        assert first[:-1] == ["global_load_lds_"] * (ahead * copies) and "vmcnt(0)" in first[-1], events[:20]
