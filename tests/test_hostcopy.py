"""The copy pool of the host-buffer calls (hostcopy.cpp), compiled by itself for the CPU: the order in which a job is published."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nncv_amd", "csrc")

CLANG = shutil.which("clang++") or "/opt/rocm/llvm/bin/clang++"


@pytest.mark.skipif(not os.path.exists(CLANG), reason="no clang")
def test_a_job_is_published_behind_a_release_fence(tmp_path):
    """x86 keeps stores in order whatever the source says, so no run there can show a missing fence; the compiler's own
    notation does: between taking back the old job's number and the first field of the new one."""
    out = str(tmp_path / "hostcopy.ll")
    subprocess.check_call([CLANG, "-O1", "-std=c++17", "-S", "-emit-llvm", "-I" + CSRC, os.path.join(CSRC, "hostcopy.cpp"), "-o", out])
    marks = re.findall(r"store atomic [^\n]* (?:monotonic|release|seq_cst)|fence \w+", open(out).read())
    taken_back = next(i for i, m in enumerate(marks) if re.match(r"store atomic i64 0, .*monotonic", m))
    assert marks[taken_back + 1] == "fence release", marks
    assert re.match(r"store atomic .*monotonic", marks[taken_back + 2]), marks
