"""Atomics of the factorization kernels cover every thread that shares their memory.  The accumulators in LDS take the
terms of several wavefronts of a workgroup between two barriers; an atomic of wavefront scope there is a data race by
the memory model, whatever instruction it becomes, and no run shows it.  The compiler's own account of each atomic's
scope is read from the device code of one width (hipcc cross-compiles without a GPU)."""
import re
import shutil
import subprocess

import pytest

from limbforge_amd import build



def test_no_atomic_is_narrower_than_a_workgroup(tmp_path):
    if not shutil.which(build.HIPCC):
        pytest.skip("hipcc is not installed")
    out = tmp_path / "factor.ll"
    subprocess.run([build.HIPCC, f"--offload-arch={build.ARCH}", "--cuda-device-only", "-S", "-emit-llvm", "-O1", "-Xclang", "-disable-llvm-passes",
                    "-std=c++17", "-DLF_WORDS=2", f"-I{build.CSRC}", f"-I{build.INCLUDE}", str(build.CSRC / "factor_w.hip"), "-o", str(out)],
                   check=True, stderr=subprocess.DEVNULL)
    atomics = [line.strip() for line in out.read_text().splitlines() if " atomicrmw " in line or " cmpxchg " in line]
    assert any("atomicrmw add" in a and " i64 " in a for a in atomics), "the 64-bit adds of the digit columns"
    narrow = [a for a in atomics if re.search(r'syncscope\("(wavefront|singlethread)', a)]
    assert not narrow, narrow
