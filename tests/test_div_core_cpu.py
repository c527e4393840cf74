"""The column division's host build against Knuth's division (tests/div_core_cpu.cpp), every width, on the CPU."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_column_division(tmp_path):
    exe = tmp_path / "div_core_cpu"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wno-unknown-pragmas", "-DLF_HOST_BUILD", f"-I{ROOT / 'limbforge_amd' / 'csrc'}",
                    str(ROOT / "tests" / "div_core_cpu.cpp"), "-o", str(exe)], check=True)
    p = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert p.returncode == 0, p.stdout
