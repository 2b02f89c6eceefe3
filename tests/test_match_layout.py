"""LDS layout of the exhaustive matcher, on the CPU: every shape that it is
launched for fits its allocation and has a kernel (match_layout_check.cpp)."""
import subprocess
from pathlib import Path

TESTS = Path(__file__).resolve().parent
CSRC = TESTS.parent / "vapoursynth-vnlb_amd" / "csrc"


def test_every_shape_fits_its_allocation(tmp_path):
    program = tmp_path / "match_layout_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{CSRC}",
                    str(TESTS / "match_layout_check.cpp"), "-o", str(program)], check=True)
    run = subprocess.run([str(program)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
    # Unguided narrow rows: 2x2 patches only, and some of them.
    assert [line.split(":")[0] for line in run.stdout.splitlines() if line.startswith("unguided")] == ["unguided 2"]
