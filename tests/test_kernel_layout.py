"""Host checks of what the kernels and their launches share, on the CPU: the
exhaustive matcher's LDS layout (every shape that it is launched for fits its
allocation and has a kernel) and the order of eigenpairs."""
import re
import subprocess
from pathlib import Path

TESTS = Path(__file__).resolve().parent
CSRC = TESTS.parent / "vapoursynth-vnlb_amd" / "csrc"


def _run(name, tmp_path):
    program = tmp_path / name
    subprocess.run(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{CSRC}",
                    str(TESTS / f"{name}.cpp"), "-o", str(program)], check=True)
    run = subprocess.run([str(program)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
    return run.stdout


def test_every_match_shape_fits_its_allocation(tmp_path):
    out = _run("match_layout_check", tmp_path)
    # Unguided narrow rows: 2x2 patches only, and some of them.
    assert [line.split(":")[0] for line in out.splitlines() if line.startswith("unguided")] == ["unguided 2"]


def test_eigenpair_places_are_a_permutation(tmp_path):
    _run("eigen_order_check", tmp_path)


def test_dynamic_lds_is_aligned_for_vector_reads(tmp_path):
    """The dynamic LDS array of every kernel in the file starts at a multiple
    of 16 bytes by its type, not by what the static arrays before it add up to
    (the learned matcher's s_dyn is read a float at a time)."""
    import build as hip_build  # vapoursynth-vnlb_amd/build.py

    ir = tmp_path / "match.ll"
    subprocess.run([hip_build.hipcc(), *hip_build.COMMON_FLAGS, "--cuda-device-only", "-emit-llvm", "-S", "-Xclang",
                    "-disable-llvm-passes", str(CSRC / "match.hip"), "-o", str(ir)], check=True, capture_output=True)
    arrays = re.findall(r"^@(\S+) = external addrspace\(3\) global .*, align (\d+)$", ir.read_text(), re.M)
    aligned = {name: int(align) for name, align in arrays if "s_dyn" not in name}
    assert len(aligned) == 1 and min(aligned.values()) >= 16, arrays
