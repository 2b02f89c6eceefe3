"""Properties of the compiled kernels that no result shows, on the CPU."""
import re
import shutil
import subprocess

import pytest

import build as hip_build  # vapoursynth-vnlb_amd/build.py

LLVM = "/opt/rocm/llvm/bin"


def _disassembly(source, tmp_path):
    obj = tmp_path / "kernels.o"
    shutil.copy(hip_build.BUILD / (source.rsplit(".", 1)[0] + ".o"), obj)
    subprocess.run([f"{LLVM}/llvm-objdump", "--offloading", obj.name], cwd=tmp_path, check=True, capture_output=True)
    (code,) = tmp_path.glob("kernels.o.*gfx950")
    return subprocess.run([f"{LLVM}/llvm-objdump", "-d", str(code)], check=True, capture_output=True, text=True).stdout


@pytest.mark.parametrize("source", ["filter.hip", "filter_fast.hip"])
def test_no_flat_memory_instructions(source, tmp_path):
    """Kernels read and write device memory and LDS by instructions of their
    own.  A FLAT access counts as both, so every wait for the LDS waits for
    the loads in flight."""
    text = _disassembly(source, tmp_path)
    assert len(re.findall(r"\bs_endpgm\b", text)) > 0
    assert not re.findall(r"\bflat_(?:load|store|atomic)\w*", text)
