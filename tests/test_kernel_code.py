"""What the compiler made of kernels that rest on it, read from the library built here: registers in the code objects' metadata and
the order of instructions in their assembly.  No GPU needed."""
import os
import re
import shutil
import subprocess

import pytest

LLVM = "/opt/rocm/llvm/bin"


def tool(name):
    return shutil.which(name) or os.path.join(LLVM, name)


@pytest.fixture(scope="module")
def code_objects(lva, tmp_path_factory):
    """the gfx950 code objects of the HIP library"""
    lib = os.path.join(os.path.dirname(lva.__file__), "libllava_hip.so")
    if not os.path.exists(lib) or not os.path.exists(tool("llvm-objdump")) or not os.path.exists(tool("llvm-readelf")):
        pytest.skip("needs the built library and llvm-objdump, llvm-readelf")
    d = tmp_path_factory.mktemp("code")
    shutil.copy(lib, d / "lib.so")
    subprocess.run([tool("llvm-objdump"), "--offloading", "lib.so"], cwd=d, check=True, stdout=subprocess.DEVNULL)
    out = sorted(str(d / f) for f in os.listdir(d) if f.endswith("gfx950"))
    assert out
    return out


@pytest.fixture(scope="module")
def spills(code_objects):
    """kernel -> registers kept in memory"""
    out = {}
    for f in code_objects:
        notes = subprocess.run([tool("llvm-readelf"), "--notes", f], check=True, capture_output=True, text=True).stdout
        out.update((n, int(v)) for n, v in re.findall(r"\.name:\s+(_Z\S+)\n(?:(?!\.name:\s+_Z).*\n)*?\s+\.vgpr_spill_count:\s+(\d+)", notes))
    return out


def test_short_products_fit_their_registers(spills):
    """a few registers of a row tile's sums in memory cost nothing that was measured; 220 made a step three times as long"""
    short = {n: v for n, v in spills.items() if "short_gemm_kernel" in n}
    assert len(short) > 40
    assert {n: v for n, v in short.items() if v > 32} == {}
