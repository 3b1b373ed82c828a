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


def test_persistent_kernels_keep_their_queue_in_registers(code_objects):
    """a loop over tiles that is too long to be unrolled indexes the queue at run time, in scratch memory: three times as long a token"""
    scratch = {}
    for f in code_objects:
        notes = subprocess.run([tool("llvm-readelf"), "--notes", f], check=True, capture_output=True, text=True).stdout
        scratch.update((n, int(v)) for n, v in re.findall(r"\.name:\s+(_Z\S+mega_decode_kernel\S+)\n(?:(?!\.name:\s+_Z).*\n)*?\s+\.private_segment_fixed_size:\s+(\d+)", notes))
    assert len(scratch) == 6 and set(scratch.values()) == {0}, scratch


def test_nothing_moves_between_matrix_products_in_inline_assembly(code_objects):
    """gemm_wide_kernel with 256-token tiles names its matrix instructions in inline assembly, where the compiler knows nothing of the
    states that have to lie between one of them and a move of its registers: it must have no move, no spill and no other matrix
    instruction between the first and the last product of a half step, and the waits around a half must be there"""
    bodies = {}
    for f in code_objects:
        text = subprocess.run([tool("llvm-objdump"), "-d", "--no-show-raw-insn", f], check=True, capture_output=True, text=True).stdout
        parts = re.split(r"\n[0-9a-f]+ <(\S+)>:\n", text)
        bodies.update((n, b) for n, b in zip(parts[1::2], parts[2::2]) if "gemm_wide_kernel" in n and "ELi128E" in n)
    assert len(bodies) >= 3
    for name, body in bodies.items():
        ins = [line.split("//")[0].strip() for line in body.split("\n") if line.strip()]
        at = [i for i, x in enumerate(ins) if "mfma" in x]
        assert len(at) == 128, name
        for half in (at[:64], at[64:]):
            inside = ins[half[0]:half[-1] + 1]
            # operands of the next half come from LDS, its loads go there; addresses are all else that is computed
            allowed = r"v_mfma_f32_16x16x32_bf16 a\[|ds_read_b128 v\[|global_load_lds_dwordx4|s_|v_(lshl_add_u64|add3_u32|add_u32_e32|add_co_u32|addc_co_u32|lshlrev_b64|mad_u64_u32)"
            assert [x for x in inside if not re.match(allowed, x)] == [], name
            assert re.match(r"s_nop [1-9]", ins[half[0] - 1]), (name, ins[half[0] - 1])
            assert ins[half[-1] + 1] == "s_nop 15", (name, ins[half[-1] + 1])


def test_nothing_moves_between_matrix_products_of_tiles_with_units(code_objects):
    """the same of the tiles of 160 and 192 tokens, whose kernels hold a loop for every number of units of 32 tokens"""
    allowed = r"v_mfma_f32_16x16x32_bf16 a\[|ds_read_b128 v\[|global_load_lds_dwordx4|s_|v_(lshl_add_u64|add3_u32|add_u32_e32|add_co_u32|addc_co_u32|lshlrev_b64|mad_u64_u32)"
    seen = 0
    for f in code_objects:
        text = subprocess.run([tool("llvm-objdump"), "-d", "--no-show-raw-insn", f], check=True, capture_output=True, text=True).stdout
        parts = re.split(r"\n[0-9a-f]+ <(\S+)>:\n", text)
        for name, body in zip(parts[1::2], parts[2::2]):
            if "gemm_wide_kernel" not in name or not re.search(r"ELi(80|96)E", name):
                continue
            seen += 1
            ins = [line.split("//")[0].strip() for line in body.split("\n") if line.strip()]
            halves, inside = 0, False
            for i, x in enumerate(ins):
                if "mfma" in x and not inside:
                    assert re.match(r"s_nop [1-9]", ins[i - 1]), (name, ins[i - 1])
                    inside = True
                if inside:
                    assert re.match(allowed, x), (name, x)
                    if x == "s_nop 15":
                        inside, halves = False, halves + 1
            assert not inside and halves == 2 * (5 if "ELi80E" in name else 6), (name, halves)
    assert seen == 6      # three epilogues of each
