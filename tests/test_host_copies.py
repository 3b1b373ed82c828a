"""Which copies of its matrices a batched step asks for on a device whose memory holds only some of them (lv_copies.h)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = r"""
#include "lv_copies.h"
#include <cstdio>
#include <cstdlib>
// memory, bytes of the prompt and of the short copy, then steps: c = whole chunks and a rest that pays, r = a step that pays, n = one that does not
int main(int, char **v)
{
    long memory = atol(v[1]);
    int state[2] = {0, 0};
    for (const char *step = v[4]; *step; step++) {
        auto make = [&](int k) {
            if (!state[k]) {
                state[k] = memory >= atol(v[2 + k]) ? 1 : -1;
                if (state[k] > 0) memory -= atol(v[2 + k]);
            }
            return state[k] > 0;
        };
        const lv::BatchCopies c = lv::batch_copies(*step == 'c', *step != 'n', [&] { return make(0); }, [&] { return make(1); },
                                                   [&] { return state[0] || state[1] || memory >= atol(v[2]) + atol(v[3]); });
        printf("%d%d ", c.batch, c.mid);
    }
    printf("prompt %d short %d", state[0], state[1]);
}
"""


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("copies")
    (d / "main.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "llama-vulkan_amd", "csrc"), str(d / "main.cpp"), "-o", str(d / "main")], check=True)
    return str(d / "main")


@pytest.mark.parametrize("memory,steps,want", [
    # room for both: each step asks for what it reads
    (30, "r", "11 prompt 0 short 1"),
    (30, "c", "11 prompt 1 short 1"),
    (30, "n", "10 prompt 1 short 0"),
    (30, "rcn", "11 11 10 prompt 1 short 1"),
    # room for the prompt copy alone: no step takes it away from the long ones
    (22, "c", "10 prompt 1 short -1"),
    (22, "r", "10 prompt 1 short -1"),
    (22, "rcr", "10 10 10 prompt 1 short -1"),
    # room for the short copy alone: steps that need no other still have it, long ones go token by token
    (10, "r", "11 prompt -1 short 1"),
    (10, "cr", "00 11 prompt -1 short 1"),
    (10, "nr", "00 11 prompt -1 short 1"),
    # room for neither
    (5, "rcn", "00 00 00 prompt -1 short -1"),
])
def test_copies_a_step_asks_for(exe, memory, steps, want):
    assert subprocess.run([exe, str(memory), "20", "8", steps], capture_output=True, text=True, check=True).stdout == want
