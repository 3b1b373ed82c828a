"""Asks the rules that choose kernels by sizes (csrc/lv_*_plan.h), compiled for the host."""
import os
import subprocess
import tempfile

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llama-vulkan_amd", "csrc")
SOURCE = r"""
#include "lv_bf_plan.h"
#include "lv_small_plan.h"
#include <cstdio>
#include <iostream>
#include <string>
int main()
{
    for (std::string what; std::cin >> what;) {
        if (what == "small") {
            lv::SmallShape m;
            std::cin >> m.D >> m.F >> m.heads >> m.rot >> m.layers >> m.vocab >> m.block_bytes;
            const lv::SmallPlan p = lv::small_plan(m);
            printf("%u %u %u\n", p.wgs, p.own, p.elements);
        } else if (what == "product") {
            uint32_t rows, n, kp, slices;
            std::cin >> rows >> n >> kp >> slices;
            const lv::BfPlan p = lv::bf_plan(rows, n, kp, slices);
            printf("%d %u\n", (int)p.tiles, p.slices);
        } else if (what == "experts") {
            uint32_t n;
            lv::ExpertShape e;
            std::cin >> n >> e.experts >> e.top >> e.rows >> e.kp >> e.down_rows >> e.down_kp;
            const lv::ExpertPlan p = lv::expert_plan(n, e);
            printf("%d %d %d\n", (int)p.gate_up, (int)p.down, (int)p.gate_up_by_expert);
        }
    }
}
"""
_exe = []
TILES = ("128x128", "256x128", "256x160", "256x192", "256x256")


def ask(lines):
    """a list of answers, tuples of numbers, to questions:
    ("small", dim, ff, heads, head size, layers, vocab, bytes of a block) -> workgroups, blocks of a workgroup, cache elements
    ("product", rows, tokens, columns, slices at most) -> TILES, slices
    ("experts", tokens, experts, of a token, rows, columns, rows, columns) -> TILES of gate and up, of down, gate and up an expert after the other"""
    if not _exe:
        d = tempfile.TemporaryDirectory()
        src, exe = os.path.join(d.name, "main.cpp"), os.path.join(d.name, "main")
        with open(src, "w") as f:
            f.write(SOURCE)
        subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, src, "-o", exe], check=True)
        _exe.extend((exe, d))
    text = "\n".join(" ".join(map(str, q)) for q in lines)
    out = subprocess.run([_exe[0]], input=text, capture_output=True, text=True, check=True).stdout
    return [tuple(map(int, line.split())) for line in out.splitlines()]
