"""The 32-lane decode asks the runtime how many workgroups a CU holds once a
launch shape: products of different steps that take turns on one instantiation
do not evict each other, and shapes whose dynamic LDS happens to be the same
do not share an answer."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include "resident.hpp"
#include <cstdio>
#include <initializer_list>
int main() {
    chm::ResidentTable table;
    int asked = 0;
    // QKV's four steps and the output projection's two, a hundred layers
    for (int layer = 0; layer < 100; ++layer)
        for (uint32_t steps : {4u, 2u})
            if (table.of(4, steps, [&] { ++asked; return 10 + steps; }) != 10 + steps) return 1;
    if (asked != 2) return 2;
    // four steps of four waves and sixteen of one: the same range sums' bytes
    if (table.of(1, 16, [&] { ++asked; return 40u; }) != 40 || table.of(4, 4, [&] { return 0u; }) != 14) return 3;
    // every shape has a place of its own
    chm::ResidentTable all;
    for (int pass = 0; pass < 2; ++pass)
        for (uint32_t waves : {1u, 4u})
            for (uint32_t steps = 1; steps <= 32; steps *= 2)
                if (all.of(waves, steps, [&] { return pass ? 0u : 64 * waves + steps; }) != 64 * waves + steps) return 4;
    std::puts("ok");
}
"""


def test_each_launch_shape_is_asked_for_once(tmp_path):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("g++ absent")
    source, program = tmp_path / "table.cpp", tmp_path / "table"
    source.write_text(PROGRAM)
    include = os.path.join(ROOT, "charlotte_amd", "csrc")
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", f"-I{include}", str(source), "-o", str(program)], check=True)
    assert subprocess.run([str(program)], capture_output=True, text=True, check=True).stdout == "ok\n"


def test_the_launch_keys_its_answer_by_the_launch_shape():
    """No cache of one answer keyed by the bytes of LDS is left in the ranges' launch."""
    text = open(os.path.join(ROOT, "charlotte_amd", "csrc", "gemv.hip")).read()
    launch = text[text.index("static void launch_ranges("):]
    launch = launch[:launch.index("\n}\n")]
    assert "ResidentTable" in launch and "cached_lds" not in launch
