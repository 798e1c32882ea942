"""Chunks of the matrix-core attention (csrc/attention_chunks.hpp) without a device: the choice ends for any number of rows and kv heads, also where one chunk a row is
already more than two workgroups a CU, and is the smallest of its multiples of 128 that asks for no more than that."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "m40-llm_amd", "csrc")
MAIN = r"""
#include "attention_chunks.hpp"
#include <cstdio>
int main() {
    unsigned long long groups; unsigned span, cus, halve;
    while (std::scanf("%llu %u %u %u", &groups, &span, &cus, &halve) == 4) std::printf("%u\n", m40_attention_chunk(groups, span, cus, halve != 0));
}
"""


def expected(groups, span, cus, halve):
    chunk = (span * groups // cus + 64) // 128 * 128
    if 256 < chunk <= 512 and halve: chunk = 256
    chunk = max(chunk, 128)
    for c in range(chunk, 2048, 128):
        if c >= span or groups * -(-span // c) <= 2 * cus: return c
    return 2048


def test_every_choice_ends(tmp_path):
    (tmp_path / "chunks.cpp").write_text(MAIN)
    exe = str(tmp_path / "chunks")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(tmp_path / "chunks.cpp"), "-o", exe], check=True)
    cases = [(g, span, cus, h) for cus in (1, 64, 256) for h in (0, 1) for g in (1, 2, 7, 64, 256, 511, 512, 513, 516, 520, 1024, 4096, 65535 * 128)
             for span in (1, 127, 128, 129, 513, 1021, 2047, 2048, 2049, 4093, 32768, 131072, 0xFFFFFFFF)]
    try:
        out = subprocess.run([exe], input="\n".join(" ".join(map(str, c)) for c in cases), capture_output=True, text=True, check=True, timeout=20).stdout
    except subprocess.TimeoutExpired:
        pytest.fail("the choice of a chunk does not end")
    assert [int(x) for x in out.split()] == [expected(*c) for c in cases]
