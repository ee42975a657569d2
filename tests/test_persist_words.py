"""Words in which the persistent kernel publishes positions and sums (md_pk_words.h), on the CPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <initializer_list>
#include "md_pk_words.h"
int main(int, char** v) {
    const unsigned n = (unsigned)strtoul(v[1], nullptr, 10);
    int bad = 0;
    for (uint32_t data : {0u, 1u, 0x7f800000u, 0xffffffffu}) {
        const uint64_t s = pk::word(data, pk::sum_tag(n));
        bad += (uint32_t)s != data || !pk::sum_of_step(s, n);
        for (unsigned fl = 0; fl < 8; fl++) {
            const uint64_t p = pk::word(data, pk::pos_tag(n, fl, data & 0xffffu));
            bad += (uint32_t)p != data || ((unsigned)(p >> 32) & 0xffffu) != (data & 0xffffu) ||
                   ((unsigned)(p >> 48) & 7u) != fl || !pk::pos_of_step(p, n);
            for (unsigned m : {n - 2, n - 1, n + 1, n + 2}) bad += pk::pos_of_step(p, m) || pk::sum_of_step(s, m);
        }
    }
    // an exchange that has not begun holds zeros
    if (n <= 3) bad += pk::pos_of_step(0, n) || pk::sum_of_step(0, n);
    printf("%d\n", bad);
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("words")
    (d / "words.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "md_gpu_amd", "csrc"), str(d / "words.cpp"),
                    "-o", str(d / "words")], check=True)
    return str(d / "words")


@pytest.mark.parametrize("n", [1, 2, 3, 8191, 8192, 8193, 2**16, 2**29 - 1, 2**29, 2**29 + 1, 2**30, 2**31 - 1])
def test_words_carry_their_step(program, n):
    """Data and flags come back, the word is its step's and no neighboring step's, up to the longest run."""
    assert subprocess.run([program, str(n)], capture_output=True, text=True, check=True).stdout == "0\n"
