"""The size rule of the kept device blocks (csrc/pt_blocks.h, plain C++), over
the whole of size_t: it ends for every size, rounds up by at most an eighth or
to 512 bytes, and is stable."""
import os
import subprocess

PROGRAM = r"""
#include "pt_blocks.h"
#include <initializer_list>
#include <stdio.h>
using pt::block_class;
static int check(size_t b)
{
    const size_t c = block_class(b);
    if (c < b || c % 512 || block_class(c) != c || (c - b >= 512 && c - b > b / 8)) {
        printf("%zu -> %zu\n", b, c);
        return 1;
    }
    return 0;
}
int main()
{
    int bad = 0;
    for (size_t b = 1; b < 100000; b++) bad += check(b);
    for (int s = 9; s < 63; s++)
        for (int k = -3; k <= 3; k++)
            for (size_t f = 8; f <= 16; f++) {
                const size_t b = ((size_t)f << s >> 3) + (size_t)(long long)k;
                if (b && b <= pt::kMaxBlockBytes) bad += check(b);
            }
    for (size_t b : {pt::kMaxBlockBytes, pt::kMaxBlockBytes - 1, pt::kMaxBlockBytes / 8 * 7}) bad += check(b);
    // above the largest request the rule is not asked, and ends all the same
    for (size_t b : {(size_t)1 << 63, SIZE_MAX, SIZE_MAX - 511}) block_class(b);
    return bad != 0;
}
"""


def test_rule(tmp_path):
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "php-gpu-tensors_amd", "csrc")
    src, exe = tmp_path / "blocks.cpp", tmp_path / "blocks"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-I", csrc, str(src), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
