"""The host block that the order stages gather a call's inputs in, built with the
standard library's own bounds checks: empty pieces anywhere, also last, where
their offset is at the block's end."""
import os
import subprocess

PROGRAM = r"""
#include "rc_block.h"
#include <stdio.h>
int main()
{
    std::vector<unsigned char> h;
    const std::vector<int> none, some = {1, 2, 3};
    for (int call = 0; call < 2; ++call) {
        RcBlock b(h, 4096);
        const double c[2] = {0.5, 0.25};
        const size_t a = b.put(c, sizeof c), e = b.put(none), s = b.put(some);
        const size_t z = b.put(none), n = b.put(nullptr, 0);
        if (a != 0 || e != 256 || s != 256 || z != 512 || n != 512 || h.size() != 512) return 1;
        if (memcmp(&h[a], c, sizeof c) != 0 || memcmp(&h[s], some.data(), 12) != 0) return 2;
    }
    RcBlock whole(h, 0);
    const std::vector<unsigned char> full(256, 7);
    whole.put(full);
    if (whole.put(none) != 256 || h.size() != 256) return 3;
    puts("ok");
    return 0;
}
"""


def test_pieces_and_empty_pieces(tmp_path):
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                        "the-rule-and-compass_amd", "csrc")
    src, exe = tmp_path / "block.cpp", tmp_path / "block"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-D_GLIBCXX_ASSERTIONS", "-I", csrc,
                    str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert (out.returncode, out.stdout) == (0, "ok\n"), out.stderr
