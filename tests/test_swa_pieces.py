"""Pieces of eight attention weights that the backward reads whole never leave the weight tensor."""
import ctypes
import os
import subprocess

from nl_hecate_amd import ffi

SOURCE = r"""
#include "swa_pieces.h"
// first piece read whole that lies outside the tensor, as a code of its case; 0 if there is none
extern "C" long long piece_outside(int heads, int s, int ws) {
    using namespace nlh;
    for (int head = 0; head < heads; head++)
        for (int t = 0; t < s; t++) {
            const int lsq = t + 1 - ws > 0 ? t + 1 - ws : 0;
            for (int key0 = lsq / 8 * 8; key0 <= t; key0 += 8) {
                const long long at = ((long long)head * s + t) * ws + (key0 - lsq);
                const bool whole = !edge_head(head, heads, s, ws) || piece_inside(t, s, ws, key0 - lsq);
                if (whole && (at < 0 || at + 8 > (long long)heads * s * ws)) return 1 + head + 1000LL * t + 1000000LL * key0;
            }
        }
    return 0;
}
"""


def test_pieces_read_whole_lie_inside_the_tensor(tmp_path):
    src, so = tmp_path / "pieces.cpp", tmp_path / "pieces.so"
    src.write_text(SOURCE)
    csrc = os.path.join(os.path.dirname(os.path.abspath(ffi.__file__)), "csrc")
    subprocess.check_call(["g++", "-O1", "-shared", "-fPIC", "-D__host__=", "-D__device__=", "-D__forceinline__=inline",
                           "-I", csrc, "-o", str(so), str(src)])
    outside = ctypes.CDLL(str(so)).piece_outside
    outside.restype = ctypes.c_longlong
    sizes = [(heads, s, ws) for heads in range(1, 6) for s in range(1, 21) for ws in range(1, 21)]
    sizes += [(4, s, ws) for s in (63, 64, 65, 127, 130) for ws in (1, 2, 5, 7, 8, 63, 64, 511)]
    assert [c for c in sizes if outside(*c)] == []
