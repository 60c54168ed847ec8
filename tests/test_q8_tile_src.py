"""Every byte the packed Q8_0 tile kernel's loads address lies inside its operands (csrc/q8_tile_src.h, the offsets the
kernel itself uses, compiled here for the CPU): all waves and lanes of the corner workgroups, the first and last stage, at
row and column counts that end inside a tile, a wave and a subtile."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "startlux-prism_amd", "csrc")
PROG = r"""
#include <stdio.h>
#include <initializer_list>
#include "q8_tile_src.h"
using namespace prism;
static long bad = 0;
static void in(const char* what, int64_t off, int bytes, int64_t size, int M, int N, int K) {
    if (off < 0 || off + bytes > size) { if (!bad++) printf("%s at %ld of %ld, M %d N %d K %d\n", what, (long)off, (long)size, M, N, K); }
}
template <bool PAN, int NT> static void check(int M, int N, int K) {
    const int NS = K / 128, last_m = (M - 1) / 128 * 128, last_n = (N - 1) / (32 * NT) * 32 * NT;
    const int64_t rows = PAN ? (M + 127) / 128 * 128 : M;
    for (int m0 : {0, last_m}) for (int n0 : {0, last_n}) for (int wv = 0; wv < 4; wv++) for (int l = 0; l < 64; l++) {
        const auto s = q8_tile_src<PAN, NT>(m0, n0, wv, l, M, N, K);
        for (int st : {0, NS - 1}) {
            for (int bi = 0; bi < 4; bi++)
                in("activations", s.a_base + (int64_t)s.a_v + (PAN ? st * 4096L + bi * 1024 : st * 128L + bi * 32), 16, rows * K, M, N, K);
            for (int i = 0; i < NT; i++)
                in("weights", s.w_base + (int64_t)s.w_v + s.w_s[i] + st * 2048L, 16, (int64_t)N * K, M, N, K);
            in("scales", s.s_base + (int64_t)s.s_v + st * 128L, 4, (int64_t)N * K / 16, M, N, K);
        }
        // a row and column inside the matrix is read where it lies
        const int m = m0 + 32 * wv + (l & 31), tid = 64 * wv + l;
        if (!PAN && m < M) in("row", s.a_base + (int64_t)s.a_v - ((int64_t)m * K + 16 * (l >> 5)), 0, 0, M, N, K);
        for (int i = 0; i < NT; i++) {
            const int64_t t = n0 / 16 + 2 * i + tid / 128;
            if (t < N / 16) in("tile", s.w_base + (int64_t)s.w_v + s.w_s[i] - (t * 16 * K + tid % 128 * 16), 0, 0, M, N, K);
        }
        const int64_t t = n0 / 16 + tid / 32;
        if (t < N / 16) in("scale tile", s.s_base + (int64_t)s.s_v - (t * K + tid % 32 * 4), 0, 0, M, N, K);
    }
}
int main() {
    for (int M : {1, 31, 32, 33, 96, 97, 127, 128, 129, 140, 777, 1024, 1100})
        for (int N = 16; N <= 272; N += 16)
            for (int K : {128, 256, 5120, 1 << 23}) {
                check<false, 2>(M, N, K), check<false, 3>(M, N, K), check<false, 4>(M, N, K);
                check<true, 2>(M, N, K), check<true, 3>(M, N, K), check<true, 4>(M, N, K);
            }
    return bad != 0;
}
"""


def test_loads_stay_inside_the_operands(tmp_path):
    src, exe = tmp_path / "src.cpp", tmp_path / "src"
    src.write_text(PROG)
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-w", "-I", CSRC, "-D__host__=", "-D__device__=",
                        "-D__forceinline__=inline", str(src), "-o", str(exe)], capture_output=True, text=True)
    if r.returncode != 0:
        pytest.fail(r.stderr)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
