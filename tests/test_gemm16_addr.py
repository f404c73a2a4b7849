"""No load of the GEMM wave tiles leaves its operand: the kernel's own offset
arithmetic (csrc/osh_gemm16_addr.h, plain C++ on the host) is enumerated over
every tile, lane and chunk at the remainders of M, K and N.

A word of a buffer load is fetched, at vector + scalar offset, when the offset
lies below the descriptor's size: the vector offset alone or (as gfx950 does it)
vector plus scalar.  Every word that the looser reading fetches must lie in the
operand, and every word the product needs must be fetched under the stricter one,
from where the matrix holds it."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "onnxsharp_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "osh_gemm16_addr.h"
using namespace osh;

static long long loads = 0;
static const char *what;
static int tile, M, K, N, lda, ldb;

static void check(G16Off o, int words, int bytes, const bool *need, const int *at) {
    loads++;
    for (int q = 0; q < words; q++) {
        const long long v = (unsigned)o.vec + 4LL * q, a = (long long)o.vec + o.scalar + 4 * q;
        const bool may = v < bytes, does = v + (unsigned)o.scalar < bytes;
        if ((may && (a < 0 || a + 4 > bytes)) || (need[q] && (!does || a != at[q]))) {
            printf("%s of tile %d, %d x %d x %d, lda %d, ldb %d: word at byte %lld of %d %s\n", what, tile, M, K, N, lda,
                   ldb, a, bytes, need[q] ? "is not the one needed" : "lies outside");
            exit(1);
        }
    }
}

template <bool TAIL>
static void chunk_a(int c, int rows, int kc) {  // the kernel clamps rows to M - 1
    what = "A";
    const int bytes = g16_bytes_a(M, K, lda);
    for (int r = 0; r < rows; r++)
        for (int kq = 0; kq < kc / 4; kq++) {
            const int row = r < M ? r : M - 1;
            bool need[4];
            int at[4];
            for (int q = 0; q < 4; q++) {
                const int k = c * kc + 4 * kq + q;
                need[q] = k < K, at[q] = (row * lda + k) * 4;
            }
            check(g16_off_a<TAIL>(g16_lane_a(row, kq, lda), c * kc), 4, bytes, need, at);
        }
}

static int first_column(int bv, int col) {
    return bv == 1 ? g16_col<1>(col, N) : bv == 2 ? g16_col<2>(col, N) : bv == 3 ? g16_col<3>(col, N) : g16_col<4>(col, N);
}

template <bool TAIL>
static void chunk_b(int c, int cols, int bv, int kc) {
    what = "B";
    const int bytes = g16_bytes_b(K, N, ldb);
    for (int s = 0; s < kc / 4; s++)
        for (int g = 0; g < 4; g++)
            for (int col = 0; col < cols; col += bv) {
                const int k = c * kc + 4 * s + g, first = first_column(bv, col);
                bool need[4];
                int at[4];
                for (int q = 0; q < bv; q++) need[q] = k < K && col < N, at[q] = (k * ldb + first + q) * 4;
                check(g16_off_b<TAIL>(g16_lane_b(g, first, ldb), c * kc + 4 * s, ldb), bv, bytes, need, at);
            }
}

// Every column is stored, by lanes whose columns all exist.
static void columns(int cols, int bv) {
    bool stored[512] = {};
    for (int col = 0; col < cols && col < N; col += bv)
        for (int q = 0; q < bv; q++) stored[first_column(bv, col) + q] = true;
    for (int j = 0; j < 512; j++)
        if (stored[j] != (j < N)) {
            printf("tile %d, N %d: column %d %s\n", tile, N, j, stored[j] ? "does not exist" : "is not stored");
            exit(1);
        }
}

int main() {
    const int tiles[][4] = {TILES};  // tm, tn, bv, kc
    const int ms[] = {1, 15, 17, 33}, ns[] = {1, 2, 3, 4, 5, 6, 7, 15, 16, 31, 32, 33, 47, 48, 50, 63, 64, 67, 129};
    for (const auto &t : tiles) {
        const int tm = t[0], tn = t[1], bv = t[2], kc = t[3];
        for (int m : ms)
            for (K = 1; K <= 2 * kc + 5; K++)
                for (int n : ns)
                    for (int pad = 0; pad < 3; pad++) {
                        M = m, N = n, lda = K + pad, ldb = N + 2 * pad;
                        const int rows = (M + 16 * tm - 1) / (16 * tm) * 16 * tm;
                        const int cols = (N + 16 * bv * tn - 1) / (16 * bv * tn) * 16 * bv * tn;
                        if (M == ms[0] && N >= bv) columns(cols, bv);
                        for (int c = 0; c * kc < K; c++) {
                            const bool tail = (c + 1) * kc > K;
                            if (N == ns[0]) tail ? chunk_a<true>(c, rows, kc) : chunk_a<false>(c, rows, kc);
                            if (M == ms[0] && N >= bv) tail ? chunk_b<true>(c, cols, bv, kc) : chunk_b<false>(c, cols, bv, kc);
                        }
                    }
        tile++;
    }
    printf("ok %lld loads\n", loads);
    return 0;
}
"""


def test_gemm_tile_loads_stay_inside_their_operands(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("no g++")
    src = open(os.path.join(CSRC, "osh_gemm.hip")).read()
    table = src[src.index("kG16[] = {"):src.index("kG16Count")]
    tiles = re.findall(r"\{(\d+), (\d+), (\d+), (\d+)\}", table)
    assert len(tiles) >= 11
    prog = tmp_path / "addr.cpp"
    prog.write_text(PROGRAM.replace("TILES", ", ".join("{%s}" % ", ".join(t) for t in tiles)))
    exe = tmp_path / "addr"
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, str(prog), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout
