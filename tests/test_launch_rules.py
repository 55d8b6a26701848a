"""The launch rules that are plain C++ (csrc/qmm_rows_shape.hpp, qmm_gemm_shape.hpp), asked on the
host: at sizes where the ways were measured on MI355X they take the fastest or one within 3%."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def run_program(tmp_path, name, text):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no C++ compiler on this machine")
    src = tmp_path / f"{name}.cpp"
    src.write_text(text)
    cmd = [cxx, "-std=c++17", "-O1", "-Wall", "-I", os.path.join(ROOT, "include"), "-I",
           os.path.join(ROOT, "openmini-v1_amd", "csrc"), str(src), "-o", str(tmp_path / name)]
    subprocess.run(cmd, check=True, capture_output=True, text=True)
    p = subprocess.run([str(tmp_path / name)], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0 and "ok" in p.stdout, p.stdout + p.stderr


ROWS = r"""
#include <cstdio>
#include <cstdlib>
#include <initializer_list>
#include "qmm_rows_shape.hpp"
using namespace qmm;

enum { Q4_0 = 2, Q4_1 = 3, Q8_0 = 7, Q4_K = 12, Q5_K = 13, Q6_K = 14 };

int main() {
    // first launch of `rows` rows; split and waves as a 16-row call on the weight has them
    struct { int type, n, k, split, waves, rows, first; } cases[] = {
        // three tiles, block minimum, eight slices: at most two row groups a launch
        {Q5_K, 12288, 8192, 1, 8, 40, 32}, {Q5_K, 11008, 16384, 1, 8, 64, 32}, {Q4_1, 9000, 8192, 1, 8, 17, 17},
        {Q4_1, 11008, 8192, 1, 8, 33, 32},
        // in four slices, and the other types: all rows
        {Q5_K, 11008, 4096, 1, 4, 40, 40}, {Q4_1, 12288, 4096, 1, 4, 64, 64}, {Q8_0, 12288, 8192, 1, 8, 64, 64},
        // one tile of a two-way split: by K, rows and type
        {Q4_1, 1536, 8192, 2, 4, 17, 16}, {Q4_1, 1536, 8192, 2, 4, 32, 32}, {Q4_1, 2048, 12288, 2, 4, 32, 16},
        {Q5_K, 2048, 12288, 2, 4, 64, 64}, {Q5_K, 2048, 12288, 2, 4, 40, 16}, {Q5_K, 1536, 4096, 2, 4, 17, 17},
        {Q4_0, 2048, 8192, 2, 4, 17, 17}, {Q4_0, 2048, 16128, 2, 4, 17, 16}, {Q8_0, 2048, 12288, 2, 4, 20, 16},
        {Q8_0, 2048, 12288, 2, 4, 64, 64}, {Q4_1, 4096, 9216, 2, 4, 17, 16}, {Q4_1, 4096, 9216, 2, 4, 24, 24},
        {Q5_K, 4096, 9216, 2, 4, 17, 17}, {Q4_0, 4096, 12288, 2, 4, 17, 17},
        // too many tiles; splits of eight waves and of four parts; one wave
        {Q4_0, 12304, 4096, 1, 4, 64, 16}, {Q4_0, 4096, 16384, 2, 8, 64, 16}, {Q4_0, 1000, 8192, 4, 4, 64, 16},
        {Q4_0, 1000, 512, 1, 1, 64, 16}};
    for (const auto& c : cases) {
        const RowsShape s = rows_shape(c.type, (c.n + 15) / 16, (c.k + 127) / 128, c.split, c.waves, false);
        const int got = next_rows(s, c.rows);
        if (got != c.first) {
            std::printf("type %d %d x %d, %d rows: first launch %d, expected %d\n", c.type, c.n, c.k, c.rows, got, c.first);
            return 1;
        }
    }
    // every call is split into launches that their kernels take
    const int types[] = {Q4_0, Q4_1, Q8_0, Q4_K, Q5_K, Q6_K}, splits[][2] = {{1, 1}, {1, 4}, {1, 8}, {2, 4}, {2, 8}, {4, 4}};
    for (int type : types)
        for (int tiles : {1, 64, 65, 128, 129, 256, 257, 512, 513, 768, 769, 2000})
            for (int groups : {1, 8, 40, 46, 64, 90, 127, 128, 300})
                for (const auto& sp : splits)
                    for (int pair = 0; pair < 2; ++pair) {
                        const RowsShape s = rows_shape(type, tiles, groups, sp[0], sp[1], pair);
                        for (int rest = 1; rest <= 200; ++rest) {
                            const int n = next_rows(s, rest);
                            const bool ok = n >= 1 && n <= rest && n <= kRowsMax && (n <= kPassRows || (s.w != 0 && n <= s.most)) &&
                                            (n == rest || n % kPassRows == 0) && s.t >= 1 && s.t <= 3 && (!pair || s.t == 1);
                            if (!ok) {
                                std::printf("type %d tiles %d groups %d split %d: %d of %d rows\n", type, tiles, groups, sp[0], n, rest);
                                return 1;
                            }
                        }
                    }
    std::printf("ok\n");
    return 0;
}
"""


def test_rows_of_a_pass(tmp_path):
    run_program(tmp_path, "rows", ROWS)


GEMM = r"""
#include <cstdio>
#include <initializer_list>
#include "qmm_gemm_shape.hpp"
using namespace qmm;

enum { Q4_0 = 2, Q8_0 = 7, Q4_K = 12, Q6_K = 14 };

// workgroups per CU: what the kernels' registers and LDS allow on gfx950
static const int kPerCu[6][kShapes] = {{1, 1, 1, 2, 2, 1, 4, 2}, {1, 1, 1, 2, 1, 1, 3, 2}, {-1, 1, 1, -1, 1, 1, 2, -1},
                                       {1, 1, 1, 2, 2, 1, 4, 2}, {1, 1, 1, 2, 2, 1, 4, 2}, {1, 1, 1, 1, 1, 1, 3, 2}};
static int pick(int type, int n, int k, int m, bool split) {
    return choose_gemm_shape(type, (n + 15) / 16, k, m, kPerCu[(split ? 3 : 0) + (type == Q8_0 ? 1 : type == Q6_K ? 2 : 0)], split);
}

int main() {
    // measured with every shape forced: those within 3% of the fastest
    struct { int type, n, k, m; bool split; unsigned good; } cases[] = {
        {Q8_0, 11008, 2048, 384, true, 1u << 0 | 1u << 7},  // 53 us; 64 x 96 64
        {Q8_0, 7168, 4096, 600, true, 1u << 0}, {Q8_0, 14336, 4096, 300, true, 1u << 0},
        {Q8_0, 13824, 4096, 100, true, 1u << 4},
        {Q8_0, 13824, 4096, 100, false, 1u << 6}, {Q8_0, 11008, 4096, 768, false, 1u << 6 | 1u << 7},
        {Q8_0, 13824, 4096, 1536, false, 1u << 7}, {Q8_0, 11008, 4096, 512, false, 1u << 0},
        {Q8_0, 4096, 11008, 100, true, 1u << 5}, {Q4_0, 4096, 4096, 128, false, 1u << 5},
        {Q6_K, 11008, 2048, 448, false, 1u << 6},
        // even in long runs (121 us); 141 against 154 in the first milliseconds after idle
        {Q6_K, 11008, 4096, 512, false, 1u << 1}};
    for (const auto& c : cases) {
        const int got = pick(c.type, c.n, c.k, c.m, c.split);
        if (got < 0 || !(c.good >> got & 1)) {
            std::printf("type %d %d x %d, %d rows, split %d: shape %d\n", c.type, c.n, c.k, c.m, c.split, got);
            return 1;
        }
    }
    // always one that is built, whatever a CU holds of it
    for (int type : {Q4_0, Q8_0, Q4_K, Q6_K})
        for (int split = 0; split < 2; ++split)
            for (int tiles : {1, 2, 100, 688, 2000, 40000})
                for (int k : {32, 4096, 65536})
                    for (int m : {1, 64, 65, 300, 4096, 300000})
                        for (int cu : {0, 1, 2, 8}) {
                            int per_cu[kShapes];
                            for (int i = 0; i < kShapes; ++i)
                                per_cu[i] = !split && type == Q6_K && (i == 0 || i == 3 || i == 7) ? -1 : cu;
                            const int got = choose_gemm_shape(type, tiles, k, m, per_cu, split);
                            if (got < 0 || got >= kShapes || per_cu[got] < 0) {
                                std::printf("type %d tiles %d k %d m %d: shape %d\n", type, tiles, k, m, got);
                                return 1;
                            }
                        }
    std::printf("ok\n");
    return 0;
}
"""


def test_gemm_shape(tmp_path):
    run_program(tmp_path, "gemm", GEMM)
