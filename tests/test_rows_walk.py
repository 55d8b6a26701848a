"""The load order of gemv_rows_kernel (csrc/qmm_rows_walk.hpp), walked on the host: the same
walk_rows the kernel runs, with callbacks that record the loads and check each wait against
them.  Loads of a wave return in the order they were issued, so a wait that leaves `a` loads
outstanding covers an item's copies only if at least `a` loads followed them."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "qmm_rows_walk.hpp"

static void check(bool ok, const char* what, int mg_count, int groups, int g, int mg) {
    if (ok) return;
    std::printf("%s: kMG=%d groups=%d group=%d item=%d\n", what, mg_count, groups, g, mg);
    std::exit(1);
}

// kCopies copies per item, R loads per group's weights (any count must do)
template <int kMG>
static void walk(int g0, int groups, int R) {
    constexpr int kCopies = 8;
    const int g1 = g0 + groups;
    long issued = 0, landed = 0;  // loads so far; of these, certainly complete
    struct { int g = -1, mg = -1; long end = 0; bool read = true; } slot[2];
    struct { int g = -1; long end = 0; bool used = true; } raw;
    int group = g0 - 1, next_mg = 0;
    auto copy = [&](int g, int mg, int s) {
        check(slot[s].read, "copy over an unread item", kMG, groups, g, mg);
        issued += kCopies;
        slot[s] = {g, mg, issued, false};
    };
    qmm::walk_rows<kMG>(
        g0, g1,
        [&](int g) {
            check(raw.used, "weights loaded over unused ones (dead loads)", kMG, groups, g, -1);
            check(g >= g0 && g < g1, "weights out of the slice", kMG, groups, g, -1);
            issued += R;
            raw = {g, issued, false};
        },
        [&] {
            check(next_mg == 0, "group begun before the last one ended", kMG, groups, group, next_mg);
            ++group;
            check(raw.g == group && !raw.used, "weights of another group", kMG, groups, group, -1);
            raw.used = true;
            if (raw.end > landed) landed = raw.end;  // the conversion waits for its own loads
        },
        copy,
        [&](int mg, int s, int raws, int ng, int nmg) {
            check(mg == next_mg, "items out of order", kMG, groups, group, mg);
            next_mg = (mg + 1) % kMG;
            check(slot[s].g == group && slot[s].mg == mg && !slot[s].read, "another item in the slot", kMG, groups, group, mg);
            const long wait = issued - (kCopies + (long)raws * R);
            if (wait > landed) landed = wait;
            // by the count itself, not by what the conversion happened to wait for
            check(wait >= slot[s].end, "copies may be in flight when they are read", kMG, groups, group, mg);
            slot[s].read = true;
            check(ng >= g0 && ng < g1, "copies out of the slice", kMG, groups, ng, nmg);
            copy(ng, nmg, s);
        },
        [&] { raw.used = true; });
    check(group == g1 - 1 && next_mg == 0 && raw.used, "slice not finished", kMG, groups, group, next_mg);
}

int main() {
    for (int R : {2, 3, 5, 7, 18, 21})
        for (int groups = 1; groups <= 40; ++groups)
            for (int g0 : {0, 5}) {
                walk<1>(g0, groups, R);
                walk<2>(g0, groups, R);
                walk<4>(g0, groups, R);
            }
    std::printf("walk ok\n");
    return 0;
}
"""


def test_every_item_waits_for_its_copies(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no C++ compiler on this machine")
    src = tmp_path / "walk.cpp"
    src.write_text(PROGRAM)
    cmd = [cxx, "-std=c++17", "-O1", "-Wall", "-Wno-unknown-pragmas", "-D__host__=", "-D__device__=",
           "-D__forceinline__=inline", "-I", os.path.join(ROOT, "openmini-v1_amd", "csrc"), str(src), "-o",
           str(tmp_path / "walk")]
    subprocess.run(cmd, check=True, capture_output=True, text=True)
    p = subprocess.run([str(tmp_path / "walk")], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0 and "walk ok" in p.stdout, p.stdout + p.stderr
