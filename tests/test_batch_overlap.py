"""Which launches of a batch may run side by side (csrc/device/overlap.hpp):
a host program holds the sweep to a byte map, over drawn blocks and at the
edges."""
from __future__ import annotations

import subprocess
from pathlib import Path

DEV = Path(__file__).resolve().parent.parent / "hlr_amd" / "csrc" / "device"

PROGRAM = r"""
#include <cstdio>
#include <random>
#include "overlap.hpp"
using hmvm::Span;

static bool by_bytes(const std::vector<Span>& v) {
    for (size_t a = 0; a < v.size(); ++a)
        for (size_t b = a + 1; b < v.size(); ++b) {
            if (v[a].launch == v[b].launch || !(v[a].write || v[b].write)) continue;
            std::vector<char> map(8192, 0);
            for (int c = 0; c < v[a].cols; ++c)
                for (int64_t k = 0; k < v[a].col; ++k) map[v[a].p + c * v[a].ld + k] = 1;
            for (int c = 0; c < v[b].cols; ++c)
                for (int64_t k = 0; k < v[b].col; ++k)
                    if (map[v[b].p + c * v[b].ld + k]) return true;
        }
    return false;
}

static int check(const char* what, std::vector<Span> v, int want) {
    std::vector<Span> w = v;
    const bool got = hmvm::launches_conflict(w), ref = by_bytes(v);
    if (got != ref || (want >= 0 && got != bool(want))) { std::printf("%s: %d %d %d\n", what, got, ref, want); return 1; }
    return 0;
}

int main() {
    int bad = 0;
    bad += check("none", {}, 0);
    bad += check("same y, other launch", {{64, 80, 80, 1, 0, true}, {64, 80, 80, 3, 1, true}}, 1);
    bad += check("same y, same launch", {{64, 80, 80, 1, 1, true}, {64, 80, 80, 3, 1, true}}, 0);
    bad += check("two reads", {{64, 80, 80, 1, 0, false}, {64, 80, 80, 3, 1, false}}, 0);
    bad += check("column of the other", {{64 + 2 * 80, 80, 80, 1, 0, true}, {64, 80, 80, 3, 1, true}}, 1);
    bad += check("behind each other", {{64, 80, 80, 3, 1, true}, {64 + 240, 80, 80, 1, 0, true}}, 0);
    bad += check("one byte", {{64, 80, 80, 3, 1, true}, {64 + 239, 80, 80, 1, 0, true}}, 1);
    bad += check("rows of one array", {{64, 40, 80, 5, 1, true}, {64 + 40, 40, 80, 5, 2, true}}, 0);
    bad += check("rows that overlap", {{64, 48, 80, 5, 1, true}, {64 + 40, 40, 80, 5, 2, true}}, 1);
    bad += check("x of one right-hand side", {{64, 80, 80, 1, 0, false}, {100, 80, 80, 2, 1, true}}, 1);
    bad += check("empty", {{64, 0, 0, 1, 0, true}, {64, 80, 80, 2, 1, true}}, 0);
    std::mt19937 g(7);
    int seen[2] = {0, 0};
    for (int k = 0; k < 20000; ++k) {
        std::vector<Span> v;
        for (int n = 2 + int(g() % 5); n > 0; --n) {
            const int64_t col = 1 + g() % 60, ld = col + (g() % 2 ? g() % 90 : 0);
            v.push_back({g() % 4000, col, ld, 1 + int(g() % 8), int(g() % 3), g() % 2 == 0});
        }
        bad += check("drawn", v, -1);
        ++seen[by_bytes(v)];
        if (bad) break;
    }
    if (seen[0] < 1000 || seen[1] < 1000) { std::printf("draws %d %d\n", seen[0], seen[1]); return 1; }
    std::puts(bad ? "bad" : "ok");
    return bad;
}
"""


def test_sweep(tmp_path):
    src, exe = tmp_path / "overlap.cpp", tmp_path / "overlap"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{DEV}", str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout
