"""The order of launches on side streams (csrc/device/fork.hpp), with every
runtime call failing in turn: a host program runs the fork over a runtime that
keeps each stream's queue, and checks that every launch sees begin() done and
that what follows end() sees every launch done."""
from __future__ import annotations

import subprocess
from pathlib import Path


DEV = Path(__file__).resolve().parent.parent / "hlr_amd" / "csrc" / "device"

PROGRAM = r"""
#include <cstdio>
#include <set>
#include <vector>
#include "fork.hpp"

// A stream holds the set of marks that its next entry is ordered behind; an
// event a copy of such a set.  Call `fail` (counted from 0) fails.
struct World {
    std::set<int> stream[8], event[8];
    int calls = 0, fail = -1, fails = 0;
    bool refuse() { if (calls++ != fail) return false; ++fails; return true; }
};
struct Order {
    World* w;
    bool record(int e, int s) const { if (w->refuse()) return false; w->event[e] = w->stream[s]; return true; }
    bool wait(int s, int e) const {
        if (w->refuse()) return false;
        w->stream[s].insert(w->event[e].begin(), w->event[e].end());
        return true;
    }
    // the host waits: everything of the stream is done before later calls
    bool finish(int s) const {
        for (auto& t : w->stream) t.insert(w->stream[s].begin(), w->stream[s].end());
        return true;
    }
};

int main() {
    constexpr int N = 3;
    const int side[N] = {1, 2, 3}, join[N] = {1, 2, 3};
    for (int launches = 0; launches <= 9; ++launches)
        for (int fail = -1; fail < 40; ++fail) {
            World w;
            w.fail = fail;
            hmvm::Fork<N, Order, int, int> f(Order{&w}, 0, side, 0, join);
            int mark = 0;
            std::set<int> all;
            for (int stage = 0; stage < 2; ++stage) {
                w.stream[0].insert(++mark);              // the caller's work so far
                all.insert(mark);
                const std::set<int> before = all;
                f.begin(launches);
                std::set<int> streams;
                for (int k = 0; k < launches; ++k) {
                    const int s = f.next();
                    streams.insert(s);
                    for (int m : before)
                        if (!w.stream[s].count(m)) { std::printf("launch before the fork: %d %d\n", launches, fail); return 1; }
                    w.stream[s].insert(++mark);
                    all.insert(mark);
                }
                f.end();
                for (int m : all)
                    if (!w.stream[0].count(m)) { std::printf("not joined: %d %d\n", launches, fail); return 1; }
                // no failure: the launches do spread
                if (fail < 0 && launches > 1 && int(streams.size()) != (launches < N + 1 ? launches : N + 1)) {
                    std::printf("spread: %d\n", launches);
                    return 1;
                }
            }
            if (f.failed() != (w.fails > 0)) { std::printf("failed(): %d %d\n", launches, fail); return 1; }
        }
    std::puts("ok");
    return 0;
}
"""


def test_order_under_failures(tmp_path):
    src, exe = tmp_path / "fork.cpp", tmp_path / "fork"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{DEV}", str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout
