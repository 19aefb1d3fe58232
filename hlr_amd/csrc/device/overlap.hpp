// overlap.hpp -- whether launches that run side by side touch the same memory.
#pragma once
#include <algorithm>
#include <cstdint>
#include <vector>

namespace hmvm {

// a column-major vector block of a launch
struct Span {
    uintptr_t p;
    int64_t col, ld;          // bytes of a column, from one column to the next (>= col)
    int cols;
    int launch;               // number of the launch that touches it
    bool write;
    uintptr_t end() const { return p + uintptr_t((cols - 1) * ld + col); }
};

// whether two blocks share a byte: their columns met in the order of their
// addresses
inline bool share_bytes(const Span& a, const Span& b) {
    uintptr_t pa = a.p, pb = b.p;
    for (int i = 0, j = 0; i < a.cols && j < b.cols;) {
        if (pa + uintptr_t(a.col) <= pb) { pa += uintptr_t(a.ld); ++i; }
        else if (pb + uintptr_t(b.col) <= pa) { pb += uintptr_t(b.ld); ++j; }
        else return true;
    }
    return false;
}

// whether launches of different numbers touch a byte that one of them writes
// (spans: reordered).  A sweep over the blocks by address; blocks of different
// addresses, the usual case, cost the sort alone.
inline bool launches_conflict(std::vector<Span>& spans) {
    spans.erase(std::remove_if(spans.begin(), spans.end(), [](const Span& s) { return s.cols < 1 || s.col < 1; }),
                spans.end());
    std::sort(spans.begin(), spans.end(), [](const Span& a, const Span& b) { return a.p < b.p; });
    std::vector<const Span*> open;
    for (const Span& s : spans) {
        open.erase(std::remove_if(open.begin(), open.end(), [&](const Span* o) { return o->end() <= s.p; }), open.end());
        for (const Span* o : open)
            if (o->launch != s.launch && (o->write || s.write) && share_bytes(*o, s)) return true;
        open.push_back(&s);
    }
    return false;
}

} // namespace hmvm
