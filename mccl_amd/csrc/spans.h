// spans.h -- byte ranges as disjoint intervals, neighbours merged: what a run of operations has
// touched so far.  The tensors of a list are usually views that follow one another, and thousands
// of them make a handful of intervals.
#pragma once

#include <cstdint>
#include <iterator>
#include <map>

namespace mcclx {

class Spans {
public:
    // Does [lo, hi) share a byte with a range that was added?
    bool hits(uintptr_t lo, uintptr_t hi) const {
        auto it = spans_.upper_bound(lo);
        if (it != spans_.end() && it->first < hi) return true;
        return it != spans_.begin() && std::prev(it)->second > lo;
    }
    void insert(uintptr_t lo, uintptr_t hi) {  // what is added may overlap what is there
        auto it = spans_.upper_bound(lo);
        if (it != spans_.begin() && std::prev(it)->second >= lo) {
            if (it == spans_.end() || it->first > hi) {  // the range before grows, and meets no other
                uintptr_t& end = std::prev(it)->second;
                end = end > hi ? end : hi;
                return;
            }
            --it;
            lo = it->first;
        }
        while (it != spans_.end() && it->first <= hi) {
            hi = hi > it->second ? hi : it->second;
            it = spans_.erase(it);
        }
        spans_.emplace(lo, hi);
    }
    void clear() { spans_.clear(); }

    // The interval that `at` lies in, to grow without a search; valid until the next insert or clear.
    using Cursor = std::map<uintptr_t, uintptr_t>::iterator;
    Cursor cursor(uintptr_t at) { return std::prev(spans_.upper_bound(at)); }
    // Does [lo, hi) begin where that interval ends, and end in front of the next one?
    bool follows(Cursor c, uintptr_t lo, uintptr_t hi) const {
        const auto next = std::next(c);
        return c->second == lo && (next == spans_.end() || hi < next->first);
    }
    static void grow(Cursor c, uintptr_t hi) { c->second = hi; }

private:
    std::map<uintptr_t, uintptr_t> spans_;  // start -> end
};

}  // namespace mcclx
