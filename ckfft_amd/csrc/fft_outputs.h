// fft_outputs.h -- outputs in memory that other transforms write too (host side).
//
// A transform above one workgroup's size keeps its intermediate in its output, so nothing else may
// write there while it runs, not even another run of the same transform, which would store the
// same values in the end.  Transforms that the library itself lets run side by side (one plan's,
// one server's) may share outputs all the same; these helpers find the ones that then need an order.
#pragma once
#include <algorithm>
#include <cstdint>
#include <vector>

namespace ckfft_gpu {

struct OutputRange {
    uintptr_t begin, end;
};

// For each of `held`, whether it shares a byte with another one of them or with one of `others`.
inline std::vector<char> shared_outputs(const std::vector<OutputRange>& held, const std::vector<OutputRange>& others)
{
    const size_t n = held.size();
    std::vector<char> shared(n, 0);
    std::vector<size_t> order(n);
    for (size_t i = 0; i < n; ++i) order[i] = i;
    std::sort(order.begin(), order.end(), [&](size_t a, size_t b) { return held[a].begin < held[b].begin; });
    uintptr_t reach = 0;   // the greatest end so far
    for (size_t i = 0; i < n; ++i) {
        const OutputRange& r = held[order[i]];
        if (reach > r.begin || (i + 1 < n && held[order[i + 1]].begin < r.end)) shared[order[i]] = 1;
        reach = std::max(reach, r.end);
    }
    // those left do not overlap, so their ends rise like their begins
    std::vector<size_t> alone;
    for (size_t i : order)
        if (!shared[i]) alone.push_back(i);
    for (const OutputRange& o : others)
        for (auto it = std::partition_point(alone.begin(), alone.end(), [&](size_t i) { return held[i].end <= o.begin; });
             it != alone.end() && held[*it].begin < o.end; ++it)
            shared[*it] = 1;
    return shared;
}

// The outputs of one batch in flight.
class BatchOutputs {
public:
    void clear()
    {
        all_.clear();
        held_.clear();
        sorted_ = false;
    }
    // holds: the transform keeps its intermediate there.
    void add(OutputRange r, bool holds)
    {
        all_.push_back(r);
        if (holds) held_.push_back(r);
    }
    // Whether a transform of one batch writes where one of the other keeps its intermediate.
    static bool conflict(BatchOutputs& a, BatchOutputs& b) { return a.hit_by(b.held_) || b.hit_by(a.held_); }

private:
    bool hit_by(const std::vector<OutputRange>& held)
    {
        if (held.empty() || all_.empty()) return false;
        if (!sorted_) {   // only batches beside multi-pass transforms get here
            std::sort(all_.begin(), all_.end(), [](const OutputRange& x, const OutputRange& y) { return x.begin < y.begin; });
            reach_.resize(all_.size());
            uintptr_t reach = 0;
            for (size_t i = 0; i < all_.size(); ++i) reach_[i] = reach = std::max(reach, all_[i].end);
            sorted_ = true;
        }
        for (const OutputRange& r : held) {
            const auto it = std::partition_point(all_.begin(), all_.end(), [&](const OutputRange& x) { return x.begin < r.end; });
            if (it != all_.begin() && reach_[it - all_.begin() - 1] > r.begin) return true;
        }
        return false;
    }

    std::vector<OutputRange> all_, held_;
    std::vector<uintptr_t> reach_;   // the greatest end among all_[0 .. i], once sorted
    bool sorted_ = false;
};

}  // namespace ckfft_gpu
