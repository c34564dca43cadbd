// How the merged adapter refresh cuts its members into workgroups: host arithmetic only, so that it
// compiles (and is checked) without a GPU.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

namespace sa3k {

constexpr int kMergeRows = 64;   // rows of a member a merge block takes
struct RefreshMember {
    int64_t in, out;
};

// Column splits of a member's 64-row blocks, by the 64 x 64 chunks of the whole refresh: a workgroup
// walks its chunks one after another, about 1.3 us each (a memory round trip and two barriers), so
// below a chip full of workgroups (four per CU) the time is that walk's length. A group that fills
// the chip by its rows alone is not split; at least kMergeMinChunks chunks stay with a workgroup.
// Measured on MI355X, whole refresh unsplit -> split, us: a 1536-wide block's seven linears (one
// launch) dora r32 117 -> 68, lora r16 111 -> 56; one linear, dora r32: 1536 x 6144 Q8_0 38 -> 21,
// 1536 x 9216 f16 34 -> 23, 6144 x 1536 f16 107 -> 20. Slots 768 / 2048 and minima of 6 / 8 chunks
// were within 5% or slower.
constexpr int kMergeSlots = 1024, kMergeMinChunks = 4;
inline int merge_splits(int64_t chunks, int64_t in) {
    const int64_t nc = in / 64, per = std::max<int64_t>(kMergeMinChunks, (chunks + kMergeSlots - 1) / kMergeSlots);
    const int64_t s = (nc + per - 1) / per, each = (nc + s - 1) / s;
    return (int)((nc + each - 1) / each);   // no split without chunks
}

// The splits of every member. dora's splits meet at an arrival counter per merge block; with more
// blocks than `counters` nothing is split (a split is only for speed). lora's need none.
inline std::vector<int> refresh_splits(const std::vector<RefreshMember>& m, bool dora, int64_t counters) {
    int64_t chunks = 0, blocks = 0;
    for (const RefreshMember& q : m) chunks += (q.out + kMergeRows - 1) / kMergeRows * (q.in / 64);
    std::vector<int> s;
    for (const RefreshMember& q : m) {
        s.push_back(merge_splits(chunks, q.in));
        blocks += (q.out + kMergeRows - 1) / kMergeRows * s.back();
    }
    if (dora && blocks > counters) s.assign(m.size(), 1);
    return s;
}

}  // namespace sa3k
