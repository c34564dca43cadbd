// C entry points over the host-only column splits of the merged adapter refresh, for the CPU tests.
#include "refresh_plan.h"

extern "C" {

// shapes: in, out per member; splits: out, per member; returns the merge blocks
int64_t refresh(const int64_t* shapes, int n, int dora, int64_t counters, int* splits) {
    std::vector<sa3k::RefreshMember> m;
    for (int i = 0; i < n; ++i) m.push_back({shapes[2 * i], shapes[2 * i + 1]});
    const std::vector<int> s = sa3k::refresh_splits(m, dora != 0, counters);
    int64_t blocks = 0;
    for (int i = 0; i < n; ++i) {
        splits[i] = s[i];
        blocks += (m[i].out + sa3k::kMergeRows - 1) / sa3k::kMergeRows * s[i];
    }
    return blocks;
}
}
