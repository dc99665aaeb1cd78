// The (schedule, search) pairs that a batch may run with: what the autotuner times, and what is taken without it.
#pragma once

#include <vector>

#include "vszipcu_bm3d.h"

namespace vszk {

struct BatchPair {
    int schedule;      // VSZ_BATCH_STAGED or VSZ_BATCH_PERSISTENT
    bool shared_cols;  // the shared-column matcher, else the row matcher (or the global-memory one)
    bool screen;       // the screened search in its place (staged only)
};

// `asked`: the schedule asked for; which matchers, the screened search (by its rule) and the persistent launch the batch
// allows. Each pair is another launch. Where the screened search may run, it is timed with the staged schedule beside one
// exhaustive matcher, so that content whose windows tie can do without it.
inline std::vector<BatchPair> batch_pairs(int asked, bool rows, bool shared_cols, bool global, bool screen, bool persistent) {
    std::vector<BatchPair> p;
    if (global) {  // the only form for such windows
        p.push_back({VSZ_BATCH_STAGED, false, false});
        return p;
    }
    if (screen && asked != VSZ_BATCH_PERSISTENT) p.push_back({VSZ_BATCH_STAGED, shared_cols, true});
    for (int sc = 1; sc >= 0; --sc) {
        if (sc ? !shared_cols : !rows) continue;
        if (asked != VSZ_BATCH_STAGED && persistent) p.push_back({VSZ_BATCH_PERSISTENT, sc != 0, false});
        if (asked != VSZ_BATCH_PERSISTENT && !(screen && shared_cols && !sc)) p.push_back({VSZ_BATCH_STAGED, sc != 0, false});
    }
    return p;
}

// Without timing: the screened search, then the shared-column matcher; the persistent launch only where asked for.
inline BatchPair batch_preferred(const std::vector<BatchPair> &pairs, int asked) {
    const int want = asked == VSZ_BATCH_PERSISTENT ? VSZ_BATCH_PERSISTENT : VSZ_BATCH_STAGED;
    for (const BatchPair &p : pairs)
        if (p.schedule == want) return p;
    return pairs[0];
}

}  // namespace vszk
