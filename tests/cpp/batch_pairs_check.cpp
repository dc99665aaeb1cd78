// CPU check of the pairs that a batch's autotuner times (csrc/batch_pairs.h), over everything a batch can allow.
#include <cstdio>
#include <set>
#include <utility>

#include "batch_pairs.h"

using namespace vszk;

int main() {
    for (int bits = 0; bits < 32; ++bits)
        for (int asked : {VSZ_BATCH_STAGED, VSZ_BATCH_PERSISTENT, VSZ_BATCH_AUTO}) {
            const bool rows = bits & 1, sc = bits & 2, global = bits & 4, screen = bits & 8, pers = bits & 16;
            if (global ? (rows || sc || screen || pers) : !rows && !sc) continue;   // global: no other form fits
            if (asked == VSZ_BATCH_PERSISTENT && !pers) continue;                      // refused at creation
            const auto pairs = batch_pairs(asked, rows, sc, global, screen, pers);
            std::set<std::pair<int, int>> launches;   // what a run launches: the screened search has no matcher beside it
            int screens = 0;
            for (const BatchPair &p : pairs) {
                const bool fits = global || (p.shared_cols ? sc : rows || p.screen);
                if (!fits || (p.schedule == VSZ_BATCH_PERSISTENT && (!pers || p.screen || asked == VSZ_BATCH_STAGED)) ||
                    (p.schedule == VSZ_BATCH_STAGED && asked == VSZ_BATCH_PERSISTENT)) {
                    std::printf("pair not allowed: flags %d asked %d\n", bits, asked);
                    return 1;
                }
                screens += p.screen;
                if (!launches.insert({p.schedule, p.screen ? 2 : p.shared_cols}).second) {
                    std::printf("one launch timed twice: flags %d asked %d\n", bits, asked);
                    return 1;
                }
            }
            const bool staged = asked != VSZ_BATCH_PERSISTENT;
            int exhaustive = 0;
            for (const BatchPair &p : pairs) exhaustive += p.schedule == VSZ_BATCH_STAGED && !p.screen;
            if (pairs.empty() || pairs.size() > 4 || screens != (screen && staged) || (staged && !exhaustive)) {
                std::printf("%zu pairs, %d screened, %d staged without: flags %d asked %d\n", pairs.size(), screens, exhaustive, bits, asked);
                return 1;
            }
            const BatchPair p = batch_preferred(pairs, asked);
            if (p.screen != (screen && staged) || p.shared_cols != sc || p.schedule != (staged ? VSZ_BATCH_STAGED : VSZ_BATCH_PERSISTENT)) {
                std::printf("preference: flags %d asked %d\n", bits, asked);
                return 1;
            }
        }
    std::printf("batch pairs: ok\n");
    return 0;
}
