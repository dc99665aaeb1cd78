// CPU check of the screened search's geometry (csrc/screen_geom.h), over every block step and window it takes: what
// a wave reads of the plane, walked as k_match_screen walks it.
#include <cstddef>
#include <cstdio>

#include "screen_geom.h"

using namespace vszk;

// The region of a tile at the plane's lower right corner: every load is in the plane or caught by the range check.
static bool region_loads(int bs, int R, const ScreenGeom &G) {
    const int H = G.ph + 3, W = G.pw + 5, S = W + 7;
    const unsigned bytes = 4u * (unsigned)(S * H);
    const int rx0 = W - G.pw, ry0 = H - G.ph, p2 = G.pw >> 1, step = G.rstep * S * 4;
    for (int lane = 0; lane < 64; ++lane) {
        const int srow = lane * G.pair_m >> 16, spair = lane - srow * p2;
        if (spair < 0) return false;
        for (int pr = spair; pr < p2; pr += 64)
            for (int r = srow; r < (srow < G.rstep ? G.ph : 0); r += kScrRows * G.rstep)
                for (int k = 0; k < kScrRows; ++k) {
                    const ScreenLoad ld = screen_region_load(((ry0 + r) * S + rx0 + 2 * pr) * 4, k, step);
                    const unsigned at = (unsigned)ld.checked, end = at + (unsigned)ld.added + 8;
                    if (at < bytes && end > bytes) {   // passes the check, but ends past the plane
                        std::printf("block_step %d bm_range %d: lane %d row %d + %d steps reads %u bytes past the plane\n", bs, R,
                                    lane, r, k, end - bytes);
                        return false;
                    }
                    if (r + k * G.rstep < G.ph && end > bytes) return false;   // a pixel that is used
                }
    }
    return true;
}

// The norms that rows of the search read: all of them before the keys kept behind the norms, and past the norms' rows
// only what their first stage wrote (the sums of the 8 region rows below).
static bool norm_reads(int bs, int R, const ScreenGeom &G) {
    const int span = 3 * bs + 2 * R + 1;
    for (int row = 0; row < span; ++row) {
        const int last = row * G.nc + 16 * G.tiles - 1;
        if (4 * (last + 1) > G.norm_bytes || last >= G.nc * (G.nr + 8)) {
            std::printf("block_step %d bm_range %d: row %d reads norm %d of %d bytes\n", bs, R, row, last, G.norm_bytes);
            return false;
        }
    }
    // ... which ends before what the wave keeps there from its start
    return G.norm_bytes + (int)offsetof(ScreenWave, cnt) >= 4 * G.nc * (G.nr + 8);
}

int main() {
    int n = 0;
    for (int bs = 1; bs <= 8; ++bs)
        for (int R = 1; screen_fits(bs, R); ++R, ++n) {
            const ScreenGeom G = screen_plan(bs, R, 1);
            if (!region_loads(bs, R, G) || !norm_reads(bs, R, G)) return 1;
        }
    std::printf("screen geometry: ok, %d plans\n", n);
    return 0;
}
