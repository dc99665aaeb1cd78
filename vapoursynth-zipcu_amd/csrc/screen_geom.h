// Geometry of the screened ssd search (k_match_screen, k_match_tied): region, norms and queue of one wave, their place in the
// LDS, and the addresses of its loads. Host code plans with it, the kernels walk by it, and a CPU check
// enumerates what they read.
#pragma once

namespace vszk {

constexpr int kScrCap = 16;    // keys kept per block between two insertions
constexpr int kScrLds8 = 20480;   // LDS bytes that each of 8 workgroups of a CU may take
constexpr int kScrLdsMax = 40960;  // a quarter of the CU's
constexpr int kScrStrides = 1 << 24;   // strides below it: the exact evaluation multiplies rows by the stride in 24 bits
constexpr int kScrRows = 28;   // region rows that a lane loads at a time, ScreenGeom::rstep apart

struct ScreenGeom {
    int ng, tiles;        // 4-row groups and 16-column tiles of a 4 x 4 block tile's candidates
    int pw, ph, nc, nr;   // half-pixel region (pitch, rows); norm array (pitch, rows)
    int queue;            // 8-byte results a wave can queue
    int slack;            // zeroed halves past the region: reads of masked columns in its last row end there
    int half_bytes, norm_bytes;
    // candidates that a wave evaluates as they come (usually 144 and up, below 200 on video with noise); where there are more, those
    // it evaluates for a block before it leaves the block (0: it leaves the tile at once)
    int most, block;
    // how 64 lanes walk the region's pairs and the norms' segments: i / d = i * m >> 16 below 4096
    int rstep, pair_m, segs, segs_m, vsegs, vsegs_m;
};

struct ScreenWave {  // per wave
    unsigned long long kbuf[16 * kScrCap];  // (distance, position) keys to insert, per block
    unsigned long long best[16 * 8];        // sorted keys of the best so far
    unsigned cnt[16];
    unsigned refpos[16];
    float th[16];                           // least result that passes in the second pass
    unsigned seen[16];                      // candidates evaluated while there were many
    unsigned zeros[4];                      // per block row, bit q: block q may have 8 distances of 0
};

// Bytes of the half region and of the norms (the last 8 rows of their first stage reach into the rest,
// which is not in use yet). Columns of the last tile past the norms' pitch belong to masked candidates and read
// the next row; after the last row, which is searched where 4 rows divide the window, they read
// values that the norms' two stages left there. What is kept behind must not be read as a norm: a mask cannot undo a NaN.
inline int screen_half_bytes(const ScreenGeom &G) { return ((G.pw * G.ph + G.slack) * 2 + 15) & ~15; }
inline int screen_norm_bytes(const ScreenGeom &G) {
    const int over = 16 * G.tiles > G.nc ? 16 * G.tiles - G.nc : 0;
    return ((G.nc * G.nr + over) * 4 + 15) & ~15;
}
inline int screen_lds_bytes(const ScreenGeom &G) {
    const int tail = 8 * G.nc * 4, rest = (int)sizeof(ScreenWave) + 8 * G.queue + 8;
    return screen_half_bytes(G) + screen_norm_bytes(G) + (tail > rest ? tail : rest);
}

inline ScreenGeom screen_geom(int bs, int R, int nt) {
    ScreenGeom G;
    const int span = 3 * bs + 2 * R + 1;
    G.ng = (span + 3) / 4;
    G.tiles = ((span + 15) / 16 + nt - 1) / nt * nt;
    G.pw = (span + 7 + 3) & ~3;   // columns past it belong to masked candidates only (they read on)
    G.nc = (span + 1) & ~1;
    if (G.nc % 16 == 0) G.nc += 2;   // rows of one column 12 apart in different banks
    G.nr = 4 * G.ng;
    G.ph = G.nr + 8;
    G.slack = (16 * G.tiles + 64 - G.pw + 7) / 8 * 8;
    G.slack = G.slack > 64 ? G.slack : 64;
    G.half_bytes = screen_half_bytes(G);
    G.norm_bytes = screen_norm_bytes(G);
    const auto magic = [](int d) { return (65536 + d - 1) / d; };
    G.rstep = G.pw / 2 <= 64 ? 64 / (G.pw / 2) : 1;
    G.pair_m = magic(G.pw / 2 <= 64 ? G.pw / 2 : 64);
    G.segs = (G.nc + 23) / 24;
    G.segs_m = magic(G.segs);
    G.vsegs = (G.nr + 11) / 12;
    G.vsegs_m = magic(G.vsegs);
    // the queue takes what is left of the LDS that lets 8 workgroups share a CU
    G.queue = 256;
    const int room = kScrLds8 - screen_lds_bytes(G);
    G.queue += (room < 0 ? 0 : room > 8 * 64 ? 8 * 64 : room) / 8;
    return G;
}

// A buffer load's byte offset: its range check covers `checked`; `added` (the scalar offset) is added past the
// check.
struct ScreenLoad {
    int checked, added;
};

// Where a lane finds the pixels k steps of `step` bytes below those at `at`. Rows past the region may lie past the
// plane, so all of it is checked: such loads return 0 and what they return is not used.
constexpr ScreenLoad screen_region_load(int at, int k, int step) {
    return ScreenLoad{(int)((unsigned)at + (unsigned)k * (unsigned)step), 0};
}

// Columns per product pass of the screened search: tiles of 16 in sets of two or three, whichever leaves
// fewer.
inline int screen_nt(int bs, int R) {
    return screen_geom(bs, R, 2).tiles < screen_geom(bs, R, 3).tiles ? 2 : 3;
}

// Which blocks a wave leaves to k_match_tied depends on what the search waits for. Up to 512 tiles leave most of the chip
// idle, so leaving a tile is quickest (640x360, block_step 8, bm_range 9, flat drawn art: 49 us, 77 with 24 and 90 with 96 for a
// block); up to 2048, all waves at once, the last wave counts (960x540, block_step 4, bm_range 12, art with noise: 384 and 24 take 94 us,
// 384 and 96 108); above, the work does (1920x1080, block_step 4, bm_range 12, text: 384 and 24 260 us, 1000 and 96 226; ordered
// dither at bm_range 16: 1080 and 248).
inline ScreenGeom screen_plan(int bs, int R, long long tiles) {
    ScreenGeom G = screen_geom(bs, R, screen_nt(bs, R));
    G.most = tiles <= 2048 ? 384 : 1000;
    G.block = tiles <= 512 ? 0 : tiles <= 2048 ? 24 : 96;
    return G;
}

// Candidates among the products' results.
inline float screen_share(const ScreenGeom &G, int R) {
    return (float)((2 * R + 1) * (2 * R + 1)) / (float)(4 * G.ng * 16 * G.tiles);
}

// Windows up to a quarter of a CU's LDS.
inline bool screen_fits(int bs, int R) { return R < 1024 && screen_lds_bytes(screen_geom(bs, R, screen_nt(bs, R))) <= kScrLdsMax; }

}  // namespace vszk
