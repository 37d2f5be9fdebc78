// How the brute-force kernels divide their sums: plain host code, so that it can be checked without a GPU.
#pragma once

#include <cstddef>
#include <cstdint>

namespace pnb {

constexpr int BF_BLOCK = 256;
constexpr int BF_TILE = 256;
constexpr int COOP_WAVES = 16;
constexpr int BF64_WAVES = 8;

inline size_t ceil_div(size_t a, size_t b) { return (a + b - 1) / b; }

constexpr int BF_COOP = 2;  // variant of the workgroup-cooperative kernel (not for tuning entries)

// A dispatch holds fewer than 2^32 work-items along x. The FP64 kernel takes 8 per affected body (2^31 for
// this many), the cooperative kernel 16, but of fewer bodies (coop_pays); the plain kernel at most one.
constexpr size_t BF64_SLICE = size_t(1) << 28;

struct BfShape {
    int variant, per_lane, j_split;
};

// What the cooperative kernel takes: sums too small for one wavefront per affected tile and range to
// fill the chip evenly. Measured, plain kernel with its best split / cooperative (us, softened): 1,000
// x 1,000 62 / 8; 4,096 x 4,096 36 / 10; 10,000 x 8,000 45 / 30; 20,000 x 20,000 142 / 122; 30,000 x
// 65,536 628 / 568; 45,000 x 130,000 1,695 / 1,659, without softening 1,861 / 1,862; 65,536 x 16,384
// 321 / 308; 90,000 x 30,000 781 / 775, 864 / 868; 130,000 x 4,000 163 / 160; 130,000 x 30,000 1,098 /
// 1,116. Below 2,048 affecting bodies the plain kernel does not split, and leaves SIMDs idle up to some
// 800,000 affected ones; the cooperative one has at most 16 tiles of 64 to share, and fewer than eight
// leave half of its wavefronts without one:
//   affected   x 257        300        400        450        512        700        1,000      2,047
//   200,000    24.6 / 24.0  27.7/26.1  34.7/31.1  38.4/31.5  46.6/32.6  59.9/43.3  85.4/58.5  175 / 115
//   262,144    25.4 / 29.4  28.5/31.8  35.5/37.9  39.0/38.2  48.2/39.8  61.1/52.8  87.4/71.3  179 / 142
//   400,000    37.4 / 43.8  42.2/48.0  54.3/57.3  61.1/58.2  70.4/60.7  93.9/80.5  133 / 109  276 / 218
//   600,000    49.4 / 63.8  56.1/69.7  72.8/83.5  81.8/84.8  93.7/88.6  125 / 118  180 / 161  369 / 322
//   1,048,576  73.9 / 109   84.3/119   110 / 142  126 / 145  142 / 151  191 / 202  273 / 275  560 / 554
//   4,194,304  269 / 424    313 / 465  413 / 558  468 / 571  521 / 596  722 / 791  1,024/1,092 2,082/2,196
// (without softening the same to 5 %). With few affecting bodies there is little to share: 256 x 100
// 6.0 / 8.8, 256 x 128 6.9 / 7.6, 256 x 200 9.8 / 8.7; 65,536 x 200 8.9 / 8.7, 90,000 x 200 11 / 13.
inline bool coop_pays(size_t n, size_t m) {
    if (m <= 256) return m > 128 && n <= 65536;
    if (m < 2048) return n <= 200000 || (n < 800000 && m > 448);
    return n <= 50000 || (n <= 100000 && m <= 16384) || (n <= 150000 && m <= 4096);
}

inline BfShape default_shape(size_t cus, size_t n, size_t m) {
    int s = 1;
    if (coop_pays(n, m)) {
        // Workgroups of 16 wavefronts over ranges of the affecting bodies: two per CU while a range
        // keeps 500 of them, which is half a tile for each wavefront, and up to 16 per CU, so that
        // no CU has twice another's work, while it keeps 700. 9,000 x 9,000 in 1 / 2 / 4 / 8 / 16
        // ranges 50 / 54 / 40 / 32 / 32 us; 6,000 x 6,000 33 / 22 / 21 / 16 / 20; 1,000 x 8,000 41 /
        // 25 / 16 / 10 / 8; 20,000 x 20,000 186 / 145 / 126 / 122 / 124.
        const size_t blocks = ceil_div(n, 64);
        while (m >= 2048 && s < 64) {
            const size_t wgs = blocks * s * 2, per = m / (size_t(s) * 2);
            if (!((wgs <= 2 * cus && per >= 500) || (wgs <= 16 * cus && per >= 700))) break;
            s <<= 1;
        }
        return {BF_COOP, 1, s};
    }
    // Otherwise one body per lane and one wavefront per affected tile and range, the affecting bodies
    // from scalar loads, or from LDS for a few of them and wavefronts too few to hide the loads (us,
    // LDS / scalar: 100,000 x 200 10.6 / 10.8, 262,144 x 256 25.2 / 27.1, 400,000 x 256 36.9 / 37.0,
    // 600,000 x 256 49.4 / 48.6, 4,194,304 x 64 79.5 / 76.2). The affecting
    // range is split from 2,048 bodies on into up to 64 workgroups per CU of at least one tile each, up
    // to 256 per CU while ranges stay at 1,024 bodies (small workgroups balance the load across CUs
    // and XCDs). 1,048,576 x 65,536 16.1 ms, with four bodies per lane 17.1.
    const size_t blocks = ceil_div(n, size_t(BF_BLOCK));
    while (m >= 2048 && s < 64 && blocks * s * 2 <= 256 * cus) {
        const size_t per = m / (size_t(s) * 2);
        if (per < (blocks * s * 2 <= 64 * cus ? size_t(BF_TILE) : size_t(1024))) break;
        s <<= 1;
    }
    return {m <= 448 && n < 400000 ? 0 : 1, 1, s};
}

struct BfPlan {
    BfShape shape;
    uint32_t splits, chunk;
    int tile;
};

// Splits of the affecting range in whole tiles. The cooperative kernel takes smaller tiles for
// small ranges, so that all its wavefronts get one.
inline BfPlan plan_for(const BfShape& sh, size_t m) {
    uint32_t splits = uint32_t(sh.j_split);
    const size_t per = m / splits / COOP_WAVES;
    const int tile = sh.variant != BF_COOP || per >= 256 ? BF_TILE : per >= 128 ? 128 : 64;
    uint32_t chunk = uint32_t(ceil_div(m, splits));
    chunk = (chunk + tile - 1) / tile * tile;
    splits = uint32_t(ceil_div(m, chunk));
    return {sh, splits, chunk, tile};
}

// Work-items per workgroup and workgroups along x (affected bodies); y counts the affecting ranges.
inline unsigned bf_block(const BfShape& sh) { return sh.variant == BF_COOP ? 64 * COOP_WAVES : BF_BLOCK; }
inline unsigned bf_grid_x(const BfShape& sh, size_t n) {
    return unsigned(ceil_div(n, sh.variant == BF_COOP ? size_t(64) : size_t(BF_BLOCK) * sh.per_lane));
}

// The FP64 sum: wavefronts per 64 affected bodies, and affecting ranges: workgroups until the launch holds
// about four rounds of wavefronts (32 per CU), with at least 32 affecting bodies for each of a
// workgroup's wavefronts. Up to eight affecting bodies one wavefront takes all: split, each has one or
// none (1,000,000 x 1 15.9 us, 10.9 so; x 8 20.4, 11.9), and adding one after the other rounds less often.
struct Bf64Plan {
    int waves;
    size_t splits;
    uint32_t chunk;
};

inline Bf64Plan plan64(size_t cus, size_t n, size_t m) {
    if (m <= BF64_WAVES) return {1, 1, m > 0 ? uint32_t(m) : 1};
    const size_t blocks = ceil_div(n, 64);
    size_t splits = 1;
    while (splits < 64 && blocks * splits * BF64_WAVES < 128 * cus && m / (splits * 2) >= 32 * BF64_WAVES)
        splits <<= 1;
    const size_t chunk = ceil_div(m, splits);
    return {BF64_WAVES, ceil_div(m, chunk), uint32_t(chunk)};
}

}  // namespace pnb
