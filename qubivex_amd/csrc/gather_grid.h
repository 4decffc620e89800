// The launch of a gather to f32: one-wave workgroups over the (item, tile) units of a batch
// (tests/test_gather_grid.py compiles this header for the host).
#pragma once
#include <algorithm>
#include <numeric>
#include <stdint.h>

#ifdef __HIPCC__
#define QVKV_HOST_DEVICE __host__ __device__
#else
#define QVKV_HOST_DEVICE
#endif

namespace qvkv {

struct GatherGrid {
    uint32_t wgs = 0;      // workgroups; 0: the launch is refused
    bool by_tile = false;  // units in order of tile, then item (else item, then tile)
    bool by_xcd = false;   // the pieces of a unit on one XCD (workgroups go to the 8 in turn)
};

// One-wave workgroups, each one batch of a tile's pieces at a time (per_tile of them share a
// tile), as for the block copy: many short workgroups keep the stores, most of the traffic, spread
// over time.  Against 256 threads x 8 pieces (a tile per workgroup), in us: q8_0 d = 128, 64 items
// of 1024-2048, 202 -> 184 (1.02 GB), d = 64 166 -> 105, f16 -> f32 225 -> 217.
// They walk the units (each_live_tile) where there are more than the grid.  held: the units with
// something in them, by the room for the output and by the tables.  An even batch takes a
// workgroup per piece of every unit, as many as a launch holds (at most 2^18 that walk, in us, 512
// of 2048, q8_0 d = 128 2054 -> 1934, d = 64 1245 -> 1080, f16 d = 128, 256 of 2048 1170 -> 1081).  An
// uneven one, with three times as many units as are held, would pay about 0.22 ns of dispatch over
// the chip for each that finds nothing to do: it takes a workgroup per held unit, at most 2^18,
// and walks tile by tile, which spreads the long items evenly.  In us, at 256 threads x 8 / one
// workgroup per piece of every unit / this, 8 KV heads, q8_0 d = 128, d = 64, f16 d = 128:
//   one item of 32 k beside 63 of 1 k    188 / 935 / 197, 192 / 477 / 118, 276 / 944 / 239
//   one of 32 k beside 255 of 64         251 / 3570 / 103, 364 / 1800 / 62, 680 / 3580 / 138
//   one of 4096 beside 15 of 64          17.6 / 31.1 / 13.2, 20.4 / 16.0 / 9.3, 19.8 / 35.1 / 17.3
//   32 of 256-4096                       155 / 150 / 147, 122 / 86 / 83, 179 / 173 / 177
// Large even q8_0 batches (one_xcd) write a unit's output from one XCD: 512 items of 2048, d = 128
// 2058 -> 1962, 128 of 2048 500 -> 493, d = 256 1268 -> 1080; 64 of 1024-2048 184 -> 189, so from 16384
// units on, and not at d = 64 (1083 -> 1120).
// A launch of more units than 2^32 threads hold at 256 each is refused.
inline GatherGrid gather_grid(uint64_t n_items, uint64_t tiles, uint64_t per_tile,
                              uint64_t out_positions, uint64_t n_table, uint64_t block,
                              bool one_xcd = false) {
    GatherGrid r;
    const uint64_t units = n_items * tiles;
    if (units * 256 > 0xffffffffull) return r;
    const uint64_t held = std::min(out_positions / 16, n_table * (block / 16)) + n_items;
    r.by_tile = units > 3 * held;
    uint64_t at_once = ((1ull << 26) - 1) / per_tile;  // 2^32 threads in all
    if (r.by_tile) at_once = std::min<uint64_t>((1ull << 18) / per_tile, held);
    at_once = std::max<uint64_t>(at_once, 1);
    // (a stride without a common factor with the inner count: the items of a tile, or the starts
    // of the items, then fall to different workgroups)
    if (units > at_once)
        while (std::gcd(at_once, r.by_tile ? n_items : tiles) != 1) at_once--;
    r.by_xcd = one_xcd && !r.by_tile && units >= 16384 && units + 7 <= at_once;
    r.wgs = (uint32_t)((r.by_xcd ? (units + 7) / 8 * 8 : std::min(units, at_once)) * per_tile);
    return r;
}

// The unit and piece of a workgroup (the first unit of its walk).
struct GatherPlace {
    uint32_t unit, part;
};
inline QVKV_HOST_DEVICE GatherPlace gather_place(uint32_t wg, uint32_t parts, bool by_xcd) {
    const uint32_t i = by_xcd ? wg / 8u : wg, q = i / parts;
    return GatherPlace{by_xcd ? q * 8u + wg % 8u : q, i - q * parts};
}

}  // namespace qvkv
