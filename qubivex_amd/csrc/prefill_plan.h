// The plan of a prefill launch (host code).
#pragma once

#include <algorithm>
#include <cstdint>

namespace qvkv {

// Workgroups per row block (64 query rows of a (segment, KV head)), and the workspace that a split
// launch (n_chunks > 1) keeps its partials in.  q8_0 launches may also keep images of their tiles
// there (img_segs segments at once, img_tiles each per KV head, img_bytes in all); the default
// plan needs no workspace.
constexpr uint32_t PREFILL_MAX_CHUNKS = 16;
constexpr uint64_t PREFILL_IMAGE_BYTES = 512ull << 20;
constexpr uint64_t PREFILL_IMAGE_TILE = 24832;  // bytes of an image: 32 positions of d = 128
struct PrefillPlan {
    uint32_t n_chunks = 1;
    uint32_t img_segs = 0, img_tiles = 0;
    uint64_t img_bytes = 0;
    uint64_t ws_bytes = 0;
};

struct PrefillShape {
    bool q8;               // the q8_0 form (d = 128), else f16 (d = 64 or 128)
    uint32_t G, D, GS;     // KV heads, head size, query heads per KV head
    uint32_t n_seg, max_pos, max_tok;
    int images, chunks;    // the knobs prefill_images, prefill_chunks
};

// The plan whose workspace is at most `limit` bytes.
//
// Chunks per row block: the count whose estimated time is least.  A CU holds 3
// workgroups (4 at d = 64); a 32-position tile takes a workgroup about `tile_us` with
// its CU full and down to 0.55-0.6 of that alone on it; each workgroup spends about
// 4 us outside its tiles, and a split launch 5 us more on its merge plus the partials'
// traffic (written and read once).  Measured at 2 k positions, f16, d = 128, in us by
// chunks 1 / 2 / 3 / 4 / 8: 32 row blocks 49 / 32 / 26 / 22 / 20, 128 blocks 51 / 36 /
// 33 / 31 / 41, 256 blocks 53 / 45 / 46 / 53 / 67, 512 blocks 65 / 83 / 81 / 92 / 134; a
// 512-token chunk at 8 k (256 blocks of 272 tiles) 188 -> 124 us with 3; d = 64, the same
// chunk by 1 / 2 / 3 / 4 / 6: 132 / 83 / 76 / 75 / 78.
//
// q8_0: tile images where enough row blocks share them (knob prefill_images: the least
// number), for as many segments at once as 512 MiB hold.  Measured at 2 k positions, 16
// segments, without / with images: 4 row blocks 143 / 150 us, 8 247 / 234, 16 427 / 388, 64 1839 /
// 1533; 4 segments at 8 k: 8 blocks 213 / 217, 32 794 / 685.  Contexts of fewer than 8 tiles do
// not pay for the extra launch: prompts of 180 tokens (12 row blocks, 6 tiles), 4 of them 18.4 / 19.6
// us, 16 37.8 / 41.5; of 256 tokens (8 tiles) 24.0 / 24.5, 55.4 / 54.7.  A limit below that makes passes of
// fewer segments only while each still fills the CUs: an underfilled pass costs more than the
// conversions that it shares.
inline PrefillPlan plan_prefill_shape(const PrefillShape &s, uint64_t limit) {
    PrefillPlan p;
    const uint64_t cus = 256, slots = (!s.q8 && s.D == 64 ? 4 : 3) * cus;
    const uint64_t n_qb = ((uint64_t)s.max_tok * s.GS + 63) / 64;
    const uint64_t tiles = ((uint64_t)s.max_pos + 32) / 32;
    const uint64_t seg_img = (uint64_t)s.G * tiles * PREFILL_IMAGE_TILE;
    uint64_t n_seg = s.n_seg;
    if (s.q8 && s.images > 0 && n_qb >= (uint64_t)s.images && (tiles >= 8 || s.images == 1) &&
        seg_img <= PREFILL_IMAGE_BYTES) {
        auto bytes = [&](uint64_t segs) { return (segs * seg_img + 255) / 256 * 256; };
        const uint64_t most = std::min<uint64_t>(PREFILL_IMAGE_BYTES / seg_img, s.n_seg);
        uint64_t fit = most;
        if (bytes(fit) > limit) {
            fit = limit / 256 * 256 / seg_img;
            if (fit * s.G * n_qb < slots) fit = 0;
        }
        if (fit > 0) {
            p.img_segs = (uint32_t)fit;
            p.img_tiles = (uint32_t)tiles;
            p.img_bytes = bytes(fit);
            n_seg = fit;
        }
    }
    const uint64_t blocks = n_seg * s.G * n_qb;
    auto partials = [&](uint32_t n) { return n > 1 ? blocks * n * 64ull * (s.D + 2) * 4ull : 0ull; };
    const double tile_us = s.q8 ? (p.img_segs ? 1.8 : 2.1) : s.D == 64 ? 0.84 : 1.14;
    double best = 0.0;
    for (uint32_t n = 1; n <= PREFILL_MAX_CHUNKS; n++) {
        if (n > 1 && (tiles < 2ull * n || blocks * n > 8 * slots) && s.chunks == 0) break;
        if (n > 1 && p.img_bytes + partials(n) > limit) break;
        const uint64_t per_cu = (blocks * n % slots + cus - 1) / cus;  // of the last round
        const double rounds = (double)(blocks * n / slots) +
                              (per_cu == 0 ? 0.0 : 0.4 + 0.6 * (double)(per_cu * cus) / (double)slots);
        double us = rounds * ((double)((tiles + n - 1) / n) * tile_us + 4.0);
        if (n > 1) us += 5.0 + (double)(blocks * n) * 64.0 * (s.D + 2) * 8.0 / 4e6;
        if (n == 1 || (s.chunks == 0 ? us < best : (int)n <= s.chunks)) {
            best = us;
            p.n_chunks = n;
        }
    }
    p.ws_bytes = p.img_bytes + partials(p.n_chunks);
    return p;
}

}  // namespace qvkv
