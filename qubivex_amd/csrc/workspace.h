// A device buffer that grows with what its launches ask for (host code; no HIP here, so that its
// rules can be tested with any allocator).
#pragma once

#include <algorithm>
#include <cstdint>

namespace qvkv {

struct Workspace {
    void *p = nullptr;
    uint64_t bytes = 0;
    uint64_t refused = ~0ull;  // the least size that the device had no memory for
    uint64_t frees = 0;        // the device's count of frees at that refusal
    uint32_t skipped = 0;      // launches since that did without
};

// Launches that do without before a refused size is tried again: memory freed outside this
// library is not seen here, and a failing allocation per launch would cost more than the launch.
constexpr uint32_t WORKSPACE_RETRY = 1024;

// Makes `w` hold at least `need` bytes (contents not kept), or leaves it as it is and returns
// false.  It grows by doubling up to `cap`, so that launches which each need a little more than
// the last (a prompt's chunks) drain the stream a few times in all and not once each.
//   alloc(bytes): a new buffer, or null;  retire(p, bytes): frees the outgrown one once no
//   launch reads it;  frees: how many buffers the device's handle has given back so far.
// The old buffer goes only after the new one exists.
template <class Alloc, class Retire>
bool grow(Workspace &w, uint64_t need, uint64_t cap, uint64_t frees, Alloc alloc, Retire retire) {
    if (w.bytes >= need) return true;
    if (need >= w.refused) {
        if (frees == w.frees && ++w.skipped < WORKSPACE_RETRY) return false;
        w.refused = ~0ull;
    }
    auto whole = [](uint64_t n) -> uint64_t { return (std::max<uint64_t>(n, 1 << 20) + 4095) & ~4095ull; };
    const uint64_t least = whole(need), most = std::max(least, whole(std::min(2 * w.bytes, cap)));
    uint64_t got = most;
    void *p = alloc(got);
    if (!p && least < most) p = alloc(got = least);
    if (!p) {
        w.refused = need;
        w.frees = frees;
        w.skipped = 0;
        return false;
    }
    if (w.p) retire(w.p, w.bytes);
    w = Workspace{p, got};
    return true;
}

}  // namespace qvkv
