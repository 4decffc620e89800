"""The prefill workspace's growth (qubivex_amd/csrc/workspace.h) and the plans that fit into it
(prefill_plan.h), compiled for the host with an allocator that refuses."""
import os
import subprocess

import pytest

HDR = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qubivex_amd", "csrc")

GROW = r"""
#include "workspace.h"
#include <stdio.h>
#include <stdlib.h>
#define CHECK(c) do { if (!(c)) { printf("FAIL line %d: %s\n", __LINE__, #c); exit(1); } } while (0)
using namespace qvkv;
static uint64_t room = ~0ull, held = 0, allocs = 0, tries = 0, retired = 0, frees = 0;
static void *alloc(uint64_t n) {
    tries++;
    if (held + n > room) return nullptr;
    held += n;
    allocs++;
    return malloc(1);
}
static void retire(void *p, uint64_t n) { held -= n; retired++; frees++; free(p); }
static bool ask(Workspace &w, uint64_t need) { return grow(w, need, 512ull << 20, frees, alloc, retire); }
int main() {
    const uint64_t M = 1 << 20;
    {   // a prompt's chunks, each needing a little more: few growths, at most twice the need
        Workspace w;
        for (uint64_t need = 20 * M; need <= 500 * M; need += 5 * M) {
            CHECK(ask(w, need) && w.bytes >= need && w.bytes <= 2 * need);
        }
        CHECK(allocs <= 6 && retired == allocs - 1 && held == w.bytes);
        CHECK(ask(w, 700 * M) && w.bytes == 700 * M);  // above the cap: what is asked for
        retire(w.p, w.bytes);
    }
    {   // a full device: the buffer at hand stays, and a refused size is not tried each time
        Workspace w;
        CHECK(ask(w, 100 * M));
        const void *p = w.p;
        room = held + 50 * M;
        tries = retired = 0;
        for (int i = 0; i < 1000; i++) CHECK(!ask(w, 300 * M) && w.p == p && w.bytes == 100 * M);
        CHECK(tries <= 2 && retired == 0);
        for (int i = 0; i < 1000; i++) CHECK(ask(w, 100 * M) && !ask(w, 400 * M));  // small and large in turn
        CHECK(tries <= 4 && retired == 0);
        CHECK(!ask(w, 150 * M) && w.p == p);      // less than was refused: tried, refused too
        room = ~0ull;
        frees++;                                  // the library gave memory back: tried at once
        CHECK(ask(w, 150 * M) && w.p != p && w.bytes >= 150 * M && retired == 1);
        retire(w.p, w.bytes);
    }
    {   // memory freed elsewhere is found again after some launches
        Workspace w;
        room = held + 10 * M;
        CHECK(!ask(w, 64 * M) && !w.p);
        room = ~0ull;
        uint32_t n = 0;
        while (!ask(w, 64 * M)) CHECK(++n <= WORKSPACE_RETRY);
        CHECK(n >= WORKSPACE_RETRY / 2);
        retire(w.p, w.bytes);
    }
    {   // doubling that does not fit falls back to the need itself
        Workspace w;
        CHECK(ask(w, 100 * M));
        room = held + 130 * M;
        CHECK(ask(w, 120 * M) && w.bytes == 120 * M && held == 120 * M);
    }
    printf("OK\n");
}
"""

PLAN = r"""
#include "prefill_plan.h"
#include <stdio.h>
#include <stdlib.h>
#include <random>
#define CHECK(c) do { if (!(c)) { printf("FAIL line %d: %s\n", __LINE__, #c); exit(1); } } while (0)
using namespace qvkv;
int main() {
    std::mt19937 r(7);
    auto pick = [&](uint32_t lo, uint32_t hi) { return lo + r() % (hi - lo + 1); };
    for (int i = 0; i < 20000; i++) {
        const bool q8 = r() & 1;
        const uint32_t max_tok = pick(1, 1 << pick(0, 10));
        const PrefillShape s{q8, pick(1, 8), q8 || (r() & 1) ? 128u : 64u, pick(1, 16), pick(1, 40),
                             max_tok + pick(0, 1 << pick(0, 15)), max_tok, r() & 1 ? 12 : 0, r() % 4 ? 0 : (int)pick(1, 16)};
        const PrefillPlan all = plan_prefill_shape(s, ~0ull);
        const uint64_t limit = r() % 3 ? all.ws_bytes * pick(0, 110) / 100 : pick(0, 1 << 30);
        const PrefillPlan p = plan_prefill_shape(s, limit);
        CHECK(p.ws_bytes <= limit && p.n_chunks >= 1 && p.n_chunks <= PREFILL_MAX_CHUNKS);
        CHECK(p.img_bytes == (p.img_segs * (uint64_t)s.G * p.img_tiles * PREFILL_IMAGE_TILE + 255) / 256 * 256);
        if (all.ws_bytes <= limit)
            CHECK(p.ws_bytes == all.ws_bytes && p.n_chunks == all.n_chunks && p.img_segs == all.img_segs);
        if (limit == 0) CHECK(p.n_chunks == 1 && p.img_segs == 0);
    }
    // 16 chunks of 512 tokens at 2 k, 8 KV heads, 4 query heads each: all images in 203 MB; half of
    // that takes fewer segments at once, a little takes none
    const PrefillShape b{true, 8, 128, 4, 16, 2046, 512, 12, 0};
    CHECK(plan_prefill_shape(b, ~0ull).img_segs == 16);
    CHECK(plan_prefill_shape(b, 100ull << 20).img_segs == 8);
    CHECK(plan_prefill_shape(b, 30ull << 20).img_segs == 0);
    // short contexts take none, unless always asked for
    PrefillShape c{true, 8, 128, 4, 16, 179, 180, 12, 0};
    CHECK(plan_prefill_shape(c, ~0ull).img_segs == 0);
    c.images = 1;
    CHECK(plan_prefill_shape(c, ~0ull).img_segs == 16);
    // one chunk at 8 k: without room for images the split is kept
    const PrefillShape one{true, 4, 128, 8, 1, 8703, 512, 12, 0};
    const PrefillPlan p = plan_prefill_shape(one, 20ull << 20);
    CHECK(plan_prefill_shape(one, ~0ull).img_segs == 1 && p.img_segs == 0 && p.n_chunks > 1);
    printf("OK\n");
}
"""


@pytest.mark.parametrize("prog", [GROW, PLAN], ids=["grow", "plan"])
def test_workspace(tmp_path, prog):
    src, exe = tmp_path / "ws.cpp", tmp_path / "ws"
    src.write_text(prog)
    try:
        subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I", HDR, str(src), "-o", str(exe)], check=True,
                       capture_output=True, text=True)
    except FileNotFoundError:
        pytest.skip("g++ is not available")
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "OK", r.stdout
