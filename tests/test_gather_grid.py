"""The grid of a gather to f32 (qubivex_amd/csrc/gather_grid.h), compiled for the host: every unit is
taken once, the workgroups are bounded whatever the batch, and a launch too large is refused."""
import os
import subprocess

import pytest

HDR = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qubivex_amd", "csrc")

PROG = r"""
#include "gather_grid.h"
#include <stdio.h>
#include <vector>
static int bad(const char *what, unsigned long long a, unsigned long long b) {
    printf("FAIL %s %llu %llu\n", what, a, b);
    return 1;
}
// the walk of each_live_tile by the workgroups of one piece
static int covers(uint64_t items, uint64_t tiles, uint64_t per_tile, uint64_t positions, bool one_xcd) {
    const qvkv::GatherGrid g = qvkv::gather_grid(items, tiles, per_tile, positions, 1ull << 40, 16, one_xcd);
    const uint64_t most = g.by_tile ? (1u << 18) + per_tile : (1u << 26) - 1;
    if (g.wgs == 0 || g.wgs % per_tile || g.wgs > most) return bad("wgs", g.wgs, per_tile);
    const uint64_t units = items * tiles, step = g.wgs / per_tile;
    if (g.by_tile && step > positions / 16 + items) return bad("more than held", step, positions);
    std::vector<uint8_t> seen(units, 0);
    std::vector<uint8_t> starts(step * per_tile, 0);
    for (uint32_t wg = 0; wg < g.wgs; wg++) {
        const qvkv::GatherPlace at = qvkv::gather_place(wg, (uint32_t)per_tile, g.by_xcd);
        if (at.part >= per_tile || at.unit >= step || starts[at.unit * per_tile + at.part]++) return bad("place", wg, step);
        if (g.by_xcd && wg % 8 != at.unit % 8) return bad("xcd", wg, at.unit);
    }
    for (uint64_t u0 = 0; u0 < step; u0++)
        for (uint64_t u = u0; u < units; u += step) {
            const uint64_t by = g.by_tile ? items : tiles, q = u / by, r = u - q * by;
            const uint64_t item = g.by_tile ? r : q, tile = g.by_tile ? q : r;
            if (item >= items || tile >= tiles || seen[item * tiles + tile]++) return bad("unit", u, step);
        }
    for (uint8_t s : seen)
        if (s != 1) return bad("missed", units, step);
    return 0;
}
int main() {
    int rc = 0;
    const uint64_t shapes[][4] = {{1, 1, 1, 16}, {64, 64, 32, 65536}, {64, 2048, 32, 97280}, {256, 2048, 16, 49088},
                                  {7, 5, 3, 560}, {64, 128, 32, 131072}, {33, 4096, 2, 4096}, {4096, 1024, 128, 65536},
                                  {1000, 1000, 1, 16000000}, {3, 1, 300000, 48}, {100, 63, 512, 6400}};
    for (auto &s : shapes)
        for (bool one_xcd : {false, true}) rc |= covers(s[0], s[1], s[2], s[3], one_xcd);
    for (uint64_t tiles : {128, 129, 131}) rc |= covers(128, tiles, 32, 128 * 16 * tiles, true);
    if (!qvkv::gather_grid(128, 129, 32, 128 * 16 * 129, 1 << 20, 16, true).by_xcd) rc |= bad("by_xcd", 0, 0);
    // an even batch: a workgroup per piece of every unit
    if (qvkv::gather_grid(512, 128, 32, 512 * 2048, 512 * 128, 16).wgs != 512 * 128 * 32) rc |= bad("even", 0, 0);
    // an uneven batch: far fewer workgroups than pieces (a workgroup costs its dispatch)
    const qvkv::GatherGrid g = qvkv::gather_grid(64, 2048, 32, 32768 + 63 * 1024, 6080, 16);
    if (!g.by_tile || g.wgs > 6144 * 32) rc |= bad("uneven", g.wgs, g.by_tile);
    // 2^24 units and more are refused, never wrapped: 65536 items bounded by 262160 positions
    if (qvkv::gather_grid(65536, 16385, 128, 1 << 20, 1 << 20, 16).wgs) rc |= bad("refuse", 0, 0);
    if (qvkv::gather_grid(1 << 12, 1 << 12, 128, 1 << 20, 1 << 20, 16).wgs) rc |= bad("refuse", 1, 0);
    // 4096 items bounded by 16384 positions, 32 heads of 128, are not
    if (!qvkv::gather_grid(4096, 1024, 128, 1 << 20, 1 << 20, 16).wgs) rc |= bad("accept", 0, 0);
    if (!rc) printf("OK\n");
    return rc;
}
"""


def test_gather_grid_takes_every_unit_once(tmp_path):
    src, exe = tmp_path / "gg.cpp", tmp_path / "gg"
    src.write_text(PROG)
    try:
        subprocess.run(["g++", "-O2", "-std=c++17", "-I", HDR, str(src), "-o", str(exe)], check=True,
                       capture_output=True, text=True)
    except FileNotFoundError:
        pytest.skip("g++ is not available")
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "OK", r.stdout
