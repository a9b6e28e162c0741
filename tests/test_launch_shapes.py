"""Grids of the per-point kernels, on the host: HIP launches fewer than 2^32
work-items in one grid dimension, so longer lines of blocks are folded; every
tile of a box must still belong to exactly one block, in either order of the
blocks over the XCDs, and blocks without one must see no point.  A host program includes the library's own launch header
and walks all block ids."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
SOURCE = r"""
#include "common.hpp"
#include <cstdlib>
#include <vector>
namespace chmy {
int set_error(int code, const char*, ...) { return code; }
int hip_status(hipError_t, const char*) { return -1; }
}
using namespace chmy;
#define CHECK(x) do { if (!(x)) { std::printf("%s:%d: %s (box %lld %lld %lld)\n", __FILE__, __LINE__, #x, \
    (long long)b.len[0], (long long)b.len[1], (long long)b.len[2]); std::exit(1); } } while (0)
static Box3 box(int64_t x, int64_t y, int64_t z) { return Box3{{0, 3, 1}, {x, y, z}}; }

// every block id of the box's grid: the tile that its lane 0 names (all lanes
// when `lanes`), in either order of the blocks
static void walk(int64_t x, int64_t y, int64_t z, bool lanes, bool spread) {
    Box3 b = box(x, y, z);
    dim3 g;
    CHECK(flat_grid(b, 8, &g) == 0);
    b.spread = spread;
    CHECK((uint64_t)g.x * kFlat < (1ull << 32) && g.y < 65536 && g.z == 1);
    const uint64_t n = (uint64_t)g.x * g.y, per = (uint64_t)((x * y + kFlat - 1) / kFlat);
    CHECK(n >= per * z && (g.y == 1 || g.x % 8 == 0));
    std::vector<bool> seen(per * z, false);
    uint64_t tiles = 0, points = 0;
    for (uint64_t id = 0; id < n; ++id) {
        int64_t i, j, k;
        if (!flat_at(b, (uint32_t)id, (uint32_t)n, 0, i, j, k)) {
            CHECK(k - 1 >= z);   // lane 0 of a tile is a point: only ids past the last tile have none
            for (uint32_t l = 1; l < kFlat; ++l) CHECK(!flat_at(b, (uint32_t)id, (uint32_t)n, l, i, j, k));
            continue;
        }
        const uint64_t q = (uint64_t)(j - 3) * x + i;
        CHECK(i >= 0 && i < x && j >= 3 && j - 3 < y && k >= 1 && k - 1 < z && q % kFlat == 0);
        const uint64_t t = (k - 1) * per + q / kFlat;
        CHECK(!seen[t]);
        seen[t] = true;
        ++tiles;
        for (uint32_t l = 0; lanes && l < kFlat; ++l) {
            int64_t i1, j1, k1;
            const bool in = flat_at(b, (uint32_t)id, (uint32_t)n, l, i1, j1, k1);
            CHECK(in == (q + l < (uint64_t)(x * y)));
            if (in) {
                CHECK(k1 == k && (uint64_t)(j1 - 3) * x + i1 == q + l);
                ++points;
            }
        }
    }
    CHECK(tiles == per * z);
    CHECK(!lanes || points == (uint64_t)(x * y * z));
}

int main() {
    for (int64_t x : {1, 3, 255, 256, 257, 700})
        for (int64_t y : {1, 2, 9})
            for (int64_t z : {1, 4, 33, 600})
                for (bool spread : {false, true}) walk(x, y, z, z < 600, spread);
    for (bool spread : {false, true}) {
        walk(65535, 65536, 1, false, spread);        // 2^32 - 2^16 points
        walk(65536, 65536, 1, false, spread);        // 2^32, the 64-bit division
        walk(1626, 1626, 1626, false, spread);
        walk(1626, 1627, 1626, false, spread);
        walk(3, 2, 16777217, false, spread);         // a block a plane
        walk((int64_t(1) << 32) + 5, 1, 1, false, spread);
    }
    for (int threads : {64, 256, 768, 1024})
        for (int64_t nb : {int64_t(1), int64_t(1) << 22, (int64_t(1) << 24) - 1, int64_t(1) << 24, (int64_t(1) << 26) + 1, kLineMost}) {
            Box3 b = box(nb, threads, 0);
            dim3 g;
            CHECK(line_grid(nb, threads, &g) == 0);
            CHECK((uint64_t)g.x * threads < (1ull << 32) && (int64_t)g.x * g.y >= nb);
            CHECK((uint64_t)nb * threads >= (1ull << 32) ? (g.y > 1 && g.x % 8 == 0) : (g.x == nb && g.y == 1));
            CHECK((uint64_t)g.x * g.y < (1ull << 31));
        }
    dim3 g;
    Box3 b = box(256, 4, 1024);   // 2^20 points: 256 bytes each are the cache's size
    CHECK(flat_grid(b, 256, &g) == 0 && !b.spread && flat_grid(b, 257, &g) == 0 && b.spread);
    b = box(0, 0, 0);
    CHECK(line_grid(kLineMost + 1, 64, &g) == CHMY_E_SIZE);
    b = box(int64_t(1) << 30, int64_t(1) << 30, 1);
    CHECK(flat_grid(b, 8, &g) == CHMY_E_SIZE);
    b = box(int64_t(1) << 40, int64_t(1) << 40, 3);
    CHECK(flat_grid(b, 8, &g) == CHMY_E_SIZE);
    std::printf("ok\n");
    return 0;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_every_tile_has_one_block(tmp_path):
    src, exe = tmp_path / "shapes.hip", tmp_path / "shapes"
    src.write_text(SOURCE)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-host-only", "-O2", "-std=c++17", "-Wno-unused-function",
                    "-I", os.path.join(ROOT, "chmy.jl_amd", "csrc"), "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
