"""The tile that the projection chooses (csrc/pvlc_internal.hpp): for every admitted geometry whose operands a device of up
to 512 GiB could hold, a tile is found, its grid stays under 2^32 threads, its weight offsets within 32 bits, and its
blocks cover every output tile; few rows of very many columns among them.  And the tiles that were measured fastest where
the choice is between sizes far apart."""

import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DRIVER = r"""
#include <cmath>
#include <cstdio>
#include <random>
#include "pvlc_internal.hpp"
using namespace pvlc;
static int fails = 0, seen[kProjectionTileCount] = {}, checks = 0;
static void check(uint64_t rows, uint64_t k, uint64_t n) {
    // as admitted: widths, rows and output tiles
    const uint64_t tiles = (rows + 127) / 128 * ((n + 127) / 128);
    if (!rows || rows > 65535u * 128u || !n || n % 4 || n > 0xffffffffu || !k || k % 32 || tiles >= 1u << 24) return;
    const double bytes = 2.0 * n * k + 4.0 * ((rows + 127) / 128 * 128) * k + 4.0 * rows * n;
    if (bytes > 512.0 * 1073741824.0) return;
    ProjectionOrder o{};
    uint64_t block = 0;
    const int i = choose_projection_tile(rows, k, n, &o, &block);
    ++checks;
    bool good = i >= 0;
    if (good) {
        const ProjectionTile t = kProjectionTiles[i];
        ++seen[i];
        const uint64_t gr = kXcds / o.col_groups;
        good = kXcds * block * t.threads < 1ull << 32 && (i + 1 < kProjectionTileCount ? (7 * (k / 8) + 7) * 16 : 15 * (k / 8) + 7) < 1ull << 32 && o.row_tiles == (rows + t.rows - 1) / t.rows &&
               o.col_tiles == (n + t.cols - 1) / t.cols && (o.row_tiles + gr - 1) / gr * ((o.col_tiles + o.col_groups - 1) / o.col_groups) <= block &&
               o.gen >= 1;
    }
    if (!good && ++fails < 10) std::printf("rows %llu k %llu n %llu: tile %d block %llu\n", (unsigned long long)rows, (unsigned long long)k, (unsigned long long)n, i, (unsigned long long)block);
}
int main() {
    std::mt19937_64 r(5);
    auto log = [&](double lo, double hi) { return std::floor(lo * std::pow(hi / lo, (r() >> 11) * 0x1p-53)); };
    for (int i = 0; i < 300000; ++i) check(log(1, 8388481), 32 * log(1, 1 << 24), 4 * log(1, 1 << 30));
    for (uint64_t n = 1ull << 29; n < 1ull << 31; n += (1ull << 25) + 4)
        for (uint64_t rows : {1, 8, 16, 17, 32, 64, 128}) check(rows, 32, n);
    for (uint64_t rows : {1, 16, 4096, 8388479, 8388480}) for (uint64_t n : {4, 12, 16, 28, 32, 60, 64, 124, 128, 188, 192}) check(rows, 32, n);
    // rows, k, n; the fastest tile of all, and its lead over 128 x 96
    const uint32_t fastest[][5] = {{2500, 1024, 6144, 128, 128},   // 67.9 us against 87.3
                                   {3500, 1024, 6144, 128, 192},   // 88.7 against 117.5
                                   {1300, 1024, 6144, 128, 160},   // 41.7 against 51.3
                                   {1836, 1152, 4304, 128, 160},   // 46.7 against 55.4
                                   {2500, 1152, 3456, 128, 160}};  // 48.9 against 59.9
    for (const auto &f : fastest) {
        ProjectionOrder o{};
        uint64_t block = 0;
        const ProjectionTile t = kProjectionTiles[choose_projection_tile(f[0], f[1], f[2], &o, &block)];
        if (t.rows != f[3] || t.cols != f[4]) std::printf("%u x %u x %u takes %u x %u\n", f[0], f[1], f[2], t.rows, t.cols), ++fails;
    }
    for (int i = 0; i < kProjectionTileCount; ++i) if (!seen[i]) { std::printf("tile %d never chosen\n", i); ++fails; }
    std::printf("%d geometries, %d failures\n", checks, fails);
    return fails != 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_every_admitted_geometry_has_a_tile_whose_grid_fits(tmp_path):
    src, exe = tmp_path / "tiles.cpp", str(tmp_path / "tiles")
    src.write_text(DRIVER)
    build = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=undefined", "-fno-sanitize-recover=all", "-I",
                            os.path.join(REPO, "include"), "-I", os.path.join(REPO, "paddleocr-vl-webgpu_amd", "csrc"), str(src),
                            "-o", exe], capture_output=True, text=True)
    assert build.returncode == 0, build.stderr[-3000:]
    run = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stdout + run.stderr[-2000:]
