"""The host's fp16 slabs of a cache block (csrc/plan.cpp): the vector form against the element-by-element definition of
the blocked layout with f32_to_f16_rne, bit for bit, over every token count and values on both sides of every rounding
case (ties, subnormals, overflow, infinities, NaN payloads of both signs)."""

import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DRIVER = r"""
#include <cstdio>
#include <cstring>
#include <vector>
#include "pvlc_internal.hpp"
using namespace pvlc;
int main() {
    uint64_t x = 88172645463325252ull;
    auto next = [&] { x ^= x << 13; x ^= x >> 7; x ^= x << 17; return x; };
    const uint32_t edges[] = {0, 1, 0x007fffff, 0x00800000, 0x33000000, 0x33000001, 0x32ffffff, 0x387fc000, 0x387fe000, 0x387fffff,
                              0x38800000, 0x38801000, 0x38801001, 0x38803000, 0x477fe000, 0x477fefff, 0x477ff000, 0x47800000,
                              0x7f7fffff, 0x7f800000, 0x7f800001, 0x7fa00000, 0x7fc051a7, 0x7fffffff};
    int checks = 0;
    for (int round = 0; round < 400; ++round)
        for (uint32_t tokens = 1; tokens <= 16; ++tokens) {
            std::vector<float> rows(tokens * 256);  // exactly the valid rows: a read past them is out of bounds
            for (float &f : rows) {
                uint32_t bits = static_cast<uint32_t>(next());
                const uint32_t kind = static_cast<uint32_t>(next() % 4);
                if (kind == 0) bits = edges[next() % (sizeof(edges) / 4)] | (bits & 0x80000000u);
                if (kind == 1) bits = (bits & 0x80ffffffu) | 0x38000000u;
                if (kind == 2) bits = (bits & 0x87ffffffu) | 0x40000000u;
                std::memcpy(&f, &bits, 4);
            }
            std::vector<uint16_t> k(4096, 0xabcd), v(4096, 0xabcd), wk(4096, 0), wv(4096, 0);
            for (uint32_t t = 0; t < tokens; ++t)
                for (uint32_t h = 0; h < 2; ++h)
                    for (uint32_t d = 0; d < 128; ++d) {
                        const uint16_t b = f32_to_f16_rne(rows[(t * 2 + h) * 128 + d]);
                        wk[key_blocked_index(t, h, d)] = b;
                        wv[value_blocked_index(t, h, d)] = b;
                    }
            key_block_slabs(rows.data(), tokens, k.data());
            value_block_slabs(rows.data(), tokens, v.data());
            if (k != wk || v != wv) return std::printf("differs at %u tokens, round %d\n", tokens, round), 1;
            ++checks;
        }
    std::printf("%d blocks equal\n", checks);
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_slabs_of_a_block_equal_the_layout_bit_for_bit(tmp_path):
    src, exe = tmp_path / "slabs.cpp", str(tmp_path / "slabs")
    src.write_text(DRIVER)
    csrc = os.path.join(REPO, "paddleocr-vl-webgpu_amd", "csrc")
    build = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                            "-I", os.path.join(REPO, "include"), "-I", csrc, str(src), os.path.join(csrc, "plan.cpp"),
                            "-lm", "-o", exe], capture_output=True, text=True)
    assert build.returncode == 0, build.stderr[-3000:]
    env = {k: v for k, v in os.environ.items() if k != "LD_PRELOAD"}
    run = subprocess.run([exe], capture_output=True, text=True, env=env, timeout=120)
    assert run.returncode == 0, run.stdout + run.stderr[-2000:]
    assert "6400 blocks equal" in run.stdout
