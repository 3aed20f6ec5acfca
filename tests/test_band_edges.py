"""The tile pass's 32-bit edge functions (csrc/band.hpp) compiled for the host
with UndefinedBehaviorSanitizer: over edges of every length up to beyond the
guard band, the sign at every centre of a band equals the 64-bit function's
where the edge is narrow, a band is only left out where the edge is negative
everywhere, and no product overflows, narrow or not."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <cstdio>
#include <random>
#define __device__
#define __forceinline__ inline
#include "band.hpp"
int main()
{
    std::mt19937_64 rng(7);
    auto upto = [&](int bits) {   // log-uniform magnitude below 2^bits, either sign, the ends among them
        const int b = (int)(rng() % (bits + 1));
        const long long m = b ? (long long)(rng() % (1ull << b)) : 0;
        const long long v = rng() % 16 == 0 ? (1ll << b) - 1 : m;
        return rng() & 1 ? v : -v;
    };
    long narrow = 0, out = 0;
    for (int k = 0; k < 200000; ++k) {
        const int ex = (int)upto(30), ey = (int)upto(30), dx = (int)upto(14), dy = (int)upto(14), w = 32, h = 16;
        // functions that change sign near the band half of the time, any others else
        long long e0 = rng() & 1 ? upto(58) : (long long)dx * ey * 256 - (long long)dy * ex * 256 + upto(36);
        const vkgv::BandEdge b = vkgv::band_edge(e0, ex, ey, dx, dy, w, h);
        if (!b.narrow) {
            if (b.out || (ex > -(1 << 22) && ex < (1 << 22) && ey > -(1 << 22) && ey < (1 << 22))) return 1;
            continue;
        }
        ++narrow;
        bool any = false;
        for (int y = 0; y < h; ++y)
            for (int x = 0; x < w; ++x) {
                const bool in = e0 - (long long)(dx + x) * ey * 256 + (long long)(dy + y) * ex * 256 >= 0;
                any = any || in;
                if ((b.start - x * ey + y * ex >= 0) != in) return 2;
            }
        if (b.out == any) return 3;
        out += b.out;
    }
    std::printf("%ld narrow edges, %ld out\n", narrow, out);
    return narrow > 50000 && out > 5000 && out < narrow ? 0 : 4;
}
"""


def test_band_edges(tmp_path):
    src, exe = tmp_path / "band.cpp", tmp_path / "band"
    src.write_text(SOURCE)
    r = subprocess.run(["g++", "-O0", "-std=c++17", "-fsanitize=undefined", "-fno-sanitize-recover=all", "-I",
                        os.path.join(ROOT, "vk_gltf_viewer_amd", "csrc"), "-o", str(exe), str(src)],
                       capture_output=True, text=True)
    if r.returncode and "ubsan" in r.stderr:
        pytest.skip("no UndefinedBehaviorSanitizer here")
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, f"case {r.returncode}: {r.stderr}"
