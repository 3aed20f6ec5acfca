// One edge function of a big triangle over a wave's band of the tile pass:
// integer arithmetic only, also compiled for the host by its test.
#pragma once

namespace vkgv {

constexpr int kNarrowEdge = 1 << 22;   // 1/256 pixel: 2^14 pixels

struct BandEdge {
    int start;      // the edge function at the band's first centre, over 256, cut to +-2^29
    bool narrow;    // ex and ey below kNarrowEdge: start, with steps of -ey and ex a pixel, has the right sign in the band
    bool out;       // narrow, and negative all over the band
};

// e0: the edge function at a centre from which the band's first one lies dx
// pixels to the right and dy down; ex, ey: the edge in 1/256 pixel, so that a
// pixel to the right adds -256 ey and one down 256 ex; w, h: the band's size, at
// most 32.  Only products of narrow edges fit 32 bits.
__device__ __forceinline__ BandEdge band_edge(long long e0, int ex, int ey, int dx, int dy, int w, int h)
{
    const long long v = (e0 - (long long)dx * ey * 256 + (long long)dy * ex * 256) >> 8, lim = 1ll << 29;
    BandEdge b;
    b.start = (int)(v < -lim ? -lim : v > lim ? lim : v);
    b.narrow = ex > -kNarrowEdge && ex < kNarrowEdge && ey > -kNarrowEdge && ey < kNarrowEdge;
    b.out = b.narrow && b.start + (ey < 0 ? -(w - 1) * ey : 0) + (ex > 0 ? (h - 1) * ex : 0) < 0;
    return b;
}

} // namespace vkgv
