// Differentiable form of the frame: triangle raster to an id/depth buffer,
// perspective-correct attribute interpolation and analytic edge antialiasing,
// each with a hand-written backward that recomputes barycentrics and edge
// crossings from the id buffer instead of storing per-pixel attributes.
//
// Conventions (shared with the torch bindings and the FP64 reference):
//  clip      [C, I, V, 4]  clip-space position of vertex v of instance i seen
//                          by camera c (reverse-Z, as the frame's cameras)
//  tris      [T, 3] int32  vertex indices, one mesh shared by the instances
//  ids       [C, H, W] int32  0 = background, else i * T + t + 1
//  depth     [C, H, W] f32    z / w at the pixel centre (larger = nearer)
//  pixel (x, y) has its centre at NDC ((x + 0.5) / (W/2) - 1, (y + 0.5) / (H/2) - 1).
//
// Interpolation: with h_k = (x, y, w) of vertex k's clip position,
// r_k = h_{k+1} x h_{k+2}, l_k = r_k . (xn, yn, 1) and lambda_k = l_k / sum(l),
// colour = sum_k lambda_k attr_k.  The kernels evaluate l_k in the equivalent
// pixel-relative form l_k = u_{k+1} x u_{k+2} (2-D cross product) with
// u_k = (x_k - xn w_k, y_k - yn w_k): subtracting the pixel's ray before the
// product keeps float32 accurate for triangles much smaller than their
// distance, where the 3-D cross product cancels.
//
// Antialiasing: for every horizontally or vertically adjacent pixel pair with
// different ids, the front pixel f (the non-background one, else the one with
// the larger depth) keeps its triangle T; the segment from f's centre to the
// other centre b leaves T through the edge of T whose edge function changes
// sign first, at parameter t in [0, 1] (an edge through a centre counts, so
// the output stays continuous when an edge crosses a centre).  The part of the pixel on the far side of the
// edge, along the pair's axis, takes the other pixel's colour:
//   t < 1/2: out_f += (1/2 - t) (c_b - c_f);   t > 1/2: out_b += (t - 1/2) (c_f - c_b).
// The output is continuous in the vertex positions; the backward gives the
// gradient of the colours and, through t, of the edge's clip positions.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "diff.hpp"

namespace vkgv_diff {
namespace {

constexpr uint32_t kBlock = 256;
constexpr int kMaxAttr = 8;

__device__ __forceinline__ uint32_t float_bits(float f) { return __float_as_uint(f); }

__device__ __forceinline__ unsigned long long make_key(float z, uint32_t id)
{
    return ((unsigned long long)(~float_bits(z + 0.0f)) << 32) | (unsigned long long)(0xFFFFFFFEu - id);
}

template <typename T> struct V2 {
    T x, y;
};
// A caller's clip position: aligned as its elements are (a contiguous tensor may
// start anywhere in its storage); loaded 16 bytes at a time all the same.
template <typename T> struct V4 {
    T x, y, z, w;
};
// A pair moved by one load or store.
template <typename T> struct alignas(2 * sizeof(T)) R2 {
    T x, y;
};

// clip = m (p, 1), m row-major.
template <typename C> __device__ __forceinline__ void transform_vertex(const C* m, const C* p, V4<C>& o)
{
    const C x = p[0], y = p[1], z = p[2];
    o.x = fma(m[0], x, fma(m[1], y, fma(m[2], z, m[3])));
    o.y = fma(m[4], x, fma(m[5], y, fma(m[6], z, m[7])));
    o.z = fma(m[8], x, fma(m[9], y, fma(m[10], z, m[11])));
    o.w = fma(m[12], x, fma(m[13], y, fma(m[14], z, m[15])));
}

struct Dims {
    int C, I, V, T, H, W;
};

struct Box {
    int x0, x1, y0, y1;
};

// boxes[(c * I + i) * T + t]: x0 | x1 << 16 | y0 << 32 | y1 << 48, or kNoBox
// for a triangle that is not gathered (or has a vertex out of range); an
// empty box (x0 > x1) for one on no pixel.
constexpr unsigned long long kNoBox = ~0ull;

__device__ __forceinline__ unsigned long long pack_box(const Box& b)
{
    return (unsigned long long)(uint16_t)b.x0 | ((unsigned long long)(uint16_t)b.x1 << 16)
           | ((unsigned long long)(uint16_t)b.y0 << 32) | ((unsigned long long)(uint16_t)b.y1 << 48);
}

__device__ __forceinline__ Box unpack_box(unsigned long long v)
{
    return Box{ (int)(v & 0xFFFFu), (int)((v >> 16) & 0xFFFFu), (int)((v >> 32) & 0xFFFFu), (int)(v >> 48) };
}

// ---------------------------------------------------------------------------
// Raster: one thread per (camera, instance, triangle); snapped vertices,
// exact integer edge functions with a top-left rule, depth plane evaluated at
// pixel centres, 64-bit atomicMin of (depth, id).  Triangles with a vertex at
// w <= 0 are skipped (the cameras of this form see the mesh from outside).
//
// render projects and snaps the vertices once each (Snap, 16 bytes), not once
// for each of the about six triangles that share one: its triangle pass has no
// division until a triangle's box holds a pixel centre.  Coordinates are 32-bit
// (below 2^28), edge functions 64-bit.  A box of more than kWaveBox pixels is
// walked by the whole wave.  Bound by the vector ALU (36.9M instructions) and the
// atomics of every front and back fragment: 6.5M triangles of about half a
// pixel in 8 views of 512x512 take 130 us; with a projection per triangle
// corner 147 us, besides the pass that rounded the clip positions to float.
// (Reading the key first and skipping the atomic of a hidden fragment puts a
// load's latency in the pixel loop: 223 us.)
struct alignas(16) Snap {
    int x, y;       // 1/256 pixel
    float z;        // z / w
    int ok;         // 0: w <= 0 or beyond the guard band, no triangle of this vertex is drawn
};
constexpr int kWaveBox = 64;

__device__ __forceinline__ Snap snap_vertex(const V4<float>& p, const Dims& d)
{
    const float hw = (float)d.W * 0.5f, hh = (float)d.H * 0.5f;
    Snap s{ 0, 0, 0.0f, 0 };
    if (!(p.w > 0.0f)) return s;
    const float xf = hw * (p.x / p.w) + hw, yf = hh * (p.y / p.w) + hh;
    if (!(fabsf(xf) < 1048576.0f && fabsf(yf) < 1048576.0f)) return s;
    s.x = (int)rintf(xf * 256.0f);
    s.y = (int)rintf(yf * 256.0f);
    s.z = p.z / p.w;
    s.ok = 1;
    return s;
}

// The start of render: clip[ci, v] = M[ci] (p_v, 1), its snapped vertex (of the
// position rounded to float), and the buffers of the passes that follow
// cleared: npx keys and nvis words of flags (the vis bytes and the wide flag
// behind them), spread over the grid.
template <typename C>
__global__ __launch_bounds__(kBlock) void project_kernel(const C* __restrict__ pos, const C* __restrict__ M, Dims d,
                                                          C* __restrict__ clip, Snap* __restrict__ snap,
                                                          unsigned long long* __restrict__ keys, size_t npx,
                                                          uint32_t* __restrict__ vis, size_t nvis)
{
    const size_t g = ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * kBlock + threadIdx.x;
    const size_t n = (size_t)gridDim.x * gridDim.y * kBlock;
    for (size_t k = g; k < npx; k += n) keys[k] = ~0ull;
    for (size_t k = g; k < nvis; k += n) vis[k] = 0u;
    const int v = (int)(blockIdx.x * kBlock + threadIdx.x);
    const size_t ci = blockIdx.y;
    if (v >= d.V || ci >= (size_t)d.C * d.I) return;
    V4<C> o;
    transform_vertex(M + ci * 16, pos + 3 * (size_t)v, o);
    reinterpret_cast<V4<C>*>(clip)[ci * d.V + v] = o;
    snap[ci * d.V + v] = snap_vertex(V4<float>{ (float)o.x, (float)o.y, (float)o.z, (float)o.w }, d);
}

// A triangle ready to be walked over its box of pixels: edge functions at the
// first centre minus the top-left bias (a centre is covered iff all are >= 0),
// the depth plane from vertex 0.
struct TriWalk {
    long long e[3];
    int ex[3], ey[3];   // a pixel to the right adds -256 ey, a row down 256 ex
    float z0, za, zb;
    int ox, oy;         // first centre from vertex 0, 1/256 pixel
    int px0, px1, py0, py1;
    uint32_t id;
    float size;         // area in pixels

    // Edge function k at pixel (i, j) of the box.
    __device__ __forceinline__ long long edge_at(int k, int i, int j) const
    {
        return e[k] + (((long long)j * ex[k] - (long long)i * ey[k]) << 8);
    }
    // Visibility-buffer key of pixel (i, j), covered or not; all ones where the
    // depth is out of range.
    __device__ __forceinline__ unsigned long long depth_key(int i, int j) const
    {
        const float z = z0 + (za * ((float)(ox + 256 * i) * 0.00390625f) + zb * ((float)(oy + 256 * j) * 0.00390625f));
        return z >= 0.0f && z <= 1.0f ? make_key(z, id) : ~0ull;
    }
    // The same, all ones also where the centre is not covered.
    __device__ __forceinline__ unsigned long long key_at(int i, int j) const
    {
        return (edge_at(0, i, j) | edge_at(1, i, j) | edge_at(2, i, j)) >= 0 ? depth_key(i, j) : ~0ull;
    }
};

__device__ __forceinline__ void key_min(unsigned long long* p, unsigned long long key)
{
    (void)__hip_atomic_fetch_min(p, key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// What render keeps a byte of per (camera, instance, triangle), vis: kSeen for
// one with a visible pixel whose box the vertex pass walks, kWide for one with a
// fragment whose terms the backward's pixel pass sums instead.  `wide` is a flag
// for the whole call: there is a kWide byte.
//
// kWide is a box of more than kWideBox pixels, or one of more than kWaveBox of
// which the triangle's area is less than 1 / kSliver.  The vertex pass reads the
// whole box, once a corner, in the one wave of the vertex, triangle after
// triangle; the pixel pass reads own pixels only but pays for every tile.  A step
// of 1, 8 or 8 cameras, 512x512, spheres of 1280 triangles (boxes up to 5000
// pixels) 1029 -> 736 us, 1841 -> 1358, of 2880 (boxes around 2000) equal; limits
// of 512 and 256 take these to 975 and 733, but cost 8 and 15 % for 8 instances
// of 5120 and 11520 triangles in float64.  Slivers: 200 triangles around one
// vertex at 96x96 854 -> 568 us, 2000 at 400x400 in 4 cameras 198 -> 5.1 ms.
constexpr int kWideBox = 1024;
constexpr float kSliver = 16.0f;
enum : uint8_t { kHidden = 0, kSeen = 1, kWide = 2 };

// boxes (null with vis and wide, for a raster alone): the pixel box of each
// triangle with a fragment.
// V: Snap, or V4<float> for clip positions, projected and snapped here for each
// corner (three times the divisions, but no pass over the vertices before).
__device__ __forceinline__ Snap snapped(const Snap& v, const Dims&) { return v; }
__device__ __forceinline__ Snap snapped(const V4<float>& v, const Dims& d) { return snap_vertex(v, d); }
template <typename V>
__global__ __launch_bounds__(kBlock) void raster_tris_kernel(const V* __restrict__ vtx, const int* __restrict__ tris,
                                                              Dims d, unsigned long long* __restrict__ keys,
                                                              unsigned long long* __restrict__ boxes,
                                                              uint8_t* __restrict__ vis, uint32_t* __restrict__ wide_flag,
                                                              int per_wave, int cull_back)
{
    const int lane = (int)(threadIdx.x & 63u), wave = (int)(blockIdx.x * (kBlock / 64u) + (threadIdx.x >> 6));
    const int t = lane < per_wave ? wave * per_wave + lane : d.T;
    for (int ci = (int)blockIdx.y; ci < d.C * d.I; ci += (int)gridDim.y) {
        const V* sv = vtx + (size_t)ci * d.V;
        unsigned long long* img = keys + (size_t)(ci / d.I) * d.H * d.W;
        TriWalk w;
        bool live = false;
        if (t < d.T) {
            const Snap a = snapped(sv[tris[3 * t]], d), b = snapped(sv[tris[3 * t + 1]], d),
                       c = snapped(sv[tris[3 * t + 2]], d);
            w.px0 = max((min(a.x, min(b.x, c.x)) + 127) >> 8, 0);
            w.px1 = min((max(a.x, max(b.x, c.x)) - 128) >> 8, d.W - 1);
            w.py0 = max((min(a.y, min(b.y, c.y)) + 127) >> 8, 0);
            w.py1 = min((max(a.y, max(b.y, c.y)) - 128) >> 8, d.H - 1);
            live = a.ok & b.ok & c.ok && w.px0 <= w.px1 && w.py0 <= w.py1;
            if (live) {
                long long area = (long long)(b.x - a.x) * (c.y - a.y) - (long long)(b.y - a.y) * (c.x - a.x);
                live = area != 0 && !(cull_back && area > 0);   // the winding the frame's back-face test keeps
                if (live) {
                    const bool flip = area < 0;
                    if (flip) area = -area;
                    const Snap p = flip ? c : b, q = flip ? b : c;
                    const int X[3] = { a.x, p.x, q.x }, Y[3] = { a.y, p.y, q.y };
                    const int sx = w.px0 * 256 + 128, sy = w.py0 * 256 + 128;
#pragma unroll
                    for (int k = 0; k < 3; ++k) {
                        const int ka = (k + 1) % 3, kb = (k + 2) % 3;
                        const int ex = X[kb] - X[ka], ey = Y[kb] - Y[ka];
                        const bool tl = ey < 0 || (ey == 0 && ex > 0);
                        w.e[k] = (long long)ex * (sy - Y[ka]) - (long long)ey * (sx - X[ka]) - (tl ? 0 : 1);
                        w.ex[k] = ex;
                        w.ey[k] = ey;
                    }
                    w.ox = sx - a.x;
                    w.oy = sy - a.y;
                    const double e1x = (double)(p.x - a.x) / 256.0, e1y = (double)(p.y - a.y) / 256.0;
                    const double e2x = (double)(q.x - a.x) / 256.0, e2y = (double)(q.y - a.y) / 256.0;
                    const double dz1 = (double)p.z - (double)a.z, dz2 = (double)q.z - (double)a.z;
                    const double det = (double)area / 65536.0;
                    w.size = 0.5f * (float)det;
                    w.z0 = a.z;
                    w.za = (float)((dz1 * e2y - dz2 * e1y) / det);
                    w.zb = (float)((dz2 * e1x - dz1 * e2x) / det);
                    w.id = (uint32_t)((ci % d.I) * d.T + t + 1);
                }
            }
        }
        const bool wide = live && (long long)(w.px1 - w.px0 + 1) * (w.py1 - w.py0 + 1) > kWaveBox;
        bool drawn = false;
        if (live && !wide) {
            unsigned long long* at = img + (size_t)w.py0 * d.W + w.px0;
            const int bw = w.px1 - w.px0 + 1, n = bw * (w.py1 - w.py0 + 1);
            for (int q = 0, i = 0, j = 0; q < n; ++q) {
                const unsigned long long key = w.key_at(i, j);
                if (key != ~0ull) {
                    key_min(at + (size_t)j * d.W + i, key);
                    drawn = true;
                }
                if (++i == bw) {
                    i = 0;
                    ++j;
                }
            }
        }
        // one wide triangle at a time in blocks of 8x8 pixels, a pixel per lane,
        // the edge functions stepped from block to block (with a division and six
        // products a pixel instead, 10240 triangles with boxes around 60x60 took 360
        // us, not 288)
        unsigned long long pending = __ballot(wide);
        while (pending != 0ull) {
            const int j = __ffsll((long long)pending) - 1;
            pending &= pending - 1ull;
            TriWalk u;
            constexpr int kWords = (int)(sizeof(TriWalk) / 4);
            static_assert(sizeof(TriWalk) % 4 == 0, "broadcast word by word");
            const uint32_t* from = reinterpret_cast<const uint32_t*>(&w);
            uint32_t* to = reinterpret_cast<uint32_t*>(&u);
#pragma unroll
            for (int k = 0; k < kWords; ++k) to[k] = (uint32_t)__builtin_amdgcn_readlane((int)from[k], j);
            const int lx = lane & 7, ly = lane >> 3, bw = u.px1 - u.px0 + 1, bh = u.py1 - u.py0 + 1;
            unsigned long long* at = img + (size_t)u.py0 * d.W + u.px0;
            long long row[3] = { u.edge_at(0, lx, ly), u.edge_at(1, lx, ly), u.edge_at(2, lx, ly) };
            bool any = false;
            for (int by = 0; by < bh; by += 8) {
                long long v[3] = { row[0], row[1], row[2] };
                for (int bx = 0; bx < bw; bx += 8) {
                    const int i = bx + lx, jj = by + ly;
                    if (i < bw && jj < bh && (v[0] | v[1] | v[2]) >= 0) {
                        const unsigned long long key = u.depth_key(i, jj);
                        if (key != ~0ull) {
                            key_min(at + (size_t)jj * d.W + i, key);
                            any = true;
                        }
                    }
#pragma unroll
                    for (int k = 0; k < 3; ++k) v[k] -= (long long)u.ey[k] * 2048;
                }
#pragma unroll
                for (int k = 0; k < 3; ++k) row[k] += (long long)u.ex[k] * 2048;
            }
            if (__ballot(any) != 0ull && lane == j) drawn = true;
        }
        if (boxes && drawn) {
            boxes[(size_t)ci * d.T + t] = pack_box(Box{ w.px0, w.px1, w.py0, w.py1 });
            const int box = (w.px1 - w.px0 + 1) * (w.py1 - w.py0 + 1);   // below 2^28
            if (box > kWideBox || (box > kWaveBox && (float)box > kSliver * w.size)) {
                vis[(size_t)ci * d.T + t] = kWide;
                *wide_flag = 1u;   // every writer stores the same value
            }
        }
    }
}

// Id and depth of a key (0 and 0 for a pixel without a triangle).
__device__ __forceinline__ void key_parts(unsigned long long k, int& id, float& depth)
{
    id = k == ~0ull ? 0 : (int)(0xFFFFFFFEu - (uint32_t)k);
    depth = k == ~0ull ? 0.0f : __uint_as_float(~(uint32_t)(k >> 32));
}

__global__ __launch_bounds__(kBlock) void keys_to_ids_kernel(const unsigned long long* __restrict__ keys, size_t n,
                                                              int* __restrict__ ids, float* __restrict__ depth)
{
    const size_t p = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (p >= n) return;
    int id;
    float dep;
    key_parts(keys[p], id, dep);
    ids[p] = id;
    depth[p] = dep;
}

// ---------------------------------------------------------------------------
// Interpolation and antialiasing, templated on the type C of the clip
// positions (and of their gradient) and the type R of attributes, images,
// their gradients and the arithmetic.  (C, R) = (float, float), (double,
// double), or (double, float): the pixel-relative offsets that the results
// are ill-conditioned in (u below, the screen offsets of the antialiasing)
// are formed in C and then rounded to R.  The raster above always works on
// float clip positions.
template <typename T> __device__ __forceinline__ V4<T> load_clip4(const T* clip, const Dims& d, int c, int i, int v)
{
    return reinterpret_cast<const V4<T>*>(clip)[((size_t)c * d.I + i) * d.V + v];
}

template <typename T> __device__ __forceinline__ T cross2(V2<T> a, V2<T> b) { return a.x * b.y - a.y * b.x; }

template <typename T> __device__ __forceinline__ T ndc_x(int px, const Dims& d)
{
    return (T(px) + T(0.5)) / (T(d.W) * T(0.5)) - T(1);
}
template <typename T> __device__ __forceinline__ T ndc_y(int py, const Dims& d)
{
    return (T(py) + T(0.5)) / (T(d.H) * T(0.5)) - T(1);
}

// Barycentrics at a pixel centre from the clip positions of a triangle.
template <typename R> struct Bary {
    V2<R> u[3];    // pixel-relative (x - xn w, y - yn w) per vertex
    R l[3], S;
    R lam[3];
    int v[3];
};

// An id outside 1..I*T or a vertex index outside 0..V-1 makes the pixel
// background: no read leaves the buffers whatever the caller's ids and tris.
__device__ __forceinline__ bool id_in_range(int id, const Dims& d) { return id > 0 && id <= d.I * d.T; }
__device__ __forceinline__ bool vertex_in_range(int v, const Dims& d) { return (unsigned)v < (unsigned)d.V; }

template <typename C, typename R>
__device__ __forceinline__ void bary_from(const V4<C> P[3], C xn, C yn, Bary<R>& b)
{
    for (int k = 0; k < 3; ++k) b.u[k] = V2<R>{ R(fma(-xn, P[k].w, P[k].x)), R(fma(-yn, P[k].w, P[k].y)) };
    for (int k = 0; k < 3; ++k) b.l[k] = cross2(b.u[(k + 1) % 3], b.u[(k + 2) % 3]);
    b.S = (b.l[0] + b.l[1]) + b.l[2];
    const R inv = R(1) / b.S;
    for (int k = 0; k < 3; ++k) b.lam[k] = b.l[k] * inv;
}

// The triangle of an in-range id: its instance, vertices (false when one is
// out of range) and clip positions.
template <typename C>
__device__ __forceinline__ bool tri_of(const C* clip, const int* tris, const Dims& d, int c, int id, int& i, int& t,
                                       int vi[3], V4<C> P[3])
{
    i = (id - 1) / d.T;
    t = (id - 1) % d.T;
    for (int k = 0; k < 3; ++k) {
        vi[k] = tris[3 * t + k];
        if (!vertex_in_range(vi[k], d)) return false;
    }
    for (int k = 0; k < 3; ++k) P[k] = load_clip4(clip, d, c, i, vi[k]);
    return true;
}

template <typename C, typename R>
__device__ __forceinline__ bool bary_at(const C* clip, const int* tris, const Dims& d, int c, int id, int px, int py,
                                        Bary<R>& b)
{
    if (!id_in_range(id, d)) return false;
    int i, t;
    V4<C> P[3];
    if (!tri_of(clip, tris, d, c, id, i, t, b.v, P)) return false;
    bary_from(P, ndc_x<C>(px, d), ndc_y<C>(py, d), b);
    return true;
}

// ---------------------------------------------------------------------------
// Gathers.  The backward of interpolation and antialiasing runs in two
// passes.  A pixel pass computes, with every lane busy, each pixel's terms
// for the three corners of its triangle (plain stores, contrib).  A vertex
// pass, a few lanes per vertex, walks the vertex's
// incident triangles (a CSR adjacency of the mesh) and sums the terms of the
// pixels in each triangle's screen box that carry the triangle's id.  No
// atomics, and the sums run in a fixed order: the gradients are the same
// bits on every run.
//
// The box holds every pixel whose centre lies in the triangle, with a margin
// of 1/64 px over the raster's 1/256-px snapping, so rasterize's ids always
// fall inside it.  A pixel outside its own triangle's box (ids from
// elsewhere), or of a triangle that is not gathered (a vertex at w <= 0 or not
// finite, a repeated vertex, or a box over kGatherMaxBox pixels), is a stray.
// The forwards flag each block of pixels that holds a stray; the backwards
// scatter those pixels' terms with atomics after the vertex pass, in a pass
// that skips unflagged blocks.
constexpr int kGatherMaxBox = 64;
constexpr int kPixBatch = 4;      // box pixels whose ids are loaded together

// Index of (camera c, the instance and triangle of in-range id) in boxes and vis.
__device__ __forceinline__ size_t tri_index(const Dims& d, int c, int id)
{
    return (size_t)c * d.I * d.T + (size_t)(id - 1);
}

__device__ __forceinline__ bool finite_coord(float x) { return fabsf(x) < 1e30f; }

// The box, in float whatever C (the raster snaps float clip positions): the
// hardware reciprocal's error (1 ulp) is far inside the margin.
template <typename C>
__device__ __forceinline__ bool gather_box(const V4<C> P[3], const int vi[3], const Dims& d, Box& b)
{
    if (vi[0] == vi[1] || vi[1] == vi[2] || vi[0] == vi[2]) return false;
    const float hw = (float)d.W * 0.5f, hh = (float)d.H * 0.5f;
    float mnx = 0.0f, mxx = 0.0f, mny = 0.0f, mxy = 0.0f;
    for (int k = 0; k < 3; ++k) {
        const float w = (float)P[k].w;
        if (!(w > 0.0f)) return false;
        // pixel coordinates: the centre of pixel (px, py) is at (px, py)
        const float r = __builtin_amdgcn_rcpf(w);
        const float sx = fmaf((float)P[k].x * r, hw, hw - 0.5f), sy = fmaf((float)P[k].y * r, hh, hh - 0.5f);
        if (!(finite_coord(sx) && finite_coord(sy))) return false;
        mnx = k ? fminf(mnx, sx) : sx;
        mxx = k ? fmaxf(mxx, sx) : sx;
        mny = k ? fminf(mny, sy) : sy;
        mxy = k ? fmaxf(mxy, sy) : sy;
    }
    const float margin = 1.0f / 64.0f;
    const float fx0 = fmaxf(ceilf(mnx - margin), 0.0f), fx1 = fminf(floorf(mxx + margin), (float)(d.W - 1));
    const float fy0 = fmaxf(ceilf(mny - margin), 0.0f), fy1 = fminf(floorf(mxy + margin), (float)(d.H - 1));
    if (fx0 > fx1 || fy0 > fy1) {   // on no pixel
        b = Box{ 1, 0, 1, 0 };
        return true;
    }
    if ((fx1 - fx0 + 1.0f) * (fy1 - fy0 + 1.0f) > (float)kGatherMaxBox) return false;
    b = Box{ (int)fx0, (int)fx1, (int)fy0, (int)fy1 };
    return true;
}

// One thread per (camera, instance, triangle).
// Also clears vis, the per-triangle flags that the forward's pixel pass sets
// for the triangles with a gathered pixel, and the nflags stray flags.
template <typename C>
__global__ __launch_bounds__(kBlock) void tri_boxes_kernel(const C* __restrict__ clip, const int* __restrict__ tris,
                                                            Dims d, unsigned long long* __restrict__ boxes,
                                                            uint8_t* __restrict__ vis, unsigned* __restrict__ flags,
                                                            size_t nflags)
{
    const size_t g = (size_t)blockIdx.x * kBlock + threadIdx.x;
    const size_t n = (size_t)d.C * d.I * d.T;
    if (g < nflags) flags[g] = 0u;
    if (g >= n) return;
    const int t = (int)(g % d.T);
    const size_t ci = g / d.T;
    const int c = (int)(ci / d.I), i = (int)(ci % d.I);
    int ii, tt, vi[3];
    V4<C> P[3];
    Box b;
    const bool ok = tri_of(clip, tris, d, c, i * d.T + t + 1, ii, tt, vi, P) && gather_box(P, vi, d, b);
    boxes[g] = ok ? pack_box(b) : kNoBox;
    vis[g] = 0;
}

// Whether pixel (px, py) of camera c with id `id` is a stray (false for
// background).
__device__ __forceinline__ bool pixel_stray(const unsigned long long* boxes, const Dims& d, int c, int id, int px,
                                            int py)
{
    if (!id_in_range(id, d)) return false;
    const unsigned long long v = boxes[tri_index(d, c, id)];
    if (v == kNoBox) return true;
    const Box b = unpack_box(v);
    return !(px >= b.x0 && px <= b.x1 && py >= b.y0 && py <= b.y1);
}

// Marks pixel p of an in-range triangle `id` for the backward: its triangle as
// one with a gathered pixel, or its run of kBlock pixels as one with a stray.
// Every writer of a flag stores the same value.
__device__ __forceinline__ void mark_pixel(const unsigned long long* boxes, const Dims& d, int c, int id, int px, int py,
                                           size_t p, unsigned* __restrict__ flags, uint8_t* __restrict__ vis)
{
    if (pixel_stray(boxes, d, c, id, px, py)) flags[p / kBlock] = 1u;
    else vis[tri_index(d, c, id)] = 1;
}

// Channel a of the interpolated attributes.
template <typename R> __device__ __forceinline__ R interp_value(const Bary<R>& b, const R* attr, int A, int a)
{
    return (b.lam[0] * attr[b.v[0] * A + a] + b.lam[1] * attr[b.v[1] * A + a]) + b.lam[2] * attr[b.v[2] * A + a];
}

template <typename C, typename R>
__global__ __launch_bounds__(kBlock) void interp_fwd_kernel(const C* __restrict__ clip, const R* __restrict__ attr,
                                                             const int* __restrict__ tris, const int* __restrict__ ids,
                                                             Dims d, int A, R* __restrict__ out,
                                                             const unsigned long long* __restrict__ boxes,
                                                             unsigned* __restrict__ stray_blocks,
                                                             uint8_t* __restrict__ vis)
{
    const size_t p = (size_t)blockIdx.x * kBlock + threadIdx.x;
    const size_t npx = (size_t)d.C * d.H * d.W;
    if (p >= npx) return;
    const int id = ids[p];
    R* o = out + p * A;
    const int c = (int)(p / ((size_t)d.H * d.W)), py = (int)((p / d.W) % d.H), px = (int)(p % d.W);
    Bary<R> b;
    if (!bary_at(clip, tris, d, c, id, px, py, b)) {
        for (int a = 0; a < A; ++a) o[a] = R(0);
        return;
    }
    for (int a = 0; a < A; ++a) o[a] = interp_value(b, attr, A, a);
    mark_pixel(boxes, d, c, id, px, py, p, stray_blocks, vis);
}

// d colour / d attr_k = lambda_k; d colour / d lambda_k = attr_k;
// d lambda_k / d l_j = (delta_kj - lambda_k) / S;
// l_k = u_{k+1} x u_{k+2}: dl_k/du_{k+1} = (u_{k+2}.y, -u_{k+2}.x), dl_k/du_{k+2} = (-u_{k+1}.y, u_{k+1}.x);
// u = (x - xn w, y - yn w): dL/dx = g.x, dL/dy = g.y, dL/dw = -(xn g.x + yn g.y).
// glam: dL/dlambda_k; gl: dL/dl_k = (glam_k - sum_j glam_j lambda_j) / S.
template <typename R> __device__ __forceinline__ void lambda_grad(const Bary<R>& b, const R glam[3], R gl[3])
{
    const R dot = (glam[0] * b.lam[0] + glam[1] * b.lam[1]) + glam[2] * b.lam[2];
    const R inv = R(1) / b.S;
    for (int k = 0; k < 3; ++k) gl[k] = (glam[k] - dot) * inv;
}

// dL/du_k from dL/dl: l_{k-1} = u_k x u_{k+1} and l_{k+1} = u_{k-1} x u_k.
template <typename R> __device__ __forceinline__ V2<R> corner_grad(const Bary<R>& b, const R gl[3], int k)
{
    const int kp = (k + 1) % 3, km = (k + 2) % 3;
    return V2<R>{ gl[km] * b.u[kp].y - gl[kp] * b.u[km].y, gl[kp] * b.u[km].x - gl[km] * b.u[kp].x };
}

// The interpolation terms of pixel p (false for a background pixel): per
// corner k, (dL/dx, dL/dy, dL/dw) of its clip position and lambda_k g_out.
template <typename C, typename R> struct InterpTerms {
    Bary<R> b;
    V2<R> gu[3];
    R gw[3];
};

// o.b set: the rest, from dL/dlambda.
template <typename C, typename R>
__device__ __forceinline__ void interp_terms_of(const R glam[3], R xn, R yn, InterpTerms<C, R>& o)
{
    R gl[3];
    lambda_grad(o.b, glam, gl);
    for (int k = 0; k < 3; ++k) {
        o.gu[k] = corner_grad(o.b, gl, k);
        o.gw[k] = -(xn * o.gu[k].x + yn * o.gu[k].y);
    }
}

template <typename C, typename R>
__device__ __forceinline__ bool interp_terms(const C* clip, const R* attr, const int* tris, const Dims& d, int A,
                                             int c, int id, int px, int py, const R* go, InterpTerms<C, R>& o)
{
    if (!bary_at(clip, tris, d, c, id, px, py, o.b)) return false;
    R glam[3] = { R(0), R(0), R(0) };
    for (int a = 0; a < A; ++a)
        for (int k = 0; k < 3; ++k) glam[k] += go[a] * attr[o.b.v[k] * A + a];
    interp_terms_of(glam, ndc_x<R>(px, d), ndc_y<R>(py, d), o);
    return true;
}

// Pixel pass: contrib[p][k] = (dL/dx, dL/dy, dL/dw, lambda_k g_out[p][0..A-1]).
template <typename C, typename R>
__global__ __launch_bounds__(kBlock) void interp_bwd_pixel_kernel(const C* __restrict__ clip,
                                                                   const R* __restrict__ attr,
                                                                   const int* __restrict__ tris,
                                                                   const int* __restrict__ ids, Dims d, int A,
                                                                   const R* __restrict__ g_out,
                                                                   R* __restrict__ contrib)
{
    const size_t p = (size_t)blockIdx.x * kBlock + threadIdx.x;
    const size_t npx = (size_t)d.C * d.H * d.W;
    if (p >= npx) return;
    const int c = (int)(p / ((size_t)d.H * d.W)), py = (int)((p / d.W) % d.H), px = (int)(p % d.W);
    const R* go = g_out + p * A;
    InterpTerms<C, R> it;
    if (!interp_terms(clip, attr, tris, d, A, c, ids[p], px, py, go, it)) return;
    R* o = contrib + p * 3 * (3 + A);
    for (int k = 0; k < 3; ++k) {
        R* ok = o + k * (3 + A);
        ok[0] = it.gu[k].x;
        ok[1] = it.gu[k].y;
        ok[2] = it.gw[k];
        for (int a = 0; a < A; ++a) ok[3 + a] = it.b.lam[k] * go[a];
    }
}

// The stray pass: a stray pixel's whole interpolation gradient, with atomics.
template <typename C, typename R>
__global__ __launch_bounds__(kBlock) void interp_bwd_stray_kernel(const C* __restrict__ clip,
                                                                   const R* __restrict__ attr,
                                                                   const int* __restrict__ tris,
                                                                   const int* __restrict__ ids, Dims d, int A,
                                                                   const R* __restrict__ g_out,
                                                                   const unsigned long long* __restrict__ boxes,
                                                                   const unsigned* __restrict__ stray_blocks,
                                                                   C* __restrict__ g_clip, R* __restrict__ g_attr)
{
    if (stray_blocks[blockIdx.x] == 0u) return;   // uniform over the block
    const size_t p = (size_t)blockIdx.x * kBlock + threadIdx.x;
    const size_t npx = (size_t)d.C * d.H * d.W;
    if (p >= npx) return;
    const int id = ids[p];
    const int c = (int)(p / ((size_t)d.H * d.W)), py = (int)((p / d.W) % d.H), px = (int)(p % d.W);
    if (!pixel_stray(boxes, d, c, id, px, py)) return;
    const R* go = g_out + p * A;
    InterpTerms<C, R> it;
    if (!interp_terms(clip, attr, tris, d, A, c, id, px, py, go, it)) return;
    const int i = (id - 1) / d.T;
    for (int k = 0; k < 3; ++k) {
        for (int a = 0; a < A; ++a) atomicAdd(&g_attr[it.b.v[k] * A + a], it.b.lam[k] * go[a]);
        C* g = g_clip + (((size_t)c * d.I + i) * d.V + it.b.v[k]) * 4;
        atomicAdd(&g[0], C(it.gu[k].x));
        atomicAdd(&g[1], C(it.gu[k].y));
        atomicAdd(&g[3], C(it.gw[k]));
    }
}

// The sums of a vertex in one camera-instance pair: dL/d(x, y, w) of its clip
// position and dL/d its attributes.
template <typename C, typename R, int NA> struct VertexSum {
    C x, y, w;
    R a[NA ? NA : kMaxAttr];
};

// NA: the attribute count, 0 for a count only known at run time (at most kMaxAttr).
#define VKGV_CHANNELS(a) _Pragma("unroll") for (int a = 0; a < (NA ? NA : kMaxAttr); ++a) if (NA || a < A)

template <typename C, typename R, int NA>
__device__ __forceinline__ void sum_clear(VertexSum<C, R, NA>& s)
{
    s.x = s.y = s.w = C(0);
#pragma unroll
    for (int a = 0; a < (NA ? NA : kMaxAttr); ++a) s.a[a] = R(0);
}

// The value of lane i's partner, i ^ 1, i ^ 2, the mirror lane of its group of
// eight, or the lane eight away in its row of 16, by a DPP move: the vector
// ALU alone (__shfl_xor goes through the LDS crossbar, which bound the vertex
// pass).
enum { kXor1 = 0xB1, kXor2 = 0x4E, kMirror8 = 0x141, kRor8 = 0x128 };
template <int CTRL> __device__ __forceinline__ float lane_move(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, true));
}
template <int CTRL> __device__ __forceinline__ double lane_move(double x)
{
    const long long b = __double_as_longlong(x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, 0xF, 0xF, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)((unsigned long long)b >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// The sum over a group of eight lanes, in each of them (every lane of the wave
// takes part): pairs, then quads, then the two quads.
template <typename T> __device__ __forceinline__ T sum8(T x)
{
    x += lane_move<kXor1>(x);
    x += lane_move<kXor2>(x);
    x += lane_move<kMirror8>(x);
    return x;
}

template <typename C, typename R, int NA> __device__ __forceinline__ void sum8(VertexSum<C, R, NA>& s, int A)
{
    s.x = sum8(s.x);
    s.y = sum8(s.y);
    s.w = sum8(s.w);
    VKGV_CHANNELS(a) s.a[a] = sum8(s.a[a]);
}

// The sum over the wave, in each lane.
template <typename T> __device__ __forceinline__ T sum64(T x)
{
    x = sum8(x);
    x += lane_move<kRor8>(x);
    x += __shfl_xor(x, 16, 64);
    x += __shfl_xor(x, 32, 64);
    return x;
}

// Adds pixel p's record of corner k: contrib[p][k][n], n = 3 + A values with
// the attributes' (ATTR), 3 without.
template <typename C, typename R, int NA, bool ATTR>
__device__ __forceinline__ void add_record(const R* contrib, size_t p, int k, int A, VertexSum<C, R, NA>& s)
{
    const R* o = contrib + (p * 3 + k) * (ATTR ? 3 + A : 3);
    if (ATTR && NA == 3) {   // six values by as few loads as there are: the lanes' records lie apart
        struct alignas(2 * sizeof(R)) Six {
            R v[6];
        };
        const Six r = *reinterpret_cast<const Six*>(o);
        s.x += C(r.v[0]);
        s.y += C(r.v[1]);
        s.w += C(r.v[2]);
        s.a[0] += r.v[3];
        s.a[1 % (NA ? NA : 2)] += r.v[4];
        s.a[2 % (NA ? NA : 3)] += r.v[5];
        return;
    }
    s.x += C(o[0]);
    s.y += C(o[1]);
    s.w += C(o[2]);
    if (ATTR) {
        VKGV_CHANNELS(a) s.a[a] += o[3 + a];
    }
}

// One lane sums the records of the pixels of box b that carry id, kPixBatch
// ids at a time in flight.  base: the camera's first pixel.  The triangle has
// a pixel in the box, so that a box of one needs no look at its id.
template <typename C, typename R, int NA, bool ATTR>
__device__ __forceinline__ void walk_box(const int* ids, size_t base, int W, const Box& b, int id, int k,
                                         const R* contrib, int A, VertexSum<C, R, NA>& s)
{
    const int bw = b.x1 - b.x0 + 1, n = bw * (b.y1 - b.y0 + 1);
    int qx = b.x0, qy = b.y0;
    if (n == 1) {
        add_record<C, R, NA, ATTR>(contrib, base + (size_t)qy * W + qx, k, A, s);
        return;
    }
    for (int q0 = 0; q0 < n; q0 += kPixBatch) {
        size_t ip[kPixBatch];
        int idq[kPixBatch];
#pragma unroll
        for (int w = 0; w < kPixBatch; ++w) {
            ip[w] = base + (size_t)qy * W + qx;
            idq[w] = q0 + w < n ? ids[ip[w]] : 0;
            if (++qx > b.x1) {
                qx = b.x0;
                ++qy;
            }
        }
#pragma unroll
        for (int w = 0; w < kPixBatch; ++w)
            if (idq[w] == id) add_record<C, R, NA, ATTR>(contrib, ip[w], k, A, s);
    }
}

// The wave sums a wide box, a pixel per lane; the total goes to lane j.
template <typename C, typename R, int NA, bool ATTR>
__device__ __forceinline__ void walk_wide(const int* ids, size_t base, int W, const Box& b, int id, int k,
                                          const R* contrib, int A, int j, VertexSum<C, R, NA>& s)
{
    const int lane = (int)(threadIdx.x & 63u), bw = b.x1 - b.x0 + 1, n = bw * (b.y1 - b.y0 + 1);
    VertexSum<C, R, NA> p;
    sum_clear(p);
    for (int q = lane; q < n; q += 64) {
        const size_t ip = base + (size_t)(b.y0 + q / bw) * W + (b.x0 + q % bw);
        if (ids[ip] == id) add_record<C, R, NA, ATTR>(contrib, ip, k, A, p);
    }
    p.x = sum64(p.x);
    p.y = sum64(p.y);
    p.w = sum64(p.w);
    VKGV_CHANNELS(a) p.a[a] = sum64(p.a[a]);
    if (lane == j) {
        s.x += p.x;
        s.y += p.y;
        s.w += p.w;
        VKGV_CHANNELS(a) s.a[a] += p.a[a];
    }
}

// Vertex passes: kVertexLanes lanes share a vertex, lane u taking incident
// triangles u, u + kVertexLanes, ... (a mesh vertex has about six), and a
// triangle without a gathered pixel (vis 0, most of them: hidden, facing away,
// between the pixel centres) costs one byte.  One lane walking all its
// triangles ran as long as the longest of 64 such walks.
constexpr int kVertexLanes = 8;   // sum8's group
constexpr int kBlockVertices = (int)kBlock / kVertexLanes;

// The vertex pass of interpolate, antialias and shade: g_clip[c, i, v]
// (written, z = 0) and, with the interpolation terms (ATTR), this
// camera-instance pair's attribute gradient part[c, i, v, A] (reduced over the
// pairs by attr_reduce_kernel).  contrib[p][k][n] as in add_record.
template <typename C, typename R, bool ATTR, int NA>
__global__ __launch_bounds__(kBlock) void vertex_gather_kernel(const int* __restrict__ ids, Dims d, int A,
                                                                const int* __restrict__ adj_off,
                                                                const int* __restrict__ adj,
                                                                const unsigned long long* __restrict__ boxes,
                                                                const uint8_t* __restrict__ vis,
                                                                const R* __restrict__ contrib, C* __restrict__ g_clip,
                                                                R* __restrict__ part)
{
    const unsigned nvb = (unsigned)((d.V + kBlockVertices - 1) / kBlockVertices);
    const int ci = (int)(blockIdx.x / nvb), u = (int)threadIdx.x % kVertexLanes;
    const int v = (int)(blockIdx.x % nvb) * kBlockVertices + (int)threadIdx.x / kVertexLanes;
    const int i = ci % d.I;
    const size_t base = (size_t)(ci / d.I) * d.H * d.W;
    const int j0 = v < d.V ? adj_off[v] : 0, j1 = v < d.V ? adj_off[v + 1] : 0;
    VertexSum<C, R, NA> s;
    sum_clear(s);
    bool any = false;
    for (int j = j0 + u; j < j1; j += kVertexLanes) {
        const int corner = adj[j], t = corner / 3;
        if (!vis[(size_t)ci * d.T + t]) continue;
        any = true;
        walk_box<C, R, NA, ATTR>(ids, base, d.W, unpack_box(boxes[(size_t)ci * d.T + t]), i * d.T + t + 1, corner - 3 * t,
                                 contrib, A, s);
    }
    if (__ballot(any) != 0ull) sum8(s, A);
    if (v >= d.V) return;
    if (u < 4) g_clip[((size_t)ci * d.V + v) * 4 + u] = u == 0 ? s.x : u == 1 ? s.y : u == 2 ? C(0) : s.w;
    if (ATTR) {
        static_assert(kVertexLanes >= kMaxAttr, "a lane writes one channel");
        VKGV_CHANNELS(a) if (u == a) part[((size_t)ci * d.V + v) * A + a] = s.a[a];
    }
}

// The vertex pass of render, which goes on through the vertex transform
// clip[ci, v] = M[ci] (p_v, 1): the clip gradient, zero for most (pair,
// vertex) entries, is never stored.  A block takes kBlockVertices vertices and
// kPairs camera-instance pairs (grid y) and writes the sums over its pairs of
// M^T g (its positions' gradient) and of the attributes' gradient to
// part_pos[y][V][3] and part_attr[y][V][A], and adds its sums over the
// vertices of g (p_v, 1)^T to g_M.  boxes: of the triangles with vis kSeen;
// what the pixel pass summed of the kWide ones, wide_pos and wide_attr, joins
// part 0.
//
// Bound by the latency of flag -> box -> ids -> records: a wave goes through
// the pairs in which any of its triangles has a pixel, the next pair's boxes in
// flight.  64 pairs of 50k vertices: 125 us, where the gather, the reduction
// over the pairs and the two passes of the vertex transform's backward over the
// stored clip gradient took 217 + 22 + 36 + 110.  With the sums over lanes
// through the LDS crossbar 142 us; each lane through its own pairs with LDS
// atomics into g_M 165 us.
constexpr int kPairs = 8;
template <typename C, typename R, int NA>
__global__ __launch_bounds__(kBlock) void vertex_render_kernel(const int* __restrict__ ids, Dims d, int A,
                                                                const C* __restrict__ pos, const C* __restrict__ M,
                                                                const int* __restrict__ adj_off,
                                                                const int* __restrict__ adj,
                                                                const unsigned long long* __restrict__ boxes,
                                                                const uint8_t* __restrict__ vis,
                                                                const R* __restrict__ contrib, C* __restrict__ part_pos,
                                                                R* __restrict__ part_attr, C* __restrict__ g_M,
                                                                const uint32_t* __restrict__ wide_flag,
                                                                const C* __restrict__ wide_pos,
                                                                const R* __restrict__ wide_attr)
{
    constexpr int kRows = (int)kBlock / 16;   // rows of 16 lanes, two vertices each
    __shared__ R2<C> s_g[kRows][kPairs][kVertexLanes];
    const int lane = (int)(threadIdx.x & 63u), row = (int)(threadIdx.x >> 4), u = lane % kVertexLanes;
    const int v = (int)blockIdx.x * kBlockVertices + (int)threadIdx.x / kVertexLanes;
    const int ci0 = (int)blockIdx.y * kPairs, np = min(kPairs, d.C * d.I - ci0);
    // a row's sums belong to its wave alone: no barrier before the end
    for (int q = u; q < kPairs * kVertexLanes; q += kVertexLanes) (&s_g[row][0][0])[q] = R2<C>{ C(0), C(0) };
    const bool live = v < d.V;
    const int j0 = live ? adj_off[v] : 0, j1 = live ? adj_off[v + 1] : 0;
    // lane u: homogeneous coordinates 2 (u & 1) and the next of its vertex
    const C h0 = live ? pos[3 * (size_t)v + (u & 1 ? 2 : 0)] : C(0);
    const C h1 = u & 1 ? C(1) : (live ? pos[3 * (size_t)v + 1] : C(0));
    C g_pos = C(0);     // lane u < 3: component u
    R g_attr = R(0);    // lane u < A: channel u
    // rounds of kVertexLanes triangles; the sums are linear in them
    for (int r = 0; __ballot(j0 + r < j1) != 0ull; r += kVertexLanes) {
        const int j = j0 + r + u;
        const int corner = j < j1 ? adj[j] : -1, t = corner / 3, k = corner - 3 * t;
        uint32_t seen = 0u;     // bit q: the triangle has a gathered pixel in pair ci0 + q
#pragma unroll
        for (int q = 0; q < kPairs; ++q)
            if (corner >= 0 && q < np && vis[(size_t)(ci0 + q) * d.T + t] == kSeen) seen |= 1u << q;
        uint32_t pairs = 0u;    // of any lane of the wave
#pragma unroll
        for (int q = 0; q < kPairs; ++q)
            if (__ballot((seen >> q) & 1u) != 0ull) pairs |= 1u << q;
        auto box_of = [&](int q) {
            return (seen >> q) & 1u ? boxes[(size_t)(ci0 + q) * d.T + t] : 1ull;   // 1: an empty box
        };
        unsigned long long next = pairs ? box_of(__ffs((int)pairs) - 1) : 1ull;
        while (pairs) {   // wave-uniform
            const int q = __ffs((int)pairs) - 1;
            const Box b = unpack_box(next);
            pairs &= pairs - 1u;
            if (pairs) next = box_of(__ffs((int)pairs) - 1);
            const int ci = ci0 + q, i = ci % d.I, id = i * d.T + t + 1;
            const size_t base = (size_t)(ci / d.I) * d.H * d.W;
            VertexSum<C, R, NA> s;
            sum_clear(s);
            const bool mine = (seen >> q) & 1u, wide = mine && (b.x1 - b.x0 + 1) * (b.y1 - b.y0 + 1) > kWaveBox;
            if (mine && !wide) walk_box<C, R, NA, true>(ids, base, d.W, b, id, k, contrib, A, s);
            unsigned long long pending = __ballot(wide);
            while (pending != 0ull) {
                const int l = __ffsll((long long)pending) - 1;
                pending &= pending - 1ull;
                const Box wb{ __builtin_amdgcn_readlane(b.x0, l), __builtin_amdgcn_readlane(b.x1, l),
                              __builtin_amdgcn_readlane(b.y0, l), __builtin_amdgcn_readlane(b.y1, l) };
                walk_wide<C, R, NA, true>(ids, base, d.W, wb, __builtin_amdgcn_readlane(id, l),
                                          __builtin_amdgcn_readlane(k, l), contrib, A, l, s);
            }
            sum8(s, A);
            const C* m = M + (size_t)ci * 16;
            const int c = u < 3 ? u : 0;
            g_pos += (m[c] * s.x + m[4 + c] * s.y) + m[12 + c] * s.w;
            VKGV_CHANNELS(a) if (u == a) g_attr += s.a[a];
            // g_M[row][col] += g_row (p, 1)_col: lane u of each vertex forms row u / 2, columns 2 (u & 1)
            // and the next, summed over the row's two vertices
            const C gr = (u >> 1) == 0 ? s.x : (u >> 1) == 1 ? s.y : (u >> 1) == 2 ? C(0) : s.w;
            C e0 = gr * h0, e1 = gr * h1;
            e0 += lane_move<kRor8>(e0);
            e1 += lane_move<kRor8>(e1);
            if ((lane & 8) == 0) {
                R2<C>& g = s_g[row][q][u];
                g.x += e0;
                g.y += e1;
            }
        }
    }
    if (live) {
        if (blockIdx.y == 0 && *wide_flag != 0u) {
            if (u < 3) g_pos += wide_pos[(size_t)v * 3 + u];
            VKGV_CHANNELS(a) if (u == a) g_attr += wide_attr[(size_t)v * A + a];
        }
        if (u < 3) part_pos[((size_t)blockIdx.y * d.V + v) * 3 + u] = g_pos;
        VKGV_CHANNELS(a) if (u == a) part_attr[((size_t)blockIdx.y * d.V + v) * A + a] = g_attr;
    }
    __syncthreads();
    for (int k = (int)threadIdx.x; k < np * 16; k += (int)kBlock) {
        C t = C(0);
        for (int w = 0; w < kRows; ++w) t += reinterpret_cast<const C*>(&s_g[w][k >> 4][0])[k & 15];
        if (t != C(0)) unsafeAtomicAdd(&g_M[(size_t)ci0 * 16 + k], t);
    }
}

// g_attr[v, a] = sum over the camera-instance pairs of part[ci, v, a], in pair order.
template <typename R>
__global__ __launch_bounds__(kBlock) void attr_reduce_kernel(const R* __restrict__ part, int CI, size_t VA,
                                                              R* __restrict__ g_attr)
{
    const size_t j = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (j >= VA) return;
    R s = R(0);
    for (int ci = 0; ci < CI; ++ci) s += part[(size_t)ci * VA + j];
    g_attr[j] = s;
}

// Sums of `parts` arrays a[.][na] and b[.][nb], in part order.
template <typename C, typename R>
__global__ __launch_bounds__(kBlock) void part_reduce_kernel(const C* __restrict__ a, size_t na, C* __restrict__ out_a,
                                                              const R* __restrict__ b, size_t nb, R* __restrict__ out_b,
                                                              int parts)
{
    const size_t j = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (j < na) {
        C s = C(0);
        for (int p = 0; p < parts; ++p) s += a[(size_t)p * na + j];
        out_a[j] = s;
    } else if (j < na + nb) {
        R s = R(0);
        for (int p = 0; p < parts; ++p) s += b[(size_t)p * nb + (j - na)];
        out_b[j - na] = s;
    }
}

// ---------------------------------------------------------------------------
// Antialiasing.  A pair is (p, q) with q the right (dir 0) or lower (dir 1)
// neighbour.  pair_eval returns false when the pair does not blend; else the
// target pixel, alpha, and what the backward needs.  Screen positions are
// taken relative to the front pixel's centre (the back centre is then one
// unit step away), which keeps the edge functions exact to the rounding of
// the small offsets rather than of the screen size.
template <typename R> struct PairEval {
    size_t f, bpx;          // front and back pixel indices
    bool to_front;          // blend into the front pixel (t < 1/2) or the back one
    R t, alpha;
    int i, va, vb;          // instance and the crossed edge's vertices
    int ka;                 // corner of the front triangle at va (vb is the next one)
    R ef, eb;               // edge functions at the two centres
    V2<R> sa, sb;           // screen offsets of the edge's vertices from the front centre
    V2<R> cb;               // back centre relative to the front one (a unit step)
    V4<R> pa, pb;           // clip positions of the edge's vertices
};

// hw (x / w - xc), hh (y / w - yc): screen offset in pixels from the centre
// with NDC (xc, yc), formed in C and rounded to R
template <typename C, typename R> __device__ __forceinline__ V2<R> screen_rel(V4<C> p, C xc, C yc, const Dims& d)
{
    const C hw = C(d.W) * C(0.5), hh = C(d.H) * C(0.5);
    return V2<R>{ R(hw * (fma(-xc, p.w, p.x) / p.w)), R(hh * (fma(-yc, p.w, p.y) / p.w)) };
}

template <typename R> __device__ __forceinline__ R edge_fn(V2<R> a, V2<R> b, V2<R> p)
{
    return (b.x - a.x) * (p.y - a.y) - (b.y - a.y) * (p.x - a.x);
}

// The triangle of a front pixel, seen from its centre: screen offsets of the
// vertices, orientation (interior on the positive side of every edge k, k+1)
// and the edge functions at the centre.  False for a triangle that blends no
// pair.  It depends on the pixel alone: the pixel's pairs share it.
template <typename R> struct FrontTri {
    V2<R> S[3];
    R sgn, ef[3];
};

template <typename C, typename R>
__device__ __forceinline__ bool front_tri(const V4<C> P[3], C xc, C yc, const Dims& d, FrontTri<R>& f)
{
    for (int k = 0; k < 3; ++k) {
        if (!(P[k].w > C(0))) return false;
        f.S[k] = screen_rel<C, R>(P[k], xc, yc, d);
    }
    const R area = edge_fn(f.S[0], f.S[1], f.S[2]);
    if (area == R(0)) return false;
    f.sgn = area > R(0) ? R(1) : R(-1);
    const V2<R> zero{ R(0), R(0) };
    for (int k = 0; k < 3; ++k) f.ef[k] = f.sgn * edge_fn(f.S[k], f.S[(k + 1) % 3], zero);
    return true;
}

// The first edge of the front triangle that the segment from the front centre
// to the back one (cb from it) leaves through: its first corner (-1: none),
// the parameter and the edge function at the back centre.
template <typename R> __device__ __forceinline__ int front_cross(const FrontTri<R>& f, V2<R> cb, R& t, R& eb)
{
    t = R(2);
    eb = R(0);
    int kb = -1;
    for (int k = 0; k < 3; ++k) {
        const R ebk = f.sgn * edge_fn(f.S[k], f.S[(k + 1) % 3], cb);
        if (!(f.ef[k] >= R(0) && ebk <= R(0) && f.ef[k] > ebk)) continue;
        const R tt = f.ef[k] / (f.ef[k] - ebk);
        if (tt < t) { t = tt; kb = k; eb = ebk; }
    }
    return kb;
}

// The k-th of three values, k known only at run time.  Scalars by value: a
// record picked through its address is placed in scratch memory.
template <typename T> __device__ __forceinline__ T pick3(T a, T b, T c, int k) { return k == 0 ? a : k == 1 ? b : c; }
template <typename T> __device__ __forceinline__ T pick3(const T (&x)[3], int k) { return pick3(x[0], x[1], x[2], k); }
template <typename R> __device__ __forceinline__ V2<R> pick3(const V2<R> (&v)[3], int k)
{
    return V2<R>{ pick3(v[0].x, v[1].x, v[2].x, k), pick3(v[0].y, v[1].y, v[2].y, k) };
}
// The k-th clip position rounded to R.
template <typename C, typename R> __device__ __forceinline__ V4<R> pick_clip(const V4<C> (&P)[3], int k)
{
    return V4<R>{ pick3(R(P[0].x), R(P[1].x), R(P[2].x), k), pick3(R(P[0].y), R(P[1].y), R(P[2].y), k),
                  pick3(R(P[0].z), R(P[1].z), R(P[2].z), k), pick3(R(P[0].w), R(P[1].w), R(P[2].w), k) };
}

// The blend of a pair whose front pixel holds the triangle with vertices vi
// and clip positions P of instance i: every field of e but f and bpx.
template <typename C, typename R>
__device__ __forceinline__ bool front_eval(const V4<C> (&P)[3], const int (&vi)[3], int i, const FrontTri<R>& f, V2<R> cb,
                                           PairEval<R>& e)
{
    R best, beb;
    const int kb = front_cross(f, cb, best, beb);
    if (kb < 0) return false;
    const int kn = kb == 2 ? 0 : kb + 1;
    e.cb = cb;
    e.i = i;
    e.t = best;
    e.to_front = best < R(0.5);
    e.alpha = e.to_front ? R(0.5) - best : best - R(0.5);
    e.ka = kb;
    e.va = pick3(vi, kb);
    e.vb = pick3(vi, kn);
    e.pa = pick_clip<C, R>(P, kb);
    e.pb = pick_clip<C, R>(P, kn);
    e.sa = pick3(f.S, kb);
    e.sb = pick3(f.S, kn);
    e.ef = f.sgn * pick3(f.ef, kb);      // unsigned-orientation values, re-signed in the backward
    e.eb = f.sgn * beb;
    return true;
}

// The front pixel of pair (a, b), b the right (dir 0) or lower (dir 1)
// neighbour of a, given their ids (0 when out of range) with ida != idb:
// the one with an id, else the one with the larger depth (a on ties).
__device__ __forceinline__ bool a_is_front(int ida, int idb, float da, float db)
{
    if (ida == 0) return false;
    if (idb == 0) return true;
    return da >= db;
}

template <typename C, typename R>
__device__ bool pair_eval(const C* clip, const int* tris, const int* ids, const float* depth, const Dims& d, int c,
                          int px, int py, int dir, PairEval<R>& e)
{
    const int qx = px + (dir == 0), qy = py + (dir == 1);
    if (qx >= d.W || qy >= d.H) return false;
    const size_t base = (size_t)c * d.H * d.W;
    const size_t ip = base + (size_t)py * d.W + px, iq = base + (size_t)qy * d.W + qx;
    const int idp = id_in_range(ids[ip], d) ? ids[ip] : 0, idq = id_in_range(ids[iq], d) ? ids[iq] : 0;
    if (idp == idq) return false;
    const bool p_front = a_is_front(idp, idq, depth[ip], depth[iq]);
    e.f = p_front ? ip : iq;
    e.bpx = p_front ? iq : ip;
    const int idf = p_front ? idp : idq;
    const int fx = p_front ? px : qx, fy = p_front ? py : qy;
    const R step = p_front ? R(1) : R(-1);
    const V2<R> cb = dir == 0 ? V2<R>{ step, R(0) } : V2<R>{ R(0), step };
    const int i = (idf - 1) / d.T, t = (idf - 1) % d.T;
    int vi[3];
    for (int k = 0; k < 3; ++k) {
        vi[k] = tris[3 * t + k];
        if (!vertex_in_range(vi[k], d)) return false;
    }
    V4<C> P[3];
    for (int k = 0; k < 3; ++k) P[k] = load_clip4(clip, d, c, i, vi[k]);
    FrontTri<R> f;
    return front_tri<C, R>(P, ndc_x<C>(fx, d), ndc_y<C>(fy, d), d, f) && front_eval<C, R>(P, vi, i, f, cb, e);
}

// The four pairs of pixel (px, py), as (a, dir) with b the right (dir 0) or
// lower (dir 1) neighbour of a: (p, right), (left, p), (p, down), (up, p).
__device__ __forceinline__ bool pair_of(int q, int px, int py, int& ax, int& ay, int& dir)
{
    ax = q == 1 ? px - 1 : px;
    ay = q == 3 ? py - 1 : py;
    dir = q >> 1;
    return ax >= 0 && ay >= 0;
}

// ---------------------------------------------------------------------------
// The pixel passes of the antialiasing.  A block of 32x16 threads takes as
// many pixels, the outer ring of which only serves its 30x14 inner ones: each
// thread evaluates the triangle of its pixel once (three vertices, six
// divisions, in the clip type) and crosses it with the up to four pairs it is
// the front of; the blends go to LDS, and an inner pixel takes those of its own
// pairs and of its neighbours'.  (One thread per pixel evaluating all four of
// its pairs did the triangle work up to four times a pixel, and again for the
// neighbours that are in front.)  shade's forward also interpolates here and
// its backward goes on through the interpolation, so that the colour gradient
// and the edge terms stay in registers.  18 % of the threads are ring.  Bound
// by the gathers of clip positions and the divisions: 8 views of 512x512 of a
// 100k-triangle mesh as 8 instances, float64 clip: forward 53 us (interpolation and
// antialiasing apart: 44 + 118), backward 106 us (107 + 242).
constexpr int kTileW = 32, kTileH = 16, kTileThreads = kTileW * kTileH;
constexpr int kInnerW = kTileW - 2, kInnerH = kTileH - 2;

struct TilePixel {
    int c, x, y;
    bool in, inner;     // in the image; one of the block's inner pixels
    size_t p;           // index (0 outside the image)
};

__device__ __forceinline__ TilePixel tile_pixel(const Dims& d)
{
    const unsigned tw = (unsigned)((d.W + kInnerW - 1) / kInnerW), th = (unsigned)((d.H + kInnerH - 1) / kInnerH);
    const unsigned col = blockIdx.x % tw, rest = blockIdx.x / tw, row = rest % th;
    const int tx = (int)threadIdx.x % kTileW, ty = (int)threadIdx.x / kTileW;
    TilePixel t;
    t.c = (int)(rest / th);
    t.x = (int)col * kInnerW + tx - 1;
    t.y = (int)row * kInnerH + ty - 1;
    t.in = t.x >= 0 && t.y >= 0 && t.x < d.W && t.y < d.H;
    t.inner = t.in && tx > 0 && ty > 0 && tx < kTileW - 1 && ty < kTileH - 1;
    t.p = t.in ? ((size_t)t.c * d.H + t.y) * d.W + t.x : 0;
    return t;
}

inline unsigned tile_blocks(const Dims& d)
{
    return (unsigned)(((d.W + kInnerW - 1) / kInnerW) * ((d.H + kInnerH - 1) / kInnerH)) * (unsigned)d.C;
}

// Directions: right, left, down, up (the order a pixel's blends are summed
// in); q ^ 1 is the opposite one.
__device__ __forceinline__ int dir_x(int q) { return q == 0 ? 1 : q == 1 ? -1 : 0; }
__device__ __forceinline__ int dir_y(int q) { return q == 2 ? 1 : q == 3 ? -1 : 0; }
__device__ __forceinline__ int dir_thread(int q) { return dir_x(q) + kTileW * dir_y(q); }

// A blend in LDS: alpha, the sign telling the target (0 the front pixel, 1
// the back one), NaN for none.
__device__ __forceinline__ bool blend_to_back(float v) { return __float_as_uint(v) >> 31; }
__device__ __forceinline__ bool blend_to_back(double v) { return __double_as_longlong(v) < 0; }
template <typename R> __device__ __forceinline__ R blend_none() { return R(__builtin_nanf("")); }

// What the pixel passes share: ids (-1 outside the image, 0 background or out
// of range) and depths of the block's pixels, and the blends of each pixel as
// the front of its pairs.
template <typename R> struct TileState {
    int id[kTileThreads];
    float depth[kTileThreads];
    R blend[4][kTileThreads];

    // Whether the pixel of thread t, with id idp > 0, is the front of its
    // differing pair in direction q.
    __device__ __forceinline__ bool front(int t, int q, int idp) const
    {
        const int n = t + dir_thread(q), idn = id[n];
        if (idn < 0 || idn == idp) return false;
        return q & 1 ? !a_is_front(idn, idp, depth[n], depth[t]) : a_is_front(idp, idn, depth[t], depth[n]);
    }
};

// Forward: out = the antialiased colour.  FROM says what it starts from:
//   kFromColor  the given `color`, ids and depth;
//   kFromIds    ids and depth; the colour is interpolated here and written;
//   kFromKeys   the raster's keys of the same clip positions: ids and depth
//               are written too, no pixel can be a stray, and the bytes of
//               triangles that the raster left as kWide stay.
// The pixels are marked for the backward as interp_fwd_kernel does.
enum { kFromColor, kFromIds, kFromKeys };
template <typename C, typename R, int FROM, int NA>
__global__ __launch_bounds__(kTileThreads) void aa_fwd_kernel(R* __restrict__ color, const C* __restrict__ clip,
                                                               const R* __restrict__ attr,
                                                               const int* __restrict__ tris, int* __restrict__ ids,
                                                               float* __restrict__ depth,
                                                               const unsigned long long* __restrict__ keys, Dims d,
                                                               int A, R* __restrict__ out,
                                                               const unsigned long long* __restrict__ boxes,
                                                               unsigned* __restrict__ stray_blocks,
                                                               uint8_t* __restrict__ vis,
                                                               const uint32_t* __restrict__ wide_flag)
{
    __shared__ TileState<R> s;
    __shared__ R s_col[NA ? NA : kMaxAttr][kTileThreads];
    const int t = (int)threadIdx.x;
    const TilePixel px = tile_pixel(d);
    int id = 0;
    float dep = 0.0f;
    if (FROM == kFromKeys) {
        if (px.in) key_parts(keys[px.p], id, dep);
        if (px.inner) {
            ids[px.p] = id;
            depth[px.p] = dep;
        }
    } else if (px.in) {
        id = ids[px.p];
        dep = depth[px.p];
    }
    id = id_in_range(id, d) ? id : 0;
    s.id[t] = px.in ? id : -1;
    s.depth[t] = dep;
    if (FROM == kFromColor) {
        VKGV_CHANNELS(a) s_col[a][t] = px.in ? color[px.p * A + a] : R(0);
    }
    int i, tri, vi[3];
    V4<C> P[3];
    const bool ok = id > 0 && tri_of(clip, tris, d, px.c, id, i, tri, vi, P);
    const C xn = ndc_x<C>(px.x, d), yn = ndc_y<C>(px.y, d);
    if (FROM != kFromColor) {
        Bary<R> b;
        if (ok) {
            bary_from(P, xn, yn, b);
            for (int k = 0; k < 3; ++k) b.v[k] = vi[k];
        }
        VKGV_CHANNELS(a) {
            const R v = ok ? interp_value(b, attr, A, a) : R(0);
            s_col[a][t] = v;
            if (px.inner) color[px.p * A + a] = v;
        }
    }
    if (ok && px.inner) {
        if (FROM == kFromKeys) {
            uint8_t& seen = vis[tri_index(d, px.c, id)];
            if (*wide_flag == 0u || seen != kWide) seen = kSeen;
        } else mark_pixel(boxes, d, px.c, id, px.x, px.y, px.p, stray_blocks, vis);
    }
    __syncthreads();
    FrontTri<R> f;
    const bool fr = ok && front_tri<C, R>(P, xn, yn, d, f);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        R v = blend_none<R>();
        // the ring's pairs towards the block's outside have no thread and no use
        const int nx = t % kTileW + dir_x(q), ny = t / kTileW + dir_y(q);
        if (fr && nx >= 0 && ny >= 0 && nx < kTileW && ny < kTileH && s.front(t, q, id)) {
            R tt, eb;
            if (front_cross(f, V2<R>{ R(dir_x(q)), R(dir_y(q)) }, tt, eb) >= 0)
                v = tt < R(0.5) ? R(0.5) - tt : -(tt - R(0.5));
        }
        s.blend[q][t] = v;
    }
    __syncthreads();
    if (!px.inner) return;
    R acc[NA ? NA : kMaxAttr];
    VKGV_CHANNELS(a) acc[a] = s_col[a][t];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int n = t + dir_thread(q);
        const R own = s.blend[q][t], nb = s.blend[q ^ 1][n];
        const bool take = (own == own && !blend_to_back(own)) || (nb == nb && blend_to_back(nb));
        if (!take) continue;
        const R alpha = own == own ? own : -nb;
        VKGV_CHANNELS(a) acc[a] += alpha * (s_col[a][n] - s_col[a][t]);
    }
    VKGV_CHANNELS(a) out[px.p * A + a] = acc[a];
}

// One blend's backward.  out_tgt = c_tgt + alpha (c_src - c_tgt):
//   d/dc_tgt = (1 - alpha), d/dc_src = alpha, d/dalpha = c_src - c_tgt;
//   alpha = +-(1/2 - t), t = ef / (ef - eb), e(P) = cross(sb - sa, P - sa).
// galpha = sum over channels of g_out[tgt] (c_src - c_tgt); returns
// dL/d(x, y, w) of the crossed edge's vertices a = va and b = vb.
template <typename R> struct EdgeGrad {
    R ax, ay, aw, bx, by, bw;
};

template <typename R> __device__ __forceinline__ EdgeGrad<R> edge_grad(const PairEval<R>& e, R galpha, const Dims& d)
{
    const R gt = e.to_front ? -galpha : galpha;   // alpha = 1/2 - t or t - 1/2
    // t = ef / (ef - eb): dt/def = -eb / (ef - eb)^2, dt/deb = ef / (ef - eb)^2
    const R den = e.ef - e.eb;
    const R gef = gt * (-e.eb / (den * den)), geb = gt * (e.ef / (den * den));
    // e(P) = (bx - ax)(Py - ay) - (by - ay)(Px - ax):
    // de/dax = by - Py, de/day = Px - bx, de/dbx = Py - ay, de/dby = ax - Px
    const V2<R> A2 = e.sa, B2 = e.sb;
    R gax = R(0), gay = R(0), gbx = R(0), gby = R(0);
    const V2<R> Ps[2] = { { R(0), R(0) }, e.cb };
    const R ge[2] = { gef, geb };
    for (int k = 0; k < 2; ++k) {
        gax += ge[k] * (B2.y - Ps[k].y);
        gay += ge[k] * (Ps[k].x - B2.x);
        gbx += ge[k] * (Ps[k].y - A2.y);
        gby += ge[k] * (A2.x - Ps[k].x);
    }
    // screen offset s = (hw (x / w - xc), hh (y / w - yc)): ds/dx = hw / w, ds/dw = -hw x / w^2
    const R hw = R(d.W) * R(0.5), hh = R(d.H) * R(0.5);
    EdgeGrad<R> g;
    g.ax = gax * hw / e.pa.w;
    g.ay = gay * hh / e.pa.w;
    g.aw = -(gax * hw * e.pa.x + gay * hh * e.pa.y) / (e.pa.w * e.pa.w);
    g.bx = gbx * hw / e.pb.w;
    g.by = gby * hh / e.pb.w;
    g.bw = -(gbx * hw * e.pb.x + gby * hh * e.pb.y) / (e.pb.w * e.pb.w);
    return g;
}

template <typename R>
__device__ __forceinline__ R blend_galpha(const PairEval<R>& e, const R* color, const R* g_out, int A)
{
    const size_t tgt = e.to_front ? e.f : e.bpx, src = e.to_front ? e.bpx : e.f;
    R galpha = R(0);
    for (int a = 0; a < A; ++a) galpha += g_out[tgt * A + a] * (color[src * A + a] - color[tgt * A + a]);
    return galpha;
}

template <typename C, typename R>
__device__ __forceinline__ void add_clip_grad(C* g_clip, const Dims& d, int c, int i, int v, R gx, R gy, R gw)
{
    C* g = g_clip + (((size_t)c * d.I + i) * d.V + v) * 4;
    atomicAdd(&g[0], C(gx));
    atomicAdd(&g[1], C(gy));
    atomicAdd(&g[3], C(gw));
}

// Orders the wave's LDS accesses before and after it.
__device__ __forceinline__ void wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// What render's pixel pass needs for the kWide triangles: the flags, the mesh
// and the matrices, and the gradients it adds to (zeroed before).
template <typename C, typename R> struct WideArgs {
    const uint8_t* vis;
    const uint32_t* flag;
    const C* pos;
    const C* M;
    C* g_pos;
    C* g_M;
    R* g_attr;
};

// The sums of a tile's kWide triangles in LDS: kWideSlots of them by a hash of
// the id, then one slot a wave for the triangles that find none.
constexpr int kWideSlots = 32, kTileWaves = kTileThreads / 64;
template <typename C, typename R, int NA> struct WideTile {
    static constexpr int kSlots = kWideSlots + kTileWaves, kAttr = 3 * (NA ? NA : kMaxAttr);
    int id[kSlots];         // 0: free
    C pos[kSlots][9];       // dL/d(x, y, w) of corner 0, 1, 2
    R attr[kSlots][kAttr];  // dL/d the attributes of corner 0, 1, 2
};

// Adds a slot to the gradients through the vertex transform (g_pos = M^T g, g_M =
// g (p, 1)^T), an atomic a lane; g_M is summed in lanes 16 .. 31 (entry lane - 16)
// while the instance stays the same.
template <typename C, typename R, int NA> struct WideFlush {
    const WideArgs<C, R>& w;
    const Dims& d;
    int A, c, lane;
    int inst = -1;
    C sum_M = C(0);

    __device__ __forceinline__ void add_M()
    {
        if (inst >= 0 && lane >= 16 && lane < 32 && (lane & 12) != 8)   // row 2 (z) has none
            unsafeAtomicAdd(&w.g_M[((size_t)c * d.I + inst) * 16 + (size_t)(lane - 16)], sum_M);
        sum_M = C(0);
    }
    __device__ __forceinline__ void add(const int* tris, const WideTile<C, R, NA>& t, int slot)
    {
        const int id = t.id[slot], i = (id - 1) / d.T;
        const int* tri = tris + 3 * (size_t)(id - 1 - i * d.T);
        if (i != inst) {
            add_M();
            inst = i;
        }
        if (lane < 9) {             // corner lane / 3, component lane % 3 of its position
            const int k = lane / 3, j = lane - 3 * k;
            const C* m = w.M + ((size_t)c * d.I + i) * 16;
            const C* g = t.pos[slot] + 3 * k;
            unsafeAtomicAdd(&w.g_pos[3 * (size_t)tri[k] + j], (m[j] * g[0] + m[4 + j] * g[1]) + m[12 + j] * g[2]);
        } else if (lane >= 16 && lane < 32) {
            const int row = (lane - 16) >> 2, col = lane & 3;
            for (int k = 0; k < 3; ++k) {
                const C p = col < 3 ? w.pos[3 * (size_t)tri[k] + col] : C(1);
                sum_M += t.pos[slot][3 * k + min(row, 2)] * p;
            }
        } else if (lane >= 32 && lane < 32 + 3 * A) {   // corner (lane - 32) / A, channel (lane - 32) % A
            const int k = (lane - 32) / A, a = (lane - 32) - k * A;
            unsafeAtomicAdd(&w.g_attr[(size_t)tri[k] * A + a], t.attr[slot][lane - 32]);
        }
    }
};

// The terms of the tile's pixels on kWide triangles, to the gradients: a
// triangle's records are summed over the wave, then over the tile's waves in
// LDS.  key: the pixel's id, 0 for one that has nothing to add; o: its record.
// Every thread of the block calls it.
//
// With atomics from every wave instead of from every tile, 2000 triangles around
// one vertex in 4 views of 400x400 take 10 ms a step instead of 4.8, and 8 views
// of 512x512 of 20 triangles 2.5 instead of 1.8; the entries of g_M are what the
// atomics meet at.
template <typename C, typename R, int NA>
__device__ __forceinline__ void add_wide(const WideArgs<C, R>& w, WideTile<C, R, NA>& t, const int* tris, const Dims& d,
                                         int A, int c, int key, const R* o)
{
    using Tile = WideTile<C, R, NA>;
    const int lane = (int)(threadIdx.x & 63u), wave = (int)(threadIdx.x >> 6);
    for (int k = (int)threadIdx.x; k < kWideSlots; k += kTileThreads) t.id[k] = 0;
    for (int k = (int)threadIdx.x; k < kWideSlots * 9; k += kTileThreads) (&t.pos[0][0])[k] = C(0);
    for (int k = (int)threadIdx.x; k < kWideSlots * Tile::kAttr; k += kTileThreads) (&t.attr[0][0])[k] = R(0);
    __syncthreads();
    WideFlush<C, R, NA> flush{ w, d, A, c, lane };
    unsigned long long pending = __ballot(key != 0);
    while (pending != 0ull) {
        const int id = __builtin_amdgcn_readlane(key, __ffsll((long long)pending) - 1);
        const bool mine = key == id;
        pending &= ~__ballot(mine);
        C gp = C(0);    // lane l < 9: entry l of the slot's pos
        R ga = R(0);    // lane 32 + l: entry l of its attr
#pragma unroll 1
        for (int k = 0; k < 3; ++k) {   // not unrolled: the pixel pass keeps its registers
            const R* ok = o + k * (3 + A);
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const C s = sum64(mine ? C(ok[j]) : C(0));
                gp = lane == 3 * k + j ? s : gp;
            }
            VKGV_CHANNELS(a) {
                const R s = sum64(mine ? ok[3 + a] : R(0));
                ga = lane == 32 + k * A + a ? s : ga;
            }
        }
        int slot = (int)((uint32_t)id * 2654435761u >> 27), tries = 0;   // the hash's 5 bits
        for (; tries < 4; ++tries, slot = (slot + 1) % kWideSlots) {
            int was = 0;
            if (lane == 0) was = atomicCAS(&t.id[slot], 0, id);
            was = __builtin_amdgcn_readfirstlane(was);
            if (was == 0 || was == id) break;
        }
        if (tries < 4) {
            if (lane < 9) unsafeAtomicAdd(&t.pos[slot][lane], gp);
            if (lane >= 32 && lane < 32 + 3 * A) unsafeAtomicAdd(&t.attr[slot][lane - 32], ga);
        } else {
            slot = kWideSlots + wave;
            if (lane == 0) t.id[slot] = id;
            if (lane < 9) t.pos[slot][lane] = gp;
            if (lane >= 32 && lane < 32 + 3 * A) t.attr[slot][lane - 32] = ga;
            wave_fence();
            flush.add(tris, t, slot);
            wave_fence();
        }
    }
    __syncthreads();
    for (int slot = wave; slot < kWideSlots; slot += kTileWaves)
        if (t.id[slot] != 0) flush.add(tris, t, slot);
    flush.add_M();
}

// Pixel pass.  The colour gradient of a pixel is g_out (the identity part)
// plus its share of the blends of its four pairs, -alpha g_out[p] where it is
// the target and alpha g_out[tgt] where it is the source.  cg[k] is dL/d(x, y,
// w) of corner k of the pixel's triangle from the blends whose front pixel it
// is.  OF says what it is the backward of:
//   kAntialias  the antialiasing alone: g_color is written, and contrib[p][k]
//               = cg[k] for every pixel with an id;
//   kShade      the colour gradient goes on through the interpolation, and
//               contrib[p][k] = (its corner terms + cg[k], lambda_k
//               g_color[0..A-1]); g_color is written only where the stray pass
//               reads it;
//   kRender     the same without a stray pass; the terms of kWide triangles
//               also go to the gradients here (add_wide).
enum { kAntialias, kShade, kRender };
template <typename C, typename R, int OF, int NA>
__global__ __launch_bounds__(kTileThreads) void aa_bwd_pixel_kernel(const R* __restrict__ color,
                                                                     const C* __restrict__ clip,
                                                                     const R* __restrict__ attr,
                                                                     const int* __restrict__ tris,
                                                                     const int* __restrict__ ids,
                                                                     const float* __restrict__ depth, Dims d, int A,
                                                                     const R* __restrict__ g_out,
                                                                     const unsigned* __restrict__ stray_blocks,
                                                                     R* __restrict__ g_color, R* __restrict__ contrib,
                                                                     WideArgs<C, R> wide)
{
    __shared__ TileState<R> s;
    constexpr int kStaged = NA ? NA : 1;   // a run-time channel count reads the neighbours from memory
    __shared__ R s_col[kStaged][kTileThreads], s_g[kStaged][kTileThreads];
    __shared__ WideTile<C, R, NA> s_wide;   // unused, and so not allocated, but for kRender
    const int t = (int)threadIdx.x;
    const TilePixel px = tile_pixel(d);
    const int raw = px.in ? ids[px.p] : 0;
    const int id = id_in_range(raw, d) ? raw : 0;
    s.id[t] = px.in ? id : -1;
    s.depth[t] = px.in ? depth[px.p] : 0.0f;
    if (NA) {
        VKGV_CHANNELS(a) {
            s_col[a % kStaged][t] = px.in ? color[px.p * A + a] : R(0);
            s_g[a % kStaged][t] = px.in ? g_out[px.p * A + a] : R(0);
        }
    }
    int i, tri, vi[3];
    V4<C> P[3];
    const bool ok = id > 0 && tri_of(clip, tris, d, px.c, id, i, tri, vi, P);
    const C xn = ndc_x<C>(px.x, d), yn = ndc_y<C>(px.y, d);
    __syncthreads();
    // pixel of direction q's neighbour (in the image wherever a pair exists)
    auto pixel_at = [&](int q) { return (size_t)((long long)px.p + dir_x(q) + (long long)dir_y(q) * d.W); };
    auto col_of = [&](int th, size_t p, int a) { return NA ? s_col[a % kStaged][th] : color[p * A + a]; };
    auto g_of = [&](int th, size_t p, int a) { return NA ? s_g[a % kStaged][th] : g_out[p * A + a]; };
    FrontTri<R> f;
    const bool fr = ok && front_tri<C, R>(P, xn, yn, d, f);
    R cg[9];
    for (int k = 0; k < 9; ++k) cg[k] = R(0);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        R v = blend_none<R>();
        const int nx = t % kTileW + dir_x(q), ny = t / kTileW + dir_y(q);
        if (fr && nx >= 0 && ny >= 0 && nx < kTileW && ny < kTileH && s.front(t, q, id)) {
            PairEval<R> e;
            if (front_eval<C, R>(P, vi, i, f, V2<R>{ R(dir_x(q)), R(dir_y(q)) }, e)) {
                v = e.to_front ? e.alpha : -e.alpha;
                if (px.inner) {
                    const int n = t + dir_thread(q);
                    const size_t pn = pixel_at(q);
                    R galpha = R(0);
                    VKGV_CHANNELS(a) {
                        const R ct = e.to_front ? col_of(t, px.p, a) : col_of(n, pn, a);
                        const R cs = e.to_front ? col_of(n, pn, a) : col_of(t, px.p, a);
                        galpha += (e.to_front ? g_of(t, px.p, a) : g_of(n, pn, a)) * (cs - ct);
                    }
                    const EdgeGrad<R> g = edge_grad(e, galpha, d);
#pragma unroll
                    for (int k = 0; k < 3; ++k) {   // corner k is vertex a of the edge, or b, or neither
                        const bool isa = e.ka == k, isb = (e.ka == 2 ? 0 : e.ka + 1) == k;
                        if (isa || isb) {
                            cg[3 * k] += isa ? g.ax : g.bx;
                            cg[3 * k + 1] += isa ? g.ay : g.by;
                            cg[3 * k + 2] += isa ? g.aw : g.bw;
                        }
                    }
                }
            }
        }
        s.blend[q][t] = v;
    }
    __syncthreads();
    R* const o = contrib + px.p * 3 * (3 + A);
    // the pixel's record; false for a pixel without one
    auto record = [&]() {
        R acc[NA ? NA : kMaxAttr];
        VKGV_CHANNELS(a) acc[a] = g_of(t, px.p, a);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int n = t + dir_thread(q);
            const R own = s.blend[q][t], nb = s.blend[q ^ 1][n];
            const bool mine = own == own;
            if (!mine && !(nb == nb)) continue;
            const R v = mine ? own : nb, alpha = blend_to_back(v) ? -v : v;
            const bool target = mine != blend_to_back(v);   // the front pixel of a blend into the front, or the back one's
            const size_t pn = pixel_at(q);
            VKGV_CHANNELS(a) acc[a] += target ? -alpha * g_of(t, px.p, a) : alpha * g_of(n, pn, a);
        }
        if (OF == kAntialias) {
            VKGV_CHANNELS(a) g_color[px.p * A + a] = acc[a];
            if (id > 0)
                for (int k = 0; k < 9; ++k) contrib[px.p * 9 + k] = cg[k];
            return false;
        }
        if (OF == kShade && stray_blocks[px.p / kBlock] != 0u) {
            VKGV_CHANNELS(a) g_color[px.p * A + a] = acc[a];
        }
        if (!ok) return false;
        InterpTerms<C, R> it;
        bary_from(P, xn, yn, it.b);
        for (int k = 0; k < 3; ++k) it.b.v[k] = vi[k];
        {
            const R xr = ndc_x<R>(px.x, d), yr = ndc_y<R>(px.y, d);
            R glam[3] = { R(0), R(0), R(0) };
            VKGV_CHANNELS(a) {
#pragma unroll
                for (int k = 0; k < 3; ++k) glam[k] += acc[a] * attr[vi[k] * A + a];
            }
            interp_terms_of(glam, xr, yr, it);
        }
        if (NA == 3) {   // 18 values as pairs (the record is a whole number of them)
            R v[18];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                v[6 * k] = it.gu[k].x + cg[3 * k];
                v[6 * k + 1] = it.gu[k].y + cg[3 * k + 1];
                v[6 * k + 2] = it.gw[k] + cg[3 * k + 2];
                VKGV_CHANNELS(a) v[6 * k + 3 + a % 3] = it.b.lam[k] * acc[a];
            }
#pragma unroll
            for (int k = 0; k < 9; ++k) reinterpret_cast<R2<R>*>(o)[k] = R2<R>{ v[2 * k], v[2 * k + 1] };
            return true;
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            R* ok3 = o + k * (3 + A);
            ok3[0] = it.gu[k].x + cg[3 * k];
            ok3[1] = it.gu[k].y + cg[3 * k + 1];
            ok3[2] = it.gw[k] + cg[3 * k + 2];
            VKGV_CHANNELS(a) ok3[3 + a] = it.b.lam[k] * acc[a];
        }
        return true;
    };
    const bool has = px.inner && record();
    if (OF == kRender && *wide.flag != 0u) {   // uniform over the grid
        const bool on_wide = has && wide.vis[tri_index(d, px.c, id)] == kWide;
        if (__syncthreads_or(on_wide)) add_wide<C, R, NA>(wide, s_wide, tris, d, A, px.c, on_wide ? id : 0, o);
    }
}

// The stray pass: the edge terms of the blends whose front pixel is a stray,
// scattered with atomics.
template <typename C, typename R>
__global__ __launch_bounds__(kBlock) void aa_bwd_stray_kernel(const R* __restrict__ color, const C* __restrict__ clip,
                                                               const int* __restrict__ tris,
                                                               const int* __restrict__ ids,
                                                               const float* __restrict__ depth, Dims d, int A,
                                                               const R* __restrict__ g_out,
                                                               const unsigned long long* __restrict__ boxes,
                                                               const unsigned* __restrict__ stray_blocks,
                                                               C* __restrict__ g_clip)
{
    if (stray_blocks[blockIdx.x] == 0u) return;   // uniform over the block
    const size_t p = (size_t)blockIdx.x * kBlock + threadIdx.x;
    const size_t npx = (size_t)d.C * d.H * d.W;
    if (p >= npx) return;
    const int c = (int)(p / ((size_t)d.H * d.W)), py = (int)((p / d.W) % d.H), px = (int)(p % d.W);
    if (!pixel_stray(boxes, d, c, ids[p], px, py)) return;
    for (int q = 0; q < 4; ++q) {
        int ax, ay, dir;
        if (!pair_of(q, px, py, ax, ay, dir)) continue;
        PairEval<R> e;
        if (!pair_eval(clip, tris, ids, depth, d, c, ax, ay, dir, e) || e.f != p) continue;
        const EdgeGrad<R> g = edge_grad(e, blend_galpha(e, color, g_out, A), d);
        add_clip_grad<C, R>(g_clip, d, c, e.i, e.va, g.ax, g.ay, g.aw);
        add_clip_grad<C, R>(g_clip, d, c, e.i, e.vb, g.bx, g.by, g.bw);
    }
}

// ---------------------------------------------------------------------------
// Vertex adjacency of a mesh (CSR): off[v] .. off[v + 1] - 1 index the
// corners 3 t + k with tris[3 t + k] = v, in increasing order.  Vertex
// indices out of range are left out (their triangles are background).
__global__ __launch_bounds__(kBlock) void adj_zero_kernel(int* __restrict__ a, size_t n)
{
    const size_t j = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (j < n) a[j] = 0;
}

__global__ __launch_bounds__(kBlock) void adj_count_kernel(const int* __restrict__ tris, size_t n, int V,
                                                            int* __restrict__ cnt)
{
    const size_t j = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (j >= n) return;
    const int v = tris[j];
    if ((unsigned)v < (unsigned)V) atomicAdd(&cnt[v], 1);
}

// One block: off[1..V] holds the counts, replaced by their inclusive sums.
constexpr int kAdjScanThreads = 1024, kAdjScanPer = 4;
__global__ __launch_bounds__(kAdjScanThreads) void adj_scan_kernel(int* __restrict__ off, int V)
{
    __shared__ int s_w[kAdjScanThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    int carry = 0;
    for (int base = 0; base < V; base += kAdjScanThreads * kAdjScanPer) {
        int x[kAdjScanPer], sum = 0;
        for (int u = 0; u < kAdjScanPer; ++u) {
            const int idx = base + tid * kAdjScanPer + u;
            x[u] = idx < V ? off[1 + idx] : 0;
            sum += x[u];
        }
        int incl = sum;
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(incl, o, 64);
            if (lane >= o) incl += y;
        }
        if (lane == 63) s_w[w] = incl;
        __syncthreads();
        int wbase = 0, total = 0;
        for (int q = 0; q < kAdjScanThreads / 64; ++q) {
            if (q < w) wbase += s_w[q];
            total += s_w[q];
        }
        int run = carry + wbase + incl - sum;
        for (int u = 0; u < kAdjScanPer; ++u) {
            const int idx = base + tid * kAdjScanPer + u;
            run += x[u];
            if (idx < V) off[1 + idx] = run;
        }
        carry += total;
        __syncthreads();   // s_w reused by the next round
    }
}

__global__ __launch_bounds__(kBlock) void adj_fill_kernel(const int* __restrict__ tris, size_t n, int V,
                                                           const int* __restrict__ off, int* __restrict__ cursor,
                                                           int* __restrict__ adj)
{
    const size_t j = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (j >= n) return;
    const int v = tris[j];
    if ((unsigned)v < (unsigned)V) adj[off[v] + atomicAdd(&cursor[v], 1)] = (int)j;
}

// Insertion sort of each vertex's corners (its valence, at most a few dozen
// in a sane mesh): the gathers then sum in a fixed order.
__global__ __launch_bounds__(kBlock) void adj_sort_kernel(const int* __restrict__ off, int V, int* __restrict__ adj)
{
    const int v = blockIdx.x * kBlock + threadIdx.x;
    if (v >= V) return;
    const int b = off[v], e = off[v + 1];
    for (int j = b + 1; j < e; ++j) {
        const int x = adj[j];
        int k = j - 1;
        while (k >= b && adj[k] > x) {
            adj[k + 1] = adj[k];
            --k;
        }
        adj[k + 1] = x;
    }
}

// ---------------------------------------------------------------------------
// Vertex transform: clip[c, i, v] = A[c, i] (p_v, 1) with A[c, i] = VP_c M_i
// (row-major 4x4).  One block covers kBlock consecutive vertices of one
// (camera, instance), so the matrix is uniform across the block.
template <typename C>
__global__ __launch_bounds__(kBlock) void transform_fwd_kernel(const C* __restrict__ pos, const C* __restrict__ A,
                                                                int V, C* __restrict__ clip)
{
    const int v = blockIdx.x * kBlock + threadIdx.x;
    const int ci = blockIdx.y;
    if (v >= V) return;
    V4<C> o;
    transform_vertex(A + (size_t)ci * 16, pos + 3 * (size_t)v, o);
    reinterpret_cast<V4<C>*>(clip)[(size_t)ci * V + v] = o;
}

// g_pos[v] = sum over (c, i) of A[c, i][:, :3]^T g_clip[c, i, v]; one thread per vertex.
template <typename C>
__global__ __launch_bounds__(kBlock) void transform_bwd_pos_kernel(const C* __restrict__ g_clip, const C* __restrict__ A,
                                                                    int V, int CI, C* __restrict__ g_pos)
{
    const int v = blockIdx.x * kBlock + threadIdx.x;
    if (v >= V) return;
    C gx = C(0), gy = C(0), gz = C(0);
    for (int ci = 0; ci < CI; ++ci) {
        const C* g = g_clip + ((size_t)ci * V + v) * 4;
        const C* m = A + (size_t)ci * 16;
        const C g0 = g[0], g1 = g[1], g2 = g[2], g3 = g[3];
        gx += ((m[0] * g0 + m[4] * g1) + m[8] * g2) + m[12] * g3;
        gy += ((m[1] * g0 + m[5] * g1) + m[9] * g2) + m[13] * g3;
        gz += ((m[2] * g0 + m[6] * g1) + m[10] * g2) + m[14] * g3;
    }
    g_pos[3 * v] = gx;
    g_pos[3 * v + 1] = gy;
    g_pos[3 * v + 2] = gz;
}

// g_A[c, i] += sum over the block's vertices of g_clip[c, i, v] (p_v, 1)^T:
// per thread 16 products, summed across the wave with lane shuffles, then
// across the block's waves in LDS, then one atomic per entry and block.
template <typename C>
__global__ __launch_bounds__(kBlock) void transform_bwd_mat_kernel(const C* __restrict__ g_clip, const C* __restrict__ pos,
                                                                    int V, C* __restrict__ g_A)
{
    constexpr int kWaves = kBlock / 64;
    __shared__ C part[kWaves][16];
    const int v = blockIdx.x * kBlock + threadIdx.x;
    const int ci = blockIdx.y;
    C acc[16];
    if (v < V) {
        const C* g = g_clip + ((size_t)ci * V + v) * 4;
        const C ph[4] = { pos[3 * v], pos[3 * v + 1], pos[3 * v + 2], C(1) };
        for (int r = 0; r < 4; ++r) {
            const C gr = g[r];
            for (int k = 0; k < 4; ++k) acc[4 * r + k] = gr * ph[k];
        }
    } else {
        for (int k = 0; k < 16; ++k) acc[k] = C(0);
    }
    for (int k = 0; k < 16; ++k)
        for (int off = 32; off > 0; off >>= 1) acc[k] += __shfl_xor(acc[k], off, 64);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0)
        for (int k = 0; k < 16; ++k) part[wave][k] = acc[k];
    __syncthreads();
    if (threadIdx.x < 16) {
        C t = C(0);
        for (int w = 0; w < kWaves; ++w) t += part[w][threadIdx.x];
        atomicAdd(&g_A[(size_t)ci * 16 + threadIdx.x], t);
    }
}

inline unsigned blocks(size_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

} // namespace

// ---------------------------------------------------------------------------
// Triangles a wave of the raster takes: 64, or fewer where 64 leave the chip
// idle (below kRasterWaves / 2 waves), so that triangles with large boxes, which a
// wave walks one after another, are spread over it: 10240 triangles with boxes
// around 60x60 288 -> 67 us, 92160 around 20x20 130 -> 112, 2000 around a vertex
// in each of 4 views of 512x512 2300 -> 128.  Below kSpreadPixels pixels a triangle
// hardly a box is large, and the smaller waves cost 2 to 4 us (1280 triangles at
// 100x70); a quarter of it still halves them, for the slivers of a fan (2000
// around a vertex in each of 4 views of 96x96 161 -> 98 us).
constexpr size_t kRasterWaves = 4096, kSpreadPixels = 16;
static int raster_per_wave(const Dims& d)
{
    const size_t px = (size_t)d.H * d.W, least = px > kSpreadPixels * d.T ? 1 : px > kSpreadPixels / 4 * d.T ? 32 : 64;
    size_t per = 64;
    while (per > least && (size_t)d.C * d.I * d.T / per < kRasterWaves / 2) per /= 2;
    return (int)per;
}
static dim3 raster_grid(const Dims& d)
{
    const size_t per_block = (size_t)raster_per_wave(d) * (kBlock / 64u);
    return dim3((unsigned)(((size_t)d.T + per_block - 1) / per_block), std::min(d.C * d.I, 65535));
}

void raster_tris(const float* clip, const int* tris, int C, int I, int V, int T, int H, int W, int cull_back,
                 unsigned long long* keys, int* ids, float* depth, hipStream_t st)
{
    const Dims d{ C, I, V, T, H, W };
    const size_t npx = (size_t)C * H * W;
    if (C * I && T && V && npx)
        raster_tris_kernel<<<raster_grid(d), kBlock, 0, st>>>(reinterpret_cast<const V4<float>*>(clip), tris, d, keys, nullptr,
                                                              nullptr, nullptr, raster_per_wave(d), cull_back);
    if (npx) keys_to_ids_kernel<<<blocks(npx), kBlock, 0, st>>>(keys, npx, ids, depth);
}

size_t stray_flag_count(int nc, int H, int W) { return blocks((size_t)nc * H * W); }

void mesh_adjacency(const int* tris, int T, int V, int* off, int* adj, hipStream_t st)
{
    if (V <= 0) return;
    const size_t n = (size_t)3 * T;
    int* cursor = off + V + 1;
    adj_zero_kernel<<<blocks((size_t)2 * V + 1), kBlock, 0, st>>>(off, (size_t)2 * V + 1);
    if (n) adj_count_kernel<<<blocks(n), kBlock, 0, st>>>(tris, n, V, off + 1);
    adj_scan_kernel<<<1, kAdjScanThreads, 0, st>>>(off, V);
    if (n) adj_fill_kernel<<<blocks(n), kBlock, 0, st>>>(tris, n, V, off, cursor, adj);
    adj_sort_kernel<<<blocks((size_t)V), kBlock, 0, st>>>(off, V, adj);
}

size_t tri_boxes_words(int nc, int I, int T)
{
    const size_t n = (size_t)nc * I * T;
    return n + (n + 7) / 8;
}

// The flag bytes that follow the box words.
static uint8_t* vis_of(unsigned long long* boxes, int nc, int I, int T)
{
    return reinterpret_cast<uint8_t*>(boxes + (size_t)nc * I * T);
}
static const uint8_t* vis_of(const unsigned long long* boxes, int nc, int I, int T)
{
    return reinterpret_cast<const uint8_t*>(boxes + (size_t)nc * I * T);
}

template <typename C>
static void tri_boxes_t(const C* clip, const int* tris, int nc, int I, int V, int T, int H, int W,
                        unsigned long long* boxes, unsigned* stray_blocks, hipStream_t st)
{
    const Dims d{ nc, I, V, T, H, W };
    const size_t nflags = stray_flag_count(nc, H, W), n = std::max((size_t)nc * I * T, nflags);
    if (n)
        tri_boxes_kernel<C><<<blocks(n), kBlock, 0, st>>>(clip, tris, d, boxes, vis_of(boxes, nc, I, T), stray_blocks,
                                                          nflags);
}

void tri_boxes(const float* clip, const int* tris, int nc, int I, int V, int T, int H, int W,
               unsigned long long* boxes, unsigned* stray_blocks, hipStream_t st)
{
    tri_boxes_t<float>(clip, tris, nc, I, V, T, H, W, boxes, stray_blocks, st);
}
void tri_boxes(const double* clip, const int* tris, int nc, int I, int V, int T, int H, int W,
               unsigned long long* boxes, unsigned* stray_blocks, hipStream_t st)
{
    tri_boxes_t<double>(clip, tris, nc, I, V, T, H, W, boxes, stray_blocks, st);
}

// The vertex pass of interpolate, antialias and shade.
template <typename C, typename R, bool ATTR>
static void vertex_gather(const int* ids, const Dims& d, int A, const int* adj_off, const int* adj,
                          const unsigned long long* boxes, const R* contrib, C* g_clip, R* part, hipStream_t st)
{
    const unsigned n = (unsigned)((d.V + kBlockVertices - 1) / kBlockVertices) * (unsigned)(d.C * d.I);
    if (n == 0) return;
    const uint8_t* vis = vis_of(boxes, d.C, d.I, d.T);
    if (A == 3)
        vertex_gather_kernel<C, R, ATTR, 3><<<n, kBlock, 0, st>>>(ids, d, A, adj_off, adj, boxes, vis, contrib, g_clip,
                                                                  part);
    else
        vertex_gather_kernel<C, R, ATTR, 0><<<n, kBlock, 0, st>>>(ids, d, A, adj_off, adj, boxes, vis, contrib, g_clip,
                                                                  part);
}

template <typename C, typename R>
static void interp_fwd_t(const C* clip, const R* attr, const int* tris, const int* ids, int nc, int I, int V, int T,
                         int H, int W, int A, R* out, unsigned long long* boxes, unsigned* stray_blocks,
                         hipStream_t st)
{
    const Dims d{ nc, I, V, T, H, W };
    if ((size_t)nc * H * W == 0) return;
    interp_fwd_kernel<C, R><<<blocks((size_t)nc * H * W), kBlock, 0, st>>>(clip, attr, tris, ids, d, A, out, boxes,
                                                                           stray_blocks, vis_of(boxes, nc, I, T));
}

template <typename C, typename R>
static void interp_bwd_t(const C* clip, const R* attr, const int* tris, const int* ids, int nc, int I, int V, int T,
                         int H, int W, int A, const unsigned long long* boxes, const unsigned* stray_blocks,
                         const int* adj_off, const int* adj, const R* g_out, R* contrib, R* part, C* g_clip, R* g_attr,
                         hipStream_t st)
{
    const Dims d{ nc, I, V, T, H, W };
    const size_t npx = (size_t)nc * H * W;
    if (V == 0) return;
    if (npx)
        interp_bwd_pixel_kernel<C, R><<<blocks(npx), kBlock, 0, st>>>(clip, attr, tris, ids, d, A, g_out,
                                                                      contrib);
    vertex_gather<C, R, true>(ids, d, A, adj_off, adj, boxes, contrib, g_clip, part, st);
    attr_reduce_kernel<R><<<blocks((size_t)V * A), kBlock, 0, st>>>(part, nc * I, (size_t)V * A, g_attr);
    if (npx)
        interp_bwd_stray_kernel<C, R><<<blocks(npx), kBlock, 0, st>>>(clip, attr, tris, ids, d, A, g_out, boxes,
                                                                      stray_blocks, g_clip, g_attr);
}

template <typename C, typename R, int FROM>
static void aa_fwd_t(R* color, const C* clip, const R* attr, const int* tris, int* ids, float* depth,
                     const unsigned long long* keys, const Dims& d, int A, R* out, const unsigned long long* boxes,
                     unsigned* stray_blocks, uint8_t* vis, const uint32_t* wide_flag, hipStream_t st)
{
    if ((size_t)d.C * d.H * d.W == 0) return;
    if (A == 3)
        aa_fwd_kernel<C, R, FROM, 3><<<tile_blocks(d), kTileThreads, 0, st>>>(color, clip, attr, tris, ids, depth, keys,
                                                                              d, A, out, boxes, stray_blocks, vis, wide_flag);
    else
        aa_fwd_kernel<C, R, FROM, 0><<<tile_blocks(d), kTileThreads, 0, st>>>(color, clip, attr, tris, ids, depth, keys,
                                                                              d, A, out, boxes, stray_blocks, vis, wide_flag);
}

template <typename C, typename R, int OF>
static void aa_bwd_pixel(const R* color, const C* clip, const R* attr, const int* tris, const int* ids,
                         const float* depth, const Dims& d, int A, const R* g_out, const unsigned* stray_blocks,
                         R* g_color, R* contrib, const WideArgs<C, R>& wide, hipStream_t st)
{
    if ((size_t)d.C * d.H * d.W == 0) return;
    if (A == 3)
        aa_bwd_pixel_kernel<C, R, OF, 3><<<tile_blocks(d), kTileThreads, 0, st>>>(
            color, clip, attr, tris, ids, depth, d, A, g_out, stray_blocks, g_color, contrib, wide);
    else
        aa_bwd_pixel_kernel<C, R, OF, 0><<<tile_blocks(d), kTileThreads, 0, st>>>(
            color, clip, attr, tris, ids, depth, d, A, g_out, stray_blocks, g_color, contrib, wide);
}

template <typename C, typename R>
static void aa_bwd_t(const R* color, const C* clip, const int* tris, const int* ids, const float* depth, int nc, int I,
                     int V, int T, int H, int W, int A, const unsigned long long* boxes, const unsigned* stray_blocks,
                     const int* adj_off, const int* adj, const R* g_out, R* contrib, R* g_color, C* g_clip,
                     hipStream_t st)
{
    const Dims d{ nc, I, V, T, H, W };
    const size_t npx = (size_t)nc * H * W;
    aa_bwd_pixel<C, R, kAntialias>(color, clip, nullptr, tris, ids, depth, d, A, g_out, stray_blocks, g_color, contrib,
                                   {}, st);
    vertex_gather<C, R, false>(ids, d, A, adj_off, adj, boxes, contrib, g_clip, static_cast<R*>(nullptr), st);
    if (npx && V)
        aa_bwd_stray_kernel<C, R><<<blocks(npx), kBlock, 0, st>>>(color, clip, tris, ids, depth, d, A, g_out, boxes,
                                                                  stray_blocks, g_clip);
}

// antialias(interpolate(...)) as one backward: one pixel pass and one vertex
// pass for both.
template <typename C, typename R>
static void shade_bwd_t(const R* color, const C* clip, const R* attr, const int* tris, const int* ids,
                        const float* depth, int nc, int I, int V, int T, int H, int W, int A,
                        const unsigned long long* boxes, const unsigned* stray_blocks, const int* adj_off,
                        const int* adj, const R* g_out, R* g_color, R* contrib, R* part, C* g_clip, R* g_attr,
                        hipStream_t st)
{
    const Dims d{ nc, I, V, T, H, W };
    const size_t npx = (size_t)nc * H * W;
    if (V == 0) return;
    aa_bwd_pixel<C, R, kShade>(color, clip, attr, tris, ids, depth, d, A, g_out, stray_blocks, g_color, contrib, {}, st);
    vertex_gather<C, R, true>(ids, d, A, adj_off, adj, boxes, contrib, g_clip, part, st);
    attr_reduce_kernel<R><<<blocks((size_t)V * A), kBlock, 0, st>>>(part, nc * I, (size_t)V * A, g_attr);
    if (npx) {
        interp_bwd_stray_kernel<C, R><<<blocks(npx), kBlock, 0, st>>>(clip, attr, tris, ids, d, A, g_color, boxes,
                                                                      stray_blocks, g_clip, g_attr);
        aa_bwd_stray_kernel<C, R><<<blocks(npx), kBlock, 0, st>>>(color, clip, tris, ids, depth, d, A, g_out, boxes,
                                                                  stray_blocks, g_clip);
    }
}

// The word of vis that holds the wide flag, behind the bytes.
static size_t wide_word(const Dims& d) { return ((size_t)d.C * d.I * d.T + 3) / 4; }

// Projection, raster and shading of a mesh, from its own keys.
template <typename C, typename R>
static void render_fwd_t(const C* pos, const C* M, const R* attr, const int* tris, const Dims& d, int A, C* clip,
                         void* snap, unsigned long long* keys, unsigned long long* boxes, uint8_t* vis, int* ids,
                         float* depth, R* color, R* out, hipStream_t st)
{
    const size_t npx = (size_t)d.C * d.H * d.W, nvis = wide_word(d) + 1;
    if (npx == 0) return;
    uint32_t* flag = reinterpret_cast<uint32_t*>(vis) + wide_word(d);
    // at least one block, which clears the keys, also without vertices
    project_kernel<C><<<dim3(std::max(1u, blocks((size_t)d.V)), std::max(1, d.C * d.I)), kBlock, 0, st>>>(
        pos, M, d, clip, static_cast<Snap*>(snap), keys, npx, reinterpret_cast<uint32_t*>(vis), nvis);
    if (d.C * d.I && d.T && d.V)
        raster_tris_kernel<<<raster_grid(d), kBlock, 0, st>>>(static_cast<const Snap*>(snap), tris, d, keys, boxes, vis,
                                                              flag, raster_per_wave(d), 0);
    aa_fwd_t<C, R, kFromKeys>(color, clip, attr, tris, ids, depth, keys, d, A, out, nullptr, nullptr, vis, flag, st);
}

int render_parts(int nc, int I) { return std::max(1, (nc * I + kPairs - 1) / kPairs); }

static size_t pad16(size_t bytes) { return (bytes + 15) / 16 * 16; }
size_t render_wide_bytes(int V, int A, size_t c, size_t r) { return pad16((size_t)V * 3 * c) + pad16((size_t)V * A * r); }

// Clears what render's backward adds to, in one launch: g_M and, behind it, the
// sums of the kWide triangles.
static __global__ __launch_bounds__(kBlock) void clear_sums_kernel(uint4* __restrict__ a, size_t na,
                                                                    uint4* __restrict__ b, size_t nb)
{
    const size_t j = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (j < na) a[j] = uint4{ 0u, 0u, 0u, 0u };
    else if (j < na + nb) b[j - na] = uint4{ 0u, 0u, 0u, 0u };
}

// part_pos and part_attr: render_parts(nc, I) gradients, reduced into g_pos and
// g_attr (with one part they are those themselves).
template <typename C, typename R>
static void render_bwd_t(const C* pos, const C* M, const R* attr, const int* tris, const Dims& d, int A, const C* clip,
                         const unsigned long long* boxes, const uint8_t* vis, const int* ids, const float* depth,
                         const R* color, const int* adj_off, const int* adj, const R* g_out, R* contrib, C* part_pos,
                         R* part_attr, void* wide, C* g_pos, C* g_M, R* g_attr, hipStream_t st)
{
    C* wide_pos = static_cast<C*>(wide);
    R* wide_attr = reinterpret_cast<R*>(static_cast<char*>(wide) + pad16((size_t)d.V * 3 * sizeof(C)));
    const size_t m4 = (size_t)d.C * d.I * 16 * sizeof(C) / 16, w4 = render_wide_bytes(d.V, A, sizeof(C), sizeof(R)) / 16;
    if (m4 + w4)
        clear_sums_kernel<<<blocks(m4 + w4), kBlock, 0, st>>>(reinterpret_cast<uint4*>(g_M), m4,
                                                              static_cast<uint4*>(wide), w4);
    if (d.V == 0) return;
    const int parts = render_parts(d.C, d.I);
    const uint32_t* flag = reinterpret_cast<const uint32_t*>(vis) + wide_word(d);
    aa_bwd_pixel<C, R, kRender>(color, clip, attr, tris, ids, depth, d, A, g_out, nullptr, nullptr, contrib,
                                { vis, flag, pos, M, wide_pos, g_M, wide_attr }, st);
    const dim3 grid((unsigned)((d.V + kBlockVertices - 1) / kBlockVertices), (unsigned)parts);
    C* pp = parts > 1 ? part_pos : g_pos;
    R* pa = parts > 1 ? part_attr : g_attr;
    if (A == 3)
        vertex_render_kernel<C, R, 3><<<grid, kBlock, 0, st>>>(ids, d, A, pos, M, adj_off, adj, boxes, vis, contrib, pp,
                                                               pa, g_M, flag, wide_pos, wide_attr);
    else
        vertex_render_kernel<C, R, 0><<<grid, kBlock, 0, st>>>(ids, d, A, pos, M, adj_off, adj, boxes, vis, contrib, pp,
                                                               pa, g_M, flag, wide_pos, wide_attr);
    if (parts > 1) {
        const size_t np = (size_t)d.V * 3, na = (size_t)d.V * A;
        part_reduce_kernel<C, R><<<blocks(np + na), kBlock, 0, st>>>(part_pos, np, g_pos, part_attr, na, g_attr, parts);
    }
}

template <typename C>
static void transform_fwd_t(const C* pos, const C* A, int CI, int V, C* clip, hipStream_t st)
{
    if (CI == 0 || V == 0) return;
    transform_fwd_kernel<C><<<dim3(blocks((size_t)V), CI), kBlock, 0, st>>>(pos, A, V, clip);
}

template <typename C>
static void transform_bwd_t(const C* g_clip, const C* pos, const C* A, int CI, int V, C* g_pos, C* g_A, hipStream_t st)
{
    if (V == 0) return;
    transform_bwd_pos_kernel<C><<<blocks((size_t)V), kBlock, 0, st>>>(g_clip, A, V, CI, g_pos);
    if (CI) transform_bwd_mat_kernel<C><<<dim3(blocks((size_t)V), CI), kBlock, 0, st>>>(g_clip, pos, V, g_A);
}

void transform_fwd(const float* pos, const float* A, int CI, int V, float* clip, hipStream_t st)
{
    transform_fwd_t<float>(pos, A, CI, V, clip, st);
}
void transform_fwd(const double* pos, const double* A, int CI, int V, double* clip, hipStream_t st)
{
    transform_fwd_t<double>(pos, A, CI, V, clip, st);
}
void transform_bwd(const float* g_clip, const float* pos, const float* A, int CI, int V, float* g_pos, float* g_A,
                   hipStream_t st)
{
    transform_bwd_t<float>(g_clip, pos, A, CI, V, g_pos, g_A, st);
}
void transform_bwd(const double* g_clip, const double* pos, const double* A, int CI, int V, double* g_pos,
                   double* g_A, hipStream_t st)
{
    transform_bwd_t<double>(g_clip, pos, A, CI, V, g_pos, g_A, st);
}

#define VKGV_DIFF_LAUNCHERS(C, R)                                                                                     \
    void interp_fwd(const C* clip, const R* attr, const int* tris, const int* ids, int nc, int I, int V, int T, int H, \
                    int W, int A, R* out, unsigned long long* boxes, unsigned* stray_blocks, hipStream_t st)           \
    {                                                                                                                  \
        interp_fwd_t<C, R>(clip, attr, tris, ids, nc, I, V, T, H, W, A, out, boxes, stray_blocks, st);                 \
    }                                                                                                                  \
    void interp_bwd(const C* clip, const R* attr, const int* tris, const int* ids, int nc, int I, int V, int T, int H, \
                    int W, int A, const unsigned long long* boxes, const unsigned* stray_blocks, const int* adj_off,   \
                    const int* adj, const R* g_out, R* contrib, R* part, C* g_clip, R* g_attr, hipStream_t st)         \
    {                                                                                                                  \
        interp_bwd_t<C, R>(clip, attr, tris, ids, nc, I, V, T, H, W, A, boxes, stray_blocks, adj_off, adj, g_out,      \
                           contrib, part, g_clip, g_attr, st);                                                         \
    }                                                                                                                  \
    void aa_fwd(const R* color, const C* clip, const int* tris, const int* ids, const float* depth, int nc, int I,     \
                int V, int T, int H, int W, int A, R* out, unsigned long long* boxes, unsigned* stray_blocks,          \
                hipStream_t st)                                                                                        \
    {                                                                                                                  \
        const Dims d{ nc, I, V, T, H, W };                                                                             \
        aa_fwd_t<C, R, kFromColor>(const_cast<R*>(color), clip, nullptr, tris, const_cast<int*>(ids),                  \
                                   const_cast<float*>(depth), nullptr, d, A, out, boxes, stray_blocks,                 \
                                   vis_of(boxes, nc, I, T), nullptr, st);                                                       \
    }                                                                                                                  \
    void shade_fwd(const C* clip, const R* attr, const int* tris, const int* ids, const float* depth, int nc, int I,   \
                   int V, int T, int H, int W, int A, R* color, R* out, unsigned long long* boxes,                     \
                   unsigned* stray_blocks, hipStream_t st)                                                             \
    {                                                                                                                  \
        const Dims d{ nc, I, V, T, H, W };                                                                             \
        aa_fwd_t<C, R, kFromIds>(color, clip, attr, tris, const_cast<int*>(ids), const_cast<float*>(depth), nullptr,   \
                                 d, A, out, boxes, stray_blocks, vis_of(boxes, nc, I, T), nullptr, st);                \
    }                                                                                                                  \
    void render_fwd(const C* pos, const C* M, const R* attr, const int* tris, int nc, int I, int V, int T, int H,      \
                    int W, int A, C* clip, void* snap, unsigned long long* keys, unsigned long long* boxes,            \
                    uint8_t* vis, int* ids, float* depth, R* color, R* out, hipStream_t st)                            \
    {                                                                                                                  \
        const Dims d{ nc, I, V, T, H, W };                                                                             \
        render_fwd_t<C, R>(pos, M, attr, tris, d, A, clip, snap, keys, boxes, vis, ids, depth, color, out, st);        \
    }                                                                                                                  \
    void render_bwd(const C* pos, const C* M, const R* attr, const int* tris, int nc, int I, int V, int T, int H,      \
                    int W, int A, const C* clip, const unsigned long long* boxes, const uint8_t* vis, const int* ids,  \
                    const float* depth, const R* color, const int* adj_off, const int* adj, const R* g_out,            \
                    R* contrib, C* part_pos, R* part_attr, void* wide, C* g_pos, C* g_M, R* g_attr, hipStream_t st)        \
    {                                                                                                                  \
        const Dims d{ nc, I, V, T, H, W };                                                                             \
        render_bwd_t<C, R>(pos, M, attr, tris, d, A, clip, boxes, vis, ids, depth, color, adj_off, adj, g_out,         \
                           contrib, part_pos, part_attr, wide, g_pos, g_M, g_attr, st);                                \
    }                                                                                                                  \
    void aa_bwd(const R* color, const C* clip, const int* tris, const int* ids, const float* depth, int nc, int I,     \
                int V, int T, int H, int W, int A, const unsigned long long* boxes, const unsigned* stray_blocks,      \
                const int* adj_off, const int* adj, const R* g_out, R* contrib, R* g_color, C* g_clip,                 \
                hipStream_t st)                                                                                        \
    {                                                                                                                  \
        aa_bwd_t<C, R>(color, clip, tris, ids, depth, nc, I, V, T, H, W, A, boxes, stray_blocks, adj_off, adj, g_out,  \
                       contrib, g_color, g_clip, st);                                                                  \
    }                                                                                                                  \
    void shade_bwd(const R* color, const C* clip, const R* attr, const int* tris, const int* ids, const float* depth,  \
                   int nc, int I, int V, int T, int H, int W, int A, const unsigned long long* boxes,                  \
                   const unsigned* stray_blocks, const int* adj_off, const int* adj, const R* g_out, R* g_color,       \
                   R* contrib, R* part, C* g_clip, R* g_attr, hipStream_t st)                                          \
    {                                                                                                                  \
        shade_bwd_t<C, R>(color, clip, attr, tris, ids, depth, nc, I, V, T, H, W, A, boxes, stray_blocks, adj_off,     \
                          adj, g_out, g_color, contrib, part, g_clip, g_attr, st);                                     \
    }

VKGV_DIFF_LAUNCHERS(float, float)
VKGV_DIFF_LAUNCHERS(double, double)
VKGV_DIFF_LAUNCHERS(double, float)
#undef VKGV_DIFF_LAUNCHERS

} // namespace vkgv_diff
