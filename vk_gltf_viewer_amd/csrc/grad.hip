// Differentiable frame: the antialiased linear image of a view's last frame
// and its gradient with respect to the instance transforms, computed from the
// frame's own 64-bit visibility buffer (no second raster).
//
// Image: each pixel's material albedo factor (the flat resolve before the
// sRGB encode, visbuffer_resolve.comp.glsl:17-41; background 0), with the
// analytic edge antialiasing of the differentiable form: for every
// horizontally or vertically adjacent pixel pair with different colours
// (different materials, or one side background), the front pixel (the
// non-background one, else the one with the smaller key, i.e. nearer) keeps
// its triangle; the segment from its centre to the other centre leaves the
// triangle through the edge whose edge function changes sign first, at t in
// [0, 1]; t < 1/2 blends (1/2 - t) of the back colour into the front pixel,
// else (t - 1/2) of the front colour into the back pixel.  Pairs of equal
// colour change nothing and are skipped.
//
// Geometry: id = draw << 7 | triangle -> the draw's raster record (vertex,
// triangle and vertex-index offsets into the packed mesh buffers, transform
// index, material) -> the triangle's object-space positions p; the clip
// position VP M (p, 1) is formed in double (VP, M are the camera's and the
// instance's float matrices), and so are the screen offsets from the front
// pixel's centre: the edge term scales as 1 / (edge function difference)^2,
// which float32 clip positions do not resolve.
//
// Work split.  Only the pairs across a material boundary blend, and each costs
// some 400 double-precision operations behind a chain of four dependent
// loads; nearly all pairs need nothing.  A block takes a 64x8-pixel tile: it
// puts the materials of the tile and its border in LDS, packs the pairs of
// different material into a list, and evaluates the list with every lane
// busy, each pair once (one thread per pixel or pair left a wave waiting for
// its few boundary lanes, and the image evaluated each pair from both sides).
// The tile is 64 wide so that a row's keys are whole 128-byte lines.  What is
// left is the latency of key -> record -> colour over the tiles (city at
// 3840x2160: image 57 us, 2.9 TB/s of its 165 MB, where a material pass and
// one thread per pixel took 21 + 123 us) and, with many boundaries, the
// evaluations (views of up to 3840x2160 of the uneven scene: image 77 us a
// view from 217, backward 114 from 488).
//   image     the pair results go to LDS by pair, and each pixel adds those of
//             its four pairs in a fixed order: the same bits on every run.
//   backward  d loss / d M_tr = sum over the crossed edge's two vertices of
//             (VP^T g_clip) (p, 1)^T.  The two vectors of each vertex go to
//             LDS; then lane j of a 16-lane group forms entry j of the product
//             for a run of the list and adds it to the gradient when the
//             transform changes (16 consecutive doubles per atomic).
#include <hip/hip_runtime.h>

#include "internal.hpp"

namespace vkgv {
namespace {

constexpr uint32_t kGradBlock = 256;

struct GradArgs {
    SceneDev s;
    const unsigned long long* keys;
    uint32_t W, H;
    double vp[16];          // column-major
};

constexpr uint32_t kNoMaterial = 0xFFFFFFFFu;   // background
constexpr uint32_t kOutside = 0xFFFFFFFEu;      // outside the view (material indices have 31 bits)
constexpr int kTileX = 64, kTileY = 8;          // pixels of a block

__device__ __forceinline__ bool key_id(unsigned long long k, uint32_t& id)
{
    if (k == ~0ull) return false;
    id = 0xFFFFFFFEu - (uint32_t)k;
    return true;
}

// material of a key's draw; kNoMaterial on background or an id outside the draw list
__device__ __forceinline__ uint32_t material_of_key(const SceneDev& s, unsigned long long k)
{
    uint32_t id;
    if (!key_id(k, id)) return kNoMaterial;
    const uint32_t d = id >> VKGV_TRIANGLE_BITS;
    if (d >= s.draw_count) return kNoMaterial;
    return s.rrec[d].material & 0x7FFFFFFFu;
}

__device__ __forceinline__ float3 albedo(const SceneDev& s, uint32_t m)
{
    if (m == kNoMaterial) return make_float3(0.0f, 0.0f, 0.0f);
    const vkgv_material& mt = s.materials[m];
    return make_float3(mt.albedo_factor[0], mt.albedo_factor[1], mt.albedo_factor[2]);
}

// One blend: what the backward needs of it.
struct DPair {
    bool to_front, to_p;    // the target is the front pixel; it is the pair's first pixel
    uint32_t tr;
    double alpha, ef, eb;
    double sa[2], sb[2], cb[2];
    double pa[4], pb[4];
    double oa[3], ob[3];
};

__device__ __forceinline__ double efn(const double* a, const double* b, const double* p)
{
    return (b[0] - a[0]) * (p[1] - a[1]) - (b[1] - a[1]) * (p[0] - a[0]);
}

// Pair (px, py) - right (dir 0) or lower (dir 1) neighbour, both in the view,
// of different materials mp and mq.
__device__ __forceinline__ bool pair_eval(const GradArgs& a, int px, int py, int dir, uint32_t mp, uint32_t mq, DPair& e)
{
    const int qx = px + (dir == 0), qy = py + (dir == 1);
    const size_t ip = (size_t)py * a.W + px, iq = (size_t)qy * a.W + qx;
    const bool hp = mp != kNoMaterial, hq = mq != kNoMaterial;
    const unsigned long long kp = a.keys[ip], kq = a.keys[iq];
    const bool p_front = !hp ? false : (!hq ? true : kp <= kq);
    uint32_t id;
    key_id(p_front ? kp : kq, id);
    const int fx = p_front ? px : qx, fy = p_front ? py : qy;
    const double step = p_front ? 1.0 : -1.0;
    e.cb[0] = dir == 0 ? step : 0.0;
    e.cb[1] = dir == 0 ? 0.0 : step;
    const RasterRec r = a.s.rrec[id >> VKGV_TRIANGLE_BITS];
    const uint32_t t = id & ((1u << VKGV_TRIANGLE_BITS) - 1u);
    if (t >= ((r.counts >> 8) & 0xFFu)) return false;
    e.tr = r.transform;
    const float* m = a.s.transforms + 16ull * r.transform;
    double M[16];
    for (int i = 0; i < 16; ++i) M[i] = (double)m[i];
    const double hw = a.W * 0.5, hh = a.H * 0.5;
    const double xc = (fx + 0.5) / hw - 1.0, yc = (fy + 0.5) / hh - 1.0;
    double P[3][4], S[3][2], O[3][3];
    for (int k = 0; k < 3; ++k) {
        const uint32_t li = a.s.tri_base[r.tri + 3u * t + (uint32_t)k];
        const uint32_t vi = a.s.vidx_base[r.vidx + li];
        const float* pp = reinterpret_cast<const float*>(reinterpret_cast<const uint8_t*>(a.s.vtx_base) + r.vtx) +
                          (size_t)vi * 6;
        O[k][0] = pp[0]; O[k][1] = pp[1]; O[k][2] = pp[2];
        double w4[4];
        for (int rr = 0; rr < 4; ++rr) w4[rr] = M[rr] * O[k][0] + M[4 + rr] * O[k][1] + M[8 + rr] * O[k][2] + M[12 + rr];
        for (int rr = 0; rr < 4; ++rr)
            P[k][rr] = a.vp[rr] * w4[0] + a.vp[4 + rr] * w4[1] + a.vp[8 + rr] * w4[2] + a.vp[12 + rr] * w4[3];
        if (!(P[k][3] > 0.0)) return false;
        S[k][0] = hw * ((P[k][0] - xc * P[k][3]) / P[k][3]);
        S[k][1] = hh * ((P[k][1] - yc * P[k][3]) / P[k][3]);
    }
    const double area = efn(S[0], S[1], S[2]);
    if (area == 0.0) return false;
    const double sgn = area > 0.0 ? 1.0 : -1.0;
    const double zero[2] = { 0.0, 0.0 };
    double best = 2.0, bef = 0.0, beb = 0.0;
    int kb = -1;
    for (int k = 0; k < 3; ++k) {
        const double ef = sgn * efn(S[k], S[(k + 1) % 3], zero);
        const double eb = sgn * efn(S[k], S[(k + 1) % 3], e.cb);
        if (!(ef >= 0.0 && eb <= 0.0 && ef > eb)) continue;
        const double tt = ef / (ef - eb);
        if (tt < best) { best = tt; kb = k; bef = ef; beb = eb; }
    }
    if (kb < 0) return false;
    e.to_front = best < 0.5;
    e.to_p = e.to_front == p_front;
    e.alpha = e.to_front ? 0.5 - best : best - 0.5;
    const int ka = kb, kc = (kb + 1) % 3;
    for (int j = 0; j < 4; ++j) { e.pa[j] = P[ka][j]; e.pb[j] = P[kc][j]; }
    for (int j = 0; j < 3; ++j) { e.oa[j] = O[ka][j]; e.ob[j] = O[kc][j]; }
    for (int j = 0; j < 2; ++j) { e.sa[j] = S[ka][j]; e.sb[j] = S[kc][j]; }
    e.ef = sgn * bef;
    e.eb = sgn * beb;
    return true;
}

// Materials of the tile at (x0, y0) and its border (rows and columns -BEFORE
// .. size, without the corners, which no pair needs), in LDS.  Thread t loads
// its own pixels (t % 64, t / 64 + 4 k) and at most one border pixel: the keys
// in flight together, then the draw records.
constexpr int kOwn = kTileX * kTileY / (int)kGradBlock;
static_assert(kTileX == 64 && kTileX * kTileY == kOwn * (int)kGradBlock, "a thread owns kOwn pixels of its column");
__device__ __forceinline__ int own_x() { return (int)(threadIdx.x & 63u); }
__device__ __forceinline__ int own_y(int k) { return (int)(threadIdx.x >> 6) + (int)(kGradBlock / 64u) * k; }

template <int BEFORE>
struct TileMat {
    static constexpr int kW = kTileX + 1 + BEFORE, kH = kTileY + 1 + BEFORE;
    static constexpr int kRowsOut = (1 + BEFORE) * kTileX;                 // border pixels above and below
    static constexpr int kBorder = kRowsOut + (1 + BEFORE) * kTileY;
    static_assert(kBorder <= (int)kGradBlock, "one border pixel per thread");
    uint32_t m[kW * kH];
    __device__ __forceinline__ uint32_t& at(int x, int y) { return m[(y + BEFORE) * kW + x + BEFORE]; }
    // fills the tile; own[k]: the thread's own pixels
    __device__ __forceinline__ void load(const GradArgs& a, int x0, int y0, uint32_t* own)
    {
        int x[kOwn + 1], y[kOwn + 1];
        bool in[kOwn + 1];
#pragma unroll
        for (int k = 0; k < kOwn; ++k) { x[k] = own_x(); y[k] = own_y(k); }
        const int t = (int)threadIdx.x;
        const bool rows = t < kRowsOut;
        const int c = t - kRowsOut;
        // below first, then (with BEFORE) above; right first, then left
        x[kOwn] = rows ? t % kTileX : (c < kTileY ? kTileX : -1);
        y[kOwn] = rows ? (t < kTileX ? kTileY : -1) : c % kTileY;
        unsigned long long key[kOwn + 1];
#pragma unroll
        for (int k = 0; k <= kOwn; ++k) {
            const int gx = x0 + x[k], gy = y0 + y[k];
            in[k] = gx >= 0 && gy >= 0 && gx < (int)a.W && gy < (int)a.H && (k < kOwn || t < kBorder);
            key[k] = in[k] ? a.keys[(size_t)gy * a.W + gx] : ~0ull;
        }
        uint32_t mat[kOwn + 1];
#pragma unroll
        for (int k = 0; k <= kOwn; ++k) mat[k] = material_of_key(a.s, key[k]);
#pragma unroll
        for (int k = 0; k <= kOwn; ++k) {
            const uint32_t v = in[k] ? mat[k] : kOutside;
            if (k < kOwn) own[k] = v;
            if (k < kOwn || t < kBorder) at(x[k], y[k]) = v;
        }
    }
};

// Whether a pair of pixels with these materials blends.
__device__ __forceinline__ bool differ(uint32_t mp, uint32_t mq) { return mp != mq && mp != kOutside && mq != kOutside; }

// Appends `code` to an LDS list on the lanes with `want` (every lane of the
// wave calls it): one LDS atomic per wave.
__device__ __forceinline__ void append(bool want, uint32_t code, uint16_t* list, uint32_t* count)
{
    const unsigned long long m = __ballot(want);
    if (m == 0ull) return;
    const int lead = __ffsll((long long)m) - 1;
    uint32_t base = 0;
    if ((int)(threadIdx.x & 63u) == lead) base = atomicAdd(count, (uint32_t)__popcll(m));
    base = (uint32_t)__shfl((int)base, lead, 64);
    const uint32_t pos = base + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
    if (want) list[pos] = (uint16_t)code;
}

// Pair codes of the image: horizontal pairs by their first pixel, columns
// -1 .. kTileX - 1 of each row, then vertical ones, rows -1 .. kTileY - 1.
constexpr int kHPairs = (kTileX + 1) * kTileY, kImagePairs = kHPairs + kTileX * (kTileY + 1);
__device__ __forceinline__ uint32_t hcode(int x, int y) { return (uint32_t)(y * (kTileX + 1) + x + 1); }
__device__ __forceinline__ uint32_t vcode(int x, int y) { return (uint32_t)(kHPairs + (y + 1) * kTileX + x); }
__device__ __forceinline__ void image_pair(int code, int& x, int& y, int& dir)
{
    dir = code >= kHPairs;
    const int k = dir ? code - kHPairs : code, w = dir ? kTileX : kTileX + 1;
    x = k % w - (dir ? 0 : 1);
    y = k / w - (dir ? 1 : 0);
}

// Gather: pixel = its colour + the blends of its four pairs that target it.
__global__ __launch_bounds__(kGradBlock) void aa_image_kernel(GradArgs a, float* __restrict__ image)
{
    __shared__ TileMat<1> s_mat;
    __shared__ double s_alpha[kImagePairs];   // of the listed pairs: sign 0 into the first pixel, 1 the second; NaN: no blend
    __shared__ uint16_t s_list[kImagePairs];
    __shared__ uint32_t s_n;
    const int x0 = (int)blockIdx.x * kTileX, y0 = (int)blockIdx.y * kTileY;
    if (threadIdx.x == 0) s_n = 0u;
    uint32_t own[kOwn];
    s_mat.load(a, x0, y0, own);
    float3 col[kOwn];
#pragma unroll
    for (int k = 0; k < kOwn; ++k) col[k] = albedo(a.s, own[k] == kOutside ? kNoMaterial : own[k]);
    __syncthreads();
    for (int k0 = 0; k0 < kImagePairs; k0 += (int)kGradBlock) {
        const int k = k0 + (int)threadIdx.x;
        bool want = false;
        if (k < kImagePairs) {
            int x, y, dir;
            image_pair(k, x, y, dir);
            want = differ(s_mat.at(x, y), s_mat.at(x + (dir == 0), y + (dir == 1)));
        }
        append(want, (uint32_t)k, s_list, &s_n);
    }
    __syncthreads();
    const uint32_t n = s_n;
    for (uint32_t i = threadIdx.x; i < n; i += kGradBlock) {
        int x, y, dir;
        image_pair((int)s_list[i], x, y, dir);
        DPair e;
        double r = __longlong_as_double(0x7FF8000000000000ll);
        if (pair_eval(a, x0 + x, y0 + y, dir, s_mat.at(x, y), s_mat.at(x + (dir == 0), y + (dir == 1)), e))
            r = e.to_p ? e.alpha : -e.alpha;
        s_alpha[s_list[i]] = r;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kOwn; ++k) {
        const int x = own_x(), y = own_y(k);
        const uint32_t m = own[k];
        if (m == kOutside) continue;
        const float3 c = col[k];
        double acc[3] = { c.x, c.y, c.z };
        if (n) {
            // left, right, upper, lower neighbour and the pair's code; this pixel is the second of the
            // left and upper pairs
            const int nx[4] = { x - 1, x + 1, x, x }, ny[4] = { y, y, y - 1, y + 1 };
            const uint32_t code[4] = { hcode(x - 1, y), hcode(x, y), vcode(x, y - 1), vcode(x, y) };
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t mn = s_mat.at(nx[q], ny[q]);
                if (!differ(m, mn)) continue;
                const double r = s_alpha[code[q]], al = fabs(r);
                if (r != r || (__double_as_longlong(r) >= 0) != ((q & 1) != 0)) continue;
                const float3 cs = albedo(a.s, mn);
                acc[0] += al * ((double)cs.x - c.x);
                acc[1] += al * ((double)cs.y - c.y);
                acc[2] += al * ((double)cs.z - c.z);
            }
        }
        float* o = image + 3 * ((size_t)(y0 + y) * a.W + (x0 + x));
        o[0] = (float)acc[0];
        o[1] = (float)acc[1];
        o[2] = (float)acc[2];
    }
}

// The tile's pixels' right (codes 0 .. kTileX * kTileY - 1) and lower pairs.
constexpr int kTilePixels = kTileX * kTileY;
constexpr int kGradWords = 14;                 // doubles a pair leaves in LDS: VP^T g_clip and p of its two vertices
constexpr int kGradStride = kGradBlock + 2;    // row of kGradBlock pairs, padded off the banks of the next one
__global__ __launch_bounds__(kGradBlock) void aa_backward_kernel(GradArgs a, const float* __restrict__ g_image,
                                                                 double* __restrict__ g_transforms)
{
    __shared__ TileMat<0> s_mat;
    __shared__ uint16_t s_list[2 * kTilePixels];
    __shared__ uint32_t s_n;
    __shared__ double s_v[kGradWords][kGradStride];
    __shared__ int s_tr[kGradBlock];
    const int x0 = (int)blockIdx.x * kTileX, y0 = (int)blockIdx.y * kTileY;
    if (threadIdx.x == 0) s_n = 0u;
    uint32_t own[kOwn];
    s_mat.load(a, x0, y0, own);
    __syncthreads();
    for (int k = (int)threadIdx.x; k < 2 * kTilePixels; k += (int)kGradBlock) {
        const int dir = k >= kTilePixels, p = k % kTilePixels, x = p % kTileX, y = p / kTileX;
        append(differ(s_mat.at(x, y), s_mat.at(x + (dir == 0), y + (dir == 1))), (uint32_t)k, s_list, &s_n);
    }
    __syncthreads();
    const uint32_t n = s_n;
    for (uint32_t i0 = 0; i0 < n; i0 += kGradBlock) {
        const uint32_t m = min(kGradBlock, n - i0);
        const uint32_t slot = threadIdx.x;
        if (slot < m) {
            const int k = (int)s_list[i0 + slot];
            const int dir = k >= kTilePixels, p = k % kTilePixels, x = p % kTileX, y = p / kTileX;
            const uint32_t mp = s_mat.at(x, y), mq = s_mat.at(x + (dir == 0), y + (dir == 1));
            DPair e;
            int key = -1;
            if (pair_eval(a, x0 + x, y0 + y, dir, mp, mq, e)) {
                const size_t ip = (size_t)(y0 + y) * a.W + (x0 + x), iq = ip + (dir == 0 ? 1 : a.W);
                const size_t tgt = e.to_p ? ip : iq;
                const float3 ct = albedo(a.s, e.to_p ? mp : mq), cs = albedo(a.s, e.to_p ? mq : mp);
                const double galpha = (double)g_image[3 * tgt] * ((double)cs.x - ct.x) +
                                      (double)g_image[3 * tgt + 1] * ((double)cs.y - ct.y) +
                                      (double)g_image[3 * tgt + 2] * ((double)cs.z - ct.z);
                const double gt = e.to_front ? -galpha : galpha;
                const double den = e.ef - e.eb;
                const double gef = gt * (-e.eb / (den * den)), geb = gt * (e.ef / (den * den));
                // e(P) = (bx - ax)(Py - ay) - (by - ay)(Px - ax) at P = 0 (front) and cb (back)
                const double gax = gef * (e.sb[1] - 0.0) + geb * (e.sb[1] - e.cb[1]);
                const double gay = gef * (0.0 - e.sb[0]) + geb * (e.cb[0] - e.sb[0]);
                const double gbx = gef * (0.0 - e.sa[1]) + geb * (e.cb[1] - e.sa[1]);
                const double gby = gef * (e.sa[0] - 0.0) + geb * (e.sa[0] - e.cb[0]);
                const double hw = a.W * 0.5, hh = a.H * 0.5;
                const double* pc[2] = { e.pa, e.pb };
                const double* po[2] = { e.oa, e.ob };
                const double gsx[2] = { gax, gbx }, gsy[2] = { gay, gby };
#pragma unroll
                for (int v = 0; v < 2; ++v) {
                    const double* c = pc[v];
                    const double gc0 = gsx[v] * hw / c[3], gc1 = gsy[v] * hh / c[3];
                    const double gc3 = -(gsx[v] * hw * c[0] + gsy[v] * hh * c[1]) / (c[3] * c[3]);
#pragma unroll
                    for (int j = 0; j < 4; ++j)   // VP^T g_clip (g_clip.z = 0)
                        s_v[7 * v + j][slot] = a.vp[j * 4] * gc0 + a.vp[j * 4 + 1] * gc1 + a.vp[j * 4 + 3] * gc3;
#pragma unroll
                    for (int j = 0; j < 3; ++j) s_v[7 * v + 4 + j][slot] = po[v][j];
                }
                key = (int)e.tr;
            }
            s_tr[slot] = key;
        }
        __syncthreads();
        {
            const int j = (int)(threadIdx.x & 15u), r = j & 3, col = j >> 2;
            const uint32_t groups = kGradBlock / 16u, per = (m + groups - 1u) / groups;
            const uint32_t first = (threadIdx.x >> 4) * per, end = min(first + per, m);
            double acc = 0.0;
            int cur = -1;
            for (uint32_t i = first; i < end; ++i) {
                const int tr = s_tr[i];
                if (tr < 0) continue;
                if (tr != cur) {
                    if (cur >= 0) atomicAdd(&g_transforms[16ull * (uint32_t)cur + j], acc);
                    cur = tr;
                    acc = 0.0;
                }
                const double p0 = col < 3 ? s_v[4 + col][i] : 1.0, p1 = col < 3 ? s_v[11 + col][i] : 1.0;
                acc += s_v[r][i] * p0 + s_v[7 + r][i] * p1;
            }
            if (cur >= 0) atomicAdd(&g_transforms[16ull * (uint32_t)cur + j], acc);
        }
        __syncthreads();   // the records are overwritten by the next round
    }
}

inline dim3 grad_tiles(uint32_t W, uint32_t H) { return dim3((W + kTileX - 1) / kTileX, (H + kTileY - 1) / kTileY); }

GradArgs make_args(const SceneDev& s, const unsigned long long* keys, uint32_t W, uint32_t H, const float* vp)
{
    GradArgs a;
    a.s = s;
    a.keys = keys;
    a.W = W;
    a.H = H;
    for (int i = 0; i < 16; ++i) a.vp[i] = (double)vp[i];
    return a;
}

} // namespace

void launch_aa_image(const SceneDev& s, const unsigned long long* keys, uint32_t W, uint32_t H, const float* vp,
                     float* image, hipStream_t st)
{
    if ((size_t)W * H == 0) return;
    aa_image_kernel<<<grad_tiles(W, H), kGradBlock, 0, st>>>(make_args(s, keys, W, H, vp), image);
}

void launch_aa_backward(const SceneDev& s, const unsigned long long* keys, uint32_t W, uint32_t H, const float* vp,
                        const float* g_image, double* g_transforms, hipStream_t st)
{
    if ((size_t)W * H == 0) return;
    aa_backward_kernel<<<grad_tiles(W, H), kGradBlock, 0, st>>>(make_args(s, keys, W, H, vp), g_image, g_transforms);
}

} // namespace vkgv
