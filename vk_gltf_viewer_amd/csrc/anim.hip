// Per-frame transform update on the device (World::updateDrawBuffers,
// world.cpp:346-354): animation sampling per node (AnimationSampler::sample,
// assets.hpp:52-110; channel application, world.cpp:192-216), then the world
// matrix of every mesh node down its ancestor chain (World::iterateNode,
// world.cpp:187-228: parent * T * R * S).
//
// Kernel 1, one thread per channel: the channel's value at `time` into its
// part of the node's TRS.  A node's later channel on a path replaces the
// earlier one's value, so that only the last is kept when the hierarchy is
// set, and the static parts stay in the buffer from then on.  The channels are
// grouped by path and interpolation, which a wave would otherwise run through
// one after another.  Kernel 2, four threads per mesh node: the product along
// its root-to-node chain, in the same operation order as the host traversal
// (so an unanimated hierarchy gives the host's matrices bit for bit), written
// to the transform buffer.  Row r of a product needs only row r of its left
// factor, so that each thread carries one row down the chain, and the next
// node's TRS is in flight meanwhile.  A chain is at most 64 nodes.
// Both are bound by the latency of a few waves' dependent loads and products:
// 65536 nodes, 65k channels: 10 us and 12 us (which also keeps the previous
// matrices, a copy of 5 us before), where one thread per node with
// its channels in turn took 28 and one per mesh node 16.
//
// slerp evaluates acos and sin in double precision with fixed series (below)
// instead of a math library, so that every platform computes the same bits.
#include "internal.hpp"

namespace vkgv {
namespace {

// asin(y), |y| <= 1/2: Maclaurin series y * sum c_n y^(2n) with
// c_{n+1} / c_n = (2n+1)^2 / ((2n+2)(2n+3)), in Horner form (31 terms).
__device__ double series_asin(double y)
{
    const double y2 = y * y;
    double acc = 1.0;
#pragma unroll
    for (int n = 29; n >= 0; --n)   // unrolled: the ratios are constants
        acc = 1.0 + (y2 * acc) * ((double)((2 * n + 1) * (2 * n + 1)) / (double)((2 * n + 2) * (2 * n + 3)));
    return y * acc;
}

// acos(x), 0 <= x <= 1.
__device__ double series_acos(double x)
{
    if (x <= 0.5) return 1.5707963267948966 - series_asin(x);
    return 2.0 * series_asin(sqrt((1.0 - x) * 0.5));
}

// sin(a), 0 <= a <= pi/2: Taylor series, 16 terms, in Horner form.
__device__ double series_sin(double a)
{
    const double a2 = a * a;
    double acc = 1.0;
#pragma unroll
    for (int n = 14; n >= 0; --n) acc = 1.0 - (a2 * acc) / (double)((2 * n + 2) * (2 * n + 3));
    return a * acc;
}

// Output k of the sampler's values (N floats per output).
template <int N>
__device__ __forceinline__ void load_out(const float* v, uint32_t k, float* o)
{
#pragma unroll
    for (int i = 0; i < N; ++i) o[i] = v[(size_t)k * N + i];
}

// AnimationSampler::sample<path>(time) (assets.hpp:52-110); N = 3 for
// translation and scale, 4 for rotation.
template <int N>
__device__ __forceinline__ void sample(const AnimDev& d, const AnimChan& sp, float time, float* out)
{
    const float* in = d.times + sp.input_offset;
    const float* val = d.values + sp.output_offset;
    const uint32_t cnt = sp.input_count, interpolation = sp.kind >> 8;
    const bool cubic = interpolation == VKGV_INTERP_CUBICSPLINE;
    time = fmodf(time, sp.last);                            // loop the animation
    // std::lower_bound (first key >= time), with libstdc++'s probe sequence so
    // that even unsorted times pick the key the reference picks
    uint32_t lo = 0, len = cnt;
    while (len > 0) {
        const uint32_t half = len >> 1;
        if (in[lo + half] < time) { lo = lo + half + 1; len = len - half - 1; }
        else len = half;
    }
    if (lo == 0) { load_out<N>(val, cubic ? 1u : 0u, out); return; }
    if (lo == cnt) { load_out<N>(val, cubic ? 3u * cnt - 2u : cnt - 1u, out); return; }
    const uint32_t i = lo;
    const float t = (time - in[i - 1]) / (in[i] - in[i - 1]);
    if (interpolation == VKGV_INTERP_STEP) { load_out<N>(val, i - 1, out); return; }
    if (!cubic) {
        float a[N], b[N];
        load_out<N>(val, i - 1, a);
        load_out<N>(val, i, b);
        if (N == 3) {
#pragma unroll
            for (int k = 0; k < N; ++k) out[k] = a[k] * (1.0f - t) + b[k] * t;
            return;
        }
        // slerp (shortest arc; linear when the keys nearly coincide)
        float cosv = 0.0f;
#pragma unroll
        for (int k = 0; k < N; ++k) cosv = k == 0 ? a[0] * b[0] : cosv + a[k] * b[k];
        if (cosv < 0.0f) {
#pragma unroll
            for (int k = 0; k < N; ++k) b[k] = -b[k];
            cosv = -cosv;
        }
        if (cosv > 1.0f - 1.1920928955078125e-7f) {
#pragma unroll
            for (int k = 0; k < N; ++k) out[k] = a[k] * (1.0f - t) + b[k] * t;
            return;
        }
        const double ang = series_acos((double)cosv);
        const double sa = series_sin(ang);
        const double w0 = series_sin((1.0 - (double)t) * ang) / sa;
        const double w1 = series_sin((double)t * ang) / sa;
#pragma unroll
        for (int k = 0; k < N; ++k) out[k] = (float)(w0 * (double)a[k] + w1 * (double)b[k]);
        return;
    }
    // cubic Hermite spline (glTF 2.0 appendix C): in-tangent, value, out-tangent per key
    const float t2 = t * t, t3 = t2 * t;
    const float dt = in[i] - in[i - 1];
    float v0[N], b0[N], v1[N], a1[N];
    load_out<N>(val, 3u * (i - 1) + 1u, v0);
    load_out<N>(val, 3u * (i - 1) + 2u, b0);
    load_out<N>(val, 3u * i + 1u, v1);
    load_out<N>(val, 3u * i + 0u, a1);
    const float h00 = (2.0f * t3 - 3.0f * t2) + 1.0f;
    const float h10 = (t3 - 2.0f * t2) + t;
    const float h01 = -2.0f * t3 + 3.0f * t2;
    const float h11 = t3 - t2;
#pragma unroll
    for (int k = 0; k < N; ++k) out[k] = ((v0[k] * h00 + (b0[k] * h10) * dt) + v1[k] * h01) + (a1[k] * h11) * dt;
    if (N == 4) {
        float l2 = 0.0f;
#pragma unroll
        for (int k = 0; k < N; ++k) l2 = k == 0 ? out[0] * out[0] : l2 + out[k] * out[k];
        const float l = sqrtf(l2);
#pragma unroll
        for (int k = 0; k < N; ++k) out[k] = out[k] / l;
    }
}

__device__ __forceinline__ NodeTrs& node_trs(const AnimDev& d, uint32_t n)
{
    return *reinterpret_cast<NodeTrs*>(d.nodes[n].translation);
}

__global__ __launch_bounds__(64) void anim_channels_kernel(AnimDev d, float time)
{
    const uint32_t c = blockIdx.x * 64u + threadIdx.x;
    if (c >= d.channel_count) return;
    const AnimChan ch = d.channels[c];
    NodeTrs& x = node_trs(d, ch.node);
    const uint32_t path = ch.kind & 0xFFu;
    if (path == VKGV_PATH_ROTATION) {
        float q[4];
        sample<4>(d, ch, time, q);
#pragma unroll
        for (int k = 0; k < 4; ++k) x.q[k] = q[k];
    } else {
        float v[3];
        sample<3>(d, ch, time, v);
        float* o = path == VKGV_PATH_TRANSLATION ? x.t : x.s;
#pragma unroll
        for (int k = 0; k < 3; ++k) o[k] = v[k];
    }
}

// Row r of m * b, each element ((m0*b0 + m1*b1) + m2*b2) + m3*b3 as mat4_mul's.
__device__ __forceinline__ float4 row_mul(const float4& m, const Mat4& b)
{
    float4 o;
    o.x = ((m.x * b.m[0] + m.y * b.m[1]) + m.z * b.m[2]) + m.w * b.m[3];
    o.y = ((m.x * b.m[4] + m.y * b.m[5]) + m.z * b.m[6]) + m.w * b.m[7];
    o.z = ((m.x * b.m[8] + m.y * b.m[9]) + m.z * b.m[10]) + m.w * b.m[11];
    o.w = ((m.x * b.m[12] + m.y * b.m[13]) + m.z * b.m[14]) + m.w * b.m[15];
    return o;
}

// A row of parent * T * R * S with the host traversal's operation order.
__device__ __forceinline__ float4 apply_trs(const float4& parent, const NodeTrs& n)
{
    const Mat4 T = {{ 1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0, n.t[0], n.t[1], n.t[2], 1 }};
    const float x = n.q[0], y = n.q[1], z = n.q[2], w = n.q[3];
    const Mat4 R = {{ 1.0f - 2.0f * (y * y + z * z), 2.0f * (x * y + w * z), 2.0f * (x * z - w * y), 0.0f,
                      2.0f * (x * y - w * z), 1.0f - 2.0f * (x * x + z * z), 2.0f * (y * z + w * x), 0.0f,
                      2.0f * (x * z + w * y), 2.0f * (y * z - w * x), 1.0f - 2.0f * (x * x + y * y), 0.0f,
                      0.0f, 0.0f, 0.0f, 1.0f }};
    const Mat4 S = {{ n.s[0], 0, 0, 0, 0, n.s[1], 0, 0, 0, 0, n.s[2], 0, 0, 0, 0, 1 }};
    return row_mul(row_mul(row_mul(parent, T), R), S);
}

__global__ __launch_bounds__(256) void world_transforms_kernel(AnimDev d, float* __restrict__ out,
                                                               float* __restrict__ prev)
{
    const uint32_t i = (blockIdx.x * 256u + threadIdx.x) >> 2, r = threadIdx.x & 3u;
    if (i >= d.mesh_count) return;
    float* o = out + 16ull * i + r;
    if (prev) {
        float* p = prev + 16ull * i + r;
#pragma unroll
        for (int c = 0; c < 4; ++c) p[4 * c] = o[4 * c];
    }
    float4 m = make_float4(r == 0 ? 1.0f : 0.0f, r == 1 ? 1.0f : 0.0f, r == 2 ? 1.0f : 0.0f, r == 3 ? 1.0f : 0.0f);
    const uint32_t* chain = d.chain_nodes + d.chain_first[i];
    const uint32_t len = d.chain_first[i + 1] - d.chain_first[i];   // at least the node itself
    NodeTrs next = node_trs(d, chain[0]);
    uint32_t after = len > 1 ? chain[1] : 0u;
    for (uint32_t k = 0; k < len; ++k) {
        const NodeTrs cur = next;
        if (k + 1 < len) next = node_trs(d, after);
        if (k + 2 < len) after = chain[k + 2];
        m = apply_trs(m, cur);
    }
    o[0] = m.x;
    o[4] = m.y;
    o[8] = m.z;
    o[12] = m.w;
}

} // namespace

void launch_update_transforms(const AnimDev& d, float time, float* transforms, float* prev, hipStream_t st)
{
    if (d.channel_count) anim_channels_kernel<<<(d.channel_count + 63) / 64, 64, 0, st>>>(d, time);
    if (d.mesh_count)
        world_transforms_kernel<<<(uint32_t)((4ull * d.mesh_count + 255) / 256), 256, 0, st>>>(d, transforms, prev);
}

} // namespace vkgv
