// Launchers of the differentiable form's kernels (diff.hip).  Plain pointers;
// the torch bindings (diff_ext.cpp) own the tensors and the autograd graph.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace vkgv_diff {

// keys: C*H*W u64 set to all ones by the caller; ids / depth: C*H*W.
void raster_tris(const float* clip, const int* tris, int C, int I, int V, int T, int H, int W, int cull_back,
                 unsigned long long* keys, int* ids, float* depth, hipStream_t st);
// Vertex transform: clip [CI, V, 4] = A [CI, 4, 4] (pos [V, 3], 1), and its
// backward: g_pos [V, 3] (written) and g_A [CI, 4, 4] (accumulated into,
// zeroed by the caller).
void transform_fwd(const float* pos, const float* A, int CI, int V, float* clip, hipStream_t st);
void transform_fwd(const double* pos, const double* A, int CI, int V, double* clip, hipStream_t st);
void transform_bwd(const float* g_clip, const float* pos, const float* A, int CI, int V, float* g_pos, float* g_A,
                   hipStream_t st);
void transform_bwd(const double* g_clip, const double* pos, const double* A, int CI, int V, double* g_pos,
                   double* g_A, hipStream_t st);

// Vertex adjacency of the mesh tris [T, 3] over V vertices, for the
// backward gathers: off [2 V + 1] (off[0..V] the CSR offsets, the rest
// scratch), adj [3 T] (corner indices 3 t + k, by vertex, increasing).
void mesh_adjacency(const int* tris, int T, int V, int* off, int* adj, hipStream_t st);

// Screen boxes of every (camera, instance, triangle), for the stray flags of
// the forwards and the gathers of the backwards: tri_boxes_words(nc, I, T)
// u64 entries (nc * I * T box words, then one flag byte per triangle that the
// forwards set for the triangles with a gathered pixel).  Also clears the
// stray flags.
size_t tri_boxes_words(int nc, int I, int T);
void tri_boxes(const float* clip, const int* tris, int nc, int I, int V, int T, int H, int W,
               unsigned long long* boxes, unsigned* stray_blocks, hipStream_t st);
void tri_boxes(const double* clip, const int* tris, int nc, int I, int V, int T, int H, int W,
               unsigned long long* boxes, unsigned* stray_blocks, hipStream_t st);

// Entries of the stray flags that the forwards set and the backwards read (one
// per 256 pixels).
size_t stray_flag_count(int nc, int H, int W);

// Interpolation and antialiasing.  C is the type of the clip positions and
// their gradient, R that of attributes, images, their gradients and the
// arithmetic: (float, float), (double, double) or (double, float).  Depth
// stays float.  The forwards take the boxes of the same clip positions and
// the cleared stray flags; the backwards take them with the adjacency of tris
// and write every output (g_clip with z = 0).  shade_fwd writes both the
// interpolated colour and the antialiased one.
// Scratch: contrib, nc * H * W * 3 * (3 + A) entries for interp_bwd and
// shade_bwd and nc * H * W * 9 for aa_bwd; part, nc * I * V * A entries; the
// g_color of shade_bwd.
// render_fwd / render_bwd: projection (clip = M (pos, 1)), raster and shading
// of a mesh in one.  Scratch: snap, 16 bytes per clip position; keys, C * H * W
// entries; contrib as for shade_bwd; part_pos [render_parts][V][3] and
// part_attr [render_parts][V][A].  Kept for the backward: clip, boxes (one
// entry per camera, instance and triangle, written for those with a fragment),
// vis (as many bytes, rounded up to 4, and a word), ids, depth, color.  wide is
// scratch of render_wide_bytes, 16-byte aligned like g_M.
int render_parts(int nc, int I);
size_t render_wide_bytes(int V, int A, size_t c, size_t r);   // c, r: bytes of a C and an R
#define VKGV_DIFF_DECLARE(C, R)                                                                                       \
    void interp_fwd(const C* clip, const R* attr, const int* tris, const int* ids, int nc, int I, int V, int T, int H, \
                    int W, int A, R* out, unsigned long long* boxes, unsigned* stray_blocks, hipStream_t st);          \
    void interp_bwd(const C* clip, const R* attr, const int* tris, const int* ids, int nc, int I, int V, int T, int H, \
                    int W, int A, const unsigned long long* boxes, const unsigned* stray_blocks, const int* adj_off,   \
                    const int* adj, const R* g_out, R* contrib, R* part, C* g_clip, R* g_attr, hipStream_t st);        \
    void aa_fwd(const R* color, const C* clip, const int* tris, const int* ids, const float* depth, int nc, int I,     \
                int V, int T, int H, int W, int A, R* out, unsigned long long* boxes, unsigned* stray_blocks,          \
                hipStream_t st);                                                                                       \
    void shade_fwd(const C* clip, const R* attr, const int* tris, const int* ids, const float* depth, int nc, int I,   \
                   int V, int T, int H, int W, int A, R* color, R* out, unsigned long long* boxes,                     \
                   unsigned* stray_blocks, hipStream_t st);                                                            \
    void render_fwd(const C* pos, const C* M, const R* attr, const int* tris, int nc, int I, int V, int T, int H,      \
                    int W, int A, C* clip, void* snap, unsigned long long* keys, unsigned long long* boxes,            \
                    uint8_t* vis, int* ids, float* depth, R* color, R* out, hipStream_t st);                           \
    void render_bwd(const C* pos, const C* M, const R* attr, const int* tris, int nc, int I, int V, int T, int H,      \
                    int W, int A, const C* clip, const unsigned long long* boxes, const uint8_t* vis, const int* ids,  \
                    const float* depth, const R* color, const int* adj_off, const int* adj, const R* g_out,            \
                    R* contrib, C* part_pos, R* part_attr, void* wide, C* g_pos, C* g_M, R* g_attr, hipStream_t st);       \
    void aa_bwd(const R* color, const C* clip, const int* tris, const int* ids, const float* depth, int nc, int I,     \
                int V, int T, int H, int W, int A, const unsigned long long* boxes, const unsigned* stray_blocks,      \
                const int* adj_off, const int* adj, const R* g_out, R* contrib, R* g_color, C* g_clip,                 \
                hipStream_t st);                                                                                       \
    void shade_bwd(const R* color, const C* clip, const R* attr, const int* tris, const int* ids, const float* depth,  \
                   int nc, int I, int V, int T, int H, int W, int A, const unsigned long long* boxes,                  \
                   const unsigned* stray_blocks, const int* adj_off, const int* adj, const R* g_out, R* g_color,       \
                   R* contrib, R* part, C* g_clip, R* g_attr, hipStream_t st);

VKGV_DIFF_DECLARE(float, float)
VKGV_DIFF_DECLARE(double, double)
VKGV_DIFF_DECLARE(double, float)
#undef VKGV_DIFF_DECLARE

} // namespace vkgv_diff
