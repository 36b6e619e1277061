// What the quantized GEMMs (csrc/gemm.hip, csrc/gemm_blocks.hip) share: operand types, the store of a tile, the division of k
// over workgroups, the workspace.
#pragma once
#include "common.h"

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float float16_t __attribute__((ext_vector_type(16)));

constexpr int kBN = 64;   // workgroup tile columns (weight rows)

static inline size_t skn_align_up(size_t v) { return (v + 255) & ~(size_t)255; }

// row blocks per tile where the tile follows the rows: 32 MT rows
static inline int skn_gemm_mt(int m) { return m <= 32 ? 1 : (m <= 64 ? 2 : 4); }

// The row scales a tile's store needs: sc[r] is that of the row register r holds (store_tile).  inv_scale has a value for every row of
// the padded tiles.  Read ahead of the exchange of the partial tiles, sixteen bytes at a time: read one by one beside their stores, each
// was waited for under its own row check (Q8_0 333 x 4096 x 4096 37.3 -> 35.9 us, Q6_K 1000 x 14336 x 4096 299 -> 286).
__device__ __forceinline__ void row_scales(const float* __restrict__ inv_scale, int row0, int lane, float (&sc)[16]) {
#pragma unroll
    for (int a = 0; a < 4; a++) {
        const float4 v = *reinterpret_cast<const float4*>(inv_scale + row0 + 8 * a + 4 * (lane >> 5));
        sc[4 * a] = v.x, sc[4 * a + 1] = v.y, sc[4 * a + 2] = v.z, sc[4 * a + 3] = v.w;
    }
}

// C tile store: acc register r of lane l holds row 8*(r/4) + 4*(l/32) + r%4, column l%32 of the 32x32 tile.  What a tile is added to is
// read as a whole first (for rows and columns outside, the edge's: unused), sixteen loads in flight instead of a load, a wait and a
// store in turn: a 512-token prompt of 32 layers of width 4096, whose residual stream two products a layer are added to, 10.81 -> 10.40 ms.
__device__ __forceinline__ void store_tile(const float16_t& acc, float* __restrict__ c, int ldc, int row0, int col0, int m, int n,
                                           const float (&sc)[16], int lane, bool accumulate) {
    const int col = col0 + (lane & 31);
    float v[16];
#pragma unroll
    for (int r = 0; r < 16; r++) v[r] = acc[r] * sc[r];
    if (accumulate) {
        float old[16];
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int row = row0 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
            old[r] = c[(size_t)min(row, m - 1) * ldc + min(col, n - 1)];
        }
#pragma unroll
        for (int r = 0; r < 16; r++) v[r] += old[r];
    }
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int row = row0 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        if (row < m && col < n) c[(size_t)row * ldc + col] = v[r];
    }
}

// a partial tile of a workgroup that holds a part of k: no scale, rows of ldc
__device__ __forceinline__ void store_tile_part(const float16_t& acc, float* __restrict__ part, int ldc, int row0, int col0, int m, int n, int lane) {
    const int col = col0 + (lane & 31);
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int row = row0 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        if (row < m && col < n) part[(size_t)row * ldc + col] = acc[r];
    }
}

__device__ __forceinline__ uint32_t bf16_rne(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}

// an element of a SwiGLU pair: silu(gate) up as the bf16 that the product it goes into is defined on
__device__ __forceinline__ uint16_t swiglu_bf16(float g, float u) { return (uint16_t)bf16_rne(g / (1.0f + expf(-g)) * u); }

// Matrices that share a division of k: the parts of their products lie side by side, col0 the first column of each.
struct skn_gemm_parts {
    float* c[3];
    int n[3], col0[3], accumulate[3];
    int count;
    uint16_t* pair;  // not null: the first two are the gate and up matrices of a SwiGLU, which goes here
};

int skn_gemm_add_parts(skn_ctx* ctx, const float* part, int splits, int cols, const skn_gemm_parts& segs, const float* inv_scale, int m);
int skn_gemm_k_splits(const skn_ctx* ctx, int m, int tiles, int nb);
// grows the context's GEMM workspace; the pointer stays valid until the next growth.  `most`: what a call of the same type, m and k may need
// with another matrix, which is there after the first call outside a capture.  `ahead`: for a later call (skn_gemm_src); what a capture does
// not allow is left out.
int skn_gemm_workspace(skn_ctx* ctx, size_t bytes, size_t most, uint8_t** out, bool ahead = false);
// Room for partial products, to be asked for behind the workspace; null where there is none: k stays undivided.  What the library's
// own divisions take at most comes with the context's first workspace, so that a call allocates no more often than it would undivided
// (a caller that captures a call has run one that needed as much of the workspace).
float* skn_gemm_parts_room(skn_ctx* ctx, size_t bytes);
