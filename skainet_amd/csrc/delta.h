// What the delta rules' kernels have in common: pieces of a state column, and the fp32 matrix instruction that sixteen tokens (a
// chunk) go through at a time.
#pragma once
#include "common.h"

namespace {

constexpr float kUnitEps = 1e-6f;  // under the root that makes a key a unit vector
constexpr int kChunk = 16;

typedef float f32x4 __attribute__((ext_vector_type(4)));

struct Vec8 {
    float v[8];
    __device__ __forceinline__ void load(const float* p) {
        const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
        v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
    }
    __device__ __forceinline__ void store(float* p) const {
        *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<float4*>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
    }
};

template <int L>
__device__ __forceinline__ float dot_over_lanes(const Vec8& a, const Vec8& s) {
    float x = a.v[0] * s.v[0], y = a.v[1] * s.v[1];
#pragma unroll
    for (int j = 2; j < 8; j += 2) x = fmaf(a.v[j], s.v[j], x), y = fmaf(a.v[j + 1], s.v[j + 1], y);
    return lane_group_sum<L>(x + y);
}

__device__ __forceinline__ f32x4 mma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f32x4 load4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
// of a lane's byte offset from an address that all lanes share
__device__ __forceinline__ f32x4 load4(const float* p, uint32_t bytes) { return *reinterpret_cast<const f32x4*>(reinterpret_cast<const char*>(p) + bytes); }
__device__ __forceinline__ float load1(const float* p, uint32_t bytes) { return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(p) + bytes); }

// The wavefronts that share a tile of sixteen state columns on a prompt.  Each has kOwn of the DP / 16 tiles of channels: its part
// of S, and of every product with S, whose sum over the wavefronts passes through LDS; of the products over the chunk's tokens and
// of the output rows it takes kRows in four.
template <int DP>
struct ScanSplit {
    static constexpr int kTiles = DP / 16, kWaves = kTiles < 4 ? kTiles : 4, kOwn = kTiles / kWaves, kRows = 4 / kWaves;
};
__device__ __forceinline__ float element(const f32x4& v, int e) { return e == 0 ? v[0] : e == 1 ? v[1] : e == 2 ? v[2] : v[3]; }
// what the wavefronts wrote to LDS is there (their requests to memory go on)
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
template <int NW>
__device__ __forceinline__ f32x4 sum_parts(const f32x4 (*part)[64], int lane) {
    f32x4 v = part[0][lane];
#pragma unroll
    for (int w = 1; w < NW; w++) v += part[w][lane];
    return v;
}

}  // namespace
