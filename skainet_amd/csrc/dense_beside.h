// A residual product of a decode step as extra workgroups of another launch: resid[row] += mult * (w[row] . x) over columns whose
// input is ready before that launch's own work.  A layer whose feed-forward runs beside its mixer has its output product over the
// mixer's and the feed-forward's columns: the latter (four fifths of the matrix at a feed-forward of four widths) are taken while
// the mixer, which is a chain of latencies on a part of the chip, runs; what is left for the output product are the mixer's columns.
// Eight layers of width 2048 and a feed-forward of 8192 in bf16, context 1000: attention 8.7 us + output product 12.5 become 10.6 +
// 6.1, a step of the delta rule 5.1 + 11.5 become 10.3 + 5.4; the decode step 311 -> 292 us.  Bound by the weight stream.
#pragma once
#include "dense.h"

struct skn_beside {
    const void* w = nullptr;  // first of the columns, 16-byte aligned; null: nothing beside
    int type = SKN_TYPE_BF16;
    int rows = 0, k_pad = 0;  // k_pad: columns, a multiple of 64 (zeros from k on)
    int64_t ld = 0;           // elements from row to row
    const float* x = nullptr; // [k], 16-byte aligned
    int k = 0;
    float* resid = nullptr;
    float mult = 1.f;
    int blocks = 0;           // workgroups, set by skn_beside_plan
};

constexpr int kBesideU = 4;  // 16-byte pieces per row and lane in flight, twice
constexpr size_t kBesideMaxLds = 64 * 1024;  // of a workgroup, with the LDS of the launch's own kernel
static inline int skn_beside_plane(const skn_beside& s) {  // float4s of either plane: whole turns of a wavefront
    const int chunk = 64 * kBesideU * (s.type == SKN_TYPE_BF16 ? 8 : 4);
    return (s.k_pad + chunk - 1) / chunk * chunk / 8;
}
static inline size_t skn_beside_lds(const skn_beside& s) { return (size_t)skn_beside_plane(s) * 32; }
// own_lds: of the launch's own kernel.  No more workgroups than fit on the device at once: a staging serves all the rows that its
// wavefronts walk through.  (Delta heads of 64, feed-forwards of 14000 columns, of which two stagings fit a compute unit: three planned
// workgroups against two, two layers of width 5120, 32 steps 6.26 | 6.16 ms; width 4608 6.26 | 6.14; width 6144 6.90 | 6.89.)
static inline void skn_beside_plan(const skn_ctx* ctx, skn_beside& s, int threads, size_t own_lds) {
    const int waves = threads / 64, fit = (int)(160 * 1024 / (skn_beside_lds(s) + own_lds)), by_threads = 1536 / threads;
    const int per_cu = by_threads < fit ? by_threads : fit, most = (per_cu > 0 ? per_cu : 1) * ctx->compute_units;
    const int want = (s.rows + waves - 1) / waves;
    s.blocks = want < most ? want : most;
}

#ifdef __HIPCC__
// `block` of s.blocks, THREADS threads, lds4: skn_beside_lds bytes.  As in csrc/dense_matvec.hip: a row per wavefront and turn, the
// input in two planes of float4 (even and odd fours of elements), both buffers of weights requested ahead of its staging.
template <typename W, int THREADS>
__device__ __forceinline__ void beside_block(const skn_beside& s, int block, int plane, float4* lds4) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    constexpr int V = 16 / (int)sizeof(W), U = kBesideU, NW = THREADS / 64;
    float4 *even = lds4, *odd = lds4 + plane;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int pieces = s.k_pad / V, turns = (pieces + 64 * U - 1) / (64 * U), stride = s.blocks * NW;
    const W* w = (const W*)s.w;
    int grp = block * NW + wave, turn = 0;         // what is multiplied next
    int fetch_grp = grp, fetch_turn = 0;           // what is requested next
    u32x4 cur[U], nxt[U];
    auto fetch = [&](u32x4(&buf)[U]) __attribute__((always_inline)) {
        const u32x4* row = reinterpret_cast<const u32x4*>(w + (int64_t)min(fetch_grp, s.rows - 1) * s.ld);
#pragma unroll
        for (int u = 0; u < U; u++) buf[u] = row[min((fetch_turn * U + u) * 64 + lane, pieces - 1)];  // (past the end: times a zero of x)
        if (++fetch_turn == turns) fetch_turn = 0, fetch_grp += stride;
    };
    fetch(cur);
    fetch(nxt);
    for (int q = tid; q < 2 * plane; q += THREADS) {
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (4 * q + 3 < s.k) v = reinterpret_cast<const float4*>(s.x)[q];
        else {
            if (4 * q < s.k) v.x = s.x[4 * q];
            if (4 * q + 1 < s.k) v.y = s.x[4 * q + 1];
            if (4 * q + 2 < s.k) v.z = s.x[4 * q + 2];
        }
        ((q & 1) ? odd : even)[q >> 1] = v;
    }
    __syncthreads();
    float acc = 0.f;
    auto step = [&](u32x4(&buf)[U]) __attribute__((always_inline)) {
        // (asked for ahead of the next weights, every turn, so that the number of requests outstanding is known)
        float resid = s.resid[min(grp, s.rows - 1)];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int p = (turn * U + u) * 64 + lane;
            if constexpr (sizeof(W) == 2) {
                const float4 a = even[p], b = odd[p];
                const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    acc = fmaf(__uint_as_float(buf[u][j] << 16), x[2 * j], acc);
                    acc = fmaf(__uint_as_float(buf[u][j] & 0xFFFF0000u), x[2 * j + 1], acc);
                }
            } else {
                const float4 a = ((p & 1) ? odd : even)[p >> 1];
                const float x[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
                for (int j = 0; j < 4; j++) acc = fmaf(__uint_as_float(buf[u][j]), x[j], acc);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        fetch(buf);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" : "+v"(resid));  // (keeps the request where it is written)
        if (++turn == turns) {
            const float z = wave_sum(acc);
            if (lane == 0 && grp < s.rows) s.resid[grp] = fmaf(s.mult, z, resid);
            acc = 0.f, turn = 0, grp += stride;
        }
    };
    while (grp < s.rows) {
        step(cur);
        step(nxt);  // (past the last row: a repeat of it, not stored)
    }
}
#endif
