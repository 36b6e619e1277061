// Batch-1 product of a stacked dense matrix (bf16 or fp32 weights) with an fp32 vector: bound by the weight stream, and a small one by
// the chain of latencies from the launch's arguments to its last store.
//
// dense_matvec_once_kernel (most calls): a workgroup has a few rows, its wavefronts share them piece by piece, and everything is asked for
// at once.  dense_matvec_kernel (inputs whose preparation is large beside the rows of one workgroup, see csrc/dense_plan.h): the input
// is staged once per workgroup in LDS -- plain, divided group by group by its root mean square (the norm ahead
// of a layer), or with the split partials of an attention merged on the way in -- as two planes of float4 (even and odd
// fours of elements), so that the eight activations of a 16-byte piece of bf16 weights are two conflict-free 16-byte
// reads; a wavefront takes a row at a time and walks on through the stacked rows; its next requests are under way while it
// multiplies, the first ones from before the staging.  Epilogue: bias and the operation
// of the segment, or the residual sum; a key projection also goes to its page of the cache.
#include "dense.h"

#include <algorithm>
#include <type_traits>

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Workgroups of T threads of the staged kernel, us of eight wavefronts | of sixteen.  Eight where that makes at most a workgroup per compute unit (two inputs 1344 x 8192
// 7.7 | 9.4, 2048 x 8192 9.3 | 10.3), and behind a norm where the rows fill the device twice (13312 x 5120 25.5 | 27.0, behind a sum too 18496 x 2048 15.1 | 16.2) or
// are a single turn of requests long, up to three per compute unit.  Sixteen, one workgroup per compute unit, for what lies between, where the compute units with two
// workgroups of eight would be the last (two inputs 2624 x 8192 11.9 | 11.3; behind a norm 2624 x 5120 10.4 | 9.4, 4096 x 5120 11.7 | 10.9), and for more rows
// behind a plain staging (6432 x 2048 7.8 | 7.5).  Over 831 calls that it gets, by type and input, 1.00 to 1.02 times the better one's time in the mean, at worst 1.22 (two
// inputs 5120 x 8192 17.2 | 21.0: where sixteen leave a turn nearly empty).
constexpr int kPerCu = 3;
constexpr int kR = 1;  // rows per wavefront and turn (measured with two as well: slower)
constexpr int kU = 4;  // 16-byte pieces per row and lane in flight, twice
constexpr int kMaxGroups = 256, kMaxMerge = 4096, kMaxSplits = 16;  // norm groups; heads x splits and splits of a merge

struct XPlanes {
    float4* even;
    float4* odd;
    __device__ __forceinline__ float4& quad(int q) const { return (q & 1) ? odd[q >> 1] : even[q >> 1]; }
    __device__ __forceinline__ float& at(int e) const { return reinterpret_cast<float*>(&quad(e >> 2))[e & 3]; }
};

// What the staging reads first, asked for ahead of the weights: requests are answered in order, so that behind the first weights
// the input came no sooner than they did, and each vector that was asked for when it was needed cost another round trip before the
// first multiplication.  Quads tid, tid + T, ... up to RQ; longer inputs read the rest as they go.  us, before -> now: 8192 x 2048 behind a
// norm 10.2 -> 9.4, behind a sum and a norm 12.4 -> 10.9, 2624 x 2048 8.0 -> 7.2, 2048 x 2048 5.2 -> 4.6; a decode step of six layers of width
// 2048 with side tables 15 us less, of eight with a delta rule 10 us less (taken before dense_matvec_once_kernel, which has these calls now and does the
// same for all that it reads).  (The partials of a merge too, or the input of the columns beside a mixer: 0.4 and 1.1 us more.)
template <int MODE, int T>
struct Ahead {
    static constexpr bool kAdd = MODE == SKN_XSRC_ADD_NORM, kNorm = MODE == SKN_XSRC_GROUP_NORM || kAdd, kPlain = MODE == SKN_XSRC_PLAIN;
    static constexpr int RQ = kPlain ? 4 : kNorm ? 2 : 1;
    float4 x[RQ], w[kNorm ? RQ : 1], y[kAdd ? RQ : 1], yw[kAdd ? RQ : 1];
    __device__ __forceinline__ void request(const skn_matvec_src& s) {
        const int quads = kNorm ? (s.k0 + 3) >> 2 : s.k0 >> 2;
#pragma unroll
        for (int i = 0; i < RQ; i++) {
            const int q = threadIdx.x + i * T;
            if ((!kPlain && !kNorm) || q >= quads) continue;
            if constexpr (kAdd) y[i] = reinterpret_cast<const float4*>(s.add)[q], yw[i] = reinterpret_cast<const float4*>(s.add_w)[q];
            x[i] = reinterpret_cast<const float4*>(s.x0)[q];
            if constexpr (kNorm) w[i] = reinterpret_cast<const float4*>(s.norm_w)[q];
        }
        __builtin_amdgcn_sched_barrier(0);
    }
};

// f(q, i): every quad of the thread's, i its place in Ahead (a constant) or -1
template <int RQ, int T, int I = 0, typename F>
__device__ __forceinline__ void each_quad(int quads, F&& f) {
    if constexpr (I < RQ) {
        const int q = threadIdx.x + I * T;
        if (q < quads) f(q, std::integral_constant<int, I>{});
        each_quad<RQ, T, I + 1>(quads, f);
    } else {
        for (int q = threadIdx.x + RQ * T; q < quads; q += T) f(q, std::integral_constant<int, -1>{});
    }
}

template <int I, int N>
__device__ __forceinline__ float4 ahead_or(std::integral_constant<int, I>, const float4 (&ahead)[N], const float* from, int q) {
    if constexpr (I >= 0) return ahead[I];
    else return reinterpret_cast<const float4*>(from)[q];
}

template <int T>
__device__ __forceinline__ void stage_group_norm(const skn_matvec_src& s, const Ahead<SKN_XSRC_GROUP_NORM, T>& ahead, const XPlanes& xs, float* red) {
    constexpr int kWaves = T / 64, kRQ = Ahead<SKN_XSRC_GROUP_NORM, T>::RQ;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, quads = (s.k0 + 3) >> 2, gs = s.k0 / s.groups;
    // (pitches are multiples of 64 elements and their padding is zero: the last quad may be read whole)
    const bool few = s.groups <= 8 && (gs & 3) == 0;
    if (few) {
        float ss[8];
#pragma unroll
        for (int g = 0; g < 8; g++) ss[g] = 0.f;
        const float inv_quads = 4.0f / (float)gs;
        each_quad<kRQ, T>(quads, [&](int q, auto i) __attribute__((always_inline)) {
            const float4 v = ahead_or(i, ahead.x, s.x0, q);
            xs.quad(q) = v;
            const float d = (v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w);
            const int g = (int)(((float)q + 0.5f) * inv_quads);
#pragma unroll
            for (int n = 0; n < 8; n++) ss[n] += n == g ? d : 0.f;
        });
#pragma unroll
        for (int g = 0; g < 8; g++)
            if (g < s.groups) {
                const float t = wave_sum(ss[g]);
                if (lane == 0) red[g * kWaves + wave] = t;
            }
        __syncthreads();
        if (tid < s.groups) {
            float t = 0.f;
            for (int i = 0; i < kWaves; i++) t += red[tid * kWaves + i];
            red[8 * kWaves + tid] = 1.0f / sqrtf(t / (float)gs + s.eps);
        }
        __syncthreads();
        each_quad<kRQ, T>(quads, [&](int q, auto i) __attribute__((always_inline)) {
            const float r = red[8 * kWaves + (int)(((float)q + 0.5f) * inv_quads)];
            const float4 v = xs.quad(q), g = ahead_or(i, ahead.w, s.norm_w, q);
            xs.quad(q) = make_float4(v.x * r * g.x, v.y * r * g.y, v.z * r * g.z, v.w * r * g.w);
        });
        return;
    }
    for (int e = tid; e < s.k0; e += T) xs.at(e) = s.x0[e];
    __syncthreads();
    for (int g = wave; g < s.groups; g += kWaves) {
        float ss = 0.f;
        for (int e = lane; e < gs; e += 64) {
            const float v = xs.at(g * gs + e);
            ss = fmaf(v, v, ss);
        }
        ss = wave_sum(ss);
        if (lane == 0) red[g] = 1.0f / sqrtf(ss / (float)gs + s.eps);
    }
    __syncthreads();
    for (int e = tid; e < s.k0; e += T) xs.at(e) *= red[e / gs] * s.norm_w[e];
}

// the sum over the workgroup (a barrier inside; red: one float per wavefront, used once)
template <int T>
__device__ __forceinline__ float block_sum(float v, float* red) {
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    v = 0.f;
#pragma unroll
    for (int i = 0; i < T / 64; i++) v += red[i];
    return v;
}

// (pitches are multiples of 64 elements and their padding is zero, as in stage_group_norm; a thread's quads stay its own)
template <int T>
__device__ __forceinline__ void stage_add_norm(const skn_matvec_src& s, const Ahead<SKN_XSRC_ADD_NORM, T>& ahead, const XPlanes& xs, float* red) {
    constexpr int kRQ = Ahead<SKN_XSRC_ADD_NORM, T>::RQ;
    const int quads = (s.k0 + 3) >> 2;
    auto square = [](const float4& v) { return (v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w); };
    float ss = 0.f;
    each_quad<kRQ, T>(quads, [&](int q, auto i) __attribute__((always_inline)) {
        const float4 v = ahead_or(i, ahead.y, s.add, q);
        xs.quad(q) = v;
        ss += square(v);
    });
    const float ry = 1.0f / sqrtf(block_sum<T>(ss, red) / (float)s.k0 + s.eps);
    ss = 0.f;
    each_quad<kRQ, T>(quads, [&](int q, auto i) __attribute__((always_inline)) {
        const float4 y = xs.quad(q), x = ahead_or(i, ahead.x, s.x0, q);
        const float4 g = ahead_or(i, ahead.yw, s.add_w, q);
        const float4 v = make_float4(fmaf(y.x * ry, g.x, x.x), fmaf(y.y * ry, g.y, x.y), fmaf(y.z * ry, g.z, x.z), fmaf(y.w * ry, g.w, x.w));
        xs.quad(q) = v;
        if (blockIdx.x == 0) reinterpret_cast<float4*>(s.x_out)[q] = v;
        ss += square(v);
    });
    const float rx = 1.0f / sqrtf(block_sum<T>(ss, red + T / 64) / (float)s.k0 + s.eps);
    each_quad<kRQ, T>(quads, [&](int q, auto i) __attribute__((always_inline)) {
        const float4 v = xs.quad(q), g = ahead_or(i, ahead.w, s.norm_w, q);
        xs.quad(q) = make_float4(v.x * rx * g.x, v.y * rx * g.y, v.z * rx * g.z, v.w * rx * g.w);
    });
}

// red: heads x splits weights.  weights(): asks for the first weights of the product; the maxima, sums and partials that are needed
// first are asked for ahead of them (see Ahead).
template <int T, typename F>
__device__ __forceinline__ void stage_merge(const skn_matvec_src& s, const XPlanes& xs, float* red, F&& weights) {
    const int tid = threadIdx.x;
    const bool quads = (s.dim & 3) == 0;
    const int dq = s.dim >> 2;
    const int64_t step = (int64_t)s.heads * s.dim_pad;
    float2 ml0[kMaxSplits];
#pragma unroll
    for (int i = 0; i < kMaxSplits; i++) ml0[i] = reinterpret_cast<const float2*>(s.ml)[min(i, s.splits - 1) * s.heads + min(tid, s.heads - 1)];
    __builtin_amdgcn_sched_barrier(0);
    weights();
    for (int h = tid; h < s.heads; h += T) {
        float2 ml[kMaxSplits];  // (all requested before the first is used)
#pragma unroll
        for (int i = 0; i < kMaxSplits; i++) ml[i] = h == tid ? ml0[i] : reinterpret_cast<const float2*>(s.ml)[min(i, s.splits - 1) * s.heads + h];
        float m = s.sink ? 0.f : -INFINITY;
#pragma unroll
        for (int i = 0; i < kMaxSplits; i++) m = fmaxf(m, ml[i].x);
        float l = s.sink ? __builtin_amdgcn_exp2f(-m) : 0.f;
#pragma unroll
        for (int i = 0; i < kMaxSplits; i++) {
            ml[i].x = i < s.splits ? __builtin_amdgcn_exp2f(ml[i].x - m) : 0.f;  // (an empty split: exp2(-inf) = 0)
            l = fmaf(ml[i].x, ml[i].y, l);
        }
        const float inv = 1.0f / l;
#pragma unroll
        for (int i = 0; i < kMaxSplits; i++)
            if (i < s.splits) red[h * s.splits + i] = ml[i].x * inv;
    }
    __syncthreads();
    if (quads) {
        for (int q = tid; q < s.heads * dq; q += T) {
            const int h = q / dq, c = q - h * dq;
            const float* p = s.x0 + (int64_t)h * s.dim_pad + 4 * c;
            float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
            for (int i0 = 0; i0 < s.splits; i0 += 8) {
                float4 v[8];
#pragma unroll
                for (int i = 0; i < 8; i++) v[i] = *reinterpret_cast<const float4*>(p + min(i0 + i, s.splits - 1) * step);
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const float f = i0 + i < s.splits ? red[h * s.splits + i0 + i] : 0.f;
                    a.x = fmaf(f, v[i].x, a.x), a.y = fmaf(f, v[i].y, a.y), a.z = fmaf(f, v[i].z, a.z), a.w = fmaf(f, v[i].w, a.w);
                }
            }
            if (s.gate) {
                const float4 g = reinterpret_cast<const float4*>(s.gate)[q];
                a.x *= g.x, a.y *= g.y, a.z *= g.z, a.w *= g.w;
            }
            xs.quad(q) = a;
        }
        return;
    }
    for (int e = tid; e < s.k0; e += T) {
        const int h = e / s.dim, d = e - h * s.dim;
        float a = 0.f;
        for (int i = 0; i < s.splits; i++) a = fmaf(red[h * s.splits + i], s.x0[((int64_t)i * s.heads + h) * s.dim_pad + d], a);
        xs.at(e) = s.gate ? a * s.gate[e] : a;
    }
}

// W: uint16_t (bf16) or float.  LDS: two planes of `plane` float4, then the scratch of the staging.
template <typename W, int MODE, int T>
__device__ __forceinline__ void dense_matvec_rows(const W* __restrict__ w, int rows, int k_pad, int ld, int plane, const float* __restrict__ bias,
                                                  const skn_matvec_src& src, const skn_dense_out& out) {
    extern __shared__ __align__(16) float4 lds4[];
    constexpr int V = 16 / (int)sizeof(W);
    const XPlanes xs = {lds4, lds4 + plane};
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int pieces = k_pad / V;                           // 16-byte pieces of a row
    const int turns = (pieces + 64 * kU - 1) / (64 * kU);   // requests per row, kU pieces per lane each
    const int groups = (rows + kR - 1) / kR, stride = (int)gridDim.x * (T / 64);
    int grp = (int)blockIdx.x * (T / 64) + wave, turn = 0;

    u32x4 cur[kR][kU], nxt[kR][kU];
    auto fetch = [&](u32x4(&buf)[kR][kU], int g, int t) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < kR; r++) {
            const u32x4* row = reinterpret_cast<const u32x4*>(w + (int64_t)min(kR * g + r, rows - 1) * ld);
#pragma unroll
            for (int u = 0; u < kU; u++) buf[r][u] = row[min((t * kU + u) * 64 + lane, pieces - 1)];  // (past the end: times a zero of x)
        }
    };
    constexpr int kRQ = Ahead<MODE, T>::RQ;
    Ahead<MODE, T> ahead;
    ahead.request(src);
    if constexpr (MODE != SKN_XSRC_MERGE) fetch(cur, min(grp, groups - 1), 0);

    // ---- staging ----
    if constexpr (MODE == SKN_XSRC_GROUP_NORM) stage_group_norm<T>(src, ahead, xs, reinterpret_cast<float*>(lds4 + 2 * plane));
    else if constexpr (MODE == SKN_XSRC_ADD_NORM) stage_add_norm<T>(src, ahead, xs, reinterpret_cast<float*>(lds4 + 2 * plane));
    else if constexpr (MODE == SKN_XSRC_MERGE) stage_merge<T>(src, xs, reinterpret_cast<float*>(lds4 + 2 * plane), [&]() __attribute__((always_inline)) { fetch(cur, min(grp, groups - 1), 0); });
    else {
        each_quad<kRQ, T>(src.k0 >> 2, [&](int q, auto i) __attribute__((always_inline)) { xs.quad(q) = ahead_or(i, ahead.x, src.x0, q); });
        for (int e = (src.k0 & ~3) + tid; e < src.k0; e += T) xs.at(e) = src.x0[e];
    }
    if (src.x1) {
        for (int q = tid; q < src.k1 >> 2; q += T) xs.quad((src.off1 >> 2) + q) = reinterpret_cast<const float4*>(src.x1)[q];
        for (int e = (src.k1 & ~3) + tid; e < src.k1; e += T) xs.at(src.off1 + e) = src.x1[e];
    }
    {
        const int gap_end = src.x1 ? src.off1 : 8 * plane, tail = src.x1 ? src.off1 + src.k1 : 8 * plane;
        if constexpr (MODE == SKN_XSRC_GROUP_NORM || MODE == SKN_XSRC_ADD_NORM) __syncthreads();  // (its last quad may have been written past k0)
        for (int e = src.k0 + tid; e < gap_end; e += T) xs.at(e) = 0.f;
        for (int e = tail + tid; e < 8 * plane; e += T) xs.at(e) = 0.f;
    }
    __syncthreads();

    const float* bias_src = bias ? bias : reinterpret_cast<const float*>(w);
    const float* resid_src = out.nseg == 0 ? out.resid : reinterpret_cast<const float*>(w);
    const int resid_last = out.nseg == 0 ? out.resid_rows - 1 : rows - 1;
    int cache_page = 0, cache_slot = 0;
    if (out.cache_seg >= 0) {
        const int pos = *out.pos_dev;
        cache_page = out.page_table[pos / out.page_tokens];
        cache_slot = pos % out.page_tokens;
    }
    const int64_t mul_at = out.mul_seg >= 0 ? (int64_t)*out.mul_tokens * out.mul_ld + out.mul_col : 0;
    float acc[kR];
#pragma unroll
    for (int r = 0; r < kR; r++) acc[r] = 0.f;
    auto multiply = [&](const u32x4(&buf)[kR][kU], int t) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const int p = (t * kU + u) * 64 + lane;
            if constexpr (sizeof(W) == 2) {
                const float4 a = xs.even[p], b = xs.odd[p];
                const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
                for (int r = 0; r < kR; r++)
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const uint32_t d = buf[r][u][j];
                        acc[r] = fmaf(__uint_as_float(d << 16), x[2 * j], acc[r]);
                        acc[r] = fmaf(__uint_as_float(d & 0xFFFF0000u), x[2 * j + 1], acc[r]);
                    }
            } else {
                const float4 a = xs.quad(p);
                const float x[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
                for (int r = 0; r < kR; r++)
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const uint32_t d = buf[r][u][j];
                        acc[r] = fmaf(__uint_as_float(d), x[j], acc[r]);
                    }
            }
        }
    };
    auto store = [&](int g, float bias_v, float resid_v) __attribute__((always_inline)) {
        float z = 0.f;
#pragma unroll
        for (int r = 0; r < kR; r++) {
            const float t = wave_sum(acc[r]);
            z = lane == r ? t : z;
            acc[r] = 0.f;
        }
        const int row = kR * g + lane;
        if (lane >= kR || row >= rows) return;
        z += bias ? bias_v : 0.f;
        if (out.nseg == 0) {
            if (row < out.resid_rows) out.resid[row] = fmaf(out.mult, z, resid_v);
            return;
        }
        int si = -1;
        for (int q = 0; q < out.nseg; q++)
            if (kR * g >= out.seg[q].row0) si = q;  // (uniform: a group of rows does not cross segments)
        if (si < 0) return;
        const skn_dense_seg sg = out.seg[si];
        const int r = row - sg.row0;
        if (r >= sg.rows) return;
        z = skn_dense_op(sg.op, z, sg.p0, sg.p1);
        if (si == out.mul_seg) z *= skn_table_at(out.mul_table, out.mul_type, mul_at + r);
        if (sg.out_type == SKN_TYPE_F32) ((float*)sg.out)[r] = z;
        else ((uint16_t*)sg.out)[r] = skn_bf16_bits(z);
        if (si == out.cache_seg) {
            const int h = r / out.dim;
            const int64_t at = (((int64_t)cache_page * out.kv_heads + h) * out.page_tokens + cache_slot) * out.dim_pad + (r - h * out.dim);
            if (out.elem_type == SKN_TYPE_F32) ((float*)out.k_pool)[at] = z;
            else ((uint16_t*)out.k_pool)[at] = __half_as_ushort(__float2half_rn(z));
        }
    };
    // one turn on `buf` while the next turn's weights arrive in `other`
    auto step = [&](u32x4(&buf)[kR][kU], u32x4(&other)[kR][kU]) __attribute__((always_inline)) {
        const int g = grp, t = turn;
        // What the store will need is asked for ahead of the weights, or waiting for it would wait for them; every turn
        // and with whatever address there is (a row of w holds at least 128 bytes), so that the number of requests
        // outstanding is known.
        const int row = min(kR * g + (lane & (kR - 1)), rows - 1);
        float bias_v = bias_src[row], resid_v = resid_src[min(row, resid_last)];
        __builtin_amdgcn_sched_barrier(0);
        if (++turn == turns) turn = 0, grp += stride;
        fetch(other, min(grp, groups - 1), turn);  // (unconditional, so that the wait below is for a known number of newer requests)
        __builtin_amdgcn_sched_barrier(0);
        multiply(buf, t);
        asm volatile("" : "+v"(bias_v), "+v"(resid_v));  // (keeps the two requests where they are written)
        if (t == turns - 1 && g < groups) store(g, bias_v, resid_v);
        __builtin_amdgcn_sched_barrier(0);
    };
    while (grp < groups) {
        step(cur, nxt);
        step(nxt, cur);  // (past the last group: a repeat of its last rows, not stored)
    }
}

template <typename W, int MODE, int T>
__global__ __launch_bounds__(T) void dense_matvec_kernel(const W* __restrict__ w, int rows, int k_pad, int ld, int plane,
                                                         const float* __restrict__ bias, const skn_matvec_src src,
                                                         const skn_dense_out out) {
    dense_matvec_rows<W, MODE, T>(w, rows, k_pad, ld, plane, bias, src, out);
}

// Behind a norm in groups the struct comes first, so that no argument arrives in registers (build.py): us of the other order | this one, 4096 x 5120
// 11.5 | 10.9, 2624 x 5120 9.7 | 9.3, 4096 x 8192 16.6 | 16.1 (a merge is 4 % slower without: 4096 x 3072 9.6 | 10.1).
template <typename W, int T>
__global__ __launch_bounds__(T) void dense_matvec_norm_kernel(const skn_matvec_src src, const W* __restrict__ w, int rows, int k_pad, int ld, int plane,
                                                              const float* __restrict__ bias, const skn_dense_out out) {
    dense_matvec_rows<W, SKN_XSRC_GROUP_NORM, T>(w, rows, k_pad, ld, plane, bias, src, out);
}

// ---- every request at once ----------------------------------------------------------------------------------------------------
// R rows to a workgroup; each of its wavefronts has PW pieces of 1 KiB of every one of them and the same pieces of the input in its
// registers, so that the input passes neither LDS nor a barrier ahead of the products, and all that the workgroup reads is under way
// before it waits for anything.  A factor of the whole input (one norm group) goes to the results; the wavefronts' sums meet in LDS, sixteen
// threads end a row.  What a launch of a few megabytes costs beside its bytes is dependent steps: arguments that are needed
// first are single values, which the device hands a wavefront in registers (build.py), and those of an epilogue that is not taken are
// not read.  us per launch in a captured graph, weights from memory, dense_matvec_kernel -> this: 2048 x 2048 4.95 -> 3.73, 256 x 2048
// 3.42 -> 2.71, 2048 x 8192 9.0 -> 7.6, behind a norm 8192 x 2048 8.8 -> 7.9 and 32000 x 2048 24.3 -> 22.4, behind a sum and
// a norm 2624 x 2048 6.6 -> 4.8; a bare read of 8.4 MB 2.95, of 33.6 MB 6.6.  In the
// mean of a mode 1.11 (merges of sixteen) to 1.27 (plain) times as fast in bf16, 1.06 to 1.26 in fp32 (profiles/dense_matvec_once.md).
struct OnceArgs {
    const float *add, *add_w;               // of a sum
    float* x_out;
    int groups, group_size;                 // of the norm
    float eps, mult;
    int cache_seg, mul_seg;
    const float *ml, *gate;                 // of a merge
    int heads, dim, dim_pad, splits, sink;
    skn_dense_seg seg;                      // the first
    int starts[kDenseMaxSegs];              // first rows of the segments
};

// a[0..N) summed over the 64 lanes, four of them in a register: lane 16 j (and the fifteen behind it) of register i has a[index(i, j)]
template <int N>
struct LaneSums {
    static constexpr int kRegs = (N + 3) / 4, kPairs = (N + 1) / 2;
    float v[kRegs];
    __device__ __forceinline__ explicit LaneSums(const float (&a)[N]) {
        float h[kPairs];
#pragma unroll
        for (int i = 0; i < kPairs; i++) {
            const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(a[2 * i]), 2 * i + 1 < N ? __float_as_uint(a[2 * i + 1]) : 0u, false, false);
            h[i] = __uint_as_float(s[0]) + __uint_as_float(s[1]);
        }
#pragma unroll
        for (int i = 0; i < kRegs; i++) {
            const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(h[2 * i]), 2 * i + 1 < kPairs ? __float_as_uint(h[2 * i + 1]) : 0u, false, false);
            v[i] = row16_sum(__uint_as_float(s[0]) + __uint_as_float(s[1]));
        }
    }
    static __device__ __forceinline__ int index(int i, int j) { return 4 * i + (j >> 1) + 2 * (j & 1); }
};

// W: uint16_t (bf16) or float.  SP: the most splits that are merged (SKN_XSRC_MERGE).  parts: a merge keeps a hundred registers of partials, a
// sum and norm four vectors, so that these have half as many wavefronts as a plain input.
// parts_nseg: wavefronts of the workgroup, segments << 16.
template <typename W, int MODE, int PW, int R, int SP>
__global__ __launch_bounds__(64 * (MODE == SKN_XSRC_PLAIN ? kOnceParts : kOnceParts / 2)) void dense_matvec_once_kernel(
    const float* __restrict__ x_in, const void* __restrict__ w, const float* __restrict__ bias, float* resid, int k, int row_bytes, int last_piece,
    uint32_t parts_nseg, int resid_rows, const float* __restrict__ norm_w, const OnceArgs args, const skn_dense_out out) {
    constexpr int V = 16 / (int)sizeof(W), Q = V / 4;
    constexpr bool kAdd = MODE == SKN_XSRC_ADD_NORM, kNorm = MODE == SKN_XSRC_GROUP_NORM || kAdd, kMerge = MODE == SKN_XSRC_MERGE;
    constexpr int SC = SP < 8 ? SP : 8;                       // splits requested ahead
    __shared__ float sums[R][kOnceParts];                     // of rows, by part
    __shared__ float squares[kOnceGroups + 1][kOnceParts];
    const int tid = threadIdx.x, lane = tid & 63, part = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int parts = (int)(parts_nseg & 0xFFFFu), nseg = (int)(parts_nseg >> 16);
    const int row0 = (int)blockIdx.x * R;

    // ---- requests: the input's first, they are answered in order ----
    const int quad0 = (part * PW * 64 + lane) * Q;
    float4 x[PW][Q], wq[kNorm ? PW : 1][Q], y[kAdd ? PW : 1][Q], yw[kAdd ? PW : 1][Q];
    int left[PW];  // columns from the lane's first one of a piece on
    float2 ml[PW][SP];
    float4 parted[PW][SC][Q], gate[kMerge ? PW : 1][Q];
    const float* of_head[PW];
    int64_t next_split = 0;
    if constexpr (kMerge) next_split = (int64_t)args.heads * args.dim_pad;
#pragma unroll
    for (int p = 0; p < PW; p++) {
        const int quad = quad0 + p * 64 * Q;
        left[p] = k - 4 * quad;
        if constexpr (kMerge) {
            const int e = min(4 * quad, k - V), h = e / args.dim;  // (a lane's columns of a piece are of one head)
            of_head[p] = x_in + (int64_t)h * args.dim_pad + (e - h * args.dim);
#pragma unroll
            for (int i = 0; i < SP; i++) ml[p][i] = reinterpret_cast<const float2*>(args.ml)[min(i, args.splits - 1) * args.heads + h];
#pragma unroll
            for (int i = 0; i < SC; i++)
#pragma unroll
                for (int j = 0; j < Q; j++) parted[p][i][j] = reinterpret_cast<const float4*>(of_head[p] + min(i, args.splits - 1) * next_split)[j];
            if (args.gate)
#pragma unroll
                for (int j = 0; j < Q; j++) gate[p][j] = reinterpret_cast<const float4*>(args.gate + e)[j];
            continue;
        }
#pragma unroll
        for (int i = 0; i < Q; i++) {
            const uint32_t at = 16u * (uint32_t)min(quad + i, (k - 1) >> 2);
            if constexpr (kAdd) y[p][i] = *reinterpret_cast<const float4*>((const char*)args.add + at), yw[p][i] = *reinterpret_cast<const float4*>((const char*)args.add_w + at);
            x[p][i] = *reinterpret_cast<const float4*>((const char*)x_in + at);
            if constexpr (kNorm) wq[p][i] = *reinterpret_cast<const float4*>((const char*)norm_w + at);
        }
    }
    const int my = row0 + min(tid >> 4, R - 1);  // the row that this thread and fifteen others end
    const float bias_v = bias ? bias[my] : 0.f;
    const float resid_v = resid ? resid[min(my, resid_rows - 1)] : 0.f;
    __builtin_amdgcn_sched_barrier(0);
    u32x4 c[R][PW];
    const char* rows = (const char*)w + (int64_t)row0 * row_bytes;
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int p = 0; p < PW; p++)
            c[r][p] = *reinterpret_cast<const u32x4*>(rows + (int64_t)r * row_bytes + (uint32_t)min((part * PW + p) * 1024 + lane * 16, last_piece));  // (past the end: times zeros)
    __builtin_amdgcn_sched_barrier(0);

    // the segment of the workgroup's rows (a power of two of them, at most 32: they are of one segment)
    int si = 0;
    if (nseg > 1) {
#pragma unroll
        for (int q = 1; q < kDenseMaxSegs; q++) si = q < nseg && row0 >= args.starts[q] ? q : si;
    }
    const skn_dense_seg sg = nseg > 1 ? out.seg[si] : args.seg;
    int cache_page = 0, cache_slot = 0;
    if (args.cache_seg == si) {
        const int pos = *out.pos_dev;
        cache_page = out.page_table[pos / out.page_tokens];
        cache_slot = pos % out.page_tokens;
    }
    auto mul_of = [&](int row) __attribute__((always_inline)) {
        return skn_table_at(out.mul_table, out.mul_type, (int64_t)*out.mul_tokens * out.mul_ld + out.mul_col + min(row - sg.row0, sg.rows - 1));
    };
    const float mul_v = args.mul_seg == si ? mul_of(my) : 1.f;

    // ---- the input ----
    auto square = [](const float4& v) { return (v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w); };
    auto sum_of = [&](const float* from) __attribute__((always_inline)) {  // of the parts
        const float t = from[lane & (kOnceParts - 1)];
        return row16_sum((lane & (kOnceParts - 1)) < parts ? t : 0.f);
    };
    if constexpr (kMerge) {
#pragma unroll
        for (int p = 0; p < PW; p++) {
            float m = args.sink ? 0.f : -INFINITY;
#pragma unroll
            for (int i = 0; i < SP; i++) m = fmaxf(m, ml[p][i].x);
            float l = args.sink ? __builtin_amdgcn_exp2f(-m) : 0.f;
#pragma unroll
            for (int i = 0; i < SP; i++) {
                ml[p][i].x = i < args.splits ? __builtin_amdgcn_exp2f(ml[p][i].x - m) : 0.f;  // (an empty split: exp2(-inf) = 0)
                l = fmaf(ml[p][i].x, ml[p][i].y, l);
            }
            const float inv = 1.0f / l;
#pragma unroll
            for (int j = 0; j < Q; j++) x[p][j] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int i = 0; i < SP; i++) {
                const float f = ml[p][i].x * inv;
#pragma unroll
                for (int j = 0; j < Q; j++) {
                    const float4 v = i < SC ? parted[p][i % SC][j] : reinterpret_cast<const float4*>(of_head[p] + min(i, args.splits - 1) * next_split)[j];
                    float4& a = x[p][j];
                    a.x = fmaf(f, v.x, a.x), a.y = fmaf(f, v.y, a.y), a.z = fmaf(f, v.z, a.z), a.w = fmaf(f, v.w, a.w);
                }
            }
            if (args.gate)
#pragma unroll
                for (int j = 0; j < Q; j++) x[p][j].x *= gate[p][j].x, x[p][j].y *= gate[p][j].y, x[p][j].z *= gate[p][j].z, x[p][j].w *= gate[p][j].w;
        }
    }
    if (4 * (parts * PW * 64 * Q) > k) {  // (what is past the last column counts as zero)
#pragma unroll
        for (int p = 0; p < PW; p++)
#pragma unroll
            for (int i = 0; i < Q; i++) {
                const int n = left[p] - 4 * i;
                auto cut = [&](float4& v) __attribute__((always_inline)) {
                    v.x = n > 0 ? v.x : 0.f, v.y = n > 1 ? v.y : 0.f, v.z = n > 2 ? v.z : 0.f, v.w = n > 3 ? v.w : 0.f;
                };
                cut(x[p][i]);
                if constexpr (kAdd) cut(y[p][i]), cut(yw[p][i]);
                if constexpr (kNorm) cut(wq[p][i]);
            }
    }
    if constexpr (kAdd) {
        float ss = 0.f;
#pragma unroll
        for (int p = 0; p < PW; p++)
#pragma unroll
            for (int i = 0; i < Q; i++) ss += square(y[p][i]);
        ss = wave_sum(ss);
        if (lane == 0) squares[kOnceGroups][part] = ss;
        __syncthreads();
        const float ry = 1.0f / sqrtf(sum_of(squares[kOnceGroups]) / (float)k + args.eps);
#pragma unroll
        for (int p = 0; p < PW; p++)
#pragma unroll
            for (int i = 0; i < Q; i++) {
                float4& v = x[p][i];
                const float4 a = y[p][i], g = yw[p][i];
                v.x = fmaf(a.x * ry, g.x, v.x), v.y = fmaf(a.y * ry, g.y, v.y), v.z = fmaf(a.z * ry, g.z, v.z), v.w = fmaf(a.w * ry, g.w, v.w);
                if (blockIdx.x == 0 && left[p] > 4 * i) reinterpret_cast<float4*>(args.x_out)[quad0 + p * 64 * Q + i] = v;
            }
    }
    const bool one_norm = kAdd || (kNorm && args.groups == 1);  // (its factor goes to the results)
    if constexpr (kNorm) {
        if (one_norm) {
            float ss = 0.f;
#pragma unroll
            for (int p = 0; p < PW; p++)
#pragma unroll
                for (int i = 0; i < Q; i++) ss += square(x[p][i]);
            ss = wave_sum(ss);
            if (lane == 0) squares[0][part] = ss;
        } else {
            int g[PW];
            float d[PW];
#pragma unroll
            for (int p = 0; p < PW; p++) {
                g[p] = min(4 * (quad0 + p * 64 * Q), k - 1) / args.group_size;  // (a lane's columns of a piece are of one group)
                d[p] = 0.f;
#pragma unroll
                for (int i = 0; i < Q; i++) d[p] += square(x[p][i]);
            }
            for (int n = 0; n < args.groups; n++) {
                float t = 0.f;
#pragma unroll
                for (int p = 0; p < PW; p++) t += g[p] == n ? d[p] : 0.f;
                t = wave_sum(t);
                if (lane == 0) squares[n][part] = t;
            }
            __syncthreads();
#pragma unroll
            for (int p = 0; p < PW; p++) {
                float t = 0.f;
                for (int i = 0; i < parts; i++) t += squares[g[p]][i];
                const float r = 1.0f / sqrtf(t / (float)args.group_size + args.eps);
#pragma unroll
                for (int i = 0; i < Q; i++) x[p][i].x *= r, x[p][i].y *= r, x[p][i].z *= r, x[p][i].w *= r;
            }
        }
#pragma unroll
        for (int p = 0; p < PW; p++)
#pragma unroll
            for (int i = 0; i < Q; i++) {
                const float4 g = wq[p][i];
                x[p][i].x *= g.x, x[p][i].y *= g.y, x[p][i].z *= g.z, x[p][i].w *= g.w;
            }
    }

    // ---- the products ----
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        acc[r] = 0.f;
#pragma unroll
        for (int p = 0; p < PW; p++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t d = c[r][p][j];
                if constexpr (sizeof(W) == 2) {
                    const float4 v = x[p][j >> 1];
                    acc[r] = fmaf(__uint_as_float(d << 16), (j & 1) ? v.z : v.x, acc[r]);
                    acc[r] = fmaf(__uint_as_float(d & 0xFFFF0000u), (j & 1) ? v.w : v.y, acc[r]);
                } else {
                    const float4 v = x[p][0];
                    acc[r] = fmaf(__uint_as_float(d), j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w, acc[r]);
                }
            }
    }
    const LaneSums<R> total(acc);
#pragma unroll
    for (int i = 0; i < LaneSums<R>::kRegs; i++) {
        const int r = LaneSums<R>::index(i, lane >> 4);
        if ((lane & 15) == 0 && r < R) sums[r][part] = total.v[i];
    }
    __syncthreads();

    // ---- a row to sixteen threads ----
    for (int m = tid >> 4; m < R; m += 4 * parts) {
        const bool first = m == tid >> 4;  // (the only turn unless there are more than four rows to a wavefront)
        const int row = row0 + m, r = row - sg.row0;
        float z = sum_of(sums[m]);
        if (one_norm) z *= 1.0f / sqrtf(sum_of(squares[0]) / (float)k + args.eps);
        z += first ? bias_v : bias ? bias[row] : 0.f;
        if ((tid & 15) != 0) continue;
        if (resid) {
            if (row < resid_rows) resid[row] = fmaf(args.mult, z, first ? resid_v : resid[row]);
            continue;
        }
        if (r >= sg.rows) continue;
        z = skn_dense_op(sg.op, z, sg.p0, sg.p1);
        if (args.mul_seg == si) z *= first ? mul_v : mul_of(row);
        if (sg.out_type == SKN_TYPE_F32) ((float*)sg.out)[r] = z;
        else ((uint16_t*)sg.out)[r] = skn_bf16_bits(z);
        if (args.cache_seg == si) {
            const int h = r / out.dim;
            const int64_t at = (((int64_t)cache_page * out.kv_heads + h) * out.page_tokens + cache_slot) * out.dim_pad + (r - h * out.dim);
            if (out.elem_type == SKN_TYPE_F32) ((float*)out.k_pool)[at] = z;
            else ((uint16_t*)out.k_pool)[at] = __half_as_ushort(__float2half_rn(z));
        }
    }
}

template <typename W, int MODE, int PW, int R, int SP>
int launch_once(skn_ctx* ctx, const skn_dense_mat& w, const skn_matvec_src& src, const skn_dense_out& out, int parts) {
    OnceArgs a = {};
    a.add = src.add, a.add_w = src.add_w, a.x_out = src.x_out;
    a.groups = src.groups, a.group_size = src.k0 / src.groups, a.eps = src.eps, a.mult = out.mult;
    a.cache_seg = out.nseg > 0 ? out.cache_seg : -1, a.mul_seg = out.nseg > 0 ? out.mul_seg : -1;  // (the residual form has no segments)
    a.ml = src.ml, a.gate = src.gate, a.heads = src.heads, a.dim = src.dim, a.dim_pad = src.dim_pad, a.splits = src.splits, a.sink = src.sink;
    if (out.nseg > 0) a.seg = out.seg[0];
    for (int q = 0; q < out.nseg; q++) a.starts[q] = out.seg[q].row0;
    skn_launch(ctx, dense_matvec_once_kernel<W, MODE, PW, R, SP>, dim3((unsigned)(w.rows / R)), dim3(64 * parts), 0, src.x0, w.w, w.bias,
               out.nseg == 0 ? out.resid : (float*)nullptr, src.k0, (w.ld ? w.ld : w.k_pad) * (int)sizeof(W), w.k_pad * (int)sizeof(W) - 16,
               (uint32_t)(parts | out.nseg << 16), out.resid_rows, src.norm_w, a, out);
    SKN_LAUNCH_CHECK(ctx);
    return SKN_OK;
}

// SKN_ERR_TYPE, without a message: not a call for dense_matvec_once_kernel
template <typename W, int MODE>
int try_once(skn_ctx* ctx, const skn_dense_mat& w, const skn_matvec_src& src, const skn_dense_out& out) {
    skn_dense_call call = {MODE, (int)sizeof(W), w.rows, w.k_pad, w.ld ? w.ld : w.k_pad, src.k0, src.groups, src.dim, src.splits, src.x1 != nullptr, out.nseg, {}};
    for (int i = 0; i < out.nseg; i++) call.row0[i] = out.seg[i].row0;
    const skn_dense_once plan = skn_dense_once_plan(call, ctx->compute_units);
    const int r = plan.rows, parts = plan.parts;
    if (r == 0) return SKN_ERR_TYPE;
    if constexpr (MODE == SKN_XSRC_MERGE) {
        auto rows = [&](auto four) {
            constexpr int R = decltype(four)::value ? 4 : 8;
            return src.splits <= 2   ? launch_once<W, MODE, 1, R, 2>(ctx, w, src, out, parts)
                   : src.splits <= 4 ? launch_once<W, MODE, 1, R, 4>(ctx, w, src, out, parts)
                   : src.splits <= 8 ? launch_once<W, MODE, 1, R, 8>(ctx, w, src, out, parts)
                                     : launch_once<W, MODE, 1, R, 16>(ctx, w, src, out, parts);
        };
        return r == 4 ? rows(std::true_type{}) : rows(std::false_type{});
    } else if constexpr (MODE == SKN_XSRC_PLAIN) {
        if (plan.pieces == 4) return launch_once<W, MODE, 4, 4, 1>(ctx, w, src, out, parts);
        if (plan.pieces == 2) return launch_once<W, MODE, 2, 4, 1>(ctx, w, src, out, parts);
        return r == 2   ? launch_once<W, MODE, 1, 2, 1>(ctx, w, src, out, parts)
               : r == 4 ? launch_once<W, MODE, 1, 4, 1>(ctx, w, src, out, parts)
                        : launch_once<W, MODE, 1, 8, 1>(ctx, w, src, out, parts);
    } else {
        switch (r) {
            case 2: return launch_once<W, MODE, 1, 2, 1>(ctx, w, src, out, parts);
            case 4: return launch_once<W, MODE, 1, 4, 1>(ctx, w, src, out, parts);
            case 8: return launch_once<W, MODE, 1, 8, 1>(ctx, w, src, out, parts);
            default: return launch_once<W, MODE, 1, 16, 1>(ctx, w, src, out, parts);
        }
    }
}

constexpr int kMaxLds = 160 * 1024;

constexpr bool stages_norm(int mode) { return mode == SKN_XSRC_GROUP_NORM || mode == SKN_XSRC_ADD_NORM; }

template <typename W, int MODE, int T>
int launch_threads(skn_ctx* ctx, const skn_dense_mat& w, const skn_matvec_src& src, const skn_dense_out& out, int per_cu) {
    constexpr int V = 16 / (int)sizeof(W), kWaves = T / 64;
    const int chunk = 64 * kU * V;  // elements of a turn: the planes hold whole turns
    const int plane = (w.k_pad + chunk - 1) / chunk * chunk / 8;
    const size_t scratch = stages_norm(MODE) ? (kMaxGroups + 16 * kWaves) * 4 : MODE == SKN_XSRC_MERGE ? (size_t)src.heads * src.splits * 4 : 0;
    const size_t lds = (size_t)plane * 32 + scratch;
    SKN_REQUIRE(ctx, lds <= kMaxLds, SKN_ERR_SHAPE, "dense matvec: %d columns need %zu bytes of LDS (at most %d)", w.k_pad, lds, kMaxLds);
    // no more workgroups than fit on the device at once: a staging serves all the rows its wavefronts walk through
    const int groups = (w.rows + kR - 1) / kR;
    const int blocks = std::min((groups + kWaves - 1) / kWaves, std::min(per_cu, (int)(kMaxLds / lds)) * ctx->compute_units);
    const int ld = w.ld ? w.ld : w.k_pad;
    if constexpr (MODE == SKN_XSRC_GROUP_NORM) skn_launch(ctx, dense_matvec_norm_kernel<W, T>, dim3((unsigned)blocks), dim3(T), lds, src, (const W*)w.w, w.rows, w.k_pad, ld, plane, w.bias, out);
    else skn_launch(ctx, dense_matvec_kernel<W, MODE, T>, dim3((unsigned)blocks), dim3(T), lds, (const W*)w.w, w.rows, w.k_pad, ld, plane, w.bias, src, out);
    SKN_LAUNCH_CHECK(ctx);
    return SKN_OK;
}

template <typename W, int MODE>
int launch(skn_ctx* ctx, const skn_dense_mat& w, const skn_matvec_src& src, const skn_dense_out& out) {
    const int round = 8 * kR * ctx->compute_units;  // rows that a workgroup of eight wavefronts per compute unit has in hand
    const bool one_turn = w.k_pad <= 64 * kU * 16 / (int)sizeof(W);
    if (w.rows <= round || (stages_norm(MODE) && (one_turn || w.rows > 2 * round))) return launch_threads<W, MODE, 512>(ctx, w, src, out, kPerCu);
    return launch_threads<W, MODE, 1024>(ctx, w, src, out, 1);
}

template <typename W>
int launch_mode(skn_ctx* ctx, const skn_dense_mat& w, const skn_matvec_src& src, const skn_dense_out& out) {
    const int rc = src.mode == SKN_XSRC_GROUP_NORM ? try_once<W, SKN_XSRC_GROUP_NORM>(ctx, w, src, out)
                   : src.mode == SKN_XSRC_ADD_NORM ? try_once<W, SKN_XSRC_ADD_NORM>(ctx, w, src, out)
                   : src.mode == SKN_XSRC_MERGE    ? try_once<W, SKN_XSRC_MERGE>(ctx, w, src, out)
                                                   : try_once<W, SKN_XSRC_PLAIN>(ctx, w, src, out);
    if (rc != SKN_ERR_TYPE) return rc;
    if (src.mode == SKN_XSRC_GROUP_NORM) return launch<W, SKN_XSRC_GROUP_NORM>(ctx, w, src, out);
    if (src.mode == SKN_XSRC_ADD_NORM) return launch<W, SKN_XSRC_ADD_NORM>(ctx, w, src, out);
    if (src.mode == SKN_XSRC_MERGE) return launch<W, SKN_XSRC_MERGE>(ctx, w, src, out);
    return launch<W, SKN_XSRC_PLAIN>(ctx, w, src, out);
}

template <typename W, int MODE>
int allow_lds(skn_ctx* ctx) {
    if constexpr (MODE == SKN_XSRC_GROUP_NORM) {
        SKN_HIP(ctx, hipFuncSetAttribute((const void*)dense_matvec_norm_kernel<W, 512>, hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds));
        SKN_HIP(ctx, hipFuncSetAttribute((const void*)dense_matvec_norm_kernel<W, 1024>, hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds));
    } else {
        SKN_HIP(ctx, hipFuncSetAttribute((const void*)dense_matvec_kernel<W, MODE, 512>, hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds));
        SKN_HIP(ctx, hipFuncSetAttribute((const void*)dense_matvec_kernel<W, MODE, 1024>, hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds));
    }
    return SKN_OK;
}

int dense_matvec_init(skn_ctx* ctx) {
    SKN_TRY((allow_lds<uint16_t, SKN_XSRC_PLAIN>(ctx)));
    SKN_TRY((allow_lds<uint16_t, SKN_XSRC_GROUP_NORM>(ctx)));
    SKN_TRY((allow_lds<uint16_t, SKN_XSRC_ADD_NORM>(ctx)));
    SKN_TRY((allow_lds<uint16_t, SKN_XSRC_MERGE>(ctx)));
    SKN_TRY((allow_lds<float, SKN_XSRC_ADD_NORM>(ctx)));
    SKN_TRY((allow_lds<float, SKN_XSRC_PLAIN>(ctx)));
    SKN_TRY((allow_lds<float, SKN_XSRC_GROUP_NORM>(ctx)));
    return allow_lds<float, SKN_XSRC_MERGE>(ctx);
}
skn_family register_family(dense_matvec_init);

}  // namespace

int skn_dense_matvec(skn_ctx* ctx, const skn_dense_mat& w, const skn_matvec_src& src, const skn_dense_out& out) {
    SKN_REQUIRE(ctx, w.w && w.rows > 0 && w.k_pad > 0 && w.k_pad % kDenseColPad == 0 && w.ld % kDenseColPad == 0 && (w.ld == 0 || w.ld >= w.k_pad) && ((uintptr_t)w.w & 15) == 0, SKN_ERR_ARG,
                "dense matvec: bad matrix (%d x %d)", w.rows, w.k_pad);
    SKN_REQUIRE(ctx, src.x0 && ((uintptr_t)src.x0 & 15) == 0 && src.k0 > 0 && src.k0 <= w.k_pad, SKN_ERR_ARG, "dense matvec: bad input");
    SKN_REQUIRE(ctx, !src.x1 || (src.off1 >= src.k0 && src.off1 % 4 == 0 && src.off1 + src.k1 <= w.k_pad && ((uintptr_t)src.x1 & 15) == 0), SKN_ERR_ARG,
                "dense matvec: bad second input");
    SKN_REQUIRE(ctx, src.mode != SKN_XSRC_GROUP_NORM || (src.norm_w && src.groups > 0 && src.groups <= kMaxGroups && src.k0 % src.groups == 0),
                SKN_ERR_SHAPE, "dense matvec: %d norm groups of %d columns (at most %d groups)", src.groups, src.k0, kMaxGroups);
    SKN_REQUIRE(ctx, src.mode != SKN_XSRC_ADD_NORM || (src.norm_w && src.add && src.add_w && src.x_out && src.x_out != src.x0), SKN_ERR_ARG,
                "dense matvec: a sum and norm without its vectors");
    SKN_REQUIRE(ctx, out.mul_seg < 0 || (out.mul_table && out.mul_tokens), SKN_ERR_ARG, "dense matvec: no table to multiply with");
    SKN_REQUIRE(ctx, src.mode != SKN_XSRC_MERGE || (src.ml && src.splits > 0 && src.splits <= kMaxSplits && src.heads * src.splits <= kMaxMerge && src.k0 == src.heads * src.dim &&
                                                     src.dim_pad % 4 == 0),
                SKN_ERR_SHAPE, "dense matvec: cannot merge %d heads x %d splits", src.heads, src.splits);
    SKN_REQUIRE(ctx, out.nseg >= 0 && out.nseg <= kDenseMaxSegs && (out.nseg > 0 || out.resid), SKN_ERR_ARG, "dense matvec: no output");
    if (w.type == SKN_TYPE_BF16) return launch_mode<uint16_t>(ctx, w, src, out);
    if (w.type == SKN_TYPE_F32) return launch_mode<float>(ctx, w, src, out);
    return skn_fail(ctx, SKN_ERR_TYPE, "dense matvec: weights of type %d (BF16 or F32)", w.type);
}
