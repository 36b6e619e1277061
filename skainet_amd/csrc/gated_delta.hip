// Gated delta rule with a decay per key channel, behind short causal convolutions (state: rstate.h).
//
//   S <- g_t S;   u_t = beta_t (v_t - S^T k_t);   S <- S + k_t u_t^T;   o_t = S^T q_t         (g_t scales the rows of S)
//
// Everything here is fp32, the matrix instructions (v_mfma_f32_16x16x4_f32) included.  On prompts sixteen tokens (a chunk) are one
// step of the chain, as in csrc/delta.hip.  With W(s, t) the product of the factors of tokens s .. t of the chunk and S the state
// before it,
//   (I + L) U = beta (V - K0 S),   L_ts = beta_t k_t^T W(s+1, t) k_s for s < t,   K0_t = k_t W(0, t)
//   O = R0 S + G U,                R0_t = q_t W(0, t),   G_ts = q_t^T W(s+1, t) k_s for s <= t
//   S' = W(0, 15) S + sum_s k_s W(s+1, 15) u_s
// gated_chunk_kernel -- one wavefront per chunk and head, all chunks at once -- leaves V1 = (I + L)^-1 beta V, -K1 = -(I + L)^-1
// beta K0, R0, G and the decayed keys as operands; gated_scan_kernel walks the chunks: U = V1 - K1 S, and so on.
// Factors may be as small as they like (a channel may forget everything in a token), so no product of them is ever divided by
// another: the pair (s, t) is taken at the level b = 8, 4, 2 or 1 at which it falls into the two halves of a block of 2 b tokens,
// where W(s+1, t) is the product of the factors from s + 1 to the end of the lower half and those of the upper half up to t -- both
// at most one, one on each operand.
#include "delta.h"
#include "dense.h"
#include "rstate.h"

#include <algorithm>

namespace {

constexpr int kTrash = 64;  // floats behind the operands that take the outputs of tokens past the end

__device__ __forceinline__ float silu(float z) { return z * skn_sigmoid(z); }
// log2 of a channel's factor
__device__ __forceinline__ float log2_factor(float z, float rate) {
    const float softplus = z > 15.f ? z + __expf(-z) : log1pf(__expf(z));
    return -1.4426950408889634f * rate * softplus;
}

// ---- convolutions ---------------------------------------------------------------------------------------------------------------

struct ConvArgs {
    const float *q, *k, *v;  // [n][ld], this portion's inputs
    int ld, n, pos0;
    const float* ring;  // inputs of the tokens before it
    const float* taps;  // [channels][n_taps]
    int n_taps, kv_heads, dim, vcols, channels;
    float *cq, *ck, *cv;
};

constexpr int kMaxTaps = 8, kConvRows = 8;

// rows t0 .. t0 + 7 of channel c (of the ring and the taps), whose inputs in the portion are src[row * ld]; past the end: the last row
__device__ __forceinline__ void conv_rows(const ConvArgs& a, const float* src, int c, int t0, float (&y)[kConvRows]) {
    float w[kMaxTaps], x[kConvRows + kMaxTaps - 1];  // w[j]: of the input j tokens back; x[i]: of row t0 - 7 + i
#pragma unroll
    for (int j = 0; j < kMaxTaps; j++) w[j] = j < a.n_taps ? a.taps[(int64_t)c * a.n_taps + a.n_taps - 1 - j] : 0.f;
#pragma unroll
    for (int i = 0; i < kConvRows + kMaxTaps - 1; i++) {
        const int t = t0 - (kMaxTaps - 1) + i, p = a.pos0 + t;
        x[i] = 0.f;
        if (i >= kMaxTaps - a.n_taps) {
            if (t >= 0) x[i] = src[(int64_t)min(t, a.n - 1) * a.ld];
            else if (p >= 0) x[i] = a.ring[(int64_t)(p % a.n_taps) * a.channels + c];
        }
    }
#pragma unroll
    for (int r = 0; r < kConvRows; r++) {
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < kMaxTaps; j++) s = fmaf(x[r + kMaxTaps - 1 - j], w[j], s);
        y[r] = silu(s);
    }
}

// grid (rows / 8, units / 4): a wavefront takes the q or the k of a q/k head, or 64 value channels
__global__ __launch_bounds__(256) void conv_rows_kernel(const ConvArgs a) {
    const int t0 = blockIdx.x * kConvRows, unit = blockIdx.y * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, qk = a.kv_heads * a.dim;
    const int rows = min(kConvRows, a.n - t0);
    float y[4][kConvRows];
    if (unit < 2 * a.kv_heads) {
        const int which = unit & 1, head = unit >> 1;
        const float* src = (which ? a.k : a.q) + head * a.dim;
        float* dst = (which ? a.ck : a.cq) + (int64_t)t0 * a.ld + head * a.dim;
        float ss[kConvRows];
#pragma unroll
        for (int r = 0; r < kConvRows; r++) ss[r] = 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int d = lane + 64 * i;
            if (64 * i >= a.dim) break;
            conv_rows(a, src + min(d, a.dim - 1), which * qk + head * a.dim + min(d, a.dim - 1), t0, y[i]);
#pragma unroll
            for (int r = 0; r < kConvRows; r++) ss[r] = d < a.dim ? fmaf(y[i][r], y[i][r], ss[r]) : ss[r];
        }
#pragma unroll
        for (int r = 0; r < kConvRows; r++) {
            const float f = (which ? 1.0f : 1.0f / sqrtf((float)a.dim)) / sqrtf(wave_sum(ss[r]) + kUnitEps);
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (lane + 64 * i < a.dim && r < rows) dst[(int64_t)r * a.ld + lane + 64 * i] = y[i][r] * f;
        }
        return;
    }
    const int c = (unit - 2 * a.kv_heads) * 64 + lane;
    if (c >= a.vcols) return;
    conv_rows(a, a.v + c, 2 * qk + c, t0, y[0]);
#pragma unroll
    for (int r = 0; r < kConvRows; r++)
        if (r < rows) a.cv[(int64_t)(t0 + r) * a.ld + c] = y[0][r];
}

// the last tokens' inputs to the ring (after every row has read what was there); grid (channels / 256, tokens kept)
__global__ __launch_bounds__(256) void conv_keep_kernel(const ConvArgs a, float* __restrict__ ring) {
    const int c = blockIdx.x * 256 + threadIdx.x, t = a.n - 1 - (int)blockIdx.y, qk = a.kv_heads * a.dim;
    if (c >= a.channels) return;
    const float* src = c < qk ? a.q + c : c < 2 * qk ? a.k + (c - qk) : a.v + (c - 2 * qk);
    ring[(int64_t)((a.pos0 + t) % a.n_taps) * a.channels + c] = src[(int64_t)t * a.ld];
}

// ---- prompts --------------------------------------------------------------------------------------------------------------------

// Operands of a chunk and head, in floats from its start, in the layouts of csrc/delta.hip: -K1 and R0 as row operands (tiles of 16
// channels), the decayed keys by channel, G as a row operand, the factors of the whole chunk, V1 as a column operand.
__host__ __device__ constexpr int off_k1(int) { return 0; }
__host__ __device__ constexpr int off_r0(int dp) { return 16 * dp; }
__host__ __device__ constexpr int off_kt(int dp) { return 32 * dp; }
__host__ __device__ constexpr int off_g(int dp) { return 48 * dp; }
__host__ __device__ constexpr int off_w(int dp) { return 48 * dp + 256; }
__host__ __device__ constexpr int off_v(int dp) { return 49 * dp + 256; }
__host__ __device__ constexpr int chunk_floats(int dp, int vdim) { return off_v(dp) + 16 * ((vdim + 15) / 16 * 16); }

struct ChunkArgs {
    const float *q, *k, *v, *beta, *z;  // convolved q, k, v; [n][ld]
    const float* rate;                  // [heads]
    int ld, n, heads, per_kv, dim, vdim;
    float* ops;
};

template <int B>
__device__ __forceinline__ void level_factors(const float (&gl)[kChunk], float (&f)[kChunk]) {
#pragma unroll
    for (int block = 0; block < kChunk; block += 2 * B) {
        float acc = 0.f;
#pragma unroll
        for (int t = block + B; t < block + 2 * B; t++) acc += gl[t], f[t] = __builtin_amdgcn_exp2f(acc);
        acc = 0.f;
#pragma unroll
        for (int s = block + B - 1; s >= block; s--) f[s] = __builtin_amdgcn_exp2f(acc), acc += gl[s];
    }
}

// one wavefront per (chunk, head); tokens past n change nothing (q = k = v = beta = 0, factor 1)
template <int DP>
__global__ __launch_bounds__(64) void gated_chunk_kernel(const ChunkArgs p) {
    constexpr int kPitch = DP + 4, kSets = (DP + 63) / 64, kTiles = DP / 16;
    __shared__ __align__(16) float op[2][kChunk * kPitch];  // a level's q and k; then K0 and R0
    __shared__ __align__(16) float tri[2][kChunk][20];      // L, G
    const int lane = threadIdx.x, chunk = blockIdx.x, h = blockIdx.y, t0 = chunk * kChunk, t16 = lane & 15, q4 = lane >> 4;
    const int kvh = h / p.per_kv, dim = p.dim, last = p.n - 1;
    float* out = p.ops + ((int64_t)h * gridDim.x + chunk) * chunk_floats(DP, p.vdim);
    const float rate = p.rate[h];
    float beta[kChunk], q[kSets][kChunk], k[kSets][kChunk], gl[kSets][kChunk];  // this lane's channels; gl: log2 of the factors
#pragma unroll
    for (int t = 0; t < kChunk; t++) beta[t] = t0 + t < p.n ? p.beta[(int64_t)min(t0 + t, last) * p.ld + h] : 0.f;
#pragma unroll
    for (int i = 0; i < kSets; i++) {
        const int d = lane + 64 * i, dd = min(d, dim - 1);
#pragma unroll
        for (int t = 0; t < kChunk; t++) {
            const int64_t row = (int64_t)min(t0 + t, last) * p.ld;
            q[i][t] = p.q[row + kvh * dim + dd];
            k[i][t] = p.k[row + kvh * dim + dd];
            gl[i][t] = p.z[row + h * dim + dd];
        }
#pragma unroll
        for (int t = 0; t < kChunk; t++) {
            const bool in = d < dim && t0 + t < p.n;
            q[i][t] = in ? q[i][t] : 0.f;
            k[i][t] = in ? k[i][t] : 0.f;
            gl[i][t] = in ? log2_factor(gl[i][t], rate) : 0.f;
        }
    }
    // the triangles, level by level; level 0: the diagonal of G
    f32x4 kk = {0.f, 0.f, 0.f, 0.f}, qk = kk;
    auto level = [&](auto width) __attribute__((always_inline)) {
        constexpr int B = decltype(width)::value;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kSets; i++) {
            const int d = lane + 64 * i;
            if (d >= DP) continue;
            float f[kChunk];
#pragma unroll
            for (int t = 0; t < kChunk; t++) f[t] = 1.f;
            if constexpr (B > 0) level_factors<B>(gl[i], f);
#pragma unroll
            for (int t = 0; t < kChunk; t++) {
                op[0][t * kPitch + d] = q[i][t] * f[t];
                op[1][t * kPitch + d] = k[i][t] * f[t];
            }
        }
        __syncthreads();
        f32x4 x[2], y[2];
#pragma unroll
        for (int i = 0; i < 2; i++) x[i] = y[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
        for (int c = 0; c < kTiles; c++) {
            const int at = t16 * kPitch + 16 * c + 4 * q4;
            const f32x4 qv = load4(&op[0][at]), kv = load4(&op[1][at]);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if constexpr (B > 0) x[e & 1] = mma(kv[e], kv[e], x[e & 1]);
                y[e & 1] = mma(qv[e], kv[e], y[e & 1]);
            }
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int t = 4 * q4 + e, s = t16, diff = t ^ s;
            const bool mine = B == 0 ? diff == 0 : t > s && diff >= B && diff < 2 * B;
            kk[e] = mine ? x[0][e] + x[1][e] : kk[e];
            qk[e] = mine ? y[0][e] + y[1][e] : qk[e];
        }
    };
    level(std::integral_constant<int, 0>());
    level(std::integral_constant<int, 8>());
    level(std::integral_constant<int, 4>());
    level(std::integral_constant<int, 2>());
    level(std::integral_constant<int, 1>());
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int t = 4 * q4 + e, s = t16;
        tri[0][t][s] = s < t ? kk[e] : 0.f;
        tri[1][t][s] = s <= t ? qk[e] : 0.f;
    }
    __syncthreads();
    // x_t = beta_t (rhs_t - sum_{s < t} (k_t W k_s) x_s)
    auto solve = [&](float (&x)[kChunk]) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < kChunk; t++) {
#pragma unroll
            for (int s = 0; s < t; s++) x[t] = fmaf(-tri[0][t][s], x[s], x[t]);
            x[t] *= beta[t];
        }
    };
#pragma unroll
    for (int i = 0; i < kSets; i++) {
        const int d = lane + 64 * i;
        if (d >= DP) continue;
        float x[kChunk], upto = 0.f;
#pragma unroll
        for (int t = 0; t < kChunk; t++) {
            upto += gl[i][t];
            const float f = __builtin_amdgcn_exp2f(upto);
            x[t] = k[i][t] * f;
            op[1][t * kPitch + d] = q[i][t] * f;
        }
        out[off_w(DP) + d] = __builtin_amdgcn_exp2f(upto);
        solve(x);
#pragma unroll
        for (int t = 0; t < kChunk; t++) op[0][t * kPitch + d] = -x[t];
        float after = 0.f;
#pragma unroll
        for (int t = kChunk - 1; t >= 0; t--) {
            x[t] = k[i][t] * __builtin_amdgcn_exp2f(after);
            after += gl[i][t];
        }
        float* frag = out + off_kt(DP) + ((d >> 4) * 64 + (d & 15)) * 4;  // tile d / 16, lane 16 q + d % 16
#pragma unroll
        for (int q = 0; q < 4; q++) *reinterpret_cast<f32x4*>(frag + 64 * q) = f32x4{x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]};
    }
    for (int d = lane; d < (p.vdim + 15) / 16 * 16; d += 64) {
        float x[kChunk];
#pragma unroll
        for (int t = 0; t < kChunk; t++)
            x[t] = d < p.vdim && t0 + t < p.n ? p.v[(int64_t)min(t0 + t, last) * p.ld + h * p.vdim + min(d, p.vdim - 1)] : 0.f;
        solve(x);
        float* frag = out + off_v(DP) + ((d >> 4) * 64 + (d & 15)) * 4;
#pragma unroll
        for (int q = 0; q < 4; q++) *reinterpret_cast<f32x4*>(frag + 64 * q) = f32x4{x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]};
    }
    __syncthreads();
#pragma unroll 2
    for (int c = 0; c < kTiles; c++) {
        *reinterpret_cast<f32x4*>(out + off_k1(DP) + (c * 64 + lane) * 4) = load4(&op[0][t16 * kPitch + 16 * c + 4 * q4]);
        *reinterpret_cast<f32x4*>(out + off_r0(DP) + (c * 64 + lane) * 4) = load4(&op[1][t16 * kPitch + 16 * c + 4 * q4]);
    }
    *reinterpret_cast<f32x4*>(out + off_g(DP) + lane * 4) = load4(&tri[1][t16][4 * q4]);
}

template <int DP>
struct GatedOps {
    using Split = ScanSplit<DP>;
    static constexpr int kOwn = Split::kOwn, kRows = Split::kRows;
    f32x4 k1[kOwn], r0[kOwn], kt[kOwn], w[kOwn], v;
    float g[kRows];
    __device__ __forceinline__ void load(const float* p, uint32_t lane, uint32_t wave, uint32_t tile) {
        const uint32_t own = (wave * kOwn * 64 + lane) * 16, row = (16 * wave * kOwn + 4 * (lane >> 4)) * 4, some = lane * 16 + wave * kRows * 4;
#pragma unroll
        for (int i = 0; i < kOwn; i++) {
            k1[i] = load4(p + off_k1(DP) + 256 * i, own);
            r0[i] = load4(p + off_r0(DP) + 256 * i, own);
        }
        v = load4(p + off_v(DP), (tile * 64 + lane) * 16);
#pragma unroll
        for (int i = 0; i < kRows; i++) {
            g[i] = load1(p + off_g(DP) + i, some);
        }
#pragma unroll
        for (int i = 0; i < kOwn; i++) {
            w[i] = load4(p + off_w(DP) + 16 * i, row);
            kt[i] = load4(p + off_kt(DP) + 256 * i, own);
        }
    }
};

// One workgroup per head and tile of sixteen value columns, its parts of S in accumulator layout (also the layout of a column
// operand); the workgroups of a head are on one XCD (blockIdx % 8), as in delta_scan_kernel.  A chunk's matrix instructions are a
// chain on one SIMD otherwise (100 of 32 clocks at 128 channels): 2048 tokens of 16 heads of 128, one wavefront 261 us, four 121.
template <int DP>
__global__ __launch_bounds__(64 * ScanSplit<DP>::kWaves) __attribute__((amdgpu_waves_per_eu(DP <= 128 ? 2 : 1, 2))) void gated_scan_kernel(const float* __restrict__ ops, int n, int chunks, int heads, int vdim, float* __restrict__ state,
                                                        float* __restrict__ o, float* __restrict__ trash) {
    using Split = ScanSplit<DP>;
    constexpr int NW = Split::kWaves, kOwn = Split::kOwn, kRows = Split::kRows, R = DP <= 64 ? 4 : DP <= 128 ? 3 : 2;  // chunks in registers (what they hold without spilling)
    __shared__ f32x4 part_u[2][NW][64], part_z[2][NW][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int tiles = (vdim + 15) / 16, turn = (int)(blockIdx.x >> 3), h = (int)(blockIdx.x & 7) + 8 * (turn / tiles), tile = turn % tiles;
    if (h >= heads) return;
    const int col = 16 * tile + (lane & 15), size = chunk_floats(DP, vdim);
    const bool live = col < vdim;  // (lanes beyond the last column compute along and store nothing)
    float* sp = state + ((int64_t)h * vdim + min(col, vdim - 1)) * DP + 16 * wave * kOwn + 4 * (lane >> 4);
    f32x4 s[kOwn];
#pragma unroll
    for (int j = 0; j < kOwn; j++) s[j] = load4(sp + 16 * j);
    const float* src = ops + (int64_t)h * chunks * size;

    const int t_own = 4 * (lane >> 4) + wave * kRows;
    float* o_own = o + ((int64_t)t_own * heads + h) * vdim + col;
    // this wavefront's rows of the outputs of a chunk
    auto store = [&](int chunk) __attribute__((always_inline)) {
        const f32x4 z = sum_parts<NW>(part_z[chunk & 1], lane);
        // (one store per row whatever the lane, so that the number of requests outstanding is known)
#pragma unroll
        for (int i = 0; i < kRows; i++) {
            const int t = chunk * kChunk + t_own + i;
            float* dst = live && t >= 0 && t < n ? o_own + (int64_t)(chunk * kChunk + i) * heads * vdim : trash + lane;
            *dst = element(z, wave * kRows + i);
        }
    };
    auto step = [&](const GatedOps<DP>& x, int chunk) __attribute__((always_inline)) {
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        f32x4 u[2] = {zero, zero}, z[2] = {zero, zero};
#pragma unroll
        for (int j = 0; j < kOwn; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) u[e & 1] = mma(x.k1[j][e], s[j][e], u[e & 1]);
        part_u[chunk & 1][wave][lane] = u[0] + u[1];
#pragma unroll
        for (int j = 0; j < kOwn; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) z[e & 1] = mma(x.r0[j][e], s[j][e], z[e & 1]);
#pragma unroll
        for (int j = 0; j < kOwn; j++) s[j] *= x.w[j];
        lds_barrier();  // (a buffer is written again two barriers after the reads of the chunk that had it)
        const f32x4 all = x.v + sum_parts<NW>(part_u[chunk & 1], lane);
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int j = 0; j < kOwn; j++) s[j] = mma(x.kt[j][e], all[e], s[j]);
#pragma unroll
        for (int i = 0; i < kRows; i++) z[i & 1] = mma(x.g[i], element(all, wave * kRows + i), z[i & 1]);
        store(chunk - 1);
        part_z[chunk & 1][wave][lane] = z[0] + z[1];
    };
    GatedOps<DP> x[R];
#pragma unroll
    for (int r = 0; r < R - 1; r++) x[r].load(src + (int64_t)min(r, chunks - 1) * size, lane, wave, tile);
    int c = 0;
    for (; c + R <= chunks; c += R) {  // (no condition inside: the number of requests outstanding is known)
#pragma unroll
        for (int r = 0; r < R; r++) {
            x[(r + R - 1) % R].load(src + (int64_t)min(c + r + R - 1, chunks - 1) * size, lane, wave, tile);
            __builtin_amdgcn_sched_barrier(0);
            step(x[r], c + r);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int r = 0; r < R - 1; r++)
        if (c + r < chunks) step(x[r], c + r);
    lds_barrier();
    store(chunks - 1);
    if (live) {
#pragma unroll
        for (int j = 0; j < kOwn; j++) *reinterpret_cast<f32x4*>(sp + 16 * j) = s[j];
    }
}

// ---- one token --------------------------------------------------------------------------------------------------------------------

struct StepArgs {
    skn_gated_step p;
    const float* taps;
    const float* rate;
    int n_taps, heads, kv_heads, dim, vdim, channels;
    float* ring;
    float* state;
};

// Eight lanes share a row of the low-rank products: lane l has the pieces of eight columns 8 l, 64 + 8 l, ..
template <typename W>
struct Piece8;
template <>
struct Piece8<uint16_t> {
    uint4 w;
    __device__ __forceinline__ void load(const uint16_t* p) { w = *reinterpret_cast<const uint4*>(p); }
    __device__ __forceinline__ void get(float (&f)[8]) const {
        const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int j = 0; j < 4; j++) f[2 * j] = __uint_as_float(u[j] << 16), f[2 * j + 1] = __uint_as_float(u[j] & 0xFFFF0000u);
    }
};
template <>
struct Piece8<float> {
    float4 c, d;
    __device__ __forceinline__ void load(const float* p) { c = *reinterpret_cast<const float4*>(p), d = *reinterpret_cast<const float4*>(p + 4); }
    __device__ __forceinline__ void get(float (&f)[8]) const { f[0] = c.x, f[1] = c.y, f[2] = c.z, f[3] = c.w, f[4] = d.x, f[5] = d.y, f[6] = d.z, f[7] = d.w; }
};

template <typename W>
__device__ __forceinline__ float piece_dot(const Piece8<W>& row, const Vec8& t) {
    float f[8];
    row.get(f);
    const float* a = t.v;
    return ((f[0] * a[0] + f[1] * a[1]) + (f[2] * a[2] + f[3] * a[3])) + ((f[4] * a[4] + f[5] * a[5]) + (f[6] * a[6] + f[7] * a[7]));
}

// The first N pieces of a row of the low-rank products (two: ranks up to 128) and of the vector, requested ahead.
template <typename W, int N>
struct LowRank {
    Piece8<W> w[N];
    Vec8 t[N];
    __device__ __forceinline__ void load(const W* row, const float* x, int rank_pad, int l) {
#pragma unroll
        for (int i = 0; i < N; i++)
            if (64 * i < rank_pad) w[i].load(row + 64 * i + 8 * l), t[i].load(x + 64 * i + 8 * l);
    }
    // row . x over rank_pad columns (zeros of the row from its rank on); the total in all eight lanes
    __device__ __forceinline__ float dot(const W* row, const float* x, int rank_pad, int l) const {
        float z = piece_dot(w[0], t[0]);
#pragma unroll
        for (int i = 1; i < N; i++)
            if (64 * i < rank_pad) z += piece_dot(w[i], t[i]);
        for (int i = 64 * N + 8 * l; i < rank_pad; i += 64) {
            Piece8<W> p;
            Vec8 v;
            p.load(row + i), v.load(x + i);
            z += piece_dot(p, v);
        }
        return lane_group_sum<8>(z);
    }
};

// what a channel's convolution reads: the inputs j tokens back and their taps
struct ConvPoint {
    float x[kMaxTaps], w[kMaxTaps];
    int which, d, c;
};

// One workgroup of NW wavefronts per head.  It is a chain of latencies on few workgroups (a megabyte of state is 64 KB for each of
// sixteen): everything that it reads is requested before the first value is waited for -- the state, rows of both low-rank products, their
// vectors, biases, taps and the convolutions' inputs -- and two barriers are met instead of three.  Sixteen heads of 128 x 128
// behind four taps and ranks of 128: 11.9 us when one loop's requests followed the other's sums, 8.7 now.
// (Up to vdim the arguments arrive in scalar registers.)
template <int L, int NW, typename W>
__global__ __launch_bounds__(64 * NW) void gated_step_kernel(float* __restrict__ states, const int32_t* __restrict__ step, const W* __restrict__ w_a,
                                                             const float* __restrict__ a_low, const W* __restrict__ w_g, const float* __restrict__ g_low,
                                                             int rank_a_pad, int rank_g_pad, int dim, int vdim, const StepArgs a) {
    constexpr int DP = 8 * L, CW = 64 / L, kThreads = 64 * NW, kCols = NW * CW, kPasses = 256 / kCols, kGroups = kThreads / 8;  // columns per wavefront, per pass
    static_assert(kThreads >= 256, "a thread for every value channel");
    __shared__ __align__(16) float vec[3][DP];  // q, k, factors
    __shared__ float sv[256], sg[256], so[256];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = blockIdx.x, rl = lane & (L - 1), per_kv = a.heads / a.kv_heads, kvh = h / per_kv;
    const int qk = a.kv_heads * dim, n_taps = a.n_taps, l = tid & 7, r0 = tid >> 3;
    const skn_gated_step& p = a.p;
    const int pos = step[1];
    // the state first: it does not wait for anything
    Vec8 s[kPasses];
    float* sp = states + ((int64_t)h * vdim) * DP + 8 * rl;
#pragma unroll
    for (int i = 0; i < kPasses; i++)
        if (i * kCols < vdim) s[i].load(sp + (int64_t)min(i * kCols + wave * CW + lane / L, vdim - 1) * DP);
    // the first rows of factors and of gates that this group of eight lanes has (DP and vdim may hold more than one turn)
    const auto row_a = [&](int r) { return w_a + (int64_t)(h * dim + min(r, dim - 1)) * rank_a_pad; };
    const auto row_g = [&](int d) { return w_g + (int64_t)(h * vdim + min(d, vdim - 1)) * rank_g_pad; };
    // (what the registers of sixteen wavefronts hold beside the state: not all of it for 32-bit weights or 256 channels)
    constexpr bool kAheadA = L <= 16, kAheadG = L < 16 || (L == 16 && sizeof(W) == 2);
    LowRank<W, kAheadG ? 2 : 1> fa, fg;
    if (kAheadA) fa.load(row_a(r0), a_low, rank_a_pad, l);
    if (kAheadG) fg.load(row_g(r0), g_low, rank_g_pad, l);
    const float bias0 = p.bias_a[h * dim + min(r0, dim - 1)], norm = p.norm[h * vdim + min(tid, vdim - 1)];
    const float beta = p.beta[h], rate = a.rate[h];
    // convolutions: channels q, k of the head's q/k head, then v
    const int slot = pos % n_taps;
    const auto conv_load = [&](ConvPoint& v, int i) __attribute__((always_inline)) {
        v.which = i < DP ? 0 : i < 2 * DP ? 1 : 2, v.d = i - v.which * DP;
        const int d = min(v.d, (v.which < 2 ? dim : vdim) - 1);  // (past the end: a valid channel, unused)
        v.c = v.which < 2 ? v.which * qk + kvh * dim + d : 2 * qk + h * vdim + d;
        v.x[0] = (v.which == 0 ? p.q + kvh * dim : v.which == 1 ? p.k + kvh * dim : p.v + h * vdim)[d];
        const float* w = a.taps + (int64_t)v.c * n_taps;
        v.w[0] = w[n_taps - 1];
#pragma unroll
        for (int j = 1; j < kMaxTaps; j++) {
            if (j >= n_taps || j > pos) break;
            const int at = slot - j < 0 ? slot - j + n_taps : slot - j;
            v.x[j] = a.ring[(int64_t)at * a.channels + v.c];
            v.w[j] = w[n_taps - 1 - j];
        }
    };
    const auto conv_finish = [&](const ConvPoint& v) __attribute__((always_inline)) {
        if (v.which < 2 && v.d >= dim) {
            vec[v.which][v.d] = 0.f;
            return;
        }
        float y = v.x[0] * v.w[0];
#pragma unroll
        for (int j = 1; j < kMaxTaps; j++) {
            if (j >= n_taps || j > pos) break;
            y = fmaf(v.x[j], v.w[j], y);
        }
        // (this token's slot is none of those that are read; the heads that share a q/k head leave it to the first)
        if (v.which == 2 || h % per_kv == 0) a.ring[(int64_t)slot * a.channels + v.c] = v.x[0];
        if (v.which < 2) vec[v.which][v.d] = silu(y);
        else sv[v.d] = silu(y);
    };
    const int points = 2 * DP + vdim;
    {
        ConvPoint first;
        if (kAheadA && tid < points) conv_load(first, tid);
        const auto factor = [&](int r, float z, float b) {
            if (l == 0) vec[2][r] = r < dim ? __builtin_amdgcn_exp2f(log2_factor(z + b, rate)) : 0.f;
        };
        if (!kAheadA) fa.load(row_a(r0), a_low, rank_a_pad, l);
        if (r0 < DP) factor(r0, fa.dot(row_a(r0), a_low, rank_a_pad, l), bias0);
        for (int r = r0 + kGroups; r < DP; r += kGroups) {
            fa.load(row_a(r), a_low, rank_a_pad, l);
            factor(r, fa.dot(row_a(r), a_low, rank_a_pad, l), p.bias_a[h * dim + min(r, dim - 1)]);
        }
        for (int d = r0; d < vdim; d += kGroups) {
            if (!kAheadG || d != r0) fg.load(row_g(d), g_low, rank_g_pad, l);
            const float z = fg.dot(row_g(d), g_low, rank_g_pad, l);
            if (l == 0) sg[d] = skn_sigmoid(z);
        }
        if (!kAheadA && tid < points) conv_load(first, tid);
        if (tid < points) conv_finish(first);
    }
    for (int i = tid + kThreads; i < points; i += kThreads) {
        ConvPoint more;
        conv_load(more, i);
        conv_finish(more);
    }
    lds_barrier();
    float sq = 0.f, sk = 0.f;  // (every wavefront for itself)
    for (int d = lane; d < DP; d += 64) sq = fmaf(vec[0][d], vec[0][d], sq), sk = fmaf(vec[1][d], vec[1][d], sk);
    const float fq = 1.0f / (sqrtf(wave_sum(sq) + kUnitEps) * sqrtf((float)dim)), fk = 1.0f / sqrtf(wave_sum(sk) + kUnitEps);
    Vec8 q, k, g;
    q.load(&vec[0][8 * rl]);
    k.load(&vec[1][8 * rl]);
    g.load(&vec[2][8 * rl]);
#pragma unroll
    for (int j = 0; j < 8; j++) q.v[j] *= fq, k.v[j] *= fk;
#pragma unroll
    for (int i = 0; i < kPasses; i++) {
        if (i * kCols >= vdim) break;
        const int col = i * kCols + wave * CW + lane / L;
#pragma unroll
        for (int j = 0; j < 8; j++) s[i].v[j] *= g.v[j];
        const float u = beta * (sv[min(col, vdim - 1)] - dot_over_lanes<L>(k, s[i]));
#pragma unroll
        for (int j = 0; j < 8; j++) s[i].v[j] = fmaf(k.v[j], u, s[i].v[j]);
        const float o = dot_over_lanes<L>(q, s[i]);
        if (col < vdim) {
            s[i].store(sp + (int64_t)col * DP);
            if (rl == 0) so[col] = o;
        }
    }
    lds_barrier();
    if (wave * 64 >= vdim) return;
    float ss = 0.f;  // (every wavefront for itself, sixty-four channels at a time)
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float o = 64 * i + lane < vdim ? so[64 * i + lane] : 0.f;
        if (64 * i < vdim) ss += wave_sum(o * o);
    }
    const float inv = 1.0f / sqrtf(ss / (float)vdim + p.eps);
    if (tid < vdim) p.y[h * vdim + tid] = so[tid] * inv * norm * sg[tid];
}

template <int DP>
int launch_rows(skn_ctx* ctx, const skn_rstate* st, const ChunkArgs& a, float* state, float* o) {
    const int chunks = (a.n + kChunk - 1) / kChunk, tiles = (a.vdim + 15) / 16;
    skn_launch(ctx, gated_chunk_kernel<DP>, dim3(chunks, a.heads), dim3(64), 0, a);
    SKN_LAUNCH_CHECK(ctx);
    float* trash = a.ops + (size_t)chunks * a.heads * chunk_floats(DP, a.vdim);
    skn_launch(ctx, gated_scan_kernel<DP>, dim3((unsigned)((a.heads + 7) / 8 * 8 * tiles)), dim3(64 * ScanSplit<DP>::kWaves), 0, (const float*)a.ops, a.n, chunks, a.heads, a.vdim, state, o,
               trash);
    SKN_LAUNCH_CHECK(ctx);
    return SKN_OK;
}

template <int L, int NW>
int launch_step(skn_ctx* ctx, const StepArgs& a) {
    const skn_gated_step& p = a.p;
    const dim3 grid(a.heads), block(64 * NW);
    if (p.w_type == SKN_TYPE_F32)
        skn_launch(ctx, gated_step_kernel<L, NW, float>, grid, block, 0, a.state, p.state, (const float*)p.w_a, p.a_low, (const float*)p.w_g, p.g_low, p.rank_a_pad,
                   p.rank_g_pad, a.dim, a.vdim, a);
    else
        skn_launch(ctx, gated_step_kernel<L, NW, uint16_t>, grid, block, 0, a.state, p.state, (const uint16_t*)p.w_a, p.a_low, (const uint16_t*)p.w_g, p.g_low,
                   p.rank_a_pad, p.rank_g_pad, a.dim, a.vdim, a);
    SKN_LAUNCH_CHECK(ctx);
    return SKN_OK;
}

}  // namespace

size_t skn_gated_delta_pack_floats(const skn_rstate* st, int n) {
    return (size_t)((n + kChunk - 1) / kChunk) * st->heads * chunk_floats(st->dim_pad, st->vdim) + kTrash;
}

int skn_gated_delta_rows(skn_ctx* ctx, skn_rstate* st, int seq, const skn_channel_delta& p, const float* q, const float* k, const float* v, const float* beta,
                         const float* z, int ld, int n, int pos0, float* cq, float* ck, float* cv, float* pack, float* o) {
    SKN_REQUIRE(ctx, st->taps > 0, SKN_ERR_STATE, "gated delta rule: the state has no convolutions");
    SKN_REQUIRE(ctx, n > 0 && st->heads <= 65535, SKN_ERR_SHAPE, "gated delta rule: %d tokens x %d heads", n, st->heads);
    ConvArgs c = {q, k, v, ld, n, pos0, st->seq_conv(seq), p.conv, st->taps, st->kv_heads, st->dim, st->heads * st->vdim, st->channels, cq, ck, cv};
    const int units = 2 * st->kv_heads + (c.vcols + 63) / 64;
    skn_launch(ctx, conv_rows_kernel, dim3((n + kConvRows - 1) / kConvRows, (units + 3) / 4), dim3(256), 0, c);
    SKN_LAUNCH_CHECK(ctx);
    skn_launch(ctx, conv_keep_kernel, dim3((st->channels + 255) / 256, std::min(n, st->taps)), dim3(256), 0, c, st->seq_conv(seq));
    SKN_LAUNCH_CHECK(ctx);
    const ChunkArgs a = {cq, ck, cv, beta, z, p.decay_rate, ld, n, st->heads, st->heads / st->kv_heads, st->dim, st->vdim, pack};
    float* s = st->seq_state(seq);
    switch (st->dim_pad) {
        case 32: return launch_rows<32>(ctx, st, a, s, o);
        case 64: return launch_rows<64>(ctx, st, a, s, o);
        case 128: return launch_rows<128>(ctx, st, a, s, o);
        default: return launch_rows<256>(ctx, st, a, s, o);
    }
}

int skn_gated_step_launch(skn_ctx* ctx, skn_rstate* st, int seq, const skn_channel_delta& c, const skn_gated_step& p) {
    SKN_REQUIRE(ctx, st->taps > 0, SKN_ERR_STATE, "gated delta rule: the state has no convolutions");
    const StepArgs a = {p, c.conv, c.decay_rate, st->taps, st->heads, st->kv_heads, st->dim, st->vdim, st->channels, st->seq_conv(seq), st->seq_state(seq)};
    switch (st->dim_pad) {
        case 32: return launch_step<4, 4>(ctx, a);
        case 64: return launch_step<8, 8>(ctx, a);
        case 128: return launch_step<16, 16>(ctx, a);
        default: return launch_step<32, 16>(ctx, a);
    }
}

extern "C" int skn_gated_delta(skn_ctx* ctx, skn_rstate* st, int seq, const skn_channel_delta* p, const float* q_dev, const float* k_dev, const float* v_dev,
                               const float* beta_dev, const float* z_dev, int n, float* out_dev) {
    SKN_REQUIRE(nullptr, ctx != nullptr, SKN_ERR_ARG, "skn_gated_delta: ctx is null");
    SKN_REQUIRE(ctx, st && p && p->conv && p->decay_rate && q_dev && k_dev && v_dev && beta_dev && z_dev && out_dev, SKN_ERR_ARG, "skn_gated_delta: null pointer");
    SKN_REQUIRE(ctx, seq >= 0 && seq < st->n_seq && n > 0, SKN_ERR_RANGE, "skn_gated_delta: %d tokens of sequence %d of %d", n, seq, st->n_seq);
    // (the rows' kernels take one pitch: the callers' tight rows are spread to it)
    const int qk = st->kv_heads * st->dim, vc = st->heads * st->vdim, zc = st->heads * st->dim, ld = std::max(qk, std::max(vc, zc));
    const size_t col = (size_t)n * ld;
    float* m = nullptr;
    SKN_HIP(ctx, hipMalloc((void**)&m, (8 * col + skn_gated_delta_pack_floats(st, n)) * sizeof(float)));
    const float* src[5] = {q_dev, k_dev, v_dev, beta_dev, z_dev};
    const int cols[5] = {qk, qk, vc, st->heads, zc};
    int rc = SKN_OK;
    for (int i = 0; i < 5 && rc == SKN_OK; i++)
        if (hipMemcpy2DAsync(m + i * col, (size_t)ld * 4, src[i], (size_t)cols[i] * 4, (size_t)cols[i] * 4, n, hipMemcpyDeviceToDevice, ctx->stream) != hipSuccess)
            rc = skn_fail(ctx, SKN_ERR_HIP, "skn_gated_delta: copy failed");
    if (rc == SKN_OK)
        rc = skn_gated_delta_rows(ctx, st, seq, *p, m, m + col, m + 2 * col, m + 3 * col, m + 4 * col, ld, n, st->pos[seq], m + 5 * col, m + 6 * col, m + 7 * col,
                                  m + 8 * col, out_dev);
    if (rc == SKN_OK) st->pos[seq] += n;
    (void)hipStreamSynchronize(ctx->stream);
    (void)hipFree(m);
    return rc;
}
