// Batched quantized GEMM  C[m,n] = sum_k A[m,k] * deq(W)[n,k]  (A bf16 [m,k], W GGUF blocks [n,k], C fp32 [m,n])
// on the matrix cores (v_mfma_f32_32x32x16_f16, fp32 accumulation).
//
// The tolerance asked of this op (1e-3 of max(|c|, 1e-3 * max|c|)) needs about 20 bits of every weight: a
// dequantized weight rounded to one fp16 / bf16 operand (11 / 8 bits) would miss it on outputs near zero.
// Both paths below therefore feed the MFMA with operands that are exact or exact to 2^-22:
//
//   * Activations: bf16 -> fp16 is exact for every value whose magnitude is within fp16's normal range; each
//     row is first scaled by a power of two that puts its largest magnitude just below 2^10 and the scale is
//     undone in the epilogue.  Products and sums are fp32 inside the MFMA.  Both paths read them in "fragment
//     order" (see prep_a_frag_kernel): a matrix-instruction operand is one coalesced 1 KiB load, no LDS.
//   * Weights, general path (every format but Q4_K): W is dequantized once into a workspace as an fp16 pair
//     hi = f16(w), lo = f16((w - hi) * 2^11) (hi + lo * 2^-11 = w to 2^-22 relative, or 2^-36 absolute for
//     weights in fp16's subnormal range), also in fragment order; each k-step issues two MFMAs per tile into two
//     sets of accumulators that are combined at the end.
//   * Weights, Q4_K path: see gemm_q4k_frag_kernel -- the 4-bit quants times their 6-bit sub-block scale are
//     integers below 2^10, exact in fp16, so one MFMA per k-step suffices; the f16 superblock scale d is the
//     unit in which a column's accumulators are kept.
#include "common.h"
#include "gemm_blocks.h"
#include "gemm_few.h"
#include "gemm_q6k.h"
#include "gemm_tiles.h"
#include "gemm_rows.h"

#include <algorithm>
#include <type_traits>

namespace {

// ---- Q4_K path: weights unpacked in the kernel, one MFMA per k-step, operands loaded by the wavefronts ------
// Workgroup of eight wavefronts, tile (64 MT) x 64.  The tile is divided in two along m; along k it is not
// divided spatially but by superblock: wavefront (mh, kq) computes rows [32 MT mh, 32 MT (mh + 1)) x all 64
// columns for superblocks kq, kq + 4, ..., and the four partial tiles of each half are added through LDS at
// the end.  The activations are prepared in "fragment order": for a block of 32 rows, a 64-element chunk and a
// k-step s, the 64 x 16 bytes that the 64 lanes feed to one matrix instruction are contiguous (lane l = 32 h + r
// holds row r and the eight elements that nibble dword 4 h + s of the chunk unpacks to), so a fragment is one
// coalesced 1 KiB load and never passes through LDS.  The weights of four superblocks (576 contiguous bytes of
// each of the 64 rows) are copied from global memory straight into LDS once per group of four superblocks --
// the only barrier in the loop -- from where each lane picks the 16 bytes of its row and k-step quartet.
// w[n, 256 b + e] = d * (sc_j * q) - dmin * m_j  (j = sub-block of e).  sc_j * q is an integer below 2^10: the
// nibble masked in place is the fp16 subnormal q * 2^-24 (or 16 q * 2^-24 for a high nibble) and one packed
// fp16 multiply by sc_j * 2^10 (or sc_j * 2^6) gives sc_j * q * 2^-14 exactly -- an fp16 operand the matrix
// core takes as is.  One set of accumulators: see the kernel.
// LDS pitch of a weight row: the 576 bytes of four superblocks plus one sixteen-byte pad piece.  With 576 (144 dwords,
// 16 mod 64) rows r, r + 4, r + 8, ... start in the same bank and the 128-bit reads of a wavefront's 32 rows were
// eight-fold bank conflicts; with 592 (148 dwords, 20 mod 64) sixteen consecutive rows tile all 64 banks.
constexpr int kWPieces = 37;
constexpr int kWPitch = kWPieces * 16;

// Activations bf16 [m, k] -> fragment order.  One workgroup per R rows of the padded row count (rows >= m are
// zero), one wavefront per row: the row's largest magnitude fixes its power-of-two scale, then the row is
// converted 4096 elements at a time into LDS, laid out so that the copy to global memory writes runs of 16 R
// bytes (the same sixteen bytes of R neighbouring rows).
// afrag: [row block][chunk][k-step][lane] x 8 halves.  sfrag: [row block][superblock][lane] x 8 halves: the eight
// sub-block sums of row r times 2^-12 as fp16 pairs, lanes 0..31 the "hi" parts, lanes 32..63 the "lo" parts
// (SUMS; k must then be a multiple of 256).
// The rows come from a source (skn_gemm_src): bf16 as given; fp32 rounded to bf16 (nearest even) on the way in;
// or fp32 RMS-normalized first (x * r * g, r = 1 / sqrt(mean(x^2) + eps)) -- the row-wise kernel that would
// otherwise run before the GEMM.
struct PrepRow {
    const void* a;   // the row
    const void* b;   // SKN_SRC_RMSNORM: the norm weights
    float r;         // SKN_SRC_RMSNORM: 1 / sqrt(mean(x^2) + eps)
};

// elements [i, i + 4) of the row as four bf16 bit patterns in two words
template <int SRC>
__device__ __forceinline__ void load_bf16x4(const PrepRow& row, int i, uint32_t& lo, uint32_t& hi) {
    if (SRC == SKN_SRC_BF16) {
        const u32x2 v = *reinterpret_cast<const u32x2*>((const uint16_t*)row.a + i);
        lo = v.x, hi = v.y;
        return;
    }
    const float4 x = *reinterpret_cast<const float4*>((const float*)row.a + i);
    float y[4] = {x.x, x.y, x.z, x.w};
    if (SRC == SKN_SRC_RMSNORM) {
        const float4 g = *reinterpret_cast<const float4*>((const float*)row.b + i);
        y[0] = x.x * row.r * g.x, y[1] = x.y * row.r * g.y, y[2] = x.z * row.r * g.z, y[3] = x.w * row.r * g.w;
    }
    lo = bf16_rne(y[0]) | (bf16_rne(y[1]) << 16);
    hi = bf16_rne(y[2]) | (bf16_rne(y[3]) << 16);
}

template <int R, int SRC, bool SUMS>
__global__ __launch_bounds__(64 * R) void prep_a_frag_kernel(const skn_gemm_src src, _Float16* __restrict__ afrag,
                                                            float* __restrict__ inv_scale, _Float16* __restrict__ sfrag,
                                                            int m, int k) {
    __shared__ __align__(16) u32x4 stage[512 * R];  // [chunk 64][k-step 4][half 2][row R] sixteen-byte pieces
    const int tid = threadIdx.x, lane = tid & 63, r8 = tid >> 6;
    const int row = blockIdx.x * R + r8;
    const bool real = row < m;
    const size_t row_off = (size_t)(real ? row : 0) * k;
    PrepRow ar;
    ar.a = SRC == SKN_SRC_BF16 ? (const void*)((const uint16_t*)src.a + row_off) : (const void*)((const float*)src.a + row_off);
    ar.b = src.b;
    ar.r = 1.f;
    if (SRC == SKN_SRC_RMSNORM) {
        const float* xr = (const float*)ar.a;
        float ss = 0.f;
        for (int i0 = 0; i0 < (k >> 2); i0 += 512) {
            float4 v[8];
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = reinterpret_cast<const float4*>(xr)[min(i0 + lane + 64 * j, (k >> 2) - 1)];
#pragma unroll
            for (int j = 0; j < 8; j++)
                if (i0 + lane + 64 * j < (k >> 2)) ss += (v[j].x * v[j].x + v[j].y * v[j].y) + (v[j].z * v[j].z + v[j].w * v[j].w);
        }
        ss = wave_sum(ss);
        ar.r = 1.0f / sqrtf(ss / (float)k + src.eps);
    }
    const int nch = k >> 6, nb = k >> 8;
    auto widen = [](uint32_t pair, int which) { return __uint_as_float(which ? pair & 0xFFFF0000u : pair << 16); };

    // pass 1: the row's largest finite magnitude
    float mx = 0.f;
    for (int i0 = 0; i0 < (k >> 3); i0 += 512) {  // eight loads in flight per lane
        u32x4 v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int i = 8 * min(i0 + lane + 64 * j, (k >> 3) - 1);
            uint32_t w0, w1, w2, w3;
            load_bf16x4<SRC>(ar, i, w0, w1);
            load_bf16x4<SRC>(ar, i + 4, w2, w3);
            v[j] = u32x4{w0, w1, w2, w3};
        }
#pragma unroll
        for (int j = 0; j < 8; j++)
#pragma unroll
            for (int x = 0; x < 8; x++) {
                const float f = fabsf(widen(v[j][x >> 1], x & 1));
                if (f == f && f < INFINITY) mx = fmaxf(mx, f);
            }
    }
    mx = wave_max(mx);
    if (!real) mx = 0.f;
    int e = 9;  // a zero row keeps scale 1
    if (mx > 0.f) e = (int)((__float_as_uint(mx) >> 23) & 0xFF) - 127;
    e = max(e, -100);  // (a subnormal maximum: exponent field 0)
    const float scale = real ? __uint_as_float((uint32_t)(127 + 9 - e) << 23) : 0.f;
    if (lane == 0 && real) inv_scale[row] = __uint_as_float((uint32_t)(127 - 9 + e) << 23);
    const int mb = row >> 5, r = row & 31;

    // pass 2: slabs of 4096 elements = 64 chunks = 512 tasks (chunk c, nibble dword dw), eight per lane
    for (int k0 = 0; k0 < k; k0 += 4096) {
        const int tasks = min(4096, k - k0) >> 3;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int task = lane + 64 * j;
            const int c = task >> 3, dw = task & 7;
            uint2 lo = make_uint2(0u, 0u), hi = lo;
            if (task < tasks) {
                load_bf16x4<SRC>(ar, k0 + 64 * c + 4 * dw, lo.x, lo.y);
                load_bf16x4<SRC>(ar, k0 + 64 * c + 32 + 4 * dw, hi.x, hi.y);
            }
            _Float16 l[4], u[4];
            l[0] = (_Float16)(widen(lo.x, 0) * scale), l[1] = (_Float16)(widen(lo.x, 1) * scale);
            l[2] = (_Float16)(widen(lo.y, 0) * scale), l[3] = (_Float16)(widen(lo.y, 1) * scale);
            u[0] = (_Float16)(widen(hi.x, 0) * scale), u[1] = (_Float16)(widen(hi.x, 1) * scale);
            u[2] = (_Float16)(widen(hi.y, 0) * scale), u[3] = (_Float16)(widen(hi.y, 1) * scale);
            float sl = ((float)l[0] + (float)l[1]) + ((float)l[2] + (float)l[3]);
            float su = ((float)u[0] + (float)u[1]) + ((float)u[2] + (float)u[3]);
            // totals over the eight lanes of the chunk
            sl += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(sl), 0xB1, 0xF, 0xF, true));
            su += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(su), 0xB1, 0xF, 0xF, true));
            sl += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(sl), 0x4E, 0xF, 0xF, true));
            su += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(su), 0x4E, 0xF, 0xF, true));
            sl += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(sl), 0x141, 0xF, 0xF, true));
            su += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(su), 0x141, 0xF, 0xF, true));
            half8_t o;
            o[0] = l[0], o[1] = l[2], o[2] = u[0], o[3] = u[2], o[4] = l[1], o[5] = l[3], o[6] = u[1], o[7] = u[3];
            const int h = dw >> 2, s = dw & 3;
            stage[((c * 4 + s) * 2 + h) * R + r8] = __builtin_bit_cast(u32x4, o);
            if (SUMS && dw == 0 && task < tasks) {
                _Float16 h0, h1, l0, l1;
                skn_split_hilo(sl * 0x1p-12f, h0, l0);
                skn_split_hilo(su * 0x1p-12f, h1, l1);
                const int cg = (k0 >> 6) + c;
                _Float16* sf = sfrag + ((size_t)mb * nb + (cg >> 2)) * 512 + 2 * (cg & 3);
                half2_t vh = {h0, h1}, vl = {l0, l1};
                *reinterpret_cast<half2_t*>(sf + r * 8) = vh;
                *reinterpret_cast<half2_t*>(sf + (32 + r) * 8) = vl;
            }
        }
        __syncthreads();
        // piece i = ((c 4 + s) 2 + h) R + row: R consecutive lanes write 16 R contiguous bytes
        u32x4* out = reinterpret_cast<u32x4*>(afrag) + ((size_t)mb * nch + (k0 >> 6)) * 256 + (blockIdx.x % (32 / R)) * R;
#pragma unroll
        for (int it = 0; it < 8; it++) {
            const int i = tid + 64 * R * it, csh = i / R;
            if (csh < tasks) out[(size_t)(csh >> 1) * 64 + (csh & 1) * 32 + (i % R)] = stage[i];
        }
        __syncthreads();
    }
}

// The same preparation with a row spread over four wavefronts (k <= 16384; two up to k = 1024): every element is read from memory once and
// stays in registers through the three steps that the one-wavefront-per-row kernel above makes three passes for (sum of
// squares, largest magnitude, conversion), two rows per workgroup.  Thread t of a row takes
// tasks t, t + 256, ... (task = chunk c, nibble dword dw: four elements at 64 c + 4 dw and four at 64 c + 32 + 4 dw);
// its sixteen-byte pieces go straight to their place in the fragment order.  Consecutive row pairs go to workgroups of
// one XCD (blockIdx % 8), so that the 128-byte lines they share are completed in one L2.
// Bound by the chain of latencies up to some thousand rows: the norm's weights are asked for with the row, and two wavefronts of a
// SIMD hide each other's.  us, two wavefronts a row and the weights asked for when the norm was known -> this: 512 rows of 4096 behind a
// norm 7.9 -> 7.4, 41 rows 5.8 -> 5.0 (0.1 to 0.2 of them for the order of the squares below); without a norm 2000 rows of 8192 25.2 -> 22.9,
// 512 rows of 11008 11.8 -> 11.7.
// Rows of up to 1024 elements have a task for 128 threads only: two wavefronts a row there.  us of a Q4_K call, four | two wavefronts: 4000 x
// 2048 x 256 22.7 | 20.0, 4000 x 2048 x 1024 36.1 | 32.9, 130 x 12000 x 512 16.6 | 16.2.
template <int NT, int SRC, bool SUMS, int T>
__global__ __launch_bounds__(2 * T) void prep_a_rows_kernel(const skn_gemm_src src, _Float16* __restrict__ afrag,
                                                         float* __restrict__ inv_scale, _Float16* __restrict__ sfrag,
                                                         int m, int k) {
    static_assert(T == 128 || T == 256);  // threads of a row
    __shared__ float red_ss[2][2], red_mx[2][T / 64];
    __shared__ float upper[SRC == SKN_SRC_RMSNORM && T == 256 ? 2 * NT * 128 : 1];
    const int tid = threadIdx.x, t = tid & (T - 1), rw = tid / T, wv = (tid >> 6) & (T / 64 - 1);
    const int n_pairs = gridDim.x, per_xcd = n_pairs >> 3;
    const int pair = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    const int row = 2 * pair + rw;
    const bool real = row < m;
    const size_t row_off = (size_t)(real ? row : 0) * k;
    const int tasks = k >> 3, nch = k >> 6, nb = k >> 8;
    const float* xf = (const float*)src.a + row_off;
    const uint16_t* xb = (const uint16_t*)src.a + row_off;
    float v[NT][8];
    float4 glo[SRC == SKN_SRC_RMSNORM ? NT : 1], ghi[SRC == SKN_SRC_RMSNORM ? NT : 1];
    float squares[SRC == SKN_SRC_RMSNORM ? NT : 1];
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const int task = min(t + T * j, tasks - 1), c = task >> 3, dw = task & 7;
        const int e0 = 64 * c + 4 * dw;
        if (SRC == SKN_SRC_BF16) {
            const u32x2 lo = *reinterpret_cast<const u32x2*>(xb + e0), hi = *reinterpret_cast<const u32x2*>(xb + e0 + 32);
            v[j][0] = __uint_as_float(lo.x << 16), v[j][1] = __uint_as_float(lo.x & 0xFFFF0000u);
            v[j][2] = __uint_as_float(lo.y << 16), v[j][3] = __uint_as_float(lo.y & 0xFFFF0000u);
            v[j][4] = __uint_as_float(hi.x << 16), v[j][5] = __uint_as_float(hi.x & 0xFFFF0000u);
            v[j][6] = __uint_as_float(hi.y << 16), v[j][7] = __uint_as_float(hi.y & 0xFFFF0000u);
        } else {
            const float4 lo = *reinterpret_cast<const float4*>(xf + e0), hi = *reinterpret_cast<const float4*>(xf + e0 + 32);
            v[j][0] = lo.x, v[j][1] = lo.y, v[j][2] = lo.z, v[j][3] = lo.w;
            v[j][4] = hi.x, v[j][5] = hi.y, v[j][6] = hi.z, v[j][7] = hi.w;
            if constexpr (SRC == SKN_SRC_RMSNORM) {
                glo[j] = *reinterpret_cast<const float4*>((const float*)src.b + e0);
                ghi[j] = *reinterpret_cast<const float4*>((const float*)src.b + e0 + 32);
                squares[j] = ((lo.x * lo.x + lo.y * lo.y) + (lo.z * lo.z + lo.w * lo.w)) + ((hi.x * hi.x + hi.y * hi.y) + (hi.z * hi.z + hi.w * hi.w));
            }
        }
    }
    float r = 1.f;
    if constexpr (SRC == SKN_SRC_RMSNORM) {
        // A row's sum of squares does not depend on how many wavefronts a row has: tasks u, u + 128, ... in turn (u < 128), then the
        // lanes of a wavefront, then the two halves.  The upper two wavefronts hand their tasks' sums to the lower two.
        float* const theirs = upper + (T == 256 ? rw * NT * 128 + (t & 127) : 0);
        if constexpr (T == 256) {
            if (t >= 128) {
#pragma unroll
                for (int j = 0; j < NT; j++) theirs[j * 128] = squares[j];
            }
            __syncthreads();
        }
        if (t < 128) {
            float ss = 0.f;
#pragma unroll
            for (int j = 0; j < NT; j++) {
                if (t + T * j < tasks) ss += squares[j];
                if (T == 256 && t + T * j + 128 < tasks) ss += theirs[j * 128];
            }
            ss = wave_sum(ss);
            if ((tid & 63) == 0) red_ss[rw][wv] = ss;
        }
        __syncthreads();
        r = 1.0f / sqrtf((red_ss[rw][0] + red_ss[rw][1]) / (float)k + src.eps);
    }
    // the bf16 values the GEMM is defined on (fp32 sources: rounded to nearest even here), and their largest magnitude
    float mx = 0.f;
#pragma unroll
    for (int j = 0; j < NT; j++) {
        if (SRC != SKN_SRC_BF16) {
            const float4 gl = SRC == SKN_SRC_RMSNORM ? glo[SRC == SKN_SRC_RMSNORM ? j : 0] : make_float4(1.f, 1.f, 1.f, 1.f);
            const float4 gh = SRC == SKN_SRC_RMSNORM ? ghi[SRC == SKN_SRC_RMSNORM ? j : 0] : make_float4(1.f, 1.f, 1.f, 1.f);
            const float g[8] = {gl.x, gl.y, gl.z, gl.w, gh.x, gh.y, gh.z, gh.w};
#pragma unroll
            for (int x = 0; x < 8; x++) {
                const float y = SRC == SKN_SRC_RMSNORM ? v[j][x] * r * g[x] : v[j][x];
                v[j][x] = __uint_as_float(bf16_rne(y) << 16);
            }
        }
#pragma unroll
        for (int x = 0; x < 8; x++) {
            const float f = fabsf(v[j][x]);
            if (f == f && f < INFINITY) mx = fmaxf(mx, f);
        }
    }
    mx = wave_max(mx);
    if ((tid & 63) == 0) red_mx[rw][wv] = mx;
    __syncthreads();
    mx = fmaxf(red_mx[rw][0], red_mx[rw][1]);
    if constexpr (T == 256) mx = fmaxf(mx, fmaxf(red_mx[rw][2], red_mx[rw][3]));
    if (!real) mx = 0.f;
    int e = 9;  // a zero row keeps scale 1
    if (mx > 0.f) e = (int)((__float_as_uint(mx) >> 23) & 0xFF) - 127;
    e = max(e, -100);
    const float scale = real ? __uint_as_float((uint32_t)(127 + 9 - e) << 23) : 0.f;
    if (t == 0 && real) inv_scale[row] = __uint_as_float((uint32_t)(127 - 9 + e) << 23);
    const int mb = row >> 5, rr = row & 31;
    u32x4* out = reinterpret_cast<u32x4*>(afrag) + (size_t)mb * nch * 256 + rr;
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const int task = t + T * j, c = task >> 3, dw = task & 7;
        _Float16 l[4], u[4];
#pragma unroll
        for (int x = 0; x < 4; x++) l[x] = (_Float16)(v[j][x] * scale), u[x] = (_Float16)(v[j][4 + x] * scale);
        float sl = ((float)l[0] + (float)l[1]) + ((float)l[2] + (float)l[3]);
        float su = ((float)u[0] + (float)u[1]) + ((float)u[2] + (float)u[3]);
        if (SUMS) {  // totals over the eight lanes of the chunk
            sl += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(sl), 0xB1, 0xF, 0xF, true));
            su += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(su), 0xB1, 0xF, 0xF, true));
            sl += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(sl), 0x4E, 0xF, 0xF, true));
            su += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(su), 0x4E, 0xF, 0xF, true));
            sl += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(sl), 0x141, 0xF, 0xF, true));
            su += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(su), 0x141, 0xF, 0xF, true));
        }
        if (task < tasks) {
            half8_t o;
            o[0] = l[0], o[1] = l[2], o[2] = u[0], o[3] = u[2], o[4] = l[1], o[5] = l[3], o[6] = u[1], o[7] = u[3];
            const int h = dw >> 2, sq = dw & 3;
            out[((size_t)c * 4 + sq) * 64 + h * 32] = __builtin_bit_cast(u32x4, o);
            if (SUMS && dw == 0) {
                _Float16 h0, h1, l0, l1;
                skn_split_hilo(sl * 0x1p-12f, h0, l0);
                skn_split_hilo(su * 0x1p-12f, h1, l1);
                _Float16* sf = sfrag + ((size_t)mb * nb + (c >> 2)) * 512 + 2 * (c & 3);
                half2_t vh = {h0, h1}, vl = {l0, l1};
                *reinterpret_cast<half2_t*>(sf + rr * 8) = vh;
                *reinterpret_cast<half2_t*>(sf + (32 + rr) * 8) = vl;
            }
        }
    }
}

// The same with four rows per workgroup, sixteen lanes of a wavefront on each, T threads a row (128; 256 where a row's elements would take too many
// registers).  The kernel above writes sixteen bytes a lane, 512 bytes apart: two million requests for 2000 rows of 8192, which the L2 takes
// one by one.  Here the lanes exchange their pieces before the store, so that four of them write the 64 bytes that four neighbouring rows have of
// a fragment.  A row's squares are added in the same order as above.
// bf16 rows, us, two rows a workgroup -> four: 2000 x 4096 12.6 -> 10.0, 2000 x 8192 20.0 -> 14.1, 4000 x 8192 31.8 -> 24.0, 2000 x 11008 25.3 -> 21.2.
template <int NT, int SRC, bool SUMS, int T>
__global__ __launch_bounds__(4 * T) void prep_a_quads_kernel(const skn_gemm_src src, _Float16* __restrict__ afrag, float* __restrict__ inv_scale,
                                                             _Float16* __restrict__ sfrag, int m, int k) {
    constexpr bool kNorm = SRC == SKN_SRC_RMSNORM;
    constexpr int W = T / 16;  // wavefronts
    static_assert(T == 128 || (T == 256 && !kNorm), "the order of the squares is that of 128 threads");
    __shared__ float red_ss[kNorm ? 4 : 1][W], red_mx[4][W];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, rw = lane >> 4, t = wave * 16 + (lane & 15);
    const int per_xcd = gridDim.x >> 3, quad = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3), row = 4 * quad + rw;
    const bool real = row < m;
    const size_t row_off = (size_t)(real ? row : 0) * k;
    const int tasks = k >> 3, nch = k >> 6, nb = k >> 8;
    const float* xf = (const float*)src.a + row_off;
    const uint16_t* xb = (const uint16_t*)src.a + row_off;
    float v[NT][8];
    float4 glo[kNorm ? NT : 1], ghi[kNorm ? NT : 1];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const int task = min(t + T * j, tasks - 1), c = task >> 3, dw = task & 7;
        const int e0 = 64 * c + 4 * dw;
        if (SRC == SKN_SRC_BF16) {
            const u32x2 lo = *reinterpret_cast<const u32x2*>(xb + e0), hi = *reinterpret_cast<const u32x2*>(xb + e0 + 32);
            v[j][0] = __uint_as_float(lo.x << 16), v[j][1] = __uint_as_float(lo.x & 0xFFFF0000u);
            v[j][2] = __uint_as_float(lo.y << 16), v[j][3] = __uint_as_float(lo.y & 0xFFFF0000u);
            v[j][4] = __uint_as_float(hi.x << 16), v[j][5] = __uint_as_float(hi.x & 0xFFFF0000u);
            v[j][6] = __uint_as_float(hi.y << 16), v[j][7] = __uint_as_float(hi.y & 0xFFFF0000u);
        } else {
            const float4 lo = *reinterpret_cast<const float4*>(xf + e0), hi = *reinterpret_cast<const float4*>(xf + e0 + 32);
            v[j][0] = lo.x, v[j][1] = lo.y, v[j][2] = lo.z, v[j][3] = lo.w;
            v[j][4] = hi.x, v[j][5] = hi.y, v[j][6] = hi.z, v[j][7] = hi.w;
            if constexpr (kNorm) {
                glo[j] = *reinterpret_cast<const float4*>((const float*)src.b + e0);
                ghi[j] = *reinterpret_cast<const float4*>((const float*)src.b + e0 + 32);
            }
        }
    }
    float r = 1.f;
    if constexpr (kNorm) {
        // tasks t, t + 128, ... in turn, then the lanes of sixteen, then the sixteens as a wavefront's sum and the two halves add them
#pragma unroll
        for (int j = 0; j < NT; j++)
            if (t + T * j < tasks) ss += ((v[j][0] * v[j][0] + v[j][1] * v[j][1]) + (v[j][2] * v[j][2] + v[j][3] * v[j][3])) +
                                         ((v[j][4] * v[j][4] + v[j][5] * v[j][5]) + (v[j][6] * v[j][6] + v[j][7] * v[j][7]));
        ss = lane_group_sum<16>(ss);
        if ((lane & 15) == 0) red_ss[rw][wave] = ss;
        __syncthreads();
        const float* z = red_ss[rw];
        r = 1.0f / sqrtf((((z[0] + z[1]) + (z[2] + z[3])) + ((z[4] + z[5]) + (z[6] + z[7]))) / (float)k + src.eps);
    }
    // the bf16 values the GEMM is defined on (fp32 sources: rounded to nearest even here), and their largest magnitude
    float mx = 0.f;
#pragma unroll
    for (int j = 0; j < NT; j++) {
        if (SRC != SKN_SRC_BF16) {
            const float4 gl = kNorm ? glo[kNorm ? j : 0] : make_float4(1.f, 1.f, 1.f, 1.f);
            const float4 gh = kNorm ? ghi[kNorm ? j : 0] : make_float4(1.f, 1.f, 1.f, 1.f);
            const float g[8] = {gl.x, gl.y, gl.z, gl.w, gh.x, gh.y, gh.z, gh.w};
#pragma unroll
            for (int x = 0; x < 8; x++) {
                const float y = kNorm ? v[j][x] * r * g[x] : v[j][x];
                v[j][x] = __uint_as_float(bf16_rne(y) << 16);
            }
        }
#pragma unroll
        for (int x = 0; x < 8; x++) {
            const float f = fabsf(v[j][x]);
            if (f == f && f < INFINITY) mx = fmaxf(mx, f);
        }
    }
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
    if ((lane & 15) == 0) red_mx[rw][wave] = mx;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < W; i++) mx = fmaxf(mx, red_mx[rw][i]);
    if (!real) mx = 0.f;
    int e = 9;  // a zero row keeps scale 1
    if (mx > 0.f) e = (int)((__float_as_uint(mx) >> 23) & 0xFF) - 127;
    e = max(e, -100);
    const float scale = real ? __uint_as_float((uint32_t)(127 + 9 - e) << 23) : 0.f;
    if (t == 0 && real) inv_scale[row] = __uint_as_float((uint32_t)(127 - 9 + e) << 23);
    const int mb = row >> 5, rr = row & 31;  // (a quad lies in one row block)
    // lane 4 i + r of the store has piece i of the wavefront's sixteen and row r of its four
    const int from = 4 * (16 * (lane & 3) + (lane >> 2)), to_row = 4 * (quad & 7) + (lane & 3);
    u32x4* out = reinterpret_cast<u32x4*>(afrag) + (size_t)mb * nch * 256 + to_row;
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const int task = t + T * j, c = task >> 3, dw = task & 7;
        _Float16 l[4], u[4];
#pragma unroll
        for (int x = 0; x < 4; x++) l[x] = (_Float16)(v[j][x] * scale), u[x] = (_Float16)(v[j][4 + x] * scale);
        half8_t o;
        o[0] = l[0], o[1] = l[2], o[2] = u[0], o[3] = u[2], o[4] = l[1], o[5] = l[3], o[6] = u[1], o[7] = u[3];
        const u32x4 mine = __builtin_bit_cast(u32x4, o);
        u32x4 theirs;
#pragma unroll
        for (int x = 0; x < 4; x++) theirs[x] = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)mine[x]);
        const int their_task = wave * 16 + (lane >> 2) + T * j, tc = their_task >> 3, tdw = their_task & 7;
        if (their_task < tasks) out[((size_t)tc * 4 + (tdw & 3)) * 64 + (tdw >> 2) * 32] = theirs;
        if (SUMS) {  // totals over the eight lanes of the chunk
            float sl = ((float)l[0] + (float)l[1]) + ((float)l[2] + (float)l[3]);
            float su = ((float)u[0] + (float)u[1]) + ((float)u[2] + (float)u[3]);
            sl += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(sl), 0xB1, 0xF, 0xF, true));
            su += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(su), 0xB1, 0xF, 0xF, true));
            sl += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(sl), 0x4E, 0xF, 0xF, true));
            su += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(su), 0x4E, 0xF, 0xF, true));
            sl += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(sl), 0x141, 0xF, 0xF, true));
            su += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(su), 0x141, 0xF, 0xF, true));
            if (dw == 0 && task < tasks) {
                _Float16 h0, h1, l0, l1;
                skn_split_hilo(sl * 0x1p-12f, h0, l0);
                skn_split_hilo(su * 0x1p-12f, h1, l1);
                _Float16* sf = sfrag + ((size_t)mb * nb + (c >> 2)) * 512 + 2 * (c & 3);
                half2_t vh = {h0, h1}, vl = {l0, l1};
                *reinterpret_cast<half2_t*>(sf + rr * 8) = vh;
                *reinterpret_cast<half2_t*>(sf + (32 + rr) * 8) = vl;
            }
        }
    }
}

template <int SRC, bool SUMS>
void launch_prep(skn_ctx* ctx, const skn_gemm_src& src, _Float16* afrag, float* isc, _Float16* sfrag, int m, int m_pad, int k) {
    // (m_pad is a multiple of 32: the pair count divides by the eight XCDs its workgroups are dealt to)
    // Four rows a workgroup where those fill the device, without a norm to wait for half of it (two rows | four, us: 333 x 4096 7.1 | 7.3, 512 x 4096
    // 7.2 | 7.0, behind a norm 7.4 | 7.9, 2000 x 2048 behind a norm 10.9 | 8.4, 333 x 11008 10.4 | 11.8, 512 x 11008 10.8 | 10.2, 1000 x 11008
    // 14.3 | 11.4), and what their registers hold: up to 4096 elements behind a norm, 12288 otherwise.  Not rows of less than 1024, which leave lanes without any
    // (whole products of Q4_K: 8192 x 256 x 256 17.8 | 20.9, 8192 x 1024 x 512 28.0 | 31.1, 4096 x 2048 x 512 24.2 | 25.6; at k = 1024 within 3 % or faster).
    constexpr int kPlain = SRC == SKN_SRC_RMSNORM ? SKN_SRC_F32 : SRC;  // (the wider forms have no norm: not reached with one)
    if (k >= 1024 && m_pad % 32 == 0 && m_pad / 4 >= ctx->compute_units / (SRC == SKN_SRC_RMSNORM ? 1 : 2) && k <= (SRC == SKN_SRC_RMSNORM ? 4096 : 12288)) {
        const dim3 grid(m_pad / 4);
        if (k <= 2048) skn_launch(ctx, prep_a_quads_kernel<2, SRC, SUMS, 128>, grid, dim3(512), 0, src, afrag, isc, sfrag, m, k);
        else if (k <= 4096) skn_launch(ctx, prep_a_quads_kernel<4, SRC, SUMS, 128>, grid, dim3(512), 0, src, afrag, isc, sfrag, m, k);
        else if (k <= 8192) skn_launch(ctx, prep_a_quads_kernel<4, kPlain, SUMS, 256>, grid, dim3(1024), 0, src, afrag, isc, sfrag, m, k);
        else skn_launch(ctx, prep_a_quads_kernel<6, kPlain, SUMS, 256>, grid, dim3(1024), 0, src, afrag, isc, sfrag, m, k);
        return;
    }
    if (k <= 16384 && m_pad % 16 == 0) {
        const dim3 grid(m_pad / 2), block(512);
        const int nt = (k / 8 + 255) / 256;
        if (k <= 1024) skn_launch(ctx, prep_a_rows_kernel<1, SRC, SUMS, 128>, grid, dim3(256), 0, src, afrag, isc, sfrag, m, k);
        else if (nt <= 2) skn_launch(ctx, prep_a_rows_kernel<2, SRC, SUMS, 256>, grid, block, 0, src, afrag, isc, sfrag, m, k);
        else if (nt <= 4) skn_launch(ctx, prep_a_rows_kernel<4, SRC, SUMS, 256>, grid, block, 0, src, afrag, isc, sfrag, m, k);
        else if (nt <= 6) skn_launch(ctx, prep_a_rows_kernel<6, SRC, SUMS, 256>, grid, block, 0, src, afrag, isc, sfrag, m, k);
        else skn_launch(ctx, prep_a_rows_kernel<8, SRC, SUMS, 256>, grid, block, 0, src, afrag, isc, sfrag, m, k);
    } else {
        skn_launch(ctx, prep_a_frag_kernel<4, SRC, SUMS>, dim3(m_pad / 4), dim3(256), 0, src, afrag, isc, sfrag, m, k);
    }
}

// up to three weight matrices [n_i, k] multiplied by the same activations in one launch
struct Q4kFragSegs {
    const uint8_t* w[3];
    float* c[3];
    int n[3];
    int accumulate[3];  // add to c instead of overwriting it
    int tile0[3];       // first column tile of each matrix (unused entries: n_tiles)
    int n_tiles;
    // pair != 0: w[0], w[1] are the gate and up matrices of a SwiGLU; a tile holds the same 32 columns of both
    // (its two 32-column halves) and stores silu(gate) * up there, in bf16
    uint16_t* pair;
    // gemm_q4k_frag_kernel with k split over workgroups (gridDim.y of them per tile): the unscaled partial products go to
    // part[blockIdx.y][m][part_cols], matrix i at column part_col0[i] (a pair: gate, then up); null: no split
    float* part;
    int part_cols, part_col0[3];
    int part_blocks;  // superblocks of a workgroup (all of a row's: no split)
};

// the kernel's LDS (weight buffers, then the tile exchange) exceeds the static limit (the scales of the tile's rows follow it): dynamic, opted in per
// device by skn_gemm_init
// A buffer of weights: the 32 rows of each half of the tile's columns in nineteen pieces of 1 KiB (32 x 37 slots of sixteen bytes, the rest unused)
constexpr int kWHalf = 19, kWBuf = 2 * kWHalf * 1024;
template <int MT, int MH>
constexpr int frag_lds_bytes() {
    return 2 * kWBuf > MT * MH * 24576 ? 2 * kWBuf : MT * MH * 24576;
}

// Accumulators: acc holds the running sum of a column in units of cs = d * 2^14 of the latest superblock whose d
// is not zero.  Entering a superblock it is rescaled by cs_old / cs_new (a relative error of 2^-23 per
// superblock, against the 1e-3 asked of the op); the superblock's integer products then add to it as they come
// out of the matrix core, and so does the "- dmin * m_j" term: one more sixteen-deep product per tile between
// the activation sub-block sums (fp16 hi | lo) and -(dmin / cs) * m_j * 2^12, itself split into an fp16 pair.
template <int MT, int MH, bool SPLIT>
__global__ __launch_bounds__(256 * MH) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_q4k_frag_kernel(const u32x4* __restrict__ afrag, const u32x4* __restrict__ sfrag, const Q4kFragSegs segs,
                          const float* __restrict__ inv_scale, int m, int k, uint32_t a_bytes) {
    extern __shared__ __align__(16) uint8_t lds[];  // max(2 kWBuf, MT x 48 KiB) bytes
    const int tid = threadIdx.x, lane = tid & 63;
    // (the wavefront's index as a scalar: everything derived from it -- its row blocks, its superblocks, the
    // base addresses of its fragments -- then lives in scalar registers, and a fragment load is scalar base +
    // lane offset instead of a 64-bit vector add per load)
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kq = wave & 3, mh = wave >> 2;
    const int h = lane >> 5, r = lane & 31;
    const int nb = k >> 8, nch = k >> 6;
    // (this workgroup's superblocks: all of them, or a part of k)
    const int sb0 = SPLIT ? (int)blockIdx.y * segs.part_blocks : 0, sb1 = SPLIT ? min(sb0 + segs.part_blocks, nb) : nb;
    const int groups = (sb1 - sb0 + 3) >> 2;
    // tile -> (row tile, weight matrix, column tile): the column tiles of up to three matrices sharing the
    // activations are laid side by side
    const int mt = blockIdx.x / segs.n_tiles, tn = blockIdx.x - mt * segs.n_tiles;
    const bool pair = segs.pair != nullptr;
    const int seg = pair ? 0 : (tn >= segs.tile0[2] ? 2 : (tn >= segs.tile0[1] ? 1 : 0));
    const uint8_t* __restrict__ w = segs.w[seg];
    float* __restrict__ c = segs.c[seg];
    const int n = segs.n[seg];
    const int mb0 = (MH * mt + mh) * MT, n0 = pair ? tn * 32 : (tn - segs.tile0[seg]) * kBN;

    // Weight staging, memory straight into LDS: a wavefront-wide load fills 64 sixteen-byte slots of a half of the buffer; slot P holds piece
    // P % 37 of row P / 37 of that half (36 pieces = the 576 bytes of four superblocks, the 37th a pad that repeats the last).  The 38 loads of a
    // group are dealt round the wavefronts (whose last may be the 38th again: no branch, so that the compiler can count).  Completion is waited
    // for with the vector-memory counter before the barrier that publishes the buffer.
    // Buffer loads: one with a 64-bit address passes for a load that LDS may answer, and from it on the compiler waited for all loads that
    // were out, the next group's weights ahead of this group's first product (us: 120 x 4096 x 4096 17.9 ->
    // 16.2, in two parts of k 11008 25.3 -> 22.3, gate and up of 11008 41.3 -> 39.2, 2000 x 2048 and 8192 66.6 -> 62.0 in the mean).
    const uint8_t* w_hi = pair ? segs.w[1] + (size_t)n0 * nb * 144 : w + (size_t)min(n0 + 32, n - 1) * nb * 144;  // (pair: rows 32 .. are the up matrix)
    const int rows_lo = min(n - n0, 32), rows_hi = pair ? rows_lo : max(min(n - n0 - 32, 32), 1);
    const __amdgpu_buffer_rsrc_t res_lo = __builtin_amdgcn_make_buffer_rsrc((void*)(w + (size_t)n0 * nb * 144), 0, rows_lo * nb * 144, 0x00020000);
    const __amdgpu_buffer_rsrc_t res_hi = __builtin_amdgcn_make_buffer_rsrc((void*)w_hi, 0, rows_hi * nb * 144, 0x00020000);
    auto wfetch = [&](int g, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int x = 0; x < (2 * kWHalf + 4 * MH - 1) / (4 * MH); x++) {
            const int i = min(wave + 4 * MH * x, 2 * kWHalf - 1), hi = i >= kWHalf;
            const int p = (i - hi * kWHalf) * 64 + lane, row = p / kWPieces, col = min(p - kWPieces * row, 35);
            const int off = min(sb0 * 144 + g * 576 + col * 16, nb * 144 - 16);  // (a short last group repeats the row's last piece)
            skn_load_to_lds(hi ? res_hi : res_lo, lds + buf * kWBuf + i * 1024, min(row, (hi ? rows_hi : rows_lo) - 1) * nb * 144 + off, 0);
        }
    };

    // The activation fragments are read with buffer loads: a scalar byte offset (row block, k-step) plus the
    // lane's sixteen bytes, no vector address arithmetic per load.
    const __amdgpu_buffer_rsrc_t arsrc = __builtin_amdgcn_make_buffer_rsrc((void*)afrag, 0, (int)a_bytes, 0x00020000);
    uint32_t abase[MT];  // byte offset of the row block's first fragment
#pragma unroll
    for (int i = 0; i < MT; i++) abase[i] = (uint32_t)(mb0 + i) * (uint32_t)nch * 4096u;
    // activation fragments: a ring of eight k-steps; the slot of step t is refilled with step t + 8 as soon as
    // the matrix instructions of step t are issued
    u32x4 a[8][MT];
    auto afetch = [&](int step, int slot) __attribute__((always_inline)) {  // step: 16 per superblock, absolute
#pragma unroll
        for (int i = 0; i < MT; i++)
            a[slot][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(arsrc, lane * 16, (int)(abase[i] + (uint32_t)step * 1024u), 0));
    };
    float16_t acc[MT][2];
    float cs[2] = {1.f, 1.f};
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int x = 0; x < 16; x++) acc[i][j][x] = 0.f;

    // the scales of the tile's rows, for the store at the end
    float* isc_lds = reinterpret_cast<float*>(lds + frag_lds_bytes<MT, MH>());
    wfetch(0, 0);
    if (tid < 32 * MT * MH) isc_lds[tid] = inv_scale[MH * mt * MT * 32 + tid];
    if (sb0 + kq < sb1) {
        // (the first eight fragment steps are requested behind the weights and stay in flight past the barrier)
#pragma unroll
        for (int s = 0; s < 8; s++) afetch(16 * (sb0 + kq) + s, s);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 * MT) : "memory");
    } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

    auto group = [&](int g, auto more) __attribute__((always_inline)) {
        const int sb = sb0 + 4 * g + kq;
        if constexpr (decltype(more)::value) wfetch(g + 1, (g + 1) & 1);
        if (sb < sb1) {
            // this lane's weight rows (one per 32-column tile): the 144 bytes of superblock sb
            const uint8_t* wl = lds + (g & 1) * kWBuf + r * kWPitch + kq * 144;
            constexpr int kTile = kWHalf * 1024;  // the lane's row of the second 32-column tile
            u32x4 hd[2], sf[MT];
#pragma unroll
            for (int j = 0; j < 2; j++) hd[j] = *reinterpret_cast<const u32x4*>(wl + j * kTile);
            // The eight 6-bit scales and mins of the superblock, four to a word: bytes 0..3 of the twelve hold the
            // low scales, 4..7 the low mins, 8..11 the low nibbles of the high ones, whose top two bits sit in
            // bits 6..7 of the first eight bytes.
            uint32_t sc4[2][2], mn4[2][2];
            float min_unit[2], sc_unit[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const uint32_t dw0 = hd[j][0], s0 = hd[j][1], s1 = hd[j][2], s2 = hd[j][3];
                const half2_t dd = __builtin_bit_cast(half2_t, dw0);
                const float d = (float)dd.x, dmin = (float)dd.y;
                const bool live = d != 0.f;  // (a zero d: the products are zeroed)
                sc4[j][0] = live ? s0 & 0x3F3F3F3Fu : 0u;
                sc4[j][1] = live ? (s2 & 0x0F0F0F0Fu) | ((s0 >> 2) & 0x30303030u) : 0u;
                mn4[j][0] = s1 & 0x3F3F3F3Fu;
                mn4[j][1] = ((s2 >> 4) & 0x0F0F0F0Fu) | ((s1 >> 2) & 0x30303030u);
                // The unit is d * 2^(14 + p) and the weight operands are sc * q * 2^-(14 + p) -- exact in fp16 for
                // p <= 10.  p = 0 unless |dmin / d| is so large (>= 2^11) that the min operands below would
                // overflow fp16; beyond 2^21 they saturate.
                const int e_d = (int)((__float_as_uint(d) >> 23) & 0xFFu), e_m = (int)((__float_as_uint(dmin) >> 23) & 0xFFu);
                const int pw = live ? min(max(e_m - e_d - 10, 0), 10) : 0;
                sc_unit[j] = __uint_as_float((uint32_t)(127 + 10 - pw) << 23);
                // (no live weights: the unit is free, and taken from dmin so that the min operands are well inside
                // fp16 -- the unit inherited from the last live superblock can be orders of magnitude off)
                const float cs_new = live ? d * __uint_as_float((uint32_t)(127 + 14 + pw) << 23)
                                          : (dmin != 0.f ? fabsf(dmin) * 512.0f : cs[j]);
                const float inv = 1.0f / cs_new, ratio = cs[j] * inv;
                // -(dmin / unit) * 2^12: times a min (< 64) it stays inside fp16
                min_unit[j] = fminf(fmaxf(-dmin * inv * 4096.0f, -1023.f), 1023.f);
                cs[j] = cs_new;
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int x = 0; x < 16; x++) acc[i][j][x] *= ratio;
            }
            auto byte_f = [](uint32_t word, int b) { return (float)((word >> (8 * b)) & 0xFFu); };
            // Sixteen k-steps, software-pipelined: the weight fragments of step t + 1 are unpacked (vector ALU)
            // while the matrix instructions of step t run.
            u32x4 q[2], qn[2];
            half2_t mul_lo[2], mul_hi[2];
            half8_t fb[2], fbn[2];
            auto load_q = [&](int cc, u32x4* dst) __attribute__((always_inline)) {
#pragma unroll
                for (int j = 0; j < 2; j++) dst[j] = *reinterpret_cast<const u32x4*>(wl + j * kTile + 16 + 32 * cc + 16 * h);
            };
            auto scales = [&](int cc) __attribute__((always_inline)) {  // sub-blocks 2 cc (low nibbles), 2 cc + 1 (high)
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const float fl = byte_f(sc4[j][cc >> 1], 2 * (cc & 1)) * sc_unit[j];
                    const float fh = byte_f(sc4[j][cc >> 1], 2 * (cc & 1) + 1) * (sc_unit[j] * 0.0625f);
                    mul_lo[j] = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(fl, fl));  // (six bits times a power of two: exact)
                    mul_hi[j] = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(fh, fh));
                }
            };
            auto decode = [&](int s, half8_t* dst) __attribute__((always_inline)) {
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const uint32_t qq = q[j][s], q8 = qq >> 8;
                    const uint32_t l02 = qq & 0x000F000Fu, h02 = qq & 0x00F000F0u;
                    const uint32_t l13 = q8 & 0x000F000Fu, h13 = q8 & 0x00F000F0u;
                    u32x4 o;
                    o.x = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, l02) * mul_lo[j]);
                    o.y = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, h02) * mul_hi[j]);
                    o.z = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, l13) * mul_lo[j]);
                    o.w = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, h13) * mul_hi[j]);
                    dst[j] = __builtin_bit_cast(half8_t, o);
                }
            };
            load_q(0, q);
            scales(0);
            decode(0, fbn);
            auto chunk = [&](auto cc_const) __attribute__((always_inline)) {
                constexpr int cc = decltype(cc_const)::value;
                if (cc == 2) {
#pragma unroll
                    for (int i = 0; i < MT; i++) sf[i] = sfrag[((size_t)(mb0 + i) * nb + sb) * 64 + lane];
                }
                if (cc < 3) load_q(cc + 1, qn);
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    fb[0] = fbn[0], fb[1] = fbn[1];
                    if (s < 3) {
                        decode(s + 1, fbn);
                    } else if (cc < 3) {
                        q[0] = qn[0], q[1] = qn[1];
                        scales(cc + 1);
                        decode(0, fbn);
                    }
                    const int step = 4 * cc + s, slot = step & 7;
#pragma unroll
                    for (int i = 0; i < MT; i++) {
                        const half8_t fa = __builtin_bit_cast(half8_t, a[slot][i]);
#pragma unroll
                        for (int j = 0; j < 2; j++)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa, fb[j], acc[i][j], 0, 0, 0);
                    }
                    // refill the slot: eight steps ahead in this superblock, or the first half of superblock sb + 4
                    // (past the end: a repeat of the last superblock, unused)
                    // (the refill stays here: moved further down by the scheduler, the ring would be shallower than it looks)
                    __builtin_amdgcn_sched_barrier(0);
                    afetch(step < 8 ? 16 * sb + step + 8 : 16 * min(sb + 4, nb - 1) + step - 8, slot);
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            chunk(std::integral_constant<int, 0>{});
            chunk(std::integral_constant<int, 1>{});
            chunk(std::integral_constant<int, 2>{});
            chunk(std::integral_constant<int, 3>{});
            // the "- dmin * m" term of the superblock
#pragma unroll
            for (int j = 0; j < 2; j++) {
                half8_t vh, vl;
#pragma unroll
                for (int s = 0; s < 8; s++) {
                    _Float16 a, b;
                    skn_split_hilo(min_unit[j] * byte_f(mn4[j][s >> 2], s & 3), a, b);
                    vh[s] = a, vl[s] = b;
                }
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    const half8_t fs = __builtin_bit_cast(half8_t, sf[i]);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fs, vh, acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fs, vl, acc[i][j], 0, 0, 0);
                }
            }
        }
        // a bare barrier: a full __syncthreads() would also wait for the fragment loads in flight
        // The next group's weights were requested before this superblock's 16 MT fragment loads, and loads
        // complete in order: once all but the newest 8 MT have landed, so have they.
        if (sb < sb1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 * MT) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), in a form that the compiler counts with
        asm volatile("s_barrier" ::: "memory");
    };
    // (the last group apart: what is out behind its fragments is known where nothing is requested on condition)
    for (int g = 0; g + 1 < groups; g++) group(g, std::true_type{});
    if (groups > 0) group(groups - 1, std::false_type{});
    // back to true units
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int x = 0; x < 16; x++) acc[i][j][x] *= cs[j];

    // Add the four partial tiles of each half.  Tile t = 2 i + j belongs to wavefront kq = t % 4 of its half and
    // the other three hand theirs over.  Pair: the two column halves of row block i are needed together, so
    // wavefront i % 4 takes accumulator registers 0..7 of both and wavefront (i + 2) % 4 registers 8..15.
    float* red = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int t = 2 * i + j;
#pragma unroll
            for (int xh = 0; xh < 2; xh++) {
                const int owner = pair ? (i + 2 * xh) & 3 : t & 3;
                if (kq != owner) {
                    float* dst = red + ((mh * 2 * MT + t) * 3 + ((kq - owner + 4) & 3) - 1) * 1024 + lane;
#pragma unroll
                    for (int x = 8 * xh; x < 8 * xh + 8; x++) dst[64 * x] = acc[i][j][x];
                }
            }
        }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MT; i++) {
        if (pair) {
#pragma unroll
            for (int xh = 0; xh < 2; xh++)
                if (kq == ((i + 2 * xh) & 3)) {
                    const int col = n0 + (lane & 31);
#pragma unroll
                    for (int x = 8 * xh; x < 8 * xh + 8; x++) {
                        float g = acc[i][0][x], u = acc[i][1][x];
#pragma unroll
                        for (int o = 0; o < 3; o++) {
                            g += red[((mh * 2 * MT + 2 * i) * 3 + o) * 1024 + 64 * x + lane];
                            u += red[((mh * 2 * MT + 2 * i + 1) * 3 + o) * 1024 + 64 * x + lane];
                        }
                        // register x of lane l: row 8 (x / 4) + 4 (l / 32) + x % 4 of the 32 x 32 tile
                        const int row = (mb0 + i) * 32 + 8 * (x >> 2) + 4 * (lane >> 5) + (x & 3);
                        if (row < m && col < n) {
                            if constexpr (SPLIT) {
                                float* dst = segs.part + ((size_t)blockIdx.y * m + row) * segs.part_cols + col;
                                dst[0] = g, dst[segs.part_col0[1]] = u;
                                continue;
                            }
                            const float sc = isc_lds[row - MH * mt * MT * 32];
                            segs.pair[(size_t)row * n + col] = swiglu_bf16(g * sc, u * sc);
                        }
                    }
                }
            continue;
        }
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int t = 2 * i + j;
            if (kq == (t & 3)) {
                float16_t sum = acc[i][j];
#pragma unroll
                for (int o = 0; o < 3; o++)
#pragma unroll
                    for (int x = 0; x < 16; x++) sum[x] += red[((mh * 2 * MT + t) * 3 + o) * 1024 + 64 * x + lane];
                float sc[16];
#pragma unroll
                for (int x = 0; x < 16; x++) sc[x] = isc_lds[(mh * MT + i) * 32 + 8 * (x >> 2) + 4 * (lane >> 5) + (x & 3)];
                if constexpr (SPLIT)
                    store_tile_part(sum, segs.part + (size_t)blockIdx.y * m * segs.part_cols + segs.part_col0[seg], segs.part_cols, (mb0 + i) * 32,
                                    n0 + 32 * j, m, n, lane);
                else
                    store_tile(sum, c, n, (mb0 + i) * 32, n0 + 32 * j, m, n, sc, lane, segs.accumulate[seg] != 0);
            }
        }
    }
}


// ---- k split over workgroups ------------------------------------------------------------------------------------
// A product of few rows has few tiles (64 of them for 41 x 4096), each a serial walk along all of k by one workgroup.
// Where the tiles leave compute units idle, k is divided over `splits` workgroups per tile as well; each leaves its
// unscaled partial products in the workspace and this kernel adds them in a fixed order, applies the row scale and does
// what the store would have done (add into c, or silu(gate) * up of a pair).
template <int W>  // columns per thread: 4, or 1 where a matrix has a number of columns that is no multiple of 4
__global__ __launch_bounds__(256) void gemm_add_parts_kernel(const float* __restrict__ part, int splits, int cols, const skn_gemm_parts segs,
                                                            const float* __restrict__ inv_scale, int m) {
    const int row = blockIdx.y, col = (blockIdx.x * 256 + threadIdx.x) * W;
    if (col >= (segs.pair ? segs.n[0] : cols)) return;
    typedef float vec __attribute__((ext_vector_type(W)));
    const float* src = part + (size_t)row * cols + col;
    const size_t stride = (size_t)m * cols;
    auto total = [&](const float* p) __attribute__((always_inline)) {
        vec sum = *reinterpret_cast<const vec*>(p);
        int z = 1;
        for (; z + 4 <= splits; z += 4) {  // four parts requested together, added one after the other
            vec v[4];
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = *reinterpret_cast<const vec*>(p + (z + i) * stride);
#pragma unroll
            for (int i = 0; i < 4; i++) sum += v[i];
        }
        for (; z < splits; z++) sum += *reinterpret_cast<const vec*>(p + z * stride);
        return sum;
    };
    const float sc = inv_scale[row];
    vec v = total(src) * sc;
    if (segs.pair) {
        const vec u = total(src + segs.col0[1]) * sc;
        typedef uint16_t bits_vec __attribute__((ext_vector_type(W)));
        bits_vec bits;
#pragma unroll
        for (int i = 0; i < W; i++) bits[i] = swiglu_bf16(v[i], u[i]);
        *reinterpret_cast<bits_vec*>(segs.pair + (size_t)row * segs.n[0] + col) = bits;
        return;
    }
    const int i = segs.count > 2 && col >= segs.col0[2] ? 2 : (segs.count > 1 && col >= segs.col0[1] ? 1 : 0);
    vec* dst = reinterpret_cast<vec*>(segs.c[i] + (size_t)row * segs.n[i] + (col - segs.col0[i]));
    *dst = segs.accumulate[i] ? *dst + v : v;
}

template <int MT, int MH>
int launch_frag(skn_ctx* ctx, int m_tiles, const u32x4* afrag, const u32x4* sfrag, const Q4kFragSegs& segs, const float* isc,
                int m, int k, int splits) {
    constexpr int kLds = frag_lds_bytes<MT, MH>() + 32 * MT * MH * 4;
    const uint32_t a_bytes = (uint32_t)((size_t)m_tiles * 32 * MT * MH * k * 2);  // (checked by the caller to fit)
    skn_launch(ctx, splits > 1 ? gemm_q4k_frag_kernel<MT, MH, true> : gemm_q4k_frag_kernel<MT, MH, false>, dim3(m_tiles * segs.n_tiles, splits), dim3(256 * MH), kLds, afrag, sfrag, segs, isc, m, k, a_bytes);
    SKN_LAUNCH_CHECK(ctx);
    return SKN_OK;
}

// ---- Q4_K path for wide weight matrices: a 256 x 128 tile, weights unpacked once for all its rows -------------
// The arithmetic of gemm_q4k_frag_kernel with its two costs divided differently.  A workgroup of eight wavefronts
// holds a 256 x 128 tile and walks k superblock by superblock.  Four consumers, one per SIMD, own 64 rows each --
// a 64 x 128 tile per wavefront: an activation fragment feeds four matrix instructions instead of two, so the
// activations a compute unit takes in per matrix instruction halve -- and four producers, their SIMD neighbours, own
// 32 columns each: a producer unpacks the fragments of its columns once for all 256 rows (a quarter of the vector
// instructions per matrix instruction of the other kernel) into LDS, two phases (a phase: a chunk of 64 elements,
// four k-steps) ahead of the consumers, three buffers, one bare barrier per phase; entering a superblock it leaves
// the min operands and the ratio by which the accumulators change their unit beside them.  The consumers load their
// activation fragments themselves (ring of eight k-steps), read the weight fragments one k-step ahead -- across the
// barrier too: what the next phase starts with was complete a phase ago -- and issue the matrix instructions; the
// change of unit between two superblocks is spread between the matrix instructions around it.  No split of k, so no
// exchange at the end.  (Timed in the kernel, the loop of one workgroup alone on the device takes as many core clocks
// as with all 224 -- nothing shared between compute units holds it -- but the core clock falls from 2.39 GHz to
// 1.8 - 1.9 GHz with all compute units at this work.)
constexpr int kTlStage = 4 * 4 * 1024;           // a phase: four k-steps x four column blocks x 1 KiB
constexpr int kTlAux = 128 * 32 + 128 * 4;       // a superblock's min operands (128 columns x (hi, lo) x 16 B) and ratios
// The last `tiles` tiles of a launch, from tile0 on, with their k divided over `splits` workgroups: part[split][tile][consumer]
// [row block][column block][register group][lane] x 4.
struct TallTail {
    int tile0, tiles, splits;
    float* part;
};
constexpr int kTlLds = 3 * kTlStage + 2 * kTlAux + 128 * 4 + 256 * 4;

// One to three matrices per launch as in gemm_q4k_frag_kernel (tile0 counts 128-column tiles here); pair: a tile holds
// the same 64 columns of the gate and the up matrix -- producers 0 and 1 unpack the gate's, 2 and 3 the up's, so a
// consumer's column blocks 0, 1 and 2, 3 meet lane by lane in the store -- and stores silu(gate) * up in bf16.
// TAIL: the last tiles are shared by tail.splits workgroups each, neighbours in the grid, with a part of k each (a template
// parameter: grids without such tiles were 0.5 us slower at 512 x 14336 x 4096 for the division).
// CB: column blocks of 32 in a tile.  Three (256 x 96) where their rounds of compute units cost less than those of four (a loop of 96 columns takes
// 0.83 of the time of one of 128, bound by the same phases: q, k and v of 512 x 4096 in 12288 columns 73.2 -> 60.8
// us, 704 -> 848 TFLOP/s; 2000 x 2048 in 3072 41.3 -> 35.9); tile0 and n_tiles count blocks of 32 there, so that a tile may hold the end of one matrix and the start of the next, and the
// fourth producer only keeps the barriers.
template <bool TAIL, int CB>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_q4k_tall_kernel(const u32x4* __restrict__ afrag, const u32x4* __restrict__ sfrag, const Q4kFragSegs segs,
                          const float* __restrict__ inv_scale, int m, int k, int m_tiles, uint32_t a_bytes, const TallTail tail) {
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const int me = wave & 3;  // consumer: its 64 rows; producer: its 32 columns
    const bool producer = wave >= 4;
    const int h = lane >> 5, r = lane & 31;
    const int nb = k >> 8, nch = k >> 6;
    int tile = (int)blockIdx.x, z = 0, parts = 1, sb0 = 0, sb1 = nb;
    if (TAIL && tile >= tail.tile0) {
        const int over = tile - tail.tile0;
        parts = tail.splits, z = over % parts, tile = tail.tile0 + over / parts;
        sb0 = nb * z / parts, sb1 = nb * (z + 1) / parts;
    }
    const int mt = tile % m_tiles, tn = tile / m_tiles;  // (the row tiles of a column tile run side by side)
    static_assert(CB == 4 || (CB == 3 && !TAIL), "tiles of 128 columns, or of 96 with k undivided");
    const bool pair = CB == 4 && segs.pair != nullptr;
    auto matrix_of = [&](int unit) __attribute__((always_inline)) { return unit >= segs.tile0[2] ? 2 : (unit >= segs.tile0[1] ? 1 : 0); };
    // (CB 3: of this producer's block of columns; a consumer looks its three up when it stores)
    const int unit = CB == 4 ? tn : tn * CB + min(me, CB - 1);
    const int seg = pair ? 0 : matrix_of(unit);
    const int n = segs.n[seg];
    const int n0 = pair ? tn * 64 : CB == 4 ? (tn - segs.tile0[seg]) * 128 : (unit - segs.tile0[seg]) * 32;  // first column of the tile in its matrix (pair: in both)
    float* __restrict__ c = segs.c[seg];
    uint8_t* stage = lds;
    uint8_t* aux = lds + 3 * kTlStage;
    uint8_t* fin = aux + 2 * kTlAux;
    float* isc_lds = reinterpret_cast<float*>(fin + 128 * 4);  // the scales of the tile's 256 rows, for the store at the end
    if (tid < 256) isc_lds[tid] = inv_scale[mt * 256 + tid];
    auto barrier = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    using C0 = std::integral_constant<int, 0>;
    using C1 = std::integral_constant<int, 1>;
    using C2 = std::integral_constant<int, 2>;
    using C3 = std::integral_constant<int, 3>;
    // the three buffers in turn: phase p is multiplied from b_cur, phase p + 1 lies complete in b_nxt, phase p + 2 is
    // being written to b_nx2 (byte offsets, uniform)
    int b_cur = 0, b_nxt = kTlStage, b_nx2 = 2 * kTlStage;
    auto turn = [&]() __attribute__((always_inline)) {
        const int t = b_cur;
        b_cur = b_nxt, b_nxt = b_nx2, b_nx2 = t;
    };

    if (CB < 4 && producer && me >= CB) {
        for (int i = 2 + 4 * (sb1 - sb0); i > 0; i--) barrier();
    } else if (producer) {
        const uint8_t* w = segs.w[pair ? me >> 1 : seg];
        const __amdgpu_buffer_rsrc_t wrsrc = __builtin_amdgcn_make_buffer_rsrc((void*)w, 0, n * nb * 144, 0x00020000);  // (checked by the caller to fit)
        const int col = 32 * me + r;  // column of the tile
        const int wrow = min(n0 + (pair ? 32 * (me & 1) + r : CB == 4 ? col : r), n - 1) * nb * 144;
        // One set of registers for the header and the four nibble pieces; each is requested again, for the next
        // superblock, right after it is unpacked: four phases before its next use.
        u32x4 hd, q[4];
        auto load_piece = [&](int sb, int cc) __attribute__((always_inline)) {
            sb = min(sb, nb - 1);  // (past the end: a repeat, unused)
            q[cc] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, wrow + 16 * h, sb * 144 + 16 + 32 * cc, 0));
        };
        auto load_header = [&](int sb) __attribute__((always_inline)) {
            sb = min(sb, nb - 1);
            hd = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, wrow, sb * 144, 0));
        };
        uint32_t sc4[2], mn4[2];
        float sc_unit = 1.f, cs = 1.f;
        auto byte_f = [](uint32_t word, int b) { return (float)((word >> (8 * b)) & 0xFFu); };
        // header of the superblock in hd -> scales, mins, units; its ratio and min operands into aux[sb & 1]
        auto enter = [&](int sb) __attribute__((always_inline)) {
            uint8_t* ax = aux + (sb & 1) * kTlAux;
            // (the header is taken up here and no earlier: without this the compiler computes on it, and waits for
            // it, phases before)
            asm volatile("" : "+v"(hd));
            const uint32_t dw0 = hd[0], s0 = hd[1], s1 = hd[2], s2 = hd[3];
            const half2_t dd = __builtin_bit_cast(half2_t, dw0);
            const float d = (float)dd.x, dmin = (float)dd.y;
            const bool live = d != 0.f;  // (a zero d: the products are zeroed)
            sc4[0] = live ? s0 & 0x3F3F3F3Fu : 0u;
            sc4[1] = live ? (s2 & 0x0F0F0F0Fu) | ((s0 >> 2) & 0x30303030u) : 0u;
            mn4[0] = s1 & 0x3F3F3F3Fu;
            mn4[1] = ((s2 >> 4) & 0x0F0F0F0Fu) | ((s1 >> 2) & 0x30303030u);
            // (units, power pw and saturation as in gemm_q4k_frag_kernel)
            const int e_d = (int)((__float_as_uint(d) >> 23) & 0xFFu), e_m = (int)((__float_as_uint(dmin) >> 23) & 0xFFu);
            const int pw = live ? min(max(e_m - e_d - 10, 0), 10) : 0;
            sc_unit = __uint_as_float((uint32_t)(127 + 10 - pw) << 23);
            const float cs_new = live ? d * __uint_as_float((uint32_t)(127 + 14 + pw) << 23)
                                      : (dmin != 0.f ? fabsf(dmin) * 512.0f : cs);
            const float inv = 1.0f / cs_new, ratio = cs * inv;
            const float min_unit = fminf(fmaxf(-dmin * inv * 4096.0f, -1023.f), 1023.f);
            cs = cs_new;
            if (h == 0) {
                half8_t vh, vl;
#pragma unroll
                for (int x = 0; x < 8; x++) {
                    _Float16 a, b;
                    skn_split_hilo(min_unit * byte_f(mn4[x >> 2], x & 3), a, b);
                    vh[x] = a, vl[x] = b;
                }
                *reinterpret_cast<half8_t*>(ax + col * 32) = vh;
                *reinterpret_cast<half8_t*>(ax + col * 32 + 16) = vl;
                *reinterpret_cast<float*>(ax + 128 * 32 + col * 4) = ratio;
            }
        };
        // chunk cc of the superblock in q -> four k-steps of this producer's column block into the buffer at `buf`
        auto unpack = [&](auto cc_const, int buf) __attribute__((always_inline)) {
            constexpr int cc = decltype(cc_const)::value;
            uint8_t* dst = stage + buf + me * 1024 + lane * 16;
            asm volatile("" : "+v"(q[cc]));  // (as for the header)
            const float fl = byte_f(sc4[cc >> 1], 2 * (cc & 1)) * sc_unit;
            const float fh = byte_f(sc4[cc >> 1], 2 * (cc & 1) + 1) * (sc_unit * 0.0625f);
            const half2_t mul_lo = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(fl, fl));  // (six bits times a power of two: exact)
            const half2_t mul_hi = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(fh, fh));
#pragma unroll
            for (int s4 = 0; s4 < 4; s4++) {
                const uint32_t qq = q[cc][s4], q8 = qq >> 8;
                const uint32_t l02 = qq & 0x000F000Fu, h02 = qq & 0x00F000F0u;
                const uint32_t l13 = q8 & 0x000F000Fu, h13 = q8 & 0x00F000F0u;
                u32x4 o;
                o.x = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, l02) * mul_lo);
                o.y = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, h02) * mul_hi);
                o.z = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, l13) * mul_lo);
                o.w = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, h13) * mul_hi);
                *reinterpret_cast<u32x4*>(dst + s4 * 4096) = o;
            }
        };
        // While the consumers multiply phase (sb, cc) the producer unpacks the phase two after it -- chunks 2 and 3 of
        // the superblock, then chunks 0 and 1 of the next, whose header it takes up with chunk 0 -- and requests the
        // same piece of the superblock after that.  (After the last superblock it unpacks a repeat into buffers that
        // nobody reads any more -- no branch, so that the requests are not moved down into one -- and keeps the unit.)
        auto phase = [&](int sb, auto cc_const) __attribute__((always_inline)) {
            constexpr int cc = decltype(cc_const)::value;
            if (cc == 0) {
                unpack(C2{}, b_nx2);
                load_piece(sb + 1, 2);
            }
            if (cc == 1) {
                unpack(C3{}, b_nx2);
                load_piece(sb + 1, 3);
            }
            if (cc == 2) {
                const float keep = cs;
                enter(sb + 1);
                if (sb + 1 >= sb1) cs = keep;
                unpack(C0{}, b_nx2);
                load_header(sb + 2);
                load_piece(sb + 2, 0);
            }
            if (cc == 3) {
                unpack(C1{}, b_nx2);
                load_piece(sb + 2, 1);
            }
            barrier();
            turn();
        };
        load_header(sb0);
#pragma unroll
        for (int x = 0; x < 4; x++) load_piece(sb0, x);
        enter(sb0);
        unpack(C0{}, b_cur);
        unpack(C1{}, b_nxt);
        load_header(sb0 + 1);
        load_piece(sb0 + 1, 0);
        load_piece(sb0 + 1, 1);
        barrier();
        for (int sb = sb0; sb < sb1; sb++) {
            phase(sb, C0{});
            phase(sb, C1{});
            phase(sb, C2{});
            phase(sb, C3{});
        }
        // the unit the accumulators ended in
        if (h == 0) *reinterpret_cast<float*>(fin + col * 4) = cs;
        barrier();
    } else {
        constexpr int MT = 2, NT = MT * CB;  // (tile t: row block t / CB, column block t % CB)
        const __amdgpu_buffer_rsrc_t arsrc = __builtin_amdgcn_make_buffer_rsrc((void*)afrag, 0, (int)a_bytes, 0x00020000);
        const int mb0 = mt * 8 + me * MT;  // first row block of this consumer
        uint32_t abase[MT];
#pragma unroll
        for (int i = 0; i < MT; i++) abase[i] = (uint32_t)(mb0 + i) * (uint32_t)nch * 4096u;
        u32x4 a[8][MT];  // ring of eight k-steps, seven ahead
        auto afetch = [&](int step, int slot) __attribute__((always_inline)) {  // step: absolute, 16 per superblock
            step = min(step, 16 * nb - 1);  // (past the end: the last step again, unused)
#pragma unroll
            for (int i = 0; i < MT; i++)
                a[slot][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(arsrc, lane * 16, (int)(abase[i] + (uint32_t)step * 1024u), 0));
        };
        float16_t acc[MT][CB];
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < CB; j++)
#pragma unroll
                for (int x = 0; x < 16; x++) acc[i][j][x] = 0.f;
        u32x4 sf[MT];
        half8_t fb[2][CB];  // the weight fragments of a k-step, read while the step before it is multiplied; step 0 of a phase in fb[0]
        float ratio[CB];  // of the superblock being entered, by column block
#pragma unroll
        for (int j = 0; j < CB; j++) ratio[j] = 1.f;
        // tile t changes its unit: half `part` of its sixteen registers
        auto rescale = [&](int t, int part) __attribute__((always_inline)) {
#pragma unroll
            for (int x = 0; x < 8; x++) acc[t / CB][t % CB][8 * part + x] *= ratio[t % CB];
        };
        auto fence = [&]() __attribute__((always_inline)) { __builtin_amdgcn_sched_barrier(0); };
        auto phase = [&](int sb, auto cc_const) __attribute__((always_inline)) {
            constexpr int cc = decltype(cc_const)::value;
            const uint8_t* ax = aux + (sb & 1) * kTlAux;
            const uint8_t* axn = aux + ((sb + 1) & 1) * kTlAux;
            if (cc == 0) {  // (the sub-block sums of the rows: needed three phases on)
#pragma unroll
                for (int i = 0; i < MT; i++) sf[i] = sfrag[((size_t)(mb0 + i) * nb + sb) * 64 + lane];
            }
            const uint8_t* src = stage + b_cur + lane * 16;
            const uint8_t* srcn = stage + b_nxt + lane * 16;
            half8_t vh[CB], vl[CB];
            float rnext[CB];
            if (cc == 3) {  // (the ratios of the next superblock, left by the producers a phase ago: used at the end of this phase)
#pragma unroll
                for (int j = 0; j < CB; j++) rnext[j] = *reinterpret_cast<const float*>(axn + 128 * 32 + (j * 32 + r) * 4);
            }
#pragma unroll
            for (int s4 = 0; s4 < 4; s4++) {
                const int step = 4 * cc + s4, slot = step & 7;
                if (s4 < 3) {
#pragma unroll
                    for (int j = 0; j < CB; j++) fb[(s4 + 1) & 1][j] = *reinterpret_cast<const half8_t*>(src + (s4 + 1) * 4096 + j * 1024);
                } else if (cc < 3) {  // the next phase's first step: complete since the barrier before this phase
#pragma unroll
                    for (int j = 0; j < CB; j++) fb[0][j] = *reinterpret_cast<const half8_t*>(srcn + j * 1024);
                } else {
#pragma unroll
                    for (int j = 0; j < CB; j++) vh[j] = *reinterpret_cast<const half8_t*>(ax + (j * 32 + r) * 32);
                }
                fence();
                if (cc == 0 && s4 == 0) {
                    // the superblock's first step: the tiles from 3 on change their unit between its matrix instructions
                    // (tiles 0 .. 2 did before the barrier)
#pragma unroll
                    for (int t = 0; t < NT; t++) {
                        acc[t / CB][t % CB] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a[slot][t / CB]), fb[0][t % CB],
                                                                                    acc[t / CB][t % CB], 0, 0, 0);
                        fence();
                        if (t < 4) rescale(3 + (t >> 1), t & 1);
                        if (t >= 4 && t < NT - 1) rescale(t + 1, 0), rescale(t + 1, 1);
                        fence();
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < MT; i++) {
                        const half8_t fa = __builtin_bit_cast(half8_t, a[slot][i]);
#pragma unroll
                        for (int j = 0; j < CB; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa, fb[s4 & 1][j], acc[i][j], 0, 0, 0);
                    }
                }
                afetch(16 * sb + step + 7, (step + 7) & 7);
                fence();
            }
            if (cc == 3) {
                // The "- dmin * m" term of the superblock (the two products of a tile eight instructions apart), and
                // under it the reads for what follows: the low parts, then the next phase's first step.
#pragma unroll
                for (int j = 0; j < CB; j++) vl[j] = *reinterpret_cast<const half8_t*>(ax + (j * 32 + r) * 32 + 16);
                fence();
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int j = 0; j < CB; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, sf[i]), vh[j], acc[i][j], 0, 0, 0);
                fence();
#pragma unroll
                for (int j = 0; j < CB; j++) fb[0][j] = *reinterpret_cast<const half8_t*>(srcn + j * 1024);
#pragma unroll
                for (int j = 0; j < CB; j++) ratio[j] = sb + 1 < sb1 ? rnext[j] : 1.0f;  // (none after the last superblock)
                fence();
                // tiles 0 .. 2 change their unit between the last of these instructions
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    acc[t / CB][t % CB] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, sf[t / CB]), vl[t % CB], acc[t / CB][t % CB], 0, 0, 0);
                    fence();
                    if (CB == 4 && t >= 2) rescale((t - 2) >> 1, t & 1);
                    if (CB == 3 && t >= 3) rescale(t - 3, 0), rescale(t - 3, 1);
                    fence();
                }
            }
            barrier();
            turn();
        };
#pragma unroll
        for (int s = 0; s < 7; s++) afetch(16 * sb0 + s, s);
        barrier();
#pragma unroll
        for (int j = 0; j < CB; j++) fb[0][j] = *reinterpret_cast<const half8_t*>(stage + b_cur + lane * 16 + j * 1024);
        for (int sb = sb0; sb < sb1; sb++) {
            phase(sb, C0{});
            phase(sb, C1{});
            phase(sb, C2{});
            phase(sb, C3{});
        }
        barrier();
        if constexpr (TAIL) if (parts > 1) {  // (unscaled, every element of the tile, in the order of the matrix core's registers: see gemm_add_tall_kernel)
            float* dst = tail.part + ((size_t)(z * tail.tiles + tile - tail.tile0) * 4 + me) * (MT * 4 * 1024) + lane * 4;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float unit = *reinterpret_cast<const float*>(fin + (j * 32 + r) * 4);
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int x = 0; x < 4; x++)
                        *reinterpret_cast<float4*>(dst + ((i * 4 + j) * 4 + x) * 256) =
                            make_float4(acc[i][j][4 * x] * unit, acc[i][j][4 * x + 1] * unit, acc[i][j][4 * x + 2] * unit, acc[i][j][4 * x + 3] * unit);
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < MT; i++) {
            float sc[16];
#pragma unroll
            for (int x = 0; x < 16; x++) sc[x] = isc_lds[(me * MT + i) * 32 + 8 * (x >> 2) + 4 * h + (x & 3)];
            if constexpr (CB == 4) if (pair) {
#pragma unroll
                for (int jj = 0; jj < 2; jj++) {
                    const float ug = *reinterpret_cast<const float*>(fin + (jj * 32 + r) * 4);
                    const float uu = *reinterpret_cast<const float*>(fin + ((jj + 2) * 32 + r) * 4);
                    const int col = n0 + 32 * jj + r;
#pragma unroll
                    for (int x = 0; x < 16; x++) {
                        // register x of lane l: row 8 (x / 4) + 4 (l / 32) + x % 4 of the 32 x 32 tile
                        const int row = (mb0 + i) * 32 + 8 * (x >> 2) + 4 * h + (x & 3);
                        if (row < m && col < n) {
                            segs.pair[(size_t)row * n + col] = swiglu_bf16(acc[i][jj][x] * ug * sc[x], acc[i][jj + 2][x] * uu * sc[x]);
                        }
                    }
                }
                continue;
            }
#pragma unroll
            for (int j = 0; j < CB; j++) {
                const float unit = *reinterpret_cast<const float*>(fin + (j * 32 + r) * 4);
#pragma unroll
                for (int x = 0; x < 16; x++) acc[i][j][x] *= unit;
                if constexpr (CB == 4) {
                    store_tile(acc[i][j], c, n, (mb0 + i) * 32, n0 + 32 * j, m, n, sc, lane, segs.accumulate[seg] != 0);
                } else {
                    const int at = tn * CB + j, s = matrix_of(at);
                    if (at < segs.n_tiles)
                        store_tile(acc[i][j], segs.c[s], segs.n[s], (mb0 + i) * 32, (at - segs.tile0[s]) * 32, m, segs.n[s], sc, lane, segs.accumulate[s] != 0);
                }
            }
        }
    }
}

// The tiles that workgroups shared: grid (tiles, 8), a wavefront per row block and column block of 32 (wavefront w of block y: row
// block y of the tile, column block w; a pair: wavefronts 0 and 1, both halves).  Lane l of register group x holds rows
// 8 x + 4 (l / 32) .. + 3 of column l % 32, as the matrix core does.
__global__ __launch_bounds__(256) void gemm_add_tall_kernel(const TallTail tail, const Q4kFragSegs segs, const float* __restrict__ inv_scale, int m, int m_tiles) {
    const int tile = tail.tile0 + (int)blockIdx.x, mt = tile % m_tiles, tn = tile / m_tiles, lane = threadIdx.x & 63, j = threadIdx.x >> 6;
    const int i = blockIdx.y, row0 = mt * 256 + 32 * i;  // (consumer i / 2, its row block i % 2)
    const bool pair = segs.pair != nullptr;
    if (row0 >= m || (pair && j > 1)) return;
    const int seg = pair ? 0 : (tn >= segs.tile0[2] ? 2 : (tn >= segs.tile0[1] ? 1 : 0));
    const int n = segs.n[seg], col = (pair ? tn * 64 : (tn - segs.tile0[seg]) * 128) + 32 * j + (lane & 31);
    float* __restrict__ c = segs.c[seg];
    auto total = [&](int jj, float (&v)[16]) __attribute__((always_inline)) {
        const float4* src = reinterpret_cast<const float4*>(tail.part) + (((size_t)blockIdx.x * 4 + (i >> 1)) * 8 + (i & 1) * 4 + jj) * 256 + lane;
        const size_t stride = (size_t)tail.tiles * 8192;
#pragma unroll
        for (int x = 0; x < 16; x++) v[x] = 0.f;
        for (int z = 0; z < tail.splits; z++)
#pragma unroll
            for (int x = 0; x < 4; x++) {
                const float4 p = src[z * stride + 64 * x];
                v[4 * x] += p.x, v[4 * x + 1] += p.y, v[4 * x + 2] += p.z, v[4 * x + 3] += p.w;
            }
    };
    float v[16], u[16], sc[16];
    row_scales(inv_scale, row0, lane, sc);
    total(j, v);
    if (pair) total(j + 2, u);
    if (pair) {
        if (col >= n) return;
#pragma unroll
        for (int x = 0; x < 16; x++) {
            const int row = row0 + 8 * (x >> 2) + 4 * (lane >> 5) + (x & 3);
            if (row < m) segs.pair[(size_t)row * n + col] = swiglu_bf16(v[x] * sc[x], u[x] * sc[x]);
        }
        return;
    }
    float16_t sum;
#pragma unroll
    for (int x = 0; x < 16; x++) sum[x] = v[x];
    store_tile(sum, c, n, row0, col - (lane & 31), m, n, sc, lane, segs.accumulate[seg] != 0);
}

// ---- general path: activations x (hi + lo * 2^-11) weights, both operands loaded in fragment order ---------
// Workgroup of four wavefronts, one per SIMD, tile (32 MT) x 64.  The tile is not divided spatially: wavefront
// kq computes all of it over a quarter of k (k is a multiple of 64, so the k-steps divide evenly) and the four
// partial tiles are added through LDS at the end, so no operand is loaded twice inside a workgroup.  Per k-step
// a wavefront loads MT activation fragments and four weight fragments (two column tiles, hi and lo) -- coalesced
// 1 KiB loads straight into the registers the matrix instructions read, D steps ahead -- and issues 4 MT matrix
// instructions.  Consecutive workgroups on an XCD (blockIdx / 8) are the row tiles of one column tile, so a
// weight fragment comes from memory once and from that XCD's L2 for the other row tiles.
template <int MT, int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void gemm_hilo_frag_kernel(const u32x4* __restrict__ afrag, const u32x4* __restrict__ bfrag,
                           const float* __restrict__ inv_scale, float* __restrict__ c, int m, int n, int steps,
                           int m_tiles, int n_tiles, int accumulate) {
    extern __shared__ __align__(16) float red[];  // 2 MT tiles x 3 copies x 1024 floats
    const int lane = threadIdx.x & 63, kq = threadIdx.x >> 6;
    const int slot_in_xcd = blockIdx.x >> 3;
    const int mt = slot_in_xcd % m_tiles, tn = (slot_in_xcd / m_tiles) * 8 + (blockIdx.x & 7);
    if (tn >= n_tiles) return;
    const int U = steps >> 2, t0 = kq * U;  // this wavefront's k-steps [t0, t0 + U)
    const u32x4* ap = afrag + ((size_t)mt * MT * steps + t0) * 64 + lane;   // + i * steps * 64 per row block
    const u32x4* bp = bfrag + ((size_t)tn * 2 * steps + t0) * 128 + lane;   // + j * steps * 128 per column block

    u32x4 ra[D][MT], rb[D][2][2];
    auto fetch = [&](int u, int slot) __attribute__((always_inline)) {
        u = min(u, U - 1);
#pragma unroll
        for (int i = 0; i < MT; i++) ra[slot][i] = ap[((size_t)i * steps + u) * 64];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            rb[slot][j][0] = bp[((size_t)j * steps + u) * 128];
            rb[slot][j][1] = bp[((size_t)j * steps + u) * 128 + 64];
        }
    };
    float16_t acc[MT][2], accl[MT][2];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int x = 0; x < 16; x++) acc[i][j][x] = accl[i][j][x] = 0.f;
    auto mac = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MT; i++) {
            const half8_t fa = __builtin_bit_cast(half8_t, ra[slot][i]);
#pragma unroll
            for (int j = 0; j < 2; j++) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa, __builtin_bit_cast(half8_t, rb[slot][j][0]), acc[i][j], 0, 0, 0);
                accl[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa, __builtin_bit_cast(half8_t, rb[slot][j][1]), accl[i][j], 0, 0, 0);
            }
        }
    };

    // Ring of D slots, D - 1 steps ahead: while the matrix instructions of step u run, the slot of step u - 1 --
    // whose registers are all free by then -- is refilled, one load after every second matrix instruction.
    // (Measured: the depth does not matter from 3 to 6 -- the loop is bound by operand delivery, 2 MiB per
    // compute unit and tile, not by its latency.)
#pragma unroll
    for (int x = 0; x < D - 1; x++) fetch(x, x);
    int u0 = 0;
    for (; u0 + D <= U; u0 += D) {
#pragma unroll
        for (int x = 0; x < D; x++) {
            fetch(u0 + x + D - 1, (x + D - 1) % D);  // (past the end: a repeat of the last step, unused)
            mac(x);
#pragma unroll
            for (int g = 0; g < MT + 4; g++) {
                __builtin_amdgcn_sched_group_barrier(0x008, (4 * MT) / (MT + 4), 0);  // matrix instructions
                __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);                    // one load
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // the last U % D steps are already in slots 0 ..
#pragma unroll
    for (int x = 0; x < D - 1; x++)
        if (u0 + x < U) mac(x);

    // hi + lo * 2^-11, then the four partial tiles: tile t = 2 i + j belongs to wavefront t % 4, the other three
    // hand theirs over
    float sc[(MT + 1) / 2][16];
#pragma unroll
    for (int y = 0; y < (MT + 1) / 2; y++) row_scales(inv_scale, (mt * MT + min((kq >> 1) + 2 * y, MT - 1)) * 32, lane, sc[y]);
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
#pragma unroll
            for (int x = 0; x < 16; x++) acc[i][j][x] += accl[i][j][x] * 0x1p-11f;
            const int t = 2 * i + j, owner = t & 3;
            if (kq != owner) {
                float* dst = red + (t * 3 + ((kq - owner + 4) & 3) - 1) * 1024 + lane;
#pragma unroll
                for (int x = 0; x < 16; x++) dst[64 * x] = acc[i][j][x];
            }
        }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int t = 2 * i + j;
            if (kq == (t & 3)) {
                float16_t sum = acc[i][j];
#pragma unroll
                for (int o = 0; o < 3; o++)
#pragma unroll
                    for (int x = 0; x < 16; x++) sum[x] += red[(t * 3 + o) * 1024 + 64 * x + lane];
                store_tile(sum, c, n, (mt * MT + i) * 32, tn * kBN + 32 * j, m, n, sc[i >> 1], lane, accumulate != 0);
            }
        }
}

template <int MT, int D>
int launch_hilo_gemm(skn_ctx* ctx, const u32x4* afrag, const u32x4* bfrag, const float* isc, float* c, int m, int n, int k,
                     int accumulate = 0) {
    constexpr int kLds = 2 * MT * 3 * 4096;
    const int m_tiles = (m + 32 * MT - 1) / (32 * MT), n_tiles = (n + kBN - 1) / kBN;
    const unsigned grid = (unsigned)(((n_tiles + 7) / 8) * 8 * m_tiles);
    skn_launch(ctx, gemm_hilo_frag_kernel<MT, D>, dim3(grid), dim3(256), kLds, afrag, bfrag, isc, c, m, n, k >> 4, m_tiles, n_tiles,
               accumulate);
    SKN_LAUNCH_CHECK(ctx);
    return SKN_OK;
}

int launch_hilo_gemm_mt(skn_ctx* ctx, int mt, const u32x4* afrag, const u32x4* bfrag, const float* isc, float* c, int m, int n,
                        int k, int accumulate) {
    if (mt == 1) return launch_hilo_gemm<1, 4>(ctx, afrag, bfrag, isc, c, m, n, k, accumulate);
    if (mt == 2) return launch_hilo_gemm<2, 4>(ctx, afrag, bfrag, isc, c, m, n, k, accumulate);
    return launch_hilo_gemm<4, 4>(ctx, afrag, bfrag, isc, c, m, n, k, accumulate);
}

// ---- Q6_K path: weights unpacked in the kernel, two matrix instructions per k-step -----------------------
// w[n, 256 b + e] = d * sc_g * (q - 32) with q in 0..63, sc_g an int8 (one per sixteen elements), d fp16.  The integer
// sc_g (q - 32) needs thirteen bits, two more than an fp16 operand holds, so the scale is split, sc = 16 s1 + s0 with
// s0 in 0..15 and s1 in -8..7: (q - 32) s1 and (q - 32) s0 / 16 are exact fp16 numbers, each goes through the matrix
// core into the same accumulator, which then holds sum a sc (q - 32) / 16 of the superblock; at its end 16 d times
// that is added to the tile's running total and the accumulator starts again from zero (the first matrix instruction
// of a superblock takes no addend).  A quant is put together in place as the fp16 number 1024 + q (0x6400 | q: the
// low four bits masked out of ql, the two high bits out of qh shifted beside them), a pair per register, and one
// packed fused multiply-add per part, (1024 + q) s - 1056 s, makes the operand: the product is exact inside the
// instruction and 1056 s = 33 s 2^5 is an fp16 number, so nothing is rounded before the fp32 accumulation.
// Workgroup of four wavefronts, one per SIMD, tile (32 MT) x 64 as in the general path below: wavefront kq takes
// superblocks kq, kq + 4, ... of all the tile and the four partial tiles are added through LDS at the end.  The
// activations come in the fragment order of the Q4_K path; the element order inside a k-step -- 4 dw + {0, 2},
// 32 + 4 dw + {0, 2}, 4 dw + {1, 3}, 32 + 4 dw + {1, 3} with dw = 4 h + s in a chunk of 64 -- is the one Q6_K's own
// layout hands out: inside a half of 128 elements, element 32 Q + l has its low bits in nibble Q / 2 of byte
// 32 (Q % 2) + l of ql and its high bits at 2 Q of byte l of qh, so chunk c of the superblock (quarters 2 (c % 2) and
// 2 (c % 2) + 1 of half c / 2) takes dword s of three sixteen-byte pieces per lane -- ql + 64 (c / 2) + 16 h, the same
// + 32, qh + 32 (c / 2) + 16 h -- shifted right by 4 (c % 2).  Each lane reads the pieces of its own weight row (32
// rows per request, 210 bytes per superblock, no alignment beyond two bytes) straight into registers, half a
// superblock ahead; nothing but the final exchange passes through LDS and the loop has no barrier.
struct Q6kHalf {
    u32x4 qa[2], qb[2], qh[2];  // per 32-column block: ql + 16 h, ql + 32 + 16 h, qh + 16 h of the half
};

template <int MT, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void gemm_q6k_frag_kernel(const u32x4* __restrict__ afrag, const uint8_t* __restrict__ w, const float* __restrict__ inv_scale,
                          float* __restrict__ c, int m, int n, int k, int m_tiles, int n_tiles, int accumulate,
                          uint32_t a_bytes, uint32_t w_bytes, int xcd_rows, float* __restrict__ part, int part_blocks) {
    extern __shared__ __align__(16) float red[];  // 2 MT tiles x 3 copies x 1024 floats
    const int lane = threadIdx.x & 63;
    const int kq = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int h = lane >> 5, r = lane & 31;
    // Workgroup -> tile.  The packed weights of a tile are small (53 KiB per 64 columns at k = 4096) beside the
    // activations of its rows (1 MiB per 128 rows), so with up to eight row tiles an XCD (blockIdx % 8) keeps to one
    // row tile, whose activations then stay in its L2 while the column tiles stream through.
    int mt, tn;
    if (xcd_rows) {
        const int xcd = blockIdx.x & 7, per = 8 / m_tiles;
        mt = xcd % m_tiles;
        tn = (blockIdx.x >> 3) * per + xcd / m_tiles;
    } else {
        const int slot_in_xcd = blockIdx.x >> 3;
        mt = slot_in_xcd % m_tiles;
        tn = (slot_in_xcd / m_tiles) * 8 + (blockIdx.x & 7);
    }
    if (tn >= n_tiles) return;
    const int nb = k >> 8, nch = k >> 6;
    // (this workgroup's superblocks: all of them, or a part of k whose products go unscaled to part[blockIdx.y][m][n])
    const int sb0 = SPLIT ? (int)blockIdx.y * part_blocks : 0, sb1 = SPLIT ? min(sb0 + part_blocks, nb) : nb;
    // The weights are read with buffer loads too: the lane's byte offset (its weight row, its sixteen-byte half) plus
    // a scalar one (superblock, piece).  A piece of an odd superblock starts at an address that is only a multiple
    // of two.
    const __amdgpu_buffer_rsrc_t wrsrc = __builtin_amdgcn_make_buffer_rsrc((void*)w, 0, (int)w_bytes, 0x00020000);
    int wrow[2];
#pragma unroll
    for (int j = 0; j < 2; j++) wrow[j] = min(tn * kBN + 32 * j + r, n - 1) * nb * 210 + 16 * h;

    const __amdgpu_buffer_rsrc_t arsrc = __builtin_amdgcn_make_buffer_rsrc((void*)afrag, 0, (int)a_bytes, 0x00020000);
    uint32_t abase[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) abase[i] = (uint32_t)(mt * MT + i) * (uint32_t)nch * 4096u;
    constexpr int RING = 4;  // ring of k-steps, RING - 1 ahead (eight deep: the same time)
    u32x4 a[RING][MT];
    auto afetch = [&](int step, int slot) __attribute__((always_inline)) {  // step: 16 per superblock, absolute
#pragma unroll
        for (int i = 0; i < MT; i++)
            a[slot][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(arsrc, lane * 16, (int)(abase[i] + (uint32_t)step * 1024u), 0));
    };
    auto wload = [&](int j, int off) __attribute__((always_inline)) {
        return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, wrow[j], off, 0));
    };
    auto load_half = [&](int sb, int hf, Q6kHalf& H) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            H.qa[j] = wload(j, sb * 210 + 64 * hf);
            H.qb[j] = wload(j, sb * 210 + 64 * hf + 32);
            H.qh[j] = wload(j, sb * 210 + 128 + 32 * hf);
        }
    };
    // the sixteen scales of the superblock (both halves of the lanes read all of them: the lane's own sixteen-byte
    // offset is taken back out) and its d, per column block
    u32x4 scl[2], scl_n[2];
    uint32_t dh[2], dh_n[2];
    auto load_head = [&](int sb, u32x4 (&sc_out)[2], uint32_t (&d_out)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            sc_out[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, wrow[j] - 16 * h, sb * 210 + 192, 0));
            d_out[j] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(wrsrc, wrow[j] - 16 * h, sb * 210 + 208, 0);
        }
    };

    float16_t acc[MT][2], total[MT][2];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int x = 0; x < 16; x++) total[i][j][x] = 0.f;

    Q6kHalf H0, H1;
    if (sb0 + kq < sb1) {
        load_head(sb0 + kq, scl_n, dh_n);
        load_half(sb0 + kq, 0, H0);
#pragma unroll
        for (int s = 0; s < RING - 1; s++) afetch(16 * (sb0 + kq) + s, s);
    }
    for (int sb = sb0 + kq; sb < sb1; sb += 4) {
        const int sb_next = min(sb + 4, nb - 1);  // (past the end: a repeat of the last superblock, unused)
        float dsc[2];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            scl[j] = scl_n[j];
            dh[j] = dh_n[j];
            dsc[j] = (float)__builtin_bit_cast(_Float16, (uint16_t)dh[j]) * 16.0f;
        }
        // one chunk of 64 elements = four k-steps; cc = 0..3, its half is cc / 2
        auto chunk = [&](auto cc_const, const Q6kHalf& H) __attribute__((always_inline)) {
            constexpr int cc = decltype(cc_const)::value;
            constexpr int par = cc & 1;
            half2_t s0v[2][2], c0v[2][2], s1v[2][2], c1v[2][2];  // [column block][low 32 / high 32 of the chunk]
            u32x4 qa[2], qb[2], qh[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                qa[j] = par ? H.qa[j] >> 4u : H.qa[j];
                qb[j] = par ? H.qb[j] >> 4u : H.qb[j];
                qh[j] = par ? H.qh[j] >> 4u : H.qh[j];
                const uint32_t dw = scl[j][cc];  // scales 4 cc .. 4 cc + 3: the lane's groups are bytes h and 2 + h
#pragma unroll
                for (int g = 0; g < 2; g++) {
                    const int sc = __builtin_amdgcn_sbfe((int)dw, (unsigned)(8 * h + 16 * g), 8u);
                    const float f0 = (float)(sc & 15) * 0.0625f, f1 = (float)(sc >> 4);
                    s0v[j][g] = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(f0, f0));  // (four bits and a power of two: exact)
                    s1v[j][g] = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(f1, f1));
                    c0v[j][g] = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(-1056.0f * f0, -1056.0f * f0));
                    c1v[j][g] = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(-1056.0f * f1, -1056.0f * f1));
                }
            }
#pragma unroll
            for (int s = 0; s < 4; s++) {
                half8_t f0[2], f1[2];
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const uint32_t x = qa[j][s], y = qb[j][s], z = qh[j][s];
                    const uint32_t x8 = x >> 8, y8 = y >> 8, z8 = z >> 8;
                    const half2_t t[4] = {
                        __builtin_bit_cast(half2_t, ((z & 0x00030003u) << 4) | ((x & 0x000F000Fu) | 0x64006400u)),
                        __builtin_bit_cast(half2_t, ((z & 0x000C000Cu) << 2) | ((y & 0x000F000Fu) | 0x64006400u)),
                        __builtin_bit_cast(half2_t, ((z8 & 0x00030003u) << 4) | ((x8 & 0x000F000Fu) | 0x64006400u)),
                        __builtin_bit_cast(half2_t, ((z8 & 0x000C000Cu) << 2) | ((y8 & 0x000F000Fu) | 0x64006400u))};
                    u32x4 o0, o1;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        o0[e] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(t[e], s0v[j][e & 1], c0v[j][e & 1]));
                        o1[e] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(t[e], s1v[j][e & 1], c1v[j][e & 1]));
                    }
                    f0[j] = __builtin_bit_cast(half8_t, o0);
                    f1[j] = __builtin_bit_cast(half8_t, o1);
                }
                const int step = 4 * cc + s, slot = step & (RING - 1);
                // (the two matrix instructions of a tile are kept eight apart; the first of a superblock takes no addend)
                const float16_t zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    const half8_t fa = __builtin_bit_cast(half8_t, a[slot][i]);
#pragma unroll
                    for (int j = 0; j < 2; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa, f1[j], step == 0 ? zero : acc[i][j], 0, 0, 0);
                }
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    const half8_t fa = __builtin_bit_cast(half8_t, a[slot][i]);
#pragma unroll
                    for (int j = 0; j < 2; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa, f0[j], acc[i][j], 0, 0, 0);
                }
                // the slot of step - 1 is free: refill it RING - 1 steps ahead
                const int ahead = step + RING - 1;
                afetch(ahead < 16 ? 16 * sb + ahead : 16 * sb_next + ahead - 16, ahead & (RING - 1));
            }
        };
        load_half(sb, 1, H1);
        chunk(std::integral_constant<int, 0>{}, H0);
        chunk(std::integral_constant<int, 1>{}, H0);
        load_head(sb_next, scl_n, dh_n);
        load_half(sb_next, 0, H0);
        chunk(std::integral_constant<int, 2>{}, H1);
        chunk(std::integral_constant<int, 3>{}, H1);
        // the superblock's sum, in units of 16 d, joins the total
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int x = 0; x < 16; x++) total[i][j][x] = fmaf(dsc[j], acc[i][j][x], total[i][j][x]);
    }

    // the four partial tiles: tile t = 2 i + j belongs to wavefront t % 4, the other three hand theirs over
    float sc[(MT + 1) / 2][16];
    if constexpr (!SPLIT)
#pragma unroll
        for (int y = 0; y < (MT + 1) / 2; y++) row_scales(inv_scale, (mt * MT + min((kq >> 1) + 2 * y, MT - 1)) * 32, lane, sc[y]);
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int t = 2 * i + j, owner = t & 3;
            if (kq != owner) {
                float* dst = red + (t * 3 + ((kq - owner + 4) & 3) - 1) * 1024 + lane;
#pragma unroll
                for (int x = 0; x < 16; x++) dst[64 * x] = total[i][j][x];
            }
        }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int t = 2 * i + j;
            if (kq == (t & 3)) {
                float16_t sum = total[i][j];
#pragma unroll
                for (int o = 0; o < 3; o++)
#pragma unroll
                    for (int x = 0; x < 16; x++) sum[x] += red[(t * 3 + o) * 1024 + 64 * x + lane];
                if constexpr (SPLIT) store_tile_part(sum, part + (size_t)blockIdx.y * m * n, n, (mt * MT + i) * 32, tn * kBN + 32 * j, m, n, lane);
                else store_tile(sum, c, n, (mt * MT + i) * 32, tn * kBN + 32 * j, m, n, sc[i >> 1], lane, accumulate != 0);
            }
        }
}

// The same arithmetic with the wavefronts specialised: a workgroup of eight, on every SIMD a producer that unpacks
// (the vector instructions above) and a consumer that loads activation fragments and issues the matrix instructions,
// so that the two kinds of instruction come from different wavefronts and overlap.  Pair kq takes superblocks kq,
// kq + 4, ...; a phase is a chunk of 64 elements (four k-steps, sixteen 1 KiB weight fragments per pair: two column
// blocks x two parts); the producer works one phase ahead into the other of two LDS buffers, one bare barrier per
// phase.  The consumer keeps one set of accumulators in units of 16 d of the latest superblock whose d is not zero,
// rescaled on entering a superblock by the ratio the producer leaves beside the fragments (gemm_q4k_frag_kernel's
// scheme), so that it needs no running total.
constexpr int kQ6Stage = 4 * 4 * 1024;         // a phase of one pair: four k-steps x (two column blocks x two parts) x 1 KiB
constexpr int kQ6Aux = 2 * 256 + 256;          // per pair: the ratios of two superblocks in turn, then the last unit
constexpr int kQ6PcLds = 4 * 2 * kQ6Stage + 4 * kQ6Aux;

template <bool SPLIT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_q6k_pc_kernel(const u32x4* __restrict__ afrag, const uint8_t* __restrict__ w, const float* __restrict__ inv_scale,
                        float* __restrict__ c, int m, int n, int k, int m_tiles, int n_tiles, int accumulate,
                        uint32_t a_bytes, uint32_t w_bytes, float* __restrict__ part, int part_blocks) {
    constexpr int MT = 4;
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const int kq = wave & 3;
    const bool producer = wave >= 4;
    const int h = lane >> 5, r = lane & 31;
    const int xcd = blockIdx.x & 7, per = 8 / m_tiles;  // (an XCD keeps to one row tile, as above; m_tiles divides 8)
    const int mt = xcd % m_tiles, tn = (blockIdx.x >> 3) * per + xcd / m_tiles;
    if (tn >= n_tiles) return;
    const int nb = k >> 8, nch = k >> 6;
    const int sb0 = SPLIT ? (int)blockIdx.y * part_blocks : 0, sb1 = SPLIT ? min(sb0 + part_blocks, nb) : nb;  // (as above)
    const int nsb = (sb1 - sb0 + 3) >> 2;  // superblocks of the busiest pair
    uint8_t* stage = lds + kq * 2 * kQ6Stage;
    uint8_t* aux = lds + 4 * 2 * kQ6Stage + kq * kQ6Aux;
    auto barrier = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    using C0 = std::integral_constant<int, 0>;
    using C1 = std::integral_constant<int, 1>;
    using C2 = std::integral_constant<int, 2>;
    using C3 = std::integral_constant<int, 3>;
    float* red = reinterpret_cast<float*>(lds);  // (for the end, when the stage buffers are free: 2 MT x 3 x 4 KiB of them)

    if (producer) {
        const __amdgpu_buffer_rsrc_t wrsrc = __builtin_amdgcn_make_buffer_rsrc((void*)w, 0, (int)w_bytes, 0x00020000);
        int wrow[2];
#pragma unroll
        for (int j = 0; j < 2; j++) wrow[j] = min(tn * kBN + 32 * j + r, n - 1) * nb * 210 + 16 * h;
        auto wload = [&](int j, int off) __attribute__((always_inline)) {
            return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, wrow[j], off, 0));
        };
        auto load_half = [&](int sb, int hf, Q6kHalf& H) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
                H.qa[j] = wload(j, sb * 210 + 64 * hf);
                H.qb[j] = wload(j, sb * 210 + 64 * hf + 32);
                H.qh[j] = wload(j, sb * 210 + 128 + 32 * hf);
            }
        };
        u32x4 scl[2], scl_n[2];
        uint32_t dh[2], dh_n[2];
        auto load_head = [&](int sb, u32x4 (&sc_out)[2], uint32_t (&d_out)[2]) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
                sc_out[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, wrow[j] - 16 * h, sb * 210 + 192, 0));
                d_out[j] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(wrsrc, wrow[j] - 16 * h, sb * 210 + 208, 0);
            }
        };
        Q6kHalf H0, H1;
        float cs[2] = {1.f, 1.f};
        bool live[2] = {true, true};
        // entering superblock i (pair-local): its head becomes current, its ratio goes to aux[i & 1]
        auto enter = [&](int i) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
                scl[j] = scl_n[j], dh[j] = dh_n[j];
                const float d = (float)__builtin_bit_cast(_Float16, (uint16_t)dh[j]);
                live[j] = d != 0.f;  // (a zero d: the products are zeroed and the unit stays)
                const float cs_new = live[j] ? d * 16.0f : cs[j];
                const float ratio = cs[j] / cs_new;
                cs[j] = cs_new;
                if (h == 0) *reinterpret_cast<float*>(aux + (i & 1) * 256 + (j * 32 + r) * 4) = ratio;
            }
        };
        // chunk cc of the current superblock -> sixteen fragments into buffer `buf`
        auto unpack = [&](auto cc_const, const Q6kHalf& H, int buf) __attribute__((always_inline)) {
            constexpr int cc = decltype(cc_const)::value;
            constexpr int par = cc & 1;
            uint8_t* dst = stage + buf * kQ6Stage + lane * 16;
            half2_t s0v[2][2], c0v[2][2], s1v[2][2], c1v[2][2];  // [column block][low 32 / high 32 of the chunk]
            u32x4 qa[2], qb[2], qh[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                qa[j] = par ? H.qa[j] >> 4u : H.qa[j];
                qb[j] = par ? H.qb[j] >> 4u : H.qb[j];
                qh[j] = par ? H.qh[j] >> 4u : H.qh[j];
                const uint32_t dw = scl[j][cc];  // scales 4 cc .. 4 cc + 3: the lane's groups are bytes h and 2 + h
#pragma unroll
                for (int g = 0; g < 2; g++) {
                    const int sc = live[j] ? __builtin_amdgcn_sbfe((int)dw, (unsigned)(8 * h + 16 * g), 8u) : 0;
                    const float f0 = (float)(sc & 15) * 0.0625f, f1 = (float)(sc >> 4);
                    s0v[j][g] = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(f0, f0));  // (four bits and a power of two: exact)
                    s1v[j][g] = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(f1, f1));
                    c0v[j][g] = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(-1056.0f * f0, -1056.0f * f0));
                    c1v[j][g] = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(-1056.0f * f1, -1056.0f * f1));
                }
            }
#pragma unroll
            for (int s4 = 0; s4 < 4; s4++)
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const uint32_t x = qa[j][s4], y = qb[j][s4], z = qh[j][s4];
                    const uint32_t x8 = x >> 8, y8 = y >> 8, z8 = z >> 8;
                    const half2_t t[4] = {
                        __builtin_bit_cast(half2_t, ((z & 0x00030003u) << 4) | ((x & 0x000F000Fu) | 0x64006400u)),
                        __builtin_bit_cast(half2_t, ((z & 0x000C000Cu) << 2) | ((y & 0x000F000Fu) | 0x64006400u)),
                        __builtin_bit_cast(half2_t, ((z8 & 0x00030003u) << 4) | ((x8 & 0x000F000Fu) | 0x64006400u)),
                        __builtin_bit_cast(half2_t, ((z8 & 0x000C000Cu) << 2) | ((y8 & 0x000F000Fu) | 0x64006400u))};
                    u32x4 o0, o1;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        o0[e] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(t[e], s0v[j][e & 1], c0v[j][e & 1]));
                        o1[e] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(t[e], s1v[j][e & 1], c1v[j][e & 1]));
                    }
                    *reinterpret_cast<u32x4*>(dst + ((s4 * 2 + j) * 2 + 0) * 1024) = o1;
                    *reinterpret_cast<u32x4*>(dst + ((s4 * 2 + j) * 2 + 1) * 1024) = o0;
                }
        };
        // While the consumers multiply phase (i, cc) the producer unpacks the phase after it.  Requests, two phases
        // before their use: head and first half of the next superblock with chunk 2, its second half with its chunk 0.
        auto phase = [&](int i, auto cc_const) __attribute__((always_inline)) {
            constexpr int cc = decltype(cc_const)::value;
            const int sb = sb0 + 4 * i + kq;
            if (sb < sb1) {
                const int sbn = min(sb + 4, nb - 1);  // (past the end: a repeat, unused)
                if (cc == 0) unpack(C1{}, H0, 1);
                if (cc == 1) {
                    load_head(sbn, scl_n, dh_n);
                    load_half(sbn, 0, H0);
                    unpack(C2{}, H1, 0);
                }
                if (cc == 2) unpack(C3{}, H1, 1);
                if (cc == 3 && sb + 4 < sb1) {
                    enter(i + 1);
                    load_half(sb + 4, 1, H1);
                    unpack(C0{}, H0, 0);
                }
            }
            barrier();
        };
        if (sb0 + kq < sb1) {
            load_head(sb0 + kq, scl_n, dh_n);
            load_half(sb0 + kq, 0, H0);
            load_half(sb0 + kq, 1, H1);
            enter(0);
            unpack(C0{}, H0, 0);
        }
        barrier();
        for (int i = 0; i < nsb; i++) {
            phase(i, C0{});
            phase(i, C1{});
            phase(i, C2{});
            phase(i, C3{});
        }
        if (h == 0) {
#pragma unroll
            for (int j = 0; j < 2; j++) *reinterpret_cast<float*>(aux + 512 + (j * 32 + r) * 4) = cs[j];
        }
        barrier();
        barrier();
    } else {
        const __amdgpu_buffer_rsrc_t arsrc = __builtin_amdgcn_make_buffer_rsrc((void*)afrag, 0, (int)a_bytes, 0x00020000);
        uint32_t abase[MT];
#pragma unroll
        for (int i = 0; i < MT; i++) abase[i] = (uint32_t)(mt * MT + i) * (uint32_t)nch * 4096u;
        u32x4 a[4][MT];  // ring of four k-steps, three ahead
        auto afetch = [&](int step, int slot) __attribute__((always_inline)) {  // step: 16 per superblock, absolute
#pragma unroll
            for (int i = 0; i < MT; i++)
                a[slot][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(arsrc, lane * 16, (int)(abase[i] + (uint32_t)step * 1024u), 0));
        };
        float16_t acc[MT][2];
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int x = 0; x < 16; x++) acc[i][j][x] = 0.f;
        auto phase = [&](int i, auto cc_const) __attribute__((always_inline)) {
            constexpr int cc = decltype(cc_const)::value;
            const int sb = sb0 + 4 * i + kq;
            if (sb < sb1) {
                if (cc == 0) {
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        const float ratio = *reinterpret_cast<const float*>(aux + (i & 1) * 256 + (j * 32 + r) * 4);
#pragma unroll
                        for (int ii = 0; ii < MT; ii++)
#pragma unroll
                            for (int x = 0; x < 16; x++) acc[ii][j][x] *= ratio;
                    }
                }
                const uint8_t* src = stage + (cc & 1) * kQ6Stage + lane * 16;
                const int sbn = min(sb + 4, nb - 1);
                // (the weight fragments of step s + 1 are read from LDS before the matrix instructions of step s are issued)
                half8_t fb[2][2][2];  // [step parity][column block][part]
#pragma unroll
                for (int j = 0; j < 2; j++)
#pragma unroll
                    for (int pt = 0; pt < 2; pt++) fb[0][j][pt] = *reinterpret_cast<const half8_t*>(src + (j * 2 + pt) * 1024);
#pragma unroll
                for (int s4 = 0; s4 < 4; s4++) {
                    const int step = 4 * cc + s4, slot = step & 3;
                    if (s4 + 1 < 4) {
#pragma unroll
                        for (int j = 0; j < 2; j++)
#pragma unroll
                            for (int pt = 0; pt < 2; pt++)
                                fb[(s4 + 1) & 1][j][pt] = *reinterpret_cast<const half8_t*>(src + (((s4 + 1) * 2 + j) * 2 + pt) * 1024);
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int pt = 0; pt < 2; pt++)
#pragma unroll
                        for (int ii = 0; ii < MT; ii++) {
                            const half8_t fa = __builtin_bit_cast(half8_t, a[slot][ii]);
#pragma unroll
                            for (int j = 0; j < 2; j++)
                                acc[ii][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa, fb[s4 & 1][j][pt], acc[ii][j], 0, 0, 0);
                        }
                    const int ahead = step + 3;
                    afetch(ahead < 16 ? 16 * sb + ahead : 16 * sbn + ahead - 16, ahead & 3);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            barrier();
        };
        if (sb0 + kq < sb1) {
#pragma unroll
            for (int s = 0; s < 3; s++) afetch(16 * (sb0 + kq) + s, s);
        }
        barrier();
        for (int i = 0; i < nsb; i++) {
            phase(i, C0{});
            phase(i, C1{});
            phase(i, C2{});
            phase(i, C3{});
        }
        barrier();
        float sc[(MT + 1) / 2][16];
        if constexpr (!SPLIT)
#pragma unroll
            for (int y = 0; y < (MT + 1) / 2; y++) row_scales(inv_scale, (mt * MT + min((kq >> 1) + 2 * y, MT - 1)) * 32, lane, sc[y]);
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const float unit = *reinterpret_cast<const float*>(aux + 512 + (j * 32 + r) * 4);
#pragma unroll
            for (int ii = 0; ii < MT; ii++) {
#pragma unroll
                for (int x = 0; x < 16; x++) acc[ii][j][x] *= unit;
                const int t = 2 * ii + j, owner = t & 3;
                if (kq != owner) {
                    float* dst = red + (t * 3 + ((kq - owner + 4) & 3) - 1) * 1024 + lane;
#pragma unroll
                    for (int x = 0; x < 16; x++) dst[64 * x] = acc[ii][j][x];
                }
            }
        }
        barrier();
#pragma unroll
        for (int ii = 0; ii < MT; ii++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int t = 2 * ii + j;
                if (kq == (t & 3)) {
                    float16_t sum = acc[ii][j];
#pragma unroll
                    for (int o = 0; o < 3; o++)
#pragma unroll
                        for (int x = 0; x < 16; x++) sum[x] += red[(t * 3 + o) * 1024 + 64 * x + lane];
                    if constexpr (SPLIT) store_tile_part(sum, part + (size_t)blockIdx.y * m * n, n, (mt * MT + ii) * 32, tn * kBN + 32 * j, m, n, lane);
                    else store_tile(sum, c, n, (mt * MT + ii) * 32, tn * kBN + 32 * j, m, n, sc[ii >> 1], lane, accumulate != 0);
                }
            }
    }
}

// The same for wide weight matrices in the form of gemm_q4k_tall_kernel: a 256 x 128 tile, k walked superblock by
// superblock by all eight wavefronts; four consumers own 64 rows each (a 64 x 128 tile per wavefront), four producers
// 32 columns each, whose blocks they unpack once for all 256 rows into LDS (per k-step and column block the two
// parts of the split scale as two fragments), two phases (chunks of 64 elements) ahead, three buffers, one bare
// barrier per phase.  The consumers take the two parts one after the other (the same activation fragment, eight
// matrix instructions each) and read the next half-step's four fragments from LDS, across the barrier too, while the
// current eight instructions run.  Accumulators in units of 16 d as in gemm_q6k_pc_kernel, the change of unit spread
// between the matrix instructions on both sides of a superblock's end.
constexpr int kQ6TlStage = 4 * 8 * 1024;          // a phase: four k-steps x (four column blocks x two parts) x 1 KiB
constexpr int kQ6TlLds = 3 * kQ6TlStage + 2 * 128 * 4 + 128 * 4 + 256 * 4;

__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_q6k_tall_kernel(const u32x4* __restrict__ afrag, const uint8_t* __restrict__ w, const float* __restrict__ inv_scale,
                          float* __restrict__ c, int m, int n, int k, int m_tiles, int accumulate, uint32_t a_bytes,
                          uint32_t w_bytes) {
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const int me = wave & 3;  // consumer: its 64 rows; producer: its 32 columns
    const bool producer = wave >= 4;
    const int h = lane >> 5, r = lane & 31;
    const int nb = k >> 8, nch = k >> 6;
    const int mt = blockIdx.x % m_tiles, tn = blockIdx.x / m_tiles;  // (the row tiles of a column tile run side by side)
    const int n0 = tn * 128;
    uint8_t* stage = lds;
    float* ratios = reinterpret_cast<float*>(lds + 3 * kQ6TlStage);  // [superblock parity][128 columns]
    float* fin = ratios + 2 * 128;                                   // the last unit of the 128 columns
    float* isc_lds = fin + 128;                                      // the scales of the tile's 256 rows
    if (tid < 256) isc_lds[tid] = inv_scale[mt * 256 + tid];
    auto barrier = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    using C0 = std::integral_constant<int, 0>;
    using C1 = std::integral_constant<int, 1>;
    using C2 = std::integral_constant<int, 2>;
    using C3 = std::integral_constant<int, 3>;
    // the three buffers in turn: phase p is multiplied from b_cur, phase p + 1 lies complete in b_nxt, phase p + 2 is
    // being written to b_nx2 (byte offsets, uniform)
    int b_cur = 0, b_nxt = kQ6TlStage, b_nx2 = 2 * kQ6TlStage;
    auto turn = [&]() __attribute__((always_inline)) {
        const int t = b_cur;
        b_cur = b_nxt, b_nxt = b_nx2, b_nx2 = t;
    };

    if (producer) {
        const __amdgpu_buffer_rsrc_t wrsrc = __builtin_amdgcn_make_buffer_rsrc((void*)w, 0, (int)w_bytes, 0x00020000);
        const int col = 32 * me + r;
        const int wrow = min(n0 + col, n - 1) * nb * 210;
        u32x4 qa[2], qb[2], qh[2];  // [half of the superblock]: ql + 16 h, ql + 32 + 16 h, qh + 16 h
        u32x4 scl, scl_n;
        uint32_t dh_n = 0;
        auto load_half = [&](int sb, int hf) __attribute__((always_inline)) {
            sb = min(sb, nb - 1);  // (past the end: a repeat, unused)
            qa[hf] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, wrow + 16 * h, sb * 210 + 64 * hf, 0));
            qb[hf] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, wrow + 16 * h, sb * 210 + 64 * hf + 32, 0));
            qh[hf] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, wrow + 16 * h, sb * 210 + 128 + 32 * hf, 0));
        };
        auto load_head = [&](int sb) __attribute__((always_inline)) {
            sb = min(sb, nb - 1);
            scl_n = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, wrow, sb * 210 + 192, 0));
            dh_n = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(wrsrc, wrow, sb * 210 + 208, 0);
        };
        float cs = 1.f;
        bool live = true;
        // entering superblock sb: its head becomes current, its ratio goes to ratios[sb & 1]
        auto enter = [&](int sb) __attribute__((always_inline)) {
            asm volatile("" : "+v"(scl_n), "+v"(dh_n));  // (taken up here and no earlier)
            scl = scl_n;
            const float d = (float)__builtin_bit_cast(_Float16, (uint16_t)dh_n);
            live = d != 0.f;  // (a zero d: the products are zeroed and the unit stays)
            const float cs_new = live ? d * 16.0f : cs;
            const float ratio = cs / cs_new;
            cs = cs_new;
            if (h == 0) ratios[(sb & 1) * 128 + col] = ratio;
        };
        // chunk cc of the current superblock -> four k-steps x two parts of this producer's column block into the buffer at `buf`
        auto unpack = [&](auto cc_const, int buf) __attribute__((always_inline)) {
            constexpr int cc = decltype(cc_const)::value;
            constexpr int par = cc & 1, hf = cc >> 1;
            uint8_t* dst = stage + buf + me * 2048 + lane * 16;
            asm volatile("" : "+v"(qa[hf]), "+v"(qb[hf]), "+v"(qh[hf]));  // (as for the head)
            const u32x4 xa = par ? qa[hf] >> 4u : qa[hf], xb = par ? qb[hf] >> 4u : qb[hf], xh = par ? qh[hf] >> 4u : qh[hf];
            half2_t s0v[2], c0v[2], s1v[2], c1v[2];  // [low 32 / high 32 of the chunk]
            const uint32_t dw = scl[cc];  // scales 4 cc .. 4 cc + 3: the lane's groups are bytes h and 2 + h
#pragma unroll
            for (int g = 0; g < 2; g++) {
                const int sc = live ? __builtin_amdgcn_sbfe((int)dw, (unsigned)(8 * h + 16 * g), 8u) : 0;
                const float f0 = (float)(sc & 15) * 0.0625f, f1 = (float)(sc >> 4);
                s0v[g] = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(f0, f0));  // (four bits and a power of two: exact)
                s1v[g] = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(f1, f1));
                c0v[g] = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(-1056.0f * f0, -1056.0f * f0));
                c1v[g] = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(-1056.0f * f1, -1056.0f * f1));
            }
#pragma unroll
            for (int s4 = 0; s4 < 4; s4++) {
                const uint32_t x = xa[s4], y = xb[s4], z = xh[s4];
                const uint32_t x8 = x >> 8, y8 = y >> 8, z8 = z >> 8;
                const half2_t t[4] = {
                    __builtin_bit_cast(half2_t, ((z & 0x00030003u) << 4) | ((x & 0x000F000Fu) | 0x64006400u)),
                    __builtin_bit_cast(half2_t, ((z & 0x000C000Cu) << 2) | ((y & 0x000F000Fu) | 0x64006400u)),
                    __builtin_bit_cast(half2_t, ((z8 & 0x00030003u) << 4) | ((x8 & 0x000F000Fu) | 0x64006400u)),
                    __builtin_bit_cast(half2_t, ((z8 & 0x000C000Cu) << 2) | ((y8 & 0x000F000Fu) | 0x64006400u))};
                u32x4 o0, o1;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    o0[e] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(t[e], s0v[e & 1], c0v[e & 1]));
                    o1[e] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(t[e], s1v[e & 1], c1v[e & 1]));
                }
                *reinterpret_cast<u32x4*>(dst + s4 * 8192) = o1;          // part 1: (q - 32) s1
                *reinterpret_cast<u32x4*>(dst + s4 * 8192 + 1024) = o0;   // part 0: (q - 32) s0 / 16
            }
        };
        // While the consumers multiply phase (sb, cc) the producer unpacks the phase two after it -- chunks 2 and 3 of
        // the superblock, then chunks 0 and 1 of the next, whose head it takes up with chunk 0.  Requests, two phases
        // before their use: head and first half of the next superblock with chunk 2, its second half with its chunk 0.
        // (After the last superblock it unpacks a repeat into buffers that nobody reads any more -- no branch, so
        // that the requests are not moved down into one -- and keeps the unit.)
        auto phase = [&](int sb, auto cc_const) __attribute__((always_inline)) {
            constexpr int cc = decltype(cc_const)::value;
            if (cc == 0) {
                load_head(sb + 1);
                load_half(sb + 1, 0);
                unpack(C2{}, b_nx2);
            }
            if (cc == 1) unpack(C3{}, b_nx2);
            if (cc == 2) {
                const float keep = cs;
                enter(sb + 1);
                if (sb + 1 >= nb) cs = keep;
                load_half(sb + 1, 1);
                unpack(C0{}, b_nx2);
            }
            if (cc == 3) unpack(C1{}, b_nx2);
            barrier();
            turn();
        };
        load_head(0);
        load_half(0, 0);
        load_half(0, 1);
        enter(0);
        unpack(C0{}, b_cur);
        unpack(C1{}, b_nxt);
        barrier();
        for (int sb = 0; sb < nb; sb++) {
            phase(sb, C0{});
            phase(sb, C1{});
            phase(sb, C2{});
            phase(sb, C3{});
        }
        if (h == 0) fin[col] = cs;
        barrier();
    } else {
        constexpr int MT = 2;
        const __amdgpu_buffer_rsrc_t arsrc = __builtin_amdgcn_make_buffer_rsrc((void*)afrag, 0, (int)a_bytes, 0x00020000);
        const int mb0 = mt * 8 + me * MT;  // first row block of this consumer
        uint32_t abase[MT];
#pragma unroll
        for (int i = 0; i < MT; i++) abase[i] = (uint32_t)(mb0 + i) * (uint32_t)nch * 4096u;
        u32x4 a[8][MT];  // ring of eight k-steps, seven ahead
        auto afetch = [&](int step, int slot) __attribute__((always_inline)) {  // step: absolute, 16 per superblock
            step = min(step, 16 * nb - 1);  // (past the end: the last step again, unused)
#pragma unroll
            for (int i = 0; i < MT; i++)
                a[slot][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(arsrc, lane * 16, (int)(abase[i] + (uint32_t)step * 1024u), 0));
        };
        float16_t acc[MT][4];
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int x = 0; x < 16; x++) acc[i][j][x] = 0.f;
        // half-step hs = 2 s4 + (part 1 first, then part 0): fragment (s4, j, part) of a phase at (s4 * 8 + j * 2 + p) KiB
        // with p = 0 for part 1; the four fragments of half-step hs + 1 are read while those of hs are multiplied,
        // half-step 0 of a phase in fb[0]
        half8_t fb[2][4];
        float ratio[4] = {1.f, 1.f, 1.f, 1.f};  // of the superblock being entered, by column block
        // tile t = 4 i + j changes its unit: half `part` of its sixteen registers
        auto rescale = [&](int t, int part) __attribute__((always_inline)) {
#pragma unroll
            for (int x = 0; x < 8; x++) acc[t >> 2][t & 3][8 * part + x] *= ratio[t & 3];
        };
        auto fence = [&]() __attribute__((always_inline)) { __builtin_amdgcn_sched_barrier(0); };
        auto phase = [&](int sb, auto cc_const) __attribute__((always_inline)) {
            constexpr int cc = decltype(cc_const)::value;
            const uint8_t* src = stage + b_cur + lane * 16;
            const uint8_t* srcn = stage + b_nxt + lane * 16;
            float rnext[4];
            if (cc == 3) {  // (the ratios of the next superblock, left by the producers a phase ago: used at the end of this phase)
#pragma unroll
                for (int j = 0; j < 4; j++) rnext[j] = ratios[((sb + 1) & 1) * 128 + j * 32 + r];
            }
#pragma unroll
            for (int hs = 0; hs < 8; hs++) {
                const int s4 = hs >> 1, step = 4 * cc + s4, slot = step & 7;
                if (hs < 7) {
                    const int s4n = (hs + 1) >> 1, ptn = (hs + 1) & 1;
#pragma unroll
                    for (int j = 0; j < 4; j++) fb[(hs + 1) & 1][j] = *reinterpret_cast<const half8_t*>(src + s4n * 8192 + j * 2048 + ptn * 1024);
                } else {  // the next phase's first half-step: complete since the barrier before this phase
#pragma unroll
                    for (int j = 0; j < 4; j++) fb[0][j] = *reinterpret_cast<const half8_t*>(srcn + j * 2048);
                }
                if (cc == 3 && hs == 7) {
#pragma unroll
                    for (int j = 0; j < 4; j++) ratio[j] = sb + 1 < nb ? rnext[j] : 1.0f;  // (none after the last superblock)
                }
                fence();
                if ((cc == 0 && hs == 0) || (cc == 3 && hs == 7)) {
                    // the two sides of a superblock's end: tiles 0 .. 2 change their unit between the last matrix
                    // instructions of the superblock, tiles 3 .. 7 between the first of the next
#pragma unroll
                    for (int t = 0; t < 8; t++) {
                        acc[t >> 2][t & 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a[slot][t >> 2]), fb[hs & 1][t & 3],
                                                                                    acc[t >> 2][t & 3], 0, 0, 0);
                        fence();
                        if (cc == 3) {
                            if (t >= 2) rescale((t - 2) >> 1, t & 1);
                        } else {
                            if (t < 4) rescale(3 + (t >> 1), t & 1);
                            if (t >= 4 && t < 7) rescale(t + 1, 0), rescale(t + 1, 1);
                        }
                        fence();
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < MT; i++) {
                        const half8_t fa = __builtin_bit_cast(half8_t, a[slot][i]);
#pragma unroll
                        for (int j = 0; j < 4; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa, fb[hs & 1][j], acc[i][j], 0, 0, 0);
                    }
                }
                if (hs & 1) afetch(16 * sb + step + 7, (step + 7) & 7);
                fence();
            }
            barrier();
            turn();
        };
#pragma unroll
        for (int s = 0; s < 7; s++) afetch(s, s);
        barrier();
#pragma unroll
        for (int j = 0; j < 4; j++) fb[0][j] = *reinterpret_cast<const half8_t*>(stage + b_cur + lane * 16 + j * 2048);
        for (int sb = 0; sb < nb; sb++) {
            phase(sb, C0{});
            phase(sb, C1{});
            phase(sb, C2{});
            phase(sb, C3{});
        }
        barrier();
#pragma unroll
        for (int i = 0; i < MT; i++) {
            float sc[16];
#pragma unroll
            for (int x = 0; x < 16; x++) sc[x] = isc_lds[(me * MT + i) * 32 + 8 * (x >> 2) + 4 * h + (x & 3)];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float unit = fin[j * 32 + r];
#pragma unroll
                for (int x = 0; x < 16; x++) acc[i][j][x] *= unit;
                store_tile(acc[i][j], c, n, (mb0 + i) * 32, n0 + 32 * j, m, n, sc, lane, accumulate != 0);
            }
        }
    }
}

template <int MT, bool SPLIT>
int launch_q6k_gemm(skn_ctx* ctx, const u32x4* afrag, const uint8_t* w, const float* isc, float* c, int m, int n, int k,
                    int accumulate, int splits, float* part) {
    constexpr int kLds = 2 * MT * 3 * 4096;
    const int m_tiles = (m + 32 * MT - 1) / (32 * MT), n_tiles = (n + kBN - 1) / kBN;
    const int xcd_rows = 8 % m_tiles == 0 ? 1 : 0, part_blocks = (k / 256 + splits - 1) / splits;
    const unsigned grid = xcd_rows ? (unsigned)(8 * ((n_tiles + 8 / m_tiles - 1) / (8 / m_tiles))) : (unsigned)(((n_tiles + 7) / 8) * 8 * m_tiles);
    const uint32_t a_bytes = (uint32_t)((size_t)m_tiles * 32 * MT * k * 2);  // (checked by the caller to fit)
    const uint32_t w_bytes = (uint32_t)((size_t)n * (k / 256) * 210);  // (checked by the caller to fit)
    // 128-row tiles: the kernel with specialised wavefronts (measured 6 - 11 % faster); option value 2 keeps to the other
    // (up to 16384 elements per row: a rescale per superblock rounds the accumulators once more, the other form does not)
    if (MT == 4 && xcd_rows && k <= 16384 && ctx->opt_gemm_q6k_fused != 2) {
        skn_launch(ctx, gemm_q6k_pc_kernel<SPLIT>, dim3(grid, splits), dim3(512), kQ6PcLds, afrag, w, isc, c, m, n, k, m_tiles, n_tiles, accumulate,
                   a_bytes, w_bytes, part, part_blocks);
        SKN_LAUNCH_CHECK(ctx);
        return SKN_OK;
    }
    skn_launch(ctx, gemm_q6k_frag_kernel<MT, SPLIT>, dim3(grid, splits), dim3(256), kLds, afrag, w, isc, c, m, n, k, m_tiles, n_tiles, accumulate,
               a_bytes, w_bytes, xcd_rows, part, part_blocks);
    SKN_LAUNCH_CHECK(ctx);
    return SKN_OK;
}

int launch_q6k_gemm_mt(skn_ctx* ctx, int mt, const u32x4* afrag, const uint8_t* w, const float* isc, float* c, int m, int n,
                       int k, int accumulate, int splits, float* part) {
    if (splits < 2) part = nullptr;
    if (!part) {
        if (mt == 1) return launch_q6k_gemm<1, false>(ctx, afrag, w, isc, c, m, n, k, accumulate, splits, part);
        if (mt == 2) return launch_q6k_gemm<2, false>(ctx, afrag, w, isc, c, m, n, k, accumulate, splits, part);
        return launch_q6k_gemm<4, false>(ctx, afrag, w, isc, c, m, n, k, accumulate, splits, part);
    }
    if (mt == 1) SKN_TRY((launch_q6k_gemm<1, true>(ctx, afrag, w, isc, c, m, n, k, accumulate, splits, part)));
    else if (mt == 2) SKN_TRY((launch_q6k_gemm<2, true>(ctx, afrag, w, isc, c, m, n, k, accumulate, splits, part)));
    else SKN_TRY((launch_q6k_gemm<4, true>(ctx, afrag, w, isc, c, m, n, k, accumulate, splits, part)));
    const skn_gemm_parts ps = {{c, nullptr, nullptr}, {n, 0, 0}, {0, 0, 0}, {accumulate, 0, 0}, 1, 0};
    return skn_gemm_add_parts(ctx, part, splits, n, ps, isc, m);
}

}  // namespace

int skn_gemm_add_parts(skn_ctx* ctx, const float* part, int splits, int cols, const skn_gemm_parts& segs, const float* isc, int m) {
    bool wide = true;
    for (int i = 0; i < segs.count; i++) wide = wide && segs.n[i] % 4 == 0 && ((uintptr_t)segs.c[i] & 15) == 0;
    const int n = segs.pair ? segs.n[0] : cols;
    if (wide) skn_launch(ctx, gemm_add_parts_kernel<4>, dim3((n / 4 + 255) / 256, m), dim3(256), 0, part, splits, cols, segs, isc, m);
    else skn_launch(ctx, gemm_add_parts_kernel<1>, dim3((n + 255) / 256, m), dim3(256), 0, part, splits, cols, segs, isc, m);
    SKN_LAUNCH_CHECK(ctx);
    return SKN_OK;
}

// How many workgroups share a tile's k: as many as there are compute units for, up to sixteen, at least one superblock for each
// of a workgroup's four k-parts.  us per call, unsplit -> chosen: Q6_K 41 x 4096 x 11008 (64 tiles) 81 -> 34.5, 120 x 4096 x 11008
// 106 -> 45, 200 x 4096 x 11008 (128 tiles) 108 -> 71; Q4_K 41 x 4096 x 11008 35.7 -> 24.6, 41 x 4096 x 4096 17.8 -> 15.1.
// Filling every compute unit twice is no gain (Q4_K 41 x 4096 x 11008 27.2, 120 x 4096 x 4096
// 21.5 against 18.7), nor is a second part for tiles that fill two thirds of the device (Q4_K 41 x 11008 x 4096 22.2 against
// 19.6, Q6_K 333 x 4096 x 4096 59 against 54): the addition costs 3 us and the parts their way through memory.
int skn_gemm_k_splits(const skn_ctx* ctx, int m, int tiles, int nb) {
    if (m > 65535) return 1;  // (a grid dimension of the addition)
    const int want = ctx->opt_gemm_split > 0 ? std::min(ctx->opt_gemm_split, nb) : std::max(1, std::min({ctx->compute_units / tiles, (nb + 3) / 4, 16}));
    const int each = (nb + want - 1) / want;
    return (nb + each - 1) / each;  // (no workgroup without a superblock)
}

static bool may_allocate(skn_ctx* ctx) {  // (asking for memory would end a capture)
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(ctx->stream, &status) == hipSuccess && status == hipStreamCaptureStatusNone) return true;
    (void)hipGetLastError();
    return false;
}

static bool grow_parts(skn_ctx* ctx, size_t bytes) {
    if (!may_allocate(ctx)) return false;
    void* p = nullptr;
    if (hipMalloc(&p, bytes) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    if (ctx->gemm_parts && (hipStreamSynchronize(ctx->stream) != hipSuccess || hipFree(ctx->gemm_parts) != hipSuccess)) {
        (void)hipGetLastError();
        (void)hipFree(p);
        return false;
    }
    ctx->gemm_parts = p;
    ctx->gemm_parts_bytes = bytes;
    return true;
}

int skn_gemm_workspace(skn_ctx* ctx, size_t bytes, size_t most, uint8_t** out, bool ahead) {
    most = std::max(bytes, most);
    bool grow = bytes > ctx->gemm_ws_bytes && !(ahead && !may_allocate(ctx));
    if (bytes <= ctx->gemm_ws_bytes && most > ctx->gemm_ws_bytes && !ctx->gemm_ws_kept) {
        grow = may_allocate(ctx);
        ctx->gemm_ws_kept = !grow;
    }
    if (grow) {
        SKN_HIP(ctx, hipStreamSynchronize(ctx->stream));
        if (ctx->gemm_ws) SKN_HIP(ctx, hipFree(ctx->gemm_ws));
        ctx->gemm_ws = nullptr;
        ctx->gemm_ws_bytes = 0;
        ctx->gemm_ws_kept = false;
        hipError_t e = hipMalloc(&ctx->gemm_ws, most);
        if (e != hipSuccess && most > bytes) {
            (void)hipGetLastError();
            e = hipMalloc(&ctx->gemm_ws, most = bytes);
        }
        if (e != hipSuccess) {
            (void)hipGetLastError();
            return skn_fail(ctx, SKN_ERR_OOM, "skn_gemm_q: %zu bytes of workspace: %s", bytes, hipGetErrorString(e));
        }
        ctx->gemm_ws_bytes = most;
        // (a workgroup per compute unit and up to 256 x 128 fp32 products of each: 32 MiB)
        if (!ctx->gemm_parts) (void)grow_parts(ctx, (size_t)ctx->compute_units * 256 * 128 * 4);
    }
    *out = (uint8_t*)ctx->gemm_ws;
    return SKN_OK;
}

float* skn_gemm_parts_room(skn_ctx* ctx, size_t bytes) {
    if (ctx->opt_test_gemm_no_parts) return nullptr;
    // (without a workspace yet, as under test or where that found no memory: what it would have brought)
    const size_t least = ctx->gemm_parts ? 0 : (size_t)ctx->compute_units * 256 * 128 * 4;
    if (bytes > ctx->gemm_parts_bytes && !grow_parts(ctx, std::max(bytes, least))) return nullptr;
    return (float*)ctx->gemm_parts;
}

// Dynamic LDS above 48 KiB must be allowed per kernel and device; done once per context here so that no launch
// path has to.
static int skn_gemm_init(skn_ctx* ctx) {
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_q4k_frag_kernel<2, 2, false>, hipFuncAttributeMaxDynamicSharedMemorySize, frag_lds_bytes<2, 2>() + 32 * 2 * 2 * 4));
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_q4k_frag_kernel<2, 2, true>, hipFuncAttributeMaxDynamicSharedMemorySize, frag_lds_bytes<2, 2>() + 32 * 2 * 2 * 4));
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_q4k_frag_kernel<2, 1, false>, hipFuncAttributeMaxDynamicSharedMemorySize, frag_lds_bytes<2, 1>() + 32 * 2 * 1 * 4));
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_q4k_frag_kernel<2, 1, true>, hipFuncAttributeMaxDynamicSharedMemorySize, frag_lds_bytes<2, 1>() + 32 * 2 * 1 * 4));
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_q4k_tall_kernel<false, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, kTlLds));
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_q4k_tall_kernel<true, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, kTlLds));
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_q4k_tall_kernel<false, 3>, hipFuncAttributeMaxDynamicSharedMemorySize, kTlLds));
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_hilo_frag_kernel<1, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * 1 * 3 * 4096));
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_hilo_frag_kernel<2, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * 2 * 3 * 4096));
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_hilo_frag_kernel<4, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * 4 * 3 * 4096));
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_q6k_tall_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kQ6TlLds));
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_q6k_pc_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize, kQ6PcLds));
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_q6k_pc_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, kQ6PcLds));
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_q6k_frag_kernel<1, false>, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * 1 * 3 * 4096));
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_q6k_frag_kernel<1, true>, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * 1 * 3 * 4096));
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_q6k_frag_kernel<2, false>, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * 2 * 3 * 4096));
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_q6k_frag_kernel<2, true>, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * 2 * 3 * 4096));
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_q6k_frag_kernel<4, false>, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * 4 * 3 * 4096));
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_q6k_frag_kernel<4, true>, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * 4 * 3 * 4096));
    return SKN_OK;
}
static skn_family register_family(skn_gemm_init);

// The tiles past the last whole round of compute units: shared where at least two workgroups each find room in that round.
static TallTail tall_tail(const skn_ctx* ctx, int tiles, int nb) {
    const int cus = ctx->compute_units, rest = tiles % cus;
    TallTail t = {tiles, 0, 1, nullptr};
    int splits = rest ? std::min(cus / rest, nb / 4) : 1;
    if (ctx->opt_gemm_split > 0) splits = std::min(ctx->opt_gemm_split, nb);
    if (rest == 0 || splits < 2) return t;
    return TallTail{tiles - rest, rest, splits, nullptr};
}

// The same for the Q4_K kernel of 64- and 128-row tiles, whose step along k is short: only where the steps saved (a group of
// four superblocks each: 1.9 us on 64 rows, 3.4 us on 128) pay for the second launch, which costs as much as one of them, and for
// the parts' way through memory (0.6 us per MB; `cols` of all the launch's matrices).  Fitted to 290 shapes of 33 to 1024 rows, 256 to
// 11008 columns and k from 1536 to 11008.  us per call, unsplit | split: 200 x 4096 x 2048 17.3 | 20.1, 512 x 2048 x 2048 19.0 | 24.4,
// 64 x 8192 x 2048 13.3 | 15.4, all three unsplit; 512 x 512 x 4096 27.0 | 20.4, 200 x 4096 x 6144 35.6 | 31.5, both split.
static int q4k_splits(const skn_ctx* ctx, int m, int tile_rows, int tiles, int nb, int cols) {
    const int splits = skn_gemm_k_splits(ctx, m, tiles, nb);
    if (splits < 2 || ctx->opt_gemm_split > 0) return splits;
    const int each = (nb + splits - 1) / splits, saved = (nb + 3) / 4 - (each + 3) / 4;
    const double gain_us = (tile_rows == 64 ? 1.9 : 3.4) * (saved - 1);
    return gain_us > 0.6e-6 * 4.0 * splits * m * cols ? splits : 1;
}

int skn_gemm_q4k_multi(skn_ctx* ctx, const skn_gemm_seg* segs, int nseg, int k, const skn_gemm_src& src, int m,
                       uint16_t* swiglu_pair) {
    SKN_REQUIRE(ctx, nseg >= 1 && nseg <= 3 && m > 0 && k > 0 && k % 256 == 0 && k <= 16384, SKN_ERR_ARG,
                "Q4_K GEMM: bad segment count or shape");
    SKN_REQUIRE(ctx, !swiglu_pair || (nseg == 2 && segs[0].n == segs[1].n && !segs[0].accumulate), SKN_ERR_ARG,
                "Q4_K GEMM: a SwiGLU pair is two matrices of the same shape");
    Q4kFragSegs fs = {};
    int tiles = 0;
    for (int i = 0; i < 3; i++) {
        const skn_gemm_seg& s = segs[i < nseg ? i : nseg - 1];
        SKN_REQUIRE(ctx, s.w && (s.c || swiglu_pair) && s.n > 0 && ((uintptr_t)s.w & 15) == 0, SKN_ERR_ARG,
                    "Q4_K GEMM: weights must be non-null and 16-byte aligned");
        fs.w[i] = (const uint8_t*)s.w, fs.c[i] = s.c, fs.n[i] = s.n, fs.accumulate[i] = s.accumulate, fs.tile0[i] = tiles;
        if (i < nseg) tiles += (s.n + kBN - 1) / kBN;
    }
    for (int i = nseg; i < 3; i++) fs.tile0[i] = tiles;
    fs.n_tiles = swiglu_pair ? (segs[0].n + 31) / 32 : tiles;
    fs.pair = swiglu_pair;
    SKN_REQUIRE(ctx, src.a && ((uintptr_t)src.a & (src.kind == SKN_SRC_BF16 ? 7 : 15)) == 0, SKN_ERR_ARG,
                "Q4_K GEMM: activations are null or misaligned");
    SKN_REQUIRE(ctx, src.kind == SKN_SRC_BF16 || src.kind == SKN_SRC_F32 || (src.b && ((uintptr_t)src.b & 15) == 0),
                SKN_ERR_ARG, "Q4_K GEMM: second activation operand is null or misaligned");
    // fragment-order workspace: rows padded to whole tiles
    // Tile rows: 128 (eight wavefronts, one workgroup per compute unit) when that gives at most one tile per
    // compute unit; otherwise 64 with four wavefronts, two independent workgroups per compute unit -- more weight
    // staging per product, but the two wavefronts of a SIMD no longer meet at the same barriers (measured 4-11 %
    // faster on grids of several rounds, 3 % slower on single-round grids).
    const int n_tiles_all = fs.n_tiles;
    // 256 x 128 tiles (the kernel that unpacks the weights once per tile) where they keep at least two thirds of the
    // compute units busy over their rounds: the 14336-column matrices, a q,k,v group and a gate / up pair at 512 rows
    int tall_cols = 0, tall_tile0[3] = {0, 0, 0}, blocks = 0, block0[3] = {0, 0, 0};
    bool tall_fits = true;
    for (int i = 0; i < nseg; i++) {
        tall_tile0[i] = tall_cols, block0[i] = blocks;
        tall_cols += (segs[i].n + 127) / 128, blocks += (segs[i].n + 31) / 32;
        tall_fits = tall_fits && (size_t)segs[i].n * (k / 256) * 144 < ((size_t)1 << 31);
    }
    for (int i = nseg; i < 3; i++) tall_tile0[i] = tall_cols, block0[i] = blocks;
    if (swiglu_pair) tall_cols = (segs[0].n + 63) / 64;
    const int tall_tiles = ((m + 255) / 256) * tall_cols;
    const int tall_rounds = (tall_tiles + ctx->compute_units - 1) / ctx->compute_units;
    const bool tall = tall_fits && (ctx->opt_gemm_tile == 3 || (ctx->opt_gemm_tile == 4 && !swiglu_pair) ||
                                    (ctx->opt_gemm_tile == 0 && m > 128 && 3 * tall_tiles >= 2 * tall_rounds * ctx->compute_units));
    TallTail tail = {tall_tiles, 0, 1, nullptr};
    if (tall) tail = tall_tail(ctx, tall_tiles, k / 256);
    // 96 columns where their rounds, at 0.85 of the time of one of 128 columns, are the shorter: one round where 128 columns leave a quarter and more of
    // it idle, and with rows of less than eight superblocks two against two, three against three or seven against six (us of 128 | of 96: 1024 x 11264 x 1024
    // 47.8 | 42.6, 1024 x 12288 x 512 35.1 | 31.2, 768 x 24000 x 1536 92.0 | 81.0, 2048 x 20608 x 1792 201 | 192; three against two, not taken: 700 x 16384 x
    // 1024 47.9 | 56.1).  Only what has no last tiles to share (their sums' chains would grow).
    const int narrow_tiles = ((m + 255) / 256) * ((blocks + 2) / 3), narrow_rounds = (narrow_tiles + ctx->compute_units - 1) / ctx->compute_units;
    const bool narrow = tall && !swiglu_pair && (ctx->opt_gemm_tile == 4 || (ctx->opt_gemm_tile == 0 && tail.tiles == 0 && 17 * narrow_rounds < 20 * tall_rounds));
    if (narrow) tail = TallTail{narrow_tiles, 0, 1, nullptr};
    const bool small_tiles = !tall && (ctx->opt_gemm_tile == 1 ||
                             (ctx->opt_gemm_tile == 0 && (m <= 128 || ((m + 127) / 128) * n_tiles_all > ctx->compute_units)));
    const int mt_rows = tall ? 256 : small_tiles ? 64 : 128;
    const int m_tiles = (m + mt_rows - 1) / mt_rows, m_pad = m_tiles * mt_rows;
    const size_t af_bytes = skn_align_up((size_t)m_pad * k * 2), sf_bytes = skn_align_up((size_t)m_pad * (k / 256) * 16 * 2);
    SKN_REQUIRE(ctx, af_bytes < ((size_t)1 << 31), SKN_ERR_SHAPE,
                "Q4_K GEMM: %d rows of %d activations exceed the 2^30 elements one call takes", m, k);
    const size_t is_bytes = skn_align_up((size_t)m_pad * 4);
    skn_gemm_parts ps = {};
    ps.count = nseg, ps.pair = fs.pair;
    for (int i = 0; i < nseg; i++) {
        ps.c[i] = segs[i].c, ps.n[i] = segs[i].n, ps.accumulate[i] = segs[i].accumulate;
        ps.col0[i] = fs.part_cols;
        fs.part_cols += segs[i].n;
    }
    for (int i = 0; i < 3; i++) fs.part_col0[i] = ps.col0[i];
    int splits = tall ? 1 : q4k_splits(ctx, m, mt_rows, m_tiles * fs.n_tiles, k / 256, fs.part_cols);
    uint8_t* ws;
    const size_t most_rows = skn_tall_rows(m), most = skn_align_up(most_rows * k * 2) + skn_align_up(most_rows * (k / 256) * 16 * 2) + skn_align_up(most_rows * 4);
    int rc = skn_gemm_workspace(ctx, af_bytes + sf_bytes + is_bytes, most, &ws, src.ahead);
    if (rc != SKN_OK) return rc;
    const size_t part_bytes = tall ? (size_t)tail.tiles * tail.splits * 131072 : splits > 1 ? (size_t)splits * m * fs.part_cols * 4 : 0;
    float* part = part_bytes ? skn_gemm_parts_room(ctx, part_bytes) : nullptr;
    if (src.ahead) return SKN_OK;
    if (!part) splits = 1, tail = TallTail{narrow ? narrow_tiles : tall_tiles, 0, 1, nullptr};
    fs.part_blocks = (k / 256 + splits - 1) / splits;
    if (splits > 1) fs.part = part;
    _Float16* afrag = (_Float16*)ws;
    _Float16* sfrag = (_Float16*)(ws + af_bytes);
    float* isc = (float*)(ws + af_bytes + sf_bytes);
    switch (src.kind) {
        case SKN_SRC_BF16: launch_prep<SKN_SRC_BF16, true>(ctx, src, afrag, isc, sfrag, m, m_pad, k); break;
        case SKN_SRC_F32: launch_prep<SKN_SRC_F32, true>(ctx, src, afrag, isc, sfrag, m, m_pad, k); break;
        case SKN_SRC_RMSNORM: launch_prep<SKN_SRC_RMSNORM, true>(ctx, src, afrag, isc, sfrag, m, m_pad, k); break;
        default: return skn_fail(ctx, SKN_ERR_ARG, "Q4_K GEMM: unknown activation source %d", src.kind);
    }
    SKN_LAUNCH_CHECK(ctx);
    if (tall) {
        for (int i = 0; i < 3; i++) fs.tile0[i] = narrow ? block0[i] : tall_tile0[i];
        fs.n_tiles = narrow ? blocks : tall_cols;
        tail.part = part;
        skn_launch(ctx, narrow ? gemm_q4k_tall_kernel<false, 3> : tail.tiles ? gemm_q4k_tall_kernel<true, 4> : gemm_q4k_tall_kernel<false, 4>, dim3(tail.tile0 + tail.tiles * tail.splits), dim3(512), kTlLds, (const u32x4*)afrag, (const u32x4*)sfrag, fs,
                   (const float*)isc, m, k, m_tiles, (uint32_t)((size_t)m_pad * k * 2), tail);
        SKN_LAUNCH_CHECK(ctx);
        if (tail.tiles) {
            skn_launch(ctx, gemm_add_tall_kernel, dim3(tail.tiles, 8), dim3(256), 0, tail, fs, (const float*)isc, m, m_tiles);
            SKN_LAUNCH_CHECK(ctx);
        }
        return SKN_OK;
    }
    if (mt_rows == 128) SKN_TRY((launch_frag<2, 2>(ctx, m_tiles, (const u32x4*)afrag, (const u32x4*)sfrag, fs, isc, m, k, splits)));
    else SKN_TRY((launch_frag<2, 1>(ctx, m_tiles, (const u32x4*)afrag, (const u32x4*)sfrag, fs, isc, m, k, splits)));
    return splits > 1 ? skn_gemm_add_parts(ctx, fs.part, splits, fs.part_cols, ps, isc, m) : SKN_OK;
}

// The product in a pass over the activations, one over the tiles and, where k is divided, one over the parts (and a pass over the
// weights, in the general path).
static int gemm_in_passes(skn_ctx* ctx, int ggml_type, const void* w_dev, int n, int k, const skn_gemm_src& src, int m, float* c_dev) {
    if (ggml_type == SKN_TYPE_Q4_K && k <= 16384) {
        SKN_REQUIRE(ctx, ((uintptr_t)w_dev & 15) == 0 && ((uintptr_t)src.a & 7) == 0, SKN_ERR_ARG,
                    "skn_gemm_q: Q4_K weights must be 16-byte aligned, activations 8-byte aligned");
        const skn_gemm_seg seg = {w_dev, n, c_dev, 0};
        // up to 32 rows (17 to 32 of matrices too large for the path above): the kernel for blocks of 32, whose tile has as many (us per
        // call, this | that: 17 x 14336 x 4096 20.1 | 19.0, 17 x 8192 x 11008 30.3 | 27.9, 32 x 28672 x 4096 28.5 | 26.4, 32 x 11008 x 8192
        // 29.5 | 29.3; on two row blocks 41 x 4096 x 4096 15.2 | 14.9, 64 x 11008 x 4096 20.1 | 23.8)
        if (ctx->opt_gemm_tile == 0 && m <= 32 && skn_gemm_blocks_ok(ctx, ggml_type, w_dev, n, k, m))
            return skn_gemm_blocks_multi(ctx, &ggml_type, &seg, 1, k, src, m);
        return skn_gemm_q4k_multi(ctx, &seg, 1, k, src, m);
    }

    // general path.  Workspace: activations in fragment order (rows padded to whole tiles) + row scales, then
    // the weights as an fp16 pair in fragment order (rows padded to whole 64-column tiles)
    SKN_REQUIRE(ctx, ((uintptr_t)src.a & 7) == 0, SKN_ERR_ARG, "skn_gemm_q: activations must be 8-byte aligned");
    // Q6_K with whole superblocks: the kernels that unpack the blocks themselves (no weight pass, no expanded copy)
    if (ggml_type == SKN_TYPE_Q6_K && skn_gemm_q6k_direct_ok(ctx, n, k, m)) {
        const skn_gemm_seg seg = {w_dev, n, c_dev, 0};
        return skn_gemm_q6k_multi(ctx, &seg, 1, k, src, m);
    }
    // formats in blocks of 32: likewise
    if (skn_gemm_blocks_ok(ctx, ggml_type, w_dev, n, k, m) && skn_gemm_blocks_pay(ggml_type, n, k, m, false)) {
        const skn_gemm_seg seg = {w_dev, n, c_dev, 0};
        return skn_gemm_blocks_multi(ctx, &ggml_type, &seg, 1, k, src, m);
    }
    if (src.ahead) return SKN_OK;  // (no product of few rows has a format or a size that would come here)
    const int mt = skn_gemm_mt(m);
    const int m_pad = (m + 32 * mt - 1) / (32 * mt) * (32 * mt), n_pad = (n + kBN - 1) / kBN * kBN;
    const size_t af_bytes = skn_align_up((size_t)m_pad * k * 2), is_bytes = skn_align_up((size_t)m_pad * 4);
    uint8_t* ws;
    const size_t bytes = af_bytes + is_bytes + (size_t)n_pad * k * 4;
    int rc = skn_gemm_workspace(ctx, bytes, bytes, &ws);
    if (rc != SKN_OK) return rc;
    _Float16* afrag = (_Float16*)ws;
    float* isc = (float*)(ws + af_bytes);
    uint8_t* bfrag = ws + af_bytes + is_bytes;
    _Float16* no_sums = nullptr;
    launch_prep<SKN_SRC_BF16, false>(ctx, src, afrag, isc, no_sums, m, m_pad, k);
    SKN_LAUNCH_CHECK(ctx);
    rc = skn_weights_hilo_frag(ctx, ggml_type, (const uint8_t*)w_dev, n, k, bfrag);
    if (rc != SKN_OK) return rc;
    return launch_hilo_gemm_mt(ctx, mt, (const u32x4*)afrag, (const u32x4*)bfrag, isc, c_dev, m, n, k, 0);
}

extern "C" int skn_gemm_q(skn_ctx* ctx, int ggml_type, const void* w_dev, int n, int k, const uint16_t* a_bf16_dev,
                          int m, float* c_dev) {
    SKN_REQUIRE(nullptr, ctx != nullptr, SKN_ERR_ARG, "skn_gemm_q: ctx is null");
    SKN_REQUIRE(ctx, skn_is_quant(ggml_type), SKN_ERR_TYPE, "skn_gemm_q: ggml type %d is not supported", ggml_type);
    SKN_REQUIRE(ctx, n >= 0 && k >= 0 && m >= 0, SKN_ERR_ARG, "skn_gemm_q: negative shape");
    int be, bb;
    skn_type_block(ggml_type, &be, &bb);
    SKN_REQUIRE(ctx, k % be == 0, SKN_ERR_SHAPE, "Quantized tensor row size (%d) is not a multiple of block size (%d)", k,
                be);
    if (n == 0 || m == 0) return SKN_OK;
    SKN_REQUIRE(ctx, c_dev != nullptr, SKN_ERR_ARG, "skn_gemm_q: c is null");
    if (k == 0) return skn_memset(ctx, c_dev, 0, (size_t)m * n * sizeof(float));
    SKN_REQUIRE(ctx, w_dev && a_bf16_dev, SKN_ERR_ARG, "skn_gemm_q: null pointer");
    SKN_REQUIRE(ctx, k % 64 == 0, SKN_ERR_SHAPE, "skn_gemm_q: k (%d) must be a multiple of %d", k, 64);

    // Few rows: one launch instead of three.  The memory that the three would take is asked for all the same: a caller that captures
    // its calls runs one of the same activations first, and one of more columns may not be of few rows.
    if (((uintptr_t)a_bf16_dev & 7) == 0 && skn_gemm_few_ok(ctx, ggml_type, w_dev, n, k, m)) {
        (void)gemm_in_passes(ctx, ggml_type, w_dev, n, k, skn_gemm_src{SKN_SRC_BF16, a_bf16_dev, nullptr, 0.f, true}, m, c_dev);
        return skn_gemm_few(ctx, ggml_type, w_dev, n, k, a_bf16_dev, m, c_dev);
    }
    return gemm_in_passes(ctx, ggml_type, w_dev, n, k, skn_gemm_src{SKN_SRC_BF16, a_bf16_dev, nullptr, 0.f}, m, c_dev);
}

namespace {
// 256 x 128 tiles for a Q6_K matrix: where they fill three quarters of the compute units or more in one round (or by option)
bool q6k_wide_tiles(const skn_ctx* ctx, int n, int k, int m) {
    const int tiles = ((m + 255) / 256) * ((n + 127) / 128);
    return k <= 16384 && ctx->opt_gemm_q6k_fused == 1 &&
           (ctx->opt_gemm_tile == 3 ||
            (ctx->opt_gemm_tile == 0 && m > 128 && 4 * tiles >= 3 * ctx->compute_units && tiles <= ctx->compute_units));
}
}  // namespace

bool skn_gemm_q6k_direct_ok(const skn_ctx* ctx, int n, int k, int m) {
    const size_t m_pad = ((size_t)m + 255) / 256 * 256;
    return ctx->opt_gemm_q6k_fused != 0 && n > 0 && m > 0 && k > 0 && k % 256 == 0 && m_pad * k * 2 + 256 < ((size_t)1 << 31) &&
           (size_t)n * (k / 256) * 210 < ((size_t)1 << 31);
}

// How many workgroups share the k of a tile of `rows` rows.  The column tiles go round the eight XCDs and their row tiles with them
// (launch_q6k_gemm), so the fullest XCD decides: parts that need a second round of its compute units are walked one behind the other.
// us per call, undivided | in two parts: 380 x 2688 x 4096 (eighteen tiles on an XCD of 32 units) 55.0 | 60.6, 600 x 1600 x 11008 (twenty) 139 | 151,
// 1300 x 700 x 11008 (22) 148 | 161, against 380 x 2560 x 8192 (fifteen) 92.6 | 60.3 and 1300 x 512 x 11008 (eleven) 150 | 97; three parts
// in two rounds gain: 1800 x 300 x 11008 154 | 127.
static int q6k_splits(const skn_ctx* ctx, int m, int n, int rows, int nb) {
    const int m_tiles = (m + rows - 1) / rows, n_tiles = (n + kBN - 1) / kBN, splits = skn_gemm_k_splits(ctx, m, m_tiles * n_tiles, nb);
    if (splits < 2 || ctx->opt_gemm_split > 0) return splits;
    const int on_xcd = 8 % m_tiles == 0 ? (n_tiles * m_tiles + 7) / 8 : (n_tiles + 7) / 8 * m_tiles, units = std::max(1, ctx->compute_units / 8);
    const int each = (nb + splits - 1) / splits;
    return (on_xcd * splits + units - 1) / units * each < (on_xcd + units - 1) / units * nb ? splits : 1;
}

int skn_gemm_q6k_multi(skn_ctx* ctx, const skn_gemm_seg* segs, int nseg, int k, const skn_gemm_src& src, int m) {
    SKN_REQUIRE(ctx, nseg >= 1 && nseg <= 3 && m > 0, SKN_ERR_ARG, "Q6_K GEMM: bad segment count or shape");
    SKN_REQUIRE(ctx, src.a && ((uintptr_t)src.a & (src.kind == SKN_SRC_BF16 ? 7 : 15)) == 0, SKN_ERR_ARG,
                "Q6_K GEMM: activations are null or misaligned");
    SKN_REQUIRE(ctx, src.kind == SKN_SRC_BF16 || src.kind == SKN_SRC_F32 || (src.b && ((uintptr_t)src.b & 15) == 0),
                SKN_ERR_ARG, "Q6_K GEMM: second activation operand is null or misaligned");
    bool any_wide = false;
    for (int i = 0; i < nseg; i++) {
        SKN_REQUIRE(ctx, segs[i].w && segs[i].c && skn_gemm_q6k_direct_ok(ctx, segs[i].n, k, m), SKN_ERR_ARG,
                    "Q6_K GEMM: a matrix is null or not one this path takes");
        any_wide = any_wide || q6k_wide_tiles(ctx, segs[i].n, k, m);
    }
    // (rows padded to the tallest tile in use: the kernels with shorter tiles address their own row blocks inside it)
    const int mt = skn_gemm_mt(m);
    const int m_rows = any_wide ? 256 : 32 * mt;
    const int m_pad = (m + m_rows - 1) / m_rows * m_rows;
    const size_t af_bytes = skn_align_up((size_t)m_pad * k * 2), is_bytes = skn_align_up((size_t)m_pad * 4);
    int splits[3] = {1, 1, 1};
    size_t part_bytes = 0;  // (the matrices' products run one after the other: they share the room for their parts)
    for (int i = 0; i < nseg; i++) {
        if (q6k_wide_tiles(ctx, segs[i].n, k, m)) continue;
        splits[i] = q6k_splits(ctx, m, segs[i].n, 32 * mt, k / 256);
        if (splits[i] > 1) part_bytes = std::max(part_bytes, (size_t)splits[i] * m * segs[i].n * 4);
    }
    uint8_t* ws;
    const size_t most_rows = skn_tall_rows(m);
    int rc = skn_gemm_workspace(ctx, af_bytes + is_bytes, skn_align_up(most_rows * k * 2) + skn_align_up(most_rows * 4), &ws, src.ahead);
    if (rc != SKN_OK) return rc;
    _Float16* afrag = (_Float16*)ws;
    float* isc = (float*)(ws + af_bytes);
    float* part = part_bytes ? skn_gemm_parts_room(ctx, part_bytes) : nullptr;
    if (src.ahead) return SKN_OK;
    if (!part) splits[0] = splits[1] = splits[2] = 1;
    _Float16* no_sums = nullptr;
    switch (src.kind) {
        case SKN_SRC_BF16: launch_prep<SKN_SRC_BF16, false>(ctx, src, afrag, isc, no_sums, m, m_pad, k); break;
        case SKN_SRC_F32: launch_prep<SKN_SRC_F32, false>(ctx, src, afrag, isc, no_sums, m, m_pad, k); break;
        case SKN_SRC_RMSNORM: launch_prep<SKN_SRC_RMSNORM, false>(ctx, src, afrag, isc, no_sums, m, m_pad, k); break;
        default: return skn_fail(ctx, SKN_ERR_ARG, "Q6_K GEMM: unknown activation source %d", src.kind);
    }
    SKN_LAUNCH_CHECK(ctx);
    for (int i = 0; i < nseg; i++) {
        const int n = segs[i].n;
        if (q6k_wide_tiles(ctx, n, k, m)) {
            const int m_tiles = m_pad / 256, tiles = m_tiles * ((n + 127) / 128);
            skn_launch(ctx, gemm_q6k_tall_kernel, dim3((unsigned)tiles), dim3(512), kQ6TlLds, (const u32x4*)afrag, (const uint8_t*)segs[i].w,
                       (const float*)isc, segs[i].c, m, n, k, m_tiles, segs[i].accumulate, (uint32_t)((size_t)m_pad * k * 2),
                       (uint32_t)((size_t)n * (k / 256) * 210));
            SKN_LAUNCH_CHECK(ctx);
        } else {
            rc = launch_q6k_gemm_mt(ctx, mt, (const u32x4*)afrag, (const uint8_t*)segs[i].w, isc, segs[i].c, m, n, k, segs[i].accumulate, splits[i], part);
            if (rc != SKN_OK) return rc;
        }
    }
    return SKN_OK;
}

// ---- expanded weights: the general path with its weight pass done once ------------------------------------
// The fp16-pair copy of a weight matrix that the general path builds per call (4 bytes per weight, rows padded to
// whole 64-column tiles) can be kept by the caller: skn_gemm_expand fills it, skn_gemm_expanded multiplies with it.

size_t skn_gemm_expanded_size(int n, int k) { return (size_t)((n + kBN - 1) / kBN * kBN) * (size_t)k * 4; }

int skn_gemm_expanded_multi(skn_ctx* ctx, const skn_gemm_seg* segs, int nseg, int k, const skn_gemm_src& src, int m) {
    SKN_REQUIRE(ctx, nseg >= 1 && m > 0 && k > 0 && k % 64 == 0, SKN_ERR_ARG, "expanded GEMM: bad segment count or shape");
    SKN_REQUIRE(ctx, src.a && ((uintptr_t)src.a & (src.kind == SKN_SRC_BF16 ? 7 : 15)) == 0, SKN_ERR_ARG,
                "expanded GEMM: activations are null or misaligned");
    SKN_REQUIRE(ctx, src.kind == SKN_SRC_BF16 || src.kind == SKN_SRC_F32 || (src.b && ((uintptr_t)src.b & 15) == 0),
                SKN_ERR_ARG, "expanded GEMM: second activation operand is null or misaligned");
    for (int i = 0; i < nseg; i++)
        SKN_REQUIRE(ctx, segs[i].w && segs[i].c && segs[i].n > 0 && ((uintptr_t)segs[i].w & 15) == 0, SKN_ERR_ARG,
                    "expanded GEMM: weights must be non-null and 16-byte aligned");
    const int mt = skn_gemm_mt(m);
    const int m_pad = (m + 32 * mt - 1) / (32 * mt) * (32 * mt);
    const size_t af_bytes = skn_align_up((size_t)m_pad * k * 2), is_bytes = skn_align_up((size_t)m_pad * 4);
    SKN_REQUIRE(ctx, af_bytes < ((size_t)1 << 31), SKN_ERR_SHAPE,
                "expanded GEMM: %d rows of %d activations exceed the 2^30 elements one call takes", m, k);
    uint8_t* ws;
    int rc = skn_gemm_workspace(ctx, af_bytes + is_bytes, af_bytes + is_bytes, &ws);
    if (rc != SKN_OK) return rc;
    _Float16* afrag = (_Float16*)ws;
    float* isc = (float*)(ws + af_bytes);
    _Float16* no_sums = nullptr;
    switch (src.kind) {
        case SKN_SRC_BF16: launch_prep<SKN_SRC_BF16, false>(ctx, src, afrag, isc, no_sums, m, m_pad, k); break;
        case SKN_SRC_F32: launch_prep<SKN_SRC_F32, false>(ctx, src, afrag, isc, no_sums, m, m_pad, k); break;
        case SKN_SRC_RMSNORM: launch_prep<SKN_SRC_RMSNORM, false>(ctx, src, afrag, isc, no_sums, m, m_pad, k); break;
        default: return skn_fail(ctx, SKN_ERR_ARG, "expanded GEMM: unknown activation source %d", src.kind);
    }
    SKN_LAUNCH_CHECK(ctx);
    for (int i = 0; i < nseg; i++) {
        rc = launch_hilo_gemm_mt(ctx, mt, (const u32x4*)afrag, (const u32x4*)segs[i].w, isc, segs[i].c, m, segs[i].n, k,
                                 segs[i].accumulate);
        if (rc != SKN_OK) return rc;
    }
    return SKN_OK;
}

extern "C" int skn_gemm_expanded_bytes(skn_ctx* ctx, int ggml_type, int n, int k, size_t* bytes_out) {
    SKN_REQUIRE(nullptr, ctx != nullptr, SKN_ERR_ARG, "skn_gemm_expanded_bytes: ctx is null");
    SKN_REQUIRE(ctx, bytes_out != nullptr, SKN_ERR_ARG, "skn_gemm_expanded_bytes: bytes_out is null");
    SKN_REQUIRE(ctx, skn_is_quant(ggml_type), SKN_ERR_TYPE, "skn_gemm_expanded_bytes: ggml type %d is not supported", ggml_type);
    SKN_REQUIRE(ctx, n >= 0 && k >= 0, SKN_ERR_ARG, "skn_gemm_expanded_bytes: negative shape");
    int be, bb;
    skn_type_block(ggml_type, &be, &bb);
    SKN_REQUIRE(ctx, k % be == 0, SKN_ERR_SHAPE, "Quantized tensor row size (%d) is not a multiple of block size (%d)", k,
                be);
    SKN_REQUIRE(ctx, k % 64 == 0, SKN_ERR_SHAPE, "skn_gemm_expanded_bytes: k (%d) must be a multiple of %d", k, 64);
    *bytes_out = skn_gemm_expanded_size(n, k);
    return SKN_OK;
}

extern "C" int skn_gemm_expand(skn_ctx* ctx, int ggml_type, const void* w_dev, int n, int k, void* expanded_dev) {
    SKN_REQUIRE(nullptr, ctx != nullptr, SKN_ERR_ARG, "skn_gemm_expand: ctx is null");
    size_t bytes = 0;
    int rc = skn_gemm_expanded_bytes(ctx, ggml_type, n, k, &bytes);
    if (rc != SKN_OK) return rc;
    if (bytes == 0) return SKN_OK;
    SKN_REQUIRE(ctx, w_dev && expanded_dev, SKN_ERR_ARG, "skn_gemm_expand: null pointer");
    SKN_REQUIRE(ctx, ((uintptr_t)expanded_dev & 15) == 0, SKN_ERR_ARG, "skn_gemm_expand: the copy must be 16-byte aligned");
    return skn_weights_hilo_frag(ctx, ggml_type, (const uint8_t*)w_dev, n, k, expanded_dev);
}

extern "C" int skn_gemm_expanded(skn_ctx* ctx, const void* expanded_dev, int n, int k, const uint16_t* a_bf16_dev, int m,
                                 float* c_dev) {
    SKN_REQUIRE(nullptr, ctx != nullptr, SKN_ERR_ARG, "skn_gemm_expanded: ctx is null");
    SKN_REQUIRE(ctx, n >= 0 && k >= 0 && m >= 0, SKN_ERR_ARG, "skn_gemm_expanded: negative shape");
    SKN_REQUIRE(ctx, k % 64 == 0, SKN_ERR_SHAPE, "skn_gemm_expanded: k (%d) must be a multiple of %d", k, 64);
    if (n == 0 || m == 0) return SKN_OK;
    SKN_REQUIRE(ctx, c_dev != nullptr, SKN_ERR_ARG, "skn_gemm_expanded: c is null");
    if (k == 0) return skn_memset(ctx, c_dev, 0, (size_t)m * n * sizeof(float));
    SKN_REQUIRE(ctx, expanded_dev && a_bf16_dev, SKN_ERR_ARG, "skn_gemm_expanded: null pointer");
    const skn_gemm_seg seg = {expanded_dev, n, c_dev, 0};
    const skn_gemm_src src = {SKN_SRC_BF16, a_bf16_dev, nullptr, 0.f};
    return skn_gemm_expanded_multi(ctx, &seg, 1, k, src, m);
}
