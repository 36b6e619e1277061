// Prompt GEMM for formats whose weights are d (q - zero) + m over blocks of 32 elements: Q8_0, Q4_0, Q4_1, Q5_0, Q5_1, the
// sub-blocks of Q5_K, and those of Q4_K for up to 32 rows (above, Q4_K has kernels of its own in gemm.hip; few rows of
// matrices that are not too large go to gemm_few.hip).
// C[m, n] = sum_k A[m, k] w[n, k], activations as in gemm.hip (bf16 rows scaled to fp16 by a power of two).
//
// Bound by the matrix cores and the vector ALUs together for many rows, by the weight stream for few.  What the general path
// does with these formats -- rewrite the weights as fp16 pairs (4 bytes per weight written and read again), then two matrix
// instructions per k-step -- is replaced by one launch that reads the blocks: q - zero is a whole number of at most 8 bits,
// exact in fp16, so a block is two matrix instructions (k = 16 each) from zero, and its sum joins the tile's total in fp32,
// times the block's scale (one fused multiply-add per element and block of 32; the lane's column fixes the scale).  Nothing is
// rounded before those sums.  Minima: sum over a superblock of m_j times the sum of the activations of block j, one more matrix
// instruction on the sums that the preparation pass leaves (fp16 pairs).
//
// Workgroup of four wavefronts, one per SIMD, tile (32 MT) x 64 (MT = 1 up to 32 rows, 2 above; in a range of sizes another kernel's 96 x 64, below), k by superblock (256 elements)
// over the wavefronts and, where the tiles do not fill the device, over workgroups too (gemm_tiles.h); the four partial tiles are
// added through LDS.  A wavefront brings its superblock of 64 rows in with coalesced 16-byte loads one superblock ahead
// (registers, then LDS of its own: no barrier in the loop) and reads the activations in fragment order, four k-steps ahead.
//
// us per call, before -> now (weights as fp16 pairs -> this): Q8_0 333 x 4096 x 4096 51.6 -> 32.1, 512 x 14336 x 4096 236 -> 115, 41 x 4096 x
// 11008 102 -> 28.5; Q5_K 512 x 4096 x 4096 60 -> 39.2; Q4_0 5 x 4096 x 4096 36.6 -> 11.5.
#include "gemm_blocks.h"
#include "gemm_rows.h"
#include "gemm_tiles.h"

#include <algorithm>
#include <type_traits>

namespace {

// ---- activations ----------------------------------------------------------------------------------------------------------
// Block order: for a block of 32 rows, a block of 32 elements and a k-step s, lane 32 h + r of a matrix instruction's operand
// holds elements 16 h + 8 s .. + 7 of row r, so that a lane's two k-steps of a weight block are sixteen consecutive quants.
// One workgroup per row (few rows are what the pass is slow for), the row in registers.  sfrag as in gemm.hip.
template <int NT, int SRC, bool SUMS>
__global__ __launch_bounds__(256) void prep_blocks_kernel(const skn_gemm_src src, u32x4* __restrict__ afrag, float* __restrict__ inv_scale,
                                                         _Float16* __restrict__ sfrag, int m, int k) {
    __shared__ float red[8];
    const int tid = threadIdx.x, bid = blockIdx.x;
    // eight neighbouring rows, whose sixteen-byte pieces share 128-byte lines, go to workgroups of one XCD (blockIdx % 8)
    const int row = (bid | 63) < (int)gridDim.x ? (bid & ~63) + (bid & 7) * 8 + ((bid >> 3) & 7) : bid;
    const bool real = row < m;
    const int pieces = k >> 3;
    const size_t off = (size_t)(real ? row : 0) * k;
    float v[NT][8];
    float4 g0[SRC == SKN_SRC_RMSNORM ? NT : 1], g1[SRC == SKN_SRC_RMSNORM ? NT : 1];  // (asked for with the row)
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const int p = min(tid + 256 * j, pieces - 1);
        if constexpr (SRC == SKN_SRC_RMSNORM) {
            const float4* g = reinterpret_cast<const float4*>((const float*)src.b + 8 * p);
            g0[j] = g[0], g1[j] = g[1];
        }
        if (SRC == SKN_SRC_BF16) {
            const u32x2* x = reinterpret_cast<const u32x2*>((const uint16_t*)src.a + off + 8 * p);
            const u32x2 a = x[0], b = x[1];
            const uint32_t w[4] = {a.x, a.y, b.x, b.y};
#pragma unroll
            for (int i = 0; i < 4; i++) v[j][2 * i] = __uint_as_float(w[i] << 16), v[j][2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
        } else {
            const float4* x = reinterpret_cast<const float4*>((const float*)src.a + off + 8 * p);
            const float4 a = x[0], b = x[1];
            v[j][0] = a.x, v[j][1] = a.y, v[j][2] = a.z, v[j][3] = a.w, v[j][4] = b.x, v[j][5] = b.y, v[j][6] = b.z, v[j][7] = b.w;
            if (SRC == SKN_SRC_RMSNORM && tid + 256 * j < pieces)
                ss += ((a.x * a.x + a.y * a.y) + (a.z * a.z + a.w * a.w)) + ((b.x * b.x + b.y * b.y) + (b.z * b.z + b.w * b.w));
        }
    }
    if constexpr (SRC == SKN_SRC_RMSNORM) {
        ss = wave_sum(ss);
        if ((tid & 63) == 0) red[tid >> 6] = ss;
        __syncthreads();
        const float r = 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)k + src.eps);
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const float4 a = g0[j], b = g1[j];
            const float gw[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
            for (int i = 0; i < 8; i++) v[j][i] = v[j][i] * r * gw[i];
        }
    }
    // the bf16 values the product is defined on, and their largest finite magnitude
    float mx = 0.f;
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < 8; i++) {
            if (SRC != SKN_SRC_BF16) v[j][i] = __uint_as_float(bf16_rne(v[j][i]) << 16);
            const float f = fabsf(v[j][i]);
            if (f == f && f < INFINITY) mx = fmaxf(mx, f);
        }
    mx = wave_max(mx);
    if ((tid & 63) == 0) red[4 + (tid >> 6)] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[4], red[5]), fmaxf(red[6], red[7]));
    int e = 9;  // a zero row keeps scale 1
    if (mx > 0.f) e = (int)((__float_as_uint(mx) >> 23) & 0xFF) - 127;
    e = max(e, -100);  // (a subnormal maximum: exponent field 0)
    const float scale = __uint_as_float((uint32_t)(127 + 9 - e) << 23);
    if (tid == 0) inv_scale[row] = __uint_as_float((uint32_t)(127 - 9 + e) << 23);
    const int mb = row >> 5, r = row & 31;
    u32x4* out = afrag + (size_t)mb * (k >> 4) * 64 + r;
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const int p = tid + 256 * j;
        half8_t o;
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            o[i] = real ? (_Float16)(v[j][i] * scale) : (_Float16)0.f;
            sum += (float)o[i];
        }
        if (SUMS) {  // over the four lanes that hold a block
            sum += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(sum), 0xB1, 0xF, 0xF, true));
            sum += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(sum), 0x4E, 0xF, 0xF, true));
        }
        if (p < pieces) {
            const int b = p >> 2, h = (p >> 1) & 1, s = p & 1;
            out[(size_t)(2 * b + s) * 64 + 32 * h] = __builtin_bit_cast(u32x4, o);
            if (SUMS && (p & 3) == 0) {
                _Float16 hi, lo;
                skn_split_hilo(sum * 0x1p-12f, hi, lo);
                _Float16* sf = sfrag + ((size_t)mb * (k >> 8) + (b >> 3)) * 512 + (b & 7);
                sf[r * 8] = hi;
                sf[(32 + r) * 8] = lo;
            }
        }
    }
}

// ---- formats --------------------------------------------------------------------------------------------------------------
// kBytes: of 256 elements (a multiple of 16).  kPitch: of a row in LDS, 16 bytes more where kBytes would put its rows on few
// banks.  `row` points at the lane's row of the superblock in LDS, h is the lane's half (elements 16 h .. 16 h + 15 of a block).
// raw: the dwords of block b; unpack: its sixteen quants minus zero as two fp16 operands, returned is what the block's sum is multiplied
// with; mins: the minima of the eight blocks as an operand, returned their unit.
struct Fields {
    u32x4 head;  // K-quants: d | dmin, scales
};
struct Raw {
    uint32_t w[8];  // what of a block the lane needs, as it lies in LDS
};

__device__ __forceinline__ uint32_t lds_u32(const uint8_t* p) { return *reinterpret_cast<const uint32_t*>(p); }
__device__ __forceinline__ float half_lo(uint32_t w) { return (float)__builtin_bit_cast(half2_t, w).x; }
__device__ __forceinline__ float half_hi(uint32_t w) { return (float)__builtin_bit_cast(half2_t, w).y; }

// four bytes (0..255) minus zero as four fp16 numbers: 0x6400 | b is 1024 + b
template <int ZERO>
__device__ __forceinline__ u32x2 bytes_to_f16(uint32_t b) {
    const half2_t c = {(_Float16)(-1024 - ZERO), (_Float16)(-1024 - ZERO)};
    const half2_t lo = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, b, 0x04010400u)) + c;
    const half2_t hi = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, b, 0x04030402u)) + c;
    return u32x2{__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)};
}

template <int ZERO>
__device__ __forceinline__ void operands(const uint32_t (&b)[4], half8_t (&f)[2]) {
#pragma unroll
    for (int s = 0; s < 2; s++) {
        const u32x2 x = bytes_to_f16<ZERO>(b[2 * s]), y = bytes_to_f16<ZERO>(b[2 * s + 1]);
        f[s] = __builtin_bit_cast(half8_t, u32x4{x.x, x.y, y.x, y.y});
    }
}

// bits 0..3 of v to bit 4 of the four bytes
__device__ __forceinline__ uint32_t fifth_bits(uint32_t v) { return (((v & 0xFu) * 0x00204081u) & 0x01010101u) << 4; }

template <int N>
__device__ __forceinline__ void align2(const uint32_t (&w)[N], uint32_t (&b)[4]) {  // the sixteen bytes from byte 2 on
#pragma unroll
    for (int i = 0; i < 4; i++) b[i] = __builtin_amdgcn_alignbyte(w[i + 1], w[i], 2);
}

struct FmtQ80 {  // 34 bytes: d, 32 int8; block pairs are 17 dwords
    static constexpr int kBytes = 272, kPitch = 272;
    static constexpr bool kMin = false;
    __device__ static void head(const uint8_t*, Fields&) {}
    __device__ static Raw raw(const uint8_t* row, int b, int h) {
        const uint8_t* p = row + 68 * (b >> 1);
        Raw x;
#pragma unroll
        for (int i = 0; i < 5 - (b & 1); i++) x.w[i] = lds_u32(p + ((b & 1) ? 36 : 0) + 16 * h + 4 * i);
        x.w[5] = lds_u32(p + ((b & 1) ? 32 : 0));
        return x;
    }
    __device__ static float unpack(const Raw& x, const Fields&, int b, int, half8_t (&f)[2]) {
        uint32_t q[4] = {x.w[0], x.w[1], x.w[2], x.w[3]};
        const float d = (b & 1) ? half_hi(x.w[5]) : half_lo(x.w[5]);
        if (!(b & 1)) align2(x.w, q);
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] ^= 0x80808080u;
        operands<128>(q, f);
        return d;
    }
};

// the formats with nibbles: low ones are elements 0..15, high ones 16..31
__device__ __forceinline__ void nibbles(uint32_t (&q)[4], int h) {
#pragma unroll
    for (int i = 0; i < 4; i++) q[i] = (q[i] >> (4 * h)) & 0x0F0F0F0Fu;
}

struct FmtQ40 {  // 18 bytes: d, nibbles; pairs are 9 dwords
    static constexpr int kBytes = 144, kPitch = 144;
    static constexpr bool kMin = false;
    __device__ static void head(const uint8_t*, Fields&) {}
    __device__ static Raw raw(const uint8_t* row, int b, int) {
        const uint8_t* p = row + 36 * (b >> 1) + ((b & 1) ? 16 : 0);
        Raw x;
#pragma unroll
        for (int i = 0; i < 5; i++) x.w[i] = lds_u32(p + 4 * i);
        return x;
    }
    __device__ static float unpack(const Raw& x, const Fields&, int b, int h, half8_t (&f)[2]) {
        uint32_t q[4] = {x.w[1], x.w[2], x.w[3], x.w[4]};
        const float d = (b & 1) ? half_hi(x.w[0]) : half_lo(x.w[0]);
        if (!(b & 1)) align2(x.w, q);
        nibbles(q, h);
        operands<8>(q, f);
        return d;
    }
};

struct FmtQ41 {  // 20 bytes: d, m, nibbles
    static constexpr int kBytes = 160, kPitch = 176;
    static constexpr bool kMin = true;
    __device__ static void head(const uint8_t*, Fields&) {}
    __device__ static Raw raw(const uint8_t* row, int b, int) {
        Raw x;
#pragma unroll
        for (int i = 0; i < 5; i++) x.w[i] = lds_u32(row + 20 * b + 4 * i);
        return x;
    }
    __device__ static float unpack(const Raw& x, const Fields&, int, int h, half8_t (&f)[2]) {
        uint32_t q[4] = {x.w[1], x.w[2], x.w[3], x.w[4]};
        nibbles(q, h);
        operands<0>(q, f);
        return half_lo(x.w[0]);
    }
    __device__ static float mins(const uint8_t* row, const Fields&, half8_t& v) {
#pragma unroll
        for (int b = 0; b < 8; b++) v[b] = __builtin_bit_cast(half2_t, lds_u32(row + 20 * b)).y;
        return 4096.0f;
    }
};

struct FmtQ50 {  // 22 bytes: d, fifth bits, nibbles; pairs are 11 dwords
    static constexpr int kBytes = 176, kPitch = 176;
    static constexpr bool kMin = false;
    __device__ static void head(const uint8_t*, Fields&) {}
    __device__ static Raw raw(const uint8_t* row, int b, int) {
        const uint8_t* p = row + 44 * (b >> 1) + ((b & 1) ? 20 : 0);
        Raw x;
#pragma unroll
        for (int i = 0; i < 6; i++) x.w[i] = lds_u32(p + 4 * i);
        return x;
    }
    __device__ static float unpack(const Raw& x, const Fields&, int b, int h, half8_t (&f)[2]) {
        const uint32_t(&w)[8] = x.w;
        uint32_t q[4] = {w[2], w[3], w[4], w[5]}, qh = w[1];
        const float d = (b & 1) ? half_hi(w[0]) : half_lo(w[0]);
        if (!(b & 1)) {
            qh = __builtin_amdgcn_alignbyte(w[1], w[0], 2);
#pragma unroll
            for (int i = 0; i < 4; i++) q[i] = __builtin_amdgcn_alignbyte(w[i + 2], w[i + 1], 2);
        }
        nibbles(q, h);
        qh >>= 16 * h;
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] |= fifth_bits(qh >> (4 * i));
        operands<16>(q, f);
        return d;
    }
};

struct FmtQ51 {  // 24 bytes: d, m, fifth bits, nibbles
    static constexpr int kBytes = 192, kPitch = 208;
    static constexpr bool kMin = true;
    __device__ static void head(const uint8_t*, Fields&) {}
    __device__ static Raw raw(const uint8_t* row, int b, int) {
        Raw x;
#pragma unroll
        for (int i = 0; i < 6; i++) x.w[i] = lds_u32(row + 24 * b + 4 * i);
        return x;
    }
    __device__ static float unpack(const Raw& x, const Fields&, int, int h, half8_t (&f)[2]) {
        uint32_t q[4] = {x.w[2], x.w[3], x.w[4], x.w[5]};
        nibbles(q, h);
        const uint32_t qh = x.w[1] >> (16 * h);
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] |= fifth_bits(qh >> (4 * i));
        operands<0>(q, f);
        return half_lo(x.w[0]);
    }
    __device__ static float mins(const uint8_t* row, const Fields&, half8_t& v) {
#pragma unroll
        for (int b = 0; b < 8; b++) v[b] = __builtin_bit_cast(half2_t, lds_u32(row + 24 * b)).y;
        return 4096.0f;
    }
};

// The K-quants with sub-blocks of 32: d, dmin, twelve bytes of 6-bit scales and minima, then (Q5_K, 176 bytes) 32 bytes of fifth bits,
// 128 bytes of nibbles.
template <bool FIVE>
struct FmtK {
    static constexpr int kBytes = FIVE ? 176 : 144, kPitch = kBytes;
    static constexpr bool kMin = true;
    __device__ static void head(const uint8_t* row, Fields& H) { H.head = *reinterpret_cast<const u32x4*>(row); }
    __device__ static uint32_t scale4(const Fields& H, int half) {  // scales of sub-blocks 4 half .. 4 half + 3
        return half ? (H.head[3] & 0x0F0F0F0Fu) | ((H.head[1] >> 2) & 0x30303030u) : H.head[1] & 0x3F3F3F3Fu;
    }
    __device__ static uint32_t min4(const Fields& H, int half) {
        return half ? ((H.head[3] >> 4) & 0x0F0F0F0Fu) | ((H.head[2] >> 2) & 0x30303030u) : H.head[2] & 0x3F3F3F3Fu;
    }
    __device__ static Raw raw(const uint8_t* row, int b, int h) {
        const u32x4 x = *reinterpret_cast<const u32x4*>(row + (FIVE ? 48 : 16) + 32 * (b >> 1) + 16 * h);
        Raw v = {{x[0], x[1], x[2], x[3]}};
        if (FIVE) {
            const u32x4 y = *reinterpret_cast<const u32x4*>(row + 16 + 16 * h);
            v.w[4] = y[0], v.w[5] = y[1], v.w[6] = y[2], v.w[7] = y[3];
        }
        return v;
    }
    __device__ static float unpack(const Raw& x, const Fields& H, int b, int, half8_t (&f)[2]) {
        uint32_t q[4];
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] = (x.w[i] >> (4 * (b & 1))) & 0x0F0F0F0Fu;
        if (FIVE) {
#pragma unroll
            for (int i = 0; i < 4; i++) q[i] |= (b < 4 ? x.w[4 + i] << (4 - b) : x.w[4 + i] >> (b - 4)) & 0x10101010u;  // (bit b of the bytes: to bit 4)
        }
        operands<0>(q, f);
        return half_lo(H.head[0]) * (float)((scale4(H, b >> 2) >> (8 * (b & 3))) & 0xFFu);  // (11 x 6 bits: exact)
    }
    __device__ static float mins(const uint8_t*, const Fields& H, half8_t& v) {
#pragma unroll
        for (int b = 0; b < 8; b++) v[b] = (_Float16)(float)((min4(H, b >> 2) >> (8 * (b & 3))) & 0xFFu);
        return -4096.0f * half_hi(H.head[0]);
    }
};
// both at once
template <typename F>
__device__ __forceinline__ float block_of(const uint8_t* row, const Fields& H, int b, int h, half8_t (&f)[2]) {
    return F::unpack(F::raw(row, b, h), H, b, h, f);
}
// (Q8_0 with each of the two kinds of block on a path of its own: as above gemm_blocks_kernel spills twelve registers instead of three, 512 x
// 4096 x 4096 40.7 us against 39.6)
template <>
__device__ __forceinline__ float block_of<FmtQ80>(const uint8_t* row, const Fields&, int b, int h, half8_t (&f)[2]) {
    const uint8_t* p = row + 68 * (b >> 1);
    uint32_t q[4];
    float d;
    if (b & 1) {
        d = half_hi(lds_u32(p + 32));
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] = lds_u32(p + 36 + 16 * h + 4 * i);
    } else {
        d = half_lo(lds_u32(p));
        uint32_t w[5];
#pragma unroll
        for (int i = 0; i < 5; i++) w[i] = lds_u32(p + 16 * h + 4 * i);
        align2(w, q);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) q[i] ^= 0x80808080u;
    operands<128>(q, f);
    return d;
}
using FmtQ4K = FmtK<false>;
using FmtQ5K = FmtK<true>;

// ---- the product ------------------------------------------------------------------------------------------------------------

template <typename F, int MT>
constexpr int blocks_lds_bytes() {
    return std::max(4 * kBN * F::kPitch, MT * 24576);
}

template <typename F, int MT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_blocks_kernel(const u32x4* __restrict__ afrag, const u32x4* __restrict__ sfrag, const uint8_t* __restrict__ w,
                        const float* __restrict__ inv_scale, float* __restrict__ c, int m, int n, int k, int m_tiles, int n_tiles, int accumulate,
                        uint32_t a_bytes, uint32_t w_bytes, float* __restrict__ part, int part_blocks) {
    extern __shared__ __align__(16) uint8_t lds[];  // a superblock of 64 rows per wavefront, then the exchange of the tiles
    constexpr int P = F::kBytes / 16;               // sixteen-byte pieces of a row's superblock
    const int lane = threadIdx.x & 63;
    const int kq = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int h = lane >> 5, r = lane & 31;
    const int slot_in_xcd = blockIdx.x >> 3;  // consecutive workgroups of an XCD: the row tiles of one column tile
    const int mt = slot_in_xcd % m_tiles, tn = (slot_in_xcd / m_tiles) * 8 + (blockIdx.x & 7);
    if (tn >= n_tiles) return;
    const int nb = k >> 8;
    const int sb0 = (int)blockIdx.y * part_blocks, sb1 = min(sb0 + part_blocks, nb);  // (all, or a part of k)

    const __amdgpu_buffer_rsrc_t wrsrc = __builtin_amdgcn_make_buffer_rsrc((void*)w, 0, (int)w_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t arsrc = __builtin_amdgcn_make_buffer_rsrc((void*)afrag, 0, (int)a_bytes, 0x00020000);
    uint8_t* mine = lds + kq * kBN * F::kPitch;
    u32x4 next[P];
    // Piece x * 64 + lane of the 64 P of a superblock of the tile's rows.  (Its row and place are formed anew each time: kept, they
    // would hold 2 P registers.)  The lanes hand each other the weights through LDS: the lane number passes through an empty asm, so
    // that a store of wstore may go anywhere as far as the compiler knows and keeps its place among the loads before and after it,
    // and the device keeps a wavefront's LDS accesses in order.  (A wavefront-scope fence or barrier there instead costs 0.5 % in the mean
    // over 576 shapes and 5 % at the worst, Q4_0 5 x 11008 x 4096 15.4 -> 16.1 us: it also holds back the other loads.)
    auto wload = [&](int sb) __attribute__((always_inline)) {
        int l = lane;
        asm("" : "+v"(l));
#pragma unroll
        for (int x = 0; x < P; x++) {
            const int p = x * 64 + l, row = p / P;
            const int from = min(tn * kBN + row, n - 1) * (nb * F::kBytes) + (p - row * P) * 16;
            next[x] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, from, sb * F::kBytes, 0));
        }
    };
    auto wstore = [&]() __attribute__((always_inline)) {
        int l = lane;
        asm("" : "+v"(l));
#pragma unroll
        for (int x = 0; x < P; x++) {
            const int p = x * 64 + l, row = p / P;
            *reinterpret_cast<u32x4*>(mine + (F::kPitch == F::kBytes ? p * 16 : row * F::kPitch + (p - row * P) * 16)) = next[x];
        }
    };
    uint32_t abase[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) abase[i] = (uint32_t)(mt * MT + i) * (uint32_t)k * 64u;
    constexpr int RING = 4;  // k-steps
    u32x4 a[RING][MT];
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
    const float16_t zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

    if (sb0 + kq < sb1) {
        wload(sb0 + kq);
#pragma unroll
        for (int s = 0; s < RING; s++) afetch(16 * (sb0 + kq) + s, s);
    }
    for (int sb = sb0 + kq; sb < sb1; sb += 4) {
        const int sbn = min(sb + 4, nb - 1);  // (past the end: a repeat, unused)
        wstore();
        wload(sbn);
        const uint8_t* row[2] = {mine + r * F::kPitch, mine + (32 + r) * F::kPitch};
        Fields H[2];
        u32x4 sf[MT];
#pragma unroll
        for (int j = 0; j < 2; j++) F::head(row[j], H[j]);
        if constexpr (F::kMin) {
#pragma unroll
            for (int i = 0; i < MT; i++) sf[i] = sfrag[((size_t)(mt * MT + i) * nb + sb) * 64 + lane];
        }
#pragma unroll
        for (int b = 0; b < 8; b++) {
            half8_t f[2][2];
            float s[2];
#pragma unroll
            for (int j = 0; j < 2; j++) s[j] = block_of<F>(row[j], H[j], b, h, f[j]);
            // (while a tile's two matrix instructions run, the other wavefront of the SIMD scales or unpacks)
            float16_t p[2];
#pragma unroll
            for (int t = 0; t <= 2 * MT; t++) {
                if (t < 2 * MT) {
                    const int i = t >> 1, j = t & 1;
                    p[t & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a[(2 * b) % RING][i]), f[j][0], zero, 0, 0, 0);
                    p[t & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a[(2 * b + 1) % RING][i]), f[j][1], p[t & 1], 0, 0, 0);
                }
                if (t > 0) {
                    const int i = (t - 1) >> 1, j = (t - 1) & 1;
#pragma unroll
                    for (int x = 0; x < 16; x++) acc[i][j][x] = fmaf(s[j], p[(t - 1) & 1][x], acc[i][j][x]);
                }
            }
            // refill the two slots: RING steps ahead here, or in the wavefront's next superblock
#pragma unroll
            for (int x = 0; x < 2; x++) {
                const int ahead = 2 * b + x + RING;
                afetch(ahead < 16 ? 16 * sb + ahead : 16 * sbn + ahead - 16, ahead % RING);
            }
            __builtin_amdgcn_sched_barrier(0);  // (later blocks' quants read early would not fit the registers)
        }
        if constexpr (F::kMin) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
                half8_t v;
                const float unit = F::mins(row[j], H[j], v);
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    const float16_t p = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, sf[i]), v, zero, 0, 0, 0);
#pragma unroll
                    for (int x = 0; x < 16; x++) acc[i][j][x] = fmaf(unit, p[x], acc[i][j][x]);
                }
            }
        }
    }

    // the four partial tiles: tile t = 2 i + j belongs to wavefront t % 4, the other three hand theirs over
    float sc[16];
    if (!part) row_scales(inv_scale, (mt * MT + min(kq >> 1, MT - 1)) * 32, lane, sc);
    __syncthreads();
    float* red = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
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
                if (part) store_tile_part(sum, part + (size_t)blockIdx.y * m * n, n, (mt * MT + i) * 32, tn * kBN + 32 * j, m, n, lane);
                else store_tile(sum, c, n, (mt * MT + i) * 32, tn * kBN + 32 * j, m, n, sc, lane, accumulate != 0);
            }
        }
}

// ---- the product on 96-row tiles: wavefronts that unpack beside wavefronts that multiply ---------------------------------------
// A workgroup of eight wavefronts for each compute unit, on every SIMD a consumer and a producer; pair kq takes superblocks kq, kq + 4, ...
// of the 96 x 64 tile.  The producer unpacks a block of 32 elements of the 64 columns into two operands per column block (matrix-core
// order) and their scales, two blocks a phase, into four buffers in LDS; the consumer multiplies the phase before, its activations in
// registers four k-steps ahead, and adds a tile's products to its sums two tiles later, eight sums between two matrix instructions.  One
// bare barrier a phase (loads stay in flight over it).  The weights are unpacked once for 96 rows, and the unpacking's vector
// instructions come from another wavefront than the matrix instructions.
// Bound by the producers' chain from LDS to LDS (0.54 us per block alone, 0.6 with the products) and by one workgroup to hide it.
constexpr int kPcBuffers = 4;                 // blocks of unpacked weights between the two
constexpr int kPcBlock = 4 * 1024 + 256;      // two column blocks x two k-steps x 1 KiB, then 64 scales
constexpr int kPcMins = 2 * 1024 + 256;       // two column blocks x 1 KiB of minima, then 64 units
constexpr int kPcMT = 3;                      // row blocks of a tile
template <typename F>
constexpr int pc_work_bytes() {  // rows of weights, blocks and minima of the four pairs, then the exchange of the tiles
    return std::max(4 * (kBN * F::kPitch + kPcBuffers * kPcBlock + (F::kMin ? 2 * kPcMins : 0)), (3 * 4 + 4 * 2) * 4096);
}
template <typename F>
constexpr int pc_lds_bytes() {
    return pc_work_bytes<F>() + 32 * kPcMT * 4;
}

template <typename F>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_blocks_pc_kernel(const u32x4* __restrict__ afrag, const u32x4* __restrict__ sfrag, const uint8_t* __restrict__ w,
                           const float* __restrict__ inv_scale, float* __restrict__ c, int m, int n, int k, int m_tiles, int n_tiles, int accumulate,
                           uint32_t a_bytes, uint32_t w_bytes) {
    extern __shared__ __align__(16) uint8_t lds[];
    constexpr int MT = kPcMT;
    static_assert(MT == 3, "skn_blocks_of_96");
    constexpr int P = F::kBytes / 16;  // sixteen-byte pieces of a row's superblock
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), kq = wave & 3;
    const int h = lane >> 5, r = lane & 31;
    const int slot_in_xcd = blockIdx.x >> 3;  // consecutive workgroups of an XCD: the row tiles of one column tile
    const int mt = slot_in_xcd % m_tiles, tn = (slot_in_xcd / m_tiles) * 8 + (blockIdx.x & 7);
    if (tn >= n_tiles) return;
    const int nb = k >> 8;
    const int turns = (nb + 3) >> 2;
    uint8_t* blocks = lds + 4 * kBN * F::kPitch + kq * kPcBuffers * kPcBlock;  // of this pair of wavefronts
    uint8_t* minima = lds + 4 * (kBN * F::kPitch + kPcBuffers * kPcBlock) + kq * 2 * kPcMins;
    float* scales = reinterpret_cast<float*>(lds + pc_work_bytes<F>());  // of the tile's rows, for the store
    auto barrier = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    auto store = [&](const float16_t& sum, int t) __attribute__((always_inline)) {
        const int row0 = (mt * MT + (t >> 1)) * 32, col0 = tn * kBN + 32 * (t & 1);
        float sc[16];
#pragma unroll
        for (int x = 0; x < 16; x++) sc[x] = scales[32 * (t >> 1) + 8 * (x >> 2) + 4 * h + (x & 3)];
        store_tile(sum, c, n, row0, col0, m, n, sc, lane, accumulate != 0);
    };

    if (wave >= 4) {
        const __amdgpu_buffer_rsrc_t wrsrc = __builtin_amdgcn_make_buffer_rsrc((void*)w, 0, (int)w_bytes, 0x00020000);
        uint8_t* mine = lds + kq * kBN * F::kPitch;
        u32x4 next[P];
        auto wload = [&](int sb) __attribute__((always_inline)) {
#pragma unroll
            for (int x = 0; x < P; x++) {
                const int p = x * 64 + lane, row = p / P;
                const int from = min(tn * kBN + row, n - 1) * (nb * F::kBytes) + (p - row * P) * 16;
                next[x] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, from, min(sb, nb - 1) * F::kBytes, 0));
            }
        };
        const uint8_t* row[2] = {mine + r * F::kPitch, mine + (32 + r) * F::kPitch};
        Fields H[2];
        Raw raw[2][2];  // of a phase's two blocks, read ahead of it
        // superblock sb's weights to LDS, those of the pair's next one on their way
        auto begin = [&](int sb) __attribute__((always_inline)) {
#pragma unroll
            for (int x = 0; x < P; x++) {
                const int p = x * 64 + lane, rw = p / P;
                *reinterpret_cast<u32x4*>(mine + (F::kPitch == F::kBytes ? p * 16 : rw * F::kPitch + (p - rw * P) * 16)) = next[x];
            }
            asm volatile("" ::: "memory");  // (the lanes hand each other the weights; the device keeps a wavefront's LDS accesses in order)
            wload(sb + 4);
#pragma unroll
            for (int j = 0; j < 2; j++) F::head(row[j], H[j]);
        };
        auto read = [&](int b) __attribute__((always_inline)) {
#pragma unroll
            for (int e = 0; e < 2; e++)
#pragma unroll
                for (int j = 0; j < 2; j++) raw[e][j] = F::raw(row[j], b + e, h);
        };
        wload(kq);
        begin(kq);
        read(0);
        for (int i = 0; i < turns; i++) {
            const int sb = kq + 4 * i;  // (past the last one: a repeat, not multiplied)
#pragma unroll
            for (int b = 0; b < 8; b += 2) {
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    uint8_t* out = blocks + ((b + e) % kPcBuffers) * kPcBlock;
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        half8_t f[2];
                        const float s = F::unpack(raw[e][j], H[j], b + e, h, f);
                        *reinterpret_cast<half8_t*>(out + (2 * j) * 1024 + lane * 16) = f[0];
                        *reinterpret_cast<half8_t*>(out + (2 * j + 1) * 1024 + lane * 16) = f[1];
                        if (h == 0) *reinterpret_cast<float*>(out + 4096 + (j * 32 + r) * 4) = s;
                    }
                }
                if constexpr (F::kMin) {
                    if (b == 0) {
                        uint8_t* mo = minima + (i & 1) * kPcMins;
#pragma unroll
                        for (int j = 0; j < 2; j++) {
                            half8_t v;
                            const float unit = F::mins(row[j], H[j], v);
                            *reinterpret_cast<half8_t*>(mo + j * 1024 + lane * 16) = v;
                            if (h == 0) *reinterpret_cast<float*>(mo + 2048 + (j * 32 + r) * 4) = unit;
                        }
                    }
                }
                if (b < 6) read(b + 2);
                else if (i + 1 < turns) begin(sb + 4), read(0);
                barrier();
            }
        }
        barrier();
        // (the exchange of the tiles: the fifth and sixth are these wavefronts')
        barrier();
        if (kq < 2) {
            const float* red = reinterpret_cast<const float*>(lds);
            float16_t sum;
#pragma unroll
            for (int x = 0; x < 16; x++) sum[x] = red[(12 + 4 * kq) * 1024 + 64 * x + lane];
#pragma unroll
            for (int o = 1; o < 4; o++)
#pragma unroll
                for (int x = 0; x < 16; x++) sum[x] += red[(12 + 4 * kq + o) * 1024 + 64 * x + lane];
            store(sum, 4 + kq);
        }
    } else {
        const __amdgpu_buffer_rsrc_t arsrc = __builtin_amdgcn_make_buffer_rsrc((void*)afrag, 0, (int)a_bytes, 0x00020000);
        int block[MT];
        uint32_t abase[MT];
#pragma unroll
        for (int i = 0; i < MT; i++) block[i] = skn_blocks_of_96(mt * MT + i, m), abase[i] = (uint32_t)block[i] * (uint32_t)k * 64u;
        constexpr int RING = 4;  // k-steps
        u32x4 a[RING][MT];
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
        const float16_t zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        half8_t f[2][2][2];
        float s[2][2];
        auto take = [&](int b, int slot) __attribute__((always_inline)) {
            const uint8_t* in = blocks + (b % kPcBuffers) * kPcBlock;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                f[slot][j][0] = *reinterpret_cast<const half8_t*>(in + (2 * j) * 1024 + lane * 16);
                f[slot][j][1] = *reinterpret_cast<const half8_t*>(in + (2 * j + 1) * 1024 + lane * 16);
                s[slot][j] = *reinterpret_cast<const float*>(in + 4096 + (j * 32 + r) * 4);
            }
        };
#pragma unroll
        for (int x = 0; x < RING; x++) afetch(16 * min(kq, nb - 1) + x, x);
        if ((int)threadIdx.x < 32 * MT)
            scales[threadIdx.x] = inv_scale[32 * skn_blocks_of_96(mt * MT + ((int)threadIdx.x >> 5), m) + r];
        barrier();
        // (a pair without a superblock in the last turn only keeps the barriers: a branch around the multiplications inside this loop would
        // have every wait for an activation wait for the newest one)
        const int mine = max(0, (nb - kq + 3) >> 2);
        for (int i = 0; i < mine; i++) {
            const int sb = kq + 4 * i, sbn = min(sb + 4, nb - 1);  // (past the end: a repeat, unused)
            float16_t p[3];
            u32x4 sf[MT];
            if constexpr (F::kMin) {
#pragma unroll
                for (int x = 0; x < MT; x++) sf[x] = sfrag[((size_t)block[x] * nb + sb) * 64 + lane];
            }
#pragma unroll
            for (int b = 0; b < 8; b++) {
                if ((b & 1) == 0) take(b, 0);
#pragma unroll
                for (int t = 0; t < 2 * MT; t++) {
                    // A tile's two matrix instructions, each with half of the sums of the tile before last behind it: issued together
                    // the second would hold the wavefront until the matrix core is free, and a tile's products are not there sooner.
                    const int x = t >> 1, j = t & 1, at = b * 2 * MT + t;
                    const int old = (at + 2 * MT - 2) % (2 * MT), y = old >> 1, oj = old & 1, ob = (at - 2 + 16 * MT) / (2 * MT) & 1;
                    p[at % 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a[(2 * b) % RING][x]), f[b & 1][j][0], zero, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    if (at >= 2) {
#pragma unroll
                        for (int e = 0; e < 8; e++) acc[y][oj][e] = fmaf(s[ob][oj], p[(at - 2) % 3][e], acc[y][oj][e]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    p[at % 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a[(2 * b + 1) % RING][x]), f[b & 1][j][1], p[at % 3], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    if (at >= 2) {
#pragma unroll
                        for (int e = 8; e < 16; e++) acc[y][oj][e] = fmaf(s[ob][oj], p[(at - 2) % 3][e], acc[y][oj][e]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    if (t == 1 && (b & 1) == 0) take(b + 1, 1);  // (behind the last use of the scales it replaces)
                }
                if (b == 7) {
#pragma unroll
                    for (int t = 2 * MT - 2; t < 2 * MT; t++)
#pragma unroll
                        for (int e = 0; e < 16; e++) acc[t >> 1][t & 1][e] = fmaf(s[1][t & 1], p[(14 * MT + t) % 3][e], acc[t >> 1][t & 1][e]);
                }
                // refill the two slots: RING steps ahead here, or in the wavefront's next superblock
#pragma unroll
                for (int x = 0; x < 2; x++) {
                    const int ahead = 2 * b + x + RING;
                    afetch(ahead < 16 ? 16 * sb + ahead : 16 * sbn + ahead - 16, ahead % RING);
                }
                if constexpr (F::kMin) {
                    if (b == 7) {
                        const uint8_t* mi = minima + (i & 1) * kPcMins;
#pragma unroll
                        for (int j = 0; j < 2; j++) {
                            const half8_t v = *reinterpret_cast<const half8_t*>(mi + j * 1024 + lane * 16);
                            const float unit = *reinterpret_cast<const float*>(mi + 2048 + (j * 32 + r) * 4);
#pragma unroll
                            for (int y = 0; y < MT; y++) {
                                const float16_t q = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, sf[y]), v, zero, 0, 0, 0);
#pragma unroll
                                for (int x = 0; x < 16; x++) acc[y][j][x] = fmaf(unit, q[x], acc[y][j][x]);
                            }
                        }
                    }
                }
                if (b & 1) barrier();
            }
        }
        if (mine < turns)
#pragma unroll
            for (int b = 0; b < 4; b++) barrier();
        // the four partial tiles: of tile t < 4 the other three go to consumer t, of the others all four to producer t - 4
        float* red = reinterpret_cast<float*>(lds);
#pragma unroll
        for (int t = 0; t < 2 * MT; t++)
            if (kq != t) {
                float* dst = red + (t < 4 ? 3 * t + ((kq - t + 4) & 3) - 1 : 12 + 4 * (t - 4) + kq) * 1024 + lane;
#pragma unroll
                for (int x = 0; x < 16; x++) dst[64 * x] = acc[t >> 1][t & 1][x];
            }
        barrier();
#pragma unroll
        for (int t = 0; t < 4; t++)
            if (kq == t) {
                float16_t sum = acc[t >> 1][t & 1];
#pragma unroll
                for (int o = 0; o < 3; o++)
#pragma unroll
                    for (int x = 0; x < 16; x++) sum[x] += red[(3 * t + o) * 1024 + 64 * x + lane];
                store(sum, t);
            }
    }
}

template <typename F, int MT>
int launch_blocks(skn_ctx* ctx, const u32x4* afrag, const u32x4* sfrag, const float* isc, const skn_gemm_seg& seg, int m, int k, int splits, float* part) {
    const int m_tiles = (m + 32 * MT - 1) / (32 * MT), n_tiles = (seg.n + kBN - 1) / kBN;
    const unsigned grid = (unsigned)(((n_tiles + 7) / 8) * 8 * m_tiles);
    const uint32_t a_bytes = (uint32_t)((size_t)m_tiles * 32 * MT * k * 2), w_bytes = (uint32_t)((size_t)seg.n * (k / 256) * F::kBytes);
    skn_launch(ctx, gemm_blocks_kernel<F, MT>, dim3(grid, splits), dim3(256), blocks_lds_bytes<F, MT>(), afrag, sfrag, (const uint8_t*)seg.w, isc, seg.c, m,
               seg.n, k, m_tiles, n_tiles, seg.accumulate, a_bytes, w_bytes, splits > 1 ? part : (float*)nullptr, (k / 256 + splits - 1) / splits);
    SKN_LAUNCH_CHECK(ctx);
    if (splits < 2) return SKN_OK;
    const skn_gemm_parts ps = {{seg.c, nullptr, nullptr}, {seg.n, 0, 0}, {0, 0, 0}, {seg.accumulate, 0, 0}, 1, 0};
    return skn_gemm_add_parts(ctx, part, splits, seg.n, ps, isc, m);
}

template <typename F>
int launch_pc(skn_ctx* ctx, const u32x4* afrag, const u32x4* sfrag, const float* isc, const skn_gemm_seg& seg, int m, int k) {
    const int m_tiles = (m + 32 * kPcMT - 1) / (32 * kPcMT), n_tiles = (seg.n + kBN - 1) / kBN;
    const uint32_t a_bytes = (uint32_t)((size_t)skn_blocks_padded_rows(m) * k * 2), w_bytes = (uint32_t)((size_t)seg.n * (k / 256) * F::kBytes);
    skn_launch(ctx, gemm_blocks_pc_kernel<F>, dim3((n_tiles + 7) / 8 * 8 * m_tiles), dim3(512), pc_lds_bytes<F>(), afrag, sfrag, (const uint8_t*)seg.w, isc, seg.c, m,
               seg.n, k, m_tiles, n_tiles, seg.accumulate, a_bytes, w_bytes);
    SKN_LAUNCH_CHECK(ctx);
    return SKN_OK;
}

template <typename F>
int launch_format(skn_ctx* ctx, int mt, const u32x4* afrag, const u32x4* sfrag, const float* isc, const skn_gemm_seg& seg, int m, int k, int splits, float* part) {
    if constexpr (!std::is_same_v<F, FmtQ4K>) {
        if (mt == kPcMT) return launch_pc<F>(ctx, afrag, sfrag, isc, seg, m, k);
    }
    if (mt == 1) return launch_blocks<F, 1>(ctx, afrag, sfrag, isc, seg, m, k, splits, part);
    return launch_blocks<F, 2>(ctx, afrag, sfrag, isc, seg, m, k, splits, part);
}

template <int SRC, bool SUMS>
void launch_prep_nt(skn_ctx* ctx, const skn_gemm_src& src, u32x4* afrag, float* isc, _Float16* sfrag, int m, int m_pad, int k) {
    const int nt = (k / 8 + 255) / 256;  // (k <= 16384)
    if (nt <= 2) skn_launch(ctx, prep_blocks_kernel<2, SRC, SUMS>, dim3(m_pad), dim3(256), 0, src, afrag, isc, sfrag, m, k);
    else if (nt <= 4) skn_launch(ctx, prep_blocks_kernel<4, SRC, SUMS>, dim3(m_pad), dim3(256), 0, src, afrag, isc, sfrag, m, k);
    else skn_launch(ctx, prep_blocks_kernel<8, SRC, SUMS>, dim3(m_pad), dim3(256), 0, src, afrag, isc, sfrag, m, k);
}

template <int SRC>
void launch_prep(skn_ctx* ctx, const skn_gemm_src& src, bool sums, u32x4* afrag, float* isc, _Float16* sfrag, int m, int m_pad, int k) {
    if (sums) launch_prep_nt<SRC, true>(ctx, src, afrag, isc, sfrag, m, m_pad, k);
    else launch_prep_nt<SRC, false>(ctx, src, afrag, isc, sfrag, m, m_pad, k);
}

template <typename F>
int allow_lds(skn_ctx* ctx) {
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_blocks_kernel<F, 1>, hipFuncAttributeMaxDynamicSharedMemorySize, blocks_lds_bytes<F, 1>()));
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_blocks_kernel<F, 2>, hipFuncAttributeMaxDynamicSharedMemorySize, blocks_lds_bytes<F, 2>()));
    if constexpr (!std::is_same_v<F, FmtQ4K>)
        SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_blocks_pc_kernel<F>, hipFuncAttributeMaxDynamicSharedMemorySize, pc_lds_bytes<F>()));
    return SKN_OK;
}

int gemm_blocks_init(skn_ctx* ctx) {
    SKN_TRY(allow_lds<FmtQ80>(ctx));
    SKN_TRY(allow_lds<FmtQ40>(ctx));
    SKN_TRY(allow_lds<FmtQ41>(ctx));
    SKN_TRY(allow_lds<FmtQ50>(ctx));
    SKN_TRY(allow_lds<FmtQ51>(ctx));
    SKN_TRY(allow_lds<FmtQ4K>(ctx));
    return allow_lds<FmtQ5K>(ctx);
}
skn_family register_family(gemm_blocks_init);

int superblock_bytes(int t) {
    switch (t) {
        case SKN_TYPE_Q8_0: return FmtQ80::kBytes;
        case SKN_TYPE_Q4_0: return FmtQ40::kBytes;
        case SKN_TYPE_Q4_1: return FmtQ41::kBytes;
        case SKN_TYPE_Q5_0: return FmtQ50::kBytes;
        case SKN_TYPE_Q5_1: return FmtQ51::kBytes;
        case SKN_TYPE_Q4_K: return FmtQ4K::kBytes;
        case SKN_TYPE_Q5_K: return FmtQ5K::kBytes;
        default: return 0;
    }
}

// The kernel of 96-row tiles: where it has a tile for each compute unit at most and the 64-row one more than that.  Those then run beside
// each other on some units and alone on others, which wait.  us per call, 64 rows | 96: Q8_0 333 x 4096 x 4096 38.4 | 35.1, 84 x 16021 x 13312 93.9 | 87.6,
// 71 x 8954 x 2048 20.7 | 17.8; 333 x 4096 x 4096 in Q4_0 35.4 | 33.2, Q4_1 38.4 | 34.8, Q5_0 38.9 | 35.0, Q5_1 43.1 | 36.4, Q5_K 37.8 | 35.0.  Over 34 shapes of
// this range each of the six formats gains: 1.02 to 1.16 times as fast, 1.07 to 1.11 in the mean of a format, Q5_1 1.10 to 1.31 and 1.21.  In more rounds the
// smaller tiles are the faster ones: Q8_0 512 x 4096 x 4096 39.6 | 56, 1000 x 4096 x 11008 163 | 189; and tiles that leave half of the device idle have their
// k divided instead.
bool one_round_of_pc(const skn_ctx* ctx, int type, int n, int m) {
    const int columns = ((n + kBN - 1) / kBN + 7) / 8 * 8;  // (of the grid)
    return type != SKN_TYPE_Q4_K && m > 64 && ctx->opt_gemm_split == 0 && (int64_t)columns * ((m + 63) / 64) > ctx->compute_units &&
           (int64_t)columns * ((m + 32 * kPcMT - 1) / (32 * kPcMT)) <= ctx->compute_units;
}

bool has_minima(int t) { return t == SKN_TYPE_Q4_1 || t == SKN_TYPE_Q5_1 || t == SKN_TYPE_Q4_K || t == SKN_TYPE_Q5_K; }

}  // namespace

bool skn_gemm_blocks_ok(const skn_ctx* ctx, int type, const void* w, int n, int k, int m) {
    const int bytes = superblock_bytes(type);
    const size_t m_pad = ((size_t)m + 127) / 128 * 128;
    return ctx->opt_gemm_q6k_fused != 0 && bytes != 0 && ((uintptr_t)w & 15) == 0 && n > 0 && m > 0 && k > 0 && k % 256 == 0 && k <= 16384 &&
           m_pad * k * 2 < ((size_t)1 << 31) && (size_t)n * (k / 256) * bytes < ((size_t)1 << 31);
}

// Unpacking a block once per 64 rows against once per call: what costs the most vector instructions, a fifth bit or minima, loses first.
// Time of the general path over this one's, 600 to 14336 columns, k from 2048 to 11008:
//   Q5_1  1280 rows 0.93 - 1.14, 1536 0.80 - 1.09, 2048 0.75 - 0.96, 4096 0.87 - 0.97; two layers' prompts of width 4096 1500 tokens 1.01,
//         1800 0.99, 2048 0.92 (5019 | 4616 us), 3000 0.98, of width 2048 above 1.04 up to 3000
//   Q4_1  1792 rows 0.95 - 1.14; 1920 to 3072 rows of 2560 to 8192 columns with k from 4096 on 0.87 - 1.06, 0.94 in the mean (2048 x 4096 x
//         6144 267 | 232 us), other sizes 0.94 - 1.12; 4096 rows 0.98 - 1.13; prompts above 1.03 throughout
//   Q8_0, Q4_0, Q5_0, Q5_K  0.91 - 1.6, above one in the mean at every number of rows; prompts above 1.1
bool skn_gemm_blocks_pay(int type, int n, int k, int m, bool in_prompt) {
    if (type == SKN_TYPE_Q5_1) return in_prompt ? m <= 1800 || k < 4096 : m <= 1400;
    if (type == SKN_TYPE_Q4_1) return in_prompt || m <= 1850 || m > 3300 || k < 4096 || n < 2560 || n > 8192;
    return true;
}

int skn_gemm_blocks_multi(skn_ctx* ctx, const int* types, const skn_gemm_seg* segs, int nseg, int k, const skn_gemm_src& src, int m) {
    SKN_REQUIRE(ctx, nseg >= 1 && nseg <= 3 && m > 0, SKN_ERR_ARG, "block GEMM: bad segment count or shape");
    SKN_REQUIRE(ctx, src.a && ((uintptr_t)src.a & (src.kind == SKN_SRC_BF16 ? 7 : 15)) == 0, SKN_ERR_ARG, "block GEMM: activations are null or misaligned");
    SKN_REQUIRE(ctx, src.kind == SKN_SRC_BF16 || src.kind == SKN_SRC_F32 || (src.b && ((uintptr_t)src.b & 15) == 0), SKN_ERR_ARG,
                "block GEMM: second activation operand is null or misaligned");
    const int mt = m <= 32 ? 1 : 2, m_pad = skn_blocks_padded_rows(m), m_tiles = m_pad / (32 * mt);
    bool pc[3] = {false, false, false};
    int splits[3] = {1, 1, 1};
    size_t part_bytes = 0;  // (the products run one after the other: they share the room for their parts)
    bool sums = false;
    for (int i = 0; i < nseg; i++) {
        SKN_REQUIRE(ctx, segs[i].w && segs[i].c && skn_gemm_blocks_ok(ctx, types[i], segs[i].w, segs[i].n, k, m), SKN_ERR_ARG,
                    "block GEMM: a matrix is null or not one this path takes");
        splits[i] = skn_gemm_k_splits(ctx, m, m_tiles * ((segs[i].n + kBN - 1) / kBN), k / 256);
        if (splits[i] > 1) part_bytes = std::max(part_bytes, (size_t)splits[i] * m * segs[i].n * 4);
        pc[i] = splits[i] == 1 && one_round_of_pc(ctx, types[i], segs[i].n, m);
        sums = sums || has_minima(types[i]);
    }
    const size_t af_bytes = skn_align_up((size_t)m_pad * k * 2), sf_bytes = sums ? skn_align_up((size_t)m_pad * (k / 256) * 32) : 0;
    const size_t is_bytes = skn_align_up((size_t)m_pad * 4);
    uint8_t* ws;
    SKN_TRY(skn_gemm_workspace(ctx, af_bytes + sf_bytes + is_bytes, af_bytes + sf_bytes + is_bytes, &ws, src.ahead));
    u32x4* afrag = (u32x4*)ws;
    _Float16* sfrag = (_Float16*)(ws + af_bytes);
    float* isc = (float*)(ws + af_bytes + sf_bytes);
    float* part = part_bytes ? skn_gemm_parts_room(ctx, part_bytes) : nullptr;
    if (src.ahead) return SKN_OK;
    if (!part) splits[0] = splits[1] = splits[2] = 1;
    switch (src.kind) {
        case SKN_SRC_BF16: launch_prep<SKN_SRC_BF16>(ctx, src, sums, afrag, isc, sfrag, m, m_pad, k); break;
        case SKN_SRC_F32: launch_prep<SKN_SRC_F32>(ctx, src, sums, afrag, isc, sfrag, m, m_pad, k); break;
        case SKN_SRC_RMSNORM: launch_prep<SKN_SRC_RMSNORM>(ctx, src, sums, afrag, isc, sfrag, m, m_pad, k); break;
        default: return skn_fail(ctx, SKN_ERR_ARG, "block GEMM: unknown activation source %d", src.kind);
    }
    SKN_LAUNCH_CHECK(ctx);
    for (int i = 0; i < nseg; i++) {
        const u32x4* sf = (const u32x4*)sfrag;
        const int tile = pc[i] ? kPcMT : mt;
        int rc = SKN_OK;
        switch (types[i]) {
            case SKN_TYPE_Q8_0: rc = launch_format<FmtQ80>(ctx, tile, afrag, sf, isc, segs[i], m, k, splits[i], part); break;
            case SKN_TYPE_Q4_0: rc = launch_format<FmtQ40>(ctx, tile, afrag, sf, isc, segs[i], m, k, splits[i], part); break;
            case SKN_TYPE_Q4_1: rc = launch_format<FmtQ41>(ctx, tile, afrag, sf, isc, segs[i], m, k, splits[i], part); break;
            case SKN_TYPE_Q5_0: rc = launch_format<FmtQ50>(ctx, tile, afrag, sf, isc, segs[i], m, k, splits[i], part); break;
            case SKN_TYPE_Q5_1: rc = launch_format<FmtQ51>(ctx, tile, afrag, sf, isc, segs[i], m, k, splits[i], part); break;
            case SKN_TYPE_Q4_K: rc = launch_format<FmtQ4K>(ctx, tile, afrag, sf, isc, segs[i], m, k, splits[i], part); break;
            default: rc = launch_format<FmtQ5K>(ctx, tile, afrag, sf, isc, segs[i], m, k, splits[i], part); break;
        }
        if (rc != SKN_OK) return rc;
    }
    return SKN_OK;
}
