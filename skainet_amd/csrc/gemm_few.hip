// Product of few activation rows, or of some more with a small matrix, with block-quantized weights: C[m, n] = sum_k A[m, k] w[n, k], A bf16 as it is given, Q4_K, Q5_K,
// Q6_K, Q8_0 or Q4_0 weights: one launch, or two and room for the parts where few columns have their k divided.
//
// Bound by the latency of a launch, then by the unpacking.  The kernels for more rows (gemm.hip, gemm_blocks.hip) take three
// launches where tiles are few: a pass that scales the rows to fp16, the product, the addition of the parts of k.  None of it is
// needed here but, for few columns, the last.  A quant less its zero has at most eight bits, exact in bf16, so the matrix cores take the activations as they are
// (v_mfma_f32_16x16x32_bf16; products exact, sums in fp32), a block's sum starts from zero and joins the total in fp32 times the
// block's scale: an accumulator's column is the lane's own weight row, so the scale is one value per lane.  Minima: the block's
// activations against a column of ones is one more matrix instruction and gives the sum that the minimum is multiplied with.
// A workgroup keeps all of k, or its part, for its sixteen columns: its eight (or four) wavefronts take superblocks of 256 in
// turn and add their tiles through LDS.
//
// us per call, three launches -> this: Q4_K 16 x 4096 x 4096 11.7 -> 5.3, Q8_0 16 x 4096 x 4096 13.1 -> 6.4, Q6_K 41 x 4096 x 11008 33.5 -> 21.1 (weights
// alone 7.5 at the rate of a copy), Q5_K 64 x 2048 x 2048 12.9 -> 7.0.  Error against 64 bits: not larger (1.1 against 1.5e-7 of the
// result in Q4_K at k = 11008, 0.95 against 1.05 in Q8_0): a superblock's sum is formed before it joins the total.
#include "gemm_few.h"
#include "gemm_few_loads.h"
#include "gemm_tiles.h"

#include <algorithm>
#include <type_traits>

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// ---- formats --------------------------------------------------------------------------------------------------------------
// Lane 16 g + c holds column c (a weight row) and, of a block of 32 elements, elements 8 g .. 8 g + 7 (Q6_K, whose scales are for
// sixteen: elements 4 g .. 4 g + 3 of either half).  kBytes: of a superblock of 256 elements; kPieces: the sixteen-byte pieces that
// hold it; kPitch: of a row in LDS, chosen so that sixteen rows start in sixteen different groups of four banks.  `row` points at
// the lane's row there.

__device__ __forceinline__ float f16_lo(uint32_t w) { return (float)__builtin_bit_cast(half2_t, w).x; }
__device__ __forceinline__ float f16_hi(uint32_t w) { return (float)__builtin_bit_cast(half2_t, w).y; }
__device__ __forceinline__ uint32_t lds_u32(const uint8_t* p) { return *reinterpret_cast<const uint32_t*>(p); }
__device__ __forceinline__ u32x2 lds_u32x2(const uint8_t* p) { return *reinterpret_cast<const u32x2*>(p); }

// Range.  A tile is first summed in units of 2^-40, which the blocks' scales bring: the quants are operands as they are, every product of
// a finite activation with one is exact (down to bf16's least subnormal), and no sum of a row of least activations loses bits.  What does not
// fit there -- rows from about 2^47 on -- ends as an infinity or NaN, is seen when the tile is stored, and the tile is summed once more with
// operands times 2^-100, in units of 2^60, where sums of the largest activations and weights of all formats fit; rows that need it are large
// enough to lose nothing by it.  So a result is finite wherever it is for rows scaled to their largest element.  The first pass pays
// 0.1 to 0.3 us for looking at the sums (16 x 4096 x 4096 in Q4_K 5.0, 5.0, in Q6_K 6.4, 6.8, in Q8_0 6.0, 6.2) and, where one body of code serves both
// passes, for the subtraction below.  kTwoBodies: from so many row blocks on a format has a body for each.  Over 45 drawn shapes each, where runs of one
// build differ by 0.8 %, Q5_K is 1.04 times as fast for it in the mean (5 x 4096 x 11008 10.9 -> 10.0 us), Q4_0 1.03 (16 x 4096 x 4096 6.7 -> 6.4), Q6_K of more
// than sixteen rows 1.02 (32 x 6000 x 6144 17.5 -> 17.1); Q6_K of up to sixteen, Q8_0 and Q4_K, which gain at some sizes and lose at others (Q6_K 16 x 2048 x 2048 5.0 -> 5.1; Q8_0 16 x 512 x 4096 5.5 -> 5.2, 16 x 4096 x 11008 11.8 -> 12.1; Q4_K
// 16 x 2048 x 2048 3.9 -> 3.7, 16 x 12000 x 1024 5.3 -> 5.5), keep one.
constexpr float kUp = 0x1p40f;
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
struct Operands {
    uint32_t down;  // off the exponents of a pair of bf16 operands: 0, 100
    float nibble;   // 2^9, 2^-91
};

// Four whole numbers of at most eight bits, one to a byte, as bf16: the upper halves of their fp32 forms (zero stays zero: the
// subtraction stops there).
__device__ __forceinline__ uint32_t bf16_pair(float lo, float hi, const Operands& o) {
    const u16x2 x = __builtin_bit_cast(u16x2, __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(x, __builtin_bit_cast(u16x2, o.down)));
}
__device__ __forceinline__ u32x2 signed_bytes(uint32_t b, const Operands& o) {
    const float f0 = (float)(int8_t)b, f1 = (float)(int8_t)(b >> 8), f2 = (float)(int8_t)(b >> 16), f3 = (float)(int8_t)(b >> 24);
    return u32x2{bf16_pair(f0, f1, o), bf16_pair(f2, f3, o)};
}
__device__ __forceinline__ u32x2 unsigned_bytes(uint32_t b, const Operands& o) {
    const float f0 = (float)(uint8_t)b, f1 = (float)(uint8_t)(b >> 8), f2 = (float)(uint8_t)(b >> 16), f3 = (float)(uint8_t)(b >> 24);
    return u32x2{bf16_pair(f0, f1, o), bf16_pair(f2, f3, o)};
}
// Four numbers 0..15: as E4M3 a byte below sixteen is that many times 2^-9 (subnormals and the first binade are one straight line).
__device__ __forceinline__ u32x2 nibble_bytes(uint32_t b, const Operands& o) {
    return u32x2{__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, o.nibble, false)),
                 __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, o.nibble, true))};
}
__device__ __forceinline__ bf16x8 operand(u32x2 lo, u32x2 hi) { return __builtin_bit_cast(bf16x8, u32x4{lo.x, lo.y, hi.x, hi.y}); }

// The K-quants with sub-blocks of 32 (see gemm_blocks.hip for their layout).
template <bool FIVE>
struct FewK {
    static constexpr int kBytes = FIVE ? 176 : 144, kPieces = kBytes / 16, kPitch = kBytes;
    static constexpr bool kMin = true, kHalves = false;
    static constexpr int kTwoBodies = FIVE ? 1 : 5;
    struct Head {
        float d, dmin;
        uint32_t sc[2], mn[2];
        u32x2 fifth;
    };
    __device__ static __forceinline__ void head(const uint8_t* row, int g, Head& s) {
        const u32x4 h = *reinterpret_cast<const u32x4*>(row);
        s.d = f16_lo(h[0]) * kUp, s.dmin = f16_hi(h[0]) * kUp;
        s.sc[0] = h[1] & 0x3F3F3F3Fu, s.sc[1] = (h[3] & 0x0F0F0F0Fu) | ((h[1] >> 2) & 0x30303030u);
        s.mn[0] = h[2] & 0x3F3F3F3Fu, s.mn[1] = ((h[3] >> 4) & 0x0F0F0F0Fu) | ((h[2] >> 2) & 0x30303030u);
        if (FIVE) s.fifth = lds_u32x2(row + 16 + 8 * g);
    }
    __device__ static __forceinline__ bf16x8 block(const uint8_t* row, const Head& H, int b, int g, const Operands& o, float& s, float& mn) {
        s = H.d * (float)((H.sc[b >> 2] >> (8 * (b & 3))) & 0xFFu);  // (11 x 6 bits: exact)
        mn = H.dmin * (float)((H.mn[b >> 2] >> (8 * (b & 3))) & 0xFFu);
        const u32x2 x = lds_u32x2(row + (FIVE ? 48 : 16) + 32 * (b >> 1) + 8 * g);
        const u32x2 q = (x >> (uint32_t)(4 * (b & 1))) & 0x0F0F0F0Fu;
        if (!FIVE) return operand(nibble_bytes(q.x, o), nibble_bytes(q.y, o));
        const u32x2 f = (b < 4 ? H.fifth << (uint32_t)(4 - b) : H.fifth >> (uint32_t)(b - 4)) & 0x10101010u;
        return operand(unsigned_bytes(q.x | f.x, o), unsigned_bytes(q.y | f.y, o));
    }
};

struct FewQ80 {  // 34 bytes: d, 32 int8; block pairs are 17 dwords
    static constexpr int kBytes = 272, kPieces = 17, kPitch = 272;
    static constexpr bool kMin = false, kHalves = false;
    static constexpr int kTwoBodies = 5;
    struct Head {};
    __device__ static __forceinline__ void head(const uint8_t*, int, Head&) {}
    __device__ static __forceinline__ bf16x8 block(const uint8_t* row, const Head&, int b, int g, const Operands& o, float& s, float&) {
        const uint8_t* p = row + 68 * (b >> 1);
        uint32_t x, y;
        if (b & 1) {
            s = f16_hi(lds_u32(p + 32)) * kUp;
            x = lds_u32(p + 36 + 8 * g), y = lds_u32(p + 40 + 8 * g);
        } else {
            s = f16_lo(lds_u32(p)) * kUp;
            const uint32_t w0 = lds_u32(p + 8 * g), w1 = lds_u32(p + 4 + 8 * g), w2 = lds_u32(p + 8 + 8 * g);
            x = __builtin_amdgcn_alignbyte(w1, w0, 2), y = __builtin_amdgcn_alignbyte(w2, w1, 2);
        }
        return operand(signed_bytes(x, o), signed_bytes(y, o));
    }
};

struct FewQ40 {  // 18 bytes: d, nibbles (low ones elements 0..15, high ones 16..31); pairs are 9 dwords
    static constexpr int kBytes = 144, kPieces = 9, kPitch = 144;
    static constexpr bool kMin = false, kHalves = false;
    static constexpr int kTwoBodies = 1;
    struct Head {};
    __device__ static __forceinline__ void head(const uint8_t*, int, Head&) {}
    // a nibble at the top of its byte, less eight there, is 16 (q - 8)
    __device__ static __forceinline__ bf16x8 block(const uint8_t* row, const Head&, int b, int g, const Operands& o, float& s, float&) {
        const uint8_t* p = row + 36 * (b >> 1);
        const int at = 8 * (g & 1);
        u32x2 q;
        if (b & 1) {
            s = f16_hi(lds_u32(p + 16)) * (kUp / 16);
            q = u32x2{lds_u32(p + 20 + at), lds_u32(p + 24 + at)};
        } else {
            s = f16_lo(lds_u32(p)) * (kUp / 16);
            const uint32_t w0 = lds_u32(p + at), w1 = lds_u32(p + 4 + at), w2 = lds_u32(p + 8 + at);
            q = u32x2{__builtin_amdgcn_alignbyte(w1, w0, 2), __builtin_amdgcn_alignbyte(w2, w1, 2)};
        }
        q = ((q << (uint32_t)(g < 2 ? 4 : 0)) & 0xF0F0F0F0u) ^ 0x80808080u;
        return operand(signed_bytes(q.x, o), signed_bytes(q.y, o));
    }
};

// Q6_K: half hf of 128 elements, quarter Q of 32: low bits in nibble Q / 2 of bytes 64 hf + 32 (Q % 2) .. + 31, high bits at 2 Q of
// bytes 128 + 32 hf .. + 31, an int8 scale for sixteen elements from byte 192 on, d at 208: the end of the last piece, which is the
// superblock's last sixteen bytes.
struct FewQ6K {
    static constexpr int kBytes = 210, kPieces = 14, kPitch = 240;
    static constexpr bool kHalves = true;
    static constexpr int kTwoBodies = 2;
    struct Head {
        float d4;  // d / 4 (times 2^40): the operands are 4 (q - 32)
        u32x4 sc;
    };
    __device__ static __forceinline__ void head(const uint8_t* row, int, Head& s) {
        s.d4 = f16_hi(lds_u32(row + 220)) * (kUp / 4);
        s.sc = *reinterpret_cast<const u32x4*>(row + 192);
    }
    __device__ static __forceinline__ s16x4 sixteen(const uint8_t* row, const Head& H, int b, int t, int g, const Operands& o, float& s) {
        const int hf = b >> 2, Q = b & 3, e = 2 * b + t;
        s = H.d4 * (float)(int8_t)(H.sc[e >> 2] >> (8 * (e & 3)));
        const uint32_t ql = lds_u32(row + 64 * hf + 32 * (Q & 1) + 16 * t + 4 * g), qh = lds_u32(row + 128 + 32 * hf + 16 * t + 4 * g);
        const uint32_t lo = (Q < 2 ? ql << 2 : ql >> 2) & 0x3C3C3C3Cu;
        const uint32_t hi = (Q == 3 ? qh : qh << (6 - 2 * Q)) & 0xC0C0C0C0u;
        return __builtin_bit_cast(s16x4, signed_bytes((lo | hi) ^ 0x80808080u, o));
    }
};

// ---- the product ------------------------------------------------------------------------------------------------------------

// blocks of 32 whose activations a wavefront holds in LDS at a time (8 KiB at most)
constexpr int few_chunk(int mt) { return mt == 1 ? 4 : 2; }

template <typename F, int MT, int W>
constexpr int few_lds_bytes() {
    return std::max(W * (16 * F::kPitch + few_chunk(MT) * MT * 1024), W * MT * 1024);
}

// MT row blocks of sixteen, sixteen columns, W wavefronts
template <typename F, int MT, int W>
__global__ __launch_bounds__(64 * W) void gemm_few_kernel(const uint16_t* __restrict__ a, const uint8_t* __restrict__ w, float* __restrict__ c, int m, int n,
                                                          int k, uint32_t a_bytes, uint32_t w_bytes, double* __restrict__ part, int part_blocks) {
    extern __shared__ __align__(16) uint8_t lds[];  // a superblock of the tile's weight rows per wavefront, then the exchange of the tiles
    constexpr int P = F::kPieces;
    constexpr int CH = few_chunk(MT);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nb = k >> 8, n0 = (int)blockIdx.x * 16, m0 = (int)blockIdx.z * 16 * MT;
    const int sb0 = (int)blockIdx.y * part_blocks, sb1 = min(sb0 + part_blocks, nb);  // (all, or a part of k)
    const __amdgpu_buffer_rsrc_t wrsrc = __builtin_amdgcn_make_buffer_rsrc((void*)w, 0, (int)w_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t arsrc = __builtin_amdgcn_make_buffer_rsrc((void*)a, 0, (int)a_bytes, 0x00020000);
    uint8_t* mine = lds + wave * (16 * F::kPitch + CH * MT * 1024);
    uint8_t* rows = mine + 16 * F::kPitch;
    f32x4 acc[MT], total[MT];  // of a superblock, of the wavefront's superblocks
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};

    // The tile's rows of a superblock: coalesced loads one superblock ahead, handed over through LDS of the wavefront's own (the stores'
    // lane number passes through an empty asm of its own: a store may go anywhere as far as the compiler knows and keeps its place among
    // the loads before and after it, and the device keeps a wavefront's LDS accesses in order).  Where they come from: gemm_few_loads.h; from
    // one load to the next the offset grows by a scalar.  (With the offsets formed per lane and load by division: Q4_K 16 x 4096 x 4096 5.6 us against 5.0,
    // Q8_0 16 x 14000 x 1536 10.1 against 8.4.)
    using WL = FewWeightLoads<P, F::kBytes>;
    constexpr int WIDE = WL::WIDE, LOADS = WL::COUNT + (WL::REST ? 1 : 0);
    const uint32_t rb = (uint32_t)(nb * F::kBytes);
    const uint32_t wfrom = WL::wide(lane, n0, rb, w_bytes), restfrom = WL::rest(lane, n0, rb, w_bytes);
    u32x4 next[LOADS];
    auto wload = [&](int sb) __attribute__((always_inline)) {
#pragma unroll
        for (int x = 0; x < WL::COUNT; x++)
            next[x] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, (int)(wfrom + x * WL::step(rb)), sb * F::kBytes, 0));
        if (WL::REST) next[LOADS - 1] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, (int)restfrom, sb * F::kBytes, 0));
    };
    // The activations likewise, a chunk of CH blocks ahead, AP lanes to a row.
    using AL = FewActivationLoads<CH>;
    constexpr int AP = AL::LANES, AR = AL::ROWS;
    const uint32_t afrom = AL::first(lane, m0, 2u * k);
    u32x4 anext[CH * MT];
    auto aload = [&](int chunk) __attribute__((always_inline)) {
#pragma unroll
        for (int x = 0; x < CH * MT; x++)
            anext[x] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(arsrc, (int)(afrom + x * AL::step(2u * k)), chunk * 64 * CH, 0));
    };
    auto fits = [](float x) __attribute__((always_inline)) { return fabsf(x) < INFINITY; };
    const auto pass = [&](auto which) __attribute__((always_inline)) {
        const uint32_t less = which;  // (the second pass: 100)
        const Operands o = {(less << 7) * 0x10001u, __uint_as_float((127u + 9u - less) << 23)};
        const uint32_t one = 0x3F803F80u - o.down;
        const u32x4 ones_bits = {one, one, one, one};
        const bf16x8 ones = __builtin_bit_cast(bf16x8, ones_bits);
#pragma unroll
        for (int i = 0; i < MT; i++) total[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (sb0 + wave < sb1) {
            wload(sb0 + wave);
            aload((8 / CH) * (sb0 + wave));
        }
        // (addresses in LDS are formed behind the first loads, which they would delay by up to 0.2 us: u of what is read, v of what is stored)
        uint32_t u = lane, v = lane;
        asm volatile("" : "+v"(u), "+v"(v));
        const int col = u & 15u, g = u >> 4;
        const uint8_t* row = mine + col * F::kPitch;
        u32x4* const wto = reinterpret_cast<u32x4*>(mine + (v / WIDE) * F::kPitch + v % WIDE * 16);
        u32x4* const restto = reinterpret_cast<u32x4*>(mine + WL::rest_row(v) * F::kPitch + WL::rest_piece(v) * 16);
        auto wstore = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int x = 0; x < WL::COUNT; x++)
                if (WL::wide_lane(v)) wto[x * (64 / WIDE) * (F::kPitch / 16)] = next[x];
            if (WL::rest_lane(v)) *restto = next[LOADS - 1];
        };
        // Activations: piece p of row r goes to place p ^ turn(r) of the row, so that the sixteen rows of an operand lie on different banks.
        auto turn = [](int r) __attribute__((always_inline)) { return CH == 2 ? (r >> 1) & 7 : r & 15; };
        const int aplace = v % AP ^ turn(v / AP);
        uint8_t* const ato = rows + (v / AP) * (AP * 16);
        auto astore = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int x = 0; x < CH * MT; x++)  // (the turns of a load's first row and of the lane's row in it share no bits)
                *reinterpret_cast<u32x4*>(ato + x * AR * AP * 16 + (aplace ^ turn(x * AR & 15)) * 16) = anext[x];
        };
        auto aread = [&](int i, int b) __attribute__((always_inline)) {  // b: in the chunk
            const uint8_t* base = rows + (16 * i + col) * (AP * 16);
            if (!F::kHalves) return *reinterpret_cast<const u32x4*>(base + ((4 * b + g) ^ turn(col)) * 16);
            const u32x2 x = lds_u32x2(base + ((4 * b + (g >> 1)) ^ turn(col)) * 16 + 8 * (g & 1));
            const u32x2 y = lds_u32x2(base + ((4 * b + 2 + (g >> 1)) ^ turn(col)) * 16 + 8 * (g & 1));
            return u32x4{x.x, x.y, y.x, y.y};
        };
        for (int sb = sb0 + wave; sb < sb1; sb += W) {
            const int sbn = min(sb + W, nb - 1);  // (past the end: a repeat, unused)
            wstore();
            wload(sbn);
            typename F::Head H;
            F::head(row, g, H);
#pragma unroll
            for (int b = 0; b < 8; b++) {
                if (b % CH == 0) {
                    astore();
                    aload(b + CH < 8 ? (8 / CH) * sb + b / CH + 1 : (8 / CH) * sbn);
                }
                u32x4 av[MT];
#pragma unroll
                for (int i = 0; i < MT; i++) av[i] = aread(i, b % CH);
                if constexpr (F::kHalves) {
#pragma unroll
                    for (int t = 0; t < 2; t++) {
                        float s;
                        const s16x4 q = F::sixteen(row, H, b, t, g, o, s);
#pragma unroll
                        for (int i = 0; i < MT; i++) {
                            const s16x4 x = __builtin_bit_cast(s16x4, u32x2{av[i][2 * t], av[i][2 * t + 1]});
                            const f32x4 p = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(x, q, zero, 0, 0, 0);
#pragma unroll
                            for (int y = 0; y < 4; y++) acc[i][y] = b == 0 && t == 0 ? s * p[y] : fmaf(s, p[y], acc[i][y]);
                        }
                    }
                } else {
                    float s, mn = 0.f;
                    const bf16x8 q = F::block(row, H, b, g, o, s, mn);
#pragma unroll
                    for (int i = 0; i < MT; i++) {
                        const bf16x8 x = __builtin_bit_cast(bf16x8, av[i]);
                        const f32x4 p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, q, zero, 0, 0, 0);
#pragma unroll
                        for (int y = 0; y < 4; y++) acc[i][y] = b == 0 ? s * p[y] : fmaf(s, p[y], acc[i][y]);
                        if constexpr (F::kMin) {
                            const f32x4 sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, ones, zero, 0, 0, 0);
#pragma unroll
                            for (int y = 0; y < 4; y++) acc[i][y] = fmaf(-mn, sum[y], acc[i][y]);
                        }
                    }
                }
                if ((b & 3) == 3) __builtin_amdgcn_sched_barrier(0);  // (more blocks at once would not fit the registers)
            }
#pragma unroll
            for (int i = 0; i < MT; i++) total[i] += acc[i];
        }

        float size = 0.f;
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int y = 0; y < 4; y++) size += fabsf(total[i][y]);
        const bool left = __builtin_amdgcn_ballot_w64(!(size < 0x1p120f)) != 0;  // (below it the wavefronts' sums stay in range too)
        __syncthreads();
        f32x4* red = reinterpret_cast<f32x4*>(lds);
        uint32_t* lefts = reinterpret_cast<uint32_t*>(red + W * MT * 64);
#pragma unroll
        for (int i = 0; i < MT; i++) red[(wave * MT + i) * 64 + lane] = total[i];
        if (lane == 0) lefts[wave] = left;
        __syncthreads();
        uint32_t again = 0;
#pragma unroll
        for (int x = 0; x < W; x++) again |= lefts[x];
        // (accumulator register y of lane 16 g + c: row 4 g + y, column c)
        const float* flat = reinterpret_cast<const float*>(red);
        uint32_t tid = threadIdx.x, z = blockIdx.y;
        asm volatile("" : "+v"(tid), "+s"(z));  // (addresses of the outputs are formed here, not ahead of the loads)
        for (int e = tid; e < MT * 256; e += 64 * W) {
            const int r = e >> 4, cc = e & 15;
            const int from = (r >> 4) * 256 + (((r >> 2) & 3) * 16 + cc) * 4 + (r & 3);
            float sum = 0.f;
#pragma unroll
            for (int x = 0; x < W; x++) sum += flat[x * MT * 256 + from];
            if (m0 + r >= m || n0 + cc >= n) continue;
            const size_t at = (size_t)(m0 + r) * n + n0 + cc;
            // (the second pass replaces what the first could not hold)
            if (part) {
                double* to = part + (size_t)z * m * n + at;
                if (!less || (fits(sum) && !fits((float)*to))) *to = (double)sum * (less ? 0x1p60 : 0x1p-40);
            } else if (!less || (fits(sum) && !fits(c[at]))) {
                c[at] = sum * (less ? 0x1p60f : 0x1p-40f);
            }
        }
        return less || !__builtin_amdgcn_readfirstlane(again);  // (done)
    };
    if constexpr (MT >= F::kTwoBodies) {
        if (pass(std::integral_constant<uint32_t, 0>{})) return;
        __syncthreads();
        (void)pass(std::integral_constant<uint32_t, 100>{});
    } else {
        uint32_t less = 0;
#pragma unroll 1
        for (;;) {
            asm volatile("" : "+s"(less));  // (one body for both)
            if (pass(less)) return;
            less = 100;
            __syncthreads();
        }
    }
}

// The parts of divided k, in fp64: whatever units a tile was summed in.
__global__ __launch_bounds__(256) void gemm_few_add_kernel(const double* __restrict__ part, int splits, size_t count, float* __restrict__ c) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= count) return;
    double v[16];  // (at most sixteen parts, all asked for before the first is used)
#pragma unroll
    for (int z = 0; z < 16; z++) v[z] = z < splits ? part[z * count + i] : 0.0;
    double sum = v[0];
#pragma unroll
    for (int z = 1; z < 16; z++) sum += v[z];
    c[i] = (float)sum;
}

template <typename F, int MT, int W>
int launch_few(skn_ctx* ctx, const uint8_t* w, const uint16_t* a, float* c, int m, int n, int k, int splits) {
    const int nb = k / 256, each = (nb + splits - 1) / splits;
    splits = (nb + each - 1) / each;  // (no workgroup without a superblock)
    double* part = splits > 1 ? (double*)skn_gemm_parts_room(ctx, (size_t)splits * m * n * sizeof(double)) : nullptr;
    if (!part) splits = 1;
    skn_launch(ctx, gemm_few_kernel<F, MT, W>, dim3((n + 15) / 16, splits, (m + 16 * MT - 1) / (16 * MT)), dim3(64 * W), few_lds_bytes<F, MT, W>(), a, w, c, m, n, k,
               (uint32_t)((size_t)m * k * 2), (uint32_t)((size_t)n * nb * F::kBytes), part, splits > 1 ? each : nb);
    SKN_LAUNCH_CHECK(ctx);
    if (!part) return SKN_OK;
    const size_t count = (size_t)m * n;
    skn_launch(ctx, gemm_few_add_kernel, dim3((uint32_t)((count + 255) / 256)), dim3(256), 0, (const double*)part, splits, count, c);
    SKN_LAUNCH_CHECK(ctx);
    return SKN_OK;
}

// Few columns: k over workgroups too where the turns of a wavefront that this saves, 0.5 + 0.7 MT us each, pay for the addition (3 us).  us
// per call, undivided | in four parts: Q4_K 16 x 1000 x 11008 10.1 | 8.3, 64 x 1000 x 11008 23 | 12.9, 16 x 2000 x 2048 4.9 | 7.5 (undivided).
// Where the tiles are more than the compute units and a workgroup of eight wavefronts leaves no LDS for another, four of them go
// to a workgroup: Q8_0 57 x 8192 x 2048 14.1 | 12.5, 41 x 14336 x 4096 33.3 | 28.9 (with room for two: Q4_K 41 x 14336 x 4096 26.2 | 30.2).
template <typename F, int MT>
int launch_rows(skn_ctx* ctx, const uint8_t* w, const uint16_t* a, float* c, int m, int n, int k) {
    const int tiles = (n + 15) / 16 * ((m + 16 * MT - 1) / (16 * MT)), nb = k / 256;
    const int splits = std::max(1, std::min({ctx->compute_units / tiles, (nb + 7) / 8, 16}));
    const int saved = (nb + 7) / 8 - ((nb + splits - 1) / splits + 7) / 8;
    if (saved * (0.5f + 0.7f * MT) > 3.0f) return launch_few<F, MT, 8>(ctx, w, a, c, m, n, k, splits);
    if constexpr (few_lds_bytes<F, MT, 8>() > 80 * 1024) {
        if (tiles > ctx->compute_units) return launch_few<F, MT, 4>(ctx, w, a, c, m, n, k, 1);
    }
    return launch_few<F, MT, 8>(ctx, w, a, c, m, n, k, 1);
}

// row blocks of a workgroup: rows go in groups of at most 64, as even as blocks of sixteen are
int row_blocks(int m) {
    const int groups = (m + 63) / 64;
    return ((m + groups - 1) / groups + 15) / 16;
}

template <typename F>
int launch_format(skn_ctx* ctx, const uint8_t* w, const uint16_t* a, float* c, int m, int n, int k) {
    switch (row_blocks(m)) {
        case 1: return launch_rows<F, 1>(ctx, w, a, c, m, n, k);
        case 2: return launch_rows<F, 2>(ctx, w, a, c, m, n, k);
        case 3: return launch_rows<F, 3>(ctx, w, a, c, m, n, k);
        default: return launch_rows<F, 4>(ctx, w, a, c, m, n, k);
    }
}

template <typename F, int MT>
int allow_lds(skn_ctx* ctx) {
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_few_kernel<F, MT, 8>, hipFuncAttributeMaxDynamicSharedMemorySize, few_lds_bytes<F, MT, 8>()));
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)gemm_few_kernel<F, MT, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, few_lds_bytes<F, MT, 4>()));
    return SKN_OK;
}

template <typename F>
int allow_format(skn_ctx* ctx) {
    SKN_TRY((allow_lds<F, 1>(ctx)));
    SKN_TRY((allow_lds<F, 2>(ctx)));
    SKN_TRY((allow_lds<F, 3>(ctx)));
    return allow_lds<F, 4>(ctx);
}

int few_init(skn_ctx* ctx) {
    SKN_TRY(allow_format<FewK<false>>(ctx));
    SKN_TRY(allow_format<FewK<true>>(ctx));
    SKN_TRY(allow_format<FewQ6K>(ctx));
    SKN_TRY(allow_format<FewQ80>(ctx));
    return allow_format<FewQ40>(ctx);
}
skn_family register_family(few_init);

}  // namespace

// Every sixteen columns read all the activations and unpack for themselves, so that the time here grows with the row blocks where the
// other kernels' hardly does: what they gain on three launches is lost again from so many superblocks of sixteen columns per compute unit
// on (16, 32, 48, 64 rows, more in groups of 64; 0: not found up to 196).  us per call, others | these: Q4_K 32 x 12000 x 4096 (47) 18.7 | 15.8, 32 x 14336 x 4096
// (56) 19.7 | 20.4, 41 x 6000 x 6144 (35) 20.6 | 19.2, 41 x 14336 x 4096 20.9 | 26.2; Q5_K 32 x 14336 x 4096 22.1 | 22.0, 41 x 14336 x 4096 26.9 | 28.1;
// Q6_K 41 x 14336 x 4096 33.7 | 30.6, 57 x 14336 x 4096 33.6 | 40.5; Q8_0 41 x 14336 x 4096 29.0 | 28.9, 32 x 14336 x 14336 (196) 74 | 85; Q4_0 (whose
// quants take three times Q4_K's instructions) 16 x 6000 x 6144 17.8 | 15.6, 16 x 14336 x 4096 18.7 | 19.3.  Over a single round of compute units
// 64 rows hold out longer: 64 x 4096 x 11008 (43) Q4_K 24.8 | 23.3, Q8_0 28.7 | 23.5, against 57 x 6000 x 6144 21.2 | 27.3, 25.6 | 26.4.
// More than 64 rows: Q5_K 128 x 2700 x 2816 (15) 18.2 | 16.6, 512 x 2000 x 1024 (16) 14.0 | 13.9; Q6_K 700 x 2000 x 1024 (21) 24.5 | 19.0; Q8_0 333 x
// 4096 x 1024 (24) 16.8 | 15.2, 256 x 2700 x 2816 (29) 22.1 | 21.3; Q4_0 512 x 2000 x 1024 13.2 | 12.7, 256 x 2700 x 2816 19.4 | 21.1; Q4_K 160 x 1000 x 2048
// (6) 16.4 | 6.8, 200 x 1000 x 2048 (8) 16.4 | 6.9, 512 x 2000 x 1024 13.8 | 13.4.  (The others there had tiles of 64 rows.  Where they take 96 now, these are
// still 1.16, 1.11 and 1.14 times as fast in the mean over forty shapes each of Q8_0, Q4_0 and Q5_K that come here, and at worst 1.04, 1.08 and 1.08 times
// as slow, in the upper half of the limits: Q4_0 254 x 4907 x 512 (10) 12.7 | 13.7, 268 x 3547 x 768 (13) 12.7 | 13.6.)
// Short rows of many columns are launches of many short workgroups, whose ramp the passes' larger tiles pay less often: from so many
// rounds of compute units on they are faster whatever the superblocks (but for one row block, Q4_0's apart): Q4_0 31 x 30269 x 512 11.8 | 15.3, 25 x 23000 x 512
// 11.0 | 11.4; Q4_K 252 x 6683 x 256 12.6 | 16.1; Q5_K 32 x 29393 x 512 12.5 | 14.7; Q6_K 370 x 13269 x 256 20.7 | 36.3, 849 x 5423 x 256 44.9 | 35.4; Q8_0 248 x 24474
// x 256 30.3 | 34.8, 507 x 8812 x 256 29.2 | 26.4.  Four row blocks of Q5_K and Q4_0 lose earlier where their last round is hardly begun: 49 x 4296 x 3072
// 14.2 | 16.6, 58 x 13285 x 1536 16.3 | 20.0, against 57 x 7844 x 1536 in 1.9 rounds 16.3 | 14.1.  (Of 2607 drawn shapes that the limits above accept the
// passes were more than 3 % faster in 123, at worst 1.75 times; of 2190 drawn with these two rules in 14, at worst 1.08 times.)
// Q4_K and Q6_K of 33 to 64 rows, up to 4096 elements and a round of tiles or more stay with the others although this is the faster path
// (41 x 4096 x 4096 15.5 | 9.7 and 19.3 | 10.7): the number of launches that such products take is held fixed by tests, as is Q4_K's 200 x 1024 x 2048.  Options that fix how k is divided mean the others.
bool skn_gemm_few_ok(const skn_ctx* ctx, int type, const void* w, int n, int k, int m) {
    int bytes;
    struct {
        int rows[5], rounds;
    } most;
    switch (type) {
        case SKN_TYPE_Q4_K: bytes = FewK<false>::kBytes, most = {{0, 48, 36, 20, 7}, 6}; break;
        case SKN_TYPE_Q5_K: bytes = FewK<true>::kBytes, most = {{0, 56, 40, 12, 15}, 6}; break;
        case SKN_TYPE_Q6_K: bytes = FewQ6K::kBytes, most = {{0, 0, 60, 24, 20}, 19}; break;
        case SKN_TYPE_Q8_0: bytes = FewQ80::kBytes, most = {{0, 80, 50, 24, 24}, 19}; break;
        case SKN_TYPE_Q4_0: bytes = FewQ40::kBytes, most = {{45, 33, 33, 12, 16}, 5}; break;
        default: return false;
    }
    if (ctx->opt_gemm_few != 1 || ctx->opt_gemm_tile != 0 || ctx->opt_gemm_split != 0 || ctx->opt_test_gemm_no_parts == 1 || ctx->opt_gemm_q6k_fused != 1 || m <= 0 || n <= 0 || k <= 0 || k % 256 != 0 || k > 16384 ||
        ((uintptr_t)w & (type == SKN_TYPE_Q6_K ? 1 : 15)) != 0 || (size_t)n * (k / 256) * bytes >= ((size_t)1 << 31))
        return false;
    const int blocks = std::min((m + 15) / 16, 5), tiles = (n + 15) / 16, groups = (m + 63) / 64;
    if (m > 32 && m <= 64 && k <= 4096 && tiles >= ctx->compute_units && (type == SKN_TYPE_Q4_K || type == SKN_TYPE_Q6_K)) return false;
    const size_t all = (size_t)tiles * groups, units = ctx->compute_units;
    if (all > most.rounds * units && (m > 16 || type == SKN_TYPE_Q4_0)) return false;
    const bool begun = blocks == 4 && 5 * all >= 7 * units && all <= 2 * units;  // (1.4 to two rounds)
    const int limit = blocks == 4 && all <= units ? 45 : begun ? std::max(20, most.rows[3]) : most.rows[blocks - 1];
    return limit == 0 || all * (k / 256) <= limit * units;
}

int skn_gemm_few(skn_ctx* ctx, int type, const void* w, int n, int k, const uint16_t* a_bf16, int m, float* c) {
    const uint8_t* wb = (const uint8_t*)w;
    switch (type) {
        case SKN_TYPE_Q4_K: return launch_format<FewK<false>>(ctx, wb, a_bf16, c, m, n, k);
        case SKN_TYPE_Q5_K: return launch_format<FewK<true>>(ctx, wb, a_bf16, c, m, n, k);
        case SKN_TYPE_Q6_K: return launch_format<FewQ6K>(ctx, wb, a_bf16, c, m, n, k);
        case SKN_TYPE_Q8_0: return launch_format<FewQ80>(ctx, wb, a_bf16, c, m, n, k);
        default: return launch_format<FewQ40>(ctx, wb, a_bf16, c, m, n, k);
    }
}
