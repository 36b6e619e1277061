// Batched product of activations [m, k] with a stacked dense matrix [rows, k], both bf16 (v_mfma_f32_32x32x16_bf16) or
// both fp32 (v_mfma_f32_32x32x2_f32: true 32-bit products and sums), fp32 accumulation, epilogue in the store.
//
// Workgroup of WM x WN wavefronts, each with a tile of 32 TM tokens x 32 TN weight rows, walked along k in slices of 128
// bytes.  Both operands of a slice go from memory straight into LDS (16 bytes per lane, eight rows per request); the lane that
// fills slot s of row r fetches piece s ^ ((r / 2) % 8) of the row, so that the fragment reads -- the same piece of 32
// consecutive rows -- touch all 64 banks per sixteen lanes.  ST slices are in LDS at once: one bare barrier per slice, which
// says both "everyone's requests for this slice have landed" and "everyone is done with the slice before it", whose
// buffer the next request may overwrite.  Within a slice the fragments of a k-step are read while the products of the one
// before it run.
// The weights are the row operand, so that a lane's accumulators are runs of four consecutive outputs of one token.
// The fp32 form reads the same 16-byte pieces (four elements, half a wavefront each) and issues four matrix instructions
// per piece: k is summed in another order than it lies in memory, the same for both operands.
#include "dense.h"

#include <type_traits>

namespace {

typedef short bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8_v __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));

constexpr int kSlice = 128;  // bytes of k per slice

// KG groups of WM x WN wavefronts share the slices of a tile in turn; their sums meet in the epilogue.
template <int WM_, int WN_, int TM_, int TN_, int ST_, int KG_ = 1>
struct Shape {
    static constexpr int WM = WM_, WN = WN_, TM = TM_, TN = TN_, ST = ST_, KG = KG_;
    static constexpr int kThreads = 64 * WM * WN * KG, kRowsA = 32 * TM * WM, kRowsW = 32 * TN * WN;
    static constexpr int kBuf = (kRowsA + kRowsW) * kSlice;
    // the epilogue passes 32 WM tokens of the tile at a time through LDS
    static constexpr int kPitch = kRowsW + 4, kOutBytes = 32 * WM * kPitch * 4;
    static constexpr int kLds = KG * (ST * kBuf > kOutBytes ? ST * kBuf : kOutBytes);
};

__device__ __forceinline__ uint32_t half_bits(float f) { return __half_as_ushort(__float2half_rn(f)); }

template <typename T>
__device__ __forceinline__ float16_t mma(const u32x4& a, const u32x4& b, float16_t c) {
    if constexpr (std::is_same<T, float>::value) {
        const f32x4 x = __builtin_bit_cast(f32x4, a), y = __builtin_bit_cast(f32x4, b);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(x.x, y.x, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(x.y, y.y, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(x.z, y.z, c, 0, 0, 0);
        return __builtin_amdgcn_mfma_f32_32x32x2f32(x.w, y.w, c, 0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_v, a), __builtin_bit_cast(bf16x8_v, b), c, 0, 0, 0);
    }
}

// T: uint16_t (bf16) or float.  lda_b, ldw_b: row pitches in bytes; slices = k_pad bytes / 128.
template <typename T, typename S>
__global__ __launch_bounds__(S::kThreads) void dense_gemm_kernel(const uint8_t* __restrict__ a, int64_t lda_b, int m, const uint8_t* __restrict__ w,
                                                                 int64_t ldw_b, int rows, int slices, int tiles_m, int tiles,
                                                                 const float* __restrict__ bias, const skn_dense_out out) {
    extern __shared__ __align__(16) uint8_t lds[];
    constexpr int WM = S::WM, WN = S::WN, TM = S::TM, TN = S::TN, ST = S::ST, KG = S::KG, kRowsA = S::kRowsA, kRowsW = S::kRowsW;
    constexpr int kReqA = kRowsA / 8 / (WM * WN), kReqW = kRowsW / 8 / (WM * WN), kReq = kReqA + kReqW;  // requests per wavefront and slice
    static_assert(kReqA * 8 * WM * WN == kRowsA && kReqW * 8 * WM * WN == kRowsW, "whole requests");
    const int tid = threadIdx.x, lane = tid & 63;
    const int all_wave = __builtin_amdgcn_readfirstlane(tid >> 6), group = all_wave / (WM * WN), wave = all_wave % (WM * WN);
    // An XCD (blockIdx % 8) takes consecutive tiles, which run down up to eight token tiles before they move on to the next
    // weight tile: what is resident on an XCD at a time shares both operands in its L2.
    const int per = (tiles + 7) / 8, tile = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (tile >= tiles || (int)(blockIdx.x >> 3) >= per) return;
    const int tiles_n = tiles / tiles_m, band = tile / (8 * tiles_n), band_m = min(8, tiles_m - 8 * band), in_band = tile - band * 8 * tiles_n;
    const int m0 = (8 * band + in_band % band_m) * kRowsA, n0 = in_band / band_m * kRowsW;

    // Requests go through buffer resources of the tile's rows: the compiler takes a load into LDS with a 64-bit address for one that LDS may
    // answer too, and every wait for a fragment then becomes a wait for all that were asked for (256 x 256
    // tiles spent 37 % of their clocks waiting; 2048 x 8192 x 2048 97.7 -> 89.3 us, 2048 x 2048 x 8192 in 128 x 64 105.9 -> 94.5, 1000 x 10752 x 2048
    // 72.2 -> 63.9).
    const int here_m = min(m - m0, kRowsA), here_n = min(rows - n0, kRowsW);
    const __amdgpu_buffer_rsrc_t res_a = __builtin_amdgcn_make_buffer_rsrc((void*)(a + (int64_t)m0 * lda_b), 0, (int)(here_m * lda_b), 0x00020000);
    const __amdgpu_buffer_rsrc_t res_w = __builtin_amdgcn_make_buffer_rsrc((void*)(w + (int64_t)n0 * ldw_b), 0, (int)(here_n * ldw_b), 0x00020000);
    int from_a[kReqA], from_w[kReqW];  // byte offsets of this lane's pieces
#pragma unroll
    for (int i = 0; i < kReqA; i++) {
        const int r = (wave * kReqA + i) * 8 + (lane >> 3);
        from_a[i] = min(r, here_m - 1) * (int)lda_b + ((lane & 7) ^ ((r >> 1) & 7)) * 16;
    }
#pragma unroll
    for (int i = 0; i < kReqW; i++) {
        const int r = (wave * kReqW + i) * 8 + (lane >> 3);  // (kRowsA is a multiple of 16: the same swizzle as by its row of the stacked buffer)
        from_w[i] = min(r, here_n - 1) * (int)ldw_b + ((lane & 7) ^ ((r >> 1) & 7)) * 16;
    }
    // the group's i-th slice is slice KG i + group of the tile
    const int own = (slices - group + KG - 1) / KG, turns = (slices + KG - 1) / KG;
    auto request = [&](int i_own) __attribute__((always_inline)) {
        const int buf = (group * ST + i_own % ST) * S::kBuf, slice = KG * i_own + group;
        uint8_t* to = lds + buf;
#pragma unroll
        for (int i = 0; i < kReqA; i++)
            skn_load_to_lds(res_a, to + (wave * kReqA + i) * 1024, from_a[i], slice * kSlice);
#pragma unroll
        for (int i = 0; i < kReqW; i++)
            skn_load_to_lds(res_w, to + kRowsA * kSlice + (wave * kReqW + i) * 1024, from_w[i], slice * kSlice);
    };

    float16_t acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; i++)
#pragma unroll
        for (int j = 0; j < TM; j++)
#pragma unroll
            for (int x = 0; x < 16; x++) acc[i][j][x] = 0.f;

    const int wv_m = wave % WM, wv_n = wave / WM, wm = wv_m * 32 * TM, wn = wv_n * 32 * TN, h = lane >> 5, r32 = lane & 31;
    const uint8_t* frag_a = lds + (wm + r32) * kSlice;
    const uint8_t* frag_w = lds + (kRowsA + wn + r32) * kSlice;
    const int swz = (r32 >> 1) & 7;  // (the 32-row blocks start at multiples of 16 rows: the same for all of them)

#pragma unroll
    for (int s = 0; s < ST - 1; s++)
        if (s < own) request(s);
    for (int s = 0; s < turns; s++) {
        // requests complete in order: all but the newest ST - 2 slices' have landed (near the end there are fewer newer ones: all)
        if (s + ST - 2 < own) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kReq * (ST - 2)) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), in a form that the compiler counts with
        asm volatile("s_barrier" ::: "memory");
        if (s + ST - 1 < own) request(s + ST - 1);
        if (KG > 1 && s >= own) continue;
        const int buf = (group * ST + s % ST) * S::kBuf;
        u32x4 fa[2][TM], fw[2][TN];
        auto read = [&](int step) __attribute__((always_inline)) {
            const int off = buf + (((2 * step + h) ^ swz) * 16);
#pragma unroll
            for (int j = 0; j < TM; j++) fa[step & 1][j] = *reinterpret_cast<const u32x4*>(frag_a + off + j * 32 * kSlice);
#pragma unroll
            for (int i = 0; i < TN; i++) fw[step & 1][i] = *reinterpret_cast<const u32x4*>(frag_w + off + i * 32 * kSlice);
        };
        read(0);
        __builtin_amdgcn_sched_barrier(0);  // (its fragments are waited for alone)
#pragma unroll
        for (int step = 0; step < 4; step++) {
            if (step < 3) read(step + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < TN; i++)
#pragma unroll
                for (int j = 0; j < TM; j++) acc[i][j] = mma<T>(fw[step & 1][i], fa[step & 1][j], acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // The tile goes through LDS (register x of lane 32 h + n: output row 8 (x / 4) + 4 h + x % 4 of its block, token n), so
    // that the epilogue is one short loop in which a thread has four consecutive outputs of one token and the threads
    // of a wavefront store whole rows of the tile.
    constexpr int kPitch = S::kPitch, kQuads = kRowsW / 4, kTurn = S::kThreads / kQuads;  // (tokens at a time; threads past a whole number have none)
    float* tile_c = reinterpret_cast<float*>(lds);
    constexpr int kPart = 32 * WM * kPitch;  // floats of a group's pass
    const int q4 = 4 * (tid % kQuads), row = n0 + q4;  // (this thread's four rows are the same in every turn)
    int si = -1;
    for (int q = 0; q < out.nseg; q++)
        if (row >= out.seg[q].row0) si = q;
    const skn_dense_seg sg = out.seg[si < 0 ? 0 : si];
    // rows of the segment from here on
    const int left = row >= rows || (out.nseg && si < 0) ? 0 : out.nseg ? sg.row0 + sg.rows - row : out.resid_rows - row;
    const float4 b = bias && left > 0 ? *reinterpret_cast<const float4*>(bias + row) : make_float4(0.f, 0.f, 0.f, 0.f);
    const bool add = out.nseg == 0 && left >= 4;
    constexpr int kPasses = (32 * WM + kTurn - 1) / kTurn;
    const auto token = [&](int tl, int j) { return m0 + (tl >> 5) * 32 * TM + 32 * j + (tl & 31); };
#pragma unroll
    for (int j = 0; j < TM; j++) {
        __syncthreads();  // (the fragments, then the pass before this one, have been read)
#pragma unroll
        for (int i = 0; i < TN; i++)
#pragma unroll
            for (int g = 0; g < 4; g++)
                *reinterpret_cast<float4*>(tile_c + group * kPart + (32 * wv_m + r32) * kPitch + wn + 32 * i + 8 * g + 4 * h) =
                    make_float4(acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]);
        __syncthreads();
        if (left <= 0 || tid >= kTurn * kQuads) continue;
        const auto sums = [&](int tl) __attribute__((always_inline)) {
            float4 c = *reinterpret_cast<const float4*>(tile_c + tl * kPitch + q4);
#pragma unroll
            for (int k = 1; k < KG; k++) {
                const float4 d = *reinterpret_cast<const float4*>(tile_c + k * kPart + tl * kPitch + q4);
                c = make_float4(c.x + d.x, c.y + d.y, c.z + d.z, c.w + d.w);
            }
            return make_float4(c.x + b.x, c.y + b.y, c.z + b.z, c.w + b.w);
        };
        if (add) {
            // What the tile is added to is read four turns at a time (tokens past the last: the last, unused): one by one, every turn's load
            // waited for the store before it (128 x 64 tiles, 2048 x 2048 outputs 31.9 -> 30.1 us, a long k's 80.4 -> 78.7; all turns
            // at once take registers that two workgroups would share).
            for (int i0 = 0; i0 < kPasses; i0 += 4) {
                float4 old[4];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int tl = min(tid / kQuads + (i0 + i) * kTurn, 32 * WM - 1);
                    old[i] = *reinterpret_cast<const float4*>(out.resid + (int64_t)min(token(tl, j), m - 1) * out.ldr + row);
                }
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int tl = tid / kQuads + (i0 + i) * kTurn, t = token(tl, j);
                    if (tl >= 32 * WM || t >= m) continue;
                    const float4 v = sums(tl), x = old[i];
                    *reinterpret_cast<float4*>(out.resid + (int64_t)t * out.ldr + row) =
                        make_float4(fmaf(out.mult, v.x, x.x), fmaf(out.mult, v.y, x.y), fmaf(out.mult, v.z, x.z), fmaf(out.mult, v.w, x.w));
                }
            }
            continue;
        }
        for (int tl = tid / kQuads; tl < 32 * WM; tl += kTurn) {
            const int t = token(tl, j);
            if (t >= m) continue;
            const float4 c = sums(tl);
            float v[4] = {c.x, c.y, c.z, c.w};
            if (out.nseg == 0) {  // (less than four rows)
                float* p = out.resid + (int64_t)t * out.ldr + row;
                for (int e = 0; e < left; e++) p[e] = fmaf(out.mult, e == 0 ? v[0] : e == 1 ? v[1] : v[2], p[e]);
                continue;
            }
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = skn_dense_op(sg.op, v[e], sg.p0, sg.p1);
            if (si == out.mul_seg) {
                const int64_t from = (int64_t)out.mul_tokens[t] * out.mul_ld + out.mul_col + (row - sg.row0);
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] *= e < left ? skn_table_at(out.mul_table, out.mul_type, from + e) : 0.f;
            }
            const int64_t at = (int64_t)t * sg.ldo + (row - sg.row0);
            if (left >= 4 && sg.out_type == SKN_TYPE_F32) {
                *reinterpret_cast<float4*>((float*)sg.out + at) = make_float4(v[0], v[1], v[2], v[3]);
            } else if (left >= 4) {
                if (sg.out_type == SKN_TYPE_F16)
                    *reinterpret_cast<uint2*>((uint16_t*)sg.out + at) = make_uint2(half_bits(v[0]) | (half_bits(v[1]) << 16), half_bits(v[2]) | (half_bits(v[3]) << 16));
                else *reinterpret_cast<uint2*>((uint16_t*)sg.out + at) = make_uint2(skn_bf16_bits(v[0]) | ((uint32_t)skn_bf16_bits(v[1]) << 16),
                                                                                skn_bf16_bits(v[2]) | ((uint32_t)skn_bf16_bits(v[3]) << 16));
            } else {
                for (int e = 0; e < left; e++) {
                    const float f = e == 0 ? v[0] : e == 1 ? v[1] : v[2];
                    if (sg.out_type == SKN_TYPE_F32) ((float*)sg.out)[at + e] = f;
                    else ((uint16_t*)sg.out)[at + e] = sg.out_type == SKN_TYPE_F16 ? (uint16_t)half_bits(f) : skn_bf16_bits(f);
                }
            }
        }
    }
}

using Tile64x64 = Shape<2, 2, 1, 1, 3>;
using Tile32x64Split = Shape<1, 2, 1, 1, 3, 4>;  // for few outputs: more and shorter chains of slices
using Tile128x64 = Shape<2, 2, 2, 1, 3>;
using Tile128x128 = Shape<2, 2, 2, 2, 2>;
using Tile128x128Split = Shape<2, 2, 2, 2, 2, 2>;  // for one round of long rows: eight wavefronts, half of the slices each four
using Tile256x256 = Shape<4, 2, 2, 4, 2>;
using Tile256x192 = Shape<4, 2, 2, 3, 2>;
using Tile128x192 = Shape<2, 2, 2, 3, 2>;

template <typename T, typename S>
int launch_gemm(skn_ctx* ctx, const skn_dense_mat& w, const void* a, int lda, int m, const skn_dense_out& out) {
    const int tm = (m + S::kRowsA - 1) / S::kRowsA, tn = (w.rows + S::kRowsW - 1) / S::kRowsW, tiles = tm * tn;
    skn_launch(ctx, dense_gemm_kernel<T, S>, dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(S::kThreads), (size_t)S::kLds, (const uint8_t*)a,
               (int64_t)lda * (int64_t)sizeof(T), m, (const uint8_t*)w.w, (int64_t)w.k_pad * (int64_t)sizeof(T), w.rows,
               (int)(w.k_pad * sizeof(T) / kSlice), tm, tiles, w.bias, out);
    SKN_LAUNCH_CHECK(ctx);
    return SKN_OK;
}

template <typename T>
int pick_gemm(skn_ctx* ctx, const skn_dense_mat& w, const void* a, int lda, int m, const skn_dense_out& out) {
    int best = skn_dense_tile((int)sizeof(T), m, w.rows, w.k_pad, ctx->compute_units);
    if (ctx->opt_dense_tile > 0) best = ctx->opt_dense_tile - 1;
    switch (best) {
        case SKN_TILE_64x64: return launch_gemm<T, Tile64x64>(ctx, w, a, lda, m, out);
        case SKN_TILE_128x64: return launch_gemm<T, Tile128x64>(ctx, w, a, lda, m, out);
        case SKN_TILE_128x128: return launch_gemm<T, Tile128x128>(ctx, w, a, lda, m, out);
        case SKN_TILE_32x64_K4: return launch_gemm<T, Tile32x64Split>(ctx, w, a, lda, m, out);
        case SKN_TILE_256x192: return launch_gemm<T, Tile256x192>(ctx, w, a, lda, m, out);
        case SKN_TILE_128x192: return launch_gemm<T, Tile128x192>(ctx, w, a, lda, m, out);
        case SKN_TILE_128x128_K2: return launch_gemm<T, Tile128x128Split>(ctx, w, a, lda, m, out);
        default: return launch_gemm<T, Tile256x256>(ctx, w, a, lda, m, out);
    }
}

template <typename T, typename S>
int allow_lds(skn_ctx* ctx) {
    SKN_HIP(ctx, hipFuncSetAttribute((const void*)dense_gemm_kernel<T, S>, hipFuncAttributeMaxDynamicSharedMemorySize, S::kLds));
    return SKN_OK;
}

template <typename T>
int allow_all(skn_ctx* ctx) {
    SKN_TRY((allow_lds<T, Tile64x64>(ctx)));
    SKN_TRY((allow_lds<T, Tile32x64Split>(ctx)));
    SKN_TRY((allow_lds<T, Tile128x64>(ctx)));
    SKN_TRY((allow_lds<T, Tile128x128>(ctx)));
    SKN_TRY((allow_lds<T, Tile128x128Split>(ctx)));
    SKN_TRY((allow_lds<T, Tile256x192>(ctx)));
    SKN_TRY((allow_lds<T, Tile128x192>(ctx)));
    return allow_lds<T, Tile256x256>(ctx);
}

int dense_gemm_init(skn_ctx* ctx) {
    SKN_TRY(allow_all<uint16_t>(ctx));
    return allow_all<float>(ctx);
}
skn_family register_family(dense_gemm_init);

}  // namespace

int skn_dense_gemm(skn_ctx* ctx, const skn_dense_mat& w, const void* a, int lda, int m, const skn_dense_out& out) {
    SKN_REQUIRE(ctx, w.w && a && m > 0 && w.rows > 0 && w.rows % kDenseRowPad == 0 && w.k_pad > 0 && w.k_pad % kDenseColPad == 0, SKN_ERR_ARG,
                "dense GEMM: bad shape (%d tokens, %d x %d)", m, w.rows, w.k_pad);
    SKN_REQUIRE(ctx, lda >= w.k_pad && lda % kDenseColPad == 0, SKN_ERR_SHAPE, "dense GEMM: activation pitch %d for %d columns", lda, w.k_pad);
    SKN_REQUIRE(ctx, skn_dense_pitch_ok(w.type == SKN_TYPE_F32 ? 4 : 2, lda), SKN_ERR_SHAPE, "dense GEMM: rows of %d elements are too long", lda);
    SKN_REQUIRE(ctx, (((uintptr_t)w.w | (uintptr_t)a) & 15) == 0, SKN_ERR_ARG, "dense GEMM: operands must be 16-byte aligned");
    SKN_REQUIRE(ctx, out.nseg >= 0 && out.nseg <= kDenseMaxSegs && (out.nseg > 0 || out.resid), SKN_ERR_ARG, "dense GEMM: no output");
    for (int i = 0; i < out.nseg; i++)
        SKN_REQUIRE(ctx, out.seg[i].out && out.seg[i].row0 % kDenseRowPad == 0 && out.seg[i].ldo % 4 == 0 && ((uintptr_t)out.seg[i].out & 15) == 0 &&
                             out.seg[i].row0 + skn_pad_rows(out.seg[i].rows) <= w.rows && (i == 0 || out.seg[i].row0 > out.seg[i - 1].row0),
                    SKN_ERR_ARG, "dense GEMM: segment %d is misplaced", i);
    SKN_REQUIRE(ctx, out.mul_seg < 0 || (out.mul_table && out.mul_tokens), SKN_ERR_ARG, "dense GEMM: no table to multiply with");
    SKN_REQUIRE(ctx, out.nseg > 0 || (out.ldr % 4 == 0 && out.resid_rows <= w.rows && ((uintptr_t)out.resid & 15) == 0), SKN_ERR_ARG,
                "dense GEMM: bad residual rows");
    if (w.type == SKN_TYPE_BF16) return pick_gemm<uint16_t>(ctx, w, a, lda, m, out);
    if (w.type == SKN_TYPE_F32) return pick_gemm<float>(ctx, w, a, lda, m, out);
    return skn_fail(ctx, SKN_ERR_TYPE, "dense GEMM: weights of type %d (BF16 or F32)", w.type);
}
