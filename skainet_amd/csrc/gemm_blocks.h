// Prompt products of weights in blocks of 32 (Q8_0, Q4_0, Q4_1, Q5_0, Q5_1, Q5_K; Q4_K too, which skn_gemm_q sends here up to 32
// rows where gemm_few.h declines) behind the activation sources of the Q4_K one (internal to the library).
#pragma once
#include "common.h"

// True where skn_gemm_blocks_multi takes a matrix: one of these formats in rows of whole groups of 256 elements from a 16-byte
// aligned address, the kernels that unpack the blocks themselves not switched off, sizes within the 32-bit offsets they use.
bool skn_gemm_blocks_ok(const skn_ctx* ctx, int type, const void* w, int n, int k, int m);
// False where the general path, whose weight pass many rows share, is the faster one for a matrix that passes.  in_prompt: the
// activations are a decoder's fp32 rows, for which the general path has a norm, a conversion and an addition more.
bool skn_gemm_blocks_pay(int type, int n, int k, int m, bool in_prompt);

// One activation pass (bf16 rows, fp32 rows, or fp32 rows with RMSNorm inside the pass) for one to three matrices [n_i, k] of any
// of the formats; a matrix with `accumulate` set is added to its output.  Every matrix must pass skn_gemm_blocks_ok.
int skn_gemm_blocks_multi(skn_ctx* ctx, const int* types, const skn_gemm_seg* segs, int nseg, int k, const skn_gemm_src& src, int m);
