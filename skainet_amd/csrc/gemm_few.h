// Products of few bf16 activation rows with Q4_K, Q5_K, Q6_K, Q8_0 or Q4_0 weights in one launch, two where k is divided (internal to the library).
#pragma once
#include "common.h"

// True where skn_gemm_few takes a product and is the faster path for it.
bool skn_gemm_few_ok(const skn_ctx* ctx, int type, const void* w, int n, int k, int m);
// c[m, n] = a w^T; a: bf16 [m, k], 8-byte aligned; the product must pass skn_gemm_few_ok.
int skn_gemm_few(skn_ctx* ctx, int type, const void* w, int n, int k, const uint16_t* a_bf16, int m, float* c);
