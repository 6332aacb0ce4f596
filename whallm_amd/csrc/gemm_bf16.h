// The bf16 GEMM of the router linear, the norm-router and the bf16 shared expert
// (gemm_bf16.hip): C[t, n] = X[t] . W[n], fp32 sums of bf16 products.
#pragma once

#include "wm_common.h"

namespace wm {

// What happens to the sums.
enum GemmEpilogue {
  GEMM_F32,     // out[t, n] = c
  GEMM_SWIGLU,  // act[t, n] = bf16(silu(x . w[n]) * (x . w2[n]))
  GEMM_DOWN,    // y[t, n] = bf16(add[t, n] + gate[t] * c)  (add optional)
};

struct GemmArgs {
  const uint16_t* x;       // [tokens, k] bf16
  const uint16_t* w;       // [n, k] bf16 (GEMM_SWIGLU: the gate rows)
  const uint16_t* w2;      // GEMM_SWIGLU: the up rows [n, k]
  int tokens, k, n;
  float* out;              // GEMM_F32
  int out_vec;             // set by gemm_bf16
  uint16_t* out16;         // GEMM_SWIGLU, GEMM_DOWN
  const float* gate;       // GEMM_DOWN: [tokens]
  const uint16_t* add;     // GEMM_DOWN: [tokens, n] or null
  const uint16_t* vec;     // GEMM_SWIGLU: [k] or null; vec_out[t] = sigmoid(x[t] . vec), 1 without vec
  float* vec_out;          // GEMM_SWIGLU: [tokens] (may be null)
};

// Whether the GEMM takes these operands: rows of a multiple of 32 values, 16-byte aligned.
bool gemm_bf16_fits(const void* x, const void* w, int k);
void gemm_bf16(GemmEpilogue ep, const GemmArgs& a, hipStream_t s);

}  // namespace wm
