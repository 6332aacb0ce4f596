// The reference's bf16 shared expert on the device:
//   y[t] = add[t] + g(t) * down(bf16(silu(x[t] . Wg^T) * (x[t] . Wu^T))),
//   g(t) = sigmoid(x[t] . gate_vec) (1 without a gate vector),
// the Qwen MLP (runtime/deepseek_v4_ssd/qwen4_exp.py:763-771) gated by
// shared_expert_gate (:1002-1003, :1045) and added to the routed combine; the native
// engine runs the same three linears with a mul_silu (Native/QwenNative/engine.mm:2075-2079).
// Weights are bf16 [I, H] (gate, up) and [H, I] (down), y = x W^T as mlx nn.Linear.
//
// Up to 5 tokens (decode): two GEMV kernels, a wave per intermediate row (gate and up rows)
// and a wave per output row, up to four 16-byte chunks of each row and of every token in flight: as many as
// the row has for a lane, since the ones past its end are loads too (96/32, 1 token: 6.0 us, 6.4 with four; 2560/640,
// 4 tokens 10.4, 11.2).
// More: the bf16 GEMM of gemm_bf16.hip twice, with the SwiGLU and the tokens' gate values in
// the first launch and the gate and add in the second.
// Measured (hidden 2560, intermediate 640): 8 tokens 24.3 us as GEMVs that looped over the
// tokens, now 14.6; 301 tokens about 290 us as three GEMMs with separate activation, gate and
// output passes, now 23; 2048 tokens 430, now 49.
#include <cmath>

#include "gemm_bf16.h"

namespace wm {

// The widths that the interface takes at 64 or more tokens: a bound of an earlier GEMM that held whole token
// rows in LDS, which the present kernels do not need; lifting it is a change of the interface.
constexpr int MLP_MAX_WIDTH = 9568;

// Tokens of the GEMVs (5 tokens, GEMVs / GEMMs, us: 2048/512 9.3/13.2, 2560/640 11.8/15.3, 7168/2048 32.3/32.4,
// 96/32 7.9/6.5).
static int mlp_gemv_max_tokens(int hidden) { return hidden <= 512 ? 4 : 5; }

// dot of 8 bf16 (one 16-byte chunk) against 8 bf16
__device__ __forceinline__ float dot8_bf16(uint4 a, uint4 b, float acc) {
  acc = dot2_bf16(bits_to_bf16x2(a.x), bits_to_bf16x2(b.x), acc);
  acc = dot2_bf16(bits_to_bf16x2(a.y), bits_to_bf16x2(b.y), acc);
  acc = dot2_bf16(bits_to_bf16x2(a.z), bits_to_bf16x2(b.z), acc);
  return dot2_bf16(bits_to_bf16x2(a.w), bits_to_bf16x2(b.w), acc);
}

// sigmoid(x[t] . v) by one wave (v may be null: 1).
__device__ __forceinline__ float wave_gate(const uint16_t* __restrict__ xr, const uint16_t* __restrict__ v, int hidden,
                                           int lane) {
  if (!v) return 1.0f;
  float a = 0.0f;
  for (int c = lane; c < hidden / 8; c += 64)
    a = dot8_bf16(reinterpret_cast<const uint4*>(xr)[c], reinterpret_cast<const uint4*>(v)[c], a);
  a = segment_sum<64>(a);
  return 1.0f / (1.0f + __expf(-a));
}

// Dot products of R weight rows with the rows of TMAX tokens, 64 chunks a step, UNROLL
// steps in flight; chunks past the end read the last one and are not used.
template <int TMAX, int R, int UNROLL>
__device__ __forceinline__ void wave_dots(const uint4* const (&wr)[R], const uint4* __restrict__ x, int tokens,
                                          int chunks, int lane, float (&acc)[R][TMAX]) {
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int t = 0; t < TMAX; ++t) acc[r][t] = 0.0f;
  for (int c0 = lane; c0 - lane < chunks; c0 += 64 * UNROLL) {
    uint4 wv[UNROLL][R], xv[UNROLL][TMAX];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int c = min(c0 + 64 * u, chunks - 1);
#pragma unroll
      for (int r = 0; r < R; ++r) wv[u][r] = gload16(&wr[r][c]);
#pragma unroll
      for (int t = 0; t < TMAX; ++t) xv[u][t] = gload16(&x[(int64_t)min(t, tokens - 1) * chunks + c]);
    }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      if (c0 + 64 * u >= chunks) continue;
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int t = 0; t < TMAX; ++t) acc[r][t] = dot8_bf16(wv[u][r], xv[u][t], acc[r][t]);
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int t = 0; t < TMAX; ++t) acc[r][t] = segment_sum<64>(acc[r][t]);
}

// grid: ceil(I / 4) + 1; wave w of block b owns intermediate row i = 4 b + w; the last block
// the tokens' gate values.
template <int TMAX, int UNROLL>
__global__ void __launch_bounds__(256) mlp_gate_up_gemv_kernel(const uint16_t* __restrict__ x, int tokens, int hidden,
                                                               int inter, const uint16_t* __restrict__ wg,
                                                               const uint16_t* __restrict__ wu,
                                                               const uint16_t* __restrict__ gate_vec,
                                                               uint16_t* __restrict__ act, float* __restrict__ gate) {
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int i = blockIdx.x * 4 + wave;
  if (blockIdx.x == gridDim.x - 1) {
    for (int t = wave; t < tokens; t += 4) {
      const float g = wave_gate(x + (int64_t)t * hidden, gate_vec, hidden, lane);
      if (lane == 0) gate[t] = g;
    }
    return;
  }
  if (i >= inter) return;
  const uint4* rows[2] = {reinterpret_cast<const uint4*>(wg + (int64_t)i * hidden),
                          reinterpret_cast<const uint4*>(wu + (int64_t)i * hidden)};
  float acc[2][TMAX];
  wave_dots<TMAX, 2, UNROLL>(rows, reinterpret_cast<const uint4*>(x), tokens, hidden / 8, lane, acc);
#pragma unroll
  for (int t = 0; t < TMAX; ++t)
    if (t < tokens && lane == 0) act[(int64_t)t * inter + i] = f32_to_bf16_bits(silu(acc[0][t]) * acc[1][t]);
}

// grid: ceil(H / 4); wave w of block b owns output row o = 4 b + w.
template <int TMAX, int UNROLL>
__global__ void __launch_bounds__(256) mlp_down_gemv_kernel(const uint16_t* __restrict__ act, int tokens, int hidden,
                                                            int inter, const uint16_t* __restrict__ wd,
                                                            const float* __restrict__ gate, const uint16_t* add,
                                                            uint16_t* y) {
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int o = blockIdx.x * 4 + wave;
  if (o >= hidden) return;
  const uint4* rows[1] = {reinterpret_cast<const uint4*>(wd + (int64_t)o * inter)};
  float acc[1][TMAX];
  wave_dots<TMAX, 1, UNROLL>(rows, reinterpret_cast<const uint4*>(act), tokens, inter / 8, lane, acc);
#pragma unroll
  for (int t = 0; t < TMAX; ++t)
    if (t < tokens && lane == 0) {
      float v = gate[t] * acc[0][t];
      if (add) v += bf16_bits_to_f32(add[(int64_t)t * hidden + o]);
      y[(int64_t)t * hidden + o] = f32_to_bf16_bits(v);
    }
}

static size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

struct MlpLayout {
  size_t gate, act, total;
};

static MlpLayout mlp_layout(int tokens, int hidden, int inter) {
  MlpLayout p{};
  size_t at = 0;
  const size_t T = tokens > 0 ? (size_t)tokens : 1;
  p.gate = at; at += align256(sizeof(float) * T);
  p.act = at;  at += align256(sizeof(uint16_t) * T * inter);
  p.total = at;
  return p;
}

}  // namespace wm

using namespace wm;

extern "C" {

WM_EXPORT size_t wm_mlp_bf16_workspace_size(int32_t tokens, int32_t hidden, int32_t inter) {
  if (tokens < 0 || hidden < 1 || inter < 1) return 0;
  return mlp_layout(tokens, hidden, inter).total;
}

WM_EXPORT int wm_mlp_bf16(const void* x, int32_t tokens, int32_t hidden, int32_t inter, const void* gate_w,
                          const void* up_w, const void* down_w, const void* gate_vec, const void* add, void* y,
                          void* workspace, size_t workspace_bytes, void* stream) {
  return guarded([&] {
    if (tokens < 0 || hidden < 32 || hidden % 32 || inter < 32 || inter % 32)
      fail("wm_mlp_bf16: hidden and intermediate must be positive multiples of 32");
    if (tokens == 0) return;
    if (!x || !gate_w || !up_w || !down_w || !y || !workspace) fail("wm_mlp_bf16: null pointer");
    for (const void* p : {x, gate_w, up_w, down_w, gate_vec, add, (const void*)y, (const void*)workspace})
      if ((uintptr_t)p % 16) fail("wm_mlp_bf16: every tensor must be 16-byte aligned");
    const MlpLayout p = mlp_layout(tokens, hidden, inter);
    if (workspace_bytes < p.total) fail("wm_mlp_bf16: workspace too small");
    if (tokens >= 64 && (hidden > MLP_MAX_WIDTH || inter > MLP_MAX_WIDTH))
      fail("wm_mlp_bf16: hidden or intermediate too large at 64 or more tokens (at most " +
           std::to_string(MLP_MAX_WIDTH) + ")");
    hipStream_t s = as_stream(stream);
    uint8_t* ws = (uint8_t*)workspace;
    float* gate = (float*)(ws + p.gate);
    uint16_t* act = (uint16_t*)(ws + p.act);
    const uint16_t *xb = (const uint16_t*)x, *gv = (const uint16_t*)gate_vec, *ab = (const uint16_t*)add;
    if (tokens <= mlp_gemv_max_tokens(hidden)) {
#define WM_GU(T, U)                                                                                                \
  hipLaunchKernelGGL((mlp_gate_up_gemv_kernel<T, U>), dim3((inter + 3) / 4 + 1), dim3(256), 0, s, xb, tokens, hidden, inter, \
                     (const uint16_t*)gate_w, (const uint16_t*)up_w, gv, act, gate)
#define WM_DN(T, U)                                                                                                \
  hipLaunchKernelGGL((mlp_down_gemv_kernel<T, U>), dim3((hidden + 3) / 4), dim3(256), 0, s, act, tokens, hidden, inter,    \
                     (const uint16_t*)down_w, gate, ab, (uint16_t*)y)
#define WM_MLP(T)                                                                                                  \
  do {                                                                                                             \
    if (hidden <= 512) WM_GU(T, 1);                                                                                \
    else if (hidden <= 1024) WM_GU(T, 2);                                                                          \
    else WM_GU(T, 4);                                                                                              \
    check_launch("mlp_gate_up_gemv");                                                                              \
    if (inter <= 512) WM_DN(T, 1);                                                                                 \
    else if (inter <= 1024) WM_DN(T, 2);                                                                           \
    else WM_DN(T, 4);                                                                                              \
    check_launch("mlp_down_gemv");                                                                                 \
  } while (0)
      if (tokens <= 1) WM_MLP(1);
      else if (tokens <= 2) WM_MLP(2);
      else if (tokens <= 4) WM_MLP(4);
      else WM_MLP(5);
#undef WM_MLP
#undef WM_DN
#undef WM_GU
      return;
    }
    GemmArgs g{};
    g.x = xb;
    g.w = (const uint16_t*)gate_w;
    g.w2 = (const uint16_t*)up_w;
    g.tokens = tokens;
    g.k = hidden;
    g.n = inter;
    g.out16 = act;
    g.vec = gv;
    g.vec_out = gate;
    gemm_bf16(GEMM_SWIGLU, g, s);
    GemmArgs d{};
    d.x = act;
    d.w = (const uint16_t*)down_w;
    d.tokens = tokens;
    d.k = inter;
    d.n = hidden;
    d.out16 = (uint16_t*)y;
    d.gate = gate;
    d.add = ab;
    gemm_bf16(GEMM_DOWN, d, s);
  });
}

}  // extern "C"
