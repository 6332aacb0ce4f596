// The step before the MoE: the residual add and RMSNorm that produce the
// expert input, with the router GEMV and the shared expert's gate GEMV fused into the
// norm's epilogue:
//   v = r + y (y optional),  x = bf16(v * rsqrt(mean(v^2) + eps) * w_norm)  (w_norm optional),
//   logits[t, e] = x[t] . W_router[e],  shared_logit[t] = x[t] . g.
// The reference runs these as separate dispatches (the norm, then linear(router),
// linear(shared_gate): Native/QwenNative/engine.mm:2074-2079, with the norm in the
// hyper-connection mix before it). Routing (wm_route_softmax_topk / wm_route_scored) follows
// on the device with no host step.
//
// Few tokens: one launch, the expert input built once per block in LDS. Grid (row blocks,
// token blocks); a block owns TB tokens and RB consecutive output rows
// (router rows, then the gate row as row E). Every block recomputes the norm of its TB
// tokens (r and y are L2-resident after the first block of a token group) and keeps x as
// a [TB][H] bf16 tile in LDS (TB up to 16, within 96 KB); row block 0 also writes x and
// r + y to HBM. Each wave takes rows wave, wave + 4, ...: a lane streams 16-byte chunks
// of the weight row once and
// applies each to the TB tokens' x chunks (V_DOT2_F32_BF16), then one wave reduction
// per token. More tokens: the norm and the GEMM as two launches (residual_norm_kernel).
#include <algorithm>
#include <cmath>

#include "gemm_bf16.h"
#include "moe_internal.h"

namespace wm {

// Statistics of v = r + y for tokens t0 .. t0 + nt, then the x tile [TB][stride] (uint4 =
// 8 bf16; tokens past nt are zero). The writer block also stores x and v to HBM. Ends with
// a block barrier.
template <int TB>
__device__ __forceinline__ void build_x_tile(const float* __restrict__ r, const uint16_t* __restrict__ y,
                                             const uint16_t* __restrict__ nw, int t0, int nt, int hidden, float eps,
                                             bool writer, uint16_t* __restrict__ x_out, float* __restrict__ r_out,
                                             uint4* tile, int stride, float* inv_s) {
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int chunks = hidden / 8;
  constexpr int QU = 8;  // float4 loads in flight per lane
  const int quads = hidden / 4;
  for (int t = wave; t < nt; t += 4) {
    const float4* rr = (const float4*)(r + (int64_t)(t0 + t) * hidden);
    const uint2* yy = y ? (const uint2*)(y + (int64_t)(t0 + t) * hidden) : nullptr;
    float ss = 0.0f;
    for (int q0 = lane; q0 < quads; q0 += 64 * QU) {
      float4 v[QU];
      uint2 b[QU];
#pragma unroll
      for (int j = 0; j < QU; ++j) {
        const int q = q0 + 64 * j;
        v[j] = q < quads ? rr[q] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        b[j] = (yy && q < quads) ? yy[q] : make_uint2(0, 0);
      }
#pragma unroll
      for (int j = 0; j < QU; ++j) {
        float4 u = v[j];
        u.x += bf16_bits_to_f32(b[j].x & 0xffffu);
        u.y += bf16_bits_to_f32(b[j].x >> 16);
        u.z += bf16_bits_to_f32(b[j].y & 0xffffu);
        u.w += bf16_bits_to_f32(b[j].y >> 16);
        ss += u.x * u.x + u.y * u.y + u.z * u.z + u.w * u.w;
      }
    }
    ss = segment_sum<64>(ss);
    if (lane == 0) inv_s[t] = rsqrtf(ss / (float)hidden + eps);
  }
  __syncthreads();
  // the tile, TU tokens at a time so their loads are in flight together
  constexpr int TU = TB < 4 ? TB : 4;
  for (int tb0 = 0; tb0 < TB; tb0 += TU) {
    for (int c = threadIdx.x; c < chunks; c += 256) {
      float4 ra[TU], rb[TU];
      uint4 yb[TU];
#pragma unroll
      for (int u = 0; u < TU; ++u) {
        const int t = tb0 + u;
        if (t < nt) {
          const float4* rr = (const float4*)(r + (int64_t)(t0 + t) * hidden) + 2 * c;
          ra[u] = rr[0];
          rb[u] = rr[1];
          yb[u] = y ? ((const uint4*)(y + (int64_t)(t0 + t) * hidden))[c] : make_uint4(0, 0, 0, 0);
        }
      }
      uint32_t nwv[4] = {0, 0, 0, 0};
      if (nw) {
        uint4 n4 = ((const uint4*)nw)[c];
        nwv[0] = n4.x, nwv[1] = n4.y, nwv[2] = n4.z, nwv[3] = n4.w;
      }
#pragma unroll
      for (int u = 0; u < TU; ++u) {
        const int t = tb0 + u;
        uint4* xt = tile + t * stride;
        if (t >= nt) {
          xt[c] = make_uint4(0, 0, 0, 0);
          continue;
        }
        const float inv = inv_s[t];
        float v[8] = {ra[u].x, ra[u].y, ra[u].z, ra[u].w, rb[u].x, rb[u].y, rb[u].z, rb[u].w};
        const uint32_t w4[4] = {yb[u].x, yb[u].y, yb[u].z, yb[u].w};
        uint32_t packed[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (y) {
            v[2 * j] += bf16_bits_to_f32(w4[j] & 0xffffu);
            v[2 * j + 1] += bf16_bits_to_f32(w4[j] >> 16);
          }
          float lo = v[2 * j] * inv, hi = v[2 * j + 1] * inv;
          if (nw) {
            lo *= bf16_bits_to_f32(nwv[j] & 0xffffu);
            hi *= bf16_bits_to_f32(nwv[j] >> 16);
          }
          packed[j] = (uint32_t)f32_to_bf16_bits(lo) | ((uint32_t)f32_to_bf16_bits(hi) << 16);
        }
        const uint4 xv = make_uint4(packed[0], packed[1], packed[2], packed[3]);
        xt[c] = xv;
        if (writer) {
          const int64_t row = (int64_t)(t0 + t) * hidden;
          ((uint4*)(x_out + row))[c] = xv;
          if (r_out) {
            float4* ro = (float4*)(r_out + row) + 2 * c;
            ro[0] = make_float4(v[0], v[1], v[2], v[3]);
            ro[1] = make_float4(v[4], v[5], v[6], v[7]);
          }
        }
      }
    }
  }
  __syncthreads();
}

// Output row e: a router row, or the shared gate as row `experts`.
__device__ __forceinline__ const uint4* weight_row(const uint16_t* router, const uint16_t* gate, int experts,
                                                   int hidden, int e) {
  return (const uint4*)(e < experts ? router + (int64_t)e * hidden : gate);
}

__device__ __forceinline__ void store_row(float* logits, float* shared_logit, int experts, int t, int e, float v) {
  if (e < experts) logits[(int64_t)t * experts + e] = v;
  else shared_logit[t] = v;
}

// Few tokens (decode): a block owns rows_per_block rows (4: one per wave), and each wave
// loads its row's first NR_PREFETCH chunks per lane before the norm, so the weight stream
// overlaps the statistics and the tile.
constexpr int NR_PREFETCH = 8;

template <int TB>
__global__ void __launch_bounds__(256) norm_router_kernel(
    const float* __restrict__ r, const uint16_t* __restrict__ y, const uint16_t* __restrict__ nw, int tokens,
    int hidden, float eps, const uint16_t* __restrict__ router, int experts, const uint16_t* __restrict__ gate,
    int rows_per_block, uint16_t* __restrict__ x_out, float* __restrict__ r_out, float* __restrict__ logits,
    float* __restrict__ shared_logit) {
  extern __shared__ uint4 x_tile[];  // [TB][hidden / 8]
  __shared__ float inv_s[TB];
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int t0 = blockIdx.y * TB;
  const int nt = min(TB, tokens - t0);
  const int chunks = hidden / 8;
  const int rows = experts + (gate ? 1 : 0);
  const int first = blockIdx.x * rows_per_block;
  const int last = min(rows, first + rows_per_block);
  const int e0 = first + wave;

  uint4 pre[NR_PREFETCH];
  if (e0 < last) {
    const uint4* w = weight_row(router, gate, experts, hidden, e0);
#pragma unroll
    for (int j = 0; j < NR_PREFETCH; ++j)
      if (lane + 64 * j < chunks) pre[j] = w[lane + 64 * j];
  }
  build_x_tile<TB>(r, y, nw, t0, nt, hidden, eps, blockIdx.x == 0, x_out, r_out, x_tile, chunks, inv_s);

  for (int e = e0; e < last; e += 4) {
    const uint4* w = weight_row(router, gate, experts, hidden, e);
    float acc[TB];
#pragma unroll
    for (int t = 0; t < TB; ++t) acc[t] = 0.0f;
    auto apply = [&](uint4 wv, int c) {
#pragma unroll
      for (int t = 0; t < TB; ++t) {
        uint4 xv = x_tile[t * chunks + c];
        float a = acc[t];
        a = dot2_bf16(bits_to_bf16x2(wv.x), bits_to_bf16x2(xv.x), a);
        a = dot2_bf16(bits_to_bf16x2(wv.y), bits_to_bf16x2(xv.y), a);
        a = dot2_bf16(bits_to_bf16x2(wv.z), bits_to_bf16x2(xv.z), a);
        a = dot2_bf16(bits_to_bf16x2(wv.w), bits_to_bf16x2(xv.w), a);
        acc[t] = a;
      }
    };
#pragma unroll
    for (int j = 0; j < NR_PREFETCH; ++j) {
      const int c = lane + 64 * j;
      if (c < chunks) apply(e == e0 ? pre[j] : w[c], c);
    }
    for (int c = lane + 64 * NR_PREFETCH; c < chunks; c += 64) apply(w[c], c);
#pragma unroll
    for (int t = 0; t < TB; ++t) {
      float s = segment_sum<64>(acc[t]);
      if (lane == t && t < nt) store_row(logits, shared_logit, experts, t0 + t, e, s);
    }
  }
}

// The packed router: [groups][hidden / 32][64 lanes] uint4, lane l of group g and step s
// holding row 16 g + l % 16 (router rows, then the gate row, then zeros; one spare zero
// group follows when the gate is packed), 8 values from column 32 s + 8 (l / 16).
__global__ void __launch_bounds__(256) repack_router_kernel(const uint4* __restrict__ router,
                                                            const uint4* __restrict__ gate, int experts, int hidden,
                                                            int64_t total, uint4* __restrict__ packed) {
  const int steps = hidden / 32, chunks = hidden / 8;
  for (int64_t o = blockIdx.x * 256 + threadIdx.x; o < total; o += (int64_t)gridDim.x * 256) {
    const int lane = (int)(o % 64);
    const int64_t gs = o / 64;
    const int st = (int)(gs % steps), g = (int)(gs / steps);
    const int row = 16 * g + lane % 16, chunk = 4 * st + lane / 16;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (row < experts) v = router[(int64_t)row * chunks + chunk];
    else if (row == experts && gate) v = gate[chunk];
    packed[o] = v;
  }
}

__device__ __forceinline__ float4 load_nt(const float4* p) {
  const wm_f32x4 v = __builtin_nontemporal_load(reinterpret_cast<const wm_f32x4*>(p));
  return make_float4(v[0], v[1], v[2], v[3]);
}
typedef uint32_t nr_u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint2 load_nt(const uint2* p) {
  const nr_u32x2 v = __builtin_nontemporal_load(reinterpret_cast<const nr_u32x2*>(p));
  return make_uint2(v.x, v.y);
}
// Many tokens: the norm as a kernel of its own (a block per token), then the GEMM of
// gemm_bf16.hip on its x. The norm passes r, y, x and r + y through memory once, which is
// what bounds a long prompt (r and y are read once: non-temporal loads, 53.8 -> 50.7 us for
// 4000 tokens of 2560 with 512 experts); the shared gate's dot product rides on the row in
// registers. In one launch every block held 8 to 32 tokens' whole rows in LDS for the GEMM and
// passed all the router rows: 120 us for the same 4000 tokens.
// Q: float4 values per thread (hidden <= 1024 Q).
template <int Q>
__global__ void __launch_bounds__(256) residual_norm_kernel(const float* __restrict__ r, const uint16_t* __restrict__ y,
                                                            const uint16_t* __restrict__ nw, int hidden, float eps,
                                                            const uint16_t* __restrict__ gate,
                                                            uint16_t* __restrict__ x_out, float* __restrict__ r_out,
                                                            float* __restrict__ shared_logit) {
  __shared__ float part[2][4];
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int quads = hidden / 4;
  const int64_t row = (int64_t)blockIdx.x * hidden;
  const float4* rr = (const float4*)(r + row);
  const uint2* yy = y ? (const uint2*)(y + row) : nullptr;
  float4 v[Q];
  uint2 b[Q];
#pragma unroll
  for (int j = 0; j < Q; ++j) {
    const int q = min((int)threadIdx.x + 256 * j, quads - 1);
    v[j] = load_nt(rr + q);
    b[j] = yy ? load_nt(yy + q) : make_uint2(0, 0);
  }
  float ss = 0.0f;
#pragma unroll
  for (int j = 0; j < Q; ++j) {
    if (yy) {  // without y, v is r with the sign of its zeros
      v[j].x += bf16_bits_to_f32(b[j].x & 0xffffu);
      v[j].y += bf16_bits_to_f32(b[j].x >> 16);
      v[j].z += bf16_bits_to_f32(b[j].y & 0xffffu);
      v[j].w += bf16_bits_to_f32(b[j].y >> 16);
    }
    if ((int)threadIdx.x + 256 * j < quads) ss += v[j].x * v[j].x + v[j].y * v[j].y + v[j].z * v[j].z + v[j].w * v[j].w;
  }
  ss = segment_sum<64>(ss);
  if (lane == 0) part[0][wave] = ss;
  __syncthreads();
  // In 64 bits up to x's rounding: memory bounds the kernel, and a row's values share the error of `inv`, which
  // moves them over bf16 rounding boundaries together: 4 x 4000 rows of 2560, 93 values off by a bf16 step, 334 in 32 bits.
  const double inv =
      1.0 / sqrt((((double)part[0][0] + part[0][1]) + ((double)part[0][2] + part[0][3])) / hidden + (double)eps);
  float dot = 0.0f;
#pragma unroll
  for (int j = 0; j < Q; ++j) {
    const int q = threadIdx.x + 256 * j;
    if (q >= quads) continue;
    double f[4] = {v[j].x * inv, v[j].y * inv, v[j].z * inv, v[j].w * inv};
    if (nw) {
      const uint2 n = ((const uint2*)nw)[q];
      f[0] *= bf16_bits_to_f32(n.x & 0xffffu);
      f[1] *= bf16_bits_to_f32(n.x >> 16);
      f[2] *= bf16_bits_to_f32(n.y & 0xffffu);
      f[3] *= bf16_bits_to_f32(n.y >> 16);
    }
    const uint2 xv =
        make_uint2((uint32_t)f32_to_bf16_bits((float)f[0]) | ((uint32_t)f32_to_bf16_bits((float)f[1]) << 16),
                   (uint32_t)f32_to_bf16_bits((float)f[2]) | ((uint32_t)f32_to_bf16_bits((float)f[3]) << 16));
    ((uint2*)(x_out + row))[q] = xv;
    if (r_out) ((float4*)(r_out + row))[q] = v[j];
    if (gate) {
      const uint2 g = ((const uint2*)gate)[q];
      dot = dot2_bf16(bits_to_bf16x2(xv.x), bits_to_bf16x2(g.x), dot);
      dot = dot2_bf16(bits_to_bf16x2(xv.y), bits_to_bf16x2(g.y), dot);
    }
  }
  if (gate) {
    dot = segment_sum<64>(dot);
    if (lane == 0) part[1][wave] = dot;
    __syncthreads();
    if (threadIdx.x == 0) shared_logit[blockIdx.x] = (part[1][0] + part[1][1]) + (part[1][2] + part[1][3]);
  }
}

constexpr int NORM_MAX_HIDDEN = 10240;

static void residual_norm(const float* r, const uint16_t* y, const uint16_t* nw, int tokens, int hidden, float eps,
                          const uint16_t* gate, uint16_t* x, float* r_out, float* shared_logit, hipStream_t s) {
#define WM_RN(Q) hipLaunchKernelGGL(residual_norm_kernel<Q>, dim3(tokens), dim3(256), 0, s, r, y, nw, hidden, eps, gate, \
                                    x, r_out, shared_logit)
  switch ((hidden + 1023) / 1024) {
    case 1: WM_RN(1); break;
    case 2: WM_RN(2); break;
    case 3: WM_RN(3); break;
    case 4: WM_RN(4); break;
    case 5: WM_RN(5); break;
    case 6: WM_RN(6); break;
    case 7: WM_RN(7); break;
    case 8: WM_RN(8); break;
    default: WM_RN(10); break;
  }
#undef WM_RN
  check_launch("residual_norm");
}

// The dot-product path's token block: the largest whose x tile (plus the 64-byte
// statistics array) fits 96 KB of LDS, no larger than the tokens.
static int pick_token_block(int tokens, int hidden) {
  const int fit = (96 * 1024 - 64) / (hidden * 2);
  for (int tb : {16, 8, 4, 2}) if (tb <= fit && tokens >= tb) return tb;
  return 1;
}

// Whether the two launches are faster than the fused kernel (us, fused / two launches). Up to hidden 6144 from 8
// tokens, where a fused block builds the rows of 8 or 16 tokens one after another: 2560, 512 experts: 4 tokens
// 9.1 / 10.9, 8 tokens 15.8 / 11.6; 4160, 512 experts, 16 tokens 26.5 / 15.6; 5120, 384: 24.4 / 19.2. Wider rows, whose
// fused blocks hold 4 tokens and whose GEMM takes as long as its K, once those blocks pass one round of
// the chip (about 20 us a round): hidden 7168: 32 experts 96 tokens (240 blocks of 512) 20.2 / 24.2, 256 experts 24 tokens
// (390) 22.2 / 24.0; 9600: 64 experts 96 tokens (408) 27.8 / 29.5, 128 tokens (544) 46 / 29.7.
static bool norm_gemm_wins(int tokens, int hidden, int rows) {
  if (hidden <= 6144) return tokens >= 8;
  const int tb = pick_token_block(tokens, hidden);
  const int64_t blocks = (int64_t)((rows + 3) / 4) * ((tokens + tb - 1) / tb);
  return blocks > 256 * (160 * 1024 / (tb * hidden * 2 + 64));  // CUs, blocks a CU by their LDS
}

}  // namespace wm

using namespace wm;

extern "C" {

WM_EXPORT size_t wm_router_packed_bytes(int32_t experts, int32_t hidden, int32_t has_gate) {
  if (experts < 1 || hidden < 32 || hidden % 32) return 0;
  // one spare zero group when the gate row is packed, so the size alone tells whether it is
  const int g = has_gate ? 1 : 0;
  return (size_t)((experts + g + 15) / 16 + g) * 16 * hidden * 2;
}

WM_EXPORT int wm_repack_router(const void* router, const void* shared_gate, int32_t experts, int32_t hidden,
                               void* packed, void* stream) {
  return guarded([&] {
    if (experts < 1 || hidden < 32 || hidden % 32) fail("wm_repack_router: hidden must be a multiple of 32");
    if (!router || !packed) fail("wm_repack_router: null pointer");
    for (const void* p : {router, shared_gate, (const void*)packed})
      if (p && ((uintptr_t)p % 16)) fail("wm_repack_router: tensors must be 16-byte aligned");
    const int64_t total = (int64_t)wm_router_packed_bytes(experts, hidden, shared_gate != nullptr) / 16;
    const int blocks = (int)std::min<int64_t>((total + 255) / 256, 4096);
    hipLaunchKernelGGL(repack_router_kernel, dim3(blocks), dim3(256), 0, as_stream(stream), (const uint4*)router,
                       (const uint4*)shared_gate, experts, hidden, total, (uint4*)packed);
    check_launch("repack_router");
  });
}

WM_EXPORT int wm_norm_router(const float* residual, const void* y, const void* norm_weight, int32_t tokens,
                             int32_t hidden, float eps, const void* router, int32_t experts, const void* shared_gate,
                             const void* router_packed, size_t router_packed_bytes, void* x,
                             float* residual_out, float* logits, float* shared_logit, void* stream) {
  return guarded([&] {
    if (tokens < 0) fail("wm_norm_router: negative token count");
    if (hidden < 8 || hidden % 8 || hidden * 2 > 64 * 1024) fail("wm_norm_router: hidden must be a multiple of 8 up to 32768");
    if (experts < 1) fail("wm_norm_router: experts must be at least 1");
    if ((shared_gate == nullptr) != (shared_logit == nullptr))
      fail("wm_norm_router: shared_gate and shared_logit go together");
    if (tokens == 0) return;
    if (!residual || !router || !x || !logits) fail("wm_norm_router: null pointer");
    // Row block 0 writes x and v while other blocks still read residual and y.
    auto overlap = [](const void* p, size_t pn, const void* q, size_t qn) {
      const char *a = (const char*)p, *b = (const char*)q;
      return p && q && a < b + qn && b < a + pn;
    };
    const size_t n4 = (size_t)tokens * hidden * sizeof(float), n2 = (size_t)tokens * hidden * 2;
    if (overlap(residual_out, n4, residual, n4) || overlap(residual_out, n4, y, n2))
      fail("wm_norm_router: residual_out must not overlap residual or y (other blocks still read them)");
    if (overlap(x, n2, residual, n4) || overlap(x, n2, y, n2))
      fail("wm_norm_router: x must not overlap residual or y (other blocks still read them)");
    if (router_packed && (hidden % 32 || router_packed_bytes != wm_router_packed_bytes(experts, hidden, shared_gate != nullptr)))
      fail("wm_norm_router: the packed router does not match experts, hidden and the shared gate (wm_router_packed_bytes)");
    for (const void* p : {(const void*)residual, y, norm_weight, router, shared_gate, router_packed, (const void*)x,
                          (const void*)residual_out})
      if (p && ((uintptr_t)p % 16)) fail("wm_norm_router: tensors must be 16-byte aligned");
    hipStream_t s = as_stream(stream);
    const int rows = experts + (shared_gate ? 1 : 0);
    if (hidden <= NORM_MAX_HIDDEN && gemm_bf16_fits(x, router, hidden) && norm_gemm_wins(tokens, hidden, rows)) {
      residual_norm(residual, (const uint16_t*)y, (const uint16_t*)norm_weight, tokens, hidden, eps,
                    (const uint16_t*)shared_gate, (uint16_t*)x, residual_out, shared_logit, s);
      GemmArgs g{};
      g.x = (const uint16_t*)x;
      g.w = (const uint16_t*)router;
      g.tokens = tokens;
      g.k = hidden;
      g.n = experts;
      g.out = logits;
      gemm_bf16(GEMM_F32, g, s);
      return;
    }
    const int tb = pick_token_block(tokens, hidden);
    // The rows spread over many blocks (4 per block, one per wave), as few tokens leave
    // the weight stream as the only work.
    const int token_blocks = (tokens + tb - 1) / tb;
    if (token_blocks > 65535) fail("wm_norm_router: too many tokens for one call");
    const int rows_per_block = 4;
    dim3 grid((rows + rows_per_block - 1) / rows_per_block, token_blocks);
    const size_t lds = (size_t)tb * hidden * 2;
#define WM_NR(TB) hipLaunchKernelGGL(norm_router_kernel<TB>, grid, dim3(256), lds, s, residual, (const uint16_t*)y, \
                                     (const uint16_t*)norm_weight, tokens, hidden, eps, (const uint16_t*)router, experts, \
                                     (const uint16_t*)shared_gate, rows_per_block, (uint16_t*)x, residual_out, logits, \
                                     shared_logit)
    switch (tb) {
      case 16: WM_NR(16); break;
      case 8: WM_NR(8); break;
      case 4: WM_NR(4); break;
      case 2: WM_NR(2); break;
      default: WM_NR(1); break;
    }
#undef WM_NR
    check_launch("norm_router");
  });
}

}  // extern "C"
