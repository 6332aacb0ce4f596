// bf16 GEMM for the linears around the experts: C[t, n] = X[t] . W[n] (both operands with K
// contiguous), fp32 accumulation, epilogues in gemm_bf16.h.
//
// The outputs are few (512 router rows, 640 intermediate columns), so what bounds these calls
// is how many of the 256 CUs get work and how many bytes of rows one block draws, not the
// matrix rate. Three kernels (the line between them: launch(), below):
//
//   small : a block owns 16 outputs x 16 tokens and its 8 waves split K (64-wide chunks
//           w, w + 8, ...), each lane loading its fragments straight from memory, four chunks
//           in flight; the partial tiles meet in LDS, summed in wave order.
//   split : a block of 4 waves owns 32 x 32 and the waves split each 128-wide K step.
//   tiled : a block of 4 waves owns a square tile of 64 or 128 outputs x tokens.
//
// split and tiled take their K steps through an LDS ring of direct loads (pieces of 16 bytes
// XOR-swizzled by row, so that a ds_read_b128 cycle's 8 rows fall on distinct banks) and run
// v_mfma_f32_32x32x16_bf16 on them. The kernel before these held 8 to 32 tokens' whole rows
// in LDS and passed every weight row by each block: 2 to 250 blocks of a serial chain. For 2048
// tokens of 2560 values and 512 outputs it took 127 us, now 17; 301 tokens of 2048: 91, now 10.
//
// Block b runs on XCD b % 8. small and split: an XCD takes every eighth output tile with all
// its token tiles, so a weight row is fetched into one L2; tiled: see TileMap.
#include "gemm_bf16.h"

#include "lds_dma.h"

namespace wm {
namespace gb {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// sigmoid(x[t] . vec) (1 without vec) of token t by one wave.
__device__ __forceinline__ void token_gate(const GemmArgs& a, int t, int lane) {
  float g = 1.0f;
  if (a.vec) {
    const uint4* xr = reinterpret_cast<const uint4*>(a.x + (int64_t)t * a.k);
    const uint4* vr = reinterpret_cast<const uint4*>(a.vec);
    float s = 0.0f;
    for (int c = lane; c < a.k / 8; c += 64) {
      const uint4 p = xr[c], q = vr[c];
      s = dot2_bf16(bits_to_bf16x2(p.x), bits_to_bf16x2(q.x), s);
      s = dot2_bf16(bits_to_bf16x2(p.y), bits_to_bf16x2(q.y), s);
      s = dot2_bf16(bits_to_bf16x2(p.z), bits_to_bf16x2(q.z), s);
      s = dot2_bf16(bits_to_bf16x2(p.w), bits_to_bf16x2(q.w), s);
    }
    s = segment_sum<64>(s);
    g = 1.0f / (1.0f + __expf(-s));
  }
  if (lane == 0) a.vec_out[t] = g;
}

// ---------------------------------------------------------------------------------
// small: 512 threads, 8 waves over K. Fragment lane (r = lane % 16, q = lane / 16) holds row
// r's K values [8 q, 8 q + 8) of each 32-wide half of a 64-wide chunk, so a load reads 64
// contiguous bytes of 16 rows. The result lane holds outputs 4 q + i for token r.
constexpr int SW = 8;  // waves
constexpr int SP = 4;  // chunks in flight

__global__ void __launch_bounds__(64 * SW) gemm_small_kernel(GemmArgs a, int n_tiles, int t_tiles) {
  __shared__ float red[SW][4][64];
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int nt = 8 * (blockIdx.x / 8 / t_tiles) + blockIdx.x % 8, tt = blockIdx.x / 8 % t_tiles;
  if (nt >= n_tiles) return;
  const int r = lane % 16, q = lane / 16;
  const int n0 = 16 * nt, t0 = 16 * tt;
  const uint16_t* ap = a.w + (int64_t)min(n0 + r, a.n - 1) * a.k + 8 * q;
  const uint16_t* bp = a.x + (int64_t)min(t0 + r, a.tokens - 1) * a.k + 8 * q;
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  const int chunks = (a.k + 63) / 64;
  const bool half_tail = a.k % 64 != 0;  // the last chunk holds 32 values
  for (int c0 = wave; c0 < chunks; c0 += SW * SP) {
    uint4 av[SP][2], bv[SP][2];
#pragma unroll
    for (int u = 0; u < SP; ++u) {
      // chunks past the end read the wave's first one again, a missing second half the first
      const int c = c0 + SW * u < chunks ? c0 + SW * u : c0;
      const int second = half_tail && c == chunks - 1 ? 0 : 32;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        av[u][h] = gload16(ap + 64 * c + h * second);
        bv[u][h] = gload16(bp + 64 * c + h * second);
      }
    }
#pragma unroll
    for (int u = 0; u < SP; ++u) {
      const int c = c0 + SW * u;
      if (c >= chunks) break;  // wave-uniform
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (h == 1 && half_tail && c == chunks - 1) break;  // wave-uniform
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av[u][h]),
                                                      __builtin_bit_cast(bf16x8, bv[u][h]), acc, 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) red[wave][i][lane] = acc[i];
  __syncthreads();
  if (threadIdx.x < 256) {
    const int tc = threadIdx.x / 16, o = threadIdx.x % 16;
    const int e = o % 4, l = 16 * (o / 4) + tc;
    float v = red[0][e][l];
#pragma unroll
    for (int w = 1; w < SW; ++w) v += red[w][e][l];
    if (t0 + tc < a.tokens && n0 + o < a.n) a.out[(int64_t)(t0 + tc) * a.n + n0 + o] = v;
  }
}

// ---------------------------------------------------------------------------------
// tiled: 256 threads, wave (wm, wn) owns 32 M outputs x 32 M tokens. v_mfma_f32_32x32x16_bf16:
// lane (r = lane % 32, g = lane / 32) holds row r's K [8 g, 8 g + 8) of a 16-wide sub-step;
// result register i is output 8 (i / 4) + 4 g + i % 4 for token r. With GEMM_SWIGLU a 32-row
// weight tile is 16 gate rows and the same 16 up rows, so registers i and i + 8 are a pair.
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// Which tile a block takes. An XCD (block b runs on XCD b % 8) fetches every row its tiles use
// once into its L2, as long as what it comes back to stays there.
enum TileMap {
  TOKENS_N_INNER,  // an XCD owns an eighth of the token tiles, their output tiles innermost
  TOKENS_T_INNER,  // the same, token tiles innermost: its x rows stay in the L2, W passes once
  LIST_TOKENS,     // an XCD takes an eighth of the tile list, token tiles outermost
  LIST_OUTPUTS,    // the same, output tiles outermost
};
__device__ __forceinline__ bool tile_of_block(TileMap map, int n_tiles, int t_tiles, int& nt, int& tt) {
  const int x = blockIdx.x % 8, j = blockIdx.x / 8;
  if (map <= TOKENS_T_INNER) {
    const int ts = (t_tiles + 7) / 8;
    nt = map == TOKENS_N_INNER ? j % n_tiles : j / ts;
    tt = x * ts + (map == TOKENS_N_INNER ? j / n_tiles : j % ts);
    return tt < t_tiles && nt < n_tiles;
  }
  const int total = n_tiles * t_tiles, tile = x * ((total + 7) / 8) + j;
  nt = map == LIST_TOKENS ? tile % n_tiles : tile / t_tiles;
  tt = map == LIST_TOKENS ? tile / n_tiles : tile % t_tiles;
  return tile < total;
}

template <int M>
struct Tile {
  static constexpr int ROWS = 64 * M;              // rows of either operand
  static constexpr int OPERAND = ROWS * 128;       // bytes of a 64-wide K step
  static constexpr int STAGE = 2 * OPERAND;
  static constexpr int STAGES = M == 1 ? 3 : 2;    // 48 or 64 KB: two or more blocks on a CU
  static constexpr int LOADS = 4 * M;              // direct loads per wave and step
};

// The top of a K step: wait until only the loads of the `ahead` steps after it are in flight
// (PER a step; at most MOST steps are issued ahead), then let every wave see every wave's.
template <int PER, int MOST>
__device__ __forceinline__ void wait_step(int ahead) {
  if (ahead >= MOST) {
    wait_loads<PER * MOST>();
  } else if constexpr (MOST > 0) {
    wait_step<PER, MOST - 1>(ahead);
  }
}

template <int EP, int M>
__global__ void __launch_bounds__(256, 2) gemm_tiled_kernel(GemmArgs a, int n_tiles, int t_tiles, TileMap map,
                                                               int gemm_blocks) {
  using T = Tile<M>;
  __shared__ __attribute__((aligned(16))) uint8_t lds[T::STAGES * T::STAGE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  if ((int)blockIdx.x >= gemm_blocks) {
    const int t = ((int)blockIdx.x - gemm_blocks) * 4 + wave;
    if (t < a.tokens) token_gate(a, t, lane);
    return;
  }
  int nt, tt;
  if (!tile_of_block(map, n_tiles, t_tiles, nt, tt)) return;
  constexpr int ON = EP == GEMM_SWIGLU ? T::ROWS / 2 : T::ROWS;
  const int n0 = nt * ON, t0 = tt * T::ROWS;
  const int wm = wave & 1, wn = wave >> 1;
  const int steps = (a.k + 63) / 64;
  const bool half_tail = a.k % 64 != 0;

  // Loads: one instruction fills 8 rows of 128 bytes; wave w takes row groups w, w + 4, ...
  // of each operand. Lane l fills row l / 8, position l % 8 with piece (l % 8) ^ (row % 8).
  const int lrow = lane / 8, piece = (lane % 8) ^ lrow;
  uint32_t aoff[2 * M], boff[2 * M];
#pragma unroll
  for (int i = 0; i < 2 * M; ++i) {
    const int row = 8 * (wave + 4 * i) + lrow;
    const int n = n0 + (EP == GEMM_SWIGLU ? 16 * (row / 32) + row % 16 : row);
    // rows past the end read the last one
    aoff[i] = (uint32_t)(min(n, a.n - 1) - n0) * (uint32_t)(2 * a.k) + 16u * piece;
    boff[i] = (uint32_t)(min(t0 + row, a.tokens - 1) - t0) * (uint32_t)(2 * a.k) + 16u * piece;
  }
  // GEMM_SWIGLU: rows 16..31 of every 32 are up rows, the 8-row groups of waves 2 and 3
  const uint8_t* wbase = (const uint8_t*)((EP == GEMM_SWIGLU && wave >= 2 ? a.w2 : a.w) + (int64_t)n0 * a.k);
  const uint8_t* xbase = (const uint8_t*)(a.x + (int64_t)t0 * a.k);
  auto issue = [&](int ks) {
    const uint32_t slot = lds_addr(lds + (ks % T::STAGES) * T::STAGE);
    // the pieces past a half step's end read the ones 64 bytes before them (not used)
    const uint32_t off = 128u * ks - (half_tail && ks == steps - 1 && piece >= 4 ? 64u : 0u);
#pragma unroll
    for (int i = 0; i < 2 * M; ++i) dma16(wbase, aoff[i] + off, slot + 1024 * (wave + 4 * i));
#pragma unroll
    for (int i = 0; i < 2 * M; ++i) dma16(xbase, boff[i] + off, slot + T::OPERAND + 1024 * (wave + 4 * i));
  };

  f32x16 acc[M][M];
#pragma unroll
  for (int m = 0; m < M; ++m)
#pragma unroll
    for (int c = 0; c < M; ++c)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[m][c][i] = 0.0f;
  const int r = lane % 32, g = lane / 32;
  const uint32_t arow = (uint32_t)(32 * M * wm + r) * 128, brow = (uint32_t)(32 * M * wn + r) * 128;

#pragma unroll
  for (int p = 0; p < T::STAGES - 1; ++p)
    if (p < steps) issue(p);
  for (int ks = 0; ks < steps; ++ks) {
    // this step's loads have landed in every wave, and every wave is done with the slot that
    // the loads issued next overwrite
    wait_step<T::LOADS, T::STAGES - 2>(steps - 1 - ks);
    if (ks + T::STAGES - 1 < steps) issue(ks + T::STAGES - 1);
    const uint8_t* sa = lds + (ks % T::STAGES) * T::STAGE;
    const uint8_t* sb = sa + T::OPERAND;
    const int subs = half_tail && ks == steps - 1 ? 2 : 4;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      if (kk >= subs) break;  // block-uniform
      const uint32_t pos = 16u * (uint32_t)((2 * kk + g) ^ (r % 8));
      bf16x8 av[M], bv[M];
#pragma unroll
      for (int m = 0; m < M; ++m) {
        av[m] = *reinterpret_cast<const bf16x8*>(sa + arow + 4096 * m + pos);
        bv[m] = *reinterpret_cast<const bf16x8*>(sb + brow + 4096 * m + pos);
      }
#pragma unroll
      for (int m = 0; m < M; ++m)
#pragma unroll
        for (int c = 0; c < M; ++c) acc[m][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[m], bv[c], acc[m][c], 0, 0, 0);
    }
  }

#pragma unroll
  for (int c = 0; c < M; ++c) {
    const int t = t0 + 32 * M * wn + 32 * c + r;
    if (t >= a.tokens) continue;
    if constexpr (EP == GEMM_SWIGLU) {
#pragma unroll
      for (int m = 0; m < M; ++m)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int n = n0 + 16 * (M * wm + m) + 8 * j + 4 * g;  // n is a multiple of 4, a.n of 32
          if (n >= a.n) continue;
          ushort4 o;
          uint16_t* p = &o.x;
#pragma unroll
          for (int i = 0; i < 4; ++i) p[i] = f32_to_bf16_bits(silu(acc[m][c][4 * j + i]) * acc[m][c][8 + 4 * j + i]);
          *reinterpret_cast<ushort4*>(a.out16 + (int64_t)t * a.n + n) = o;
        }
    } else {
      const float gate = EP == GEMM_DOWN ? a.gate[t] : 0.0f;
#pragma unroll
      for (int m = 0; m < M; ++m)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int n = n0 + 32 * (M * wm + m) + 8 * j + 4 * g;
          const int64_t at = (int64_t)t * a.n + n;
          if constexpr (EP == GEMM_DOWN) {
            if (n >= a.n) continue;  // a.n is a multiple of 32
            ushort4 o;
            uint16_t* p = &o.x;
            ushort4 ad = make_ushort4(0, 0, 0, 0);
            if (a.add) ad = *reinterpret_cast<const ushort4*>(a.add + at);
            const uint16_t* q = &ad.x;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              float v = gate * acc[m][c][4 * j + i];
              if (a.add) v += bf16_bits_to_f32(q[i]);
              p[i] = f32_to_bf16_bits(v);
            }
            *reinterpret_cast<ushort4*>(a.out16 + at) = o;
          } else if (a.out_vec && n < a.n) {
            *reinterpret_cast<f32x4*>(a.out + at) =
                f32x4{acc[m][c][4 * j], acc[m][c][4 * j + 1], acc[m][c][4 * j + 2], acc[m][c][4 * j + 3]};
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (n + i < a.n) a.out[at + i] = acc[m][c][4 * j + i];
          }
        }
    }
  }
}

// split: a block of 4 waves owns 32 outputs x 32 tokens and its waves split each 128-wide K
// step (wave w the sub-steps 2 w and 2 w + 1); operands through an LDS ring of 8 steps (rows of
// 256 bytes, pieces XOR-swizzled by row % 16); the four partial tiles meet in LDS.
constexpr int KS_STAGES = 8, KS_OPERAND = 32 * 256, KS_STAGE = 2 * KS_OPERAND;

template <int EP>
__global__ void __launch_bounds__(256) gemm_split_kernel(GemmArgs a, int n_tiles, int t_tiles, int gemm_blocks) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[KS_STAGES * KS_STAGE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  if ((int)blockIdx.x >= gemm_blocks) {
    const int t = ((int)blockIdx.x - gemm_blocks) * 4 + wave;
    if (t < a.tokens) token_gate(a, t, lane);
    return;
  }
  const int nt = 8 * (blockIdx.x / 8 / t_tiles) + blockIdx.x % 8, tt = blockIdx.x / 8 % t_tiles;
  if (nt >= n_tiles) return;
  constexpr int ON = EP == GEMM_SWIGLU ? 16 : 32;
  const int n0 = nt * ON, t0 = tt * 32;
  const int steps = (a.k + 127) / 128;
  const int tail = a.k % 128 / 8;  // pieces of a partial last step (0: it is whole)

  // one load instruction fills 4 rows; wave w takes rows 4 (w + 4 i) .. + 3 of each operand
  const int lrow = lane / 16;
  uint32_t aoff[2], boff[2], step_piece[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = 4 * (wave + 4 * i) + lrow;
    const int n = n0 + (EP == GEMM_SWIGLU ? row % 16 : row);  // i = 1: the up rows
    const int piece = (lane % 16) ^ (row % 16);
    aoff[i] = (uint32_t)(min(n, a.n - 1) - n0) * (uint32_t)(2 * a.k);
    boff[i] = (uint32_t)(min(t0 + row, a.tokens - 1) - t0) * (uint32_t)(2 * a.k);
    step_piece[i] = (uint32_t)piece;
  }
  const uint8_t* wbase = (const uint8_t*)(a.w + (int64_t)n0 * a.k);
  const uint8_t* ubase = EP == GEMM_SWIGLU ? (const uint8_t*)(a.w2 + (int64_t)n0 * a.k) : wbase;
  const uint8_t* xbase = (const uint8_t*)(a.x + (int64_t)t0 * a.k);
  auto issue = [&](int ks) {
    const uint32_t slot = lds_addr(lds + (ks % KS_STAGES) * KS_STAGE);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      // pieces past a partial step's end read its first 64 bytes (not used)
      const uint32_t p = tail && ks == steps - 1 && step_piece[i] >= (uint32_t)tail ? step_piece[i] & 3 : step_piece[i];
      const uint32_t off = 256u * ks + 16u * p, dst = slot + 1024 * (wave + 4 * i);
      dma16(i ? ubase : wbase, aoff[i] + off, dst);
      dma16(xbase, boff[i] + off, dst + KS_OPERAND);
    }
  };
  f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
  const int r = lane % 32, g = lane / 32;
  for (int p = 0; p < KS_STAGES - 1; ++p)
    if (p < steps) issue(p);
  for (int ks = 0; ks < steps; ++ks) {
    wait_step<4, KS_STAGES - 2>(steps - 1 - ks);
    if (ks + KS_STAGES - 1 < steps) issue(ks + KS_STAGES - 1);
    const uint8_t* sa = lds + (ks % KS_STAGES) * KS_STAGE;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int p = 4 * wave + 2 * h;
      if (tail && ks == steps - 1 && p >= tail) break;  // wave-uniform
      const uint32_t at = (uint32_t)(r * 256 + 16 * ((p + g) ^ (r % 16)));
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8*>(sa + at),
                                                    *reinterpret_cast<const bf16x8*>(sa + KS_OPERAND + at), acc, 0, 0, 0);
    }
  }
  wait_loads<0>();
  float(*red)[16][64] = reinterpret_cast<float(*)[16][64]>(lds);
#pragma unroll
  for (int i = 0; i < 16; ++i) red[wave][i][lane] = acc[i];
  __syncthreads();
  auto total = [&](int o, int tc) {  // output row o of the tile, token tc
    const int i = o / 8 * 4 + o % 4, l = 32 * (o / 4 % 2) + tc;
    return (red[0][i][l] + red[1][i][l]) + (red[2][i][l] + red[3][i][l]);
  };
  for (int idx = threadIdx.x; idx < ON * 32; idx += 256) {
    const int tc = idx / ON, o = idx % ON;
    const int t = t0 + tc, n = n0 + o;
    if (t >= a.tokens || n >= a.n) continue;
    const int64_t at = (int64_t)t * a.n + n;
    if constexpr (EP == GEMM_SWIGLU) {
      a.out16[at] = f32_to_bf16_bits(silu(total(o, tc)) * total(16 + o, tc));
    } else if constexpr (EP == GEMM_F32) {
      a.out[at] = total(o, tc);
    } else {
      float v = a.gate[t] * total(o, tc);
      if (a.add) v += bf16_bits_to_f32(a.add[at]);
      a.out16[at] = f32_to_bf16_bits(v);
    }
  }
}

template <int EP>
static void launch_split(const GemmArgs& a, hipStream_t s) {
  constexpr int ON = EP == GEMM_SWIGLU ? 16 : 32;
  const int n_tiles = (a.n + ON - 1) / ON, t_tiles = (a.tokens + 31) / 32;
  const int blocks = 8 * ((n_tiles + 7) / 8) * t_tiles;
  const int extra = EP == GEMM_SWIGLU && a.vec_out ? (a.tokens + 3) / 4 : 0;
  hipLaunchKernelGGL((gemm_split_kernel<EP>), dim3(blocks + extra), dim3(256), 0, s, a, n_tiles, t_tiles, blocks);
  check_launch("gemm_bf16 (split)");
}

static void launch_small(const GemmArgs& a, hipStream_t s) {
  const int n_tiles = (a.n + 15) / 16, t_tiles = (a.tokens + 15) / 16;
  hipLaunchKernelGGL(gemm_small_kernel, dim3(8 * ((n_tiles + 7) / 8) * t_tiles), dim3(64 * SW), 0, s, a, n_tiles, t_tiles);
  check_launch("gemm_bf16 (small)");
}

template <int EP, int M>
static void launch_tiled(const GemmArgs& a, hipStream_t s) {
  constexpr int ROWS = Tile<M>::ROWS, ON = EP == GEMM_SWIGLU ? ROWS / 2 : ROWS;
  const int n_tiles = (a.n + ON - 1) / ON, t_tiles = (a.tokens + ROWS - 1) / ROWS;
  const int64_t xb = (int64_t)a.tokens * a.k * 2, wb = (int64_t)a.n * (EP == GEMM_SWIGLU ? 2 : 1) * a.k * 2;
  TileMap map;
  int blocks;
  if (xb >= wb && (t_tiles % 8 == 0 || t_tiles >= 32)) {
    map = xb / 8 <= (5 << 19) ? TOKENS_T_INNER : TOKENS_N_INNER;
    blocks = 8 * ((t_tiles + 7) / 8) * n_tiles;
  } else {
    map = xb >= wb ? LIST_TOKENS : LIST_OUTPUTS;
    blocks = 8 * (int)(((int64_t)n_tiles * t_tiles + 7) / 8);
  }
  const int extra = EP == GEMM_SWIGLU && a.vec_out ? (a.tokens + 3) / 4 : 0;
  hipLaunchKernelGGL((gemm_tiled_kernel<EP, M>), dim3(blocks + extra), dim3(256), 0, s, a, n_tiles, t_tiles,
                     map, blocks);
  check_launch("gemm_bf16 (tiled)");
}

// Blocks a kernel may have to itself: past one per CU it takes a second round.
constexpr int64_t ONE_ROUND = 256;

// The kernel of a shape. A CU draws about 38 KB/us of rows that are not yet in its XCD's L2
// however many loads it has in flight, so a block's time is the bytes of its rows: the
// smallest tile whose blocks still fit one round wins, and past that the tile whose rows are
// reused most. Measured (K 2048, 512 outputs, weights and tokens not in the L2): 64 tokens small
// 5.9 us, split 9.6, 64 x 64 tiles 13; 301 tokens small 13 (608 blocks), split 10.0, 64 x 64
// 13.4; 600 tokens split 18.2 (304 blocks), 64 x 64 13.4; 4096 tokens 64 x 64 19.0, 128 x 128
// 23.7; 16384 tokens 71 against 45.5.
template <int EP>
static void launch(const GemmArgs& a, hipStream_t s) {
  auto blocks = [&](int64_t outputs, int64_t tokens) {
    return ((a.n * (EP == GEMM_SWIGLU ? 2 : 1) + outputs - 1) / outputs) * ((a.tokens + tokens - 1) / tokens);
  };
  if constexpr (EP == GEMM_F32) {
    if (blocks(16, 16) <= ONE_ROUND) return launch_small(a, s);
  }
  if (blocks(32, 32) <= ONE_ROUND) return launch_split<EP>(a, s);
  if (blocks(128, 128) >= ONE_ROUND) return launch_tiled<EP, 2>(a, s);
  launch_tiled<EP, 1>(a, s);
}

}  // namespace gb

bool gemm_bf16_fits(const void* x, const void* w, int k) {
  return k % 32 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0;
}

void gemm_bf16(GemmEpilogue ep, const GemmArgs& args, hipStream_t s) {
  GemmArgs a = args;
  a.out_vec = a.n % 4 == 0 && (uintptr_t)a.out % 16 == 0;  // rows of 16-byte stores
  if (ep == GEMM_SWIGLU) gb::launch<GEMM_SWIGLU>(a, s);
  else if (ep == GEMM_DOWN) gb::launch<GEMM_DOWN>(a, s);
  else gb::launch<GEMM_F32>(a, s);
}

}  // namespace wm
