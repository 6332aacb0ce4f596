// The grouped GEMMs' tiles for few rows an expert: a part of grouped_mfma.hip (which includes it
// after its 128-row tiles and its tile, term and scalar-load helpers).
//
// With up to a few dozen rows an expert the weights, each read once, bound the call. What 128-row
// tiles spend there instead: MFMAs on empty rows (128 for 1 to 64), two load slots that wait
// a memory round trip each K step, and, in the row layout, half a 128-byte line of every
// MXFP4 row a step. Here:
//
//   tile    : BM rows of one expert x TW = 32 WAVES weight rows in 32-row weight tiles, for gate_up
//             16 gate rows and the same 16 up rows, so that a lane holds both results of a column.
//             With 16 rows wave w owns weight tile w; with 64, wave (wm, wn) = (w / 4, w % 4) owns the
//             weight tiles 2 wn and 2 wn + 1 and the row tile of 32 rows wm, so that a step reads
//             96 KB of LDS (MXFP4) where 32 weight rows x 64 rows a wave read 144, as many
//             LDS cycles as MFMA ones (2048 tokens over 512 experts of 2560/640: gate_up 320 ->
//             301 us, down 194 -> 186; 219 and 136 without the compute, 217 and 139 without the
//             loads, so what is left is how far the two overlap).
//   weights : a unit is 128 bytes of every row (two 128-wide K steps of MXFP4, one of FP8), eight
//             whole lines of 8 rows a load, in either layout, with the non-temporal hint (a
//             plain read of HBM: 7.0 against 5.9 TB/s).
//   rows    : the split rows by K step, as in the 128-row tiles.
//
// Both go to LDS rings of three slots by direct loads, two units (steps) ahead, across tiles.
// Two shapes: 64 rows x 256 weight rows (8 waves, 154 KB), one row tile an expert; and, for MXFP4, 16
// rows x 128 (4 waves, 77 KB), two workgroups on a CU, one's epilogue and tile set-up under the
// other's loads. row_tiles() says which call takes which, with times. WIDE: the 16-row shape for calls
// of a few tokens, 4 rows a tile with activations of eight terms (see run_few). At 2 rows an expert of
// 7168/2048 FP8 weights (11.3 GB): 1486 us a call against 2791 with 128-row tiles, 7.6 TB/s.
#pragma once

namespace wm {
namespace mf {

typedef float v4f __attribute__((ext_vector_type(4)));

template <bool FP8_, bool A_SCALED_, int BM_, int WAVES_, bool WIDE_ = false>
struct StreamF {
  // WIDE: eight terms, two in each of SETS operand rows; operand row r holds set r / ROWS of tile row r % ROWS
  static constexpr bool WIDE = WIDE_;
  static constexpr int SETS = WIDE_ ? 4 : 1, ROWS = BM_ / SETS;  // rows of a tile
  static constexpr bool FP8 = FP8_, A_SCALED = A_SCALED_, BLOCK_F32 = FP8_ && !A_SCALED_;
  static constexpr int BM = BM_, WAVES = WAVES_, TW = 32 * WAVES_;
  static constexpr int MI = BM_ == 16 ? 1 : 2;             // a wave's weight tiles
  static constexpr int SUB = FP8_ ? 1 : 2;                 // K steps of a weight unit
  static constexpr int BSUB = BM_ == 16 ? SUB : 1;         // K steps of a split-row slot
  static constexpr int GRAN = SUB / BSUB;                  // split-row slots of a unit
  static constexpr int A_FMT = FP8_ ? FMT_FP8 : FMT_FP4;
  static constexpr int A_SLOT = TW * 128 + (A_SCALED_ ? TW * 4 * SUB : 0);
  static constexpr int B_TERMS = BM_ * XSTEP8 * BSUB, B_SLOT = B_TERMS + BM_ * 4 * BSUB;
  static constexpr int RINGS = 3 * (A_SLOT + B_SLOT), BYTES = RINGS + (BM_ == 16 ? WAVES_ * BM_ * 4 : 0);  // and block maxima
  static constexpr int NQA = 4, NQB = BM_ / 4 / WAVES_;    // 1 KB loads of a wave: a unit's, a K step's rows
  // about how many of its tiles take as long as one 128-row tile (twice the weight rows for MXFP4, and
  // bound by its MFMAs)
  static constexpr int HOT_COST = FP8_ ? 1 : 3;
  // loads of a wave: a unit's, and at least a split-row slot's (see issue_rows)
  static constexpr int UNIT_LOADS = NQA + (A_SCALED_ ? 1 : 0), ROW_LOADS = BM_ == 16 ? BSUB + 1 : 2;
  static_assert(BM_ == 16 ? NQB == 1 && !FP8_ : BM_ == 64 && NQB == 2, "the loader's split-row loads");
  static_assert(!WIDE_ || BM_ == 16, "eight terms: 16-row tiles");
};

// Loads of one tile. Weight load i of wave w fills rows 8 (w + WAVES i) .. + 7 of the tile: lane l
// row l / 8, LDS position l % 8 holding piece (l % 8) ^ (l / 8) of the row's 128 bytes (8 rows at
// one piece then lie on distinct banks). The second half of a unit's pieces (the odd K step of MXFP4)
// is `half` bytes on; a last unit of one step reads its first half twice.
template <typename F>
struct StreamLoads {
  const uint8_t *w, *s, *b, *bs;
  uint32_t woff[F::NQA], whalf, wunit, soff, shalf, sunit;
  uint32_t boff[F::NQB], bsoff;

  // rows: the region's rows, k its K; row_of(j): the region row of tile row j (8-row groups stay
  // together)
  template <typename RowOf>
  __device__ __forceinline__ void weights(const uint8_t* region, const uint8_t* scales, int rows, int k, int tiled,
                                          int wave, int lane, RowOf row_of) {
    w = uniform_u8(region);
    s = uniform_u8(scales);
    const int p = (lane % 8) ^ (lane / 8);
#pragma unroll
    for (int i = 0; i < F::NQA; ++i) {
      const int row = row_of(8 * (wave + F::WAVES * i) + lane / 8);
      if (tiled)
        woff[i] = (uint32_t)(row / 16 * (F::FP8 ? 2048 : 1024) + (F::FP8 ? p : p % 4) * 256 + row % 16 * 16);
      else
        woff[i] = (uint32_t)(row * (F::FP8 ? k : k / 2) + (F::FP8 ? p : p % 4) * 16);
    }
    const uint32_t step = tiled ? (uint32_t)rows * (F::FP8 ? 128 : 64) : (F::FP8 ? 128 : 64);
    wunit = F::SUB * step;
    whalf = F::FP8 || p < 4 ? 0 : step;
    soff = shalf = sunit = 0;
    if constexpr (F::A_SCALED && F::FP8) {  // E8M0 32 x 32 blocks: lanes 0..31, a dword a row and step
      soff = (uint32_t)(row_of(32 * wave + lane % 32) / 32 * (k / 32));
      sunit = 4;
    } else if constexpr (F::A_SCALED) {  // lane l: row 32 w + l / 2, step l % 2
      const int row = row_of(32 * wave + lane / 2);
      const uint32_t sstep = tiled ? (uint32_t)rows * 4 : 4;
      soff = (uint32_t)(tiled ? row * 4 : row * (k / 32));
      sunit = 2 * sstep;
      shalf = lane % 2 ? sstep : 0;
    }
  }
  // row_index(r): the split row of tile row r (wave-uniform r). Load i of wave w fills rows
  // 4 (w + WAVES i) .. + 3, and the scale load their dwords.
  template <typename RowIndex>
  __device__ __forceinline__ void rows(const uint8_t* terms, const uint8_t* scales, int k, int wave, int lane,
                                       RowIndex row_index) {
    b = uniform_u8(terms);
    bs = uniform_u8(scales);
    bsoff = 0;
#pragma unroll
    for (int i = 0; i < F::NQB; ++i) {
      const int q0 = 4 * (wave + F::WAVES * i);
      int idx[4];
#pragma unroll
      for (int d = 0; d < 4; ++d) idx[d] = row_index(q0 + d);
      const int d = lane / 16, e = lane % 4;
      const int mine = d == 0 ? idx[0] : d == 1 ? idx[1] : d == 2 ? idx[2] : idx[3];
      boff[i] = (uint32_t)mine * (uint32_t)(k / 128 * XSTEP8) + 16u * (uint32_t)((lane % 16) ^ ((q0 + d) & 15));
      const int srow = e == 0 ? idx[0] : e == 1 ? idx[1] : e == 2 ? idx[2] : idx[3];
      if (lane / 4 == i || F::NQB == 1) bsoff = (uint32_t)srow * (uint32_t)(k / 128 * 4);
    }
  }
  // Weight unit u; whole: both its steps exist. UNIT_LOADS instructions.
  __device__ __forceinline__ void issue_unit(uint8_t* slot, int u, bool whole, int wave, int lane) const {
    const uint32_t at = (uint32_t)u * wunit + (whole ? whalf : 0);
#pragma unroll
    for (int i = 0; i < F::NQA; ++i) dma16<true>(w, woff[i] + at, lds_addr(slot + (wave + F::WAVES * i) * 1024));
    if constexpr (F::A_SCALED) {
      if (!F::FP8 || lane < 32)
        dma4(s, soff + (uint32_t)u * sunit + (whole ? shalf : 0),
             lds_addr(slot + F::TW * 128 + wave * (F::FP8 ? 128 : 256)));
    }
  }
  // The split rows' K steps BSUB k .. of a tile of `n` rows into a slot: ROW_LOADS instructions or one
  // more (the second load's rows only where the tile has them; what it leaves in LDS feeds unused
  // columns). A step past the last reads the last again.
  __device__ __forceinline__ void issue_rows(uint8_t* slot, int k, int steps, int n, int wave, int lane) const {
    const int ks = min(F::BSUB * k, steps - 1);
    if constexpr (F::BM == 16) {
      const bool two = ks + 1 < steps;
#pragma unroll
      for (int h = 0; h < F::BSUB; ++h)
        dma16(b, boff[0] + (uint32_t)(h && two ? ks + 1 : ks) * XSTEP8, lds_addr(slot + h * 16 * XSTEP8 + wave * 1024));
      // lanes 0..3 the first step's scale dwords of rows 4 w .. + 3, lanes 4..7 the second's
      if (lane < 4 * F::BSUB)
        dma4(bs, bsoff + (uint32_t)(lane >= 4 && two ? ks + 1 : ks) * 4, lds_addr(slot + F::B_TERMS + 16 * F::BSUB * wave));
    } else {
#pragma unroll
      for (int i = 0; i < F::NQB; ++i)
        if (4 * F::WAVES * i < n)
          dma16(b, boff[i] + (uint32_t)ks * XSTEP8, lds_addr(slot + (wave + F::WAVES * i) * 1024));
      if (lane < 4 * F::NQB) dma4(bs, bsoff + (uint32_t)ks * 4, lds_addr(slot + F::B_TERMS + 16 * F::NQB * wave));
    }
  }
};

template <typename F>
struct StreamTile {
  StreamLoads<F> ld;
  int expert, begin, end, nt;
  float limit;
  const_f32_ptr s0, s1;  // FP8 with fp32 blocks: the block scales of the wave's registers 0..7 and 8..15
};

// Tile `logical` of the list. With 64 rows every expert has one row tile, so the list is row tile by
// row tile; otherwise an expert's row tiles that read the same weights run together (order_tile).
template <typename F>
__device__ __forceinline__ void stream_locate(const Lists& L, int logical, int n_tiles, StreamTile<F>& t) {
  int mt = logical / n_tiles;
  t.nt = logical - mt * n_tiles;
  if constexpr (F::BM == 16) order_tile<F::ROWS>(L, logical, n_tiles, mt, t.nt);
  resolve_tile_s<F::ROWS>(L, mt, t.expert, t.begin, t.end);
}

// A wave's results: MI weight tiles of 32 rows x a row tile of 32 columns (v_mfma_scale_f32_32x32x64 in the
// order of the 128-row tiles, so that a row's results do not depend on the tile that held it: with 16
// rows half the columns go unused, 2.5% of a call of 64 tokens of 5120/2304 over 16x16x128, whose sums of
// 128 products round otherwise). WIDE: its two 16-row weight tiles (gate_up: the gate and the up rows) x 16
// columns (16x16x128).
template <typename F>
struct StreamAcc {
  v16f v[F::MI];
  v4f q[2];
  __device__ __forceinline__ void clear() {
    q[0] = q[1] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int mi = 0; mi < F::MI; ++mi)
#pragma unroll
      for (int i = 0; i < 16; ++i) v[mi][i] = 0.0f;
  }
};

// WIDE: acc += K step `sub` of an MXFP4 weight unit and of a split-row slot. Lane (c, q) holds row
// c's E2M1 K [32 q, +32), or E4M3 K [16 q, +16) and [64 + 16 q, +16); scale lane (c, q) covers K block q.
template <typename F>
__device__ __forceinline__ void stream_step16(const uint8_t* wa, const uint8_t* rb, int sub, int wave, int lane,
                                              v4f (&acc)[2]) {
  const int c = lane % 16, q = lane / 16;
  uint4 p[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) p[e] = *reinterpret_cast<const uint4*>(rb + sub * 16 * XSTEP8 + e4_piece(c, 4 * e + q));
  const uint32_t sw =
      *reinterpret_cast<const uint32_t*>(rb + F::B_TERMS + 16 * F::BSUB * (c / 4) + 16 * sub + 4 * (c % 4)) >> (8 * q);
  const v8i hi = {(int)p[0].x, (int)p[0].y, (int)p[0].z, (int)p[0].w, (int)p[1].x, (int)p[1].y, (int)p[1].z, (int)p[1].w};
  const v8i lo = {(int)p[2].x, (int)p[2].y, (int)p[2].z, (int)p[2].w, (int)p[3].x, (int)p[3].y, (int)p[3].z, (int)p[3].w};
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int row = 32 * wave + 16 * t + c;
    const uint4 u = *reinterpret_cast<const uint4*>(wa + row * 128 + 16 * ((4 * sub + q) ^ (row % 8)));
    const v8i a = {(int)u.x, (int)u.y, (int)u.z, (int)u.w, 0, 0, 0, 0};
    const int sa = (int)(*reinterpret_cast<const uint32_t*>(wa + F::TW * 128 + row * 8 + 4 * sub) >> (8 * q));
    // lo scales: hi - 4 (every hi scale byte is >= 5, so the low byte takes no borrow)
    acc[t] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, hi, acc[t], F::A_FMT, FMT_FP8, 0, sa, 0, (int)sw);
    acc[t] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, lo, acc[t], F::A_FMT, FMT_FP8, 0, sa, 0, (int)(sw - 4));
  }
}

// acc += K step `sub` of a weight unit x a step of split rows, for the weight rows w0 .. and the tile's rows
// row0 ..; f0, f1: the fp32 block scales of result registers 0..7 and 8..15. A half's fragment reads run
// under the other half's MFMAs. With 16 rows the slot holds BSUB steps and columns 16..31 repeat the
// rows of 0..15.
template <typename F>
__device__ __forceinline__ void stream_step(const uint8_t* wa, const uint8_t* rb, int sub, int w0, int row0, int lane,
                                            float f0, float f1, v16f (&acc)[F::MI]) {
  const int r = lane % 32, g = lane / 32;
  const int row = row0 + r % F::BM;
  const uint8_t* arow = wa + (w0 + r) * 128;
  uint32_t sa[F::MI];
#pragma unroll
  for (int mi = 0; mi < F::MI; ++mi)
    sa[mi] = F::A_SCALED ? *reinterpret_cast<const uint32_t*>(wa + F::TW * 128 + (w0 + 32 * mi + r) * 4 * F::SUB + 4 * sub)
                         : 127;
  // where the loader put the row's scale dword
  const uint32_t sw = *reinterpret_cast<const uint32_t*>(
      rb + F::B_TERMS + (F::BM == 16 ? 16 * (F::BSUB * (row / 4) + sub) + 4 * (row % 4)
                                     : 4 * (8 * (row / 4 % F::WAVES) + 4 * (row / (4 * F::WAVES)) + row % 4)));
  const uint8_t* terms = rb + (F::BM == 16 ? sub * 16 * XSTEP8 : 0);
  v8i a[2][F::MI], t[2][2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int mi = 0; mi < F::MI; ++mi) {
      auto piece = [&](int p) { return *reinterpret_cast<const uint4*>(arow + 4096 * mi + 16 * (p ^ (r % 8))); };
      if constexpr (F::FP8) {
        const uint4 u = piece(4 * h + g), v = piece(4 * h + 2 + g);
        a[h][mi] = v8i{(int)u.x, (int)u.y, (int)u.z, (int)u.w, (int)v.x, (int)v.y, (int)v.z, (int)v.w};
      } else {
        const uint4 u = piece(4 * sub + 2 * h + g);
        a[h][mi] = v8i{(int)u.x, (int)u.y, (int)u.z, (int)u.w, 0, 0, 0, 0};
      }
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const uint4 u = *reinterpret_cast<const uint4*>(terms + e4_piece(row, 8 * e + 4 * h + g));
      const uint4 v = *reinterpret_cast<const uint4*>(terms + e4_piece(row, 8 * e + 4 * h + 2 + g));
      t[h][e] = v8i{(int)u.x, (int)u.y, (int)u.z, (int)u.w, (int)v.x, (int)v.y, (int)v.z, (int)v.w};
    }
  }
  v16f blk[F::BLOCK_F32 ? F::MI : 1];
  if constexpr (F::BLOCK_F32) {
#pragma unroll
    for (int mi = 0; mi < F::MI; ++mi)
#pragma unroll
      for (int i = 0; i < 16; ++i) blk[mi][i] = 0.0f;
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int sh = 8 * g + 16 * h;
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int mi = 0; mi < F::MI; ++mi) {
        v16f& sum = F::BLOCK_F32 ? blk[F::BLOCK_F32 ? mi : 0] : acc[mi];
        // lo scales: hi - 4 (every hi scale byte is >= 5)
        sum = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a[h][mi], t[h][e], sum, F::A_FMT, FMT_FP8, 0,
                                                              F::A_SCALED ? (int)(sa[mi] >> sh) : 127, 0,
                                                              (int)((sw - (e ? 0x04040404u : 0u)) >> sh));
      }
  }
  if constexpr (F::BLOCK_F32) {  // the fp32 block scale cannot ride on the MFMA's E8M0 scales
#pragma unroll
    for (int mi = 0; mi < F::MI; ++mi)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[mi][i] = fmaf(i < 8 ? f0 : f1, blk[mi][i], acc[mi][i]);
  }
}

// The tiles of this workgroup as one sequence of split-row slots, GRAN to a weight unit (a tile's
// last unit counts whole; its missing K step is skipped). At the top of slot step g: wait until its
// rows and its unit have landed, a barrier (which also frees the slots of step g - 1), then the
// loads of the rows of step g + 2 and, on a unit's first step, of the unit two on, the next tile's
// where this one ends. Issue order is ..., rows g, unit g / GRAN + 1 (first steps), rows g + 1, so
// UNIT_LOADS + ROW_LOADS may stay in flight while those were issued. The epilogue's stores count
// too: they may complete out of order with loads, but loads do not among themselves, so at most that
// many of the youngest loads are outstanding. At least two units a tile.
// locate(j, tile) finds a tile (at the start of the one before it, so that its scalar loads'
// round trips are not where the loads of its first unit wait), setup(tile) its addresses.
template <typename F, typename Locate, typename Setup, typename Epilogue>
__device__ __forceinline__ void stream_tiles(const TileRange& tr, int steps, uint8_t* lds, int wave, int lane, Locate locate,
                                             Setup setup, Epilogue epilogue) {
  if (tr.count == 0) return;
  const int units = (steps + F::SUB - 1) / F::SUB, n = units * F::GRAN;
  auto wslot = [&](int u) { return lds + u % 3 * F::A_SLOT; };
  auto rslot = [&](int g) { return lds + 3 * F::A_SLOT + g % 3 * F::B_SLOT; };
  auto unit = [&](const StreamTile<F>& t, int at, int u) {
    t.ld.issue_unit(wslot(at), u, F::SUB * (u + 1) <= steps, wave, lane);
  };
  auto rows = [&](const StreamTile<F>& t, int at, int k) {
    t.ld.issue_rows(rslot(at), k, steps, t.end - t.begin, wave, lane);
  };
  StreamAcc<F> acc;
  StreamTile<F> cur, nxt;
  locate(0, cur);
  setup(cur);
  rows(cur, 0, 0);
  unit(cur, 0, 0);
  rows(cur, 1, 1);
  unit(cur, 1, 1);
  acc.clear();
  int g = 0, gu = 0;  // slot steps and units before this one
  for (int j = 0; j < tr.count; ++j) {
    const bool more = j + 1 < tr.count;
    for (int k = 0; k < n; ++k, ++g) {
      const int sub = F::GRAN == 2 ? k & 1 : 0, u = F::GRAN == 2 ? k >> 1 : k;
      // units issued after this step's rows: the next (a unit's first step) or the one after it
      const bool kept = more || u + 1 + sub < units;
      if (kept)
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(F::UNIT_LOADS + F::ROW_LOADS) : "memory");
      else
        ring_wait_all();
      if (k == 0 && more) locate(j + 1, nxt);
      if (sub == 0 && more && u + 2 == units) setup(nxt);
      if (k + 2 < n) rows(cur, g + 2, k + 2);
      else if (more) rows(nxt, g + 2, k + 2 - n);
      if (sub == 0) {
        if (u + 2 < units) unit(cur, gu + 2, u + 2);
        else if (more) unit(nxt, gu + 2, u + 2 - units);
      }
#pragma unroll
      for (int h = 0; h < F::BSUB; ++h) {
        const int ks = F::BSUB * k + h;
        if (ks >= steps) break;  // uniform
        if constexpr (F::BM == 16) {
          if constexpr (F::WIDE) stream_step16<F>(wslot(gu), rslot(g), h, wave, lane, acc.q);
          else stream_step<F>(wslot(gu), rslot(g), h, 32 * wave, 0, lane, 1.0f, 1.0f, acc.v);
        } else {
          const int wm = wave / 4, wn = wave % 4;
          if (32 * wm >= cur.end - cur.begin) continue;  // no rows in this row tile (uniform)
          float f0 = 1.0f, f1 = 1.0f;
          if constexpr (F::BLOCK_F32) f0 = cur.s0[ks], f1 = cur.s1[ks];
          stream_step<F>(wslot(gu), rslot(g), sub, 64 * wn, 32 * wm, lane, f0, f1, acc.v);
        }
      }
      if (sub == F::GRAN - 1) ++gu;
    }
    epilogue(cur, acc);
    acc.clear();
    cur = nxt;
  }
}

// WIDE: in the lanes of the first set, its product plus those of the others, the smallest first.
template <typename F>
__device__ __forceinline__ float sum_sets(float v, int lane) {
  float low = __shfl(v, lane + (F::SETS - 1) * F::ROWS, 64);
#pragma unroll
  for (int h = F::SETS - 2; h > 0; --h) low += __shfl(v, lane + h * F::ROWS, 64);
  return v + low;
}

// The lists of a launch. WIDE: without the shared expert's rows where its table says that it is not resident, so
// that no weights are read for it (the routed experts' rows are left out of the lists themselves).
template <typename F, typename Table>
__device__ __forceinline__ Lists resident_lists(const Lists& all, const Table& shared) {
  Lists L = all;
  if constexpr (F::WIDE)
    if (L.has_shared && shared.slots && scalar_i32(shared.slots, 0) < 0) L.has_shared = 0;
  return L;
}

// act rows of TW / 2 intermediate columns, 16 a weight tile: result lane (r, g) register i < 8 is the
// gate and i + 8 the up product of column 8 (i / 4) + 4 g + i % 4 for row r of the row tile.
// Weight tiles 2 p and 2 p + 1 share a 32-value block of the act row: a wave's own two, or with 16 rows
// those of two waves.
template <typename F, typename Table>
__device__ __forceinline__ void stream_gate_up(uint8_t* lds, const uint8_t* __restrict__ x8, const uint8_t* __restrict__ x8s,
                                               const int32_t* __restrict__ row_token, const Lists& all, const Table& routed,
                                               const Table& shared, int before, int x_rows, int a_rows,
                                               uint8_t* __restrict__ a8, uint8_t* __restrict__ a8s) {
  float(*block_max)[F::BM] = reinterpret_cast<float(*)[F::BM]>(lds + F::RINGS);  // 16 rows
  const Lists L = resident_lists<F>(all, shared);
  constexpr int TG = F::TW / 2;
  const int H = routed.hidden, I = routed.inter;
  const int n_tiles = I / TG;  // I is a multiple of 128
  const TileRange tr = tile_range_after(active_row_tiles<F::ROWS>(L) * n_tiles, before, F::HOT_COST);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  auto locate = [&](int j, StreamTile<F>& t) { stream_locate<F>(L, tr.at(j), n_tiles, t); };
  auto setup = [&](StreamTile<F>& t) {
    const TileWeights tw = tile_weights_s(routed, shared, t.expert);
    t.limit = tw.limit;
    const int gate0 = (tw.up_first ? I : 0) + t.nt * TG, up0 = (tw.up_first ? 0 : I) + t.nt * TG;
    t.ld.weights(tw.w13, tw.w13s, 2 * I, H, table_tiled(routed), wave, lane,
                 [=](int j) { return (j % 32 < 16 ? gate0 : up0) + j / 32 * 16 + j % 16; });
    if constexpr (F::BLOCK_F32) {
      t.s0 = uniform_ptr(reinterpret_cast<const float*>(tw.w13s) + (int64_t)(gate0 / 128) * (H / 128));
      t.s1 = uniform_ptr(reinterpret_cast<const float*>(tw.w13s) + (int64_t)(up0 / 128) * (H / 128));
    }
    const int begin = t.begin, end = t.end;
    t.ld.rows(x8, x8s, H, wave, lane, [&](int r) {
      const int q = begin + r % F::ROWS;
      return scalar_i32(row_token, q < end ? q : begin) + r / F::ROWS * x_rows;
    });
  };
  auto epilogue = [&](const StreamTile<F>& t, StreamAcc<F>& acc) {
    const int rows = t.end - t.begin;
    auto act = [&](float gv, float uv) {
      if (t.limit > 0.0f) {
        gv = fminf(gv, t.limit);
        uv = fminf(fmaxf(uv, -t.limit), t.limit);
      }
      return silu(gv) * uv;
    };
    if constexpr (F::BM == 16) {
      constexpr int COLS = F::WIDE ? 16 : 32, GROUPS = F::WIDE ? 1 : 2;  // result columns; a lane's groups of 4 values
      const int row = lane % COLS, g = lane / COLS;
      float v[GROUPS][4], amax = 0.0f;
#pragma unroll
      for (int i = 0; i < 4 * GROUPS; ++i) {
        float gv = F::WIDE ? acc.q[0][i % 4] : acc.v[0][i], uv = F::WIDE ? acc.q[1][i % 4] : acc.v[0][i + 8];
        if constexpr (F::WIDE) gv = sum_sets<F>(gv, lane), uv = sum_sets<F>(uv, lane);
        v[i / 4][i % 4] = act(gv, uv);
        amax = fmaxf(amax, fabsf(v[i / 4][i % 4]));
      }
      if constexpr (F::WIDE) amax = fmaxf(amax, __shfl_xor(amax, 16, 64));
      amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
      if (lane < F::BM) block_max[wave][lane] = amax;
      stage_barrier();
      if (row >= rows) return;
      const float block = fmaxf(amax, block_max[wave ^ 1][row]);
      const int s = F::WIDE ? fp8_term_exponent_wide(block) : fp8_term_exponent(block);
      const int n = t.nt * TG + 16 * wave;  // the wave's first column
      const int64_t at = (int64_t)(t.begin + row) * (I / 128);
      uint8_t* dst = a8 + (at + n / 128) * XSTEP8 + n % 128 + 4 * g;
#pragma unroll
      for (int q = 0; q < GROUPS; ++q) {  // columns 8 q + 4 g .. + 3
        if constexpr (F::WIDE) {
          uint32_t w[WIDE_TERMS];
          fp8_terms4_wide(v[q], pow2_biased(254 - s), w);
#pragma unroll
          for (int e = 0; e < WIDE_TERMS; ++e)
            *reinterpret_cast<uint32_t*>(dst + 8 * q + (int64_t)(e / 2) * a_rows * (I / 128) * XSTEP8 + e % 2 * 128) = w[e];
        } else {
          uint32_t hi, lo;
          fp8_terms4(v[q], pow2_biased(254 - s), hi, lo);
          *reinterpret_cast<uint32_t*>(dst + 8 * q) = hi;
          *reinterpret_cast<uint32_t*>(dst + 8 * q + 128) = lo;
        }
      }
      if (wave % 2 == 0 && g == 0) {
#pragma unroll
        for (int h = 0; h < F::SETS; ++h) a8s[(at + (int64_t)h * a_rows * (I / 128)) * 4 + n / 32] = (uint8_t)(s - 8 * h);
      }
    } else {
      const int wm = wave / 4, wn = wave % 4, g = lane / 32, row = 32 * wm + lane % 32;
      if (32 * wm >= rows) return;  // uniform
      float v[F::MI][2][4], amax = 0.0f;
#pragma unroll
      for (int mi = 0; mi < F::MI; ++mi)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          v[mi][i / 4][i % 4] = act(acc.v[mi][i], acc.v[mi][i + 8]);
          amax = fmaxf(amax, fabsf(v[mi][i / 4][i % 4]));
        }
      amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
      const int s = fp8_term_exponent(amax);
      // words [term][8-column group 2 mi + q] of columns 4 g .. + 3 of the group; two swaps between the lane
      // halves (groups of a tile, then tiles) leave each lane the 16 columns of weight tile g
      uint32_t w[2][4];
#pragma unroll
      for (int c = 0; c < 4; ++c) fp8_terms4(v[c / 2][c % 2], pow2_biased(254 - s), w[0][c], w[1][c]);
      const int n = t.nt * TG + 32 * wn;  // the wave's first column
      const int64_t at = (int64_t)(t.begin + row) * (I / 128);
      uint8_t* dst = a8 + (at + n / 128) * XSTEP8 + n % 128 + 16 * g;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        uint32_t o[4];
#pragma unroll
        for (int q = 0; q < 2; ++q) {  // group q of tile 0 and of tile 1
          const auto pr = __builtin_amdgcn_permlane32_swap(w[e][q], w[e][2 + q], false, false);
          o[2 * q] = pr[0];
          o[2 * q + 1] = pr[1];
        }
        if (row < rows) *reinterpret_cast<uint4*>(dst + 128 * e) = make_uint4(o[0], o[1], o[2], o[3]);
      }
      if (row < rows && g == 0) a8s[at * 4 + n / 32] = (uint8_t)s;
    }
  };
  stream_tiles<F>(tr, H / 128, lds, wave, lane, locate, setup, epilogue);
}

// Output rows (bf16, permuted order) of TW columns, 32 a weight tile.
template <typename F, typename Table>
__device__ __forceinline__ void stream_down(uint8_t* lds, const uint8_t* __restrict__ a8, const uint8_t* __restrict__ a8s,
                                            const Lists& all, const Table& routed, const Table& shared, int before,
                                            int a_rows, void* __restrict__ out_rows) {
  uint16_t* __restrict__ out = (uint16_t*)out_rows;
  const Lists L = resident_lists<F>(all, shared);
  const int H = routed.hidden, I = routed.inter;
  const int n_tiles = (H + F::TW - 1) / F::TW;
  const TileRange tr = tile_range_after(active_row_tiles<F::ROWS>(L) * n_tiles, before, F::HOT_COST);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  auto locate = [&](int j, StreamTile<F>& t) { stream_locate<F>(L, tr.at(j), n_tiles, t); };
  auto setup = [&](StreamTile<F>& t) {
    const TileWeights tw = tile_weights_s(routed, shared, t.expert);
    // a multiple of 128; the rows past a narrow last tile's columns read its first ones
    const int col0 = t.nt * F::TW, valid = min(F::TW, H - col0);
    t.ld.weights(tw.w2, tw.w2s, H, I, table_tiled(routed), wave, lane, [=](int j) { return col0 + j % valid; });
    if constexpr (F::BLOCK_F32)
      t.s0 = t.s1 = uniform_ptr(reinterpret_cast<const float*>(tw.w2s) +
                                (int64_t)((col0 + 64 * (wave % 4) % valid) / 128) * (I / 128));
    const int begin = t.begin, end = t.end;
    t.ld.rows(a8, a8s, I, wave, lane, [&](int r) {
      const int q = begin + r % F::ROWS;
      return (q < end ? q : begin) + r / F::ROWS * a_rows;
    });
  };
  auto epilogue = [&](const StreamTile<F>& t, StreamAcc<F>& acc) {
    const int col = t.nt * F::TW + (F::BM == 16 ? 32 * wave : 64 * (wave % 4));
    if (col >= H) return;
    if constexpr (F::WIDE) {  // fp32 rows
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc.q[q][i] = sum_sets<F>(acc.q[q][i], lane);
      const int row = t.begin + lane % 16;
      if (lane % 16 >= F::ROWS || row >= t.end) return;
      float* dst = (float*)out_rows + (int64_t)row * H + col + lane / 16 * 4;
#pragma unroll
      for (int q = 0; q < 2; ++q) *reinterpret_cast<v4f*>(dst + 16 * q) = acc.q[q];
    } else {
      const int row0 = t.begin + (F::BM == 16 ? 0 : 32 * (wave / 4)), row = row0 + lane % 32, g = lane / 32;
      if (row0 >= t.end) return;  // uniform
      // a swap between the lane halves gives each lane 8 columns in a row: stores of 16 bytes
#pragma unroll
      for (int mi = 0; mi < F::MI; ++mi)
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const v16f& a = acc.v[mi];
          uint32_t o[4];
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const auto pr = __builtin_amdgcn_permlane32_swap(pack_bf16x2(a[8 * p + 2 * q], a[8 * p + 2 * q + 1]),
                                                             pack_bf16x2(a[8 * p + 4 + 2 * q], a[8 * p + 4 + 2 * q + 1]),
                                                             false, false);
            o[q] = pr[0];
            o[2 + q] = pr[1];
          }
          if (row < t.end)
            *reinterpret_cast<uint4*>(out + (int64_t)row * H + col + 32 * mi + 16 * p + 8 * g) = make_uint4(o[0], o[1], o[2], o[3]);
        }
    }
  };
  stream_tiles<F>(tr, I / 128, lds, wave, lane, locate, setup, epilogue);
}

// 16-row tiles alone.
template <typename F, typename Table>
__global__ void __launch_bounds__(64 * F::WAVES, 2) stream_gate_up_kernel(const uint8_t* __restrict__ x8,
                                                                          const uint8_t* __restrict__ x8s,
                                                                          const int32_t* __restrict__ row_token, Lists L,
                                                                          Table routed, Table shared, int x_rows,
                                                                          int a_rows, uint8_t* __restrict__ a8,
                                                                          uint8_t* __restrict__ a8s) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[F::BYTES];
  stream_gate_up<F>(lds, x8, x8s, row_token, L, routed, shared, 0, x_rows, a_rows, a8, a8s);
}
template <typename F, typename Table>
__global__ void __launch_bounds__(64 * F::WAVES, 2) stream_down_kernel(const uint8_t* __restrict__ a8,
                                                                       const uint8_t* __restrict__ a8s, Lists L,
                                                                       Table routed, Table shared, int a_rows,
                                                                       void* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[F::BYTES];
  stream_down<F>(lds, a8, a8s, L, routed, shared, 0, a_rows, out);
}

// 128-row tiles of the experts with more than 64 rows (`hot`), then 64-row tiles of the others
// (`cold`, one tile an expert, so its weights are read once). One launch, so that the workgroups
// with a 128-row tile less take more of the others (tile_range_after: with routing as skewed as
// natural text's, 2048 tokens over 128 MXFP4 experts of 2048/768, 303 us without and 249 with).
template <typename F>
using StreamOf = StreamF<F::FP8, F::A_SCALED, 64, 8>;
template <typename F>
constexpr int MIXED_LDS = RingMx<F, F::DA, F::DB>::BYTES > StreamOf<F>::BYTES ? RingMx<F, F::DA, F::DB>::BYTES
                                                                              : StreamOf<F>::BYTES;

template <typename Table>
struct MixedArgs {
  const uint8_t *terms, *scales;  // x's (gate_up) or act's (down)
  const int32_t* row_token;
  Lists hot, cold;
  Table routed, shared;
  uint8_t* a8;
  uint32_t* a8s;
  uint16_t* out;
};
// The launch's arguments read again from its argument buffer. The second part's copies of pointers and table fields
// otherwise live through the first, whose tiles then spill and reload scalar registers at each set-up.
template <typename Args>
__device__ __forceinline__ const Args& args_again() {
  auto p = __builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const Args*)p;
}

template <typename F, typename Table>
__global__ void __launch_bounds__(512, 2) mixed_gate_up_kernel(MixedArgs<Table> a) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[MIXED_LDS<F>];
  gate_up_mx<F, F::DA, F::DB>(lds, a.terms, a.scales, a.row_token, a.hot, a.routed, a.shared, a.a8, a.a8s);
  ring_wait_all();  // no load into the rings and no LDS access of the first part is left
  const MixedArgs<Table>& b = args_again<MixedArgs<Table>>();
  stream_gate_up<StreamOf<F>>(lds, b.terms, b.scales, b.row_token, b.cold, b.routed, b.shared,
                              active_row_tiles(b.hot) * ((b.routed.inter + F::TW / 2 - 1) / (F::TW / 2)), 0, 0, b.a8,
                              (uint8_t*)b.a8s);
}
template <typename F, typename Table>
__global__ void __launch_bounds__(512, 2) mixed_down_kernel(MixedArgs<Table> a) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[MIXED_LDS<F>];
  down_mx<F, F::DA, F::DB>(lds, a.terms, a.scales, a.hot, a.routed, a.shared, a.out);
  ring_wait_all();
  const MixedArgs<Table>& b = args_again<MixedArgs<Table>>();
  stream_down<StreamOf<F>>(lds, b.terms, b.scales, b.cold, b.routed, b.shared,
                           active_row_tiles(b.hot) * ((b.routed.hidden + F::TW - 1) / F::TW), 0, b.out);
}

}  // namespace mf
}  // namespace wm
