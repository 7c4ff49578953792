// FP8 / bf16 MFMA GEMMs of the FP8 MLP block (gfx950, CDNA4).
//
// Every GEMM here is C[m, n] = sum_k A[m, k] * B[n, k]: both operands are
// K-contiguous rows in HBM, except that a weight gradient (K = tokens) may
// read either operand as the token-major activation its producer wrote,
// through transposing LDS reads (MainLoop TR_A / TR_B).  One work-group
// computes an output tile with the pipelined main loop of mainloop.h: 256 x 256
// by 8 waves of 128 x 64, 192 x 256 or 128 x 256 by 8, 128 x 128 by 4 of 64 x 64
// (Tile below), each wave's share as blocks of 32 x 32 MFMA accumulators.
//
// MFMA: v_mfma_f32_32x32x64_f8f6f4 (e4m3/e5m2 chosen per operand) or
// v_mfma_f32_32x32x16_bf16.  The B fragment is passed as the instruction's
// first operand and the A fragment as its second, so each lane holds ONE A
// row (lane % 32) and, in a 32x32 block, 16 accumulators for B-tile rows
// 8*(v/4) + 4*(lane/32) + v%4, v = 0..15.  Within one instruction both
// operands use the same (lane-half, byte) -> k assignment, so any consistent
// placement of K inside a fragment gives the same dot product.
//
// Output-column permutation: the B tile is filled with its rows permuted
// (plain_col_nb, paired_col8 and paired_col64 below), so that accumulator v of
// block nb of the lane in half g is output column  base + 16*nb + v  -- 16 (and
// across blocks 32) consecutive columns per lane.  Every epilogue access is then a
// 16-byte vector; LDS staging remains only for the transposed copies.
#include "common.h"
#include "mainloop.h"
#include "scale.h"

namespace sfp8 {

// Logical tile lid -> (tm, tn): tile rows in groups of 8, walking the tile
// columns of a group before the next group, so a column of B tiles is reused
// from L2 across the group's A tiles.
SFP8_DEV void raster(int lid, int tiles_m, int tiles_n, int& tm, int& tn) {
  constexpr int G = 8;
  const int group = G * tiles_n;
  const int first_m = (lid / group) * G;
  const int gsz = (tiles_m - first_m) < G ? (tiles_m - first_m) : G;
  tm = first_m + (lid % group) % gsz;
  tn = (lid % group) / gsz;
}

// Work-groups are dispatched round-robin over the 8 XCDs (pid % 8): the
// logical index of work-group pid of nwg when each XCD (with its own L2)
// takes a contiguous run of logical indices (walked from its end with rev).
// A bijection of [0, nwg).
SFP8_DEV int xcd_run(int pid, int nwg, bool rev = false) {
  const int per = nwg >> 3, rem = nwg & 7;
  const int xcd = pid & 7;
  const int len = xcd < rem ? per + 1 : per;
  const int local = rev ? len - 1 - (pid >> 3) : (pid >> 3);
  return (xcd < rem) ? xcd * (per + 1) + local : rem * (per + 1) + (xcd - rem) * per + local;
}

// Work-group -> tile mapping: XCD-contiguous runs of logical tiles, rastered
// as above.  rev: each XCD walks its run backwards, so that a consumer of the
// previous kernel's output (run in the same order, forwards) reads the most
// recently written row blocks first, while they may still be in the memory-
// side cache.
SFP8_DEV void tile_coords(int pid, int nwg, int tiles_m, int tiles_n, int& tm, int& tn, bool rev = false) {
  raster(xcd_run(pid, nwg, rev), tiles_m, tiles_n, tm, tn);
}

// Split-K mapping of a 1-D grid of tiles * splits work-groups.  Work-groups
// are dispatched round-robin over the 8 XCDs (pid % 8); each XCD takes a
// contiguous run of the split-major order (split, tile), so the work-groups
// resident on one XCD read the same K range of A and B (one split, or two
// where a run crosses a split boundary) and share it in that XCD's L2.  With
// splits a multiple of 8 each XCD runs whole splits over every tile; with 2
// or 4 each split takes 8 / splits XCDs (1.5-2 % faster than split-major
// order over all XCDs at 4 and 2 splits).  Tiles of a split are rastered as
// in tile_coords.
// The grid may be padded past tiles * splits (wgrad_grid); padding work-groups
// get split = splits and do nothing.
SFP8_DEV void split_tile_coords(int pid, int nwg, int tiles_m, int tiles_n, int splits, int& tm, int& tn,
                                int& split) {
  const int tiles = tiles_m * tiles_n;
  const int lid = xcd_run(pid, nwg);
  split = lid / tiles;
  raster(lid % tiles, tiles_m, tiles_n, tm, tn);
}

// Output column (within the tile) held in B-tile row r, plain layout of NB
// blocks of 32 rows per wave: wave column wn owns rows 32*NB*wn.., lane half g
// of block nb element v (row 32*nb + 8*(v/4) + 4*g + v%4) gets column 32*NB*wn +
// 16*NB*g + 16*nb + v, so a lane's NB blocks cover 16*NB consecutive columns.
template <int NB>
SFP8_DEV int plain_col_nb(int r) {
  const int wn = r / (32 * NB), rl = r % (32 * NB);
  return 32 * NB * wn + 16 * NB * ((rl >> 2) & 1) + 16 * (rl >> 5) + 4 * ((rl >> 3) & 3) + (rl & 3);
}

// Paired (gate/up) layout, 8 waves: rows 0..127 are gate, 128..255 up; wave
// column wn (0..3) owns rows 32*wn.. of each half (one block); column (within
// the 128-column half) 32*wn + 16*g + v.
SFP8_DEV int paired_col8(int r) {
  const int rl = r & 127;
  return 32 * (rl >> 5) + 16 * ((rl >> 2) & 1) + 4 * ((rl >> 3) & 3) + (rl & 3);
}

// B-tile row r of the 128-row paired tile -> (half, column within 64):
// half = r / 64 (gate, up); column = 32*wn + 16*g + v for the lane layout.
SFP8_DEV int paired_col64(int r) {
  const int rl = r & 63, wn = rl >> 5, w = rl & 31;
  return 32 * wn + 16 * ((w >> 2) & 1) + 4 * (w >> 3) + (w & 3);
}

// Copy of an LDS tile (nrows rows of 64 * NP bytes, LDS row stride `stride`)
// into a K-slab matrix: 64-byte column block p of tile row r goes to
// dst + (c0 / 64 + p) * ldrows * 64 + (r0 + r) * 64.  Sixteen consecutive
// threads read one contiguous LDS row (no bank conflicts for NP = 4); the
// global writes are 256-byte runs of 4 rows per block.
template <int NP, int NT = 256>
SFP8_DEV void lds_rows_to_kslab(const uint8_t* lds, int nrows, int stride, uint8_t* dst, int64_t ldrows, int64_t r0,
                                int64_t c0) {
  const int total = nrows * NP * 4;
  for (int idx = threadIdx.x; idx < total; idx += NT) {
    const int ch = idx & 3, pb = (idx >> 2) % NP, r = idx / (4 * NP);
    *reinterpret_cast<intx4*>(dst + (c0 / 64 + pb) * ldrows * 64 + (r0 + r) * 64 + ch * 16) =
        *reinterpret_cast<const intx4*>(lds + r * stride + pb * 64 + ch * 16);
  }
}

SFP8_DEV void store16(void* p, const uint32_t (&w)[4]) {
  *reinterpret_cast<intx4*>(p) = intx4{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
}

// Round 16 accumulators to bf16 (as fp32 values), after scaling by s.
SFP8_DEV void round16_bf16(const floatx16& a, float s, float (&o)[16]) {
#pragma unroll
  for (int v = 0; v < 16; v += 2) {
    const uint32_t p = pack2_bf16(a[v] * s, a[v + 1] * s);
    o[v] = __uint_as_float(p << 16);
    o[v + 1] = __uint_as_float(p & 0xffff0000u);
  }
}

// Tile shapes of the GEMMs below: 64 TB rows by 64 WN columns, 2 WN waves of
// 32 TB x 64.  <4, 4> is 256 x 256 by 8 waves, one work-group per CU, <3, 4>
// the same with 192 rows; <2, 2> is 128 x 128 by 4 waves, two work-groups per
// CU.  The B rows of each are permuted by plain_col_nb<2>,
// or with PAIRED (gate rows in the first half of the B tile, up rows in the
// second) by paired_col8 (WN = 4) and paired_col64 (WN = 2).
template <int TB, int WN>
struct Tile {
  static constexpr int kM = 64 * TB, kN = 64 * WN, kTB = TB, kWN = WN;
  static constexpr int kThreads = 128 * WN;
  static constexpr int kMinWaves = WN == 2 ? 2 : 1;  // per SIMD: two work-groups of 4 waves fit a CU
  template <bool BF16, int FA, int FB, bool TRA = false, bool TRB = false, bool PAIRED = false>
  using Loop = MainLoop<BF16, FA, FB, PAIRED, 2, kStages, TRA, TRB, WN, TB, TB == 3 ? 256 : kM>;
  static constexpr int kLds = Loop<true, 0, 0>::kLds;
  static constexpr int kOutStride = 2 * kN + 16;        // a staged bf16 row
  static constexpr int kPieces = kM * kN / 8 / kThreads;  // 16-byte pieces of it per thread
  // the plan's tile of tile row tm, and that tile row's first row in it
  static SFP8_DEV int plan_tile(int tm) { return tm / (256 / kM); }
  static SFP8_DEV int plan_skip(int tm) { return kM * (tm % (256 / kM)); }
};
template <bool SMALL>
using TileShape = Tile<SMALL ? 2 : 4, SMALL ? 2 : 4>;

// The last round of a kernel of 256 x 256 tiles, one per CU, in halves: when
// the remainder r of a round of nwg work-groups is at most half of it, these
// tiles are split into 128-row halves (half: tm counts rows of 128), a
// work-group each, so that the last round takes half as long.  False: no work
// for this index.  Measured (us): gate/up dgrad, D = 1024, I = 3072, 121 -> 106
// at 320 tiles, 369 -> 341 at 1040; down dgrad 102 -> 94 at 576 tiles, 457 ->
// 447 at 3084; a block's step, T = 20000, D = 1024, I = 2048, 563 -> 549;
// unchanged where the rounds are full.
SFP8_DEV int tail_full(int ntiles, int nwg) {
  const int r = ntiles % nwg;
  return 2 * r <= nwg ? ntiles - r : ntiles;
}
SFP8_DEV bool tail_half(int h, int full, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int tile = full + (h >> 1);
  if (tile >= tiles_m * tiles_n) return false;
  raster(tile, tiles_m, tiles_n, tm, tn);
  tm = 2 * tm + (h & 1);
  return true;
}
constexpr int kRound = 256;  // work-groups of a round: one per CU
SFP8_DEV bool tail_tile(int tiles_m, int tiles_n, int& tm, int& tn, bool& half, bool rev = false) {
  const int full = tail_full(tiles_m * tiles_n, kRound), pid = blockIdx.x;
  half = pid >= full;
  if (half) return tail_half(pid - full, full, tiles_m, tiles_n, tm, tn);
  tile_coords(pid, full, tiles_m, tiles_n, tm, tn, rev);
  return true;
}

// ---------------------------------------------------------------------------
// (a6) gate/up forward + SwiGLU epilogue (spark-gpt train.py:975-1016).
// Tile: 256 tokens x 128 intermediate columns; the B tile holds gate rows
// n0..n0+127 then up rows I+n0..I+n0+127 (paired layout), so a lane holds g and
// u of the same 32 consecutive columns.
// staging row: the tile's 128 (64) bytes of one output, and 16
template <bool SMALL>
constexpr int kEpiStride = SMALL ? 80 : 144;

// With a MoE plan (grouped experts): tile row tm of padded expert order,
// its expert's W8 at w8 + e * w_estride and weight scale wscale[e]; tile
// rows past the plan's count exit.
// 8 waves (two per SIMD): wave (wm, wn) owns tile rows 128*wm.. and the gate
// and up columns 32*wn.. (one 32-column block of each), so the serial
// epilogue of one wave overlaps the other's on the same SIMD.
// SMALL: 128 tokens x 64 columns by 4 waves of 64 rows.
template <bool SMALL>
__global__ __launch_bounds__(TileShape<SMALL>::kThreads, TileShape<SMALL>::kMinWaves) void swiglu_fwd_kernel(
    const uint8_t* __restrict__ x8, const uint8_t* __restrict__ w8, int64_t T, int64_t D, int64_t I,
    const float* __restrict__ scale, const float* __restrict__ wscale, float* __restrict__ amax,
    uint8_t* __restrict__ gu8, uint8_t* __restrict__ h8, uint8_t* __restrict__ h8t, int64_t ldt,
    int tiles_m, int tiles_n, const int* __restrict__ plan, int64_t w_estride) {
  using TS = TileShape<SMALL>;
  constexpr int kN = TS::kM / 2;  // (gate, up) columns of a tile
  constexpr int kWaves = TS::kThreads / 64, kEs = kEpiStride<SMALL>;
  extern __shared__ __align__(16) uint8_t lds[];
  int tm, tn;
  tile_coords(blockIdx.x, gridDim.x, tiles_m, tiles_n, tm, tn);
  if (plan) {
    const MoePlan P{plan};
    const int pt = TS::plan_tile(tm);
    if (pt >= P.ntiles()) return;  // work-group uniform
    const int e = P.expert(pt);
    w8 += e * w_estride;
    wscale += e;
  }
  const int64_t m0 = (int64_t)tm * TS::kM, n0 = (int64_t)tn * kN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  floatx16 acc[TS::kTB][2];  // [tb][0] gate, [tb][1] up
  // K-slab operands: x8 [D/64][ldt][64], w8 [D/64][2I][64]; one K stage of
  // the tile is kM contiguous rows of A and two runs of kN rows of B
  TS::template Loop<false, kFmtE4M3, kFmtE4M3, false, false, true>::run(
      lds, x8 + m0 * kStage, D * ldt - m0 * kStage, [=](int r) { return r * kStage; }, (int)(ldt * kStage), w8,
      D * 2 * I, [=](int r) {
        return ((r / kN) * (int)I + (int)n0 + (SMALL ? paired_col64(r) : paired_col8(r))) * kStage;
      },
      (int)(2 * I * kStage), (int)(D / kStage), acc);
  // All scales are powers of two, so the dequantization factor commutes with
  // every rounding step: with gb, ub = bf16(acc) (unscaled),
  //   g = gb*deq, u = ub*deq, h = (g*sig(g))*u = hb*deq^2, hb = (gb*sig)*ub,
  //   gu8 = e4m3(g*q1) = e4m3(gb*(deq*q1)),  h8 = e4m3(hb*(deq^2*q2)),
  //   amax1 = deq*max(|gb|,|ub|),  amax2 = deq^2*max|hb|.
  // Rows past T are zero in x8 (K-slab padding): they add 0 to the amax and
  // 0 bytes to the padding of h8 and h8t.
  const float deq = 1.0f / (scale[0] * wscale[0]);
  const float c_exp = deq * -1.4426950408889634f;
  const float m1 = deq * scale[1], m2 = deq * deq * scale[2];
  const float inv1 = 1.0f / m1, inv2 = 1.0f / m2;
  const float bnd1 = kE4M3Max * inv1, bnd2 = kE4M3Max * inv2;
  // epilogue LDS: the tile's g8, u8 and h8 bytes (kM x kN each), then the amax slots
  uint8_t* Gt = lds;
  uint8_t* Ut = lds + TS::kM * kEs;
  uint8_t* Ht = lds + 2 * TS::kM * kEs;
  float* red = reinterpret_cast<float*>(lds + 3 * TS::kM * kEs);
  float m_gu = 0.f, m_h = 0.f;
  const int fr = lane & 31, g = lane >> 5;
  const int cb = 32 * wn + 16 * g;  // first of this lane's 16 columns
  // g, u (bf16-rounded, unscaled) and h of unit (tb, q): 4 columns
  auto unit = [&](int tb, int q, float (&gb)[4], float (&ub)[4], float (&hb)[4]) {
    // g, u rounded to bf16 as in the bf16 path (train.py:1006-1007)
#pragma unroll
    for (int e = 0; e < 4; e += 2) {
      const uint32_t pg = pack2_bf16(acc[tb][0][4 * q + e], acc[tb][0][4 * q + e + 1]);
      const uint32_t pu = pack2_bf16(acc[tb][1][4 * q + e], acc[tb][1][4 * q + e + 1]);
      gb[e] = __uint_as_float(pg << 16);
      gb[e + 1] = __uint_as_float(pg & 0xffff0000u);
      ub[e] = __uint_as_float(pu << 16);
      ub[e + 1] = __uint_as_float(pu & 0xffff0000u);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float sg = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(gb[e] * c_exp));
      hb[e] = gb[e] * sg * ub[e];
    }
  };
#pragma unroll
  for (int tb = 0; tb < TS::kTB; ++tb) {
    const int row = 32 * TS::kTB * wm + 32 * tb + fr;  // token within the tile
    uint32_t gw[4], uw[4], hw[4];
    bool bad = false;
    {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float gb[4], ub[4], hb[4];
        unit(tb, q, gb, ub, hb);
        // NaN-propagating maxima: inside the e4m3 range (after scaling) the
        // unclamped conversions are exact; otherwise the row block is redone
        float a = max3_nan(fabsf(gb[0]), fabsf(ub[0]), fabsf(gb[1]));
        a = max3_nan(a, fabsf(ub[1]), fabsf(gb[2]));
        a = max3_nan(a, fabsf(ub[2]), fabsf(gb[3]));
        a = __builtin_elementwise_maximum(a, fabsf(ub[3]));
        float b = max3_nan(fabsf(hb[0]), fabsf(hb[1]), fabsf(hb[2]));
        b = __builtin_elementwise_maximum(b, fabsf(hb[3]));
        bad |= !(a <= bnd1) | !(b <= bnd2);
        m_gu = fmaxf(m_gu, a);  // a NaN here is redone by the exact path
        m_h = fmaxf(m_h, b);
        const int k = q;
        gw[k] = pack4_e4m3_scaled_noclamp(gb[0], gb[1], gb[2], gb[3], inv1, 0u);
        uw[k] = pack4_e4m3_scaled_noclamp(ub[0], ub[1], ub[2], ub[3], inv1, 0u);
        hw[k] = pack4_e4m3_scaled_noclamp(hb[0], hb[1], hb[2], hb[3], inv2, 0u);
      }
    }
    if (__builtin_amdgcn_ballot_w64(bad)) {  // wave-uniform; NaN or out-of-range data only
      asm volatile("" ::: "memory");
      {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float gb[4], ub[4], hb[4];
          unit(tb, q, gb, ub, hb);
#pragma unroll
          for (int e = 0; e < 4; ++e) {  // amax over the non-NaN values
            m_gu = fmaxf(m_gu, fmaxf(fabsf(gb[e]), fabsf(ub[e])));
            m_h = fmaxf(m_h, fabsf(hb[e]));
          }
          const int k = q;
          gw[k] = fix_nan4(pack4_e4m3_scaled(gb[0], gb[1], gb[2], gb[3], inv1, bnd1), gb[0], gb[1], gb[2], gb[3]);
          uw[k] = fix_nan4(pack4_e4m3_scaled(ub[0], ub[1], ub[2], ub[3], inv1, bnd1), ub[0], ub[1], ub[2], ub[3]);
          hw[k] = fix_nan4(pack4_e4m3_scaled(hb[0], hb[1], hb[2], hb[3], inv2, bnd2), hb[0], hb[1], hb[2], hb[3]);
        }
      }
    }
    store16(Gt + row * kEs + cb, {gw[0], gw[1], gw[2], gw[3]});
    store16(Ut + row * kEs + cb, {uw[0], uw[1], uw[2], uw[3]});
    store16(Ht + row * kEs + cb, {hw[0], hw[1], hw[2], hw[3]});
  }
  m_gu *= deq;
  m_h *= deq * deq;
  __syncthreads();
  // gu8 (gate and up halves) and h8 as 64-column K-slab blocks (every tile
  // row: rows past T are zero padding), then, when asked for, the
  // token-contiguous h8t
  lds_rows_to_kslab<kN / 64, TS::kThreads>(Gt, TS::kM, kEs, gu8, ldt, m0, n0);
  lds_rows_to_kslab<kN / 64, TS::kThreads>(Ut, TS::kM, kEs, gu8, ldt, m0, I + n0);
  lds_rows_to_kslab<kN / 64, TS::kThreads>(Ht, TS::kM, kEs, h8, ldt, m0, n0);
  if (h8t) {
    if constexpr (SMALL) {
      lds_rows_store_slab_tr<64, kWaves>(Ht, kN, kEs, h8t, slab_rows(I), m0, n0);
      lds_rows_store_slab_tr<64, kWaves>(Ht + 64 * kEs, kN, kEs, h8t, slab_rows(I), m0 + 64, n0);
    } else {
      lds_tile_store_slab_tr<8, 8>(Ht, kEs, h8t, slab_rows(I), m0, n0);
    }
  }
  m_gu = wave_max(m_gu);
  m_h = wave_max(m_h);
  if (lane == 0) { red[wave] = m_gu; red[kWaves + wave] = m_h; }
  __syncthreads();
  if (tid == 0) {
    float a1 = red[0], a2 = red[kWaves];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) {
      a1 = fmaxf(a1, red[w]);
      a2 = fmaxf(a2, red[kWaves + w]);
    }
    atomic_max_nonneg(amax + 1, a1);
    atomic_max_nonneg(amax + 2, a2);
  }
}

// ---------------------------------------------------------------------------
// (a6) gate/up forward + SwiGLU, persistent with a deferred epilogue.
//
// Tile 256 tokens x 64 (gate, up) column pairs: B tile = 64 gate rows + 64 up
// rows (MainLoop NB = 2, paired), so each lane holds g and u of the same 16
// consecutive columns for each of its TB row blocks.  One work-group per CU
// walks its tiles; after tile i's K loop the lane packs bf16(g), bf16(u) of
// its 16 TB pairs into registers (E), and the SwiGLU of tile i runs in 4 TB
// units of 4 pairs over the K stages of tile i+1, in the same instruction
// stream as its MFMAs (the matrix pipe runs them while the vector ALU does the
// epilogue): each unit in six pieces, spread evenly after the MFMAs past the
// stages' barriers (one per MFMA at NK = 16, two at 8, four at 4; there the
// vector ALU, not the matrix core, sets the pace).  The h bytes of a tile also
// go to one of two LDS tiles; its token-contiguous (K-slab) copy is written at
// the next tile boundary with LDS transpose reads.  The last tile's epilogue
// runs alone.
// NK = D / 64 K stages, fully unrolled so each piece has a fixed stage; the K
// stream runs on across tiles (the last three stages of a tile load the next
// tile's first three), so a tile boundary waits for no DMA.
constexpr int kPipeHStride = 80;                    // 64 h bytes + 16 per LDS row
constexpr int kPipeHBytes = kTile * kPipeHStride;   // one h tile
constexpr int kPipeRing = MainLoop<false, kFmtE4M3, kFmtE4M3, true, 2, 4>::kLds;  // 96 KiB
constexpr int kPipeLds = kPipeRing + 2 * kPipeHBytes + 64;
// the pipe's waves: 8 of 64 x 64 (two row blocks each)
constexpr int kPipeTB = 2;
constexpr int kPipeThreads = kPipeTB == 4 ? 256 : 512;

// The h tile's 256 rows of 64 bytes to 256 consecutive K-slab rows (NT
// threads, 16 bytes each per pass).
template <int NT>
SFP8_DEV void pipe_h8_rows(const uint8_t* hbuf, uint8_t* dst) {
#pragma unroll
  for (int k = 0; k < 1024 / NT; ++k) {
    const int idx = NT * k + (int)threadIdx.x, r = idx >> 2, ch = idx & 3;
    *reinterpret_cast<intx4*>(dst + r * 64 + 16 * ch) =
        *reinterpret_cast<const intx4*>(hbuf + r * kPipeHStride + 16 * ch);
  }
}

// TB = row blocks of 32 per wave: 4 (4 waves of 128 x 64) or 2 (8 waves of
// 64 x 64, two per SIMD: each wave's waits are covered by the other's
// MFMAs).
template <int NK, int TB>
struct SwigluPipe {
  using ML = MainLoop<false, kFmtE4M3, kFmtE4M3, true, 2, 4, false, false, 2, TB>;
  static constexpr int kWaves = ML::kWaves, kWM = ML::kWM;
  static constexpr int kUnits = 4 * TB;  // 4 pairs each: unit u = row block u/4, pairs 4*(u%4) ..
  static constexpr int kSt = 4;          // LDS ring stages
  static constexpr int kDma = ML::kDma;
  static constexpr int kPre = TB == 4 ? 2 : 1;  // MFMAs of a stage issued before its wait
  static constexpr int kSlots = ML::kMfma - kPre;  // MFMAs past the barrier, one slot each
  static constexpr int kDmaSlots = TB == 4 ? 2 : kSlots;  // slots carrying the DMA
  static_assert(NK >= kSt && NK % kSt == 0, "whole rings of K stages: a tile's stage s sits in slot s % kSt");
  // the units' pieces, six each, fill the tile's slots in order
  static constexpr int kPer = 6 * kUnits / (NK * kSlots);  // pieces per slot
  static_assert(kPer * NK * kSlots == 6 * kUnits, "whole pieces per slot");
  // row blocks whose units are complete after stage KT
  static constexpr int blocks_done(int kt) { return (kt + 1) * kSlots * kPer / 24; }

  // A unit's working values between its pieces.
  struct UnitTmp {
    float gb[4], ub[4], hb[4], ex[4], sg[4];
  };

  struct Ctx {
    // main loop; the last kSt - 1 stages of a tile load the first stages of
    // the next tile (nra, nvoff_b), or repeat this tile's last stage when
    // there is none (has_next false: nra, nvoff_b = ra, voff_b)
    uint8_t* lds;
    __amdgpu_buffer_rsrc_t ra, rb, nra, nrb;
    uint32_t voff_a[4], voff_b[2], nvoff_b[2], aoff[8], boff[8];
    bool has_next;
    int wave;
    typename ML::Frag f[2];
    floatx16 acc[TB][2];
    // previous tile's epilogue
    uint32_t E[TB][16];
    uint32_t gw[4], uw[4], hw[4];
    UnitTmp ut;  // the current unit's working values (its pieces may span two stages)
    bool bad;  // a unit of the current row block saw NaN or out-of-range data
    float m_gu, m_h;
    bool prev;            // a previous tile exists
    int64_t pm0, pn0;     // its origin
    uint8_t* hbuf;        // its LDS h tile
    // scales (of the previous tile's weight: the epilogue's) and outputs
    float deq, c_exp, inv1, bnd1, inv2, bnd2;
    float s0, s1, s2;  // scale[0], scale[1], scale[2]
    float mx_gu, mx_h;  // amax so far, dequantized
    int64_t T, I, ldt;
    // gu8 (the K-slab [2I/64][ldt][64]) and the previous tile's byte offsets
    // in it: gate block (pn0/64, rows pm0..) and up block (I + pn0)/64
    __amdgpu_buffer_rsrc_t rgu;
    uint32_t so_g, so_u;
    uint8_t* h8;
  };

  // One unit: 4 pairs of row block TB, packed into byte Q of gw/uw/hw.
  template <int U>
  static SFP8_DEV void unit_compute(Ctx& c) {
    constexpr int RB = U / 4, Q = U % 4;
    float gb[4], ub[4], hb[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t p = c.E[RB][4 * Q + e];
      gb[e] = __uint_as_float(p << 16);
      ub[e] = __uint_as_float(p & 0xffff0000u);
      const float sg = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(gb[e] * c.c_exp));
      hb[e] = gb[e] * sg * ub[e];
    }
    // NaN-propagating maxima of the magnitudes: when both are inside the
    // e4m3 range (after scaling) no clamp can act and no NaN needs patching,
    // so the unclamped conversions are exact; otherwise the row block's
    // block_store redoes them (wave-uniform, rare)
    float a = max3_nan(fabsf(gb[0]), fabsf(ub[0]), fabsf(gb[1]));
    a = max3_nan(a, fabsf(ub[1]), fabsf(gb[2]));
    a = max3_nan(a, fabsf(ub[2]), fabsf(gb[3]));
    a = __builtin_elementwise_maximum(a, fabsf(ub[3]));
    float b = max3_nan(fabsf(hb[0]), fabsf(hb[1]), fabsf(hb[2]));
    b = __builtin_elementwise_maximum(b, fabsf(hb[3]));
    c.bad |= !(a <= c.bnd1) | !(b <= c.bnd2);
    c.m_gu = fmaxf(c.m_gu, a);  // a NaN here is redone by the exact path
    c.m_h = fmaxf(c.m_h, b);
    c.gw[Q] = pack4_e4m3_scaled_noclamp(gb[0], gb[1], gb[2], gb[3], c.inv1, c.gw[Q]);
    c.uw[Q] = pack4_e4m3_scaled_noclamp(ub[0], ub[1], ub[2], ub[3], c.inv1, c.uw[Q]);
    c.hw[Q] = pack4_e4m3_scaled_noclamp(hb[0], hb[1], hb[2], hb[3], c.inv2, c.hw[Q]);
  }

  // Piece P of unit U: the arithmetic of unit_compute<U>, the same
  // operations in the same order per value, cut into six parts that go one
  // after each of the stage's MFMAs past the barrier and software-pipelined
  // over the unit's four pairs (the exponent of a pair one piece before its
  // reciprocal), so that each part holds at most two transcendental
  // instructions (a quarter of the vector ALU's rate) beside independent
  // others.  A wave issues in order: more vector work between two MFMAs
  // than the first one's 64 cycles holds back the second.  Each part reads
  // its inputs and publishes its results through empty asm statements, so
  // the compiler keeps it in its slot.
  template <int RB, int Q, int E>
  static SFP8_DEV void unit_unpack(Ctx& c, UnitTmp& t) {
    uint32_t p = c.E[RB][4 * Q + E];
    asm volatile("" : "+v"(p));
    t.gb[E] = __uint_as_float(p << 16);
    t.ub[E] = __uint_as_float(p & 0xffff0000u);
    t.ex[E] = __builtin_amdgcn_exp2f(t.gb[E] * c.c_exp);
  }
  template <int U, int P>
  static SFP8_DEV void unit_piece(Ctx& c, UnitTmp& t) {
    constexpr int RB = U / 4, Q = U % 4;
    if constexpr (P == 0) {
      unit_unpack<RB, Q, 0>(c, t);
      unit_unpack<RB, Q, 1>(c, t);
      asm volatile("" ::"v"(t.ex[0]), "v"(t.ex[1]));
    } else if constexpr (P == 1) {
      t.sg[0] = __builtin_amdgcn_rcpf(1.0f + t.ex[0]);
      t.sg[1] = __builtin_amdgcn_rcpf(1.0f + t.ex[1]);
      unit_unpack<RB, Q, 2>(c, t);
      asm volatile("" ::"v"(t.sg[0]), "v"(t.sg[1]), "v"(t.ex[2]));
    } else if constexpr (P == 2) {
      unit_unpack<RB, Q, 3>(c, t);
      t.sg[2] = __builtin_amdgcn_rcpf(1.0f + t.ex[2]);
      t.hb[0] = t.gb[0] * t.sg[0] * t.ub[0];
      t.hb[1] = t.gb[1] * t.sg[1] * t.ub[1];
      asm volatile("" ::"v"(t.ex[3]), "v"(t.sg[2]), "v"(t.hb[0]), "v"(t.hb[1]));
    } else if constexpr (P == 3) {
      t.sg[3] = __builtin_amdgcn_rcpf(1.0f + t.ex[3]);
      t.hb[2] = t.gb[2] * t.sg[2] * t.ub[2];
      // NaN-propagating maximum of the gate and up magnitudes: inside the
      // e4m3 range (after scaling) no clamp can act and no NaN needs
      // patching, so the unclamped conversions are exact; otherwise the row
      // block's block_store redoes them (wave-uniform, rare)
      float a = max3_nan(fabsf(t.gb[0]), fabsf(t.ub[0]), fabsf(t.gb[1]));
      a = max3_nan(a, fabsf(t.ub[1]), fabsf(t.gb[2]));
      a = max3_nan(a, fabsf(t.ub[2]), fabsf(t.gb[3]));
      a = __builtin_elementwise_maximum(a, fabsf(t.ub[3]));
      c.bad |= !(a <= c.bnd1);
      c.m_gu = fmaxf(c.m_gu, a);  // a NaN here is redone by the exact path
      asm volatile("" ::"v"(t.sg[3]), "v"(t.hb[2]), "v"(c.m_gu));
    } else if constexpr (P == 4) {
      t.hb[3] = t.gb[3] * t.sg[3] * t.ub[3];
      float b = max3_nan(fabsf(t.hb[0]), fabsf(t.hb[1]), fabsf(t.hb[2]));
      b = __builtin_elementwise_maximum(b, fabsf(t.hb[3]));
      c.bad |= !(b <= c.bnd2);
      c.m_h = fmaxf(c.m_h, b);
      c.gw[Q] = pack4_e4m3_scaled_noclamp(t.gb[0], t.gb[1], t.gb[2], t.gb[3], c.inv1, c.gw[Q]);
      asm volatile("" ::"v"(c.m_h), "v"(c.gw[Q]));
    } else {
      c.uw[Q] = pack4_e4m3_scaled_noclamp(t.ub[0], t.ub[1], t.ub[2], t.ub[3], c.inv1, c.uw[Q]);
      c.hw[Q] = pack4_e4m3_scaled_noclamp(t.hb[0], t.hb[1], t.hb[2], t.hb[3], c.inv2, c.hw[Q]);
      asm volatile("" ::"v"(c.uw[Q]), "v"(c.hw[Q]));
    }
  }

  // After the last unit of row block TB: the exact conversions when a unit
  // of the block saw NaN or out-of-range data (wave-uniform, rare), the
  // three 16-byte global stores and the h bytes into the LDS tile.
  template <int RB>
  static SFP8_DEV void block_store(Ctx& c) {
    const int lane = threadIdx.x & 63, wm = c.wave % kWM, wn = c.wave / kWM;
    const int fr = lane & 31, g = lane >> 5;
    if (__builtin_amdgcn_ballot_w64(c.bad)) {
      asm volatile("" ::: "memory");
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float gb[4], ub[4], hb[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t p = c.E[RB][4 * q + e];
          gb[e] = __uint_as_float(p << 16);
          ub[e] = __uint_as_float(p & 0xffff0000u);
          const float sg = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(gb[e] * c.c_exp));
          hb[e] = gb[e] * sg * ub[e];
          // amax over the non-NaN values
          c.m_gu = fmaxf(c.m_gu, fmaxf(fabsf(gb[e]), fabsf(ub[e])));
          c.m_h = fmaxf(c.m_h, fabsf(hb[e]));
        }
        c.gw[q] = fix_nan4(pack4_e4m3_scaled(gb[0], gb[1], gb[2], gb[3], c.inv1, c.bnd1), gb[0], gb[1], gb[2], gb[3]);
        c.uw[q] = fix_nan4(pack4_e4m3_scaled(ub[0], ub[1], ub[2], ub[3], c.inv1, c.bnd1), ub[0], ub[1], ub[2], ub[3]);
        c.hw[q] = fix_nan4(pack4_e4m3_scaled(hb[0], hb[1], hb[2], hb[3], c.inv2, c.bnd2), hb[0], hb[1], hb[2], hb[3]);
      }
    }
    c.bad = false;
    const int row = 32 * TB * wm + 32 * RB + fr;
    const int col = 32 * wn + 16 * g;
    if (c.prev) {
      // gu8 is a K-slab [2I/64][ldt][64], h8 one of [I/64][ldt][64]: the
      // tile's 64 gate, 64 up and 64 h columns are one block each (rows past
      // T hold the zeros computed from x8's zero padding); the block's origin
      // goes in the vector offset (Bf16Pipe::row_write says why)
      const uint32_t vo = (uint32_t)(row * 64 + col);
      __builtin_amdgcn_raw_buffer_store_b128(intx4{(int)c.gw[0], (int)c.gw[1], (int)c.gw[2], (int)c.gw[3]},
                                             c.rgu, vo + c.so_g, 0, 0);
      __builtin_amdgcn_raw_buffer_store_b128(intx4{(int)c.uw[0], (int)c.uw[1], (int)c.uw[2], (int)c.uw[3]},
                                             c.rgu, vo + c.so_u, 0, 0);
    }
    store16(c.hbuf + row * kPipeHStride + col, c.hw);
  }

  // Stage KT: the first kPre MFMAs, then the wait for stage KT+1 and the
  // barrier, then six slots (slot below), then the row-block stores the
  // stage's unit completed.  vmcnt counts loads and stores and falls in
  // issue order.  The wait allows the kDma operations issued last: all of
  // them the previous stage's loads, or after a stage that stored (which not
  // every one does: c.prev) its stores and fewer of its loads, which are then
  // waited for a stage early.
  template <int KT>
  static SFP8_DEV void stage(Ctx& c, int a_ss, int b_ss) {
    constexpr int cur = KT & 1, nxt = cur ^ 1;
    // the first kPre MFMAs (register operands only) go ahead of the wait,
    // so the matrix core stays busy while it blocks
    ML::template mfma_range<0, kPre>(c.f[cur], c.acc);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kDma * (kSt - 3)) : "memory");
    __builtin_amdgcn_sched_barrier(0);
    slots<KT, 0>(c, c.ut, a_ss, b_ss);
    // the stage that finishes a row block's last unit stores it
    if constexpr (blocks_done(KT) > blocks_done(KT - 1)) block_store<blocks_done(KT) - 1>(c);
  }
  template <int KT, int J>
  static SFP8_DEV void slots(Ctx& c, UnitTmp& t, int a_ss, int b_ss) {
    if constexpr (J < kSlots) {
      slot<KT, J>(c, t, a_ss, b_ss);
      slots<KT, J + 1>(c, t, a_ss, b_ss);
    }
  }

  // Slot J of stage KT: one MFMA past the barrier, then (J < 2) half of the
  // DMA of stage KT+3 (of the next tile past the last stage), one fragment
  // of stage KT+1 (B blocks first: the next stage's first MFMAs use b[0],
  // b[1] and a[0]) and the slot's pieces of the epilogue units; the scheduling
  // barrier keeps the slot's work after its MFMA.
  template <int KT, int J>
  static SFP8_DEV void slot(Ctx& c, UnitTmp& t, int a_ss, int b_ss) {
    constexpr int cur = KT & 1, nxt = cur ^ 1;
    ML::template mfma_range<kPre + J, kPre + J + 1>(c.f[cur], c.acc);
    if constexpr (J < kDmaSlots) {
      constexpr int slot_ = (KT + kSt - 1) % kSt;
#pragma unroll
      for (int j = J * kDma / kDmaSlots; j < (J + 1) * kDma / kDmaSlots; ++j) {
        if constexpr (KT + kSt - 1 < NK) {
          constexpr int ld = KT + kSt - 1;
          ML::load_one(j, c.lds, slot_, c.ra, c.rb, c.voff_a, c.voff_b, stage_off<ld>(a_ss), stage_off<ld>(b_ss),
                       c.wave);
        } else {
          const int ld = c.has_next ? KT + kSt - 1 - NK : NK - 1;
          ML::load_one(j, c.lds, slot_, c.nra, c.nrb, c.voff_a, c.nvoff_b, ld * a_ss, ld * b_ss, c.wave);
        }
      }
    }
    if constexpr (TB == 4) {
      ML::template read_frag<J < 2 ? 4 + J : J - 2>(c.lds, (KT + 1) % kSt, c.aoff, c.boff, c.f[nxt]);
    } else if constexpr (J == 0) {
      // a[0] and b[0] first (the next stage's MFMA ahead of its wait), then
      // b[1], then a[1]
      ML::template read_frag<0>(c.lds, (KT + 1) % kSt, c.aoff, c.boff, c.f[nxt]);
      ML::template read_frag<2>(c.lds, (KT + 1) % kSt, c.aoff, c.boff, c.f[nxt]);
    } else {
      ML::template read_frag<J == 1 ? 3 : 1>(c.lds, (KT + 1) % kSt, c.aoff, c.boff, c.f[nxt]);
    }
    pieces<(KT * kSlots + J) * kPer, kPer>(c, t);
    __builtin_amdgcn_sched_barrier(0);
  }
  // Pieces P .. P + N - 1 of the tile's units, in order.
  template <int P, int N>
  static SFP8_DEV void pieces(Ctx& c, UnitTmp& t) {
    if constexpr (N > 0) {
      unit_piece<P / 6, P % 6>(c, t);
      pieces<P + 1, N - 1>(c, t);
    }
  }

  // Stage LD's byte offset LD * ss, computed where it is used (otherwise
  // the products for all fixed stages stay live in scalar registers across
  // the tile loop).
  template <int LD>
  static SFP8_DEV int stage_off(int ss) {
    asm volatile("" : "+s"(ss));
    return LD * ss;
  }

  template <int KT>
  static SFP8_DEV void stages(Ctx& c, int a_ss, int b_ss) {
    if constexpr (KT < NK) {
      stage<KT>(c, a_ss, b_ss);
      stages<KT + 1>(c, a_ss, b_ss);
    }
  }
  template <int U0>
  static SFP8_DEV void tail_units(Ctx& c) {
    if constexpr (U0 < kUnits) {
      unit_compute<U0>(c);
      if constexpr (U0 % 4 == 3) block_store<U0 / 4>(c);
      tail_units<U0 + 1>(c);
    }
  }

  // The finished epilogue's maxima, dequantized with its tile's scale, join
  // the running amax (exact: the scales are powers of two); then the next
  // epilogue's constants for weight scale q (all powers of two).
  static SFP8_DEV void next_scales(Ctx& c, float q) {
    c.mx_gu = fmaxf(c.mx_gu, c.m_gu * c.deq);
    c.mx_h = fmaxf(c.mx_h, c.m_h * (c.deq * c.deq));
    c.m_gu = 0.f;
    c.m_h = 0.f;
    c.deq = 1.0f / (c.s0 * q);
    c.c_exp = c.deq * -1.4426950408889634f;
    const float m1 = c.deq * c.s1, m2 = c.deq * c.deq * c.s2;
    c.inv1 = 1.0f / m1;
    c.inv2 = 1.0f / m2;
    c.bnd1 = kE4M3Max * c.inv1;
    c.bnd2 = kE4M3Max * c.inv2;
  }
};

template <int NK, int TB>
__global__ __launch_bounds__(TB == 4 ? 256 : 512, 1) void swiglu_pipe_kernel(
    const uint8_t* __restrict__ x8, const uint8_t* __restrict__ w8, int64_t T, int64_t D, int64_t I,
    const float* __restrict__ scale, const float* __restrict__ wscale, float* __restrict__ amax,
    uint8_t* __restrict__ gu8, uint8_t* __restrict__ h8, uint8_t* __restrict__ h8t, int64_t ldt, int tiles_m,
    int tiles_n, const int* __restrict__ plan, int64_t w_estride) {
  using P = SwigluPipe<NK, TB>;
  using ML = typename P::ML;
  extern __shared__ __align__(16) uint8_t lds[];
  typename P::Ctx c;
  c.lds = lds;
  c.wave = threadIdx.x >> 6;
  // scales folded as in swiglu_fwd_kernel (all powers of two); with a plan
  // each tile's expert has its own weight scale wscale[e]
  c.s0 = scale[0];
  c.s1 = scale[1];
  c.s2 = scale[2];
  c.m_gu = 0.f;
  c.m_h = 0.f;
  c.mx_gu = 0.f;
  c.mx_h = 0.f;
  c.deq = 1.f;
  P::next_scales(c, wscale[0]);
  if (plan) tiles_m = MoePlan{plan}.ntiles();
  c.T = T;
  c.I = I;
  c.ldt = ldt;
  c.rgu = make_rsrc(gu8, 2 * I * ldt);
  c.so_g = c.so_u = 0u;
  c.h8 = h8;
  c.bad = false;
#pragma unroll
  for (int q = 0; q < 4; ++q) c.gw[q] = c.uw[q] = c.hw[q] = 0u;
  c.prev = false;
  c.pm0 = 0;
  c.pn0 = 0;
  c.hbuf = lds + kPipeRing;
  // the first tile's K loop runs the epilogue units with no previous tile:
  // on zeros they add nothing to the amax slots (and store nothing)
#pragma unroll
  for (int tb = 0; tb < TB; ++tb)
#pragma unroll
    for (int v = 0; v < 16; ++v) c.E[tb][v] = 0u;
  const int lane = threadIdx.x & 63, wm = c.wave % P::kWM, wn = c.wave / P::kWM;
  const int fr = lane & 31, g = lane >> 5;
  const uint32_t chunk = (uint32_t)(((lane & 3) ^ ((lane >> 4) & 3)) << 4);
  const int sw = (fr >> 2) & 3;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    c.aoff[h] = (uint32_t)((32 * TB * wm + fr) * kStage + (((2 * g + h) ^ sw) << 4));
    c.boff[h] = (uint32_t)(ML::kLdsB + (BLayout<true, 2>::kWaveStride * wn + fr) * kStage + (((2 * g + h) ^ sw) << 4));
  }
  const int64_t rpad = slab_rows(I);
  const int ntiles = tiles_m * tiles_n;
  const int a_ss = (int)(ldt * kStage), b_ss = (int)(2 * I * kStage);
#pragma unroll
  for (int j = 0; j < ML::kDmaA; ++j)
    c.voff_a[j] = (uint32_t)(((kTile / P::kWaves) * c.wave + 16 * j + (lane >> 2)) * kStage) + chunk;
  // K-slab operands: x8 [D/64][ldt][64], w8 [D/64][2I][64] (with a plan:
  // tile row tm's expert e at w8 + e * w_estride, its scale wscale[e]); tile
  // origin (m0, n0) -> A and B descriptors, B lane offsets, weight scale
  auto tile_operands = [&](int tile, int64_t& m0, int64_t& n0, __amdgpu_buffer_rsrc_t& ra,
                           __amdgpu_buffer_rsrc_t& rb, uint32_t (&voff_b)[2], float& q) {
    int tm, tn;
    tile_coords(tile, ntiles, tiles_m, tiles_n, tm, tn);
    m0 = (int64_t)tm * kTile;
    n0 = (int64_t)tn * 64;
    ra = make_rsrc(x8 + m0 * kStage, D * ldt - m0 * kStage);
    const int e = plan ? MoePlan{plan}.expert(tm) : 0;
    rb = make_rsrc(w8 + e * w_estride, D * 2 * I);
    q = wscale[e];
#pragma unroll
    for (int j = 0; j < ML::kDmaB; ++j) {
      const int r = (128 / P::kWaves) * c.wave + 16 * j + (lane >> 2);
      voff_b[j] = (uint32_t)(((r >> 6) * (int)I + (int)n0 + paired_col64(r)) * kStage) + chunk;
    }
  };
  int it = 0;
  int64_t m0 = 0, n0 = 0;
  float q = 1.f, nq = 1.f;  // weight scale of the current tile and of the next
  if (blockIdx.x < ntiles) {
    // prologue, once per work-group: the first tile's stages 0..2 in flight,
    // stage 0 landed, its fragments read.  Later tiles' first stages are
    // loaded by the last stages of the tile before.
    tile_operands(blockIdx.x, m0, n0, c.ra, c.rb, c.voff_b, q);
#pragma unroll
    for (int s = 0; s < 3; ++s) ML::load_stage(lds, s, c.ra, c.rb, c.voff_a, c.voff_b, s * a_ss, s * b_ss, c.wave);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * ML::kDma) : "memory");
    ML::read_frags(lds, 0, c.aoff, c.boff, c.f[0]);
  }
  for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x, ++it) {
    int64_t nm0 = m0, nn0 = n0;
    c.has_next = tile + (int)gridDim.x < ntiles;
    if (c.has_next) {
      tile_operands(tile + (int)gridDim.x, nm0, nn0, c.nra, c.nrb, c.nvoff_b, nq);
    } else {
      c.nra = c.ra;
      c.nrb = c.rb;
      c.nvoff_b[0] = c.voff_b[0];
      c.nvoff_b[1] = c.voff_b[1];
    }
#pragma unroll
    for (int i = 0; i < TB; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) c.acc[i][j] = floatx16{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f,
                                                          0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    P::template stages<0>(c, a_ss, b_ss);
    // every wave's h-tile writes are done (the next tile's first stages stay
    // in flight)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // the previous tile's h tile is complete: its K-slab copies (h8: 256
    // token rows of 64 bytes, one contiguous block; the optional h8t
    // transposed)
    if (c.prev) {
      pipe_h8_rows<64 * P::kWaves>(c.hbuf, h8 + (c.pn0 >> 6) * ldt * 64 + c.pm0 * 64);
      if (h8t) lds_tile_store_slab_tr<4, P::kWaves>(c.hbuf, kPipeHStride, h8t, rpad, c.pm0, c.pn0);
    }
    // this tile's g, u (bf16, unscaled) become the next epilogue's input
#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
#pragma unroll
      for (int v = 0; v < 16; ++v) c.E[tb][v] = pack2_bf16(c.acc[tb][0][v], c.acc[tb][1][v]);
    c.prev = true;
    c.pm0 = m0;
    c.pn0 = n0;
    c.so_g = (uint32_t)((n0 >> 6) * ldt * 64 + m0 * 64);
    c.so_u = (uint32_t)(((I + n0) >> 6) * ldt * 64 + m0 * 64);
    c.hbuf = lds + kPipeRing + (it & 1) * kPipeHBytes;
    // the previous epilogue is complete: its amax joins, and this tile's
    // weight scale sets the next epilogue's constants
    P::next_scales(c, q);
    m0 = nm0;
    n0 = nn0;
    q = nq;
    c.ra = c.nra;
    c.rb = c.nrb;
    c.voff_b[0] = c.nvoff_b[0];
    c.voff_b[1] = c.nvoff_b[1];
  }
  // the last tile's repeated loads of its last stage are still in flight
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (c.prev) {
    P::template tail_units<0>(c);
    __syncthreads();
    pipe_h8_rows<64 * P::kWaves>(c.hbuf, h8 + (c.pn0 >> 6) * ldt * 64 + c.pm0 * 64);
    if (h8t) lds_tile_store_slab_tr<4, P::kWaves>(c.hbuf, kPipeHStride, h8t, rpad, c.pm0, c.pn0);
  }
  P::next_scales(c, 1.f);  // folds the last epilogue's maxima
  float* red = reinterpret_cast<float*>(lds + kPipeRing + 2 * kPipeHBytes);
  float mg = wave_max(c.mx_gu), mh = wave_max(c.mx_h);
  if (lane == 0) {
    red[c.wave] = mg;
    red[P::kWaves + c.wave] = mh;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    float a1 = red[0], a2 = red[P::kWaves];
#pragma unroll
    for (int w = 1; w < P::kWaves; ++w) {
      a1 = fmaxf(a1, red[w]);
      a2 = fmaxf(a2, red[P::kWaves + w]);
    }
    atomic_max_nonneg(amax + 1, a1);
    atomic_max_nonneg(amax + 2, a2);
  }
}

// bf16 epilogues stage the tile in two passes of 128 rows (256 bf16 columns,
// row stride kBf16Stride: consecutive rows shift by 4 banks) and then write
// whole rows.  Pass P holds tile rows 64P..64P+63 and 128+64P..128+64P+63.
constexpr int kBf16Stride = 528;

// Wave (wm, wn), wn = 0..3, owns A rows 128 wm.. and output columns 64 wn.. as 4
// x 2 blocks; lane half g of block nb holds columns 64 wn + 32 g + 16 nb + v.
template <int P>
SFP8_DEV void stage_bf16_half8(uint8_t* lds, const floatx16 (&acc)[4][2], float s) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave & 1, wn = wave >> 1;
  const int fr = lane & 31, g = lane >> 5, cb = 64 * wn + 32 * g;
#pragma unroll
  for (int tt = 0; tt < 2; ++tt) {
    const int lr = 64 * wm + 32 * tt + fr;
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      uint32_t w0[4], w1[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        w0[i] = pack2_bf16(acc[2 * P + tt][nb][2 * i] * s, acc[2 * P + tt][nb][2 * i + 1] * s);
        w1[i] = pack2_bf16(acc[2 * P + tt][nb][8 + 2 * i] * s, acc[2 * P + tt][nb][8 + 2 * i + 1] * s);
      }
      uint8_t* q = lds + lr * kBf16Stride + (cb + 16 * nb) * 2;
      store16(q, w0);
      store16(q + 16, w1);
    }
  }
}

// A tile of at most 192 rows staged at once: the bf16 tile of kM rows and kN
// columns (row stride kOutStride: consecutive rows shift by 4 banks), written
// as whole tile rows.
template <class TS>
SFP8_DEV void stage_bf16_tile(uint8_t* lds, const floatx16 (&acc)[TS::kTB][2], float s) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave & 1, wn = wave >> 1;
  const int fr = lane & 31, g = lane >> 5, cb = 64 * wn + 32 * g;
#pragma unroll
  for (int tb = 0; tb < TS::kTB; ++tb) {
    const int lr = 32 * TS::kTB * wm + 32 * tb + fr;
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      uint32_t w0[4], w1[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        w0[i] = pack2_bf16(acc[tb][nb][2 * i] * s, acc[tb][nb][2 * i + 1] * s);
        w1[i] = pack2_bf16(acc[tb][nb][8 + 2 * i] * s, acc[tb][nb][8 + 2 * i + 1] * s);
      }
      uint8_t* q = lds + lr * TS::kOutStride + (cb + 16 * nb) * 2;
      store16(q, w0);
      store16(q + 16, w1);
    }
  }
}

// Tile row held in staging row lr of pass p.
SFP8_DEV int half_tile_row(int lr, int p) { return 128 * (lr >> 6) + 64 * p + (lr & 63); }

// Byte offset of out[t, n] (bf16, leading dimension ld) from out + m0 * ld,
// or 2^31 -- past the range of any descriptor, so the store is dropped --
// for t >= T or n >= N.  A bit mask rather than a select keeps the stores
// free of branches (one store instruction per chunk, a fixed count per
// wave).  Tile rows t - m0 < 256, so the offset needs ld < 2^22.
SFP8_DEV uint32_t bf16_out_off(int64_t t, int64_t n, int64_t m0, int64_t T, int64_t N, int64_t ld) {
  const uint32_t in = 0u - (uint32_t)(t < T && n < N);
  return ((uint32_t)(((t - m0) * ld + n) * 2) & in) | (~in & 0x80000000u);
}

// Writes one staged pass to out[t, n] (bf16, leading dimension ld) for rows
// m0.. of the tile below T and columns below N.  NT = threads of the
// work-group.
template <int NT = 256>
SFP8_DEV void write_bf16_half(const uint8_t* lds, int p, int64_t m0, int64_t n0, int64_t T, int64_t N,
                              int64_t ld, uint16_t* __restrict__ out) {
  const __amdgpu_buffer_rsrc_t ro = make_rsrc(out + m0 * ld, (T - m0) * ld * 2);
#pragma unroll
  for (int k = 0; k < 4096 / NT; ++k) {
    const int idx = (int)threadIdx.x + NT * k;
    const int lr = idx >> 5, c = idx & 31;
    const int64_t t = m0 + half_tile_row(lr, p), n = n0 + 8 * c;
    const intx4 o = *reinterpret_cast<const intx4*>(lds + lr * kBf16Stride + c * 16);
    __builtin_amdgcn_raw_buffer_store_b128(o, ro, bf16_out_off(t, n, m0, T, N, ld), 0, 0);
  }
}

// Residual words of staged half p, in write_bf16_half's order (4096 / NT per
// thread); rows past T read as zero through the descriptor.
template <int NT>
SFP8_DEV void load_res_half(__amdgpu_buffer_rsrc_t rres, int p, int64_t n0, int64_t D, intx4 (&rv)[4096 / NT]) {
#pragma unroll
  for (int k = 0; k < 4096 / NT; ++k) {
    const int idx = (int)threadIdx.x + NT * k;
    const int lr = idx >> 5, c = idx & 31;
    const uint32_t off = (uint32_t)((half_tile_row(lr, p) * D + n0 + 8 * c) * 2);
    rv[k] = __builtin_amdgcn_raw_buffer_load_b128(rres, off, 0, kNT);
  }
}

// write_bf16_half after adding the bf16 residual, already in registers:
// out = bf16(res + staged).
template <int NT>
SFP8_DEV void write_bf16_half_res(const uint8_t* lds, int p, int64_t m0, int64_t n0, int64_t T, int64_t D,
                                  const intx4 (&rv)[4096 / NT], uint16_t* __restrict__ out) {
  const __amdgpu_buffer_rsrc_t ro = make_rsrc(out + m0 * D, (T - m0) * D * 2);
#pragma unroll
  for (int k = 0; k < 4096 / NT; ++k) {
    const int idx = (int)threadIdx.x + NT * k;
    const int lr = idx >> 5, c = idx & 31;
    const int64_t t = m0 + half_tile_row(lr, p), n = n0 + 8 * c;
    intx4 o = *reinterpret_cast<const intx4*>(lds + lr * kBf16Stride + c * 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t a = (uint32_t)rv[k][i], b = (uint32_t)o[i];
      o[i] = (int)pack2_bf16(__uint_as_float(b << 16) + __uint_as_float(a << 16),
                             __uint_as_float(b & 0xffff0000u) + __uint_as_float(a & 0xffff0000u));
    }
    __builtin_amdgcn_raw_buffer_store_b128(o, ro, bf16_out_off(t, n, m0, T, D, D), 0, 0);
  }
}

// The tile staged by stage_bf16_tile to out[t, n] (bf16, leading dimension
// ld), rows m0.. below T, columns below N; with RES the bf16 residual rv
// (requested by load_res_tile) is added first: out = bf16(res + staged).
template <class TS>
SFP8_DEV void load_res_tile(__amdgpu_buffer_rsrc_t rres, int64_t n0, int64_t D, intx4 (&rv)[TS::kPieces]) {
#pragma unroll
  for (int k = 0; k < TS::kPieces; ++k) {
    const int idx = (int)threadIdx.x + TS::kThreads * k;
    const int lr = idx / (TS::kN / 8), c = idx % (TS::kN / 8);
    rv[k] = __builtin_amdgcn_raw_buffer_load_b128(rres, (uint32_t)((lr * D + n0 + 8 * c) * 2), 0, kNT);
  }
}
template <class TS, bool RES>
SFP8_DEV void write_bf16_tile(const uint8_t* lds, int64_t m0, int64_t n0, int64_t T, int64_t N, int64_t ld,
                              const intx4 (&rv)[TS::kPieces], uint16_t* __restrict__ out) {
  const __amdgpu_buffer_rsrc_t ro = make_rsrc(out + m0 * ld, (T - m0) * ld * 2);
#pragma unroll
  for (int k = 0; k < TS::kPieces; ++k) {
    const int idx = (int)threadIdx.x + TS::kThreads * k;
    const int lr = idx / (TS::kN / 8), c = idx % (TS::kN / 8);
    intx4 o = *reinterpret_cast<const intx4*>(lds + lr * TS::kOutStride + c * 16);
    if constexpr (RES) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t a = (uint32_t)rv[k][i], b = (uint32_t)o[i];
        o[i] = (int)pack2_bf16(__uint_as_float(b << 16) + __uint_as_float(a << 16),
                               __uint_as_float(b & 0xffff0000u) + __uint_as_float(a & 0xffff0000u));
      }
    }
    __builtin_amdgcn_raw_buffer_store_b128(o, ro, bf16_out_off(m0 + lr, n0 + 8 * c, m0, T, N, ld), 0, 0);
  }
}

// A tile's accumulators times s, as bf16, to out[t, n] (leading dimension N)
// for rows u0.. below uend and columns n0.. below N.
template <class TS>
SFP8_DEV void store_bf16_tile(uint8_t* lds, const floatx16 (&acc)[TS::kTB][2], float s, int64_t u0, int64_t n0,
                              int64_t uend, int64_t N, uint16_t* __restrict__ out) {
  if constexpr (TS::kTB < 4) {
    const intx4 none[TS::kPieces] = {};
    stage_bf16_tile<TS>(lds, acc, s);
    __syncthreads();
    write_bf16_tile<TS, false>(lds, u0, n0, uend, N, N, none, out);
  } else {
    stage_bf16_half8<0>(lds, acc, s);
    __syncthreads();
    write_bf16_half<512>(lds, 0, u0, n0, uend, N, N, out);
    __syncthreads();
    stage_bf16_half8<1>(lds, acc, s);
    __syncthreads();
    write_bf16_half<512>(lds, 1, u0, n0, uend, N, N, out);
  }
}

// ---------------------------------------------------------------------------
// (a7) down forward + residual (spark-gpt train.py:1019-1046):
//   y = bf16(res + bf16(acc / (s2 * q_d)))
// With a MoE plan: no residual; tile row tm of padded expert order writes
// its rows(tm) valid rows to y rows urow(tm).. (expert order, unpadded);
// W_down8 of expert e at wd8 + e * w_estride, its scale wscale[e] (the dense
// call passes wscale + 1: [q_gu, q_d]).
template <class TS>
SFP8_DEV void down_fwd_tile(
    uint8_t* lds, int tm, int tn, const uint8_t* __restrict__ h8, const uint8_t* __restrict__ wd8,
    const uint16_t* __restrict__ res, int64_t T, int64_t D, int64_t I, const float* __restrict__ scale,
    const float* __restrict__ wscale, uint16_t* __restrict__ y, int64_t ldt, const int* __restrict__ plan,
    int64_t w_estride) {
  int64_t u0 = 0, urows = 0;
  if (plan) {
    const MoePlan P{plan};
    const int pt = TS::plan_tile(tm);
    if (pt >= P.ntiles()) return;  // work-group uniform
    const int e = P.expert(pt);
    wd8 += e * w_estride;
    wscale += e;
    u0 = P.urow(pt) + TS::plan_skip(tm);
    urows = P.rows(pt) - TS::plan_skip(tm);
    if (urows <= 0) return;  // nothing but padding rows, which have no output
  }
  const int64_t m0 = (int64_t)tm * TS::kM, n0 = (int64_t)tn * TS::kN;
  if (!plan && m0 >= T) return;  // the second half of the last tile, past the last row
  floatx16 acc[TS::kTB][2];
  // K-slab operands: h8 [I/64][ldt][64], wd8 [I/64][slab_rows(D)][64]
  const int64_t dp = slab_rows(D);
  TS::template Loop<false, kFmtE4M3, kFmtE4M3>::run(
      lds, h8 + m0 * kStage, I * ldt - m0 * kStage, [=](int r) { return r * kStage; }, (int)(ldt * kStage),
      wd8 + n0 * kStage, I * dp - n0 * kStage, [=](int r) { return plain_col_nb<2>(r) * kStage; },
      (int)(dp * kStage), (int)(I / kStage), acc);
  const float deq = 1.0f / (scale[2] * wscale[0]);
  if constexpr (TS::kTB < 4) {
    intx4 rv[TS::kPieces];
    if (!plan) load_res_tile<TS>(make_rsrc(res + m0 * D, (T - m0) * D * 2), n0, D, rv);
    stage_bf16_tile<TS>(lds, acc, deq);
    __syncthreads();
    if (plan) write_bf16_tile<TS, false>(lds, u0, n0, u0 + urows, D, D, rv, y);
    else write_bf16_tile<TS, true>(lds, m0, n0, T, D, D, rv, y);
  } else {
  if (plan) {
    // expert rows, no residual: out rounded to bf16 (train.py:1377-1378 stores acc / (s2 q_d) as bf16)
    stage_bf16_half8<0>(lds, acc, deq);
    __syncthreads();
    write_bf16_half<512>(lds, 0, u0, n0, u0 + urows, D, D, y);
    __syncthreads();
    stage_bf16_half8<1>(lds, acc, deq);
    __syncthreads();
    write_bf16_half<512>(lds, 1, u0, n0, u0 + urows, D, D, y);
    return;
  }
  const __amdgpu_buffer_rsrc_t rres = make_rsrc(res + m0 * D, (T - m0) * D * 2);
  // Every residual word the two staged halves add is requested at once (one
  // memory latency), in the order the staged rows are written, so both the
  // residual reads and the y writes are whole rows; rows past T read as zero
  // through the descriptor's range check and are not stored.
  intx4 rv0[8], rv1[8];
  load_res_half<512>(rres, 0, n0, D, rv0);
  load_res_half<512>(rres, 1, n0, D, rv1);
  // out rounded to bf16 before the residual add (train.py:1043)
  stage_bf16_half8<0>(lds, acc, deq);
  __syncthreads();
  write_bf16_half_res<512>(lds, 0, m0, n0, T, D, rv0, y);
  __syncthreads();
  stage_bf16_half8<1>(lds, acc, deq);
  __syncthreads();
  write_bf16_half_res<512>(lds, 1, m0, n0, T, D, rv1, y);
  }
}
template <class TS>
__global__ __launch_bounds__(TS::kThreads, TS::kMinWaves) void down_fwd_kernel(
    const uint8_t* __restrict__ h8, const uint8_t* __restrict__ wd8, const uint16_t* __restrict__ res,
    int64_t T, int64_t D, int64_t I, const float* __restrict__ scale, const float* __restrict__ wscale,
    uint16_t* __restrict__ y, int64_t ldt, int tiles_m, int tiles_n, const int* __restrict__ plan,
    int64_t w_estride) {
  extern __shared__ __align__(16) uint8_t lds[];
  int tm, tn;
  if constexpr (TS::kTB == 4) {
    bool half;
    if (!tail_tile(plan ? MoePlan{plan}.ntiles() : tiles_m, tiles_n, tm, tn, half)) return;
    if (half) {
      down_fwd_tile<Tile<2, 4>>(lds, tm, tn, h8, wd8, res, T, D, I, scale, wscale, y, ldt, plan, w_estride);
      return;
    }
  } else {
    tile_coords(blockIdx.x, gridDim.x, tiles_m, tiles_n, tm, tn);
  }
  down_fwd_tile<TS>(lds, tm, tn, h8, wd8, res, T, D, I, scale, wscale, y, ldt, plan, w_estride);
}

// ---------------------------------------------------------------------------
// (a9) bf16 down dgrad + SwiGLU backward (spark-gpt train.py:1049-1094):
//   dh = bf16(dy @ Wd); g, u = gu8 / s1; sig = sigmoid(g)
//   d_gate = dh*u*(sig*(1+g*(1-sig))), d_up = dh*g*sig
//   dgu8 = e5m2(d * s3) as the K-slab of [T, 2I] (and optionally of [2I,
//   ldt]: the token-contiguous dgu8t), amax slot 3.
// B = Wd^T (bf16, [I, D]).  Tile 256 tokens x 256 intermediate columns,
// one work-group of 8 waves (two per SIMD, each 128 x 64 of the tile): the
// second wave on a SIMD runs while the first waits, in the K loop and above
// all in the epilogue, whose loads, LDS round trips and barriers a single
// wave per SIMD left exposed.
constexpr int kEpiStride2 = 272;
// LDS: the SwiGLU backward's table at offset 0 (so that an entry's address
// is its code times 8), then the main loop's ring, later the epilogue's
// staging tiles and 8 reduction slots
constexpr int kDgradLutBytes = 256 * 8;

// dg, du of the 4 columns of group w of a 16-column chunk: dh from the
// staged bf16 words h0 (columns 0-7) and h1 (8-15), the gate and up codes
// from gw and uw, the two factors per gate code from the table at LDS
// address 0 (entry b at 8 b: the kernel has no static LDS, so its dynamic
// LDS begins at 0, and one shift of the selected byte is the address); the
// reference's order (train.py:1083-1087).
typedef __attribute__((address_space(3))) const floatx2* lds_floatx2_ptr;
SFP8_DEV void dgrad_swiglu4(const intx4& h0, const intx4& h1, uint32_t gw, uint32_t uw, int w, float (&dg)[4],
                            float (&du)[4]) {
  const uint32_t hw0 = (uint32_t)(w < 2 ? h0[2 * w] : h1[2 * w - 4]);
  const uint32_t hw1 = (uint32_t)(w < 2 ? h0[2 * w + 1] : h1[2 * w - 3]);
  const float dhv[4] = {__uint_as_float(hw0 << 16), __uint_as_float(hw0 & 0xffff0000u), __uint_as_float(hw1 << 16),
                        __uint_as_float(hw1 & 0xffff0000u)};
  const floatx2 g01 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(gw, 1.0f, false);
  const floatx2 g23 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(gw, 1.0f, true);
  const floatx2 u01 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(uw, 1.0f, false);
  const floatx2 u23 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(uw, 1.0f, true);
  const float g8v[4] = {g01.x, g01.y, g23.x, g23.y}, u8v[4] = {u01.x, u01.y, u23.x, u23.y};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    // (sig, sig * (1 + g * (1 - sig)))
    const floatx2 f = *reinterpret_cast<lds_floatx2_ptr>((uintptr_t)(((gw >> (8 * e)) & 0xFFu) << 3));
    dg[e] = (dhv[e] * u8v[e]) * f.y;
    du[e] = (dhv[e] * g8v[e]) * f.x;
  }
}

// With a MoE plan: tile rows are padded expert order (gu8, dgu8, dgu8t over
// ldt padded rows); dy is the row-major upstream gradient of the expert-order
// rows (its rows urow(tm).. for tile row tm), W_down^T of expert e at
// wdt + e * w_estride (bytes); the tile count comes from the plan.
// TCOPY: dgu8t is written too (staged in LDS per pass).
// SMALL: 128 x 128 tiles by 4 waves of 64 x 64, two work-groups per CU, one
// epilogue pass (not with TCOPY).
template <bool TCOPY, bool SMALL>
__global__ __launch_bounds__(TileShape<SMALL>::kThreads, TileShape<SMALL>::kMinWaves) void down_dgrad_swiglu_kernel(
    const uint16_t* __restrict__ dy, const uint16_t* __restrict__ wdt, const uint8_t* __restrict__ gu8,
    int64_t T, int64_t D, int64_t I, const float* __restrict__ scale, float* __restrict__ amax,
    uint8_t* __restrict__ dgu8, uint8_t* __restrict__ dgu8t, int64_t ldt, int tiles_m, int tiles_n,
    const int* __restrict__ plan, int64_t w_estride) {
  static_assert(!(TCOPY && SMALL), "the copy is staged by the larger tile");
  constexpr int kWaves = TileShape<SMALL>::kThreads / 64;
  extern __shared__ __align__(16) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t ldb = D * 2;  // bytes
  const int64_t ip = slab_rows(I);
  // The gate operand of the SwiGLU backward is an e4m3 code here, so its two
  // factors take 256 values per launch: entry b of this table holds
  //   sig = sigmoid(g), sig * (1 + g * (1 - sig))   for g = e4m3(b) / s1,
  // rounded in the reference's order (train.py:1083-1087, no contraction).
  // Its LDS range is disjoint from the main loop's ring and the staging
  // tiles; the main loop's first barrier publishes it.
  floatx2* lut = reinterpret_cast<floatx2*>(lds);
  uint8_t* const base = lds + kDgradLutBytes;  // the ring and the staging tiles
  if (tid < 256) {
#pragma clang fp contract(off)
    const float gl = __builtin_amdgcn_cvt_f32_fp8(tid, 0) * (1.0f / scale[1]);
    const float sig = 1.0f / (1.0f + expf(-gl));
    lut[tid] = floatx2{sig, sig * (1.0f + gl * (1.0f - sig))};
  }
  // g = g8*s_gu, u = u8*s_gu with g8, u8 the stored e4m3 values; as the scales
  // are powers of two, d_gate = dg*s_gu and d_up = du*s_gu with
  //   dg = (dh*u8)*(sig*(1 + g*(1-sig))),  du = (dh*g8)*sig  (factors from lut),
  //   dgu8 = e5m2(d*q3) = e5m2(d'*(s_gu*q3)),  amax3 = s_gu*max(|dg|,|du|).
  const float m3s = (1.0f / scale[1]) * scale[3];
  const float inv3 = 1.0f / m3s, bnd3 = kE5M2Max * inv3;
  float* red = reinterpret_cast<float*>(base + (SMALL ? 128 * TileShape<SMALL>::kOutStride : 2 * kTile * kEpiStride2));  // after the staging tiles
  float m3 = 0.f;
  // Persistent: work-group pid runs tiles pid, pid + gridDim.x, ...  (Work-
  // groups started a quarter of a tile apart per XCD, so that the tiles'
  // 256 KiB store bursts would not coincide, measured 2 % slower.)
  if (plan) tiles_m = MoePlan{plan}.ntiles() * (kTile / TileShape<SMALL>::kM);
  const int ntiles = tiles_m * tiles_n;
  // A = dy row-major (rows past the tile's last read as zero through the
  // range check); B = Wd^T as a bf16 K-slab [2D/64][slab_rows(I)][64] (bytes)
  const auto arow = [=](int r) { return r * (int)ldb; };
  const auto brow = [=](int r) { return plain_col_nb<2>(r) * kStage; };
  const int nk = (int)(ldb / kStage);
  // the operands of tile `tile`: dy rows m0.. (dense) or the expert rows
  // urow(tm).. (MoE), and W_down^T (of the tile's expert) from column n0
  struct Ops {
    const uint8_t* a;
    int64_t a_bytes;
    const uint8_t* b;
    int64_t b_bytes;
  };
  const auto ops_of = [=](auto shape, int tm, int tn) {
    using TS = decltype(shape);
    const int64_t m0 = (int64_t)tm * TS::kM, n0 = (int64_t)tn * TS::kN;
    int64_t a_row = m0, a_rows = T - m0;
    const uint8_t* wb = reinterpret_cast<const uint8_t*>(wdt);
    if (plan) {
      const MoePlan P{plan};
      const int pt = TS::plan_tile(tm);
      a_row = P.urow(pt) + TS::plan_skip(tm);
      a_rows = P.rows(pt) - TS::plan_skip(tm);  // 0 or less: every row reads as zero
      wb += P.expert(pt) * w_estride;
    }
    return Ops{reinterpret_cast<const uint8_t*>(dy) + a_row * ldb, a_rows * ldb, wb + n0 * kStage,
               ldb * ip - n0 * kStage};
  };
  const auto run_tile = [&](auto shape, int tm, int tn) {
  using TS = decltype(shape);
  using Loop = typename TS::template Loop<true, 0, 0>;
  const int64_t m0 = (int64_t)tm * TS::kM, n0 = (int64_t)tn * TS::kN;
  floatx16 acc[TS::kTB][2];
  {
    const Ops o = ops_of(shape, tm, tn);
    Loop::run(base, o.a, o.a_bytes, arow, kStage, o.b, o.b_bytes, brow, (int)(ip * kStage), nk, acc);
  }
  // Row-order epilogue, in two passes (128-row tiles: one) of 128 tile rows (the rows
  // of stage_bf16_half8<P>): dh staged in LDS as bf16, then each thread takes
  // 16-column chunks of one row, reading gu8 and writing dgu8 as whole K-slab
  // rows; with dgu8t the codes also go to LDS for the token-contiguous copy.
  const __amdgpu_buffer_rsrc_t rgu = make_rsrc(gu8 + m0 * 64, 2 * I * ldt - m0 * 64);
  uint8_t* DH = base;
  // chunk k of this thread in a pass: 16 columns from chunk_col(k) of staging
  // row chunk_row(k), tile row tile_row(k, P)
  constexpr int kSlabs = TS::kN / 64, kDh = TS::kOutStride;
  constexpr bool kOne = TS::kTB == 2;  // one pass
  static_assert(kDh == (SMALL ? kDh : kBf16Stride), "the staging rows of stage_bf16_half8");
  const auto chunk_row = [=](int k) { return 16 * ((kWaves * k + wave) / kSlabs) + (lane >> 2); };
  const auto chunk_col = [=](int k) { return 64 * ((kWaves * k + wave) % kSlabs) + 16 * (lane & 3); };
  const auto tile_row = [=](int k, int P) { return kOne ? chunk_row(k) : half_tile_row(chunk_row(k), P); };
  // the staging tiles of the token-contiguous copy (MoE only); their offset
  // goes through an empty asm so that the compiler does not hoist per-lane
  // addresses into them out of the tile loop (a register it had to spill)
  int g2off = kDgradLutBytes + 128 * kBf16Stride;
  asm volatile("" : "+s"(g2off));
  uint8_t* G2 = lds + g2off;
  uint8_t* U2 = G2 + 128 * kEpiStride2;
  // Byte offset from gu8 / dgu8 + m0 * 64 of tile row `row`, tile column c
  // of the gate half (the up half lies I * ldt further, and I * ldt < 2^31):
  // a column past I gets offset 2^31, beyond the descriptors' range in both
  // halves, so its loads return zero and its stores are dropped -- every
  // chunk issues its instructions, a fixed count per wave, with no branch
  // around them (a bit mask rather than a select, which the compiler turned
  // into one).
  const auto gu_off = [=](int c, int row) {
    const int64_t j = n0 + c;
    const uint32_t in = 0u - (uint32_t)(j < I);  // all ones for a column inside I
    return ((uint32_t)((j >> 6) * ldt * 64 + row * 64 + (j & 63)) & in) | (~in & 0x80000000u);
  };
  const __amdgpu_buffer_rsrc_t rdg = make_rsrc(dgu8 + m0 * 64, 2 * I * ldt - m0 * 64);
  // gu8 words of this thread's 4 chunks of pass P, requested at once
  intx4 wg[4], wu[4];
  const auto gu_loads = [&](int P) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t o = gu_off(chunk_col(k), tile_row(k, P));
      wg[k] = __builtin_amdgcn_raw_buffer_load_b128(rgu, o, 0, kNT);
      wu[k] = __builtin_amdgcn_raw_buffer_load_b128(rgu, o + (uint32_t)(I * ldt), 0, kNT);
    }
  };
  // the codes of chunk k of the loaded pass (dh from the staged tile, gate and up
  // codes from wg[k], wu[k]); the running amax in m3
  const auto swiglu_chunk = [&](int k, uint32_t (&pg)[4], uint32_t (&pu)[4]) {
    const int lr = chunk_row(k), c = chunk_col(k);
    const intx4 h0 = *reinterpret_cast<const intx4*>(DH + lr * kDh + 2 * c);
    const intx4 h1 = *reinterpret_cast<const intx4*>(DH + lr * kDh + 2 * c + 16);
    // The 16 values' unclamped codes and their NaN-propagating maximum
    // magnitude (the first maximum3 of each group of four takes the
    // running maximum): when it is inside the e5m2 range (after scaling)
    // no clamp can act and no NaN needs its code, so the codes are
    // exact; otherwise (wave-uniform, NaN or out-of-range data only) the
    // chunk is computed again with the clamps and NaN codes, and the amax
    // over its non-NaN values.
    float mc = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      float dg[4], du[4];
      dgrad_swiglu4(h0, h1, (uint32_t)wg[k][w], (uint32_t)wu[k][w], w, dg, du);
      mc = max3_nan(mc, fabsf(dg[0]), fabsf(du[0]));
      mc = max3_nan(mc, fabsf(dg[1]), fabsf(du[1]));
      mc = max3_nan(mc, fabsf(dg[2]), fabsf(du[2]));
      mc = max3_nan(mc, fabsf(dg[3]), fabsf(du[3]));
      // the unclamped packs overwrite both halves of their third argument:
      // the dead dh words, rather than a copy of a live register
      pg[w] = pack4_e5m2_scaled_noclamp(dg[0], dg[1], dg[2], dg[3], inv3,
                                        (uint32_t)(w < 2 ? h0[2 * w] : h1[2 * w - 4]));
      pu[w] = pack4_e5m2_scaled_noclamp(du[0], du[1], du[2], du[3], inv3,
                                        (uint32_t)(w < 2 ? h0[2 * w + 1] : h1[2 * w - 3]));
    }
    if (__builtin_amdgcn_ballot_w64(!(mc <= bnd3))) {
      asm volatile("" ::: "memory");
      mc = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        float dg[4], du[4];
        dgrad_swiglu4(h0, h1, (uint32_t)wg[k][w], (uint32_t)wu[k][w], w, dg, du);
        pg[w] = fix_nan4(pack4_e5m2_scaled(dg[0], dg[1], dg[2], dg[3], inv3, bnd3), dg[0], dg[1], dg[2], dg[3]);
        pu[w] = fix_nan4(pack4_e5m2_scaled(du[0], du[1], du[2], du[3], inv3, bnd3), du[0], du[1], du[2], du[3]);
#pragma unroll
        for (int e = 0; e < 4; ++e) mc = fmaxf(mc, fmaxf(fabsf(dg[e]), fabsf(du[e])));
      }
    }
    m3 = fmaxf(m3, mc);
    if constexpr (TCOPY) {  // staged for the token-contiguous copy
      store16(G2 + lr * kEpiStride2 + c, pg);
      store16(U2 + lr * kEpiStride2 + c, pu);
    }
  };
  // dgu8 is a K-slab [2I/64][ldt][64]; four lanes write one 64-byte row
  const auto store_chunk = [&](int P, int k, const uint32_t (&pg)[4], const uint32_t (&pu)[4]) {
    const uint32_t o = gu_off(chunk_col(k), tile_row(k, P));
    __builtin_amdgcn_raw_buffer_store_b128(intx4{(int)pg[0], (int)pg[1], (int)pg[2], (int)pg[3]}, rdg, o, 0, 0);
    __builtin_amdgcn_raw_buffer_store_b128(intx4{(int)pu[0], (int)pu[1], (int)pu[2], (int)pu[3]}, rdg,
                                           o + (uint32_t)(I * ldt), 0, 0);
  };
  if constexpr (TCOPY) {
#pragma unroll
    for (int P = 0; P < 2; ++P) {
      gu_loads(P);
      if (P == 1) __syncthreads();  // pass 0's dgu8t copy has read the LDS
      // dh rounded to bf16 (train.py:1082)
      if (P == 0) stage_bf16_half8<0>(DH, acc, 1.0f);
      else stage_bf16_half8<1>(DH, acc, 1.0f);
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        uint32_t pg[4], pu[4];
        swiglu_chunk(k, pg, pu);
        store_chunk(P, k, pg, pu);
      }
      __syncthreads();
      // the token-contiguous dgu8t: local rows 0-63 are tile rows 64P.., rows
      // 64-127 tile rows 128 + 64P.. (rows past T hold zero codes)
      const int64_t rp2 = slab_rows(2 * I);
      const int cols = (int)((I - n0) < kTile ? (I - n0) : kTile);  // 128 or 256
      lds_rows_store_slab_tr<64, 8>(G2, cols, kEpiStride2, dgu8t, rp2, m0 + 64 * P, n0);
      lds_rows_store_slab_tr<64, 8>(G2 + 64 * kEpiStride2, cols, kEpiStride2, dgu8t, rp2, m0 + 128 + 64 * P, n0);
      lds_rows_store_slab_tr<64, 8>(U2, cols, kEpiStride2, dgu8t, rp2, m0 + 64 * P, I + n0);
      lds_rows_store_slab_tr<64, 8>(U2 + 64 * kEpiStride2, cols, kEpiStride2, dgu8t, rp2, m0 + 128 + 64 * P,
                                    I + n0);
    }
    __syncthreads();  // the next tile's DMA overwrites the staging tiles
  } else if constexpr (kOne) {
    uint32_t pg[4], pu[4];
    gu_loads(0);
    stage_bf16_tile<TS>(DH, acc, 1.0f);  // dh rounded to bf16 (train.py:1082)
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      swiglu_chunk(k, pg, pu);
      store_chunk(0, k, pg, pu);
    }
    __syncthreads();  // the next tile's DMA overwrites the staging tile
  } else {
    // Each chunk is stored as soon as its codes are made, so that the stores
    // drain while the rest is computed.  (Deferring the first pass's stores
    // behind the second pass's gu8 requests, so that waiting for those
    // leaves the stores in flight, measured 2 % slower.)  The second pass's
    // gu8 words are requested before its staging.
    uint32_t pg[4][4], pu[4][4];
    gu_loads(0);
    stage_bf16_half8<0>(DH, acc, 1.0f);  // dh rounded to bf16 (train.py:1082)
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      swiglu_chunk(k, pg[k], pu[k]);
      store_chunk(0, k, pg[k], pu[k]);
    }
    gu_loads(1);
    __syncthreads();  // every wave has read pass 0's staged rows
    stage_bf16_half8<1>(DH, acc, 1.0f);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      swiglu_chunk(k, pg[k], pu[k]);
      store_chunk(1, k, pg[k], pu[k]);
    }
    __syncthreads();  // the next tile's DMA overwrites the staging tile
  }
  };
  // the last round in halves (tail_full), except with the copy and the small
  // tiles
  const int nwg = gridDim.x, full = TCOPY || SMALL ? ntiles : tail_full(ntiles, nwg);
  int tm, tn;
  for (int tile = blockIdx.x; tile < full; tile += nwg) {
    tile_coords(tile, full, tiles_m, tiles_n, tm, tn);
    run_tile(TileShape<SMALL>{}, tm, tn);
  }
  if constexpr (!TCOPY && !SMALL) {
    if (tail_half(blockIdx.x, full, tiles_m, tiles_n, tm, tn)) run_tile(Tile<2, 4>{}, tm, tn);
  }
  m3 *= 1.0f / scale[1];  // s_gu, read again rather than held across the tile loop
  block_amax_atomic<kWaves>(m3, red, amax + 3);
}

// ---------------------------------------------------------------------------
// (a10) gate/up dgrad (spark-gpt train.py:1239-1241):
//   dxn = bf16(acc * (1/s3) * (1/q_gu)), A = d_gu8 (e5m2, [T, 2I]), B = W8^T (e4m3, [D, 2I]).
// One work-group per 256 x 256 tile; the bf16 tile is staged in LDS in two
// passes of 128 rows and written as whole rows.
// With a MoE plan: tile row tm of padded expert order writes its rows(tm)
// valid rows to dxn rows urow(tm).. (expert order, unpadded); W8^T of
// expert e at w8t + e * w_estride, its scale wscale[e].
template <class TS>
SFP8_DEV void gateup_dgrad_tile(
    uint8_t* lds, int tm, int tn, const uint8_t* __restrict__ dgu8, const uint8_t* __restrict__ w8t, int64_t T,
    int64_t D, int64_t I, const float* __restrict__ scale, const float* __restrict__ wscale,
    uint16_t* __restrict__ dxn, int64_t ldt, const int* __restrict__ plan, int64_t w_estride) {
  const int64_t K = 2 * I;
  const int64_t dp = slab_rows(D);
  int64_t u0 = (int64_t)tm * TS::kM, uend = T;  // output rows of this tile
  if (plan) {
    const MoePlan P{plan};
    const int pt = TS::plan_tile(tm);
    if (pt >= P.ntiles()) return;  // work-group uniform
    const int e = P.expert(pt);
    w8t += e * w_estride;
    wscale += e;
    u0 = P.urow(pt) + TS::plan_skip(tm);
    uend = P.urow(pt) + P.rows(pt);
    if (u0 >= uend) return;  // nothing but padding rows, which have no output
  }
  const int64_t m0 = (int64_t)tm * TS::kM, n0 = (int64_t)tn * TS::kN;
  if (!plan && m0 >= T) return;  // the second half of the last tile, past the last row
  floatx16 acc[TS::kTB][2];
  // K-slab operands: dgu8 [2I/64][ldt][64], w8t [2I/64][slab_rows(D)][64]
  TS::template Loop<false, kFmtE5M2, kFmtE4M3>::run(
      lds, dgu8 + m0 * kStage, K * ldt - m0 * kStage, [=](int r) { return r * kStage; }, (int)(ldt * kStage),
      w8t + n0 * kStage, K * dp - n0 * kStage, [=](int r) { return plain_col_nb<2>(r) * kStage; },
      (int)(dp * kStage), (int)(K / kStage), acc);
  // the scales are read after the K loop, so that nothing is held across it
  const float sab = (1.0f / scale[3]) * (1.0f / wscale[0]);  // both powers of two
  store_bf16_tile<TS>(lds, acc, sab, u0, n0, uend, D, dxn);
}
template <class TS>
__global__ __launch_bounds__(TS::kThreads, TS::kMinWaves) void gateup_dgrad_kernel(
    const uint8_t* __restrict__ dgu8, const uint8_t* __restrict__ w8t, int64_t T, int64_t D, int64_t I,
    const float* __restrict__ scale, const float* __restrict__ wscale, uint16_t* __restrict__ dxn,
    int64_t ldt, int tiles_m, int tiles_n, const int* __restrict__ plan, int64_t w_estride) {
  extern __shared__ __align__(16) uint8_t lds[];
  int tm, tn;
  // backwards: the dgrad wrote d_gu8 in forward order (0.304 -> 0.302 ms)
  if constexpr (TS::kTB == 4) {
    bool half;
    if (!tail_tile(plan ? MoePlan{plan}.ntiles() : tiles_m, tiles_n, tm, tn, half, true)) return;
    if (half) {
      gateup_dgrad_tile<Tile<2, 4>>(lds, tm, tn, dgu8, w8t, T, D, I, scale, wscale, dxn, ldt, plan, w_estride);
      return;
    }
  } else {
    tile_coords(blockIdx.x, gridDim.x, tiles_m, tiles_n, tm, tn, true);
  }
  gateup_dgrad_tile<TS>(lds, tm, tn, dgu8, w8t, T, D, I, scale, wscale, dxn, ldt, plan, w_estride);
}

// ---------------------------------------------------------------------------
// (a12, a13) weight gradients, reduced over tokens:
//   out[m, n] = sum_t A[m, t] * B[n, t] / (sa * sb)
// A, B are K-slab token-contiguous fp8 copies (common.h) over ldt tokens
// (zeros past T): a tile's K stage is one contiguous 16 KiB block of each.
// The grid is tiles * splits work-groups (split_tile_coords); split sp takes
// K bytes [sp * kchunk, min((sp + 1) * kchunk, ldt)) (the last split may be
// shorter; every split is a whole number of 128-byte stage pairs); with splits > 1
// each split writes its raw fp32 accumulators to ws in accumulator order
// (acc_order_rc: each wave store instruction is one contiguous 1 KiB
// run) and splitk_reduce_kernel sums them in split order (deterministic) and
// scatters them to [M, N].
// With `partials` the raw partials go to `out` as the workspace, also for one
// split (the reduction that applies the optimizer's momentum stage); without,
// there is one split and the gradient itself goes to `out` (store_grad_tile).
// BF16: bf16 operands (2 bytes per token: `ldt` and `kchunk` count K bytes)
// and a bf16 gradient.
// TRA / TRB: that operand is instead a row K-slab of the token-major
// activation ([M/64][ldt][64] or [N/64][ldt][64]: h8 and dgu8 as their
// producers write them for the forward GEMMs), read through transposing LDS
// reads (MainLoop TR_A / TR_B); with TRB the accumulator columns are
// unpermuted (splitk_reduce_kernel<true>).
// SMALL: 128 x 128 tiles (4 waves of 64 x 64, two work-groups per CU) instead
// of 256 x 256 (8 waves of 128 x 64, one per CU); the partials' tiles and
// accumulator order follow the shape (acc_order_rc), the sums do not.
// Addressing of a transposed-read operand: row r of block r / 64 (fp8) or
// r / 32 (bf16) at token t lies at base + block * bs + t * ts, and ext bytes
// are readable from base (the rest reads as zero).  A row K-slab of [T, L]
// over ldt tokens: ts = 64, bs = ldt * 64; row-major [T, L] rows: ts = the row
// bytes, bs = 64, ext = T * ts.
struct TrOp {
  int64_t ts, bs, ext;
};

// One split's gradient tile, in place of its partials: the accumulators times
// s to out[m, n] (fp32, or rounded to bf16) for m below M, n below N, through
// LDS in passes of 64 tile rows (32 of each wave row; rows of 4 kN + 16 bytes,
// which shift by 4 banks), so that whole tile rows are written: a lane holds
// four consecutive columns of 32 rows.  The values are the reductions' with one
// split.  A write, a read and a launch less: gate/up and down gradient with one
// split (us), D = 1024, I = 3072, 1024 tokens 26 -> 15 and 18 -> 11; D = 2048, I =
// 6144, 3000 tokens 102 -> 77 and 54 -> 38 (bf16 gate/up 161 -> 134).
template <class TS, bool BF16, bool TRB>
SFP8_DEV void store_grad_tile(uint8_t* lds, const floatx16 (&acc)[TS::kTB][2], float s, int64_t m0, int64_t n0,
                              int64_t M, int64_t N, float* __restrict__ out) {
  constexpr int kRow = 4 * TS::kN + 16, kQuads = TS::kN / 4;  // bytes of a staged row, float4s in it
  static_assert(64 * kRow <= TS::kLds, "a pass fits the ring");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave & 1, wn = wave >> 1;
  const int fr = lane & 31, g = lane >> 5;
#pragma unroll
  for (int tb = 0; tb < TS::kTB; ++tb) {
    if (tb) __syncthreads();  // the pass before has been read
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = 64 * wn + (TRB ? 32 * nb + 8 * i + 4 * g : 32 * g + 16 * nb + 4 * i);  // acc_order_rc
        *reinterpret_cast<floatx4*>(lds + (32 * wm + fr) * kRow + 4 * c) =
            floatx4{acc[tb][nb][4 * i] * s, acc[tb][nb][4 * i + 1] * s, acc[tb][nb][4 * i + 2] * s,
                    acc[tb][nb][4 * i + 3] * s};
      }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 64 * kQuads / TS::kThreads; ++k) {
      const int idx = (int)threadIdx.x + TS::kThreads * k, lr = idx / kQuads, q = idx % kQuads;
      const int64_t m = m0 + 32 * TS::kTB * (lr >> 5) + 32 * tb + (lr & 31), n = n0 + 4 * q;
      const floatx4 v = *reinterpret_cast<const floatx4*>(lds + lr * kRow + 16 * q);
      if (m >= M || n >= N) continue;  // N % 4 == 0: the 4 values are wholly inside or past the row
      if constexpr (BF16)
        *reinterpret_cast<intx2*>(reinterpret_cast<uint16_t*>(out) + m * N + n) =
            intx2{(int)pack2_bf16(v[0], v[1]), (int)pack2_bf16(v[2], v[3])};
      else
        *reinterpret_cast<floatx4*>(out + m * N + n) = v;
    }
  }
}

template <class TS, bool BF16, int FMT_A, int FMT_B, bool TRA, bool TRB>
SFP8_DEV void wgrad_tile(
    uint8_t* lds, int tm, int tn, int sp, const uint8_t* __restrict__ at, const uint8_t* __restrict__ bt, int64_t M, int64_t N, int64_t ldt,
    int64_t kchunk, const float* __restrict__ sa, const float* __restrict__ sb, float* __restrict__ out,
    int tiles_m, int tiles_n, int partials, TrOp tra, TrOp trb) {
  const int64_t m0 = (int64_t)tm * TS::kM, n0 = (int64_t)tn * TS::kN;
  if (m0 >= M) return;  // the second half of a tile past the last row (work-group uniform)
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  floatx16 acc[TS::kTB][2];
  const int64_t kb = (int64_t)sp * kchunk;
  {
    // K-slab operands: slab (kb / 64) of A starts at (kb / 64) * rpa * 64.
    // TR operands (TrOp): tile row r is row r % kRows of block r / kRows at
    // the stage's tokens; a stage (64 K bytes: kRows tokens) is kRows * ts on.
    constexpr int kRows = BF16 ? 32 : 64;
    const int64_t rpa = slab_rows(M), rpb = slab_rows(N);
    const int64_t t0 = kb / (BF16 ? 2 : 1);  // first token of the split
    const int ats = (int)tra.ts, abs_ = (int)tra.bs, bts = (int)trb.ts, bbs = (int)trb.bs;
    const uint8_t* a0 = TRA ? at + (m0 / kRows) * tra.bs + t0 * tra.ts : at + (kb / kStage) * rpa * kStage + m0 * kStage;
    const uint8_t* b0 = TRB ? bt + (n0 / kRows) * trb.bs + t0 * trb.ts : bt + (kb / kStage) * rpb * kStage + n0 * kStage;
    const uint8_t* a_end = TRA ? at + tra.ext : at + ldt * rpa;
    const uint8_t* b_end = TRB ? bt + trb.ext : bt + ldt * rpb;
    TS::template Loop<BF16, FMT_A, FMT_B, TRA, TRB>::run(
        lds, a0, a_end - a0, [=](int r) { return TRA ? (r / kRows) * abs_ + (r % kRows) * ats : r * kStage; },
        TRA ? kRows * ats : (int)(rpa * kStage), b0, b_end - b0,
        [=](int r) { return TRB ? (r / kRows) * bbs + (r % kRows) * bts : plain_col_nb<2>(r) * kStage; },
        TRB ? kRows * bts : (int)(rpb * kStage), (int)((kchunk < ldt - kb ? kchunk : ldt - kb) / kStage), acc);
  }
  if (partials) {
    // accumulator order: [split][tile][wave][tb][nb][i][lane][4]
    float* frag = out + ((int64_t)sp * tiles_m * tiles_n + (int64_t)tm * tiles_n + tn) * (TS::kM * TS::kN) +
                  wave * (TS::kM * TS::kN / (TS::kThreads / 64));
#pragma unroll
    for (int tb = 0; tb < TS::kTB; ++tb)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          reinterpret_cast<floatx4*>(frag + (tb * 2 + nb) * 1024 + i * 256)[lane] =
              floatx4{acc[tb][nb][4 * i], acc[tb][nb][4 * i + 1], acc[tb][nb][4 * i + 2], acc[tb][nb][4 * i + 3]};
    return;
  }
  store_grad_tile<TS, BF16, TRB>(lds, acc, BF16 ? 1.0f : 1.0f / (sa[0] * sb[0]), m0, n0, M, N, out);
}
template <bool SMALL, bool BF16, int FMT_A, int FMT_B, bool TRA = false, bool TRB = false>
__global__ __launch_bounds__(TileShape<SMALL>::kThreads, TileShape<SMALL>::kMinWaves) void wgrad_kernel(
    const uint8_t* __restrict__ at, const uint8_t* __restrict__ bt, int64_t M, int64_t N, int64_t ldt,
    int64_t kchunk, const float* __restrict__ sa, const float* __restrict__ sb, float* __restrict__ out,
    int tiles_m, int tiles_n, int splits, int partials, TrOp tra, TrOp trb) {
  extern __shared__ __align__(16) uint8_t lds[];
  int tm, tn, sp = 0;
  if (!SMALL && !partials) {
    // one split: the last round in halves (tail_tile); a block's step, 16384
    // tokens, D = 2048, I = 6144 (384 gate/up tiles), 1963 -> 1940 us
    bool half;
    if (!tail_tile(tiles_m, tiles_n, tm, tn, half)) return;
    if (half) {
      wgrad_tile<Tile<2, 4>, BF16, FMT_A, FMT_B, TRA, TRB>(lds, tm, tn, 0, at, bt, M, N, ldt, kchunk, sa, sb, out,
                                                           tiles_m, tiles_n, 0, tra, trb);
      return;
    }
  } else {
    split_tile_coords(blockIdx.x, gridDim.x, tiles_m, tiles_n, splits, tm, tn, sp);
    if (sp >= splits) return;  // grid padding (work-group uniform)
  }
  wgrad_tile<TileShape<SMALL>, BF16, FMT_A, FMT_B, TRA, TRB>(lds, tm, tn, sp, at, bt, M, N, ldt, kchunk, sa, sb, out,
                                                             tiles_m, tiles_n, partials, tra, trb);
}

// K splits of expert e of a grouped gradient: `longest` for one with more than
// one and a half times the average rows, else `even`.
SFP8_DEV int moe_expert_splits(const int* __restrict__ plan, int e, int even, int longest) {
  const MoePlan P{plan};
  return 2 * (P.pcount(e) / kTile) * P.experts() > 3 * P.ntiles() ? longest : even;
}

// Grouped (MoE) weight gradient: out[e, m, n] = sum over expert e's padded
// rows t of A[m, t] * B[n, t] / (sa * sb), A and B token-contiguous K-slab
// copies over the padded expert order (zeros in padding rows).  Work-group
// Work-group (expert e, split sp, tile) of a 1-D grid over the three, tile
// fastest, takes split sp of the expert's 64-token stages (an even number of
// them; none for an expert without rows, whose gradient comes out zero).
// Each XCD takes a contiguous run of that order, so the work-groups resident
// on one XCD share one (expert, split) K range of A and B in its L2 (with the
// tile index spread over the XCDs, every XCD read every expert's operands:
// 3.9x the algorithmic bytes at the MoE workload).  With one split it
// writes out[e] itself; otherwise its raw partial in accumulator order to
// ws[e][sp][tile], summed in split order by splitk_reduce_kernel.
// BF16: bf16 operands, 2 bytes per padded row (`ldp` counts K bytes), and a
// bf16 gradient (bf16_wgrad_reduce_kernel).
// longest > splits: each expert has its own count (moe_expert_splits), read
// from the plan; the work-groups past it exit, and the reductions skip experts
// of one split.
template <class TS, bool BF16, int FMT_A, int FMT_B, bool TRA, bool TRB>
SFP8_DEV void moe_wgrad_tile(
    uint8_t* lds, int tm, int tn, int e, int sp, const uint8_t* __restrict__ at, const uint8_t* __restrict__ bt, int64_t M, int64_t N, int64_t ldp,
    const float* __restrict__ sa, const float* __restrict__ sb, float* __restrict__ out, float* __restrict__ ws,
    const int* __restrict__ plan, int tiles_m, int tiles_n, int splits, int ws_splits) {
  const MoePlan P{plan};
  const int64_t m0 = (int64_t)tm * TS::kM, n0 = (int64_t)tn * TS::kN;
  if (m0 >= M) return;  // the second half of a tile past the last row (work-group uniform)
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  constexpr int64_t kBpe = BF16 ? 2 : 1;  // K bytes per padded row
  const int64_t nst = P.pcount(e) * kBpe / kStage;  // a multiple of 4
  int64_t q = (nst + splits - 1) / splits;
  q = (q + 1) & ~(int64_t)1;
  const int64_t k0 = (int64_t)sp * q;
  const int64_t nk = nst - k0 < 0 ? 0 : (nst - k0 < q ? nst - k0 : q);
  const int64_t rpa = slab_rows(M), rpb = slab_rows(N);
  const int64_t s0 = P.pstart(e) * kBpe / kStage + k0;  // first 64-byte stage
  // Token-contiguous operands: stage s at s * rows * 64.  Row K-slab (TR)
  // operands ([rows/kRows][padded rows][64], as for wgrad_kernel): tile row r
  // is token r % kRows of slab r / kRows, and a stage (kRows tokens) is
  // kRows * 64 bytes on in every slab.
  constexpr int kRows = BF16 ? 32 : 64;
  const int64_t ldt_tok = ldp / kBpe;  // padded rows (ldp counts K bytes)
  const int ltok = (int)ldt_tok;
  const uint8_t* a0 = TRA ? at + (m0 / kRows) * ldt_tok * kStage + s0 * kRows * kStage : at + s0 * rpa * kStage + m0 * kStage;
  const uint8_t* b0 = TRB ? bt + (n0 / kRows) * ldt_tok * kStage + s0 * kRows * kStage : bt + s0 * rpb * kStage + n0 * kStage;
  const uint8_t* a_end = TRA ? at + (M / kRows) * ldt_tok * kStage : at + ldp * rpa;
  const uint8_t* b_end = TRB ? bt + (N / kRows) * ldt_tok * kStage : bt + ldp * rpb;
  const int64_t a_bytes = nk > 0 ? a_end - a0 : 0, b_bytes = nk > 0 ? b_end - b0 : 0;
  floatx16 acc[TS::kTB][2];
  TS::template Loop<BF16, FMT_A, FMT_B, TRA, TRB>::run(
      lds, a0, a_bytes, [=](int r) { return TRA ? ((r / kRows) * ltok + (r % kRows)) * kStage : r * kStage; },
      TRA ? kRows * kStage : (int)(rpa * kStage), b0, b_bytes,
      [=](int r) { return TRB ? ((r / kRows) * ltok + (r % kRows)) * kStage : plain_col_nb<2>(r) * kStage; },
      TRB ? kRows * kStage : (int)(rpb * kStage), (int)nk, acc);
  if (splits > 1) {
    // accumulator order: [expert][split of ws_splits][tile][wave][tb][nb][i][lane][4]
    float* frag = ws + (((int64_t)e * ws_splits + sp) * tiles_m * tiles_n + (int64_t)tm * tiles_n + tn) * (TS::kM * TS::kN) +
                  wave * (TS::kM * TS::kN / (TS::kThreads / 64));
#pragma unroll
    for (int tb = 0; tb < TS::kTB; ++tb)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          reinterpret_cast<floatx4*>(frag + (tb * 2 + nb) * 1024 + i * 256)[lane] =
              floatx4{acc[tb][nb][4 * i], acc[tb][nb][4 * i + 1], acc[tb][nb][4 * i + 2], acc[tb][nb][4 * i + 3]};
    return;
  }
  const int64_t skip = (int64_t)e * M * N;
  store_grad_tile<TS, BF16, TRB>(lds, acc, BF16 ? 1.0f : 1.0f / (sa[0] * sb[0]), m0, n0, M, N,
                                 BF16 ? reinterpret_cast<float*>(reinterpret_cast<uint16_t*>(out) + skip) : out + skip);
}
template <bool SMALL, bool BF16, int FMT_A, int FMT_B, bool TRA = false, bool TRB = false>
__global__ __launch_bounds__(TileShape<SMALL>::kThreads, TileShape<SMALL>::kMinWaves) void moe_wgrad_kernel(
    const uint8_t* __restrict__ at, const uint8_t* __restrict__ bt, int64_t M, int64_t N, int64_t ldp,
    const float* __restrict__ sa, const float* __restrict__ sb, float* __restrict__ out, float* __restrict__ ws,
    const int* __restrict__ plan, int tiles_m, int tiles_n, int splits, int longest, int experts) {
  extern __shared__ __align__(16) uint8_t lds[];
  const int tiles = tiles_m * tiles_n, n = tiles * splits * experts, pid = blockIdx.x;
  int lid, e, sp, count = splits, tm, tn;
  if (longest > splits) {
    // the grid has `longest` splits, one after the other; a split's run over
    // the XCDs is turned by its share of them, so that the splits of one expert
    // lie on different XCDs
    const int n0 = tiles * experts;
    sp = pid / n0;
    lid = (xcd_run(pid % n0, n0) + (int)((int64_t)n0 * sp / longest)) % n0;
    e = lid / tiles;
    count = moe_expert_splits(plan, e, splits, longest);
    if (sp >= count) return;
  } else {
    int full = n;
    if constexpr (!SMALL) {
      // one split: the last round in halves, as tail_tile (the run of full tiles
      // is the grid's without them); 8 experts, 131072 rows, D = 1024, I = 1536
      // (384 gate/up tiles), the experts' step 2344 -> 2329 us
      if (splits == 1) full = tail_full(n, kRound);
      if (pid >= full) {
        lid = full + ((pid - full) >> 1);
        if (lid >= n) return;
        raster(lid % tiles, tiles_m, tiles_n, tm, tn);
        moe_wgrad_tile<Tile<2, 4>, BF16, FMT_A, FMT_B, TRA, TRB>(lds, 2 * tm + ((pid - full) & 1), tn, lid / tiles, 0,
                                                                 at, bt, M, N, ldp, sa, sb, out, ws, plan, tiles_m,
                                                                 tiles_n, 1, 1);
        return;
      }
    }
    lid = xcd_run(pid, full);
    e = lid / (tiles * splits);
    sp = (lid / tiles) % splits;
  }
  raster(lid % tiles, tiles_m, tiles_n, tm, tn);
  moe_wgrad_tile<TileShape<SMALL>, BF16, FMT_A, FMT_B, TRA, TRB>(lds, tm, tn, e, sp, at, bt, M, N, ldp, sa, sb, out, ws,
                                                                 plan, tiles_m, tiles_n, count, longest);
}

// out[0, n) = 0: four floats per thread (n % 4 == 0, out 16-byte aligned).
__global__ __launch_bounds__(256) void zero_fill_kernel(float* __restrict__ out, int64_t n) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i < n) *reinterpret_cast<floatx4*>(out + i) = floatx4{0.f, 0.f, 0.f, 0.f};
}

// Tile row r and column c of the first value of float4 q of one partial tile
// of wgrad_kernel<SMALL, ..> in accumulator order [wave][tb][nb][i][lane][4]
// (kTileQ float4s; wave (wm, wn) = (wave & 1, wave >> 1) owns rows
// 32 kTB wm.. and columns 64 wn..): B-tile rows permuted by plain_col_nb<2>
// (accumulator v of block nb, lane half g is column 64 wn + 32 g + 16 nb + v),
// or with TR_B unpermuted (column 64 wn + 32 nb + 8 (v / 4) + 4 g + v % 4).
template <bool SMALL>
constexpr int kTileQLog = SMALL ? 12 : 14;  // log2 of the float4s of a tile
template <bool SMALL, bool TR_B>
SFP8_DEV void acc_order_rc(int q, int& r, int& c) {
  constexpr int TBB = SMALL ? 1 : 2;  // bits of tb
  const int lane = q & 63, i = (q >> 6) & 3, nb = (q >> 8) & 1, tb = (q >> 9) & (TileShape<SMALL>::kTB - 1);
  const int wave = (q >> (9 + TBB)) & (TileShape<SMALL>::kThreads / 64 - 1), g = lane >> 5;
  r = 32 * TileShape<SMALL>::kTB * (wave & 1) + 32 * tb + (lane & 31);
  c = 64 * (wave >> 1) + (TR_B ? 32 * nb + 8 * i + 4 * g : 32 * g + 16 * nb + 4 * i);
}

// Split-K reduction of the accumulator-order partials of wgrad_kernel:
// out[m, n] = (sum over s ascending of ws[s]) / (sa * sb).  Thread q owns the
// q-th float4 of one split's partials; its (m, n) follows from the MFMA
// accumulator layout (acc_order_rc; TR_B: partials of wgrad_kernel<..,
// true>).
template <bool SMALL, bool TR_B>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ ws, int splits,
                                                            int64_t n4, int tiles_n, int64_t M, int64_t N,
                                                            const float* __restrict__ sa,
                                                            const float* __restrict__ sb, float* __restrict__ out,
                                                            const int* __restrict__ plan, int even) {
  // expert blockIdx.y of a grouped gradient: its splits' partials, its [M, N];
  // with a plan the splits that it has (one: the gradient is written)
  ws += (int64_t)blockIdx.y * splits * n4 * 4;
  if (plan) splits = moe_expert_splits(plan, blockIdx.y, even, splits);
  if (splits == 1) return;
  out += (int64_t)blockIdx.y * M * N;
  const floatx4* w4 = reinterpret_cast<const floatx4*>(ws);
  for (int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x; q < n4; q += (int64_t)gridDim.x * 256) {
    floatx4 acc = __builtin_nontemporal_load(w4 + q);
    for (int s = 1; s < splits; ++s) acc += __builtin_nontemporal_load(w4 + (int64_t)s * n4 + q);
    int r, c;
    acc_order_rc<SMALL, TR_B>((int)(q & ((1 << kTileQLog<SMALL>) - 1)), r, c);
    const int64_t tile = q >> kTileQLog<SMALL>;
    const int64_t tm = tile / tiles_n, tn = tile % tiles_n;
    const int64_t m = tm * TileShape<SMALL>::kM + r, n = tn * TileShape<SMALL>::kM + c;
    if (m < M && n < N) {
      const float deq = 1.0f / (sa[0] * sb[0]);
      *reinterpret_cast<floatx4*>(out + m * N + n) = acc * deq;
    }
  }
}

// ---------------------------------------------------------------------------
// bf16 SwiGLU MLP path (spark-gpt's default, non-FP8 path): the gate/up GEMM
// with the SwiGLU epilogue of _swiglu_gemm_kernel (train.py:1625-1716), the
// plain bf16 GEMM of its dgrad and the rounding reduce of its weight
// gradient.  Operands are bf16 K-slabs (2 bytes per element: a 64-byte
// stage is 32 elements of K) or, for the forward's A, the caller's
// row-major x.

// Forward: gate/up = x @ W^T per tile (fp32 accumulate), then
//   g = bf16(acc_g * rs), u = bf16(acc_u * rs)   (rs = rstd[row] when the
//   RMSNorm is folded into W, else 1; train.py:1696-1702),
//   h = bf16(g * sigmoid(g) * u)                (train.py:1709-1715),
// gu = [g | u] row-major [rows, 2I] (saved for the backward), h row-major
// [rows, I].  Tile: 256 rows x 128 (gate, up) column pairs; B is the bf16
// K-slab of W [2D/64][slab_rows(2I)][64] in the paired layout (a lane holds
// g and u of the same 32 consecutive columns).  A = x row-major [rows, D]
// (rows past the tile's last read as zero through the range check).
// With a MoE plan: tile row tm of padded expert order reads and writes the
// expert-order rows urow(tm) .. + rows(tm); W of expert e at w + e * w_estride
// (bytes).  Columns from I on (the last tile when I % 128 != 0) are not
// written.
// staging row: 128 (64) bf16 columns and 16 bytes
template <bool SMALL>
constexpr int kGuStride = SMALL ? 144 : 272;

// 8 waves (two per SIMD): wave (wm, wn) owns tile rows 128*wm.. and one
// 32-column block of gate and one of up, columns 32*wn.. of each half.
// SMALL: 128 rows x 64 columns by 4 waves of 64 rows, staged in one pass.
// w_rows: W is row-major [2I, D] bf16 as the caller has it instead of its
// K-slab; gu may be null (evaluation: nothing is saved).
template <bool SMALL>
__global__ __launch_bounds__(TileShape<SMALL>::kThreads, TileShape<SMALL>::kMinWaves) void bf16_swiglu_fwd_kernel(
    const uint16_t* __restrict__ x, const uint8_t* __restrict__ w, int64_t T, int64_t D, int64_t I,
    const float* __restrict__ rstd, uint16_t* __restrict__ gu, uint16_t* __restrict__ h, int tiles_m, int tiles_n,
    const int* __restrict__ plan, int64_t w_estride, int64_t ldxs, int w_rows) {
  using TS = TileShape<SMALL>;
  constexpr int kN = TS::kM / 2;  // (gate, up) columns of a tile
  constexpr int kGs = kGuStride<SMALL>;
  extern __shared__ __align__(16) uint8_t lds[];
  int tm, tn;
  tile_coords(blockIdx.x, gridDim.x, tiles_m, tiles_n, tm, tn);
  int64_t r0 = (int64_t)tm * TS::kM, nrows = T - r0;
  if (plan) {
    const MoePlan P{plan};
    const int pt = TS::plan_tile(tm);
    if (pt >= P.ntiles()) return;  // work-group uniform
    r0 = P.urow(pt) + TS::plan_skip(tm);
    nrows = P.rows(pt) - TS::plan_skip(tm);
    if (nrows <= 0) return;  // nothing but padding rows, which have no output
    w += P.expert(pt) * w_estride;
  }
  const int64_t n0 = (int64_t)tn * kN;
  const int64_t ldx = D * 2;  // bytes per x row = K bytes
  const int64_t wr = slab_rows(2 * I);
  // the outputs from the tile's first row (gu [rows, 2I], h [rows, I], bf16)
  const __amdgpu_buffer_rsrc_t rgu = make_rsrc(gu + r0 * 2 * I, gu ? nrows * 4 * I : 0);
  const __amdgpu_buffer_rsrc_t rho = make_rsrc(h + r0 * I, nrows * 2 * I);
  floatx16 acc[TS::kTB][2];  // [tb][0] gate, [tb][1] up
  // A: x row-major [T, D] (rows past the tile's last read as zero through
  // the range check), or with ldxs > 0 its row K-slab [2D/64][ldxs][64]
  // (zero padding rows): a K stage of the tile is then one 16 KiB block of
  // whole 128-byte lines instead of 256 half lines 2D bytes apart
  const bool xslab = ldxs > 0;
  TS::template Loop<true, 0, 0, false, false, true>::run(
      lds, reinterpret_cast<const uint8_t*>(x) + r0 * (xslab ? kStage : ldx),
      xslab ? ldx * ldxs - r0 * kStage : nrows * ldx, [=](int r) { return r * (xslab ? kStage : (int)ldx); },
      xslab ? (int)(ldxs * kStage) : kStage, w, ldx * (w_rows ? 2 * I : wr), [=](int r) {
        return ((r / kN) * (int)I + (int)n0 + (SMALL ? paired_col64(r) : paired_col8(r))) * (w_rows ? (int)ldx : kStage);
      },
      w_rows ? kStage : (int)(wr * kStage), (int)(ldx / kStage), acc);
  // Epilogue in two passes (SMALL: one) of 128 tile rows: pass P takes the
  // lanes' row blocks tb = 2P, 2P+1 (tile row 32 kTB wm + 64 P + 32 (tb & 1) +
  // fr, staging row 64 wm + 32 (tb & 1) + fr), stages g, u and h as bf16 rows in LDS,
  // then writes them as whole 256-byte row runs.
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave & 1, wn = wave >> 1, fr = lane & 31, g = lane >> 5;
  const int cb = 32 * wn + 16 * g;  // first of this lane's 16 columns in the tile
  uint8_t* Gs = lds;
  uint8_t* Us = lds + 128 * kGs;
  uint8_t* Hs = lds + 2 * 128 * kGs;
  const float c_exp = -1.4426950408889634f;
#pragma unroll
  for (int P = 0; P < TS::kTB / 2; ++P) {
    if (P) __syncthreads();  // the first pass's rows are out of the staging tiles
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int tb = 2 * P + q;
      const int lr = 32 * TS::kTB * wm + 32 * tb + fr;  // row within the tile
      const float rs = (rstd && lr < nrows) ? rstd[r0 + lr] : 1.0f;
      uint32_t gw[8], uw[8], hw[8];
#pragma unroll
      for (int v = 0; v < 16; v += 2) {
        const uint32_t pg = pack2_bf16(acc[tb][0][v] * rs, acc[tb][0][v + 1] * rs);
        const uint32_t pu = pack2_bf16(acc[tb][1][v] * rs, acc[tb][1][v + 1] * rs);
        const float g0 = __uint_as_float(pg << 16), g1 = __uint_as_float(pg & 0xffff0000u);
        const float u0 = __uint_as_float(pu << 16), u1 = __uint_as_float(pu & 0xffff0000u);
        const float s0 = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g0 * c_exp));
        const float s1 = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g1 * c_exp));
        const int k = v / 2;
        gw[k] = pg;
        uw[k] = pu;
        hw[k] = pack2_bf16(g0 * s0 * u0, g1 * s1 * u1);
      }
      const int sr = 64 * wm + 32 * q + fr;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        store16(Gs + sr * kGs + 2 * cb + 16 * j, {gw[4 * j], gw[4 * j + 1], gw[4 * j + 2], gw[4 * j + 3]});
        store16(Us + sr * kGs + 2 * cb + 16 * j, {uw[4 * j], uw[4 * j + 1], uw[4 * j + 2], uw[4 * j + 3]});
        store16(Hs + sr * kGs + 2 * cb + 16 * j, {hw[4 * j], hw[4 * j + 1], hw[4 * j + 2], hw[4 * j + 3]});
      }
    }
    __syncthreads();
    // 128 rows x kN / 8 pieces of 16 bytes per output: kN / 8 lanes per row;
    // buffer stores from the tile's first row, a piece past the valid rows or
    // past I (I % 8 == 0: whole pieces) at offset 2^31 (beyond the range:
    // dropped), so every thread issues the same stores without a branch
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int idx = (int)threadIdx.x + TS::kThreads * k;
      const int sr = idx / (kN / 8), c = idx % (kN / 8);
      const int lr = SMALL ? sr : half_tile_row(sr, P);
      const int64_t col = n0 + 8 * c;
      const uint32_t in = 0u - (uint32_t)(lr < nrows && col < I);
      const uint32_t og = ((uint32_t)((lr * 2 * I + col) * 2) & in) | (~in & 0x80000000u);
      const uint32_t oh = ((uint32_t)((lr * I + col) * 2) & in) | (~in & 0x80000000u);
      if (gu) {  // uniform
        __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const intx4*>(Gs + sr * kGs + 16 * c), rgu,
                                               og, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const intx4*>(Us + sr * kGs + 16 * c), rgu,
                                               og + (uint32_t)(2 * I), 0, 0);
      }
      __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const intx4*>(Hs + sr * kGs + 16 * c), rho,
                                             oh, 0, 0);
    }
  }
}

// Evaluation of a few rows (generation): h = bf16(g * sigmoid(g) * u), g, u =
// bf16(x W^T), for up to 64 rows of x and W row-major [2I, D] bf16 as the
// caller has it.  The call reads W once and little else, so it is bound by the
// memory's bandwidth and latency: a work-group of 8 waves takes 16 gate and
// the 16 up rows of W (one MFMA's 32) against NT tiles of 32 rows of x.  K runs
// in chunks of 128 through a ring of kRing LDS slots, kRing - 1 of them in
// flight; all waves load, wave t multiplies x tile t.  One chain of MFMAs runs
// over the whole K, 16 at a time, with the K values of MainLoop's fragments in
// MainLoop's order, so that a row's h has the bytes of the tiled kernels,
// training's and those from 65 rows on (K shared by the waves and their sums
// added differed from them in the last bit now and then, and was no faster: us
// at 1, 8 and 64 rows with weights out of the caches, D = 1024, I = 3072, 5.4 5.8
// 9.6 -> 5.5 5.5 7.1 (2.3 TB/s at 8 rows); D = 2048, I = 8192, 17.2 18.5 29.5 ->
// 17.5 17.9 21.5 (3.7 TB/s); D = 256, I = 1024, 2.8 3.0 3.9 -> 3.0 3.1 3.3).  At 65
// rows the tiled kernel takes 16.4, 31.6 and 6.1.
// LDS rows are 128 bytes (64 of K); row r keeps its 16-byte chunk c at c ^ ((r
// >> 1) & 7), so that 16 lanes reading one chunk of 16 rows meet every bank
// once.  Rows of x past T lie past the descriptor's records and cost no traffic.
constexpr int kEvalRows = 64;  // most rows of x
template <int NT>
struct EvalShape {
  static constexpr int kRows = 32 + 32 * NT;     // LDS rows of a 64-wide K step: W, then x
  static constexpr int kSteps = 2;               // K steps of 64 in a chunk
  static constexpr int kSlot = kSteps * kRows * 128;
  static constexpr int kRing = NT == 1 ? 4 : 3;  // two work-groups fit a CU
  static constexpr int kLds = kRing * kSlot;
  static constexpr int kDma = 1 + NT;            // 1 KiB loads of each wave per chunk
};
template <int NT>
__global__ __launch_bounds__(512) void bf16_swiglu_eval_kernel(const uint16_t* __restrict__ x,
                                                               const uint16_t* __restrict__ w, int T, int D, int I,
                                                               uint16_t* __restrict__ h) {
  using S = EvalShape<NT>;
  extern __shared__ __align__(16) uint8_t lds[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, fr = lane & 31, g = lane >> 5;
  const int n0 = (int)blockIdx.x * 16, ldx = 2 * D;
  const int steps = D / 64, chunks = (steps + S::kSteps - 1) / S::kSteps;
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(w, (int64_t)2 * I * ldx), rx = make_rsrc(x, (int64_t)T * ldx);
  // a load covers 8 rows of 128 bytes; this wave's: row group j of W in K step
  // wave / 4, and of x (NT = 1: the same) in one (NT = 2: each) step
  const auto chunk_of = [=](int row) { return (uint32_t)(((lane & 7) ^ ((row >> 1) & 7)) << 4); };
  const int wj = wave & 3, wr = 8 * wj + (lane >> 3);
  const int xj = NT == 1 ? wj : wave, xr = 8 * xj + (lane >> 3);
  const uint32_t voff_w = (uint32_t)(((wr >> 4) * I + n0 + (wr & 15)) * ldx) + chunk_of(wr);
  const uint32_t voff_x = (uint32_t)(xr * ldx) + chunk_of(xr);
  const auto load = [&](int c) {  // chunk c; steps past the last are aimed out of range
    uint8_t* slot = lds + (c % S::kRing) * S::kSlot;
    const int s0 = c * S::kSteps + (wave >> 2);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_ptr_t)(slot + (wave >> 2) * S::kRows * 128 + wj * 1024), 16,
                                             s0 < steps ? voff_w + 128 * s0 : 0x80000000u, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int st = NT == 1 ? wave >> 2 : i, s = c * S::kSteps + st;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_ptr_t)(slot + (st * S::kRows + 32) * 128 + xj * 1024), 16,
                                               s < steps ? voff_x + 128 * s : 0x80000000u, 0, 0, 0);
    }
  };
  for (int c = 0; c < S::kRing - 1; ++c) load(c);
  floatx16 acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  // a chunk's operands, in the order of MainLoop's fragments: per 64 bytes of a
  // row the lane half's first 16-byte chunk, then its second
  struct Frag {
    bf16x8 w[4 * S::kSteps], x[4 * S::kSteps];
  };
  const auto read = [&](Frag& f, int c) {
    const uint8_t* pw = lds + (c % S::kRing) * S::kSlot + fr * 128;
#pragma unroll
    for (int k = 0; k < 4 * S::kSteps; ++k) {
      const int at = (k >> 2) * S::kRows * 128 + (((2 * (k & 2) + 2 * g + (k & 1)) ^ ((fr >> 1) & 7)) << 4);
      f.w[k] = *reinterpret_cast<const bf16x8*>(pw + at);
      f.x[k] = *reinterpret_cast<const bf16x8*>(pw + (32 + 32 * wave) * 128 + at);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  const auto multiply = [&](const Frag& f, int nk) {
#pragma unroll
    for (int st = 0; st < S::kSteps; ++st) {
      if (st >= nk) break;
#pragma unroll
      for (int k = 4 * st; k < 4 * st + 4; ++k)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.w[k], f.x[k], acc, 0, 0, 0);
    }
  };
  // chunk c has landed, and every wave's reads of chunk c - 1, whose slot the
  // next load fills, are done; its operands come while chunk c - 1 multiplies
  const auto chunk = [&](int c, Frag& cur, const Frag& prev) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(S::kDma * (S::kRing - 2)) : "memory");
    load(c + S::kRing - 1);
    if (wave >= NT) return;
    read(cur, c);
    if (c) multiply(prev, S::kSteps);
  };
  Frag f0, f1;
  for (int c = 0; c < chunks; c += 2) {
    chunk(c, f0, f1);
    if (c + 1 < chunks) chunk(c + 1, f1, f0);
  }
  if (wave < NT) {
    const int last = steps - (chunks - 1) * S::kSteps;
    if (chunks & 1) multiply(f0, last);
    else multiply(f1, last);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the loads past the last chunk
  // accumulator 4 q + i is W row 8 q + 4 g + i of the 32: gate for q < 2, up of
  // the same columns for q + 2
  const int row = 32 * wave + fr;
  if (wave >= NT || row >= T) return;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    uint32_t o[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int v = 4 * q + 2 * i;
      float g0 = acc[v], g1 = acc[v + 1], u0 = acc[8 + v], u1 = acc[8 + v + 1];
      round2_bf16(g0, g1);
      round2_bf16(u0, u1);
      o[i] = pack2_bf16(g0 * sigmoid_fast(g0) * u0, g1 * sigmoid_fast(g1) * u1);
    }
    *reinterpret_cast<intx2*>(h + (int64_t)row * I + n0 + 8 * q + 4 * g) = intx2{(int)o[0], (int)o[1]};
  }
}

// The bf16 gate/up forward, persistent, with the SwiGLU of each tile under the
// K loop of the next, after swiglu_pipe_kernel: tiles of 256 rows x 64 (gate,
// up) column pairs, 8 waves of 64 x 64, one work-group per CU.  At K = 16
// stages (D = 512) the one-tile kernel spends as long writing its 6 bytes per
// pair as in its K loop, each with the other idle.
//
// At a tile's end a lane packs bf16(g * rs), bf16(u * rs) of its 32 pairs into
// 32 registers (rs = rstd of the row, brought to LDS by DMA with the tile's
// first stages); the next tile's first KE stages run the 8 units of 4 pairs in
// six pieces each.  A unit leaves its gate and up words in place of the pairs
// and two h words; a finished row block goes to LDS and, in the next stage,
// out as whole 128-byte rows.  (Stored from the registers, 32 contiguous bytes
// of each row per instruction, the stores took as long as the rest: 224
// against 149 us without them.)  Stages past KE have a plain loop of four, so
// D is any multiple of 128 from 32 KE on.  Operands, plan and rounding as
// bf16_swiglu_fwd_kernel.
template <int KE, bool EXACT>
struct Bf16Pipe {
  using ML = MainLoop<true, 0, 0, true, 2, kStages, false, false, 2, 2>;
  static constexpr int kUnits = 8, kPre = 2, kSlots = ML::kMfma - kPre;
  // the pieces fill the slots of stages 0 .. KE - 2; a row block staged at the
  // end of a stage is written in the next
  static constexpr int kAllSlots = (KE - 1) * kSlots, kPieces = 6 * kUnits;
  static constexpr int first_piece(int slot) { return slot < kAllSlots ? slot * kPieces / kAllSlots : kPieces; }
  static constexpr int blocks_done(int kt) { return first_piece((kt + 1) * kSlots) / 24; }
  static constexpr int kRow = 144, kOut = 128 * kRow;  // staging: row stride, bytes per output
  static constexpr int kWrites = 6;  // stores per thread of a row block: 128 rows x 8 pieces x 3 outputs
  // the row block written in stage kt, or -1
  static constexpr int written(int kt) { return kt > 0 && blocks_done(kt - 1) > blocks_done(kt - 2) ? blocks_done(kt - 1) - 1 : -1; }

  struct Ctx {
    uint8_t* lds;
    uint8_t* stg;  // staging rows
    intx4 rv;      // the piece read last
    __amdgpu_buffer_rsrc_t ra, rb, nra, nrb;  // this tile's operands and the next's (no records: none)
    uint32_t voff_a[4], voff_b[2], aoff[8], boff[8];
    int nk, a_ss, b_ss, wave;
    typename ML::Frag f[2];
    floatx16 acc[2][2];
    // the previous tile's epilogue
    uint32_t E[2][16], hw[8];
    float gb[4], ub[4], hb[4], ex[4], sg[4];
    __amdgpu_buffer_rsrc_t rgu, rh;  // its outputs from its first row (no records: no previous tile)
    int so_g, so_u, so_h;            // its first column's byte offsets
    int ld_gu, ld_h;                 // bytes per output row
  };

  template <int RB, int Q, int I>
  static SFP8_DEV void unpack(Ctx& c) {
    uint32_t p = c.E[RB][4 * Q + I];
    asm volatile("" : "+v"(p));
    c.gb[I] = __uint_as_float(p << 16);
    c.ub[I] = __uint_as_float(p & 0xffff0000u);
    c.ex[I] = __builtin_amdgcn_exp2f(c.gb[I] * -1.4426950408889634f);
  }
  // Piece P of unit U, kept in its slot by empty asm statements as in
  // SwigluPipe::unit_piece.
  template <int U, int P>
  static SFP8_DEV void unit_piece(Ctx& c) {
    constexpr int RB = U / 4, Q = U % 4;
    if constexpr (P == 0) {
      unpack<RB, Q, 0>(c);
      unpack<RB, Q, 1>(c);
      asm volatile("" ::"v"(c.ex[0]), "v"(c.ex[1]));
    } else if constexpr (P == 1) {
      c.sg[0] = __builtin_amdgcn_rcpf(1.0f + c.ex[0]);
      c.sg[1] = __builtin_amdgcn_rcpf(1.0f + c.ex[1]);
      unpack<RB, Q, 2>(c);
      asm volatile("" ::"v"(c.sg[0]), "v"(c.sg[1]), "v"(c.ex[2]));
    } else if constexpr (P == 2) {
      unpack<RB, Q, 3>(c);
      c.sg[2] = __builtin_amdgcn_rcpf(1.0f + c.ex[2]);
      c.hb[0] = c.gb[0] * c.sg[0] * c.ub[0];
      c.hb[1] = c.gb[1] * c.sg[1] * c.ub[1];
      asm volatile("" ::"v"(c.ex[3]), "v"(c.sg[2]), "v"(c.hb[0]), "v"(c.hb[1]));
    } else if constexpr (P == 3) {
      c.sg[3] = __builtin_amdgcn_rcpf(1.0f + c.ex[3]);
      c.hb[2] = c.gb[2] * c.sg[2] * c.ub[2];
      c.hw[2 * Q] = pack2_bf16(c.hb[0], c.hb[1]);
      asm volatile("" ::"v"(c.sg[3]), "v"(c.hb[2]), "v"(c.hw[2 * Q]));
    } else if constexpr (P == 4) {
      c.hb[3] = c.gb[3] * c.sg[3] * c.ub[3];
      c.hw[2 * Q + 1] = pack2_bf16(c.hb[2], c.hb[3]);
      asm volatile("" ::"v"(c.hw[2 * Q + 1]));
    } else {
      // four pairs -> two gate words, two up words
      const uint32_t e0 = c.E[RB][4 * Q], e1 = c.E[RB][4 * Q + 1], e2 = c.E[RB][4 * Q + 2], e3 = c.E[RB][4 * Q + 3];
      c.E[RB][4 * Q] = __builtin_amdgcn_perm(e1, e0, 0x05040100u);
      c.E[RB][4 * Q + 1] = __builtin_amdgcn_perm(e3, e2, 0x05040100u);
      c.E[RB][4 * Q + 2] = __builtin_amdgcn_perm(e1, e0, 0x07060302u);
      c.E[RB][4 * Q + 3] = __builtin_amdgcn_perm(e3, e2, 0x07060302u);
      asm volatile("" ::"v"(c.E[RB][4 * Q]), "v"(c.E[RB][4 * Q + 1]), "v"(c.E[RB][4 * Q + 2]),
                   "v"(c.E[RB][4 * Q + 3]));
    }
  }
  template <int P, int END>
  static SFP8_DEV void pieces(Ctx& c) {
    if constexpr (P < END) {
      unit_piece<P / 6, P % 6>(c);
      pieces<P + 1, END>(c);
    }
  }

  // Row block RB of the previous tile (128 rows: 32 of each wave row) into the
  // staging rows: gate, up, h, each 64 columns.
  template <int RB>
  static SFP8_DEV void block_stage(Ctx& c) {
    const int lane = threadIdx.x & 63, wm = c.wave % ML::kWM, wn = c.wave / ML::kWM;
    uint8_t* p = c.stg + (32 * wm + (lane & 31)) * kRow + 64 * wn + 32 * (lane >> 5);
    uint32_t(&E)[16] = c.E[RB];
    store16(p, {E[0], E[1], E[4], E[5]});
    store16(p + 16, {E[8], E[9], E[12], E[13]});
    store16(p + kOut, {E[2], E[3], E[6], E[7]});
    store16(p + kOut + 16, {E[10], E[11], E[14], E[15]});
    store16(p + 2 * kOut, {c.hw[0], c.hw[1], c.hw[2], c.hw[3]});
    store16(p + 2 * kOut + 16, {c.hw[4], c.hw[5], c.hw[6], c.hw[7]});
  }
  // Piece K of this thread of the staged row block RB: read, and stored as part
  // of a whole 128-byte row.  Rows past the tile's last lie past the
  // descriptors' records and are dropped (so are all when there is no previous
  // tile).
  template <int K>
  static SFP8_DEV intx4 row_read(const Ctx& c) {
    const int tid = threadIdx.x;
    return *reinterpret_cast<const intx4*>(c.stg + (K / 2) * kOut + ((tid >> 3) + 64 * (K & 1)) * kRow + 16 * (tid & 7));
  }
  template <int RB, int K>
  static SFP8_DEV void row_write(const Ctx& c, const intx4& v) {
    const int tid = threadIdx.x, sr = (tid >> 3) + 64 * (K & 1);
    const int row = 64 * (sr >> 5) + 32 * RB + (sr & 31);
    // the column goes in the vector offset: with a scalar register there the
    // compiler sees no hazard in a vector instruction that overwrites the data
    // right after the store, and such stores wrote that instruction's result
    const uint32_t vo = (uint32_t)(row * (K < 4 ? c.ld_gu : c.ld_h) + 16 * (tid & 7)) +
                        (uint32_t)(K < 2 ? c.so_g : K < 4 ? c.so_u : c.so_h);
    __builtin_amdgcn_raw_buffer_store_b128(v, K < 4 ? c.rgu : c.rh, vo, 0, 0);
  }

  // One stage: kPre MFMAs, the wait for the next stage's DMA and the barrier,
  // then a slot per MFMA with the DMA (instruction j of stage kt + 3, or of
  // stage NEXT of the next tile), the fragment reads (those the next stage
  // starts with first) and, in the first KE stages, the pieces.
  // PH = stage % 4; KT = the stage, or -1 past KE; PREV = the stage before, if
  // it may be one that writes
  template <int PH, int KT, int NEXT, int PREV = KT - 1>
  static SFP8_DEV void stage(Ctx& c, int kt) {
    static_assert(kSlots == kWrites, "a piece per slot");
    ML::template mfma_range<0, kPre>(c.f[PH & 1], c.acc);
    __builtin_amdgcn_sched_barrier(0);
    // what the stage before issued may still fly: its DMA and, after a write
    // stage, its stores (vmcnt counts both and falls in issue order; every wave
    // issues the same number); block_stage's LDS writes must have landed
    constexpr int kFly = ML::kDma + (PREV >= 0 && written(PREV) >= 0 ? kWrites : 0);
    if constexpr (KT >= 0 && written(KT) >= 0)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kFly) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kFly) : "memory");
    __builtin_amdgcn_sched_barrier(0);
    slots<PH, KT, NEXT, 0>(c, kt);
    if constexpr (KT >= 0) {
      if constexpr (written(KT) >= 0) row_write<written(KT), kSlots - 1>(c, c.rv);
      if constexpr (blocks_done(KT) > blocks_done(KT - 1)) block_stage<blocks_done(KT) - 1>(c);
    }
  }
  template <int PH, int KT, int NEXT, int J>
  static SFP8_DEV void slots(Ctx& c, int kt) {
    if constexpr (J < kSlots) {
      ML::template mfma_range<kPre + J, kPre + J + 1>(c.f[PH & 1], c.acc);
#pragma unroll
      for (int j = J * ML::kDma / kSlots; j < (J + 1) * ML::kDma / kSlots; ++j) {
        const int s = NEXT >= 0 ? NEXT : kt + kStages - 1;
        int ass = c.a_ss, bss = c.b_ss;
        asm volatile("" : "+s"(ass), "+s"(bss));  // the products are made here, not kept for every stage
        ML::load_one(j, c.lds, (PH + 3) % kStages, NEXT >= 0 ? c.nra : c.ra, NEXT >= 0 ? c.nrb : c.rb, c.voff_a,
                     c.voff_b, s * ass, s * bss, c.wave);
      }
      if constexpr (J == 0) {
        ML::template read_frag<0>(c.lds, (PH + 1) % kStages, c.aoff, c.boff, c.f[(PH & 1) ^ 1]);
        ML::template read_frag<2>(c.lds, (PH + 1) % kStages, c.aoff, c.boff, c.f[(PH & 1) ^ 1]);
      } else if constexpr (J < 3) {
        ML::template read_frag<J == 1 ? 3 : 1>(c.lds, (PH + 1) % kStages, c.aoff, c.boff, c.f[(PH & 1) ^ 1]);
      }
      if constexpr (KT >= 0) {
        if constexpr (written(KT) >= 0) {  // each piece stored a slot after it is read
          if constexpr (J > 0) row_write<written(KT), J - 1>(c, c.rv);
          c.rv = row_read<J>(c);
        }
        pieces<first_piece(KT * kSlots + J), first_piece(KT * kSlots + J + 1)>(c);
      }
      __builtin_amdgcn_sched_barrier(0);
      slots<PH, KT, NEXT, J + 1>(c, kt);
    }
  }
  // Stages KT .. KE - 1; EXACT: the tile has no others, so the last three
  // load the next tile's first.
  template <int KT>
  static SFP8_DEV void stages(Ctx& c) {
    if constexpr (KT < KE) {
      stage<KT % kStages, KT, (EXACT ? KT + kStages - 1 - KE : -1)>(c, KT);
      stages<KT + 1>(c);
    }
  }
  static SFP8_DEV void rest(Ctx& c) {
    int kt = KE;
    // (the first of these follows a write stage; waiting for the stores there
    // too keeps one loop body)
    for (; kt < c.nk - 4; kt += 4) {
      stage<0, -1, -1>(c, kt);
      stage<1, -1, -1>(c, kt + 1);
      stage<2, -1, -1>(c, kt + 2);
      stage<3, -1, -1>(c, kt + 3);
    }
    stage<0, -1, -1>(c, kt);
    stage<1, -1, 0>(c, kt + 1);
    stage<2, -1, 1>(c, kt + 2);
    stage<3, -1, 2>(c, kt + 3);
  }
  template <int RB, int K = 0>
  static SFP8_DEV void write_all(Ctx& c) {
    if constexpr (K < kWrites) {
      row_write<RB, K>(c, row_read<K>(c));
      write_all<RB, K + 1>(c);
    }
  }
  // The last tile's epilogue.  The barrier first: EXACT tiles read row block 1
  // of the tile before from the staging rows in their last stage, which another
  // wave may still be in.
  static SFP8_DEV void tail(Ctx& c) {
    __syncthreads();
    pieces<0, kPieces / 2>(c);
    block_stage<0>(c);
    __syncthreads();
    write_all<0>(c);
    pieces<kPieces / 2, kPieces>(c);
    __syncthreads();
    block_stage<1>(c);
    __syncthreads();
    write_all<1>(c);
  }
};
// the ring, three slots of rstd, the staging rows
constexpr int kBf16PipeRing = Bf16Pipe<8, true>::ML::kLds;
constexpr int kBf16PipeStg = kBf16PipeRing + 3 * kTile * 4;
constexpr int kBf16PipeLds = kBf16PipeStg + 3 * Bf16Pipe<8, true>::kOut;
static_assert(kBf16PipeLds <= 160 * 1024, "fits the LDS");

template <int KE, bool EXACT>
__global__ __launch_bounds__(512, 1) void bf16_swiglu_pipe_kernel(
    const uint16_t* __restrict__ x, const uint8_t* __restrict__ w, int64_t T, int64_t D, int64_t I,
    const float* __restrict__ rstd, uint16_t* __restrict__ gu, uint16_t* __restrict__ h, int tiles_m, int tiles_n,
    const int* __restrict__ plan, int64_t w_estride, int64_t ldxs) {
  using P = Bf16Pipe<KE, EXACT>;
  using ML = typename P::ML;
  extern __shared__ __align__(16) uint8_t lds[];
  typename P::Ctx c;
  c.lds = lds;
  c.stg = lds + kBf16PipeStg;
  c.wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63, wm = c.wave % ML::kWM, wn = c.wave / ML::kWM;
  const int fr = lane & 31, g = lane >> 5;
  const uint32_t chunk = (uint32_t)(((lane & 3) ^ ((lane >> 4) & 3)) << 4);
  const int sw = (fr >> 2) & 3;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    c.aoff[k] = (uint32_t)((64 * wm + fr) * kStage + (((2 * g + k) ^ sw) << 4));
    c.boff[k] = (uint32_t)(ML::kLdsB + (BLayout<true, 2>::kWaveStride * wn + fr) * kStage + (((2 * g + k) ^ sw) << 4));
  }
  const bool xslab = ldxs > 0;
  const int64_t ldx = D * 2, wr = slab_rows(2 * I);
  c.nk = (int)(ldx / kStage);
  c.a_ss = xslab ? (int)(ldxs * kStage) : kStage;
  c.b_ss = (int)(wr * kStage);
  c.ld_gu = (int)(4 * I);
  c.ld_h = (int)(2 * I);
#pragma unroll
  for (int j = 0; j < ML::kDmaA; ++j) {
    const int r = (kTile / ML::kWaves) * c.wave + 16 * j + (lane >> 2);
    c.voff_a[j] = (uint32_t)(r * (xslab ? kStage : (int)ldx)) + chunk;
  }
#pragma unroll
  for (int j = 0; j < ML::kDmaB; ++j) {
    const int r = (128 / ML::kWaves) * c.wave + 16 * j + (lane >> 2);
    c.voff_b[j] = (uint32_t)(((r >> 6) * (int)I + paired_col64(r)) * kStage) + chunk;
  }
  if (plan) tiles_m = MoePlan{plan}.ntiles();
  const int ntiles = tiles_m * tiles_n;
  // tile -> its first row, rows and first column, and its operands
  auto tile_of = [&](int tile, int64_t& r0, int64_t& nrows, int64_t& n0, __amdgpu_buffer_rsrc_t& ra,
                     __amdgpu_buffer_rsrc_t& rb) {
    int tm, tn;
    tile_coords(tile, ntiles, tiles_m, tiles_n, tm, tn);
    r0 = (int64_t)tm * kTile;
    nrows = T - r0;
    const uint8_t* wb = w;
    if (plan) {
      const MoePlan M{plan};
      r0 = M.urow(tm);
      nrows = M.rows(tm);
      wb += M.expert(tm) * w_estride;
    }
    n0 = (int64_t)tn * 64;
    ra = make_rsrc(reinterpret_cast<const uint8_t*>(x) + r0 * (xslab ? kStage : ldx),
                   xslab ? ldx * ldxs - r0 * kStage : nrows * ldx);
    rb = make_rsrc(wb + n0 * kStage, ldx * wr - n0 * kStage);
  };
  // rstd of the 256 rows from r0 into LDS slot `slot` (rows past T read as
  // zero; every wave brings the same 1 KiB, so that its waits count it).  Three
  // slots: while a wave requests the next tile's, another may still read the
  // previous tile's.
  auto load_rstd = [&](int64_t r0, int slot) {
    if (rstd)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(make_rsrc(rstd + r0, (T - r0) * 4),
                                               (lds_ptr_t)(lds + kBf16PipeRing + slot * kTile * 4), 16,
                                               (uint32_t)(lane * 16), 0, 0, 0);
  };
#pragma unroll
  for (int tb = 0; tb < 2; ++tb)
#pragma unroll
    for (int v = 0; v < 16; ++v) c.E[tb][v] = 0u;
  c.rgu = make_rsrc(gu, 0);  // no previous tile: its stores are dropped
  c.rh = make_rsrc(h, 0);
  c.so_g = c.so_u = c.so_h = 0;
  int64_t r0 = 0, nrows = 0, n0 = 0;
  int it = 0;
  if ((int)blockIdx.x < ntiles) {
    tile_of(blockIdx.x, r0, nrows, n0, c.ra, c.rb);
    load_rstd(r0, 0);
#pragma unroll
    for (int s = 0; s < 3; ++s)
      ML::load_stage(lds, s, c.ra, c.rb, c.voff_a, c.voff_b, s * c.a_ss, s * c.b_ss, c.wave);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * ML::kDma) : "memory");
    ML::read_frags(lds, 0, c.aoff, c.boff, c.f[0]);
  }
  for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x, ++it) {
    int64_t nr0 = 0, nnrows = 0, nn0 = 0;
    const bool has_next = tile + (int)gridDim.x < ntiles;
    if (has_next) {
      tile_of(tile + (int)gridDim.x, nr0, nnrows, nn0, c.nra, c.nrb);
      load_rstd(nr0, (it + 1) % 3);
    } else {  // no records: the stages past the last read nothing
      c.nra = make_rsrc(x, 0);
      c.nrb = make_rsrc(w, 0);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) c.acc[i][j] = floatx16{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f,
                                                          0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    P::template stages<0>(c);
    if constexpr (!EXACT) P::rest(c);
    // this tile's g, u times rstd (bf16) become the next epilogue's input; its
    // rstd landed with its first stages, many barriers ago
    const float* rs = reinterpret_cast<const float*>(lds + kBf16PipeRing + (it % 3) * kTile * 4);
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
      const float s = rstd ? rs[64 * wm + 32 * tb + fr] : 1.0f;
#pragma unroll
      for (int v = 0; v < 16; ++v) c.E[tb][v] = pack2_bf16(c.acc[tb][0][v] * s, c.acc[tb][1][v] * s);
    }
    c.rgu = make_rsrc(gu + r0 * 2 * I, nrows * 4 * I);
    c.rh = make_rsrc(h + r0 * I, nrows * 2 * I);
    c.so_g = (int)(n0 * 2);
    c.so_u = (int)((I + n0) * 2);
    c.so_h = (int)(n0 * 2);
    r0 = nr0;
    nrows = nnrows;
    n0 = nn0;
    c.ra = c.nra;
    c.rb = c.nrb;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (it) P::tail(c);
}

// out[u, n] = bf16(sum_k A[m, k] * B[n, k]) with A a bf16 K-slab over lda
// rows (Kb bytes of K) and B a bf16 K-slab [Kb/64][slab_rows(N)][64]: the
// dgrad of the SwiGLU path (_swiglu_dgrad_kernel, train.py:1907-1980, its
// d_gu operand precomputed).  One work-group per 256 x 256 tile; the bf16
// tile is staged in LDS in two passes of 128 rows and written as whole rows.
// With a MoE plan: A in padded expert order, tile row tm writes its rows(tm)
// valid rows to out rows urow(tm).. (expert order); B of expert e at
// b + e * b_estride (bytes).
// 8 waves (two per SIMD), each 128 x 64.
template <class TS>
SFP8_DEV void bf16_gemm_tile(
    uint8_t* lds, int tm, int tn, const uint8_t* __restrict__ a, const uint8_t* __restrict__ b, int64_t T,
    int64_t N, int64_t Kb, int64_t lda, uint16_t* __restrict__ out, const int* __restrict__ plan,
    int64_t b_estride) {
  const int64_t bp = slab_rows(N);
  int64_t u0 = (int64_t)tm * TS::kM, uend = T;  // output rows of this tile
  if (plan) {
    const MoePlan P{plan};
    const int pt = TS::plan_tile(tm);
    if (pt >= P.ntiles()) return;  // work-group uniform
    b += P.expert(pt) * b_estride;
    u0 = P.urow(pt) + TS::plan_skip(tm);
    uend = P.urow(pt) + P.rows(pt);
    if (u0 >= uend) return;  // nothing but padding rows, which have no output
  }
  const int64_t m0 = (int64_t)tm * TS::kM, n0 = (int64_t)tn * TS::kN;
  if (!plan && m0 >= T) return;  // the second half of the last tile, past the last row
  floatx16 acc[TS::kTB][2];
  TS::template Loop<true, 0, 0>::run(
      lds, a + m0 * kStage, Kb * lda - m0 * kStage, [=](int r) { return r * kStage; }, (int)(lda * kStage),
      b + n0 * kStage, Kb * bp - n0 * kStage, [=](int r) { return plain_col_nb<2>(r) * kStage; }, (int)(bp * kStage),
      (int)(Kb / kStage), acc);
  store_bf16_tile<TS>(lds, acc, 1.0f, u0, n0, uend, N, out);
}
template <class TS>
__global__ __launch_bounds__(TS::kThreads, TS::kMinWaves) void bf16_gemm_kernel(
    const uint8_t* __restrict__ a, const uint8_t* __restrict__ b, int64_t T, int64_t N, int64_t Kb, int64_t lda,
    uint16_t* __restrict__ out, int tiles_m, int tiles_n, const int* __restrict__ plan, int64_t b_estride) {
  extern __shared__ __align__(16) uint8_t lds[];
  int tm, tn;
  if constexpr (TS::kTB == 4) {
    bool half;
    if (!tail_tile(plan ? MoePlan{plan}.ntiles() : tiles_m, tiles_n, tm, tn, half)) return;
    if (half) {
      bf16_gemm_tile<Tile<2, 4>>(lds, tm, tn, a, b, T, N, Kb, lda, out, plan, b_estride);
      return;
    }
  } else {
    tile_coords(blockIdx.x, gridDim.x, tiles_m, tiles_n, tm, tn);
  }
  bf16_gemm_tile<TS>(lds, tm, tn, a, b, T, N, Kb, lda, out, plan, b_estride);
}

// The bf16 weight gradient's reduction: out[m, n] = bf16(sum over s
// ascending of ws[s]) (the bf16 result of _swiglu_wgrad_kernel,
// train.py:1983-2026), partials in wgrad_kernel's accumulator order;
// blockIdx.y = expert of a grouped gradient (out [E, M, N]).
template <bool SMALL, bool TR_B>
__global__ __launch_bounds__(256) void bf16_wgrad_reduce_kernel(const float* __restrict__ ws, int splits, int64_t n4,
                                                                int tiles_n, int64_t M, int64_t N,
                                                                uint16_t* __restrict__ out,
                                                                const int* __restrict__ plan, int even) {
  ws += (int64_t)blockIdx.y * splits * n4 * 4;
  if (plan) splits = moe_expert_splits(plan, blockIdx.y, even, splits);  // as splitk_reduce_kernel
  if (splits == 1) return;
  out += (int64_t)blockIdx.y * M * N;
  const floatx4* w4 = reinterpret_cast<const floatx4*>(ws);
  for (int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x; q < n4; q += (int64_t)gridDim.x * 256) {
    floatx4 acc = __builtin_nontemporal_load(w4 + q);
    for (int s = 1; s < splits; ++s) acc += __builtin_nontemporal_load(w4 + (int64_t)s * n4 + q);
    int r, c;
    acc_order_rc<SMALL, TR_B>((int)(q & ((1 << kTileQLog<SMALL>) - 1)), r, c);
    const int64_t tile = q >> kTileQLog<SMALL>;
    const int64_t tm = tile / tiles_n, tn = tile % tiles_n;
    const int64_t m = tm * TileShape<SMALL>::kM + r, n = tn * TileShape<SMALL>::kM + c;
    if (m < M && n < N)  // N % 4 == 0: the 4 values are wholly inside or past the row
      *reinterpret_cast<intx2*>(out + m * N + n) =
          intx2{(int)pack2_bf16(acc[0], acc[1]), (int)pack2_bf16(acc[2], acc[3])};
  }
}

// The weight gradient with the optimizer's momentum stage fused into its
// reduction (the consumer of dW, train.py:2805-2820, applied as the split
// sum leaves the registers): d = (sum over s ascending of ws[s]) / (sa * sb),
// then v <- lerp(v, d, w_v) in place and u = bf16(lerp(d, v, 1 - w_u1)) into
// the Newton-Schulz staging matrix ([M, N] bf16, the parameter's layout);
// grad[m, n] = d when grad is given.  splits == 0: d = 0 (no tokens).  TR_B:
// the partials' columns are in the transposed-read B order, as for
// splitk_reduce_kernel<true>; SMALL: the partials of wgrad_kernel<SMALL, ..>.
template <bool SMALL, bool TR_B>
__global__ __launch_bounds__(256) void splitk_momentum_kernel(const float* __restrict__ ws, int splits, int64_t n4,
                                                              int tiles_n, int64_t M, int64_t N,
                                                              const float* __restrict__ sa,
                                                              const float* __restrict__ sb, float* __restrict__ grad,
                                                              float* __restrict__ v, uint16_t* __restrict__ u,
                                                              float w_v, float w_u1) {
  // Work-group b sums the b-th 256 float4s of every split: a 32 x 32 block of
  // dW (fixed tile, wave, row block tb, column block nb), passed through LDS
  // so that eight lanes then cover 32 contiguous columns of one row of v, u
  // and grad (n4 is a multiple of 256: no partial work-group).
  __shared__ floatx4 blk[32][9];
  const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const floatx4* w4 = reinterpret_cast<const floatx4*>(ws);
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < splits; ++s) acc += __builtin_nontemporal_load(w4 + (int64_t)s * n4 + q);
  using TS = TileShape<SMALL>;
  constexpr int TBB = SMALL ? 1 : 2;  // bits of tb
  const int lane = threadIdx.x & 63, i = threadIdx.x >> 6;
  const int64_t b = blockIdx.x;
  const int nb = (int)(b & 1), tb = (int)(b >> 1) & (TS::kTB - 1);
  const int wave = (int)(b >> (1 + TBB)) & (TS::kThreads / 64 - 1);
  const int64_t tile = b >> (kTileQLog<SMALL> - 8);
  const int64_t tm = tile / tiles_n, tn = tile % tiles_n;
  // local column (0..31) of this thread's float4 in the block
  const int c = TR_B ? 8 * i + 4 * (lane >> 5) : 16 * (lane >> 5) + 4 * i;
  blk[lane & 31][c >> 2] = acc * (1.0f / (sa[0] * sb[0]));
  __syncthreads();
  const int r = threadIdx.x >> 3, c2 = 4 * (threadIdx.x & 7);
  const int64_t m = tm * TS::kM + 32 * TS::kTB * (wave & 1) + 32 * tb + r;
  // local column -> output column: TR_B blocks are 32 contiguous columns,
  // the plain layout's two 16-column halves lie 32 columns apart
  const int64_t n =
      tn * TS::kM + 64 * (wave >> 1) + (TR_B ? 32 * nb + c2 : 16 * nb + (c2 < 16 ? c2 : 16 + c2));
  if (m >= M || n >= N) return;
  const floatx4 d = blk[r][c2 >> 2];
  if (grad) *reinterpret_cast<floatx4*>(grad + m * N + n) = d;
  floatx4 vv = *reinterpret_cast<const floatx4*>(v + m * N + n);
  uint32_t uu[2];
  momentum4(d, vv, w_v, w_u1, uu);
  *reinterpret_cast<floatx4*>(v + m * N + n) = vv;
  *reinterpret_cast<intx2*>(u + m * N + n) = intx2{(int)uu[0], (int)uu[1]};
}

}  // namespace sfp8

static_assert(3 * sfp8::kTile * sfp8::kEpiStride<false> + 64 <= sfp8::kMainLds &&
                  3 * 128 * sfp8::kEpiStride<true> + 64 <= sfp8::TileShape<true>::kLds, "swiglu epilogue tiles fit the main loop's LDS");
static_assert(sfp8::kPipeLds <= 160 * 1024, "deferred-epilogue SwiGLU fits the 160 KiB LDS");
static_assert(128 * sfp8::kBf16Stride <= sfp8::kMainLds, "bf16 epilogue staging fits the main loop's LDS");
static_assert(3 * 128 * sfp8::kGuStride<false> <= sfp8::kMainLds &&
                  3 * 128 * sfp8::kGuStride<true> <= sfp8::TileShape<true>::kLds, "bf16 SwiGLU staging fits the main loop's LDS");

// ============================================================================
// C ABI
// ============================================================================
using namespace sfp8;

namespace {

// epilogue tiles (2 x 256 x 272) + 4 amax floats, or the main loop's ring
constexpr int kDgradEpiLds = 2 * kTile * kEpiStride2 + 32;
constexpr int kDgradLds = kDgradLutBytes + (kDgradEpiLds > kMainLds ? kDgradEpiLds : kMainLds);

template <typename K>
int prep(K kernel, int lds_bytes) {
  // dynamic LDS above 64 KiB must be opted into once per kernel
  const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           lds_bytes);
  return e == hipSuccess ? kOk : (int)e;
}

inline int status() {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? kOk : (int)e;
}

inline bool al16(const void* p) { return (((uintptr_t)p) & 15u) == 0; }
inline int cdiv(int64_t a, int64_t b) { return (int)((a + b - 1) / b); }

// Compute units of the current device (queried on every call: no cached state).
inline int cu_count(int* n) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(n, hipDeviceAttributeMultiprocessorCount, dev);
  if (e != hipSuccess) return (int)e;
  if (*n <= 0) *n = 1;
  return 0;
}
// offsets inside one operand tile are 32-bit
inline bool fits32(int64_t rows, int64_t ld) { return rows * ld < (int64_t)1 << 31; }

// Work-groups launched for a split-K weight gradient of `tiles` tiles: when
// padding the grid to whole 32-tile runs per XCD (256 work-groups a round)
// adds no round of work-groups, it is padded, so that every round of an XCD
// runs 32 consecutive tiles of one split (one raster group of 8 tile rows x
// 4 tile columns at 4 tile columns); the padding work-groups exit at once.
inline int wgrad_grid(int tiles, int splits) {
  const int n = tiles * splits, padded = (n + 255) / 256 * 256;
  return splits > 1 && (tiles % 32) == 0 ? padded : n;
}

// K bytes per weight-gradient split: ldt / s rounded up to whole 128-byte
// stage pairs (the last split takes what remains).
inline int64_t wgrad_chunk(int64_t ldt, int64_t s) {
  const int64_t per = (ldt + s - 1) / s;
  return (per + 2 * kStage - 1) / (2 * kStage) * (2 * kStage);
}

}  // namespace

namespace {
constexpr int64_t kCUs = 256;

// Whether an M x N output (of each of `parts` K splits times experts) is
// computed in 128 x 128 tiles (two work-groups per CU) instead of 256 x 256
// ones (one per CU): when the larger tiles would leave half of the 256 CUs or
// more without one.  A CU runs its tile at the same speed however many others
// are idle, so the quarter tiles, spread over up to four times the CUs, win
// until they fill the chip; from then on their K loop, with twice the LDS-DMA
// bytes per FLOP, is the slower one.  Measured (us, 256 -> 128 tiles): weight
// gradient with its reduction 25 -> 15 at 16 work-groups of 256 x 256, 26 ->
// 17 at 32, 27 -> 25 at 96, 55 -> 52 at 192 but 40 -> 43 at another 192; down
// dgrad 27 -> 13 at 48 tiles, 17 -> 13 at 128, 39 -> 44 at 240; FP8 SwiGLU
// forward 11 -> 6 at 32, 12 -> 9 at 128, 15 -> 15 at 256.
// second: also when the larger tiles would take a second round of 1 to
// `second` of them, for the kernels whose epilogue is a large part of a tile,
// which the second work-group of a CU then overlaps: with 128, FP8 SwiGLU
// forward 32 -> 26 at 272 tiles and 28 -> 26 at 384, bf16 one 49 -> 41 and
// 42 -> 39, down dgrad 46 -> 41 and 68 -> 66 at 384.
inline bool use_small_tiles(int64_t M, int64_t N, int64_t parts, int second) {
  const int64_t tiles = (int64_t)cdiv(M, kTile) * cdiv(N, kTile) * parts;
  return tiles <= kCUs / 2 || (tiles > kCUs && tiles <= kCUs + second);
}

// A GEMM's tile shape Tile<tb, wn> over an M x N output (of each of `parts` K
// splits times experts), and its launch.
struct Tiling {
  bool small;  // Tile<2, 2>; else of 256 columns
  int tb;
  int m, n, lds;  // tile rows and columns, dynamic LDS
  dim3 grid, block;
};
template <int TB, int WN>
Tiling tiling_of(int64_t M, int64_t N, int64_t parts = 1) {
  using TS = Tile<TB, WN>;
  Tiling t;
  t.small = WN == 2;
  t.tb = TB;
  t.m = cdiv(M, TS::kM);
  t.n = cdiv(N, TS::kN);
  t.lds = TS::kLds;
  t.grid = dim3((unsigned)(t.m * t.n * parts));
  t.block = dim3((unsigned)TS::kThreads);
  return t;
}
inline Tiling tiling(int64_t M, int64_t N, int64_t parts = 1, int second = 0) {
  return use_small_tiles(M, N, parts, second) ? tiling_of<2, 2>(M, N, parts) : tiling_of<4, 4>(M, N, parts);
}
// The kernels with bf16 outputs have every shape; K: their K bytes.  By the
// number of 256 x 256 tiles: 128 x 128 ones up to 128; from there on 192 x 256
// ones where their rounds of 256 work-groups cost less (15 units a round
// against 20, or 12 for a last one in halves) and the K loop is long enough to
// outweigh the larger share of prologue and epilogue; else 256 x 256.
// Measured (us, D = 1024, I = 3072, gate/up dgrad and bf16 dgrad, 256 x 256 /
// 192 x 256 / 128 x 128): 16 tiles 48 40 25, 91 75 46; 80 tiles 50 41 37, 93 77
// 71; 192 tiles 63 62 71, 126 120 136; 256 tiles 77 97 89, 150 194 177; with
// the halves 320 tiles 106 108, 234 218; 448 tiles 138 161, 303 334; 544 tiles
// 191 179, 381 367; 640 tiles 210 229, 407 460.  At 24 K stages (down forward,
// I = 1536, 384 tiles) 192 x 256 is no faster.  128 x 256 tiles, one per CU,
// were the faster ones alone at 80 tiles (34 against 37), but the block's step
// was 3 % slower with them.  Grouped rows come in whole tiles of 256, which
// 192-row tiles do not divide.
inline Tiling out_shape(int64_t M, int64_t N, int64_t K, bool grouped) {
  const int64_t tiles = (int64_t)cdiv(M, kTile) * cdiv(N, kTile);
  if (tiles <= kCUs / 2) return tiling_of<2, 2>(M, N);
  const int64_t r = tiles % kCUs, cost = 20 * (tiles / kCUs) + (r == 0 ? 0 : 2 * r <= kCUs ? 12 : 20);
  const int64_t cost192 = 15 * cdiv((int64_t)cdiv(M, 192) * cdiv(N, kTile), kCUs);
  if (!grouped && K >= 48 * kStage && cost192 < cost) return tiling_of<3, 4>(M, N);
  return tiling_of<4, 4>(M, N);
}
// The grid of the 256 x 256 tiles and their halves (tail_tile); grouped: an
// upper bound, the kernel reads the plan's count.
inline Tiling with_tail(Tiling tl, bool grouped) {
  const int n = tl.m * tl.n, r = n % kRound;
  if (!tl.small && tl.tb == 4) tl.grid.x = (unsigned)(grouped ? n + kRound / 2 : 2 * r <= kRound ? n + r : n);
  return tl;
}
inline Tiling out_tiling(int64_t M, int64_t N, int64_t K, bool grouped) {
  return with_tail(out_shape(M, N, K, grouped), grouped);
}
#define OUT_KERNEL(kernel, tl) \
  ((tl).small ? kernel<Tile<2, 2>> : (tl).tb == 3 ? kernel<Tile<3, 4>> : kernel<Tile<4, 4>>)

// The gate/up forward's: a tile covers half as many (gate, up) columns as rows.
inline Tiling swiglu_tiling(int64_t M, int64_t I) {
  return tiling(M, 2 * I, 1, 128);
}

// Whether the gate/up forward runs the persistent kernel: at the widths it is
// built for (4, 8 or 16 K stages), from 640 tiles of 256 x 64 pairs on (2.5 per
// CU).  Its gain is the epilogue of one tile under the K loop of the next, so
// it needs several tiles per CU, and the shorter the K loop the larger the
// epilogue that it hides.  Measured (us, one tile per work-group -> persistent,
// at 256, 512, 768 and 4096 or more tiles): D = 256 9 -> 11, 15 -> 15, 21 ->
// 19, 92 -> 74; D = 512 (384, 640, 768, 4608) 16 -> 17, 23 -> 23, 26 -> 24,
// 149 -> 107; D = 1024 14 -> 15, 23 -> 24, 36 -> 32, 530 -> 423 (640: 31 ->
// 29).  At D = 2048 the longer K loop prefers the 256-column tile's lower
// DMA traffic (1.81 against 1.55 ms at T = 65536).
inline bool use_pipe(int64_t rows, int64_t D, int64_t I) {
  return (D == 256 || D == 512 || D == 1024) && (int64_t)cdiv(rows, kTile) * (I / 64) >= 5 * kCUs / 2;
}

// The persistent gate/up forward over `rows` token rows (with a plan an upper
// bound: the kernel reads the plan's count), one work-group per CU.
int pipe_launch(const void* x8, const void* w8, int64_t T, int64_t rows, int64_t D, int64_t I, const float* scale,
                const float* wscale, float* amax, void* gu8, void* h8, void* h8t, int64_t ldt, const int* plan,
                int64_t w_estride, hipStream_t st) {
  const auto kern = D == 1024  ? swiglu_pipe_kernel<16, kPipeTB>
                    : D == 512 ? swiglu_pipe_kernel<8, kPipeTB>
                               : swiglu_pipe_kernel<4, kPipeTB>;
  const int tiles_m = cdiv(rows, kTile), tiles_n = (int)(I / 64);
  const int ntiles = tiles_m * tiles_n;
  int n_cu = 0;
  int rc = cu_count(&n_cu);
  if (rc) return rc;
  rc = prep(kern, kPipeLds);
  if (rc) return rc;
  hipLaunchKernelGGL(kern, dim3(ntiles < n_cu ? ntiles : n_cu), dim3(kPipeThreads), kPipeLds, st, (const uint8_t*)x8,
                     (const uint8_t*)w8, T, D, I, scale, wscale, amax, (uint8_t*)gu8, (uint8_t*)h8, (uint8_t*)h8t,
                     ldt, tiles_m, tiles_n, plan, w_estride);
  return status();
}

// The persistent down dgrad over `rows` token rows, the padding that its
// K-slab output needs among them (with a plan an upper bound: the kernel reads
// the plan's count), T rows of dy.
int dgrad_launch(const void* dy, const void* wdt, const void* gu8, int64_t rows, int64_t T, int64_t D, int64_t I,
                 const float* scale, float* amax, void* dgu8, void* dgu8t, int64_t ldt, const int* plan,
                 int64_t w_estride, hipStream_t st) {
  const Tiling tl = dgu8t ? tiling_of<4, 4>(rows, I) : tiling(rows, I, 1, 128);
  const auto kern = dgu8t ? down_dgrad_swiglu_kernel<true, false>
                          : (tl.small ? down_dgrad_swiglu_kernel<false, true> : down_dgrad_swiglu_kernel<false, false>);
  int n_cu = 0;
  int rc = cu_count(&n_cu);
  if (rc) return rc;
  const int lds = tl.small ? kDgradLutBytes + TileShape<true>::kLds : kDgradLds;
  rc = prep(kern, lds);
  if (rc) return rc;
  const unsigned wgs = (unsigned)(tl.small ? 2 * n_cu : n_cu);  // resident at once
  hipLaunchKernelGGL(kern, dim3(tl.grid.x < wgs ? tl.grid.x : wgs), tl.block, lds, st, (const uint16_t*)dy,
                     (const uint16_t*)wdt, (const uint8_t*)gu8, T, D, I, scale, amax, (uint8_t*)dgu8,
                     (uint8_t*)dgu8t, ldt, tl.m, tl.n, plan, w_estride);
  return status();
}

// wgrad_kernel over one weight gradient's tiles and splits (tl of M x N and
// `splits` parts): `ldt` and `chunk` K bytes in all and per split.
template <bool BF16, int FMT_A, int FMT_B, bool TRA, bool TRB>
int launch_wgrad(const Tiling& tl, const void* a, const void* b, int64_t M, int64_t N, int64_t ldt, int64_t chunk,
                 const float* sa, const float* sb, float* out, int splits, int partials, TrOp tra, TrOp trb,
                 hipStream_t st) {
  const auto kern = tl.small ? wgrad_kernel<true, BF16, FMT_A, FMT_B, TRA, TRB>
                             : wgrad_kernel<false, BF16, FMT_A, FMT_B, TRA, TRB>;
  const int rc = prep(kern, tl.lds);
  if (rc) return rc;
  const dim3 grid = !partials ? with_tail(tl, false).grid
                    : BF16 || tl.small ? tl.grid : dim3((unsigned)wgrad_grid(tl.m * tl.n, splits));
  hipLaunchKernelGGL(kern, grid, tl.block, tl.lds, st, (const uint8_t*)a, (const uint8_t*)b, M, N, ldt, chunk, sa, sb,
                     out, tl.m, tl.n, splits, partials, tra, trb);
  return status();
}

// K splits of each expert of a grouped gradient, and of those with more than
// one and a half times the average rows (moe_expert_splits).
struct MoeSplits {
  int even, longest;
};
// moe_wgrad_kernel over every expert's tiles and splits (tl of M x N and
// E * splits.even parts).
template <bool BF16, int FMT_A, int FMT_B, bool TRA, bool TRB>
int launch_moe_wgrad(const Tiling& tl, const void* a, const void* b, int64_t M, int64_t N, int64_t ldp,
                     const float* sa, const float* sb, float* out, float* ws, const int* plan, MoeSplits splits,
                     hipStream_t st) {
  const auto kern = tl.small ? moe_wgrad_kernel<true, BF16, FMT_A, FMT_B, TRA, TRB>
                             : moe_wgrad_kernel<false, BF16, FMT_A, FMT_B, TRA, TRB>;
  const int rc = prep(kern, tl.lds);
  if (rc) return rc;
  const int n = (int)tl.grid.x, r = n % kRound, n0 = n / splits.even;
  const dim3 grid(splits.longest > splits.even                     ? n0 * splits.longest
                  : !tl.small && splits.even == 1 && 2 * r <= kRound ? n + r
                                                                     : n);
  hipLaunchKernelGGL(kern, grid, tl.block, tl.lds, st, (const uint8_t*)a, (const uint8_t*)b, M, N, ldp, sa, sb, out, ws,
                     plan, tl.m, tl.n, splits.even, splits.longest, n0 / (tl.m * tl.n));
  return status();
}

// Whether a weight gradient's workspace is missing or smaller than its size
// query says.  The answer does not depend on the splits that the call takes,
// which may be fewer than the query's; a size of 0 needs no pointer.
inline bool no_workspace(const float* ws, int64_t have, int64_t floats) {
  return floats > 0 && (!ws || have < floats);
}

// float4s of one split's partials, and the launches of the reductions over
// them (E experts; tr_b: the partials of a transposed-read B; plan: the
// experts' counts are `even` or `splits`, moe_expert_splits).
inline int64_t partial_quads(const Tiling& tl) { return (int64_t)tl.m * tl.n << (tl.small ? 12 : 14); }
inline dim3 reduce_grid(const Tiling& tl, int64_t E, bool few = false) {
  // few: most experts have nothing to add, and work-groups that exit at once
  // cost a launch's time too (16 experts, M = 2944, N = 896: 49152 of them 10 us,
  // 6144 none); down to 512 an expert, which the others still need
  const int64_t n = (partial_quads(tl) + 255) / 256;
  return dim3((unsigned)(few && n > 512 ? (n > 4096 ? n / 8 : 512) : n), (unsigned)E);
}
int launch_reduce(const Tiling& tl, bool tr_b, const float* ws, int splits, int64_t E, int64_t M, int64_t N,
                  const float* sa, const float* sb, float* out, hipStream_t st, const int* plan = nullptr, int even = 0) {
  const auto kern = tl.small ? (tr_b ? splitk_reduce_kernel<true, true> : splitk_reduce_kernel<true, false>)
                             : (tr_b ? splitk_reduce_kernel<false, true> : splitk_reduce_kernel<false, false>);
  hipLaunchKernelGGL(kern, reduce_grid(tl, E, plan && even == 1), dim3(256), 0, st, ws, splits, partial_quads(tl), tl.n, M, N, sa, sb,
                     out, plan, even);
  return status();
}
int launch_bf16_reduce(const Tiling& tl, bool tr_b, const float* ws, int splits, int64_t E, int64_t M, int64_t N,
                       void* out, hipStream_t st, const int* plan = nullptr, int even = 0) {
  const auto kern = tl.small
                        ? (tr_b ? bf16_wgrad_reduce_kernel<true, true> : bf16_wgrad_reduce_kernel<true, false>)
                        : (tr_b ? bf16_wgrad_reduce_kernel<false, true> : bf16_wgrad_reduce_kernel<false, false>);
  hipLaunchKernelGGL(kern, reduce_grid(tl, E, plan && even == 1), dim3(256), 0, st, ws, splits, partial_quads(tl), tl.n, M, N,
                     (uint16_t*)out, plan, even);
  return status();
}

// The split partials ws[split][tile] (one fp32 tile each, in accumulator
// order) of the FP8 weight gradient; a_rows / b_rows: that operand is the row
// K-slab of the token-major activation instead of a token-contiguous copy.
// partials 0: one split, whose gradient goes to `out`.
int wgrad_partials(const Tiling& tl, bool a_rows, bool b_rows, const void* a, const void* b, int64_t M, int64_t N,
                   int64_t ldt, const float* sa, const float* sb, float* out, int splits, int partials,
                   hipStream_t st) {
  // row K-slabs over ldt tokens
  const TrOp tra{kStage, ldt * kStage, (M / 64) * ldt * kStage}, trb{kStage, ldt * kStage, (N / 64) * ldt * kStage};
  const auto launch = a_rows ? (b_rows ? launch_wgrad<false, kFmtE5M2, kFmtE4M3, true, true>
                                       : launch_wgrad<false, kFmtE5M2, kFmtE4M3, true, false>)
                             : (b_rows ? launch_wgrad<false, kFmtE5M2, kFmtE4M3, false, true>
                                       : launch_wgrad<false, kFmtE5M2, kFmtE4M3, false, false>);
  return launch(tl, a, b, M, N, ldt, wgrad_chunk(ldt, splits), sa, sb, out, splits, partials, tra, trb, st);
}
}  // namespace

extern "C" {

int sfp8_gemm_gateup_swiglu_fwd(const void* x8, const void* w8, int64_t T, int64_t D, int64_t I,
                                const float* scale, const float* wscale, float* amax, void* gu8, void* h8,
                                void* h8t, int64_t ldt, void* stream) {
  // token-sized buffers may be null when there are no tokens
  if (!w8 || !scale || !wscale || !amax || (T > 0 && (!x8 || !gu8 || !h8))) return kErrNullPointer;
  // the grid covers ceil(T / 256) token tiles, which write every padding
  // token of the outputs only when ldt is T rounded up to 256
  if (T < 0 || D <= 0 || I <= 0 || D % (2 * kStage) || I % 128 || ldt != (int64_t)cdiv(T, kTile) * kTile)
    return kErrBadShape;
  if (!fits32(ldt, D) || !fits32(2 * I, D) || !fits32(ldt, I) || !fits32(ldt, 2 * I)) return kErrBadShape;
  if (!al16(x8) || !al16(w8) || !al16(gu8) || !al16(h8) || !al16(h8t)) return kErrBadAlignment;
  if (T == 0) return kOk;
  if (use_pipe(ldt, D, I))
    return pipe_launch(x8, w8, T, ldt, D, I, scale, wscale, amax, gu8, h8, h8t, ldt, nullptr, 0, (hipStream_t)stream);
  const Tiling tl = swiglu_tiling(ldt, I);  // the padding rows' zeros too
  const auto kern = tl.small ? swiglu_fwd_kernel<true> : swiglu_fwd_kernel<false>;
  const int rc = prep(kern, tl.lds);
  if (rc) return rc;
  hipLaunchKernelGGL(kern, tl.grid, tl.block, tl.lds, (hipStream_t)stream,
                     (const uint8_t*)x8, (const uint8_t*)w8, T, D, I, scale, wscale, amax, (uint8_t*)gu8,
                     (uint8_t*)h8, (uint8_t*)h8t, ldt, tl.m, tl.n, (const int*)nullptr, (int64_t)0);
  return status();
}

int sfp8_gemm_down_fwd(const void* h8, const void* wd8, const void* res, int64_t T, int64_t D, int64_t I,
                       const float* scale, const float* wscale, void* y, int64_t ldt, void* stream) {
  if (!wd8 || !scale || !wscale || (T > 0 && (!h8 || !res || !y))) return kErrNullPointer;
  if (T < 0 || D <= 0 || I <= 0 || I % (2 * kStage) || D % 16 || ldt < T || ldt % kTile) return kErrBadShape;
  if (!fits32(ldt, I) || !fits32(slab_rows(D), I) || !fits32(kTile, 2 * D)) return kErrBadShape;
  if (!al16(h8) || !al16(wd8) || !al16(res) || !al16(y)) return kErrBadAlignment;
  if (T == 0) return kOk;
  const Tiling tl = out_tiling(T, D, I, false);
  const auto kern = OUT_KERNEL(down_fwd_kernel, tl);
  const int rc = prep(kern, tl.lds);
  if (rc) return rc;
  hipLaunchKernelGGL(kern, tl.grid, tl.block, tl.lds, (hipStream_t)stream,
                     (const uint8_t*)h8, (const uint8_t*)wd8, (const uint16_t*)res, T, D, I, scale, wscale + 1,
                     (uint16_t*)y, ldt, tl.m, tl.n, (const int*)nullptr, (int64_t)0);
  return status();
}

int sfp8_gemm_down_dgrad_swiglu(const void* dy, const void* wdt, const void* gu8, int64_t T, int64_t D,
                                int64_t I, const float* scale, float* amax, void* dgu8, void* dgu8t,
                                int64_t ldt, void* stream) {
  if (!wdt || !scale || !amax || (T > 0 && (!dy || !gu8 || !dgu8))) return kErrNullPointer;
  if (T < 0 || D <= 0 || I <= 0 || (2 * D) % (2 * kStage) || I % 128 || ldt != (int64_t)cdiv(T, kTile) * kTile)
    return kErrBadShape;  // ldt = T rounded up to 256: the grid writes every padding token
  if (!fits32(kTile, 2 * D) || !fits32(slab_rows(I), 2 * D) || !fits32(ldt, 2 * I)) return kErrBadShape;
  if (!al16(dy) || !al16(wdt) || !al16(gu8) || !al16(dgu8) || !al16(dgu8t)) return kErrBadAlignment;
  if (T == 0) return kOk;
  return dgrad_launch(dy, wdt, gu8, ldt, T, D, I, scale, amax, dgu8, dgu8t, ldt, nullptr, 0, (hipStream_t)stream);
}

int sfp8_gemm_gateup_dgrad(const void* dgu8, const void* w8t, int64_t T, int64_t D, int64_t I,
                           const float* scale, const float* wscale, void* dxn, int64_t ldt, void* stream) {
  if (!w8t || !scale || !wscale || (T > 0 && (!dgu8 || !dxn))) return kErrNullPointer;
  if (T < 0 || D <= 0 || I <= 0 || (2 * I) % (2 * kStage) || D % 16 || ldt < T || ldt % kTile) return kErrBadShape;
  if (!fits32(ldt, 2 * I) || !fits32(slab_rows(D), 2 * I) || !fits32(kTile, 2 * D)) return kErrBadShape;
  if (!al16(dgu8) || !al16(w8t) || !al16(dxn)) return kErrBadAlignment;
  if (T == 0) return kOk;
  const Tiling tl = out_tiling(T, D, 2 * I, false);
  const auto kern = OUT_KERNEL(gateup_dgrad_kernel, tl);
  const int rc = prep(kern, tl.lds);
  if (rc) return rc;
  hipLaunchKernelGGL(kern, tl.grid, tl.block, tl.lds, (hipStream_t)stream,
                     (const uint8_t*)dgu8, (const uint8_t*)w8t, T, D, I, scale, wscale, (uint16_t*)dxn, ldt,
                     tl.m, tl.n, (const int*)nullptr, (int64_t)0);
  return status();
}

// Number of K splits the library uses for an (M, N, ldt) weight gradient and
// the workspace (floats) it needs: splits * M * N when splits > 1, else 0.
// Split sp covers K [sp * c, min((sp + 1) * c, ldt)) with c = wgrad_chunk:
// ldt / s rounded up to whole 128-token (128-byte) stage pairs, so the last
// split may be shorter.  s is usable when every split has at least 2048
// tokens' worth of chunk and the last split is not empty.
static bool wgrad_split_ok(int64_t s, int64_t ldt) {
  if (s == 1) return true;
  const int64_t c = wgrad_chunk(ldt, s);
  return c >= 2048 && ldt - (s - 1) * c > 0;
}

static int64_t wgrad_splits(int64_t M, int64_t N, int64_t kbytes) {
  // The count (any, not only a power of two) that minimises the modelled
  // time: the rounds of work-groups the 256 CUs run, times the longest
  // split's 64-byte K stages, plus the split partials' traffic (4 bytes
  // written and read per output and split, at about 5 TB/s: M * N * 8 /
  // 3.5e6 stage times of 0.7 us).  At T = 65536 this gives 5 splits for both
  // the down gradient (48 tiles: 240 work-groups in one round, where 4
  // splits leave 64 CUs idle) and the gate/up one (96 tiles: 480 work-groups
  // in two rounds, against three rounds of 256 with 8).  Ties go to fewer
  // splits.  A bf16 stage holds half the tokens in the same bytes and takes as
  // long: at T = 49152, M = 3072, N = 512 (24 tiles) it gives 10 splits in one
  // round, 150 us with the reduction against 186 for 16 (a round and a half).
  const int64_t tiles = (int64_t)cdiv(M, kTile) * cdiv(N, kTile);
  const double part = (double)M * (double)N * 8.0 / 3.5e6;
  int64_t best = 1;
  double best_cost = 0.0;
  for (int64_t s = 1; s <= 64 && tiles * s <= 2048; ++s) {
    if (!wgrad_split_ok(s, kbytes)) continue;
    const double stages = (double)wgrad_chunk(kbytes, s) / kStage;
    const double cost = (double)((tiles * s + kCUs - 1) / kCUs) * stages + (s > 1 ? s * part : 0.0);
    if (s == 1 || cost < best_cost - 1e-9) {
      best = s;
      best_cost = cost;
    }
  }
  return best;
}

// The modelled time (us) of `parts` M x N gradients (the experts') over
// `stages` 64-byte K stages each, in s splits.  A stage of a 256 x 256 tile
// takes 0.4 us, and up to 0.35 more the fuller the rounds are (the clock
// falls); one of a 128 x 128 tile 0.3 us alone on its CU and 0.4 (bf16: 0.48)
// beside another.  With one split the gradient is written by its own
// work-group; several write and read 8 bytes per output each, at about 5
// TB/s, and launch the reduction.  Measured against it (us, gradient and
// reduction, 1 / 2 / 4 splits of even rows; the model's choice is marked): 8 experts, M =
// 3072, N = 1024, 131072 rows 332* 362 410, 16384 rows 57* 124 181; M = 1536, N
// = 512, 65536 rows fp8 52* 59 75, bf16 130 107* 128; 4 experts, M = 1024, N =
// 512, 16384 rows bf16 38 31* 32; 16 experts, M = 512, N = 256 10* 19 25.
static inline double wgrad_us(int64_t M, int64_t N, int64_t parts, double stages, int64_t s, bool bf16) {
  const Tiling tl = tiling(M, N, parts * s);
  const int64_t n = (int64_t)tl.m * tl.n * parts * s;
  const int64_t rounds = cdiv(n, tl.small ? 2 * kCUs : kCUs);
  const double us = !tl.small ? 0.4 + 0.35 * (double)n / (double)(rounds * kCUs) : n <= kCUs ? 0.3 : bf16 ? 0.48 : 0.4;
  const int64_t r = n % kCUs;  // one split's last round in halves costs 0.6
  const double cost = !tl.small && s == 1 && r > 0 && 2 * r <= kCUs ? (double)rounds - 0.4 : (double)rounds;
  return cost * us * stages / (double)s +
         (s > 1 ? 2.5 + (double)s * (double)parts * (double)M * (double)N * 8.0 / 5e6 : 0.0);
}
// The K splits that a dense call takes: those of wgrad_splits, which counts
// rounds of 256 x 256 tiles only and sizes the workspace, or one or two splits
// where this model, which knows the smaller tiles, gains a twentieth or so
// (counts between, taken at 24 tiles and 49152 tokens, were no slower alone but
// made the block's step 4 % slower).  Measured (us, gradient and reduction):
// gate/up, D = 1024, I = 3072, 5003 tokens 51 -> 36 (2 -> 1 splits), 8192 67 ->
// 52, 16384 109 -> 100; D = 2048, I = 6144, 16384 tokens 355 -> 329; bf16, D =
// 1024, I = 3072, 16384 tokens 200 -> 182 (5 -> 2); within 3 % of each other
// where the model is near even.
static int64_t dense_splits(int64_t M, int64_t N, int64_t kbytes, bool bf16) {
  const int64_t most = wgrad_splits(M, N, kbytes);
  const double stages = (double)kbytes / (double)kStage;
  int64_t best = most;
  double best_us = 0.96 * wgrad_us(M, N, 1, stages, most, bf16);
  for (int64_t s = 1; s <= 2 && s < most; ++s) {
    if (!wgrad_split_ok(s, kbytes)) continue;
    const double us = wgrad_us(M, N, 1, stages, s, bf16);
    if (us < best_us) {
      best = s;
      best_us = us;
    }
  }
  return best;
}

int64_t sfp8_wgrad_splits(int64_t M, int64_t N, int64_t ldt) { return wgrad_splits(M, N, ldt); }

int64_t sfp8_slab_bytes(int64_t rows, int64_t k) {
  if (rows < 0 || k < 0 || k % kStage) return -1;
  return slab_rows(rows) * k;
}

int64_t sfp8_wgrad_workspace_floats(int64_t M, int64_t N, int64_t ldt) {
  // one 256 x 256 fp32 tile per (split, tile)
  const int64_t s = sfp8_wgrad_splits(M, N, ldt);
  return s > 1 ? s * (int64_t)cdiv(M, kTile) * cdiv(N, kTile) * kTile * kTile : 0;
}



int sfp8_gemm_wgrad(const void* at, int fmt_a, const void* bt, int fmt_b, int64_t M, int64_t N, int64_t ldt,
                    const float* sa, const float* sb, float* out, float* ws, int64_t ws_floats, void* stream) {
  if (!sa || !sb || !out || (ldt > 0 && (!at || !bt))) return kErrNullPointer;
  if (M <= 0 || N <= 0 || ldt < 0 || ldt % kTile || N % 4) return kErrBadShape;
  if (fmt_a != kFmtE5M2 || fmt_b != kFmtE4M3) return kErrBadShape;
  // every K-slab offset (stage * rows * 64 + row * 64) is 32-bit
  if (!fits32(slab_rows(M), ldt) || !fits32(slab_rows(N), ldt)) return kErrBadShape;
  if (!al16(at) || !al16(bt) || !al16(out)) return kErrBadAlignment;
  hipStream_t st = (hipStream_t)stream;
  const int64_t splits = dense_splits(M, N, ldt, false);
  if (no_workspace(ws, ws_floats, sfp8_wgrad_workspace_floats(M, N, ldt))) return kErrWorkspaceTooSmall;
  if (ldt == 0) {
    // no tokens: the gradient is zero (a fill kernel, not a memset node, so
    // that a captured graph replays it correctly)
    const int64_t n = M * N;
    hipLaunchKernelGGL(zero_fill_kernel, dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, st, out, n);
    return status();
  }
  const Tiling tl = tiling(M, N, splits);
  const int rc = launch_wgrad<false, kFmtE5M2, kFmtE4M3, false, false>(
      tl, at, bt, M, N, ldt, wgrad_chunk(ldt, splits), sa, sb, splits > 1 ? ws : out, (int)splits, (int)(splits > 1),
      TrOp{}, TrOp{}, st);
  if (rc || splits == 1) return rc;
  return launch_reduce(tl, false, ws, (int)splits, 1, M, N, sa, sb, out, st);
}

// ---- grouped (MoE expert) GEMMs over padded expert order (common.h) ----
// ldp = padded rows (256 * sfp8_moe_padded_rows); plan from sfp8_moe_plan.
namespace {
// Most K splits of a grouped gradient, by which its workspace is sized before
// its rows are known: at least 2, then doubling until the grid has 384
// work-groups (8 at most).
inline int64_t moe_splits_most(int64_t M, int64_t N, int64_t E) {
  const int64_t wgs = (int64_t)cdiv(M, kTile) * cdiv(N, kTile) * E;
  int64_t s = 2;
  while (s < 8 && wgs * s < 384) s *= 2;
  return s;
}
// The modelled time (us) of a grouped gradient whose rows all went to one
// expert: `stages` K stages in `longest` splits, with the tiles of E * even
// parts.  With one count for all, its work-groups are one run of the grid's, so
// they share the XCDs of that run (32 CUs each) and the others idle; with a
// count of its own each split has such a run to itself.  A stage takes 0.5 us
// for a 256 x 256 tile on a full XCD; 0.27 for a 128 x 128 one alone on its CU
// and 0.4 (bf16: 0.42) beside another.
static inline double one_expert_us(int64_t M, int64_t N, int64_t E, double stages, MoeSplits c, bool bf16) {
  const Tiling tl = tiling(M, N, E * c.even);
  const bool own = c.longest > c.even;
  const int64_t w = (int64_t)tl.m * tl.n * (own ? 1 : c.even), n = w * E, r = n % kCUs;
  const int64_t full = !own && !tl.small && c.even == 1 && r < n && 2 * r <= kCUs ? n - r : n;  // as tail_full
  const int64_t wgs = own ? w * c.longest : w, xcds = (8 * w + full - 1) / full * (own ? c.longest : 1);
  const int64_t cus = 32 * (xcds < 8 ? xcds : 8), slots = tl.small ? 2 * cus : cus, rounds = (wgs + slots - 1) / slots;
  const double fill = wgs <= cus ? 0.0 : wgs >= 2 * cus ? 1.0 : (double)(wgs - cus) / (double)cus;
  const double us = !tl.small ? 0.5 : 0.27 + (bf16 ? 0.15 : 0.13) * fill;
  return (double)rounds * us * stages / (double)c.longest +
         (c.longest > 1 ? 2.5 + (double)c.longest * (double)(own ? 1 : E) * (double)M * (double)N * 8.0 / 5e6 : 0.0);
}
// Its K splits (1, 2, 4 or 8) over ldp padded rows.  The routing is known on
// the device only, so they have to do for all of them: the count that is fastest
// over even rows (more only where that gains a tenth), if it is no slower than
// the most when one expert has every row; else the faster over even rows of two
// ways to make it so, a larger count for all or one for the long experts only
// (the fewest splits that do), which costs the reduction's launch.  Measured
// (us, even rows / half on one expert / all on one; one split for all -> 1 and 2
// to 4 for long ones): 16 experts, M = 512, N = 256, 16384 rows bf16 15/65/123
// -> 17/28/40; M = 2944, N = 896, 68546 rows fp8 170/541/998 -> 173/374/542; 4
// experts, M = 2048, N = 1024, 65536 rows fp8 117/181/325 -> 122/170/179.  The
// most splits for all take 35/44/68, 311/630/993 and 142/203/325.
inline MoeSplits moe_wgrad_splits(int64_t M, int64_t N, int64_t E, int64_t ldp, bool bf16) {
  const double per = (bf16 ? 2.0 : 1.0) / (double)kStage;  // stages per row
  const int64_t pad = (int64_t)kTile * (E - 1);            // the other experts' padding
  const double one = (double)(ldp - pad < kTile ? kTile : ldp - pad) * per, even = (double)ldp * per / (double)E;
  const int most = (int)moe_splits_most(M, N, E);
  const double bound = 1.05 * one_expert_us(M, N, E, one, {most, most}, bf16);
  int best = 0, fixed = 0;  // of all counts; of those within the bound
  double best_us = 0.0, fixed_us = 0.0;
  for (int s = 1; s <= most; s *= 2) {
    const double us = wgrad_us(M, N, E, even, s, bf16);
    if (!best || us < 0.9 * best_us) {
      best = s;
      best_us = us;
    }
    if (s < most && one_expert_us(M, N, E, one, {s, s}, bf16) > bound) continue;
    if (!fixed || us < 0.9 * fixed_us) {
      fixed = s;
      fixed_us = us;
    }
  }
  if (fixed == best) return {best, best};
  for (int s = 2 * best; s <= most; s *= 2)
    if (one_expert_us(M, N, E, one, {best, s}, bf16) <= bound)
      return best_us + 3.0 < fixed_us ? MoeSplits{best, s} : MoeSplits{fixed, fixed};
  return {fixed, fixed};
}
// The plan for the reductions when the experts' counts differ.
inline const int* uneven(MoeSplits c, const int* plan) { return c.longest > c.even ? plan : nullptr; }
inline bool moe_shape(int64_t E, int64_t D, int64_t I, int64_t ldp) {
  return E > 0 && D > 0 && I > 0 && D % 128 == 0 && I % 128 == 0 && ldp > 0 && ldp % kTile == 0;
}
}  // namespace

int sfp8_moe_gemm_gateup_swiglu_fwd(const void* x8, const void* w8, int64_t E, int64_t D, int64_t I, const int* plan,
                                    int64_t ldp, const float* scale, const float* q_gu, float* amax, void* gu8,
                                    void* h8, void* h8t, void* stream) {
  if (!x8 || !w8 || !plan || !scale || !q_gu || !amax || !gu8 || !h8) return kErrNullPointer;
  if (!moe_shape(E, D, I, ldp) || !fits32(ldp, D) || !fits32(2 * I, D) || !fits32(ldp, 2 * I)) return kErrBadShape;
  if (!al16(x8) || !al16(w8) || !al16(gu8) || !al16(h8) || !al16(h8t)) return kErrBadAlignment;
  if (use_pipe(ldp, D, I))
    return pipe_launch(x8, w8, ldp, ldp, D, I, scale, q_gu, amax, gu8, h8, h8t, ldp, plan, D * slab_rows(2 * I),
                       (hipStream_t)stream);
  const Tiling tl = swiglu_tiling(ldp, I);
  const auto kern = tl.small ? swiglu_fwd_kernel<true> : swiglu_fwd_kernel<false>;
  const int rc = prep(kern, tl.lds);
  if (rc) return rc;
  hipLaunchKernelGGL(kern, tl.grid, tl.block, tl.lds, (hipStream_t)stream,
                     (const uint8_t*)x8, (const uint8_t*)w8, ldp, D, I, scale, q_gu, amax, (uint8_t*)gu8,
                     (uint8_t*)h8, (uint8_t*)h8t, ldp, tl.m, tl.n, plan, D * slab_rows(2 * I));
  return status();
}

int sfp8_moe_gemm_down_fwd(const void* h8, const void* wd8, int64_t E, int64_t D, int64_t I, const int* plan,
                           int64_t ldp, const float* scale, const float* q_d, void* out, int64_t R, void* stream) {
  if (!h8 || !wd8 || !plan || !scale || !q_d || (R > 0 && !out)) return kErrNullPointer;
  if (!moe_shape(E, D, I, ldp) || R < 0 || !fits32(ldp, I) || !fits32(slab_rows(D), I) || !fits32(kTile, 2 * D))
    return kErrBadShape;
  if (!al16(h8) || !al16(wd8) || !al16(out)) return kErrBadAlignment;
  const Tiling tl = out_tiling(ldp, D, I, true);
  const auto kern = OUT_KERNEL(down_fwd_kernel, tl);
  const int rc = prep(kern, tl.lds);
  if (rc) return rc;
  hipLaunchKernelGGL(kern, tl.grid, tl.block, tl.lds, (hipStream_t)stream,
                     (const uint8_t*)h8, (const uint8_t*)wd8, (const uint16_t*)nullptr, R, D, I, scale, q_d,
                     (uint16_t*)out, ldp, tl.m, tl.n, plan, I * slab_rows(D));
  return status();
}

int sfp8_moe_gemm_down_dgrad_swiglu(const void* dout, const void* wdt, const void* gu8, int64_t E, int64_t D,
                                    int64_t I, int64_t R, const int* plan, int64_t ldp, const float* scale,
                                    float* amax, void* dgu8, void* dgu8t, void* stream) {
  if (!wdt || !gu8 || !plan || !scale || !amax || !dgu8 || (R > 0 && !dout)) return kErrNullPointer;
  if (!moe_shape(E, D, I, ldp) || R < 0) return kErrBadShape;
  if (!fits32(kTile, 2 * D) || !fits32(slab_rows(I), 2 * D) || !fits32(ldp, 2 * I)) return kErrBadShape;
  if (!al16(dout) || !al16(wdt) || !al16(gu8) || !al16(dgu8) || !al16(dgu8t)) return kErrBadAlignment;
  return dgrad_launch(dout, wdt, gu8, ldp, R, D, I, scale, amax, dgu8, dgu8t, ldp, plan, 2 * D * slab_rows(I),
                      (hipStream_t)stream);
}

int sfp8_moe_gemm_gateup_dgrad(const void* dgu8, const void* w8t, int64_t E, int64_t D, int64_t I, const int* plan,
                               int64_t ldp, const float* scale, const float* q_gu, void* dx, int64_t R, void* stream) {
  if (!dgu8 || !w8t || !plan || !scale || !q_gu || (R > 0 && !dx)) return kErrNullPointer;
  if (!moe_shape(E, D, I, ldp) || R < 0 || !fits32(ldp, 2 * I) || !fits32(slab_rows(D), 2 * I) ||
      !fits32(kTile, 2 * D))
    return kErrBadShape;
  if (!al16(dgu8) || !al16(w8t) || !al16(dx)) return kErrBadAlignment;
  const Tiling tl = out_tiling(ldp, D, 2 * I, true);
  const auto kern = OUT_KERNEL(gateup_dgrad_kernel, tl);
  const int rc = prep(kern, tl.lds);
  if (rc) return rc;
  hipLaunchKernelGGL(kern, tl.grid, tl.block, tl.lds, (hipStream_t)stream,
                     (const uint8_t*)dgu8, (const uint8_t*)w8t, R, D, I, scale, q_gu, (uint16_t*)dx, ldp, tl.m,
                     tl.n, plan, 2 * I * slab_rows(D));
  return status();
}

int64_t sfp8_moe_wgrad_splits(int64_t M, int64_t N, int64_t E) { return moe_splits_most(M, N, E); }

int64_t sfp8_wgrad_splits_of(int64_t M, int64_t N, int64_t E, int64_t rows, int bf16, int longest) {
  if (M <= 0 || N <= 0 || E < 0 || rows <= 0 || rows % kTile) return -1;
  if (!E) return dense_splits(M, N, bf16 ? 2 * rows : rows, bf16);
  const MoeSplits s = moe_wgrad_splits(M, N, E, rows, bf16);
  return longest ? s.longest : s.even;
}

int64_t sfp8_moe_wgrad_workspace_floats(int64_t M, int64_t N, int64_t E) {
  const int64_t s = sfp8_moe_wgrad_splits(M, N, E);
  return s > 1 ? E * s * (int64_t)cdiv(M, kTile) * cdiv(N, kTile) * kTile * kTile : 0;
}

int sfp8_moe_gemm_wgrad(const void* at, int fmt_a, const void* bt, int fmt_b, int64_t M, int64_t N, int64_t E,
                        const int* plan, int64_t ldp, const float* sa, const float* sb, float* out, float* ws,
                        int64_t ws_floats, void* stream) {
  if (!at || !bt || !plan || !sa || !sb || !out) return kErrNullPointer;
  if (M <= 0 || N <= 0 || E <= 0 || N % 4 || ldp <= 0 || ldp % kTile) return kErrBadShape;
  if (fmt_a != kFmtE5M2 || fmt_b != kFmtE4M3) return kErrBadShape;
  if (!fits32(slab_rows(M), ldp) || !fits32(slab_rows(N), ldp)) return kErrBadShape;
  if (!al16(at) || !al16(bt) || !al16(out) || !al16(ws)) return kErrBadAlignment;
  const MoeSplits splits = moe_wgrad_splits(M, N, E, ldp, false);
  if (no_workspace(ws, ws_floats, sfp8_moe_wgrad_workspace_floats(M, N, E))) return kErrWorkspaceTooSmall;
  hipStream_t st = (hipStream_t)stream;
  const Tiling tl = tiling(M, N, E * splits.even);
  const int rc = launch_moe_wgrad<false, kFmtE5M2, kFmtE4M3, false, false>(tl, at, bt, M, N, ldp, sa, sb, out, ws,
                                                                           plan, splits, st);
  if (rc || splits.longest == 1) return rc;
  return launch_reduce(tl, false, ws, splits.longest, E, M, N, sa, sb, out, st, uneven(splits, plan), splits.even);
}

// ---- the grouped weight gradient with row K-slab operands ----
int64_t sfp8_moe_wgrad_rows_workspace_floats(int64_t M, int64_t N, int64_t E) {
  return sfp8_moe_wgrad_workspace_floats(M, N, E);
}

int sfp8_moe_gemm_wgrad_rows(const void* a, int fmt_a, int a_rows, const void* b, int fmt_b, int b_rows, int64_t M,
                             int64_t N, int64_t E, const int* plan, int64_t ldp, const float* sa, const float* sb,
                             float* out, float* ws, int64_t ws_floats, void* stream) {
  if (!a || !b || !plan || !sa || !sb || !out || !ws) return kErrNullPointer;
  if (M <= 0 || N <= 0 || E <= 0 || N % 4 || ldp <= 0 || ldp % kTile || !(a_rows || b_rows)) return kErrBadShape;
  if ((a_rows && M % 64) || (b_rows && N % 64)) return kErrBadShape;
  if (fmt_a != kFmtE5M2 || fmt_b != kFmtE4M3) return kErrBadShape;
  if (!fits32(slab_rows(M), ldp) || !fits32(slab_rows(N), ldp)) return kErrBadShape;
  if (!al16(a) || !al16(b) || !al16(out) || !al16(ws)) return kErrBadAlignment;
  const MoeSplits splits = moe_wgrad_splits(M, N, E, ldp, false);
  if (ws_floats < sfp8_moe_wgrad_rows_workspace_floats(M, N, E)) return kErrWorkspaceTooSmall;
  hipStream_t st = (hipStream_t)stream;
  const Tiling tl = tiling(M, N, E * splits.even);
  const auto launch = a_rows ? (b_rows ? launch_moe_wgrad<false, kFmtE5M2, kFmtE4M3, true, true>
                                       : launch_moe_wgrad<false, kFmtE5M2, kFmtE4M3, true, false>)
                             : launch_moe_wgrad<false, kFmtE5M2, kFmtE4M3, false, true>;
  const int rc = launch(tl, a, b, M, N, ldp, sa, sb, out, ws, plan, splits, st);
  if (rc || splits.longest == 1) return rc;
  return launch_reduce(tl, b_rows, ws, splits.longest, E, M, N, sa, sb, out, st, uneven(splits, plan), splits.even);
}


// ---- bf16 SwiGLU path (the default, non-FP8 path) ----
namespace {
// (a tile's gu rows, 256 x 2I bf16, are addressed with 32-bit offsets)
inline bool bf16_shape(int64_t D, int64_t I) {
  return D > 0 && I > 0 && D % 64 == 0 && I % 64 == 0 && fits32(kTile, 4 * I);
}

// Whether the bf16 gate/up forward runs the persistent kernel: from 640 tiles
// of 64 column pairs on (2.5 per CU) and up to the width where its K loop,
// which reads a third more LDS per FLOP than 256 x 256 tiles, loses more than
// the hidden epilogue gains.  Measured (us, one tile per work-group ->
// persistent, reading the row K-slab): D = 256 39 -> 33 at 1024 tiles (21 ->
// 21 at 512), 155 -> 128 at 4096; D = 512 40 -> 35 at 768, 225 -> 190 at 4608;
// D = 640 98 -> 82 at 1728; D = 768 42 -> 41 at 544, 362 -> 337 at 6144; D =
// 1024 201 -> 225 at 3072.  Reading row-major rows (half lines per K stage):
// D = 640 99 -> 86, D = 768 117 -> 120.  Widths of whole 4-stage rings only.
inline bool use_bf16_pipe(int64_t rows, int64_t D, int64_t I, bool slab) {
  return D % 128 == 0 && D >= 256 && D <= (slab ? 768 : 640) &&
         (int64_t)cdiv(rows, kTile) * (I / 64) >= 5 * kCUs / 2;
}

int bf16_swiglu_launch(const void* x, const void* w, int64_t T, int64_t D, int64_t I, const float* rstd, void* gu,
                       void* h, const int* plan, int64_t ldp, int64_t ldxs, hipStream_t st) {
  if (use_bf16_pipe(plan ? ldp : T, D, I, ldxs > 0)) {
    const auto kern = D == 256   ? bf16_swiglu_pipe_kernel<8, true>
                      : D == 384 ? bf16_swiglu_pipe_kernel<8, false>
                      : D == 512 ? bf16_swiglu_pipe_kernel<16, true>
                                 : bf16_swiglu_pipe_kernel<16, false>;
    const int tiles_m = cdiv(plan ? ldp : T, kTile), tiles_n = (int)(I / 64), ntiles = tiles_m * tiles_n;
    int n_cu = 0;
    int rc = cu_count(&n_cu);
    if (rc) return rc;
    rc = prep(kern, kBf16PipeLds);
    if (rc) return rc;
    hipLaunchKernelGGL(kern, dim3(ntiles < n_cu ? ntiles : n_cu), dim3(512), kBf16PipeLds, st, (const uint16_t*)x,
                       (const uint8_t*)w, T, D, I, rstd, (uint16_t*)gu, (uint16_t*)h, tiles_m, tiles_n, plan,
                       plan ? 2 * D * slab_rows(2 * I) : 0, ldxs);
    return status();
  }
  const Tiling tl = swiglu_tiling(plan ? ldp : T, I);
  const auto kern = tl.small ? bf16_swiglu_fwd_kernel<true> : bf16_swiglu_fwd_kernel<false>;
  const int rc = prep(kern, tl.lds);
  if (rc) return rc;
  hipLaunchKernelGGL(kern, tl.grid, tl.block, tl.lds, st,
                     (const uint16_t*)x, (const uint8_t*)w, T, D, I, rstd, (uint16_t*)gu, (uint16_t*)h, tl.m,
                     tl.n, plan, plan ? 2 * D * slab_rows(2 * I) : 0, ldxs, 0);
  return status();
}

int bf16_gemm_launch(const void* a, const void* b, int64_t T, int64_t N, int64_t K, int64_t lda, void* out,
                     const int* plan, hipStream_t st) {
  const Tiling tl = out_tiling(plan ? lda : T, N, 2 * K, plan != nullptr);
  const auto kern = OUT_KERNEL(bf16_gemm_kernel, tl);
  const int rc = prep(kern, tl.lds);
  if (rc) return rc;
  hipLaunchKernelGGL(kern, tl.grid, tl.block, tl.lds, st,
                     (const uint8_t*)a, (const uint8_t*)b, T, N, 2 * K, lda, (uint16_t*)out, tl.m, tl.n, plan,
                     plan ? 2 * K * slab_rows(N) : 0);
  return status();
}
}  // namespace

int sfp8_bf16_gemm_swiglu_fwd(const void* x, int x_slab, const void* w, int64_t T, int64_t D, int64_t I,
                              const float* rstd, void* gu, void* h, void* stream) {
  if (!w || (T > 0 && (!x || !gu || !h))) return kErrNullPointer;
  if (T < 0 || !bf16_shape(D, I) || !fits32(kTile, 2 * D) || !fits32(slab_rows(2 * I), 2 * D)) return kErrBadShape;
  if (x_slab && !fits32(slab_rows(T), 2 * D)) return kErrBadShape;
  if (!al16(x) || !al16(w) || !al16(gu) || !al16(h)) return kErrBadAlignment;
  if (T == 0) return kOk;
  return bf16_swiglu_launch(x, w, T, D, I, rstd, gu, h, nullptr, 0, x_slab ? slab_rows(T) : 0,
                            (hipStream_t)stream);
}

int sfp8_bf16_swiglu_eval(const void* x, const void* w, int64_t T, int64_t D, int64_t I, void* h, void* stream) {
  if (!w || (T > 0 && (!x || !h))) return kErrNullPointer;
  if (T < 0 || !bf16_shape(D, I) || !fits32(kTile, 2 * D) || !fits32(2 * I, 2 * D)) return kErrBadShape;
  if (!al16(x) || !al16(w) || !al16(h)) return kErrBadAlignment;
  if (T == 0) return kOk;
  hipStream_t st = (hipStream_t)stream;
  if (T <= kEvalRows) {
    const auto kern = T <= 32 ? bf16_swiglu_eval_kernel<1> : bf16_swiglu_eval_kernel<2>;
    const int lds = T <= 32 ? EvalShape<1>::kLds : EvalShape<2>::kLds, rc = prep(kern, lds);
    if (rc) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)(I / 16)), dim3(512), lds, st, (const uint16_t*)x, (const uint16_t*)w,
                       (int)T, (int)D, (int)I, (uint16_t*)h);
    return status();
  }
  const Tiling tl = swiglu_tiling(T, I);
  const auto kern = tl.small ? bf16_swiglu_fwd_kernel<true> : bf16_swiglu_fwd_kernel<false>;
  const int rc = prep(kern, tl.lds);
  if (rc) return rc;
  hipLaunchKernelGGL(kern, tl.grid, tl.block, tl.lds, st, (const uint16_t*)x, (const uint8_t*)w, T, D, I,
                     (const float*)nullptr, (uint16_t*)nullptr, (uint16_t*)h, tl.m, tl.n, (const int*)nullptr,
                     (int64_t)0, (int64_t)0, 1);
  return status();
}

int sfp8_bf16_moe_gemm_swiglu_fwd(const void* x, const void* w, int64_t E, int64_t D, int64_t I, const int* plan,
                                  int64_t ldp, void* gu, void* h, void* stream) {
  if (!w || !plan || (ldp > 0 && (!x || !gu || !h))) return kErrNullPointer;
  if (E <= 0 || ldp < 0 || ldp % kTile || !bf16_shape(D, I) || !fits32(kTile, 2 * D) ||
      !fits32(slab_rows(2 * I), 2 * D))
    return kErrBadShape;
  if (!al16(x) || !al16(w) || !al16(gu) || !al16(h)) return kErrBadAlignment;
  if (ldp == 0) return kOk;
  return bf16_swiglu_launch(x, w, 0, D, I, nullptr, gu, h, plan, ldp, 0, (hipStream_t)stream);
}

int sfp8_bf16_gemm(const void* a, const void* b, int64_t T, int64_t N, int64_t K, int64_t lda, void* out,
                   void* stream) {
  if (!b || (T > 0 && (!a || !out))) return kErrNullPointer;
  if (T < 0 || N <= 0 || N % 8 || K <= 0 || K % 32 || lda < T || lda % kTile) return kErrBadShape;
  if (!fits32(lda, 2 * K) || !fits32(slab_rows(N), 2 * K) || !fits32(kTile, 2 * N)) return kErrBadShape;
  if (!al16(a) || !al16(b) || !al16(out)) return kErrBadAlignment;
  if (T == 0) return kOk;
  return bf16_gemm_launch(a, b, T, N, K, lda, out, nullptr, (hipStream_t)stream);
}

int sfp8_bf16_moe_gemm(const void* a, const void* b, int64_t E, int64_t N, int64_t K, const int* plan, int64_t ldp,
                       void* out, void* stream) {
  if (!b || !plan || (ldp > 0 && (!a || !out))) return kErrNullPointer;
  if (E <= 0 || N <= 0 || N % 8 || K <= 0 || K % 32 || ldp < 0 || ldp % kTile) return kErrBadShape;
  if (!fits32(ldp, 2 * K) || !fits32(slab_rows(N), 2 * K)) return kErrBadShape;
  if (!al16(a) || !al16(b) || !al16(out)) return kErrBadAlignment;
  if (ldp == 0) return kOk;
  return bf16_gemm_launch(a, b, 0, N, K, ldp, out, plan, (hipStream_t)stream);
}

int64_t sfp8_bf16_wgrad_splits(int64_t M, int64_t N, int64_t ldt) { return wgrad_splits(M, N, 2 * ldt); }

int64_t sfp8_bf16_wgrad_workspace_floats(int64_t M, int64_t N, int64_t ldt) {
  const int64_t s = sfp8_bf16_wgrad_splits(M, N, ldt);
  return s > 1 ? s * (int64_t)cdiv(M, kTile) * cdiv(N, kTile) * kTile * kTile : 0;
}

int sfp8_bf16_gemm_wgrad(const void* at, const void* bt, int64_t M, int64_t N, int64_t ldt, void* out, float* ws,
                         int64_t ws_floats, void* stream) {
  if (!out || (ldt > 0 && (!at || !bt))) return kErrNullPointer;
  if (M <= 0 || N <= 0 || ldt < 0 || ldt % kTile || N % 4 || (M * N) % 8) return kErrBadShape;
  if (!fits32(slab_rows(M), 2 * ldt) || !fits32(slab_rows(N), 2 * ldt)) return kErrBadShape;
  if (!al16(at) || !al16(bt) || !al16(out) || !al16(ws)) return kErrBadAlignment;
  hipStream_t st = (hipStream_t)stream;
  if (ldt == 0) {
    // no tokens: a zero gradient (M * N bf16 = M * N / 2 floats of zero bits)
    const int64_t n = M * N / 2;
    hipLaunchKernelGGL(zero_fill_kernel, dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, st, (float*)out, n);
    return status();
  }
  const int64_t splits = dense_splits(M, N, 2 * ldt, true);
  if (no_workspace(ws, ws_floats, sfp8_bf16_wgrad_workspace_floats(M, N, ldt))) return kErrWorkspaceTooSmall;
  const Tiling tl = tiling(M, N, splits);
  const int rc = launch_wgrad<true, 0, 0, false, false>(tl, at, bt, M, N, 2 * ldt, wgrad_chunk(2 * ldt, splits), nullptr, nullptr,
                                                        splits > 1 ? ws : (float*)out, (int)splits, splits > 1, TrOp{},
                                                        TrOp{}, st);
  if (rc || splits == 1) return rc;
  return launch_bf16_reduce(tl, false, ws, (int)splits, 1, M, N, out, st);
}

int64_t sfp8_bf16_moe_wgrad_workspace_floats(int64_t M, int64_t N, int64_t E) {
  return sfp8_moe_wgrad_workspace_floats(M, N, E);
}

int sfp8_bf16_moe_gemm_wgrad(const void* at, const void* bt, int64_t M, int64_t N, int64_t E, const int* plan,
                             int64_t ldp, void* out, float* ws, int64_t ws_floats, void* stream) {
  if (!at || !bt || !plan || !out) return kErrNullPointer;
  if (M <= 0 || N <= 0 || E <= 0 || N % 4 || ldp <= 0 || ldp % kTile) return kErrBadShape;
  if (!fits32(slab_rows(M), 2 * ldp) || !fits32(slab_rows(N), 2 * ldp)) return kErrBadShape;
  if (!al16(at) || !al16(bt) || !al16(out) || !al16(ws)) return kErrBadAlignment;
  const MoeSplits splits = moe_wgrad_splits(M, N, E, ldp, true);
  if (no_workspace(ws, ws_floats, sfp8_bf16_moe_wgrad_workspace_floats(M, N, E))) return kErrWorkspaceTooSmall;
  hipStream_t st = (hipStream_t)stream;
  const Tiling tl = tiling(M, N, E * splits.even);
  const int rc = launch_moe_wgrad<true, 0, 0, false, false>(tl, at, bt, M, N, 2 * ldp, nullptr, nullptr, (float*)out,
                                                           ws, plan, splits, st);
  if (rc || splits.longest == 1) return rc;
  return launch_bf16_reduce(tl, false, ws, splits.longest, E, M, N, out, st, uneven(splits, plan), splits.even);
}

// ---- the bf16 weight gradients read through transposing LDS reads ----
int sfp8_bf16_gemm_wgrad_rows(const void* a, const void* x, int x_rows, int64_t M, int64_t N, int64_t T, int64_t ldt,
                              void* out, float* ws, int64_t ws_floats, void* stream) {
  if (!out || (T > 0 && (!a || !x))) return kErrNullPointer;
  if (M <= 0 || N <= 0 || M % 32 || N % (x_rows ? 32 : 4) || T < 0 || ldt < T || ldt % kTile || (M * N) % 8)
    return kErrBadShape;
  if (!fits32(slab_rows(M), 2 * ldt) || !fits32(slab_rows(N), 2 * ldt) || T * N * 2 >= ((int64_t)1 << 31))
    return kErrBadShape;
  if (!al16(a) || !al16(x) || !al16(out) || !al16(ws)) return kErrBadAlignment;
  hipStream_t st = (hipStream_t)stream;
  if (ldt == 0) {
    const int64_t n = M * N / 2;
    hipLaunchKernelGGL(zero_fill_kernel, dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, st, (float*)out, n);
    return status();
  }
  const int64_t splits = dense_splits(M, N, 2 * ldt, true);
  if (no_workspace(ws, ws_floats, sfp8_bf16_wgrad_workspace_floats(M, N, ldt))) return kErrWorkspaceTooSmall;
  // a: the bf16 K-slab of [ldt, M] (32 columns per 64-byte row); x (x_rows):
  // row-major [T, N] bf16, tokens T..ldt-1 read as zero through the range
  // check, or else the token-contiguous bf16 K-slab of x^T over ldt tokens
  const TrOp tra{kStage, ldt * kStage, (M / 32) * ldt * kStage}, trb{2 * N, kStage, T * 2 * N};
  const Tiling tl = tiling(M, N, splits);
  const auto launch = x_rows ? launch_wgrad<true, 0, 0, true, true> : launch_wgrad<true, 0, 0, true, false>;
  const int rc = launch(tl, a, x, M, N, 2 * ldt, wgrad_chunk(2 * ldt, splits), nullptr, nullptr,
                        splits > 1 ? ws : (float*)out, (int)splits, splits > 1, tra, x_rows ? trb : TrOp{}, st);
  if (rc || splits == 1) return rc;
  return launch_bf16_reduce(tl, x_rows, ws, (int)splits, 1, M, N, out, st);
}

int sfp8_bf16_moe_gemm_wgrad_rows(const void* a, const void* bt, int64_t M, int64_t N, int64_t E, const int* plan,
                                  int64_t ldp, void* out, float* ws, int64_t ws_floats, void* stream) {
  if (!a || !bt || !plan || !out) return kErrNullPointer;
  if (M <= 0 || N <= 0 || E <= 0 || M % 32 || N % 4 || ldp <= 0 || ldp % kTile) return kErrBadShape;
  if (!fits32(slab_rows(M), 2 * ldp) || !fits32(slab_rows(N), 2 * ldp)) return kErrBadShape;
  if (!al16(a) || !al16(bt) || !al16(out) || !al16(ws)) return kErrBadAlignment;
  const MoeSplits splits = moe_wgrad_splits(M, N, E, ldp, true);
  if (no_workspace(ws, ws_floats, sfp8_bf16_moe_wgrad_workspace_floats(M, N, E))) return kErrWorkspaceTooSmall;
  hipStream_t st = (hipStream_t)stream;
  const Tiling tl = tiling(M, N, E * splits.even);
  const int rc = launch_moe_wgrad<true, 0, 0, true, false>(tl, a, bt, M, N, 2 * ldp, nullptr, nullptr, (float*)out,
                                                           ws, plan, splits, st);
  if (rc || splits.longest == 1) return rc;
  return launch_bf16_reduce(tl, false, ws, splits.longest, E, M, N, out, st, uneven(splits, plan), splits.even);
}

// ---- the weight gradient with row K-slab operands ----
int64_t sfp8_wgrad_rows_workspace_floats(int64_t M, int64_t N, int64_t ldt) {
  return sfp8_wgrad_workspace_floats(M, N, ldt);
}

int sfp8_gemm_wgrad_rows(const void* a, int fmt_a, int a_rows, const void* b, int fmt_b, int b_rows, int64_t M,
                         int64_t N, int64_t ldt, const float* sa, const float* sb, float* out, float* ws,
                         int64_t ws_floats, void* stream) {
  if (!sa || !sb || !out || (ldt > 0 && (!a || !b))) return kErrNullPointer;
  if (M <= 0 || N <= 0 || ldt < 0 || ldt % kTile || N % 4 || !(a_rows || b_rows)) return kErrBadShape;
  if ((a_rows && M % 64) || (b_rows && N % 64)) return kErrBadShape;
  if (fmt_a != kFmtE5M2 || fmt_b != kFmtE4M3) return kErrBadShape;
  if (!fits32(slab_rows(M), ldt) || !fits32(slab_rows(N), ldt)) return kErrBadShape;
  if (!al16(a) || !al16(b) || !al16(out) || !al16(ws)) return kErrBadAlignment;
  hipStream_t st = (hipStream_t)stream;
  if (ldt == 0) {
    const int64_t n = M * N;
    hipLaunchKernelGGL(zero_fill_kernel, dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, st, out, n);
    return status();
  }
  const int splits = (int)dense_splits(M, N, ldt, false);
  const int64_t most = sfp8_wgrad_rows_workspace_floats(M, N, ldt);
  if (no_workspace(ws, ws_floats, most)) return ws ? kErrWorkspaceTooSmall : kErrNullPointer;
  const Tiling tl = tiling(M, N, splits);
  const int rc =
      wgrad_partials(tl, a_rows, b_rows, a, b, M, N, ldt, sa, sb, splits > 1 ? ws : out, splits, splits > 1, st);
  if (rc || splits == 1) return rc;
  return launch_reduce(tl, b_rows, ws, splits, 1, M, N, sa, sb, out, st);
}

// ---- the weight gradient fused with the optimizer's momentum stage ----
int64_t sfp8_wgrad_momentum_workspace_floats(int64_t M, int64_t N, int64_t ldt) {
  return sfp8_wgrad_splits(M, N, ldt) * (int64_t)cdiv(M, kTile) * cdiv(N, kTile) * kTile * kTile;
}

int sfp8_gemm_wgrad_momentum(const void* a, int fmt_a, int a_rows, const void* b, int fmt_b, int b_rows, int64_t M,
                             int64_t N, int64_t ldt, const float* sa, const float* sb, float* grad, float* v, void* u,
                             float w_v, float w_u, float* ws, int64_t ws_floats, void* stream) {
  if (!sa || !sb || !v || !u || (ldt > 0 && (!a || !b || !ws))) return kErrNullPointer;
  if (M <= 0 || N <= 0 || ldt < 0 || ldt % kTile || N % 4) return kErrBadShape;
  if ((a_rows && M % 64) || (b_rows && N % 64)) return kErrBadShape;
  if (fmt_a != kFmtE5M2 || fmt_b != kFmtE4M3 || !(w_v > -0.5f && w_v < 0.5f) || !(w_u >= 0.5f)) return kErrBadShape;
  if (!fits32(slab_rows(M), ldt) || !fits32(slab_rows(N), ldt)) return kErrBadShape;
  if (!al16(a) || !al16(b) || !al16(grad) || !al16(v) || !al16(ws) || (((uintptr_t)u) & 7u)) return kErrBadAlignment;
  hipStream_t st = (hipStream_t)stream;
  int splits = 0;
  if (ldt > 0) {
    splits = (int)dense_splits(M, N, ldt, false);
    if (ws_floats < sfp8_wgrad_momentum_workspace_floats(M, N, ldt)) return kErrWorkspaceTooSmall;
  }
  const Tiling tl = tiling(M, N, splits);
  if (ldt > 0) {
    const int rc = wgrad_partials(tl, a_rows, b_rows, a, b, M, N, ldt, sa, sb, ws, splits, 1, st);
    if (rc) return rc;
  }
  const auto kern = tl.small ? (b_rows ? splitk_momentum_kernel<true, true> : splitk_momentum_kernel<true, false>)
                             : (b_rows ? splitk_momentum_kernel<false, true> : splitk_momentum_kernel<false, false>);
  hipLaunchKernelGGL(kern, reduce_grid(tl, 1), dim3(256), 0, st, ws, splits, partial_quads(tl), tl.n, M, N, sa, sb,
                     grad, v, (uint16_t*)u, w_v, 1.0f - w_u);
  return status();
}

}  // extern "C"
