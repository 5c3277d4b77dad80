// The tile loop of the large-tile expert GEMMs for tiles of 8 to 20 row tiles: both operands through LDS.
//
// A workgroup (4 waves, one per SIMD) multiplies up to 320 rows x 256 columns.  The waves stand in a 2 x 2 grid: wave
// (wm, wn) owns half of the row tiles and 128 columns, so that a K slice of 128 bytes costs it 8 + 8 operand fragments for
// 64 MFMAs (one wave across all rows needs 16 activation fragments and 4 weight fragments, which then have to come
// from memory straight into registers, with moves into operand order and a wait at the head of every slice).
//   * Both operands go global -> LDS without touching a register (buffer_load ... lds), two stages each.  Nothing that a
//     load writes is a register, so the waits below are all there is to get right.
//   * Weights lie in LDS as they do in memory, [32 partitions][256 columns][4 K values]: one 1 KB row per partition,
//     columns in any order of 4-column pieces (the DMA's lanes fetch what their LDS place wants), the 64-byte units of
//     row p at unit ^ ((p >> 2) & 3).  A fragment (16 columns x 8 partitions of the lane's K group) is then four
//     ds_read2st64_b32, each of which brings two partitions of the lane's column into consecutive registers: MFMA
//     operand order without a move, from the reference layout and from the packed copies alike, and free of conflicts.
//   * The weights are the MFMA's first operand, the activations the second: a lane then holds four neighbouring columns of
//     one token's row, and the epilogues pack and store 16 bytes per lane without any exchange between lanes (the MX
//     re-quantisation needs one, its blocks span two lane groups).
//   * Per slice two barriers.  B1, behind the slice's first 8 MFMAs: every wave holds its weight fragments, the slice's
//     weight stage is free, and the loads of the weights two slices ahead go out into it.  B2, ahead of the slice's last
//     16 MFMAs: every wave holds its last activation fragments and what it has requested of the next slice has
//     landed; the loads of the activations two slices ahead go out, and under the last 16 MFMAs the fragments of the next
//     slice are read: a weight fragment is read into the registers of the one whose last MFMA has just been issued.
//     No slice begins with a wait for LDS.
// What bounds it: the matrix pipes with bf16 (a slice of 16 row tiles takes 2690 cycles, its MFMAs alone 2480: 128 of
// 16 x 16 x 32, one in 19.35 cycles); with 8 bits, where the MFMAs take 2048, the DMA's latency (fp8-row 2540 cycles, MXFP8 with
// the weights from HBM 3050); all of them at the clock that the part's power leaves, 1.7 to 2.1 GHz.  Layers back to back, against the loop before (weights through registers, one wave
// across all rows, some 4000 cycles per slice): 8192 tokens over 256 MXFP8 experts of H = 7168, I = 2048 3155 -> 3010 us;
// 4096 tokens, top-2 of 8 bf16 experts of H = 2048, I = 4096 440 -> 409; 8192 tokens, top-8 of 128 MXFP8 experts of H = 2048,
// I = 768 539 -> 502; 1999 tokens, top-4 of 32 MXFP4 experts of H = 3072, I = 1536 203 -> 196.
// (Dense kinds: no vector ALU instruction in the K loop; MX: one per slice, the address of the activation scales, and with
// 4-bit weights the 32 that pick a column's halves.)
#pragma once

#include "mx_tile.hpp"

namespace moe {

template <int NMT>
struct MxWideCfg {
  static constexpr int RT = NMT / 2;             // row tiles of a wave
  static constexpr int SA = NMT * 16 * MXROW;    // bytes of an activation stage
  static constexpr int SW = 32 * 1024;           // ... of a weight stage
  static constexpr int OFF_W = 2 * SA;
  static constexpr int OFF_AS = OFF_W + 2 * SW;  // activation scales of four slices: [row][slice % 4][K block]
  static constexpr int AS = (NMT > 16 ? 320 : 256) * 16;
  static constexpr int OFF_WS = OFF_AS + AS;     // weight scales, two stages: [K block][256 columns], rows of WSP bytes
  static constexpr int WSP = 256 + 16;
  static constexpr int WS = 4 * WSP;
  static constexpr int LDS_PLAIN = OFF_AS, LDS_SCALED = OFF_WS + 2 * WS;
  // The epilogue's exchange, 4 KB per wave: behind the rest, or, where that fills the LDS, in the part of the second
  // activation stage that is loaded by the next tile's first slice.
  static constexpr int OFF_EX_BIG = SA + ((RT + 1) / 2) * 4096;
  static_assert(NMT <= 16 || OFF_EX_BIG + 16384 <= 2 * SA, "the exchange fits the part of the stage that is free");
};
static_assert(MxWideCfg<16>::LDS_PLAIN + 16384 <= MxWideCfg<20>::LDS_PLAIN &&
              MxWideCfg<16>::LDS_SCALED + 16384 <= MxWideCfg<20>::LDS_SCALED, "the exchange of the smaller tiles fits");
constexpr int MX_WIDE_LDS_PLAIN = MxWideCfg<20>::LDS_PLAIN, MX_WIDE_LDS_SCALED = MxWideCfg<20>::LDS_SCALED;

// One MFMA: weight fragment wf (first operand, element format WFMT) x activation fragment af into the fixed accumulators
// ACC .. ACC + 3.  Scales sit in byte 0 of their registers.
#define MXW_MFMA(FMT_)                                                                                          \
  asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 a[%0:%1], %2, %3, a[%0:%1], %4, %5 op_sel_hi:[0,0,0]" FMT_     \
               : : "n"(ACC), "n"(ACC + 3), "v"(wf), "v"(af), "v"(sw), "v"(sa))
template <int ACC, int WFMT, int HALF, class WFrag>
__device__ __forceinline__ void mxw_mfma(const WFrag& wf, const v8i& af, int sw, int sa) {
  if constexpr (WFMT == MX_WFMT_E2M1) {
    MXW_MFMA(" cbsz:4");
  } else if constexpr (WFMT == MX_WFMT_BF16) {
    const v4i w4 = HALF ? (v4i){wf[4], wf[5], wf[6], wf[7]} : (v4i){wf[0], wf[1], wf[2], wf[3]};
    const v4i a4 = HALF ? (v4i){af[4], af[5], af[6], af[7]} : (v4i){af[0], af[1], af[2], af[3]};
    asm volatile("v_mfma_f32_16x16x32_bf16 a[%0:%1], %2, %3, a[%0:%1]" : : "n"(ACC), "n"(ACC + 3), "v"(w4), "v"(a4));
  } else if constexpr (WFMT == MX_WFMT_E5M2) {
    MXW_MFMA(" cbsz:1");
  } else {
    MXW_MFMA("");
  }
}
#undef MXW_MFMA
// The same with the accumulator tile in ordinary registers (row tiles 8, 9 of a wave).
#define MXW_MFMA(FMT_)                                                                                       \
  asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel_hi:[0,0,0]" FMT_              \
               : "+v"(acc) : "v"(wf), "v"(af), "v"(sw), "v"(sa))
template <int WFMT, int HALF, class WFrag>
__device__ __forceinline__ void mxw_mfma_v(v4f& acc, const WFrag& wf, const v8i& af, int sw, int sa) {
  if constexpr (WFMT == MX_WFMT_E2M1) {
    MXW_MFMA(" cbsz:4");
  } else if constexpr (WFMT == MX_WFMT_BF16) {
    const v4i w4 = HALF ? (v4i){wf[4], wf[5], wf[6], wf[7]} : (v4i){wf[0], wf[1], wf[2], wf[3]};
    const v4i a4 = HALF ? (v4i){af[4], af[5], af[6], af[7]} : (v4i){af[0], af[1], af[2], af[3]};
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(w4), "v"(a4));
  } else if constexpr (WFMT == MX_WFMT_E5M2) {
    MXW_MFMA(" cbsz:1");
  } else {
    MXW_MFMA("");
  }
}
#undef MXW_MFMA

// 16 (4) bytes per lane straight into LDS at base + OFF + 16 (4) * lane.  M0 carries the LDS address; a memory instruction
// that reads M0 needs a wait state behind the scalar instruction that wrote it, and one that reads a scalar register five
// behind a vector instruction that wrote that (see MX_SGPR_WAIT).  LOOP: the K loop's loads, which carry the first of the two
// only: the loop keeps all its scalars in scalar registers and has no vector instruction that writes one (build.py reads
// the compiled code for that); four issue slots less per load are 5 % of the bf16 loop.
#define MXW_DMA(WAIT_, OP_)                                                                    \
  asm volatile("s_add_u32 m0, %0, %4\n\t" WAIT_ "buffer_load_" OP_                             \
               : : "s"(base), "v"(voff), "s"(rsrc), "s"(soff), "n"(OFF) : "memory", "m0", "scc")
#define MXW_M0_WAIT "s_nop 0\n\t"
template <int OFF, bool NT, bool LOOP>
__device__ __forceinline__ void dma_b128(uint32_t base, uint32_t voff, const v4i& rsrc, int soff) {
  if constexpr (NT && LOOP) MXW_DMA(MXW_M0_WAIT, "dwordx4 %1, %2, %3 offen nt lds");
  else if constexpr (NT) MXW_DMA(MX_SGPR_WAIT, "dwordx4 %1, %2, %3 offen nt lds");
  else if constexpr (LOOP) MXW_DMA(MXW_M0_WAIT, "dwordx4 %1, %2, %3 offen lds");
  else MXW_DMA(MX_SGPR_WAIT, "dwordx4 %1, %2, %3 offen lds");
}
template <int OFF, bool LOOP>
__device__ __forceinline__ void dma_b32(uint32_t base, uint32_t voff, const v4i& rsrc, int soff) {
  if constexpr (LOOP) MXW_DMA(MXW_M0_WAIT, "dword %1, %2, %3 offen lds");
  else MXW_DMA(MX_SGPR_WAIT, "dword %1, %2, %3 offen lds");
}
#undef MXW_DMA
#undef MXW_M0_WAIT
__device__ __forceinline__ void st_b8(int d, uint32_t voff, const v4i& rsrc, int soff) {
  asm volatile(MX_SGPR_WAIT "buffer_store_byte %0, %1, %2, %3 offen" : : "v"(d), "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}
__device__ __forceinline__ void st_b128_plain(const v4i& d, uint32_t voff, const v4i& rsrc, int soff) {
  asm volatile(MX_SGPR_WAIT "buffer_store_dwordx4 %0, %1, %2, %3 offen" : : "v"(d), "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}

// One class of tiles (see mx_gemm_tiles in bwmm_mx.hip for the walk over the queue, LASTUSE and the order of requests
// around the epilogue).
template <int STAGE, int NMT, bool LASTUSE, int WFMT, bool KTAIL>
__device__ __forceinline__ int mx_gemm_tiles_wide(const MxArgs& a, uint8_t* smem, int (*s_tok)[MX_ROWS_MAX],
                                                  float (*s_aff)[MX_ROWS_MAX], float (*s_bias)[MXT],
                                                  float (*s_rs)[MX_ROWS_MAX], float (*s_wsc)[MXT], int L, int& step, const MxRun& run) {
  static_assert(NMT >= 8 && NMT % 2 == 0, "at least four row tiles per wave");
  using Cfg = MxWideCfg<NMT>;
  constexpr bool BF16 = WFMT == MX_WFMT_BF16;
  constexpr bool ROW8 = WFMT == MX_WFMT_ROW8 || BF16;
  constexpr bool SCALED = !ROW8;
  constexpr bool FP4 = WFMT == MX_WFMT_E2M1;
  constexpr int ES = FP4 ? 2 : 4;  // bytes of a weight element (four K values of a column)
  constexpr int RT = Cfg::RT, SA = Cfg::SA, SW = Cfg::SW;
  constexpr bool BIG = NMT > 16;  // row tiles 8, 9 of a wave accumulate in ordinary registers

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = uni(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int wm = w >> 1, wn = w & 1;
  const int nH = (int)(a.H / 512);
  typedef MxTileWalk<STAGE, NMT, WFMT> TW;
  const TW tw{a, s_tok, s_aff, s_bias, s_rs, s_wsc, tid, run};

  // ---- columns ------------------------------------------------------------------------------------------------
  // Position Q = (wn, column tile tt, piece gq) of a 4-column piece among the workgroup's 64; a lane of group g ends up
  // with the four columns of piece gq = g of every column tile of its wave.
  //   gate/up: even column tiles hold gate columns, odd ones the up columns that belong to them.
  //     MX: tile pair = quarter q, pieces = 4 of the 8 pieces (of 4 partitions) that wave wn owns of each quarter
  //     bf16: tile pairs 2j, 2j+1 = quarter 2 wn + j, a lane gets 8 neighbouring columns of the two pairs (16-byte stores)
  //     fp8-row: the same quarters, a lane 4 neighbouring columns of each pair (fp32 results, 16-byte stores)
  //   down: tile pairs, a lane gets 8 neighbouring columns of a pair (4-bit weights, whose DMA brings two pieces at a time:
  //     twice 4)
  struct Piece {
    int q, gu, cl;  // gate/up: quarter, gate or up, piece of 4 partitions among the column tile's 8; down: cl alone
  };
  auto piece_at = [&](int pwn, int tt, int gq) {
    Piece p;
    const int t = tt >> 1, odd = tt & 1;
    if (STAGE == 2) {
      p.q = 0; p.gu = 0;
      p.cl = pwn * 32 + t * 8 + (FP4 ? 4 * odd + gq : 2 * gq + odd);
    } else if (SCALED) {
      p.q = t; p.gu = odd;
      p.cl = pwn * 4 + gq;
    } else {
      p.q = 2 * pwn + (t >> 1); p.gu = odd;
      p.cl = BF16 ? 2 * gq + (t & 1) : 4 * (t & 1) + gq;
    }
    return p;
  };

  // ---- K schedule (slice ks: tile of 512 ks >> 2, partition group ks & 3; see bwmm_mx.hip) ------------------------
  int nks;
  if (STAGE == 1) nks = (int)(a.H / 128);
  else nks = (int)mx_col_tiles(a.I);
  // KTAIL: K ends inside the last slice, behind partition nP - 1 counted through all slices (whole MX blocks of
  // 8); weights and scales past that are not read (see aim_w)
  static_assert(!KTAIL || (STAGE == 2 && SCALED), "the other stages' K are whole slices");
  const int nP = uni((int)(a.I >> 2));

  // ---- operand addressing -----------------------------------------------------------------------------------
  const int64_t w_pstride = (STAGE == 1) ? 2 * (int64_t)nH * a.I : (int64_t)a.nI * a.H;  // elements between partitions
  const int64_t w_tstride = (STAGE == 1) ? a.I : a.H;                                     // ... between tiles of 512
  const bool pk = a.w_packed != 0;
  constexpr int PK_LANE = FP4 ? 8 : 16, PK_LOAD = 64 * PK_LANE, PK_WAVE = 8 * PK_LOAD, PK_SLICE = 4 * PK_WAVE;
  const int64_t w_expert_bytes = pk ? (int64_t)a.col_tiles * nks * PK_SLICE
                                    : (STAGE == 1 ? 128 : (int64_t)a.pI) * w_pstride * ES;
  const int64_t ws_expert_bytes = (STAGE == 1 ? 16 : ((int64_t)a.pI + 7) / 8) * w_pstride;
  // a weight slice: wave w brings partitions 4 w .. 4 w + 3 and 16 + 4 w .. 16 + 4 w + 3, one per load, or (4-bit weights)
  // 8 w .. 8 w + 7, two per load; all of these have the swizzle w
  const int w_step = uni(pk ? 1024 : (int)(w_pstride * 4)), w_jump = uni(pk ? 4 * PK_LOAD : (int)(w_pstride * 64));
  const int w_pb = uni(pk ? PK_SLICE : (int)(w_pstride * 32 * ES)), w_kt = uni(pk ? 4 * PK_SLICE : (int)(w_tstride * ES));
  const int ws_pb = uni((int)(w_pstride * 4)), ws_kt = uni((int)w_tstride);
  const int lu = FP4 ? ((lane & 31) >> 1) ^ w : (lane >> 2) ^ w;  // logical column tile that belongs at the lane's place
  const Piece lp = piece_at(lu >> 3, lu & 7, FP4 ? 2 * (lane & 1) : lane & 3);  // ... its (first) piece, for the weights
  const Piece sp = piece_at(lane >> 5, (lane >> 2) & 7, lane & 3);         // the lane's piece of the weight scales (no swizzle)

  // ---- loads ----------------------------------------------------------------------------------------------------
  constexpr int NAJ = NMT / 2;            // activation loads of a slice per wave (8 rows x 128 bytes each)
  constexpr int NA1 = (NAJ + 1) / 2;      // ... of these behind B2, the others under the next slice's first MFMAs
  constexpr int NAS = SCALED ? (BIG ? 2 : 1) : 0;  // loads of the activation scales, one set for four slices
  constexpr int NWL = FP4 ? 4 : 8;        // weight loads of a slice per wave
  constexpr int NW = NWL + (SCALED ? 1 : 0);
  constexpr int NAV = (STAGE == 1) ? NAJ : 1;
  const int arow0 = tid >> 3, ach = tid & 7;
  uint32_t a_voff[NAV], as_voff = 0, as_voff2 = 0, w_voff = 0, ws_voff = 0;
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
  const uint32_t lds_a = (uint32_t)uni((int)(lds0 + (uint32_t)w * 1024u));
  const uint32_t lds_w = (uint32_t)uni((int)(lds0 + (uint32_t)(Cfg::OFF_W + w * 4096)));
  const uint32_t lds_as = (uint32_t)uni((int)(lds0 + (uint32_t)(Cfg::OFF_AS + w * 1024)));
  const uint32_t lds_as2 = (uint32_t)uni((int)(lds0 + (uint32_t)(Cfg::OFF_AS + 4096)));
  const uint32_t lds_ws = (uint32_t)uni((int)(lds0 + (uint32_t)(Cfg::OFF_WS + w * Cfg::WSP)));
  v4i ra_ = make_rsrc(a.A, (uint32_t)(a.a_rows * a.a_stride)),
      ras_ = make_rsrc(a.A_scale, (uint32_t)(a.a_scale_bytes ? a.a_scale_bytes : a.a_rows * a.a_scale_stride));
  v4i rw_ = ra_, rs_ = ras_;
  const int ra_rec = ra_[2], ras_rec = ras_[2];
  int rw_rec = 0, rs_rec = 0, w_base = 0, ws_base = 0;
  const int a_group_bytes = uni((int)(32 * a.a_stride));
  int tile_live = -1;
  // Point the loads at a tile (its token ids sit in s_tok[buf]).
  auto aim_loads_at = [&](const MxTile& t, int buf) {
#pragma unroll
    for (int j = 0; j < NAV; ++j) {
      const int row = arow0 + 32 * j;
      uint32_t r;
      if (STAGE == 1) {
        // a row without a token points past the end of the buffer: the range check turns its loads into zeros
        const int tok = s_tok[buf][row];
        r = (tok >= 0) ? (uint32_t)tok : (uint32_t)a.a_rows;
      } else {
        r = (uint32_t)(t.slot0 + row);
      }
      a_voff[j] = r * (uint32_t)a.a_stride + (uint32_t)((ach ^ (arow0 & 7)) * 16);
    }
    auto scale_row_off = [&](int row) {
      if (STAGE == 1) {
        const int tok = s_tok[buf][row];
        return ((tok >= 0) ? (uint32_t)tok : 0u) * (uint32_t)a.a_scale_stride;
      }
      return (uint32_t)(t.slot0 + ((row < t.nrows) ? row : (t.nrows - 1))) * (uint32_t)a.a_scale_stride;
    };
    if constexpr (SCALED) {
      as_voff = scale_row_off(tid);
      if constexpr (BIG) as_voff2 = scale_row_off(256 + lane);
    }
    const int Pt = tw.tile_Pt(t);
    const int colu = (STAGE == 1) ? tw.tile_tI(t) * 512 + tw.tile_p0(t) : (int)tw.tile_h0(t);
    auto piece_elem = [&](const Piece& p) {
      return (STAGE == 1) ? (uint32_t)(p.gu * nH) * (uint32_t)a.I + (uint32_t)(p.q * Pt + p.cl * 4) : (uint32_t)(p.cl * 4);
    };
    // (4-bit weights: the upper half of the wave brings the second partition of a load)
    if (pk)
      w_voff = ((STAGE == 1) ? (uint32_t)(lp.q * PK_WAVE + (w * 16 + ((lp.cl >> 2) & 1) * 8 + lp.gu * 4 + (lp.cl & 3)) * PK_LANE)
                             : (uint32_t)((lp.cl >> 4) * PK_WAVE + (w * 16 + (lp.cl & 15)) * PK_LANE)) +
               (FP4 ? (uint32_t)((lane >> 5) * PK_LOAD) : 0u);
    else
      w_voff = (uint32_t)(FP4 ? 8 * w + (lane >> 5) : 4 * w) * (uint32_t)(w_pstride * ES) + piece_elem(lp) * (uint32_t)ES;
    w_base = uni(pk ? t.xt * nks * PK_SLICE : colu * ES);
    rw_ = make_rsrc((const uint8_t*)a.W + (int64_t)t.e * w_expert_bytes, (uint32_t)w_expert_bytes);
    rw_rec = rw_[2];
    if constexpr (SCALED) {
      ws_voff = (uint32_t)w * (uint32_t)w_pstride + piece_elem(sp);
      ws_base = uni(colu);
      rs_ = make_rsrc(a.W_scale + (int64_t)(a.w_scale_shared ? 0 : t.e) * ws_expert_bytes, (uint32_t)ws_expert_bytes);
      rs_rec = rs_[2];
    }
  };
  // The loads of slice ks into stage U = ks & 1 (of a slice past the end: through descriptors of zero records, no traffic).
  // Activations, row group j.
  int a_off = 0;
  auto aim_a = [&](int ks) {
    a_off = ks * 128;
    ra_[2] = uni(ra_rec & ((ks < nks) ? tile_live : 0));
  };
  auto load_a = [&](auto u_, auto j_, auto loop_) {
    constexpr int U = decltype(u_)::value, j = decltype(j_)::value;
    constexpr bool LOOP = decltype(loop_)::value;
    if constexpr (STAGE == 1) dma_b128<U * SA + j * 4096, false, LOOP>(lds_a, a_voff[j], ra_, a_off);
    else dma_b128<U * SA + j * 4096, false, LOOP>(lds_a, a_voff[0], ra_, a_off + j * a_group_bytes);
  };
  // Weights and their scales: load i of NW.
  int w_off = 0, ws_off = 0, rw_hi = 0;
  auto aim_w = [&](int ks) {
    const int kt = ks >> 2, pb = ks & 3, live = (ks < nks) ? tile_live : 0;
    w_off = w_base + pb * w_pb + kt * w_kt;
    // (KTAIL: the wave's first partitions, 4-bit weights all of them, and those of its second half; its scales' block)
    rw_[2] = uni(rw_rec & (KTAIL ? (ks * 32 + (FP4 ? 8 : 4) * w < nP ? tile_live : 0) : live));
    if constexpr (KTAIL && !FP4) rw_hi = uni(rw_rec & (ks * 32 + 16 + 4 * w < nP ? tile_live : 0));
    if constexpr (SCALED) {
      ws_off = ws_base + pb * ws_pb + kt * ws_kt;
      rs_[2] = uni(rs_rec & (KTAIL ? (ks * 32 + 8 * w < nP ? tile_live : 0) : live));
    }
  };
  auto load_w = [&](auto u_, auto i_, auto loop_) {
    constexpr int U = decltype(u_)::value, i = decltype(i_)::value;
    constexpr bool LOOP = decltype(loop_)::value;
    if constexpr (KTAIL && !FP4 && i == 4) rw_[2] = rw_hi;
    if constexpr (i < NWL)
      dma_b128<U * SW + (FP4 || i < 4 ? i : 12 + i) * 1024, LASTUSE, LOOP>(
          lds_w, w_voff, rw_, w_off + (FP4 || i < 4 ? i * w_step : w_jump + (i - 4) * w_step));
    else
      dma_b32<U * Cfg::WS, LOOP>(lds_ws, ws_voff, rs_, ws_off);
  };
  // Activation scales of the four slices from ks0 (a multiple of four) on.  (The loop requests them in every second slice:
  // ahead of a group's first slice the group, and once more from within it, the same bytes to the same places.)
  auto load_as = [&](int ks0, auto loop_) {
    constexpr bool LOOP = decltype(loop_)::value;
    if constexpr (SCALED) {
      ras_[2] = uni(ras_rec & ((ks0 < nks) ? tile_live : 0));
      dma_b128<0, false, LOOP>(lds_as, as_voff, ras_, ks0 * 4);
      if constexpr (BIG) dma_b128<0, false, LOOP>(lds_as2, as_voff2, ras_, ks0 * 4);
    }
  };

  // ---- fragments --------------------------------------------------------------------------------------------------
  // Row tile i of the wave: rows wm * RT * 16 + i * 16 + c, 16-byte chunks g and g + 4, at chunk ^ (row & 7).
  const uint8_t* pa_lo = smem + (wm * RT * 16 + c) * MXROW + ((g ^ (c & 7)) * 16);
  const uint8_t* pa_hi = smem + (wm * RT * 16 + c) * MXROW + (((g + 4) ^ (c & 7)) * 16);
  // Column tile 4 x + b of the wave: 64-byte unit wn * 8 + 4 x + (b ^ g), dword c, of partitions 4 g + r and 16 + 4 g + r.
  // (4-bit weights: 32-byte units, a dword holds two columns, partitions 8 g + r)
  const uint8_t* pw[FP4 ? 8 : 4];
#pragma unroll
  for (int b = 0; b < (FP4 ? 8 : 4); ++b)
    pw[b] = smem + Cfg::OFF_W + 4096 * g + (wn * 8 + ((b & 4) | ((b & 3) ^ g))) * (16 * ES) + (FP4 ? c >> 1 : c) * 4;
  const uint8_t* pas = smem + Cfg::OFF_AS + (wm * RT * 16 + c) * 16 + g;
  const uint8_t* pws = smem + Cfg::OFF_WS + g * Cfg::WSP + wn * 128 + c;
  typedef typename std::conditional<FP4, v4i, v8i>::type WFrag;
  WFrag wf[8];
  v8i af[2][2];
  v8i wraw[4];  // 4-bit weights as read, column tile t in t & 3: two columns to a dword, see finish_w
  const uint32_t half_sel = (c & 1) ? 0x07060302u : 0x05040100u;  // the lane's column of the two
  int wsc[8], asc[RT];
#pragma unroll
  for (int i = 0; i < 8; ++i) wsc[i] = 0x7f;
#pragma unroll
  for (int i = 0; i < RT; ++i) asc[i] = 0x7f;
  auto read_w = [&](auto u_, auto t_) {
    constexpr int U = decltype(u_)::value, tt = decltype(t_)::value;
    if constexpr (FP4) {
      const uint8_t* p = pw[tt] + U * SW;
#pragma unroll
      for (int r = 0; r < 8; ++r) wraw[tt & 3][r] = *(const int*)(p + r * 512);
    } else {
      const uint8_t* p = pw[tt & 3] + U * SW + (tt >> 2) * 256;
      v8i f;
#pragma unroll
      for (int r = 0; r < 8; ++r) f[r] = *(const int*)(p + (r < 4 ? r : 12 + r) * 1024);
      wf[tt] = f;
    }
    if constexpr (SCALED) wsc[tt] = *(pws + U * Cfg::WS + tt * 16);
  };
  // 4-bit weights: two partitions of the lane's column to a register (and the distance that an MFMA needs behind a vector
  // instruction that wrote its operand)
  auto finish_w = [&](auto t_) {
    constexpr int tt = decltype(t_)::value;
    if constexpr (FP4) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        wf[tt][r] = (int)__builtin_amdgcn_perm((uint32_t)wraw[tt & 3][2 * r + 1], (uint32_t)wraw[tt & 3][2 * r], half_sel);
      asm volatile("s_nop 1" : "+v"(wf[tt]));
    }
  };
  auto read_a = [&](auto u_, auto i_, v8i& f) {
    constexpr int o = decltype(u_)::value * SA + decltype(i_)::value * 16 * MXROW;
    const v4i lo = *(const v4i*)(pa_lo + o), hi = *(const v4i*)(pa_hi + o);
    f = (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  };
  auto read_as = [&](auto i_, int ks) {
    constexpr int i = decltype(i_)::value;
    if constexpr (SCALED) asc[i] = *(pas + i * 256 + (ks & 3) * 4);
  };

  v4f accv[2][8];  // row tiles 8, 9

  // ---- a K slice --------------------------------------------------------------------------------------------------
  // Row tiles in groups of two (the first group holds one when their number is odd); fragments of the next group are
  // read under the MFMAs of a group.  Two slices are written out, so that stages and fragment sets are compile-time.
  constexpr int G = (RT + 1) / 2, ODD = RT & 1;
  constexpr int MB1 = 8, MB2 = 8 * (RT - 2);  // MFMAs ahead of the barriers
  auto slice = [&](auto u_, int ks, auto loop_) {
    constexpr int U = decltype(u_)::value;
    typedef std::integral_constant<int, U> UC;
    typedef std::integral_constant<int, U ^ 1> UN;
    acc_fence();
    static_for<0, G>([&](auto gi_) {
      constexpr int gi = decltype(gi_)::value;
      constexpr int r0 = gi == 0 ? 0 : 2 * gi - ODD, nr = (gi == 0 && ODD) ? 1 : 2;
      constexpr int set = (U * G + gi) & 1;
      constexpr bool LASTG = gi == G - 1;
      if constexpr (gi == 0) {
        // the scales of the last two row tiles (their registers were in use when the others were read)
        read_as(std::integral_constant<int, RT - 2>{}, ks);
        read_as(std::integral_constant<int, RT - 1>{}, ks);
        aim_a(ks + 1);
      }
      if constexpr (!LASTG) {
        constexpr int n0 = r0 + nr;
        read_a(UC{}, std::integral_constant<int, n0>{}, af[set ^ 1][0]);
        read_a(UC{}, std::integral_constant<int, n0 + 1>{}, af[set ^ 1][1]);
        asm volatile("" ::: "memory");
      } else {
        // B2 (the loads issued since the next slice's were: the weights two slices ahead)
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(NW) : "memory");
        constexpr int first_n = ODD ? 1 : 2;
        static_for<0, first_n>([&](auto i_) { read_a(UN{}, i_, af[set ^ 1][decltype(i_)::value]); });
        static_for<0, RT - 2>([&](auto i_) { read_as(i_, ks + 1); });
        asm volatile("" ::: "memory");
        aim_a(ks + 2);
      }
      // the group's MFMAs: row tile by row tile; in the last group column tile by column tile
      static_for<0, nr * 8>([&](auto j_) {
        constexpr int j = decltype(j_)::value;
        constexpr int m = r0 * 8 + j;  // MFMA number within the slice
        if constexpr (m == MB1) {
          // B1 (with a single row tile in the first group the reads for the group after it are the last four out)
          asm volatile("s_waitcnt lgkmcnt(%0)\n\ts_barrier" : : "n"(ODD ? 4 : 0) : "memory");
          aim_w(ks + 2);
          if constexpr (U == 1) load_as((ks + 1) & ~3, loop_);
        }
        auto mul = [&](auto jj_, auto half_) {
          constexpr int jj = decltype(jj_)::value, half = decltype(half_)::value;
          // (8-bit formats: there and back, so that every MFMA shares an operand with the one before: less switching, a
          // clock 2 % higher in a loop of nothing but these MFMAs, 8 % against both operands changing every time)
          constexpr int turn = BF16 ? 0 : LASTG ? (jj / 2) & 1 : (jj / 8) & 1;
          constexpr int xx = LASTG ? (jj % 2) ^ turn : jj / 8, cc = LASTG ? jj / 2 : turn ? 7 - jj % 8 : jj % 8, rr = r0 + xx;
          if constexpr (rr < 8) mxw_mfma<(rr * 8 + cc) * 4, WFMT, half>(wf[cc], af[set][xx], wsc[cc], asc[rr]);
          else mxw_mfma_v<WFMT, half>(accv[rr - 8][cc], wf[cc], af[set][xx], wsc[cc], asc[rr]);
        };
        mul(j_, std::integral_constant<int, 0>{});
        if constexpr (BF16 && j % 2 == 1) {  // (the second halves of two tiles behind the first ones: not back to back on one)
          mul(std::integral_constant<int, j - 1>{}, std::integral_constant<int, 1>{});
          mul(j_, std::integral_constant<int, 1>{});
        }
        if constexpr (m == 3) {  // the last two column tiles that were read
          finish_w(std::integral_constant<int, 6>{});
          finish_w(std::integral_constant<int, 7>{});
        }
        // loads, spread over the MFMAs between the barriers
        if constexpr (m < MB1) {
          constexpr int NA2 = NAJ - NA1;
          static_for<NA1 + m * NA2 / MB1, NA1 + (m + 1) * NA2 / MB1>([&](auto i_) { load_a(UN{}, i_, loop_); });
        } else if constexpr (m < MB2) {
          constexpr int n = m - MB1, span = MB2 - MB1;
          static_for<n * NW / span, (n + 1) * NW / span>([&](auto i_) { load_w(UC{}, i_, loop_); });
        } else {
          constexpr int n = m - MB2;
          if constexpr (n % 2 == 1) {
            read_w(UN{}, std::integral_constant<int, n / 2>{});
            if constexpr (n / 2 >= 2) finish_w(std::integral_constant<int, n / 2 - 2>{});
          }
          static_for<n * NA1 / 16, (n + 1) * NA1 / 16>([&](auto i_) { load_a(UC{}, i_, loop_); });
          if constexpr (n % 2 == 1) asm volatile("" ::: "memory");
        }
      });
    });
    if constexpr (BIG) asm volatile("s_nop 15");
    acc_fence();
  };

  // The loads a tile starts on, numbered in issue order (so that a part of them can be asked for at a time): scales of the
  // first four slices, slices 0 and 1 (the second part of slice 1's activations is requested by slice 0).
  constexpr int NFIRST = 1 + NW + NAJ + NW + NA1;
  constexpr int NFIRST_LOADS = NFIRST - 1 + NAS;  // instructions (the scales are none, one or two)
  static_assert(NFIRST_LOADS < 64, "the counter of outstanding memory instructions");
  auto request_first = [&](auto n0_, auto n1_) {
    static_for<decltype(n0_)::value, (decltype(n1_)::value < NFIRST ? decltype(n1_)::value : NFIRST)>([&](auto n_) {
      constexpr int n = decltype(n_)::value;
      typedef std::integral_constant<int, 0> S0;
      typedef std::integral_constant<int, 1> S1;
      if constexpr (n == 0) {
        load_as(0, std::false_type{});
        aim_w(0);
        aim_a(0);
      } else if constexpr (n < 1 + NW) {
        load_w(S0{}, std::integral_constant<int, n - 1>{}, std::false_type{});
      } else if constexpr (n < 1 + NW + NAJ) {
        load_a(S0{}, std::integral_constant<int, n - 1 - NW>{}, std::false_type{});
        if constexpr (n == NW + NAJ) {
          aim_w(1);
          aim_a(1);
        }
      } else if constexpr (n < 1 + 2 * NW + NAJ) {
        load_w(S1{}, std::integral_constant<int, n - 1 - NW - NAJ>{}, std::false_type{});
      } else {
        load_a(S1{}, std::integral_constant<int, n - 1 - 2 * NW - NAJ>{}, std::false_type{});
      }
    });
  };

  // ---- first tile: nothing is in flight yet, so plain waits do --------------------------------------------------
  // (every round trip to memory is a microsecond of the launch: what does not depend on the token ids goes out with them, in the
  // down stage the first slices, whose rows are slots)
  MxTile cur = tw.tile_at(L);
  int ids_nn[2] = {0, 0}, aff_n[2] = {0, 0}, bias_n = 0;  // requested ahead of an epilogue, put in place after it
  int rs_n[2] = {0, 0}, wsc_n = 0;                          // (fp8-row and bf16 kinds only)
  auto first_slices = [&]() {
    aim_loads_at(cur, 0);
    request_first(std::integral_constant<int, 0>{}, std::integral_constant<int, NFIRST>{});
  };
  tw.ids_raw(cur, ids_nn);
  tw.bias_raw(cur, bias_n);
  tw.wsc_raw(cur, wsc_n);
  if constexpr (STAGE == 2) {
    first_slices();
    tw.template loads_landed<NFIRST_LOADS>(ids_nn, aff_n, bias_n, rs_n, wsc_n);
  } else {
    tw.all_loads_landed(ids_nn, aff_n, bias_n, rs_n, wsc_n);
  }
  tw.ids_put(0, cur.nrows, ids_nn);
  tw.bias_put(cur, 0, bias_n);
  tw.wsc_put(cur, 0, wsc_n);
  lds_barrier();
  if (TW::AFF_ROWS) {
    tw.aff_raw(cur, 0, aff_n);
    tw.rs_raw(cur, 0, rs_n);
  }
  if constexpr (STAGE == 1) first_slices();
  int Ln = L + step;  // the item after the current one
  bool have_next = Ln < run.end;
  MxTile nxt = tw.tile_at(have_next ? Ln : L);
  tw.ids_raw(nxt, ids_nn);
  tw.all_loads_landed(ids_nn, aff_n, bias_n, rs_n, wsc_n);
  if (TW::AFF_ROWS) {
    if (STAGE == 2) tw.aff_put(cur.e, 0, aff_n);
    tw.rs_put(cur.e, 0, rs_n, aff_n);
  }
  if (have_next) tw.ids_put(1, nxt.nrows, ids_nn);  // published by the barrier below
  int buf = 0;  // which of the two row tables belongs to the current tile
  auto zero_accumulators = [&]() {
    acc_fence();
    static_for<0, (RT < 8 ? RT : 8) * 32>([&](auto i_) { acc_zero<decltype(i_)::value>(); });
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) accv[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
  };
  zero_accumulators();
  bool have_nn = L + run.W2 < run.end;
  MxTile nn = tw.tile_at(have_nn ? L + run.W2 : L);  // the tile after the next one

  for (;;) {
    // (what the tile's first slice needs has landed: every wave has waited for its own loads)
    lds_barrier();
    {
      typedef std::integral_constant<int, 0> S0;
      static_for<0, (ODD ? 1 : 2)>([&](auto i_) { read_a(S0{}, i_, af[0][decltype(i_)::value]); });
      static_for<0, RT - 2>([&](auto i_) { read_as(i_, 0); });
      static_for<0, 8>([&](auto t_) {
        read_w(S0{}, t_);
        if constexpr (decltype(t_)::value >= 2) finish_w(std::integral_constant<int, decltype(t_)::value - 2>{});
        asm volatile("" ::: "memory");  // (reads of two column tiles are not to be merged: their halves would need moves)
      });
    }
    int ks = 0;
#pragma clang loop unroll(disable)
    for (; ks + 2 <= nks; ks += 2) {
      slice(std::integral_constant<int, 0>{}, ks, std::true_type{});
      slice(std::integral_constant<int, 1>{}, ks + 1, std::true_type{});
    }
    if (ks < nks) slice(std::integral_constant<int, 0>{}, ks, std::false_type{});
    // (the loads past the end, and the MFMAs still in the pipe)
    asm volatile("s_waitcnt vmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");
    if constexpr (BIG) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(accv[i][j]));
    }

    // (the exchange shares LDS with the loads past the end then: those of all waves have to be over)
    if constexpr (BIG) asm volatile("s_barrier" ::: "memory");

    // ---- the next tile's first loads, and what the tile after it needs, go out around the epilogue ----------------
    // (Every wave is past B2 of the last slice: nothing in LDS that the epilogues of the others need is overwritten.  No
    // branch surrounds a load into registers, see bwmm_mx.hip: behind the last tile they are issued all the same.)
    const int nbuf = have_next ? buf ^ 1 : buf;
    tile_live = have_next ? -1 : 0;
    aim_loads_at(nxt, nbuf);
    if (TW::AFF_ROWS) tw.aff_raw(nxt, nbuf, aff_n);
    tw.rs_raw(nxt, nbuf, rs_n);
    tw.bias_raw(nxt, bias_n);
    tw.wsc_raw(nxt, wsc_n);
    tw.ids_raw(nn, ids_nn);
    // The epilogue's steps; behind each of the first half of them a share of the first loads.  (All at once they fill the
    // CU's load queue, and this arithmetic, which could run meanwhile, waits behind the first that does not fit.)
    constexpr int STEPS = (STAGE == 1 && ROW8) ? 2 * RT : RT, LSTEPS = (STEPS + 1) / 2;
    constexpr int STORES = (STAGE == 2) ? 4 : (SCALED || !BF16) ? 2 : 1;  // at least, per step
    auto loads_by = [](int i) constexpr { return i >= LSTEPS ? NFIRST : i * NFIRST / LSTEPS; };  // requested ahead of step i
    auto spread = [&](auto i_) {
      constexpr int i = decltype(i_)::value;
      request_first(std::integral_constant<int, loads_by(i)>{}, std::integral_constant<int, loads_by(i + 1)>{});
    };
    // Loads and stores that may still be out when the next tile starts, those issued behind the last load that its first
    // slice needs: slice 1's loads and the stores of the later steps (vector loads and stores share one counter on this
    // target, which counts down in issue order: the compiler relies on it as well and waits for vmcnt(2) ahead of the use
    // of a load with two stores behind it; a store that is not counted here only makes the wait a longer one).
    constexpr int NEED = 1 + NW + NAJ;
    auto last_need_step = [=]() constexpr {
      int i = 0;
      while (loads_by(i + 1) < NEED) ++i;
      return i;
    };
    constexpr int OUT = NFIRST - NEED + STORES * (STEPS - 1 - last_need_step());
    static_assert(OUT < 64, "the counter of outstanding memory instructions");

    // ---- epilogue -------------------------------------------------------------------------------------------------
    // (lane-derived values are derived again from a copy the compiler cannot see through: they would otherwise be kept
    // in registers across the K loop)
    int tid_e = threadIdx.x;
    asm volatile("" : "+v"(tid_e));
    const int c_e = tid_e & 15, g_e = (tid_e & 63) >> 4;
    const int row0 = wm * RT * 16 + c_e;  // the lane's row in row tile 0
    auto acc_of = [&](auto rt_, auto ct_, float (&v)[4]) {
      constexpr int rt = decltype(rt_)::value, ct = decltype(ct_)::value;
      static_for<0, 4>([&](auto r_) {
        constexpr int r = decltype(r_)::value;
        if constexpr (rt < 8) v[r] = acc_get<(rt * 8 + ct) * 4 + r>();
        else v[r] = accv[rt - 8][ct][r];
      });
    };
    typedef __bf16 v2bf_ __attribute__((ext_vector_type(2)));
    typedef float v2f_ __attribute__((ext_vector_type(2)));
    auto pack2 = [](float x, float y) {
      const v2f_ p = {x, y};
      return __builtin_bit_cast(int, __builtin_convertvector(p, v2bf_));
    };
    // A lane holds 16-byte pieces of one row and its neighbours pieces of other rows, which is what a store makes a request
    // each of (64 per instruction instead of 8 or 16 whole lines: the epilogue of a 256 x 256 down tile took 15 k cycles,
    // half of them in its stores).  So the wave's 16 rows go through 4 KB of LDS of its own: PIECES pieces per row, written
    // by row, read back with a row's pieces in neighbouring lanes; pieces are swizzled with the row.
    constexpr int PIECES = (STAGE == 2) ? 16 : (ROW8 && !BF16) ? 8 : 4, PITCH = PIECES * 16, NST = PIECES / 4;
    constexpr int FOLD = PIECES == 16 ? 0 : PIECES == 8 ? 1 : 2;
    constexpr int OFF_EX = BIG ? Cfg::OFF_EX_BIG : SCALED ? Cfg::LDS_SCALED : Cfg::LDS_PLAIN;
    const int lane_e = tid_e & 63;
    uint8_t* const ex = smem + OFF_EX + w * 4096;
    uint8_t* const ex_w = ex + c_e * PITCH;
    auto ex_put = [&](int piece, const v4i& o) { *(v4i*)(ex_w + ((piece ^ (c_e >> FOLD)) & (PIECES - 1)) * 16) = o; };
    const int st_row = lane_e / PIECES, st_piece = lane_e % PIECES;  // of the first store; 64 / PIECES rows more per store
    auto ex_get = [&](v4i (&o)[NST]) {
      asm volatile("" ::: "memory");
#pragma unroll
      for (int k = 0; k < NST; ++k) {
        const int row = k * (64 / PIECES) + st_row;
        o[k] = *(const v4i*)(ex + row * PITCH + ((st_piece ^ (row >> FOLD)) & (PIECES - 1)) * 16);
      }
      asm volatile("" ::: "memory");
    };
    const int st_row0 = wm * RT * 16 + st_row;
    if constexpr (STAGE == 1) {
      int cmask = a.clamp_mask;
      asm volatile("" : "+s"(cmask));
      const float inf = __builtin_inff();
      auto limit = [&](int bit, float v, float none) {
        return __builtin_bit_cast(float, uni(__builtin_bit_cast(int, (cmask & bit) ? v : none)));
      };
      // clamps as an unconditional median of three against +-inf (with lo > hi every value becomes hi once lo is lowered to
      // it), the activation as a compile-time constant of the pass: per-element decisions would double this code
      const float g_hi = limit(MOE_CLAMP_GATE_HI, a.clamp[0], inf);
      const float g_lo = limit(MOE_CLAMP_GATE_LO, fminf(a.clamp[1], g_hi), -inf);
      const float u_hi = limit(MOE_CLAMP_UP_HI, a.clamp[2], inf);
      const float u_lo = limit(MOE_CLAMP_UP_LO, fminf(a.clamp[3], u_hi), -inf);
      auto table = [&](const float* t, float (&v)[4]) {
        const float4 x = *(const float4*)t;
        v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
      };
      // bias (and scales) of the lane's four columns of tile pair t
      struct PairTab {
        float bg[4], bu[4], sg[4], su[4];
      };
      auto pair_tab = [&](int t) {
        const Piece p = piece_at(wn, 2 * t, g_e);
        const int col = p.q * 32 + p.cl * 4;
        PairTab r;
        table(s_bias[buf] + col, r.bg);
        table(s_bias[buf] + 128 + col, r.bu);
        if constexpr (ROW8) {
          table(s_wsc[buf] + col, r.sg);
          table(s_wsc[buf] + 128 + col, r.su);
        }
        return r;
      };
      const int tI = tw.tile_tI(cur), p0 = tw.tile_p0(cur), Pt = tw.tile_Pt(cur);
      // results: MX rows of bytes, bf16 or fp32 rows; rows past the chunk's last are dropped by the range check
      const int y_rowb = uni(SCALED ? (int)a.y_stride : BF16 ? (int)(a.y_stride * 2) : (int)(a.y32_stride * 4));
      const uint8_t* ybase = SCALED || BF16 ? (const uint8_t*)a.Yq : (const uint8_t*)a.Y32;
      const v4i rdy = make_rsrc(ybase + (int64_t)cur.slot0 * y_rowb, (uint32_t)(cur.nrows * y_rowb));
      const int ys_rowb = uni((int)a.ys_stride);
      const v4i rdys = make_rsrc(SCALED ? (const void*)(a.Ys + (int64_t)cur.slot0 * ys_rowb) : (const void*)a.tp2id,
                                 SCALED ? (uint32_t)(cur.nrows * ys_rowb) : 0u);
      const int pl = p0 + 16 * wn + 4 * g_e;  // MX: the lane's first partition
      const int p_live = pl < Pt ? -1 : 0;    // ... past the last one of a short tile: zeros, whatever the columns hold
      const uint32_t yq_voff = (uint32_t)(st_row0 * y_rowb + tI * 512 + (p0 + 16 * wn) * 4 + st_piece * 16);
      // (the scale byte of a block is stored by the even one of its two lane groups; the other's store is out of range)
      const uint32_t ys_voff = (g_e & 1) ? 0xffffffffu : (uint32_t)(row0 * ys_rowb + tI * 16 + (pl >> 3));
      // dense kinds: natural column of the lane's first value of quarter 2 wn + j
      auto nat_col = [&](int j) { return tI * 512 + (2 * wn + j) * Pt + p0 + (BF16 ? 8 : 4) * g_e; };
      // Activation checkpoint [N, 2, I, B] (bwmm_shard_on_I.py:160-176), bf16 kind: gate / up projections after scale, bias and
      // clamp, transposed, ahead of the results' pass.  Up to 64 of the wave's rows x a quarter's 32 columns at a time go through
      // its 4 KB of LDS, column by column, and leave as 16-byte pieces of 8 rows, eight of them side by side (in blocks of a
      // multiple of 8 rows; row by row otherwise).  (Stored from the registers 4 bytes at a time, in every activation's copy of
      // the results' pass: a layer of 1024 tokens, top-4 of 8 experts of H = 3072, I = 2048 243 us, now 241, and half of this
      // file's compile time; without streaming stores 247.)  A block's gate or up half is less than 4 GiB (the call's
      // intermediate rows are), so 32 bits hold an offset inside a half, and which half is a matter of 64 bits.
      auto ckpt_pass = [&]() {
        if constexpr (BF16) {
          const uint32_t ck_B = (uint32_t)a.ckpt_B, ck_half = (uint32_t)a.ckpt_I * ck_B * 2u;  // bytes
          const bool whole = (ck_B & 7) == 0 && (uni((int)(uintptr_t)a.ckpt) & 15) == 0;
          static_for<0, 2>([&](auto j_) {
            constexpr int j = decltype(j_)::value;
            const PairTab tab[2] = {pair_tab(2 * j), pair_tab(2 * j + 1)};
            const int col0 = tI * 512 + (2 * wn + j) * Pt + p0;  // the quarter's first column
            static_for<0, (RT + 3) / 4>([&](auto grp_) {
              constexpr int r0 = 4 * decltype(grp_)::value, nr = RT - r0 < 4 ? RT - r0 : 4;
              if ((wm * RT + r0) * 16 >= cur.nrows) return;
              // the lane's piece when they leave: column 8 k + lane / 8, rows 8 (lane % 8) ..
              const int unit = lane_e & 7, row = (wm * RT + r0) * 16 + 8 * unit;
              const uint32_t slot = (uint32_t)(cur.slot0 + row);
              const int rows = unit < 2 * nr ? cur.nrows - row : 0;  // of the piece, rows that exist (8 and more: all)
              static_for<0, 2>([&](auto gu_) {
                constexpr int gu = decltype(gu_)::value;
                const float lo = gu ? u_lo : g_lo, hi = gu ? u_hi : g_hi;
                static_for<0, nr>([&](auto i_) {
                  constexpr int i = decltype(i_)::value;
                  const float rs = s_rs[buf][row0 + (r0 + i) * 16];
                  float v[8];  // columns 8 g_e .. 8 g_e + 7 of the quarter
                  static_for<0, 2>([&](auto h_) {
                    constexpr int h = decltype(h_)::value;
                    float x[4];
                    acc_of(std::integral_constant<int, r0 + i>{}, std::integral_constant<int, 2 * (2 * j + h) + gu>{}, x);
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                      v[4 * h + r] = __builtin_amdgcn_fmed3f((x[r] * (gu ? tab[h].su : tab[h].sg)[r]) * rs + (gu ? tab[h].bu : tab[h].bg)[r], lo, hi);
                  });
                  // neighbouring lanes hold neighbouring rows: the even one takes the first four columns for both, the odd one
                  // the last four
                  const int odd = c_e & 1;
#pragma unroll
                  for (int k = 0; k < 4; ++k) {
                    const float own = odd ? v[4 + k] : v[k], give = odd ? v[k] : v[4 + k];
                    const float got = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, give), 0xb1 /* quad_perm 1 0 3 2 */, 0xf, 0xf, true));
                    const int col = 8 * g_e + 4 * odd + k, u = (2 * i + (c_e >> 3)) ^ (2 * g_e + odd);
                    *(uint32_t*)(ex + col * 128 + u * 16 + ((c_e >> 1) & 3) * 4) = odd ? pack2_bf16(got, own) : pack2_bf16(own, got);
                  }
                });
                asm volatile("" ::: "memory");
                v4i d[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                  const int col = 8 * k + (lane_e >> 3);
                  d[k] = *(const v4i*)(ex + col * 128 + (unit ^ (col >> 2)) * 16);
                }
                const int ccol = col0 + (lane_e >> 3);
                if (whole && rows >= 8) {
                  const uint32_t n = slot / ck_B, rr = slot - n * ck_B;
                  uint8_t* const at = (uint8_t*)a.ckpt + (uint64_t)(2u * n + gu) * ck_half + ((uint32_t)ccol * ck_B + rr) * 2u;
#pragma unroll
                  for (int k = 0; k < 4; ++k)
                    if (ccol + 8 * k < (int)a.ckpt_I) __builtin_nontemporal_store(d[k], (v4i*)(at + (uint32_t)(8 * k) * ck_B * 2u));
                } else {
#pragma clang loop unroll(disable)
                  for (int r = 0; r < (rows < 8 ? rows : 8); ++r) {
                    const uint32_t n = (slot + r) / ck_B, rr = slot + r - n * ck_B;
                    uint8_t* const at = (uint8_t*)a.ckpt + (uint64_t)(2u * n + gu) * ck_half + ((uint32_t)ccol * ck_B + rr) * 2u;
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                      const int w01 = (r & 2) ? d[k][1] : d[k][0], w23 = (r & 2) ? d[k][3] : d[k][2];
                      const uint32_t word = (uint32_t)((r & 4) ? w23 : w01) >> (16 * (r & 1));
                      if (ccol + 8 * k < (int)a.ckpt_I) *(uint16_t*)(at + (uint32_t)(8 * k) * ck_B * 2u) = (uint16_t)word;
                    }
                  }
                }
                asm volatile("" ::: "memory");
              });
            });
          });
        }
      };
      auto passes = [&](auto act_, auto plain_) {
        constexpr int ACT = decltype(act_)::value;
        constexpr bool PLAIN = decltype(plain_)::value;
        // gate and up of a tile pair, scaled, biased and clamped
        auto gate_up = [&](auto rt_, auto t_, const PairTab& tab, float rs, float (&gg)[4], float (&uu)[4]) {
          constexpr int t = decltype(t_)::value;
          float gv[4], uv[4];
          acc_of(rt_, std::integral_constant<int, 2 * t>{}, gv);
          acc_of(rt_, std::integral_constant<int, 2 * t + 1>{}, uv);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            if constexpr (ROW8 && !(BF16 && PLAIN)) {
              gv[r] = (gv[r] * tab.sg[r]) * rs;
              uv[r] = (uv[r] * tab.su[r]) * rs;
            }
            gg[r] = PLAIN ? gv[r] : __builtin_amdgcn_fmed3f(gv[r] + tab.bg[r], g_lo, g_hi);
            uu[r] = PLAIN ? uv[r] : __builtin_amdgcn_fmed3f(uv[r] + tab.bu[r], u_lo, u_hi);
          }
        };
        if constexpr (SCALED) {
          PairTab tab[4];
          if constexpr (!PLAIN)
#pragma unroll
            for (int t = 0; t < 4; ++t) tab[t] = pair_tab(t);
          v4i ex_o[NST];
          static_for<0, RT>([&](auto rt_) {
            constexpr int rt = decltype(rt_)::value;
            float y[4][4];
            static_for<0, 4>([&](auto t_) {
              constexpr int t = decltype(t_)::value;
              float gg[4], uu[4];
              gate_up(rt_, t_, tab[t], 1.f, gg, uu);
#pragma unroll
              for (int r = 0; r < 4; ++r) y[t][r] = act_apply(gg[r], ACT) * uu[r];
            });
            // MX block: 8 partitions x 4 quarters of a row = the lane's 16 values and the 16 of its neighbour group's lane
            float am = 0.f;
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
              for (int r = 0; r < 4; ++r) am = fmaxf(am, fabsf(y[t][r]));
            am = fmaxf(am, __shfl_xor(am, 16, 64));
            const uint32_t sb = mx_scale_byte(am);
            const float is = mx_inv_scale(sb);
            v4i o;
#pragma unroll
            for (int r = 0; r < 4; ++r)
              o[r] = (int)pack4_e4m3(clip448(y[0][r] * is), clip448(y[1][r] * is), clip448(y[2][r] * is), clip448(y[3][r] * is)) & p_live;
            // (the rows before are stored while these values wait for theirs)
            if constexpr (rt > 0) st_b128_plain(ex_o[0], yq_voff, rdy, (rt - 1) * 16 * y_rowb);
            ex_put(g_e, o);
            ex_get(ex_o);
            st_b8((int)sb & p_live, ys_voff, rdys, rt * 16 * ys_rowb);
            spread(rt_);
          });
          st_b128_plain(ex_o[0], yq_voff, rdy, (RT - 1) * 16 * y_rowb);
        } else {
          static_for<0, 2>([&](auto j_) {  // quarter 2 wn + j: tile pairs 2 j and 2 j + 1
            constexpr int j = decltype(j_)::value;
            const PairTab tab[2] = {pair_tab(2 * j), pair_tab(2 * j + 1)};
            int y_live[4];  // bf16: columns that only pad the weights go out as zeros whatever they hold
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const int n = (int)a.I_tab - (nat_col(j) + 2 * k);
              y_live[k] = n >= 2 ? -1 : n == 1 ? 0xffff : 0;
            }
            constexpr int ES = BF16 ? 2 : 4;
            const int col0 = tI * 512 + (2 * wn + j) * Pt + p0;  // the quarter's first column
            const uint32_t y_voff = (uint32_t)(st_row0 * y_rowb + col0 * ES + st_piece * 16);
            v4i ex_o[NST];
            auto store = [&](int rt) {
#pragma unroll
              for (int k = 0; k < NST; ++k) st_b128(ex_o[k], y_voff, rdy, (rt * 16 + k * (64 / PIECES)) * y_rowb);
            };
            static_for<0, RT>([&](auto rt_) {
              constexpr int rt = decltype(rt_)::value;
              const float rs = s_rs[buf][row0 + rt * 16];
              float gg[2][4], uu[2][4], y[2][4];
              static_for<0, 2>([&](auto h_) {
                constexpr int h = decltype(h_)::value;
                gate_up(rt_, std::integral_constant<int, 2 * j + h>{}, tab[h], rs, gg[h], uu[h]);
#pragma unroll
                for (int r = 0; r < 4; ++r) y[h][r] = act_apply(gg[h][r], ACT) * uu[h][r];
              });
              if constexpr (BF16) {
                const v4i o = {pack2(y[0][0], y[0][1]) & y_live[0], pack2(y[0][2], y[0][3]) & y_live[1],
                               pack2(y[1][0], y[1][1]) & y_live[2], pack2(y[1][2], y[1][3]) & y_live[3]};
                if constexpr (rt > 0) store(rt - 1);
                ex_put(g_e, o);
              } else {
                if constexpr (rt > 0) store(rt - 1);
#pragma unroll
                for (int h = 0; h < 2; ++h)
                  ex_put(4 * h + g_e, (v4i){__builtin_bit_cast(int, y[h][0]), __builtin_bit_cast(int, y[h][1]),
                                            __builtin_bit_cast(int, y[h][2]), __builtin_bit_cast(int, y[h][3])});
              }
              ex_get(ex_o);
              spread(std::integral_constant<int, j * RT + rt>{});
            });
            store(RT - 1);
          });
        }
      };
      // (the plain form, without bias and clamps, exists for SiLU alone: every instance of this code lengthens the build)
      // (bf16: nor scales; a row without a token is zeros then as it is)
      const bool pre = a.scaling_mode == MOE_SCALE_PRE || a.scaling_mode == MOE_SCALE_PRE_DELAYED;
      const bool plain = cmask == 0 && a.bias == nullptr && (!BF16 || (a.w_cscale == nullptr && !pre));
      if (BF16 && a.ckpt != nullptr) ckpt_pass();
      switch (a.act_fn) {
        case MOE_ACT_SILU:
          if (plain) passes(std::integral_constant<int, MOE_ACT_SILU>{}, std::true_type{});
          else passes(std::integral_constant<int, MOE_ACT_SILU>{}, std::false_type{});
          break;
        case MOE_ACT_GELU: passes(std::integral_constant<int, MOE_ACT_GELU>{}, std::false_type{}); break;
        case MOE_ACT_GELU_TANH: passes(std::integral_constant<int, MOE_ACT_GELU_TANH>{}, std::false_type{}); break;
        default: passes(std::integral_constant<int, MOE_ACT_SWISH>{}, std::false_type{}); break;
      }
    } else {
      const bool post = a.scaling_mode == MOE_SCALE_POST;
      const int rowb = uni((int)(a.H * 2));
      // rows past the chunk's last are dropped by the range check (rows of padding slots inside the chunk are written:
      // nothing reads them)
      const v4i rd = make_rsrc(a.D + (int64_t)cur.slot0 * a.H, (uint32_t)((int64_t)cur.nrows * a.H * 2));
      // bf16 kind: the down checkpoint [N, B, H] = [slots, H] takes the same rows ahead of the affinity
      const v4i rdc = make_rsrc((BF16 ? a.ckpt : a.D) + (int64_t)cur.slot0 * a.H, (uint32_t)((int64_t)cur.nrows * a.H * 2));
      const int lcol = 128 * wn + (FP4 ? 4 : 8) * g_e;  // the lane's first column of tile pair 0 within the tile
      constexpr int HI = FP4 ? 16 : 4;                  // ... of the pair's second tile behind that of its first
      auto put = [&](int t, const v4i& o) {
        if constexpr (FP4) {
#pragma unroll
          for (int h = 0; h < 2; ++h)
            *(v2i*)(ex_w + (((4 * t + 2 * h + (g_e >> 1)) ^ c_e) & 15) * 16 + (g_e & 1) * 8) = (v2i){o[2 * h], o[2 * h + 1]};
        } else {
          ex_put(4 * t + g_e, o);
        }
      };
      const uint32_t d_voff = (uint32_t)(st_row0 * rowb) + (uint32_t)(((int)tw.tile_h0(cur) + 128 * wn) * 2 + st_piece * 16);
      float affs[RT], rss[RT];
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        affs[i] = post ? s_aff[buf][row0 + i * 16] : 1.f;
        if constexpr (ROW8) rss[i] = s_rs[buf][row0 + i * 16];
      }
      // (PLAIN: no bias and, bf16, no scales, what most layers are; CKPT: the bf16 kind's checkpoint is written)
      auto passes = [&](auto plain_, auto ckpt_) {
        constexpr bool PLAIN = decltype(plain_)::value, CKPT = decltype(ckpt_)::value;
        float bd[4][8], sd[4][8];
        if constexpr (!PLAIN || (ROW8 && !BF16)) {
#pragma unroll
          for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int k = 0; k < 8; k += 4) {
              const float4 vb = *(const float4*)(s_bias[buf] + lcol + 32 * t + (k ? HI : 0));
              bd[t][k] = vb.x; bd[t][k + 1] = vb.y; bd[t][k + 2] = vb.z; bd[t][k + 3] = vb.w;
              if constexpr (ROW8) {
                const float4 vs = *(const float4*)(s_wsc[buf] + lcol + 32 * t + (k ? HI : 0));
                sd[t][k] = vs.x; sd[t][k + 1] = vs.y; sd[t][k + 2] = vs.z; sd[t][k + 3] = vs.w;
              }
            }
        }
        v4i ex_o[NST];
        auto store = [&](int rt, const v4i& d) {
#pragma unroll
          for (int k = 0; k < NST; ++k) st_b128(ex_o[k], d_voff, d, (rt * 16 + k * (64 / PIECES)) * rowb);
        };
        static_for<0, RT>([&](auto rt_) {
          constexpr int rt = decltype(rt_)::value;
          v4i o[4], oc[4];
          static_for<0, 4>([&](auto t_) {
            constexpr int t = decltype(t_)::value;
            float lo[4], hi[4], v[8];
            acc_of(rt_, std::integral_constant<int, 2 * t>{}, lo);
            acc_of(rt_, std::integral_constant<int, 2 * t + 1>{}, hi);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
              float x = k < 4 ? lo[k & 3] : hi[k & 3];
              if constexpr (ROW8 && !(BF16 && PLAIN)) x = (x * sd[t][k]) * rss[rt];
              v[k] = PLAIN ? x : x + bd[t][k];
            }
            if constexpr (CKPT) oc[t] = (v4i){pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]), pack2(v[6], v[7])};
            o[t] = (v4i){pack2(v[0] * affs[rt], v[1] * affs[rt]), pack2(v[2] * affs[rt], v[3] * affs[rt]),
                         pack2(v[4] * affs[rt], v[5] * affs[rt]), pack2(v[6] * affs[rt], v[7] * affs[rt])};
          });
          // (the rows before are stored while these values wait for theirs)
          if constexpr (rt > 0) store(rt - 1, rd);
          if constexpr (CKPT) {
#pragma unroll
            for (int t = 0; t < 4; ++t) put(t, oc[t]);
            ex_get(ex_o);
            store(rt, rdc);
          }
#pragma unroll
          for (int t = 0; t < 4; ++t) put(t, o[t]);
          ex_get(ex_o);
          spread(rt_);
        });
        store(RT - 1, rd);
      };
      const bool plain = a.bias == nullptr && (!BF16 || a.w_cscale == nullptr);
      if constexpr (BF16) {
        if (a.ckpt != nullptr) passes(std::false_type{}, std::true_type{});
        else if (plain) passes(std::true_type{}, std::false_type{});
        else passes(std::false_type{}, std::false_type{});
      } else {
        if (plain) passes(std::true_type{}, std::false_type{});
        else passes(std::false_type{}, std::false_type{});
      }
    }
    tile_live = -1;

    // ---- hand over to the next tile -----------------------------------------------------------------------------
    // The loads of the next tile's first slice and the small loads land here (the latter may be used from here on); the
    // stores drain under the next tile's first slice, whose B2 waits for all of them.
    zero_accumulators();
    if (!have_next) {
      tw.all_loads_landed(ids_nn, aff_n, bias_n, rs_n, wsc_n);
      break;
    }
    const bool have_n3 = Ln + run.W2 < run.end;
    const MxTile n3 = tw.tile_at(have_n3 ? Ln + run.W2 : L);
    tw.template loads_landed<OUT>(ids_nn, aff_n, bias_n, rs_n, wsc_n);
    if (STAGE == 2) tw.aff_put(nxt.e, buf ^ 1, aff_n);
    tw.rs_put(nxt.e, buf ^ 1, rs_n, aff_n);
    tw.bias_put(nxt, buf ^ 1, bias_n);
    tw.wsc_put(nxt, buf ^ 1, wsc_n);
    if (have_nn) tw.ids_put(buf, nn.nrows, ids_nn);  // the table of the tile that has just ended
    cur = nxt;
    nxt = nn;
    nn = n3;
    L = Ln;
    step = run.W2 - step;
    Ln += step;
    have_next = have_nn;
    have_nn = have_n3;
    buf ^= 1;
  }
  step = run.W2 - step;
  return Ln;
}

}  // namespace moe
