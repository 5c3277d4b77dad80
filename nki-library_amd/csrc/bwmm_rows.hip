// Blockwise expert GEMMs for launches with few rows per expert (decode batches, short prompts) on gfx950: the operands,
// layouts and epilogues of the large-tile kernels (bwmm_mx.hip), another split of the work.
//
// What bounds these launches is the stream of the expert weights (a 16-row tile multiplies a weight byte 16 times, a
// 256-row tile 256 times).  The large-tile kernel gives a CU one workgroup of four waves that walk a tile's K slices in
// step: CUs stay without a tile when experts x column tiles are fewer than CUs (one token of 8 experts of H = 7168,
// I = 2048: 128 of 256), and every tile pays its prologue and epilogue alone on its CU.  Here
//   * the waves of a workgroup split K between them (slice ks belongs to wave ks mod KP) and do not meet before the end
//     of the K loop: no barrier and no LDS in the loop, both operands straight from memory into MFMA operand registers,
//     two slices of loads in flight per wave;
//   * a workgroup owns few columns: 64 or 128 where columns are independent (down stage, bf16 and fp8-row gate/up), half
//     a column tile for the MX gate/up stage, whose re-quantisation blocks take 8 partitions of all four quarters of an
//     intermediate tile; four waves per workgroup (eight for MX gate/up), so that a CU holds one or two of them and one
//     streams while the other starts or ends;
//   * the partial sums meet in LDS once, and every thread finishes a few results.
// A wave is held to 256 registers: with 128 the K loop's two slices of weights spill, and the launch is slower than the
// large-tile kernel's.
// Measured (gate/up + down, large-tile kernel -> this one): one token, 8 MXFP8 experts of H = 7168, I = 2048:
// 58 + 29 -> 49 + 24 us (363 MB in all: 4.9 and 5.0 TB/s);
// 20 tokens, 128 bf16 experts of H = 2048, I = 768: 117 + 54 -> 91 + 48 us (6.2 TB/s); 256 tokens, 8 bf16 experts of
// H = 512, I = 1024: 21 + 23 -> 15 + 17 us.
// A chunk with more rows than the instance multiplies at once (MT row tiles of 16) is walked in passes that stream the
// weights again: right for any table, meant for the few-rows case (see mx_rows_fits).
#include <type_traits>

#include "bwmm.hpp"

namespace moe {

namespace {

typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ int uni32(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ rsrc_t rsrc_of(const void* p, uint32_t bytes) {
  const uint64_t addr = (uint64_t)p;
  const uint64_t u = (uint64_t)(uint32_t)uni32((int)(uint32_t)addr) | ((uint64_t)(uint32_t)uni32((int)(uint32_t)(addr >> 32)) << 32);
  return __builtin_amdgcn_make_buffer_rsrc((void*)u, 0, (int)uni32((int)bytes), 0x00020000);
}
constexpr int AUX_NT = 2;  // non-temporal: the weights of a launch like this are read once

__device__ __forceinline__ v4i mk4(const v8i& x, int h) { return h ? (v4i){x[4], x[5], x[6], x[7]} : (v4i){x[0], x[1], x[2], x[3]}; }

}  // namespace

template <int STAGE, int WFMT, int MT, int CGT, int KP>
struct RowsCfg {
  static constexpr bool BF16 = WFMT == MX_WFMT_BF16;
  static constexpr bool ROW8 = WFMT == MX_WFMT_ROW8 || BF16;
  static constexpr bool FP4 = WFMT == MX_WFMT_E2M1;
  // groups of 64 columns per workgroup (a wave multiplies one).  MX gate/up: 16 partitions x 4 quarters, gate and up, i.e.
  // half a column tile of the large-tile kernel; group h holds quarters 2h and 2h + 1.  Otherwise: 64 columns of a tile.
  static constexpr bool HALF = STAGE == 1 && !ROW8;
  static constexpr int CG = HALF ? 2 : CGT;
  static constexpr int NW = CG * KP;                         // waves
  static constexpr int ROWS = 16 * MT;
  static constexpr int PITCH = CG * 64 + 4;                  // floats per row of partial sums in LDS
  static constexpr int LDS = KP * ROWS * PITCH * 4;
};

// KTAIL: MX down stage whose K may end inside the last slice (an instance of its own: the offsets that it needs per slice
// cost the one-token launch half a microsecond)
template <int STAGE, int WFMT, int MT, int CGT, int KP, bool KTAIL>
__global__ __launch_bounds__(64 * (RowsCfg<STAGE, WFMT, MT, CGT, KP>::NW))
__attribute__((amdgpu_waves_per_eu(2, 8))) void mx_rows_kernel(const MxArgs a) {
  using Cfg = RowsCfg<STAGE, WFMT, MT, CGT, KP>;
  constexpr bool BF16 = Cfg::BF16, ROW8 = Cfg::ROW8, FP4 = Cfg::FP4, SCALED = !ROW8;
  constexpr int CG = Cfg::CG, NTHR = 64 * Cfg::NW, ROWS = Cfg::ROWS, PITCH = Cfg::PITCH;
  extern __shared__ __attribute__((aligned(16))) float s_part[];  // [KP][ROWS][PITCH]
  __shared__ float s_aff[ROWS], s_rs[ROWS];

  __shared__ long long s_clk[2];  // (start of the launch, see MxArgs::clk; the K loop has no scalar registers to spare)
  const int tid = threadIdx.x, lane = tid & 63;
  if (a.clk && blockIdx.x == 0 && tid == 0) {
    s_clk[0] = clock64();
    s_clk[1] = wall_clock64();
  }
  const int w = uni32(tid >> 6);
  const int cg = w % CG, kp = w / CG;
  const int c = lane & 15, g = lane >> 4;
  const int64_t nH = a.H / 512;
  // the lane's four neighbouring columns: gate or up (gu), first column within the group's 32 (16: HALF) partitions; HALF:
  // the lane's quarter is 2 cg + (c >> 3)
  constexpr bool HALF = Cfg::HALF;
  const int gu = (STAGE == 1) ? (HALF ? (c >> 2) & 1 : c >> 3) : 0;
  const int cl = HALF ? (c & 3) : (STAGE == 1) ? (c & 7) : c;

  int nks;
  if (STAGE == 1) nks = (int)(a.H / 128);
  else nks = (int)mx_col_tiles(a.I);
  // K ends behind partition nP - 1 counted through all slices (whole MX blocks of
  // 8); a load of partitions past that is aimed past the end of the expert's weights (less than 2^31 bytes) and returns zeros
  // (where even the first partition of a load does not exist: through a descriptor of zero records)
  static_assert(!KTAIL || (STAGE == 2 && SCALED), "the other stages' K are whole slices");
  constexpr uint32_t PAST_END = 0x80000000u;
  const int nP = (int)(a.I >> 2);

  // weight addressing: as in mx_gemm_tiles (same layouts, one wave per 64 columns)
  constexpr int ES = FP4 ? 2 : 4, GROWS = FP4 ? 8 : 4;
  const int64_t w_pstride = (STAGE == 1) ? 2 * nH * a.I : (int64_t)a.nI * a.H;
  const int64_t w_tstride = (STAGE == 1) ? a.I : a.H;
  const bool pk = a.w_packed != 0;
  constexpr int PK_LANE = FP4 ? 8 : 16, PK_LOAD = 64 * PK_LANE, PK_WAVE = 8 * PK_LOAD, PK_SLICE = 4 * PK_WAVE;
  const int64_t w_expert_bytes = pk ? (int64_t)a.col_tiles * nks * PK_SLICE
                                    : (STAGE == 1) ? 128 * w_pstride * ES : (int64_t)a.pI * w_pstride * ES;
  const int64_t ws_expert = (STAGE == 1) ? 16 * w_pstride : (int64_t)((a.pI + 7) / 8) * w_pstride;

  typedef typename std::conditional<FP4, v2i, v4i>::type RawLoad;
  struct Slice {  // a slice's weights as loaded, with their scale bytes
    RawLoad b[8];
    int bs;
  };
  struct ASlice {  // and its activation fragments
    v4i a[MT][2];
    int as[MT];
  };

  constexpr int SUB = 4 / CG;  // items per column tile of 256
  const int n_items = uni32(*a.n_chunks) * a.col_tiles * SUB;
  // MX gate/up: neighbouring items (column groups of one expert) share the lines that hold the block scales, 16 bytes of a
  // line each, so every XCD takes a contiguous eighth of the items (workgroup ids go round the XCDs; the grid is a multiple
  // of 8): dealt round-robin, every XCD fetched nearly every such line (one token on 8 experts of H = 7168, I = 2048: 294
  // MB where 242 are needed, the layer 91 us; now 84).  Elsewhere nothing is shared, and round-robin | by XCD came out the
  // same within the spread of the runs (20 tokens on 128 bf16 experts of H = 2048, I = 768, gate/up + down: 95 + 49.7 |
  // 96 + 50.1 us; 16 on 64 fp8-row experts of 4096, 768: 48.2 + 30.1 | 48.6 + 29.4) but for the smallest: 256 tokens on 8 bf16
  // experts of 512, 1024: 17.4 + 18.2 | 16.7 + 19.4.  Those keep the order that deals neighbouring items to all XCDs.
  constexpr bool BY_XCD = STAGE == 1 && SCALED;
  const int xcd = blockIdx.x & 7;
  const int item0 = BY_XCD ? (int)((int64_t)n_items * xcd / 8) + (int)(blockIdx.x >> 3) : (int)blockIdx.x;
  const int item1 = BY_XCD ? (int)((int64_t)n_items * (xcd + 1) / 8) : n_items;
  const int item_step = BY_XCD ? (int)(gridDim.x >> 3) : (int)gridDim.x;
  for (int item = item0; item < item1; item += item_step) {
    const int per_chunk = a.col_tiles * SUB;
    const int ci = item / per_chunk, ct = item - ci * per_chunk;
    const int xt = ct / SUB, sub = ct - xt * SUB;
    const int slot0 = uni32(a.chunk_slot[ci]), nrows = uni32(a.chunk_rows[ci]), e = uni32(a.chunk_expert[ci]);
    const int tI = xt >> 2, p0 = (xt & 3) * 32;
    const int Pt = (int)((a.I - (int64_t)tI * 512 < 512 ? a.I - (int64_t)tI * 512 : 512) / 4);  // (gate/up)
    // first column of the workgroup's group, and the lane's offsets from it (HALF: the quarter is the lane's)
    const int q = HALF ? 2 * cg + (c >> 3) : sub * CG + cg;
    const int64_t colu = (STAGE == 1) ? (int64_t)tI * 512 + (HALF ? 16 * sub + p0 : (int64_t)q * Pt + p0) : (int64_t)xt * 256 + 64 * q;
    const int64_t lane_col = (STAGE == 1) ? (HALF ? (int64_t)q * Pt : 0) + gu * nH * a.I + 4 * cl : 4 * cl;
    // packed copies: the lane's place within a load (see mx_pack_lane) and, HALF, its quarter's block
    const int pl = HALF ? g * 16 + sub * 8 + gu * 4 + cl : (STAGE == 1) ? mx_pack_lane(lane) : lane;
    const uint32_t w_voff = pk ? (uint32_t)((HALF ? q * PK_WAVE : 0) + pl * PK_LANE) : (uint32_t)((GROWS * g * w_pstride + lane_col) * ES);
    const uint32_t s_voff = (uint32_t)(g * w_pstride + lane_col);
    // scalar byte offset of load i: one base and one step (the loads' partition rows are 0..3 and 16..19; 0..7 for
    // 4-bit weights), so that no table of offsets occupies scalar registers
    const int w_base = uni32(pk ? (xt * nks) * PK_SLICE + (HALF ? 0 : q * PK_WAVE) : (int)(colu * ES));
    const int s_base = uni32((int)colu);
    const int w_step = uni32(pk ? PK_LOAD : (int)(w_pstride * ES)), w_jump = uni32(pk ? 4 : 16);
    const uint8_t* Wp = (const uint8_t*)a.W + (int64_t)e * w_expert_bytes;
    const uint8_t* Sp = a.W_scale + (int64_t)e * ws_expert;

    for (int row0 = 0; row0 < nrows; row0 += ROWS) {
      // rows of this pass: affinities, row scales (read behind the barrier that ends the K loop)
      __syncthreads();  // (the results of the pass before have been read)
      for (int r = tid; r < ROWS; r += NTHR) {
        const int row = row0 + r, slot = slot0 + row;
        int id = (row < nrows) ? a.tp2id[slot] : -1;
        if (id < 0 || id >= a.n_real) id = -1;
        float af = 0.f;
        if (a.aff && id >= 0)
          af = a.aff_dtype == MOE_DT_BF16 ? bf16_bits_to_f32(((const uint16_t*)a.aff)[(int64_t)id * a.E + e])
                                          : ((const float*)a.aff)[(int64_t)id * a.E + e];
        s_aff[r] = af;
        if constexpr (ROW8) {
          float v = 1.f;
          if (STAGE == 1) {
            if (!BF16 && id >= 0) v = *(const float*)(a.A + (int64_t)id * a.a_stride + a.H);
            if (id < 0) v = 0.f;
            if ((a.scaling_mode == MOE_SCALE_PRE || a.scaling_mode == MOE_SCALE_PRE_DELAYED) && a.aff && id >= 0) v *= af;
          } else if (!BF16) {
            v = (row < nrows) ? a.a_rscale[slot] : 0.f;
          }
          s_rs[r] = v;
        }
      }
      // the lane's A rows; a row that does not exist points past the end of the table and loads as zeros
      uint32_t a_voff[MT], as_voff[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int row = row0 + 16 * m + c;
        int64_t r = a.a_rows;
        if (row < nrows) {
          if (STAGE == 1) {
            const int id = a.tp2id[slot0 + row];
            if (id >= 0 && id < a.n_real) r = id;
          } else {
            r = slot0 + row;
          }
        }
        a_voff[m] = (uint32_t)r * (uint32_t)a.a_stride + 16u * (uint32_t)g;
        if constexpr (SCALED) as_voff[m] = (uint32_t)((r < a.a_rows) ? r : 0) * (uint32_t)a.a_scale_stride + (uint32_t)g;
      }

      v4f acc[MT][4];
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[m][t] = (v4f){0.f, 0.f, 0.f, 0.f};

      // a slice behind the last one loads through descriptors of zero records: no traffic, zeros, no branch
      auto load_b = [&](Slice& s, int ks) {
        const bool live = ks < nks;
        const int kt = ks >> 2, pb = ks & 3;
        const rsrc_t rw = rsrc_of(Wp, live ? (uint32_t)w_expert_bytes : 0u);
        const int w_off = w_base + uni32(pk ? ks * PK_SLICE : (int)(((int64_t)(pb * 32) * w_pstride + (int64_t)kt * w_tstride) * ES));
        const uint32_t w_lo = (!KTAIL || ks * 32 + GROWS * g < nP) ? w_voff : PAST_END;
        const uint32_t w_hi = (!KTAIL || ks * 32 + 16 + GROWS * g < nP) ? w_voff : PAST_END;
        const rsrc_t rw_hi = (KTAIL && !FP4) ? rsrc_of(Wp, ks * 32 + 16 < nP ? (uint32_t)w_expert_bytes : 0u) : rw;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int soff = w_off + (FP4 ? i : (i < 4) ? i : w_jump + i - 4) * w_step;
          if constexpr (FP4) s.b[i] = __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(rw, w_lo, soff, AUX_NT));
          else s.b[i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(i < 4 ? rw : rw_hi, i < 4 ? w_lo : w_hi, soff, AUX_NT));
        }
        if constexpr (SCALED) {
          const rsrc_t rs = rsrc_of(Sp, live ? (uint32_t)ws_expert : 0u);
          s.bs = (int)__builtin_amdgcn_raw_buffer_load_b32(rs, (!KTAIL || ks * 32 + 8 * g < nP) ? s_voff : PAST_END, s_base + uni32((int)((int64_t)(pb * 4) * w_pstride + (int64_t)kt * w_tstride)), 0);
        }
      };
      auto load_a = [&](ASlice& s, int ks) {
        const bool live = ks < nks;
        const rsrc_t ra = rsrc_of(a.A, live ? (uint32_t)(a.a_rows * a.a_stride) : 0u);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          s.a[m][0] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(ra, a_voff[m], ks * 128, 0));
          s.a[m][1] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(ra, a_voff[m], ks * 128 + 64, 0));
          if constexpr (SCALED) {
            const rsrc_t rsa = rsrc_of(a.A_scale, live ? (uint32_t)(a.a_rows * a.a_scale_stride) : 0u);
            s.as[m] = (int)__builtin_amdgcn_raw_buffer_load_b8(rsa, as_voff[m], ks * 4, 0);
          }
        }
      };
      auto mul = [&](const Slice& s, const ASlice& x) {
        v8i bf[4];
        if constexpr (FP4) {
#pragma unroll
          for (int t = 0; t < 4; ++t) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const uint32_t lo = (uint32_t)s.b[2 * r][t >> 1], hi = (uint32_t)s.b[2 * r + 1][t >> 1];
              bf[t][r] = (int)__builtin_amdgcn_perm(hi, lo, (t & 1) ? 0x07060302u : 0x05040100u);
              bf[t][4 + r] = 0;
            }
          }
        } else {
#pragma unroll
          for (int r = 0; r < 8; ++r)
#pragma unroll
            for (int t = 0; t < 4; ++t) bf[t][r] = s.b[r][t];
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          if constexpr (BF16) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
              for (int h = 0; h < 2; ++h)
                acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, x.a[m][h]),
                                                                    __builtin_bit_cast(v8bf, mk4(bf[t], h)), acc[m][t], 0, 0, 0);
          } else {
            const v8i af = (v8i){x.a[m][0][0], x.a[m][0][1], x.a[m][0][2], x.a[m][0][3],
                                 x.a[m][1][0], x.a[m][1][1], x.a[m][1][2], x.a[m][1][3]};
            constexpr int BLGP = WFMT == MX_WFMT_E5M2 ? 1 : FP4 ? 4 : 0;
            const int sa = SCALED ? x.as[m] : 127, sb = SCALED ? s.bs : 0x7f7f7f7f;
            acc[m][0] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(af, bf[0], acc[m][0], 0, BLGP, 0, sa, 0, sb);
            acc[m][1] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(af, bf[1], acc[m][1], 0, BLGP, 0, sa, 1, sb);
            acc[m][2] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(af, bf[2], acc[m][2], 0, BLGP, 0, sa, 2, sb);
            acc[m][3] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(af, bf[3], acc[m][3], 0, BLGP, 0, sa, 3, sb);
          }
        }
      };
      // (four row tiles: one set of activation fragments, requested when the one before has been multiplied; two do not
      // fit the registers beside two slices of weights)
      constexpr bool ONE_A = MT == 4;
      Slice s0, s1;
      ASlice x0, x1;
      load_b(s0, kp);
      load_a(x0, kp);
#pragma clang loop unroll(disable)
      for (int ks = kp; ks < nks; ks += 2 * KP) {
        load_b(s1, ks + KP);
        if constexpr (!ONE_A) load_a(x1, ks + KP);
        mul(s0, x0);
        if constexpr (ONE_A) load_a(x0, ks + KP);
        load_b(s0, ks + 2 * KP);
        if constexpr (!ONE_A) load_a(x0, ks + 2 * KP);
        mul(s1, ONE_A ? x0 : x1);  // (zeros when there is no such slice)
        if constexpr (ONE_A) load_a(x0, ks + 2 * KP);
      }

      // ---- partial sums to LDS: [kp][row][64-column group][column], a lane's four columns side by side ----
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          *(float4*)(s_part + ((size_t)kp * ROWS + 16 * m + 4 * g + r) * PITCH + cg * 64 + 4 * c) =
              make_float4(acc[m][0][r], acc[m][1][r], acc[m][2][r], acc[m][3][r]);
      __syncthreads();

      auto bias_at = [&](int64_t i) {
        return a.bias_dtype == MOE_DT_BF16 ? bf16_bits_to_f32(((const uint16_t*)a.bias)[i]) : ((const float*)a.bias)[i];
      };
      auto part = [&](int r, int col) {
        float v = 0.f;
#pragma unroll
        for (int k = 0; k < KP; ++k) v += s_part[((size_t)k * ROWS + r) * PITCH + col];
        return v;
      };
      auto limit = [&](int bit, float v, float none) { return (a.clamp_mask & bit) ? v : none; };
      const float inf = __builtin_inff();
      const float g_hi = limit(MOE_CLAMP_GATE_HI, a.clamp[0], inf), g_lo = limit(MOE_CLAMP_GATE_LO, fminf(a.clamp[1], g_hi), -inf);
      const float u_hi = limit(MOE_CLAMP_UP_HI, a.clamp[2], inf), u_lo = limit(MOE_CLAMP_UP_LO, fminf(a.clamp[3], u_hi), -inf);
      auto gate_up = [&](float gv, float uv) {
        // (the medians of the large-tile kernels' epilogue, not minima and maxima: these would turn a NaN under an upper
        // clamp alone into that clamp; without clamps the values go through as they are)
        if (a.clamp_mask) {
          gv = __builtin_amdgcn_fmed3f(gv, g_lo, g_hi);
          uv = __builtin_amdgcn_fmed3f(uv, u_lo, u_hi);
        }
        return act_apply(gv, a.act_fn) * uv;
      };
      const int live_rows = (nrows - row0 < ROWS) ? nrows - row0 : ROWS;
      if constexpr (STAGE == 1 && !ROW8) {
        // thread = (row, partition): its four quarters are the four bytes of one dword of the down stage's row, and
        // eight neighbouring lanes hold one MX block
        for (int i = tid; i < live_rows * 16; i += NTHR) {
          const int r = i >> 4, pp = i & 15, p = p0 + 16 * sub + pp;
          float y[4], am = 0.f;
#pragma unroll
          for (int qq = 0; qq < 4; ++qq) {
            float gv = part(r, qq * 32 + pp), uv = part(r, qq * 32 + 16 + pp);
            if (a.bias && p < Pt) {
              const int64_t b0 = ((((int64_t)e * a.pI + p) * 2) * a.nI + tI) * 4 + qq;
              gv += bias_at(b0);
              uv += bias_at(b0 + (int64_t)a.nI * 4);
            }
            y[qq] = gate_up(gv, uv);
            am = fmaxf(am, fabsf(y[qq]));
          }
          am = fmaxf(am, __shfl_xor(am, 1, 64));
          am = fmaxf(am, __shfl_xor(am, 2, 64));
          am = fmaxf(am, __shfl_xor(am, 4, 64));
          const uint32_t sb = mx_scale_byte(am);
          const float is = mx_inv_scale(sb);
          const int64_t slot = slot0 + row0 + r;
          const uint32_t p_live = p < Pt ? ~0u : 0u;  // past the last partition of a short tile: zeros, whatever the columns hold
          *(uint32_t*)(a.Yq + slot * a.y_stride + tI * 512 + p * 4) =
              pack4_e4m3(clip448(y[0] * is), clip448(y[1] * is), clip448(y[2] * is), clip448(y[3] * is)) & p_live;
          if ((pp & 7) == 0) a.Ys[slot * a.ys_stride + tI * 16 + (p >> 3)] = (uint8_t)(sb & p_live);
        }
      } else if constexpr (STAGE == 1) {
        // thread = (row, two neighbouring columns)
        for (int i = tid; i < live_rows * 16 * CG; i += NTHR) {
          const int r = i / (16 * CG), k2 = i % (16 * CG), qq = k2 >> 4, j = (k2 & 15) * 2;
          const int64_t col = (int64_t)tI * 512 + (int64_t)(sub * CG + qq) * Pt + p0 + j;
          const float rs = s_rs[r];
          float y[2];
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            float gv = part(r, qq * 64 + j + k), uv = part(r, qq * 64 + 32 + j + k);
            float sg = 1.f, su = 1.f;
            const bool live = col + k < a.I_tab;  // (a column that only pads the weights is zero, also for a row with an infinity)
            if (a.w_cscale && live) {
              const float* ws = a.w_cscale + (a.cscale_experts > 1 ? (int64_t)e * 2 * a.I_tab : 0);
              sg = ws[col + k];
              su = ws[a.I_tab + col + k];
            }
            gv = (gv * sg) * rs;
            uv = (uv * su) * rs;
            if (a.bias && live) {
              gv += bias_at((int64_t)e * 2 * a.I_tab + col + k);
              uv += bias_at((int64_t)e * 2 * a.I_tab + a.I_tab + col + k);
            }
            y[k] = live ? gate_up(gv, uv) : 0.f;
          }
          const int64_t slot = slot0 + row0 + r;
          if constexpr (BF16) *(uint32_t*)((uint16_t*)a.Yq + slot * a.y_stride + col) = pack2_bf16(y[0], y[1]);
          else *(float2*)(a.Y32 + slot * a.y32_stride + col) = make_float2(y[0], y[1]);
        }
      } else {
        const bool post = a.scaling_mode == MOE_SCALE_POST;
        for (int i = tid; i < live_rows * 32 * CG; i += NTHR) {
          const int r = i / (32 * CG), j = (i % (32 * CG)) * 2;
          const int64_t h = (int64_t)xt * 256 + 64 * (sub * CG) + j;
          float d[2];
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            d[k] = part(r, j + k);
            if constexpr (ROW8) {
              const float sd = a.w_cscale ? a.w_cscale[(a.cscale_experts > 1 ? (int64_t)e * a.H : 0) + h + k] : 1.f;
              d[k] = (d[k] * sd) * s_rs[r];
            }
            if (a.bias) d[k] += bias_at((int64_t)e * a.H + h + k);
            if (post) d[k] *= s_aff[r];
          }
          *(uint32_t*)(a.D + (int64_t)(slot0 + row0 + r) * a.H + h) = pack2_bf16(d[0], d[1]);
        }
      }
    }
  }
  if (a.clk && blockIdx.x == 0 && tid == 0) {
    a.clk[0] = clock64() - s_clk[0];
    a.clk[1] = wall_clock64() - s_clk[1];
  }
}

// the kinds that have an instance of four row tiles
template <int STAGE, int WFMT>
constexpr bool ROWS_MT4 = WFMT == MX_WFMT_BF16 || (STAGE == 2 && (WFMT == MX_WFMT_ROW8 || WFMT == MX_WFMT_E2M1));

// One workgroup per item, as many as the GPU holds at a time (the waves per SIMD that mx_rows_kernel is compiled for);
// workgroups beyond the items end at once.
template <int STAGE, int WFMT, int MT, int CGT, int KP, bool KTAIL>
static int launch_instance(const MxArgs& m, int64_t max_chunks, int cus, hipStream_t s) {
  using Cfg = RowsCfg<STAGE, WFMT, MT, CGT, KP>;
  const int64_t items = max_chunks * m.col_tiles * (4 / Cfg::CG);
  const int64_t resident = (int64_t)cus * (8 / Cfg::NW);
  const unsigned grid = ((unsigned)(items < resident ? items : resident) + 7u) & ~7u;
  if (allow_lds<&mx_rows_kernel<STAGE, WFMT, MT, CGT, KP, KTAIL>>(Cfg::LDS) != hipSuccess) return MOE_E_LAUNCH;
  hipLaunchKernelGGL((mx_rows_kernel<STAGE, WFMT, MT, CGT, KP, KTAIL>), dim3(grid), dim3(64 * Cfg::NW), Cfg::LDS, s, m);
  MOE_CHECK_LAUNCH();
  return MOE_OK;
}
template <int STAGE, int WFMT, int MT, int CGT, int KP>
static int launch_one(const MxArgs& m, int64_t max_chunks, int cus, hipStream_t s) {
  if constexpr (STAGE == 2 && !RowsCfg<STAGE, WFMT, MT, CGT, KP>::ROW8)
    if (m.I % 128 != 0) return launch_instance<STAGE, WFMT, MT, CGT, KP, true>(m, max_chunks, cus, s);
  return launch_instance<STAGE, WFMT, MT, CGT, KP, false>(m, max_chunks, cus, s);
}

// Columns per workgroup.  64 (four waves on a quarter of K each) unless that leaves a second, partly filled round of
// workgroups that 128 (two waves each on half of K) avoids or, in the down stage with its short K loop, unless there are
// enough workgroups anyway.  `groups` = 64-column groups of the launch, 512 workgroups run at a time.  Measured, 64 | 128
// columns: gate/up of 8 fp8-row experts, I = 3584 (896 groups) 53 | 44 us; of 64 bf16 experts, I = 768 (1536 groups)
// 49 | 55 us; down of 8 bf16 experts, H = 2048 (256 groups) 25 | 30 us; of 32 MXFP8 experts, H = 7168 (3584 groups)
// 57 | 50 us; of 64 bf16 experts, H = 2048 (2048 groups) 39 | 33 us.
template <int STAGE, int WFMT, int MT>
static int launch_mt(const MxArgs& m, int64_t max_chunks, int cus, hipStream_t s) {
  const int64_t groups = max_chunks * m.col_tiles * 4, at_once = 2 * (int64_t)cus;
  constexpr bool HALF = RowsCfg<STAGE, WFMT, MT, 1, 4>::HALF;
  if constexpr (!HALF)
    if (groups > at_once && (STAGE == 2 || groups <= 2 * at_once)) return launch_one<STAGE, WFMT, MT, 2, 2>(m, max_chunks, cus, s);
  return launch_one<STAGE, WFMT, MT, 1, 4>(m, max_chunks, cus, s);
}

template <int STAGE, int WFMT>
static int launch_rows(const MxArgs& m, int64_t rows, int64_t max_chunks, int cus, hipStream_t s) {
  if (rows <= 16) return launch_mt<STAGE, WFMT, 1>(m, max_chunks, cus, s);
  if constexpr (ROWS_MT4<STAGE, WFMT>)
    if (rows > 32) return launch_mt<STAGE, WFMT, 4>(m, max_chunks, cus, s);
  if constexpr (STAGE == 1 && WFMT == MX_WFMT_E2M1) return MOE_E_BAD_ARG;  // (mx_rows_fits: up to 8 rows)
  else return launch_mt<STAGE, WFMT, 2>(m, max_chunks, cus, s);
}

// How many rows a launch holds is known from the number of tokens; how many experts they hit stands in the table, on the
// device: one of N >= E blocks is taken to hit all E, a shorter one so many per token as models of E experts route to.
// Times below are us between two events on the stream, large-tile kernel | this one.
//   MX gate/up.  A half column tile per CU and round: one round (128 tiles) beats the large-tile kernel's, from then on
//     both are bound by the stream, where the large tiles' longer runs are the better ones (8-bit weights) or the 8-byte
//     loads of this kernel's 4-bit weights by far the worse.  Up to four experts always: the large-tile kernel gives an
//     expert's tiles to one XCD.  8-bit, experts hit of H, I: 8 of 7168, 2048: 58 | 49; 16: 86 | 90; 57: 280 | 317; 8 of
//     5120, 1536: 51 | 31; 14: 52 | 57; 2 of 4096, 14336: 126 | 51; 8: 167 | 174.  4-bit: 8 of 7168, 2048: 47 | 50;
//     16: 52 | 90; 57: 166 | 314; 8 of 3072, 1536: 26 | 21; 15: 29 | 40; 3 of 4096, 14336: 94 | 73; 6: 100 | 139.  Between
//     one round and two the estimate decides (a low one for 8-bit weights, where a wrong choice costs 10 % at most, a high
//     one for 4-bit): over random shapes up to 32 (8) tokens the stage then takes 1.034 (1.012) times the better kernel's
//     time, the large-tile kernel 1.41 (1.29), this one 1.017 (1.12) with losses up to 1.29 (1.9).
//   Dense gate/up: up to 32 rows (fp8-row) or 64 (bf16), except a long K over many tiles (bf16, 64 experts of 7168, 2048,
//     16 rows: 667 | 695, 32: 702 | 754, 64: 706 | 775; of 5120, 1536, 16 rows: 277 | 239, 32: 307 | 329; 104 of 2048, 768,
//     32 rows: 127 | 113; 59 of 1024, 768, 64: 51 | 41; 8 of 4096, 1024, 64: 65 | 34.  fp8-row, 58 of 4096, 768, 16 rows:
//     85 | 64; 56 of 4096, 2048, 32: 177 | 185, 64: 192 | 215).
//   Down: up to 32 rows (MXFP8, 32 rows: 159 experts of 7168, 2048: 376 | 362; 32 of 3072, 1536: 42 | 31), up to 64 for
//     the kinds whose four row tiles fit the registers (bf16, 64 rows: 64 of 7168, 2048: 303 | 308; 128 of 2048, 768:
//     80 | 70); 4-bit ones there while the tiles are few (48 rows: 119 of 4096, 2048: 115 | 131; 59 of 2048, 6400: 81 | 104;
//     32 of 3072, 1536: 31 | 28).
//   bf16 beyond 64 rows, one pass of 64 on average, while the large-tile kernel has a tile for half of the CUs or less: 256
//     tokens over 8 experts, two of them each, of H = 512, I = 1024: gate/up 19 | 17, down 23 | 18; of H = 4096, I = 1024:
//     70 | 61 and 27 | 33; 384 tokens of the former: 21 | 20 and 25 | 21, not taken: a pass more per expert and falling.
//   (Every time with chunks of more than 64 rows, i.e. this paragraph and the table below, is of the present loop of
//     mx_wide.hpp.  Over 260 random shapes of up to 64 tokens, bf16 up to 256: gate/up 1.049 and down 1.016
//     times the better kernel's time, the large-tile kernels alone 1.67 and 1.72, this one alone 1.007 and 1.002.  What the
//     rule leaves is small launches that it still gives to the large tiles, MX kinds with 33 to 64 tokens over four experts
//     above all: 46 tokens of H = 2048, I = 512: 37 | 15 and 21 | 9.)
bool mx_rows_fits(int stage, int wfmt, const RowsCall& c) {
  const bool fp4 = wfmt == MX_WFMT_E2M1, bf16 = wfmt == MX_WFMT_BF16, mx = !bf16 && wfmt != MX_WFMT_ROW8;
  if (stage == 1 && mx) {
    if (c.rows > (fp4 ? 8 : 32)) return false;
    const int64_t per = c.E / (fp4 ? 4 : 16), hit = c.rows * (per < 1 ? 1 : per > 8 ? 8 : per);
    const bool some = c.N < c.E && hit < c.E;
    const int64_t experts = some ? hit : c.E, tiles = experts * c.col_tiles;
    return experts <= 4 || tiles <= 128 || (some && tiles < (fp4 ? 192 : 256));
  }
  if (c.rows <= 16) return true;
  if (stage == 1) {
    if (c.rows <= (bf16 ? 64 : 32)) return !(c.N >= c.E && c.H > 5120 && c.E * c.col_tiles > 512);
  } else {
    if (c.rows <= 32) return true;
    if (c.rows <= 64) return bf16 || wfmt == MX_WFMT_ROW8 || (fp4 && (c.N < c.E ? c.N : c.E) * c.col_tiles <= 384);
  }
  if (!bf16 || c.rows > 256 || c.col_tiles * c.max_chunks > 128) return false;
  // A table of N blocks is made for about (N - (E - 1)) * B routed rows.  One with fewer blocks than experts was cut by the
  // caller to what it holds, which may be whole blocks: several passes, worth it while the large-tile kernel has a chunk
  // for an XCD or less (gate/up, 7 blocks of 128 rows over H = 2048, I = 1024: 72 | 43; 4 of 256: 95 | 75; 16 of 256 over
  // H = 4096: 100 | 273).
  if (c.N < c.E) return c.max_chunks <= 8 || (c.B < c.rows ? c.B : c.rows) <= 64;
  return (c.N - (c.E - 1)) * c.B / c.E <= 64;
}

int launch_mx_rows(int stage, const MxArgs& m0, unsigned gx, int64_t max_chunks, int64_t rows, hipStream_t s) {
  if (gx == 0 || max_chunks == 0) return MOE_OK;
  MxArgs m = m0;
  m.col_tiles = (int32_t)gx;
  const int cus = device_cus();
  if (cus < 8) return MOE_E_LAUNCH;
  switch (m.wfmt) {
    case MX_WFMT_E4M3: return stage == 1 ? launch_rows<1, MX_WFMT_E4M3>(m, rows, max_chunks, cus, s) : launch_rows<2, MX_WFMT_E4M3>(m, rows, max_chunks, cus, s);
    case MX_WFMT_E5M2: return stage == 1 ? launch_rows<1, MX_WFMT_E5M2>(m, rows, max_chunks, cus, s) : launch_rows<2, MX_WFMT_E5M2>(m, rows, max_chunks, cus, s);
    case MX_WFMT_E2M1: return stage == 1 ? launch_rows<1, MX_WFMT_E2M1>(m, rows, max_chunks, cus, s) : launch_rows<2, MX_WFMT_E2M1>(m, rows, max_chunks, cus, s);
    case MX_WFMT_ROW8: return stage == 1 ? launch_rows<1, MX_WFMT_ROW8>(m, rows, max_chunks, cus, s) : launch_rows<2, MX_WFMT_ROW8>(m, rows, max_chunks, cus, s);
    case MX_WFMT_BF16: return stage == 1 ? launch_rows<1, MX_WFMT_BF16>(m, rows, max_chunks, cus, s) : launch_rows<2, MX_WFMT_BF16>(m, rows, max_chunks, cus, s);
    default: return MOE_E_BAD_ARG;
  }
}

}  // namespace moe
