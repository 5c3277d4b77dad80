// What the tile loops of the large-tile expert GEMMs share (bwmm_mx.hip: weights through registers, mx_wide.hpp: both
// operands through LDS): accumulators in fixed registers, loads and stores written as instructions, and the walk over a
// queue of tiles with the small per-tile tables (token ids, affinities, bias, scales).
#pragma once

#include <type_traits>

#include "bwmm.hpp"

namespace moe {

constexpr int MXT = 256;                     // threads
constexpr int MX_ROWS_MAX = CHUNK_ROWS_MAX;  // rows of the largest chunk (320)
constexpr int MXROW = 128;                   // LDS pitch of one staged activation row; 16-byte chunk ch of row r sits in
                                             // slot ch ^ (r & 7), which makes the fragment reads (16 rows x 4 chunks
                                             // per instruction) and the staging writes conflict free

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}
// The accumulators live in fixed accumulation registers that only the statements below name: tile
// (mt, nt) of a wave's 16 x 4 tiles is a[16 mt + 4 nt .. + 3].  They are not C++ values, so the
// compiler never moves, copies or spills them (it would do so without the wait that a read of an
// MFMA result needs: it does not know these statements as MFMAs).  Every accumulation register is
// declared clobbered at both ends of each K slice, so the compiler keeps nothing of its own there.
#define MX_A10(p) "a" #p "0", "a" #p "1", "a" #p "2", "a" #p "3", "a" #p "4", "a" #p "5", "a" #p "6", "a" #p "7", "a" #p "8", "a" #p "9"
#define MX_ALL_ACC                                                                                               \
  "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", MX_A10(1), MX_A10(2), MX_A10(3), MX_A10(4),        \
      MX_A10(5), MX_A10(6), MX_A10(7), MX_A10(8), MX_A10(9), MX_A10(10), MX_A10(11), MX_A10(12), MX_A10(13),     \
      MX_A10(14), MX_A10(15), MX_A10(16), MX_A10(17), MX_A10(18), MX_A10(19), MX_A10(20), MX_A10(21), MX_A10(22), \
      MX_A10(23), MX_A10(24), "a250", "a251", "a252", "a253", "a254", "a255"
__device__ __forceinline__ void acc_fence() { asm volatile("" ::: MX_ALL_ACC); }
template <int I>
__device__ __forceinline__ void acc_zero() {
  asm volatile("v_accvgpr_write_b32 a[%0], 0" : : "n"(I));
}
template <int I>
__device__ __forceinline__ float acc_get() {
  float x;
  asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(x) : "n"(I));
  return x;
}

// A vector memory instruction that reads a scalar register (descriptor, scalar offset) needs five wait states
// after a vector ALU instruction that wrote that register (v_readfirstlane, v_readlane: the compiler reloads
// spilled scalars with the latter right where they are used).  The compiler keeps that distance for instructions
// of its own; for the instructions written out in this file it cannot (it does not see which operands an inline
// statement reads when), so each of them carries the wait states itself.  They are issue slots in the shadow of
// the MFMAs between which the loads sit.
#define MX_SGPR_WAIT "s_nop 4\n\t"

// Raw buffer descriptor over [p, p + bytes): loads take a per-lane 32-bit byte offset (VGPR) plus a
// wave-uniform 32-bit byte offset (SGPR), which is exactly the shape of every address in this
// kernel, so no 64-bit per-lane pointer is ever formed.
// (The descriptor and the uniform offsets are passed through readfirstlane: 64-bit address
// arithmetic on uniform values is done by the vector ALU, and without the hint the compiler wraps
// every load in a loop that checks whether all lanes agree on the descriptor.)
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int uni(int64_t v) { return __builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ v4i make_rsrc(const void* p, uint32_t bytes) {
  const uint64_t addr = (uint64_t)p;
  v4i d;
  d[0] = uni((int)(uint32_t)addr);
  d[1] = uni((int)(uint32_t)(addr >> 32)) & 0xffff;  // stride 0: raw buffer
  d[2] = uni((int)bytes);
  d[3] = 0x00020000;
  return d;
}
// The K loop's loads are written as instructions, not builtins: the compiler orders the results of
// its own loads with a counter that completes in order, and places those waits as if every load it
// can see on any path had just been issued -- which with two alternating weight sets means waiting
// for the set that was only just requested.  Loads the compiler cannot see get no waits from it;
// the waits are placed by hand where the data is first used (vm_wait).  The destination is an
// in/out operand so that the load updates the variable's register in place.
// NT: non-temporal, for data that nobody will ask the L2 for again.
template <bool NT>
__device__ __forceinline__ void ld_b128(v4i& d, uint32_t voff, const v4i& rsrc, int soff) {
  if constexpr (NT)
    asm volatile(MX_SGPR_WAIT "buffer_load_dwordx4 %0, %1, %2, %3 offen nt" : "+v"(d) : "v"(voff), "s"(rsrc), "s"(soff) : "memory");
  else
    asm volatile(MX_SGPR_WAIT "buffer_load_dwordx4 %0, %1, %2, %3 offen" : "+v"(d) : "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}
__device__ __forceinline__ void st_b64(const v2i& d, uint32_t voff, const v4i& rsrc, int soff) {
  asm volatile(MX_SGPR_WAIT "buffer_store_dwordx2 %0, %1, %2, %3 offen nt" : : "v"(d), "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}
__device__ __forceinline__ void st_b128(const v4i& d, uint32_t voff, const v4i& rsrc, int soff) {
  asm volatile(MX_SGPR_WAIT "buffer_store_dwordx4 %0, %1, %2, %3 offen nt" : : "v"(d), "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}
// 16 bytes per lane straight into LDS at lds + 16 * lane (no destination registers).  The instruction takes its
// LDS base from M0, which is set in the same statement.  M0 is declared clobbered: the compiler warns that it
// does not save reserved registers around a statement, which is what is wanted here -- on this target it never
// carries a value in M0 from one instruction to the next (it writes M0 itself immediately before each instruction
// of its own that reads it), so there is nothing to save.
__device__ __forceinline__ void ld_lds_b128(uint32_t lds, uint32_t voff, const v4i& rsrc, int soff) {
  asm volatile(MX_SGPR_WAIT "s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               : : "s"(lds), "v"(voff), "s"(rsrc), "s"(soff) : "memory", "m0");
}
template <bool NT>
__device__ __forceinline__ void ld_b64(v2i& d, uint32_t voff, const v4i& rsrc, int soff) {
  if constexpr (NT)
    asm volatile(MX_SGPR_WAIT "buffer_load_dwordx2 %0, %1, %2, %3 offen nt" : "+v"(d) : "v"(voff), "s"(rsrc), "s"(soff) : "memory");
  else
    asm volatile(MX_SGPR_WAIT "buffer_load_dwordx2 %0, %1, %2, %3 offen" : "+v"(d) : "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}
typedef int v3i __attribute__((ext_vector_type(3)));
__device__ __forceinline__ void ld_dwords(v3i& d, uint32_t voff, const v4i& rsrc, int soff) {
  asm volatile(MX_SGPR_WAIT "buffer_load_dwordx3 %0, %1, %2, %3 offen" : "+v"(d) : "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}
__device__ __forceinline__ void ld_dwords(v2i& d, uint32_t voff, const v4i& rsrc, int soff) {
  asm volatile(MX_SGPR_WAIT "buffer_load_dwordx2 %0, %1, %2, %3 offen" : "+v"(d) : "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}
__device__ __forceinline__ void ld_b32(int& d, uint32_t voff, const v4i& rsrc, int soff) {
  asm volatile(MX_SGPR_WAIT "buffer_load_dword %0, %1, %2, %3 offen" : "+v"(d) : "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}

// A workgroup barrier that orders LDS traffic only.  (__syncthreads also makes the workgroup's global stores
// visible, for which the compiler waits until every vector memory operation has completed -- the loads in flight
// for the next tile included.)
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

struct MxTile {
  int nrows, e, slot0, xt;
};

// A run of a workgroup's items on one instance of a tile loop.  The items of an XCD's queue go to its W workgroups in rounds of W,
// every other round in reverse: of a queue in order of falling size the workgroup with the largest of one round gets the
// smallest of the next (in the same order every round, the first workgroups got the largest of all of them).  Nor does a workgroup
// then stay with the same column tile of one expert after the other.  Over 164 layers of 90 us and more, both orders on one card:
// 0.990 times the time in turns, 0.988 for the 105 of them whose experts hold up to 60 rows, 0.996 up to 320, 0.991 from 600 on; 38
// layers more than 2 % shorter, 6 longer.  The same order every round | in turns, us: 453 tokens, top-3 of 60 bf16 experts of
// H = 3584, I = 4096 1056 | 951; 2185, top-4 of 128 MXFP4 experts of 1536, 384 128 | 113; 352, top-7 of 32 MXFP8 experts of 4608, 1152
// 198 | 176; and the worst: 549, top-5 of 16 bf16 experts of 4608, 2304 298 | 317; 3191, one of 64 MXFP8 experts of 6656, 1536,
// popular and unpopular ones 462 | 483 (with even ones 427 | 426); 688, top-3 of 32 fp8-row experts of 7168, 1920 379 | 395.  What
// a launch gains or loses does not follow from rows, rounds or format: the same tiles in another order of memory accesses.
// (Few words: they are live in scalar registers through the tile loops, whose epilogues have none to spare.)
struct MxRun {
  int end;  // the run ends ahead of this item
  int W2;   // 2 W: from an item of the workgroup's to the one after the next
  int qbase, interleave;
  int pos0, npos;  // the chunks of the class: first place in the queue, number
  int cut;  // whole << 2 | shift: items from `whole` on are pieces, 1 << shift of a tile, equal parts of its chunk's rows
  __device__ __forceinline__ static int rows_per_piece(int rows, int shift) {
    const int per = (((rows + (1 << shift) - 1) >> shift) + 31) & ~31;
    return rows <= 128 ? rows : per < 64 ? 64 : per;
  }
};

// The tiles of a run.
template <int STAGE, int NMT, int WFMT>
struct MxTileWalk {
  // ROW8: the fp8-row kind (and the bf16 kind): per-channel weight scale x per-row activation scale ahead of the bias,
  // bias and scales indexed by natural column, and two more row / column tables (s_rs, s_wsc)
  static constexpr bool BF16 = WFMT == MX_WFMT_BF16;
  static constexpr bool ROW8 = WFMT == MX_WFMT_ROW8 || BF16;
  static constexpr int TAB_ROWS = NMT > 16 ? 320 : 256;  // rows of the row tables that are kept up
  const MxArgs& a;
  int (*s_tok)[MX_ROWS_MAX];
  float (*s_aff)[MX_ROWS_MAX];
  float (*s_bias)[MXT];
  float (*s_rs)[MX_ROWS_MAX];  // (token entries for the MX formats)
  float (*s_wsc)[MXT];
  int tid;
  const MxRun& run;

  // ---- tiles ------------------------------------------------------------------------------------
  // Everything that says which tile: uniform values, kept in scalar registers.  A tile's queue entry (two words)
  // is read through the scalar cache where it is needed, with an instruction of this file's own: a plain load is a
  // vector load to the compiler (it cannot know that no store aliases the queue), and a vector load in the wrong
  // place waits for every load in flight.
  // Item l of the class -> (chunk position, column tile).  G = `interleave` chunks at a time (chosen with the queues): within a
  // group of G queue positions the chunk varies fastest, so that workgroups with neighbouring items work on the
  // same column tile of different chunks (of one expert: they share the weight tile); G = 1 is column tiles
  // innermost.  The last group of a class may hold fewer than G chunks.
  // (items are numbered through the XCD's whole queue)
  __device__ __forceinline__ auto tile_at(int l0) const {
    int pos, xt;
    const int whole = run.cut >> 2, shift = run.cut & 3, over = l0 - whole;
    const int l = over < 0 ? l0 : whole + (over >> shift);
    if (run.interleave == 1) {
      pos = l / a.col_tiles;
      xt = l - pos * a.col_tiles;
    } else {
      const int per_group = run.interleave * a.col_tiles;
      const int lr = l - run.pos0 * a.col_tiles;
      const int grp = lr / per_group, j = lr - grp * per_group;
      const int base = grp * run.interleave;
      const int G = (run.npos - base < run.interleave) ? run.npos - base : run.interleave;
      xt = j / G;
      pos = run.pos0 + base + (j - xt * G);
    }
    v2i raw;
    asm volatile(MX_SGPR_WAIT "s_load_dwordx2 %0, %1, %2\n\ts_waitcnt lgkmcnt(0)"
                 : "=s"(raw) : "s"(a.q_chunk), "s"((run.qbase + pos) * 8) : "memory");
    MxTile t;
    t.xt = xt;
    const int rows = raw[1] & 0xffff, per = over < 0 ? rows : MxRun::rows_per_piece(rows, shift);
    const int row0 = over < 0 ? 0 : (over & ((1 << shift) - 1)) * per;
    t.slot0 = raw[0] + row0;
    t.nrows = rows - row0 < per ? rows - row0 : per;
    t.e = raw[1] >> 16;
    return t;
  }
  // gate/up: column tiles are numbered over the existing ones, 4 per full intermediate tile, then those of a
  // short last tile (the last of them may hold fewer than 32 partitions per q): intermediate tile, first
  // partition, partitions per q.  down: first hidden column.
  __device__ __forceinline__ auto tile_tI(const MxTile& t) const { return t.xt >> 2; }
  __device__ __forceinline__ auto tile_p0(const MxTile& t) const { return (t.xt & 3) * 32; }
  __device__ __forceinline__ auto tile_Pt(const MxTile& t) const {
    const int64_t rows_t = (a.I - (int64_t)(t.xt >> 2) * 512 < 512) ? (a.I - (int64_t)(t.xt >> 2) * 512) : 512;
    return (int)(rows_t / 4);
  }
  __device__ __forceinline__ auto tile_h0(const MxTile& t) const { return (int64_t)t.xt * 256; }
  // Rows: a thread looks after rows tid and 256 + tid of the chunk (token id, affinity), and after one of the
  // tile's 256 bias values.  Each of these is fetched in two steps: `*_raw` issues loads (always from a valid
  // address, no branch), `*_put` turns what arrived into the value and stores it in LDS.  Between the two lies an
  // epilogue with a tile's first loads in flight.  The loads are instructions of this file's own, like those of
  // the K loop: the compiler waits for a load of its own wherever it first touches the result or reuses the
  // register, and such a wait would hold the epilogue until everything issued before it has arrived.
  static constexpr bool ROWS2 = NMT * 16 > 256;
  __device__ __forceinline__ auto ids_raw(const MxTile& t, int (&raw)[2]) const {
    const v4i rd = make_rsrc(a.tp2id, 0xffffffffu);
#pragma unroll
    for (int j = 0; j < (ROWS2 ? 2 : 1); ++j) {
      const int r = tid + 256 * j;
      ld_b32(raw[j], (uint32_t)(t.slot0 + ((r < t.nrows) ? r : t.nrows - 1)) * 4u, rd, 0);
    }
  }
  __device__ __forceinline__ auto ids_put(int buf, int nrows, const int (&raw)[2]) const {
#pragma unroll
    for (int j = 0; j < (ROWS2 ? 2 : 1); ++j) {
      const int r = tid + 256 * j;
      if (r < TAB_ROWS) s_tok[buf][r] = (r < nrows && raw[j] >= 0 && raw[j] < a.n_real) ? raw[j] : -1;
    }
  }
  // (No branch may surround such a load: where two paths that load into the same variable meet, the compiler
  // copies the register right behind the load instruction, i.e. before the data has arrived.  So there is one
  // load instruction for both element types -- the aligned word that holds the element, the half picked later --
  // and a table that is absent is replaced by an address that is valid.)
  __device__ __forceinline__ auto elem_offset(uint32_t idx, bool two_byte) const { return two_byte ? ((idx << 1) & ~3u) : (idx << 2); }
  __device__ __forceinline__ auto elem_value(int word, uint32_t idx, bool two_byte) const {
    return two_byte ? bf16_bits_to_f32((uint16_t)((uint32_t)word >> ((idx & 1u) * 16u))) : __builtin_bit_cast(float, word);
  }
  __device__ __forceinline__ auto aff_index(int e, int buf, int r) const {
    const int id = s_tok[buf][(r < NMT * 16) ? r : 0];
    return (uint32_t)((id >= 0) ? id : 0) * (uint32_t)a.E + (uint32_t)e;
  }
  __device__ __forceinline__ auto aff_raw(const MxTile& t, int buf, int (&raw)[2]) const {
    const v4i rd = make_rsrc(a.aff ? a.aff : (const void*)a.tp2id, 0xffffffffu);
#pragma unroll
    for (int j = 0; j < (ROWS2 ? 2 : 1); ++j) {
      const uint32_t off = a.aff ? elem_offset(aff_index(t.e, buf, tid + 256 * j), a.aff_dtype == MOE_DT_BF16) : 0u;
      ld_b32(raw[j], off, rd, 0);
    }
  }
  __device__ __forceinline__ auto aff_put(int e, int buf, const int (&raw)[2]) const {
#pragma unroll
    for (int j = 0; j < (ROWS2 ? 2 : 1); ++j) {
      const int r = tid + 256 * j;
      if (r < NMT * 16) {
        float v = 0.f;
        if (a.aff && s_tok[buf][r] >= 0) v = elem_value(raw[j], aff_index(e, buf, r), a.aff_dtype == MOE_DT_BF16);
        s_aff[buf][r] = v;
      }
    }
  }
  // gate/up: bias value (gu*4 + q)*32 + pl belongs to partition p0 + pl; down: value j to column h0 + j.
  // the natural column of the thread's table entry: gate/up (gu = tid/128, q = tid/32 % 4, pl = tid % 32) ->
  // gu * I + tile*512 + q*Pt + p0 + pl; down -> h0 + tid
  // (columns that only pad the weights have no entry: natural_live is false, and natural_col the last real column's)
  __device__ __forceinline__ auto tile_col(const MxTile& t) const {
    return (uint32_t)tile_tI(t) * 512u + (uint32_t)((tid >> 5) & 3) * (uint32_t)tile_Pt(t) + (uint32_t)(tile_p0(t) + (tid & 31));
  }
  __device__ __forceinline__ auto natural_live(const MxTile& t) const { return STAGE != 1 || tile_col(t) < (uint32_t)a.I_tab; }
  __device__ __forceinline__ auto natural_col(const MxTile& t) const {
    if (STAGE == 1) {
      const uint32_t col = tile_col(t);
      return (uint32_t)(tid >> 7) * (uint32_t)a.I_tab + (col < (uint32_t)a.I_tab ? col : (uint32_t)a.I_tab - 1u);
    }
    return (uint32_t)tile_h0(t) + (uint32_t)tid;
  }
  // table entries per expert
  __device__ __forceinline__ uint32_t ncols() const { return (STAGE == 1) ? 2u * (uint32_t)a.I_tab : (uint32_t)a.H; }
  __device__ __forceinline__ auto bias_index(const MxTile& t) const {
    if (ROW8) return (uint32_t)t.e * ncols() + natural_col(t);
    if (STAGE == 1) {
      // (partitions that a short last tile does not have: the table may end with the last one that exists)
      const int p_ = tile_p0(t) + (tid & 31), Pt = tile_Pt(t);
      const uint32_t p = (uint32_t)(p_ < Pt ? p_ : Pt - 1);
      return ((((uint32_t)t.e * (uint32_t)a.pI + p) * 2u + (uint32_t)(tid >> 7)) * (uint32_t)a.nI + (uint32_t)tile_tI(t)) * 4u +
             (uint32_t)((tid >> 5) & 3);
    }
    return (uint32_t)t.e * (uint32_t)a.H + (uint32_t)tile_h0(t) + (uint32_t)tid;
  }
  __device__ __forceinline__ auto bias_raw(const MxTile& t, int& raw) const {
    const v4i rd = make_rsrc(a.bias ? a.bias : (const void*)a.tp2id, 0xffffffffu);
    ld_b32(raw, a.bias ? elem_offset(bias_index(t), a.bias_dtype == MOE_DT_BF16) : 0u, rd, 0);
  }
  __device__ __forceinline__ auto bias_put(const MxTile& t, int buf, int raw) const {
    s_bias[buf][tid] = (a.bias && (!ROW8 || natural_live(t))) ? elem_value(raw, bias_index(t), a.bias_dtype == MOE_DT_BF16) : 0.f;
  }
  // ROW8: the weights' per-channel scale of the thread's column (fp32), and the activation rows' scales: gate/up,
  // the fp32 behind the H codes of the token's record, times the affinity under PRE_SCALE (the affinity scales
  // the token's row, i.e. its dequantisation scale); down, the scale of the re-quantised intermediate row.
  __device__ __forceinline__ auto wsc_raw(const MxTile& t, int& raw) const {
    if constexpr (ROW8) {
      const v4i rd = make_rsrc(a.w_cscale ? (const void*)a.w_cscale : (const void*)a.tp2id, 0xffffffffu);
      ld_b32(raw, a.w_cscale ? ((a.cscale_experts > 1 ? (uint32_t)t.e * ncols() : 0u) + natural_col(t)) << 2 : 0u, rd, 0);
    }
  }
  __device__ __forceinline__ auto wsc_put(const MxTile& t, int buf, int raw) const {
    if constexpr (ROW8) s_wsc[buf][tid] = (a.w_cscale && natural_live(t)) ? __builtin_bit_cast(float, raw) : 1.f;
  }
  __device__ __forceinline__ auto rs_raw(const MxTile& t, int buf, int (&raw)[2]) const {
    if constexpr (ROW8) {
      // (bf16: nothing to fetch; the load stays, from an address that is valid, so that every format issues the
      // same loads)
      const v4i rd = make_rsrc((BF16 || (STAGE == 1 && !a.a_rscale)) ? (const void*)a.A : (const void*)a.a_rscale, 0xffffffffu);
#pragma unroll
      for (int j = 0; j < (ROWS2 ? 2 : 1); ++j) {
        const int r = tid + 256 * j;
        uint32_t off;
        if (STAGE == 1) {
          const int id = s_tok[buf][(r < NMT * 16) ? r : 0];
          off = (uint32_t)((id >= 0) ? id : 0) * (a.a_rscale ? 4u : (uint32_t)a.a_stride) +
                ((BF16 || a.a_rscale) ? 0u : (uint32_t)a.H);
        } else {
          off = (uint32_t)(t.slot0 + ((r < t.nrows) ? r : t.nrows - 1)) << 2;
        }
        ld_b32(raw[j], off, rd, 0);
      }
    }
  }
  // (gate/up under PRE_SCALE: `aff` holds what aff_raw fetched for the same rows)
  __device__ __forceinline__ auto rs_put(int e, int buf, const int (&raw)[2], const int (&aff)[2]) const {
    if constexpr (ROW8) {
      const bool pre = STAGE == 1 && (a.scaling_mode == MOE_SCALE_PRE || a.scaling_mode == MOE_SCALE_PRE_DELAYED);
#pragma unroll
      for (int j = 0; j < (ROWS2 ? 2 : 1); ++j) {
        const int r = tid + 256 * j;
        if (r < NMT * 16) {
          float v = BF16 ? 1.f : __builtin_bit_cast(float, raw[j]);
          if (STAGE == 1 && s_tok[buf][r] < 0) v = 0.f;
          if (pre && a.aff && s_tok[buf][r] >= 0) v *= elem_value(aff[j], aff_index(e, buf, r), a.aff_dtype == MOE_DT_BF16);
          s_rs[buf][r] = v;
        }
      }
    }
  }
  // which stages fetch the affinities: down always; gate/up of the fp8-row kind, for PRE_SCALE
  static constexpr bool AFF_ROWS = STAGE == 2 || ROW8;
  // what has been requested with the *_raw functions above may be used once this has passed (OUT: memory instructions
  // issued behind them that may still be out)
  template <int OUT>
  __device__ __forceinline__ void loads_landed(int (&x)[2], int (&y)[2], int& z, int (&u)[2], int& v) const {
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(OUT) : "memory");
    asm volatile("" : "+v"(x[0]), "+v"(x[1]), "+v"(y[0]), "+v"(y[1]), "+v"(z));
    if constexpr (ROW8) asm volatile("" : "+v"(u[0]), "+v"(u[1]), "+v"(v));
  }
  __device__ __forceinline__ void all_loads_landed(int (&x)[2], int (&y)[2], int& z, int (&u)[2], int& v) const {
    loads_landed<0>(x, y, z, u, v);
  }
};

}  // namespace moe
