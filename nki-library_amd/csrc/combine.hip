// Block bookkeeping and the affinity-weighted combine (scatter-add) for the blockwise MoE.
//
// The reference accumulates each block's bf16 contribution into the output rows with a
// read-modify-write scatter in block order (bwmm_shard_on_block.py:1005-1038; golden
// test_moe_cte_common.py:430-434).  On the GPU the down GEMM writes every slot's contribution
// once (bf16, already multiplied by the affinity) and one pass per token then adds that
// token's contributions in ascending slot order -- the same order and the same bf16
// arithmetic as the golden, deterministic, and without atomics.  HBM traffic: each
// contribution row is written once and read once, each output row written once.
#include "combine.hpp"
#include "chunks.hpp"

namespace moe {

// n_active = index of the first zero in conditions (N when there is none / no conditions);
// valid_rows[b] = 1 + last row of block b holding a real token id (0 for an all-padding block
// or a block at/after n_active or with an expert id outside [0, E)).
__global__ __launch_bounds__(256) void prep_blocks_kernel(const int32_t* __restrict__ tp2id,
                                                          const int32_t* __restrict__ b2e,
                                                          const int32_t* __restrict__ conditions, int64_t n_conditions,
                                                          int64_t N, int64_t B, int64_t E, int64_t n_real,
                                                          int32_t* __restrict__ n_active,
                                                          int32_t* __restrict__ valid_rows,
                                                          int32_t* __restrict__ cnt) {
  __shared__ int s_first_zero;
  __shared__ int s_red[4];
  if (threadIdx.x == 0) s_first_zero = (int)N;
  __syncthreads();
  if (conditions) {
    const int64_t lim = n_conditions < N ? n_conditions : N;
    for (int64_t i = threadIdx.x; i < lim; i += blockDim.x)
      if (conditions[i] == 0) atomicMin(&s_first_zero, (int)i);
  }
  __syncthreads();
  const int na = s_first_zero;
  if (blockIdx.x == 0 && threadIdx.x == 0) *n_active = na;
  for (int64_t b = blockIdx.x; b < N; b += gridDim.x) {
    int v = 0;
    const int e = b2e[b];
    if (b < na && e >= 0 && e < E) {
      for (int64_t r = threadIdx.x; r < B; r += blockDim.x) {
        const int id = tp2id[b * B + r];
        if (id >= 0 && id < n_real) {
          v = (int)r + 1;
          atomicAdd(&cnt[id], 1);  // slots per token, for the token -> slot lists of the combine
        }
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) valid_rows[b] = max(max(s_red[0], s_red[1]), max(s_red[2], s_red[3]));
  }
}

__global__ __launch_bounds__(256) void fill_zero_kernel(int32_t* __restrict__ p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// Exclusive scan of cnt[0..n) into off[0..n] by one workgroup of 1024 threads: a thread owns 8 consecutive
// elements of each 8192-element tile.
__device__ __forceinline__ void inv_scan(const int32_t* __restrict__ cnt, int32_t* __restrict__ off, int64_t n,
                                         int* s_ws) {
  int carry = 0;
  for (int64_t base = 0; base < n; base += 8192) {
    const int64_t i0 = base + 8 * (int64_t)threadIdx.x;
    int v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (i0 + j < n) ? cnt[i0 + j] : 0;
    int mine = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) mine += v[j];
    int total;
    int run = carry + block_excl_scan(mine, s_ws, &total);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (i0 + j < n) off[i0 + j] = run;
      run += v[j];
    }
    carry += total;
  }
  if (threadIdx.x == 0) off[n] = carry;
}

// Two workgroups of 1024 threads, run after prep_blocks_kernel: workgroup 0 builds the expert chunks,
// workgroup 1 turns the slots-per-token counts into list offsets.  They share no data.
__global__ __launch_bounds__(1024) void chunks_and_offsets_kernel(
    const int32_t* __restrict__ b2e, const int32_t* __restrict__ n_active, const int32_t* __restrict__ valid_rows,
    int64_t N, int64_t B, int64_t E, int32_t* __restrict__ n_chunks, int32_t* __restrict__ chunk_slot,
    int32_t* __restrict__ chunk_rows, int32_t* __restrict__ chunk_expert, int32_t* __restrict__ chunk_xcd,
    int32_t* __restrict__ q_chunk, int32_t* __restrict__ q_off, int64_t max_chunks,
    const int32_t* __restrict__ cnt, int32_t* __restrict__ off, int64_t n_real, bool pad_row) {
  __shared__ int s_ws[16];
  if (blockIdx.x == 0)
    build_chunks(b2e, n_active, valid_rows, N, B, E, n_chunks, chunk_slot, chunk_rows, chunk_expert, chunk_xcd, q_chunk,
                 q_off, max_chunks, s_ws, pad_row);
  else
    inv_scan(cnt, off, n_real, s_ws);
}

// One workgroup: chunks and work queues from a block build's own valid rows (moe_build_blocks_plan).
__global__ __launch_bounds__(1024) void plan_chunks_kernel(
    const int32_t* __restrict__ b2e, const int32_t* __restrict__ n_active, const int32_t* __restrict__ valid_rows,
    int64_t N, int64_t B, int64_t E, int32_t* __restrict__ n_chunks, int32_t* __restrict__ chunk_slot,
    int32_t* __restrict__ chunk_rows, int32_t* __restrict__ chunk_expert, int32_t* __restrict__ chunk_xcd,
    int32_t* __restrict__ q_chunk, int32_t* __restrict__ q_off, int64_t max_chunks) {
  __shared__ int s_ws[16];
  build_chunks(b2e, n_active, valid_rows, N, B, E, n_chunks, chunk_slot, chunk_rows, chunk_expert, chunk_xcd, q_chunk,
               q_off, max_chunks, s_ws, false);
}

// ---- activation checkpoints: the rows behind the last token -------------------------------------------------
//
// The gate_up checkpoint [N, 2, I, B] and the down checkpoint [N, B, H] hold every row of every executed block; blocks
// that do not run stay zero.  Behind an expert's last token all rows are padding, i.e. a zero hidden row each, with the
// same results: the GEMMs compute the first of them (see build_chunks), and these kernels copy it to the rest of the
// expert's blocks and clear the blocks that do not run.  A training-shaped call has as many padding rows as tokens:
// T = 1024, top-4 of 8 experts of H = 3072, I = 2048, B = 512 lists 7680 rows for 4096 routed ones: the GEMMs over all of them
// took 205 + 134 us and clearing both checkpoints beforehand 33; over the routed ones 125 + 82, and 16 + 9 for these copies.

// A block's run (the executed blocks of its expert around it): the slot of the row to copy, and the block's first row
// behind it; rows 0 .. B of a block that does not run are to be cleared (src = -1).  Every thread of the workgroup gets it.
struct CkptPad {
  int64_t src;
  int first;
};
__device__ __forceinline__ CkptPad ckpt_pad_of(int64_t b, const int32_t* __restrict__ b2e, const int32_t* __restrict__ n_active,
                                               const int32_t* __restrict__ valid_rows, int64_t B, int64_t E, int* s_w) {
  const int na = *n_active, e = b2e[b];
  if (b >= na || e < 0 || e >= E) return CkptPad{-1, 0};  // (the same for the whole workgroup)
  if (threadIdx.x == 0) {
    s_w[0] = 0;   // first block of the run
    s_w[1] = na;  // the one behind it
    s_w[2] = -1;  // its last block that holds a token
  }
  __syncthreads();
  for (int j = threadIdx.x; j < na; j += blockDim.x)
    if (b2e[j] != e) {
      if (j < b) atomicMax(&s_w[0], j + 1);
      else atomicMin(&s_w[1], j);
    }
  __syncthreads();
  const int j0 = s_w[0], j1 = s_w[1];
  for (int j = j0 + (int)threadIdx.x; j < j1; j += blockDim.x)
    if (valid_rows[j] > 0) atomicMax(&s_w[2], j);
  __syncthreads();
  const int last = s_w[2];
  const int64_t src = last < 0 ? j0 * B : last * B + valid_rows[last];  // (its block may be the next one, or past the run)
  const int64_t first = src + 1 - b * B;
  return CkptPad{src, (int)(first < 0 ? 0 : first > B ? B : first)};
}

constexpr int CKPT_COLS = 64;  // columns of the gate_up checkpoint per workgroup
// workgroup y of ny that share block b
__device__ __forceinline__ void ckpt_pad_gate_up(uint16_t* __restrict__ ck, const int32_t* __restrict__ b2e,
                                                 const int32_t* __restrict__ n_active,
                                                 const int32_t* __restrict__ valid_rows, int64_t B, int64_t E, int64_t cols,
                                                 int64_t b, int64_t y, int64_t ny) {
  __shared__ int s_w[3];
  __shared__ uint16_t s_v[CKPT_COLS];
  const CkptPad p = ckpt_pad_of(b, b2e, n_active, valid_rows, B, E, s_w);
  if (p.first >= B) return;
  for (int64_t c0 = y * CKPT_COLS; c0 < cols; c0 += ny * CKPT_COLS) {
    __syncthreads();  // (s_v of the pass before)
    const int nc = (int)(cols - c0 < CKPT_COLS ? cols - c0 : CKPT_COLS);
    if ((int)threadIdx.x < nc) {
      uint16_t v = 0;
      if (p.src >= 0) v = ck[(p.src / B * cols + c0 + threadIdx.x) * B + p.src % B];
      s_v[threadIdx.x] = v;
    }
    __syncthreads();
    uint16_t* base = ck + (b * cols + c0) * B;
    if (B % 8 == 0 && ((uintptr_t)ck & 15) == 0) {
      // pieces of eight rows, 2^lw threads side by side along a column; the first piece may begin with rows to keep
      const int g0 = p.first / 8, g1 = (int)(B / 8), lw = g1 >= 64 ? 6 : g1 >= 32 ? 5 : g1 >= 16 ? 4 : 3;
      for (int col = (int)threadIdx.x >> lw; col < nc; col += 256 >> lw) {
        const uint32_t v = s_v[col], w = v | (v << 16);
        for (int gr = g0 + ((int)threadIdx.x & ((1 << lw) - 1)); gr < g1; gr += 1 << lw) {
          uint16_t* q = base + (int64_t)col * B + gr * 8;
          if (gr * 8 >= p.first) *(uint4*)q = make_uint4(w, w, w, w);
          else
            for (int r = p.first - gr * 8; r < 8; ++r) q[r] = (uint16_t)v;
        }
      }
    } else {
      const int nr = (int)B - p.first;
      for (int64_t i = threadIdx.x; i < (int64_t)nc * nr; i += 256) base[i / nr * B + p.first + i % nr] = s_v[i / nr];
    }
  }
}

constexpr int CKPT_ROWS = 16;  // rows of the down checkpoint per workgroup
__device__ __forceinline__ void ckpt_pad_down(uint16_t* __restrict__ ck, const int32_t* __restrict__ b2e,
                                              const int32_t* __restrict__ n_active, const int32_t* __restrict__ valid_rows,
                                              int64_t B, int64_t E, int64_t H, int64_t b, int64_t y, int64_t ny) {
  __shared__ int s_w[3];
  const CkptPad p = ckpt_pad_of(b, b2e, n_active, valid_rows, B, E, s_w);
  for (int64_t rb = y * CKPT_ROWS; rb < B; rb += ny * CKPT_ROWS) {
    const int64_t r0 = rb < p.first ? p.first : rb, r1 = rb + CKPT_ROWS < B ? rb + CKPT_ROWS : B;
    if (r0 >= r1) continue;
    if (H % 8 == 0 && ((uintptr_t)ck & 15) == 0) {
      for (int64_t h = threadIdx.x; h < H / 8; h += 256) {
        uint4 v = make_uint4(0, 0, 0, 0);
        if (p.src >= 0) v = *(const uint4*)(ck + p.src * H + h * 8);
        for (int64_t r = r0; r < r1; ++r) *(uint4*)(ck + (b * B + r) * H + h * 8) = v;
      }
    } else {
      for (int64_t h = threadIdx.x; h < H; h += 256) {
        const uint16_t v = p.src >= 0 ? ck[p.src * H + h] : (uint16_t)0;
        for (int64_t r = r0; r < r1; ++r) ck[(b * B + r) * H + h] = v;
      }
    }
  }
}

// up to this many slots, tokens and blocks the bookkeeping is one launch of one workgroup (prep_small_kernel)
constexpr int64_t PREP_SMALL_SLOTS = 40960, PREP_SMALL_TOKENS = 4096, PREP_SMALL_BLOCKS = 2048;

// The whole bookkeeping of a small problem (up to a few ten thousand slots) by ONE workgroup of 1024 threads in one
// launch: find the active blocks and their valid rows, count the slots per token, build the expert chunks and the work
// queues, scan the counts and fill the token -> slot lists.  The four launches it replaces take longer to start than to
// run at such sizes.  It is a chain of steps, so what counts is the latency of each: the counts, the list positions and
// the valid rows live in LDS, and the two passes over the slots deal units of 64 slots to all sixteen waves, four in
// flight per wave (a wave per block with the counts behind global atomics left three quarters of the waves idle and took 27
// us at 15 blocks of 512 slots over 1024 tokens; now 15).
__global__ __launch_bounds__(1024) void prep_small_kernel(
    const int32_t* __restrict__ tp2id, const int32_t* __restrict__ b2e, const int32_t* __restrict__ conditions,
    int64_t n_conditions, int64_t N, int64_t B, int64_t E, int64_t n_real, int32_t* __restrict__ n_active,
    int32_t* __restrict__ valid_rows, int32_t* __restrict__ n_chunks, int32_t* __restrict__ chunk_slot,
    int32_t* __restrict__ chunk_rows, int32_t* __restrict__ chunk_expert, int32_t* __restrict__ chunk_xcd,
    int32_t* __restrict__ q_chunk, int32_t* __restrict__ q_off, int64_t max_chunks, int32_t* __restrict__ off,
    int32_t* __restrict__ list, bool pad_row) {
  __shared__ int s_ws[16];
  __shared__ int s_first_zero;
  __shared__ int s_cnt[PREP_SMALL_TOKENS];    // slots per token, then the next free place of its list
  __shared__ int s_valid[PREP_SMALL_BLOCKS];  // valid rows per block = 1 + last row with a real token
  const int tid = threadIdx.x;
  for (int i = tid; i < (int)n_real; i += 1024) s_cnt[i] = 0;
  for (int b = tid; b < (int)N; b += 1024) s_valid[b] = 0;
  if (tid == 0) s_first_zero = (int)N;
  __syncthreads();
  if (conditions) {
    const int64_t lim = n_conditions < N ? n_conditions : N;
    for (int64_t i = tid; i < lim; i += 1024)
      if (conditions[i] == 0) atomicMin(&s_first_zero, (int)i);
    __syncthreads();
  }
  const int na = s_first_zero;  // (blocks from the first zero condition on hold nothing)
  if (tid == 0) *n_active = na;
  // body(block, slot, row, id, live): 64 neighbouring slots of one block per call; live: a token in a block of an expert
  constexpr int U = 4;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int iB = (int)B, per = (iB + 63) / 64, units = na * per;
  auto over_slots = [&](auto&& body) {
    for (int u0 = wave; u0 < units; u0 += 16 * U) {
      int e[U], id[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int un = u0 + 16 * u, b = un / per, r = (un - b * per) * 64 + lane;
        e[u] = un < units ? b2e[b] : -1;
        id[u] = (un < units && r < iB) ? tp2id[b * iB + r] : -1;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int un = u0 + 16 * u, b = un / per, r = (un - b * per) * 64 + lane;
        if (e[u] >= 0 && e[u] < E) body(b, b * iB + r, r, id[u], id[u] >= 0 && id[u] < n_real);
      }
    }
  };
  over_slots([&](int b, int, int r, int id, bool live) {
    if (live) atomicAdd(&s_cnt[id], 1);
    const uint64_t m = __ballot(live);
    if (m != 0 && lane == 0) atomicMax(&s_valid[b], r + 64 - __builtin_clzll(m));  // (lane 0: r is the unit's first row)
  });
  __syncthreads();
  for (int b = tid; b < (int)N; b += 1024) valid_rows[b] = s_valid[b];
  __threadfence_block();
  __syncthreads();
  build_chunks(b2e, n_active, valid_rows, N, B, E, n_chunks, chunk_slot, chunk_rows, chunk_expert, chunk_xcd, q_chunk,
               q_off, max_chunks, s_ws, pad_row);
  // counts -> list offsets: four consecutive tokens per thread
  static_assert(PREP_SMALL_TOKENS == 4 * 1024, "one round of the workgroup");
  {
    const int i0 = 4 * tid;
    int v[4], total;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = (i0 + j < n_real) ? s_cnt[i0 + j] : 0;
    int run = block_excl_scan(v[0] + v[1] + v[2] + v[3], s_ws, &total);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (i0 + j < n_real) off[i0 + j] = s_cnt[i0 + j] = run;
      run += v[j];
    }
    if (tid == 0) off[n_real] = total;
  }
  __syncthreads();
  over_slots([&](int, int sl, int, int id, bool live) {
    if (live) list[atomicAdd(&s_cnt[id], 1)] = sl;
  });
}

__global__ __launch_bounds__(256) void inv_fill_kernel(const int32_t* __restrict__ tp2id,
                                                       const int32_t* __restrict__ valid_rows, int64_t N, int64_t B,
                                                       int64_t n_real, const int32_t* __restrict__ off,
                                                       int32_t* __restrict__ cursor, int32_t* __restrict__ list) {
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= N * B) return;
  const int64_t b = s / B, r = s % B;
  if (r >= valid_rows[b]) return;
  const int id = tp2id[s];
  if (id >= 0 && id < n_real) {
    const int p = atomicAdd(&cursor[id], 1);
    list[off[id] + p] = (int32_t)s;
  }
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// One workgroup per output row t (a few, side by side along the row, when the rows are too few to fill the GPU: y of
// ny).  D: bf16 [N*B, H] contributions.
__device__ __forceinline__ void combine_row(const uint16_t* __restrict__ D, const int32_t* __restrict__ off,
                                            const int32_t* __restrict__ list, uint16_t* __restrict__ out,
                                            uint16_t* __restrict__ out_shard1, int64_t out_row_stride, int64_t H,
                                            int64_t n_real, int64_t t, int64_t y, int64_t ny) {
  __shared__ int s_sorted[COMBINE_MAX_K];
  int cnt = 0, base = 0;
  if (t < n_real) {
    base = off[t];
    cnt = off[t + 1] - base;
    if (cnt > COMBINE_MAX_K) cnt = COMBINE_MAX_K;  // rejected on the host: a token has at most E <= MAX_K slots
  }
  // rank sort: ascending slot index == block order of the reference's accumulation.  (A list handed over by the
  // block build has a fixed number of entries per token, -1 where the token has no slot: those are left out.)
  int holes = 0;
  for (int j = 0; j < cnt; ++j) holes += list[base + j] < 0;
  for (int i = threadIdx.x; i < cnt; i += blockDim.x) {
    const int mine = list[base + i];
    if (mine < 0) continue;
    int rank = 0;
    for (int j = 0; j < cnt; ++j) {
      const int other = list[base + j];
      rank += (other >= 0 && other < mine);
    }
    s_sorted[rank] = mine;
  }
  cnt -= holes;
  __syncthreads();
  uint16_t* orow = out + t * out_row_stride;
  uint16_t* zrow = out_shard1 ? out_shard1 + t * out_row_stride : nullptr;  // the other shard's row: zeros
  const bool vec = (H % 8 == 0) && ((out_row_stride % 8) == 0) && (((uintptr_t)out & 15) == 0) &&
                   (((uintptr_t)out_shard1 & 15) == 0);
  const int64_t vt = y * blockDim.x + threadIdx.x, vstride = ny * blockDim.x;
  if (vec) {
    for (int64_t c = vt * 8; c < H; c += vstride * 8) {
      float acc[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) acc[k] = 0.f;
      // the additions form one dependent chain (bf16 rounding after each, in slot order), so the loads
      // are what can overlap: up to eight rows are requested before the first is added
      for (int j0 = 0; j0 < cnt; j0 += 8) {
        // (the contributions are read once and the result rows are not read again by this kernel: non-temporal,
        // so that neither displaces the other in the caches)
        u32x4 d[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (j0 + j < cnt) d[j] = __builtin_nontemporal_load((const u32x4*)(D + (int64_t)s_sorted[j0 + j] * H + c));
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          if (j0 + j < cnt) {
            const uint32_t w[4] = {d[j][0], d[j][1], d[j][2], d[j][3]};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              acc[2 * k] = round_to_bf16(acc[2 * k] + bf16_bits_to_f32((uint16_t)(w[k] & 0xffff)));
              acc[2 * k + 1] = round_to_bf16(acc[2 * k + 1] + bf16_bits_to_f32((uint16_t)(w[k] >> 16)));
            }
          }
        }
      }
      uint32_t o[4];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        o[k] = (uint32_t)f32_to_bf16_bits(acc[2 * k]) | ((uint32_t)f32_to_bf16_bits(acc[2 * k + 1]) << 16);
      __builtin_nontemporal_store((u32x4){o[0], o[1], o[2], o[3]}, (u32x4*)(orow + c));
      if (zrow) __builtin_nontemporal_store((u32x4){0, 0, 0, 0}, (u32x4*)(zrow + c));
    }
  } else {
    for (int64_t c = vt; c < H; c += vstride) {
      float acc = 0.f;
      for (int j = 0; j < cnt; ++j) acc = round_to_bf16(acc + bf16_bits_to_f32(D[(int64_t)s_sorted[j] * H + c]));
      orow[c] = f32_to_bf16_bits(acc);
      if (zrow) zrow[c] = 0;
    }
  }
}

__global__ __launch_bounds__(256) void combine_kernel(const uint16_t* __restrict__ D, const int32_t* __restrict__ off,
                                                      const int32_t* __restrict__ list, uint16_t* __restrict__ out,
                                                      uint16_t* __restrict__ out_shard1, int64_t out_row_stride,
                                                      int64_t H, int64_t n_real) {
  combine_row(D, off, list, out, out_shard1, out_row_stride, H, n_real, blockIdx.x, blockIdx.y, gridDim.y);
}

// The checkpoints' padding rows and the combine of one layer in one launch: three jobs that share no data and are each too
// short to fill the memory system from start to end.  Workgroups [0, n_gu) take the gate_up checkpoint (y_gu per block), the
// next n_dn the down checkpoint, the rest the output rows.  T = 1024, top-4 of 8 experts of H = 3072, I = 2048, B = 512:
// 16.5 + 9 + 10 us in three launches, 21 in this one.
struct CkptTail {
  uint16_t *ck_gu, *ck_dn;
  const int32_t *b2e, *n_active, *valid_rows;
  int64_t B, E, cols, H;
  int64_t n_gu, y_gu, n_dn, y_dn, y_c;
};
__global__ __launch_bounds__(256) void ckpt_tail_kernel(const CkptTail k, const uint16_t* __restrict__ D,
                                                        const int32_t* __restrict__ off, const int32_t* __restrict__ list,
                                                        uint16_t* __restrict__ out, uint16_t* __restrict__ out_shard1,
                                                        int64_t out_row_stride, int64_t n_real) {
  int64_t i = blockIdx.x;
  if (i < k.n_gu) {
    ckpt_pad_gate_up(k.ck_gu, k.b2e, k.n_active, k.valid_rows, k.B, k.E, k.cols, i / k.y_gu, i % k.y_gu, k.y_gu);
    return;
  }
  i -= k.n_gu;
  if (i < k.n_dn) {
    ckpt_pad_down(k.ck_dn, k.b2e, k.n_active, k.valid_rows, k.B, k.E, k.H, i / k.y_dn, i % k.y_dn, k.y_dn);
    return;
  }
  i -= k.n_dn;
  combine_row(D, off, list, out, out_shard1, out_row_stride, k.H, n_real, i / k.y_c, i % k.y_c, k.y_c);
}
// (one stage of a layer that is issued stage by stage)
__global__ __launch_bounds__(256) void ckpt_pad_kernel(const CkptTail k) {
  if (k.n_gu)
    ckpt_pad_gate_up(k.ck_gu, k.b2e, k.n_active, k.valid_rows, k.B, k.E, k.cols, blockIdx.x / k.y_gu, blockIdx.x % k.y_gu, k.y_gu);
  else
    ckpt_pad_down(k.ck_dn, k.b2e, k.n_active, k.valid_rows, k.B, k.E, k.H, blockIdx.x / k.y_dn, blockIdx.x % k.y_dn, k.y_dn);
}

// ---- host-side orchestration used by moe_blockwise() -------------------------------------

size_t bookkeeping_bytes(int64_t T1, int64_t N, int64_t B) {
  // n_active[4] | valid_rows[N] | cnt[T1] | cursor[T1] | off[T1+1] | list[N*B] | n_chunks[4] | 6 x chunk[max_chunks] |
  // q_off[8][CHUNK_CLASSES + 1], each region 256-byte aligned
  auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
  return al(16) + al((size_t)N * 4) + 2 * al((size_t)T1 * 4) + al((size_t)(T1 + 1) * 4) + al((size_t)N * B * 4) +
         al(16) + 6 * al((size_t)max_chunks_for(N, B) * 4) + al((size_t)(8 * (CHUNK_CLASSES + 1) + 1) * 4);
}

Bookkeeping carve_bookkeeping(void* base, int64_t T1, int64_t N, int64_t B) {
  auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
  Bookkeeping k;
  uint8_t* p = (uint8_t*)base;
  k.n_active = (int32_t*)p; p += al(16);
  k.valid_rows = (int32_t*)p; p += al((size_t)N * 4);
  k.cnt = (int32_t*)p; p += al((size_t)T1 * 4);
  k.cursor = (int32_t*)p; p += al((size_t)T1 * 4);
  k.off = (int32_t*)p; p += al((size_t)(T1 + 1) * 4);
  k.list = (int32_t*)p; p += al((size_t)N * B * 4);
  k.max_chunks = max_chunks_for(N, B);
  k.n_chunks = (int32_t*)p; p += al(16);
  k.chunk_slot = (int32_t*)p; p += al((size_t)k.max_chunks * 4);
  k.chunk_rows = (int32_t*)p; p += al((size_t)k.max_chunks * 4);
  k.chunk_expert = (int32_t*)p; p += al((size_t)k.max_chunks * 4);
  k.chunk_xcd = (int32_t*)p; p += al((size_t)k.max_chunks * 4);
  k.q_chunk = (int32_t*)p; p += 2 * al((size_t)k.max_chunks * 4);
  k.q_off = (int32_t*)p;
  return k;
}

int launch_prep(const Bookkeeping& k, const moe_bwmm_args* a, int64_t n_real, hipStream_t s) {
  const bool pad_row = a->gate_up_activations_T != nullptr || a->down_activations != nullptr;
  // cnt and cursor are adjacent: one clear covers both.  A fill kernel rather than a memset
  // node, so that the sequence stays safe to record into a HIP graph.
  const int64_t clear_words = (int64_t)((uint8_t*)k.off - (uint8_t*)k.cnt) / 4;
  if (a->N * a->B <= PREP_SMALL_SLOTS && n_real <= PREP_SMALL_TOKENS && a->N <= PREP_SMALL_BLOCKS) {
    hipLaunchKernelGGL(prep_small_kernel, dim3(1), dim3(1024), 0, s, a->token_position_to_id, a->block_to_expert,
                       a->conditions, a->n_conditions, a->N, a->B, a->E, n_real, k.n_active, k.valid_rows, k.n_chunks,
                       k.chunk_slot, k.chunk_rows, k.chunk_expert, k.chunk_xcd, k.q_chunk, k.q_off, k.max_chunks, k.off,
                       k.list, pad_row);
    MOE_CHECK_LAUNCH();
    return MOE_OK;
  }
  hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)((clear_words + 255) / 256)), dim3(256), 0, s, k.cnt,
                     clear_words);
  MOE_CHECK_LAUNCH();
  const unsigned g = (unsigned)(a->N < 1024 ? a->N : 1024);
  hipLaunchKernelGGL(prep_blocks_kernel, dim3(g), dim3(256), 0, s, a->token_position_to_id, a->block_to_expert,
                     a->conditions, a->n_conditions, a->N, a->B, a->E, n_real, k.n_active, k.valid_rows, k.cnt);
  MOE_CHECK_LAUNCH();
  hipLaunchKernelGGL(chunks_and_offsets_kernel, dim3(2), dim3(1024), 0, s, a->block_to_expert, k.n_active, k.valid_rows,
                     a->N, a->B, a->E, k.n_chunks, k.chunk_slot, k.chunk_rows, k.chunk_expert, k.chunk_xcd, k.q_chunk, k.q_off,
                     k.max_chunks, k.cnt, k.off, n_real, pad_row);
  MOE_CHECK_LAUNCH();
  const int64_t slots = a->N * a->B;
  const unsigned gs = (unsigned)((slots + 255) / 256);
  hipLaunchKernelGGL(inv_fill_kernel, dim3(gs), dim3(256), 0, s, a->token_position_to_id, k.valid_rows, a->N, a->B,
                     n_real, k.off, k.cursor, k.list);
  MOE_CHECK_LAUNCH();
  return MOE_OK;
}

int launch_plan_chunks(const Bookkeeping& k, const int32_t* block_to_expert, int64_t N, int64_t B, int64_t E,
                       hipStream_t s) {
  hipLaunchKernelGGL(plan_chunks_kernel, dim3(1), dim3(1024), 0, s, block_to_expert, k.n_active, k.valid_rows, N, B, E,
                     k.n_chunks, k.chunk_slot, k.chunk_rows, k.chunk_expert, k.chunk_xcd, k.q_chunk, k.q_off,
                     k.max_chunks);
  MOE_CHECK_LAUNCH();
  return MOE_OK;
}

static int64_t at_most(int64_t v, int64_t lim) { return v < lim ? v : lim; }
// few rows (decode): up to 8 workgroups share a row of the result, 8 columns per thread each
static int64_t combine_split(const moe_bwmm_args* a) {
  return a->T1 <= 256 ? at_most((a->H + 256 * 8 - 1) / (256 * 8), 8) : 1;
}
// A launch holds fewer than 2^32 threads along x (hipLaunchKernel refuses more).
constexpr int64_t MAX_WORKGROUPS = (((int64_t)1 << 32) - 1) / 256;
// A workgroup per block and 64 columns (16 rows), or, beyond a million of them, as many per block as stay below that: every
// further one would only search the blocks' table again.
CkptGrid ckpt_grid(int64_t N, int64_t B, int64_t cols, bool gate_up, bool down) {
  const int64_t per_block = N < ((int64_t)1 << 20) ? ((int64_t)1 << 20) / N : 1;
  CkptGrid g;
  g.y_gu = at_most((cols + CKPT_COLS - 1) / CKPT_COLS, per_block);
  g.y_dn = at_most((B + CKPT_ROWS - 1) / CKPT_ROWS, per_block);
  g.n_gu = gate_up ? N * g.y_gu : 0;
  g.n_dn = down ? N * g.y_dn : 0;
  return g;
}
static CkptTail ckpt_tail(const Bookkeeping& k, const moe_bwmm_args* a, bool gate_up, bool down) {
  CkptTail t;
  t.ck_gu = (uint16_t*)a->gate_up_activations_T;
  t.ck_dn = (uint16_t*)a->down_activations;
  t.b2e = a->block_to_expert; t.n_active = k.n_active; t.valid_rows = k.valid_rows;
  t.B = a->B; t.E = a->E; t.cols = 2 * a->I; t.H = a->H;
  const CkptGrid g = ckpt_grid(a->N, a->B, t.cols, gate_up, down);
  t.n_gu = g.n_gu; t.y_gu = g.y_gu; t.n_dn = g.n_dn; t.y_dn = g.y_dn;
  t.y_c = combine_split(a);
  return t;
}

int launch_ckpt_pad(int stage, const Bookkeeping& k, const moe_bwmm_args* a, hipStream_t s) {
  const CkptTail t = ckpt_tail(k, a, stage == 1, stage == 2);
  hipLaunchKernelGGL(ckpt_pad_kernel, dim3((unsigned)(t.n_gu + t.n_dn)), dim3(256), 0, s, t);
  MOE_CHECK_LAUNCH();
  return MOE_OK;
}

int launch_ckpt_tail(const Bookkeeping& k, const moe_bwmm_args* a, const void* D, int64_t n_real, hipStream_t s) {
  const CkptTail t = ckpt_tail(k, a, a->gate_up_activations_T != nullptr, a->down_activations != nullptr);
  const int64_t grid = t.n_gu + t.n_dn + a->T1 * t.y_c;
  if (grid > MAX_WORKGROUPS) {  // (millions of blocks or tokens: each of the three fits a launch of its own)
    for (int stage = 1; stage <= 2; ++stage) {
      const int rc = (stage == 1 ? t.n_gu : t.n_dn) > 0 ? launch_ckpt_pad(stage, k, a, s) : MOE_OK;
      if (rc != MOE_OK) return rc;
    }
    return launch_combine(k, a, D, n_real, s);
  }
  hipLaunchKernelGGL(ckpt_tail_kernel, dim3((unsigned)grid), dim3(256), 0, s, t, (const uint16_t*)D, k.off, k.list,
                     (uint16_t*)a->output, (uint16_t*)a->output_shard1, a->out_row_stride, n_real);
  MOE_CHECK_LAUNCH();
  return MOE_OK;
}

int launch_combine(const Bookkeeping& k, const moe_bwmm_args* a, const void* D, int64_t n_real, hipStream_t s) {
  hipLaunchKernelGGL(combine_kernel, dim3((unsigned)a->T1, (unsigned)combine_split(a)), dim3(256), 0, s, (const uint16_t*)D,
                     k.off, k.list, (uint16_t*)a->output, (uint16_t*)a->output_shard1, a->out_row_stride, a->H, n_real);
  MOE_CHECK_LAUNCH();
  return MOE_OK;
}

int launch_fill_zero_bytes(void* p, size_t bytes, hipStream_t s) {
  if (bytes == 0) return MOE_OK;
  if ((bytes & 3) != 0 || ((uintptr_t)p & 3) != 0) return MOE_E_BAD_ARG;
  const int64_t words = (int64_t)(bytes / 4);
  const int64_t grid = (words + 255) / 256;
  if (grid >= (int64_t)1 << 31) return MOE_E_BAD_SHAPE;
  hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)grid), dim3(256), 0, s, (int32_t*)p, words);
  MOE_CHECK_LAUNCH();
  return MOE_OK;
}

}  // namespace moe
