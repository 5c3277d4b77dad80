// Router top-k front end for gfx950: logits = x @ w (+ bias), top-k selection, affinities.
//
// Semantics: router_topk_torch_ref, src/nkilib_src/nkilib/core/router_topk/router_topk_torch.py:23-135
// (kernel signature src/nkilib_src/nkilib/core/router_topk/router_topk.py:55-75).
//
// Three launches where the caller's workspace holds the partial logits (moe_router_topk_workspace_bytes_for):
//   1. router_pack_w_kernel      w [H, E] -> 16-byte MFMA fragments in the order the next launch reads them, and the
//                                cleared row of the padding token;
//   2. router_split_kernel       partial logits: a workgroup multiplies a token tile and up to 256 experts over one of
//                                several parts of K.  One workgroup per 64 tokens, which is what a selection in the same
//                                launch asks for, left half of the CUs idle at 8192 tokens and all but one at 64;
//   3. router_select_kernel      sums the parts, selects, writes the table.
// T = 8192, H = 7168, E = 256 (117 MB of tokens, 21 us at the rate of a large copy): 4 + 37 + 13 us, a pass 136 -> 56 us;
// T = 64 of the same: one workgroup walked all of K, now 24 us, most of it the host's.
//
// Two launches with the smaller workspace (moe_router_topk_workspace_bytes) or a token table that is not 16-byte aligned:
//   1. transpose_w_kernel   w [H,E] -> wt [E,H] (a few MB), so that both GEMM operands are contiguous
//                           along K, which is what an MFMA lane wants (8 consecutive K values);
//   2. router_kernel<NT,MT> a workgroup of 4 waves owns 64*MT tokens and all E = 16*NT experts.  Each wave
//                           multiplies its 16*MT tokens (fragments straight from global) with the
//                           K slice of wt that the workgroup stages in LDS, with
//                           v_mfma_f32_16x16x32_bf16 into MT*NT accumulator tiles, and then selects the top
//                           k per token without leaving registers: a token's E logits sit in 16 lanes x
//                           NT registers, so k rounds of (local argmax, 4-step lane reduction, retire the
//                           winner) pick them in descending order, ties to the lower expert index.
// Everything after the GEMM is fp32: softmax over all E (or over the k selected), sigmoid, the optional
// division by the sum of the selected values.
// For E <= 256 the K loop of router_kernel is software-pipelined (MT = 1): the 64-wide K slices of wt go global -> LDS
// directly into a ring of three stages (two steps ahead), XOR-swizzled on the global side so that the
// fragment reads are conflict free, and the token fragments into six register sets (five steps ahead:
// that stream comes from HBM); loads and waits are written as instructions (a wave's loads complete in
// issue order, so a wait names how many of the most recent ones may still be out), one barrier per
// step.
#include <type_traits>

#include "common.hpp"

namespace moe {

constexpr int RT_THREADS = 256;
constexpr int RT_K = 64;         // K elements per LDS stage
constexpr int RT_PITCH = RT_K + 8;  // bf16 elements per staged row of wt (16-byte aligned, conflict-spreading pad)

__global__ __launch_bounds__(256) void transpose_w_kernel(const uint16_t* __restrict__ w, uint16_t* __restrict__ wt,
                                                          int64_t H, int64_t E) {
  __shared__ uint16_t tile[32][33];
  const int64_t h0 = (int64_t)blockIdx.x * 32, e0 = (int64_t)blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int r = ty; r < 32; r += 8) {
    const int64_t h = h0 + r, e = e0 + tx;
    tile[r][tx] = (h < H && e < E) ? w[h * E + e] : (uint16_t)0;
  }
  __syncthreads();
  for (int r = ty; r < 32; r += 8) {
    const int64_t e = e0 + r, h = h0 + tx;
    if (e < E && h < H) wt[e * H + h] = tile[tx][r];
  }
}

__global__ __launch_bounds__(256) void fill_zero_bytes_kernel(uint8_t* __restrict__ p, int64_t n) {
  for (int64_t i = threadIdx.x; i < n; i += 256) p[i] = 0;
}

struct RouterArgs {
  const uint16_t* x;   // bf16 [T, H]
  const uint16_t* wt;  // bf16 [E, H]
  const void* bias;    // [E] or null
  int bias_dtype;
  int64_t T, H, E;
  int k, act_fn, pre_norm, norm_topk, mask_to_topk;
  void* logits_out;    // [T, E] or null
  int logits_dtype;
  int32_t* index_out;  // [T, k] or null
  void* aff_out;       // [T (+1), E]
  int aff_dtype;
  float* topk_aff_out; // [T, k] or null
};

__device__ __forceinline__ void store_val(void* p, int dtype, int64_t i, float v) {
  if (dtype == MOE_DT_BF16) ((uint16_t*)p)[i] = f32_to_bf16_bits(v);
  else ((float*)p)[i] = v;
}

// max / sum over the 16 lanes that share a token row (lanes with equal lane >> 4)
__device__ __forceinline__ float row16_max(float v) {
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ float row16_sum(float v) {
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) v += __shfl_xor(v, o, 64);
  return v;
}

template <int I, int N, class F>
__device__ __forceinline__ void rt_static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    rt_static_for<I + 1, N>(f);
  }
}
__device__ __forceinline__ int rt_uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ v4i rt_rsrc(const void* p, uint32_t bytes) {
  const uint64_t addr = (uint64_t)p;
  v4i d;
  d[0] = rt_uni((int)(uint32_t)addr);
  d[1] = rt_uni((int)(uint32_t)(addr >> 32)) & 0xffff;
  d[2] = rt_uni((int)bytes);
  d[3] = 0x00020000;
  return d;
}
// (s_nop 4: a scalar operand that a vector instruction has just written -- the compiler reloads spilled scalars
// with v_readlane -- must not be read by a memory instruction within the next few cycles, and the compiler does
// not know that these statements are memory instructions)
__device__ __forceinline__ void rt_ld_lds(uint32_t lds, uint32_t voff, const v4i& rsrc, int soff) {
  asm volatile("s_nop 4\n\ts_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               : : "s"(lds), "v"(voff), "s"(rsrc), "s"(soff) : "memory", "m0");
}
__device__ __forceinline__ void rt_ld(v4i& d, uint32_t voff, const v4i& rsrc, int soff) {
  asm volatile("s_nop 4\n\tbuffer_load_dwordx4 %0, %1, %2, %3 offen" : "+v"(d) : "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}

// Experts of a lane: lane c of the 16 that share a token holds NT logits.
struct ColsOf16 {  // expert n * 16 + c: the accumulators of router_kernel
  static __device__ __forceinline__ int expert(int n, int c) { return n * 16 + c; }
  static __device__ __forceinline__ int lane(int e) { return e & 15; }
  static __device__ __forceinline__ int slot(int e) { return e >> 4; }
};
struct ColsOf4 {  // four neighbouring experts per 16-byte load: the partial sums of router_split_kernel
  static __device__ __forceinline__ int expert(int n, int c) { return (n >> 2) * 64 + c * 4 + (n & 3); }
  static __device__ __forceinline__ int lane(int e) { return (e >> 2) & 15; }
  static __device__ __forceinline__ int slot(int e) { return (e >> 6) * 4 + (e & 3); }
};

__device__ __forceinline__ float expert_bias(const RouterArgs& a, int e) {
  return (a.bias && e < a.E) ? load_as_f32(a.bias, a.bias_dtype, e) : 0.f;
}

// One token per 16 lanes: logits out, activation, top k, affinities out.  v: the lane's logits; `live` (t is a token)
// is uniform over the 16 lanes.
template <int NT, class MAP>
__device__ __forceinline__ void select_and_store(const RouterArgs& a, int64_t t, bool live, int c, float (&v)[NT]) {
  const float NEG = -__builtin_inff();
#pragma unroll
  for (int n = 0; n < NT; ++n)
    if (MAP::expert(n, c) >= a.E) v[n] = NEG;
  if (a.logits_out && live) {
#pragma unroll
    for (int n = 0; n < NT; ++n)
      if (MAP::expert(n, c) < a.E) store_val(a.logits_out, a.logits_dtype, t * a.E + MAP::expert(n, c), v[n]);
  }
  // full activation (pre-norm pipeline)
  float fullv[NT];
  if (a.pre_norm) {
    if (a.act_fn == 1) {  // softmax over all experts
      float mx = NEG;
#pragma unroll
      for (int n = 0; n < NT; ++n) mx = fmaxf(mx, v[n]);
      mx = row16_max(mx);
      float sum = 0.f;
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        fullv[n] = (v[n] == NEG) ? 0.f : expf(v[n] - mx);
        sum += fullv[n];
      }
      sum = row16_sum(sum);
#pragma unroll
      for (int n = 0; n < NT; ++n) fullv[n] = fullv[n] / sum;
    } else {
#pragma unroll
      for (int n = 0; n < NT; ++n) fullv[n] = 1.0f / (1.0f + expf(-v[n]));
    }
  }
  // k rounds of argmax, ties to the lower expert index
  unsigned taken = 0;  // bit n: the lane's n-th expert has been selected
  float selv[8];
  int seli[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    selv[j] = 0.f;
    seli[j] = 0;
  }
  for (int j = 0; j < a.k; ++j) {
    float bv = NEG;
    int bi = 0x7fffffff;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const bool free_ = !((taken >> n) & 1u) && (MAP::expert(n, c) < a.E);
      if (free_ && v[n] > bv) {  // ascending n: the lower index wins ties inside the lane
        bv = v[n];
        bi = MAP::expert(n, c);
      }
    }
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
      const float ov = __shfl_xor(bv, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (ov > bv || (ov == bv && oi < bi)) {
        bv = ov;
        bi = oi;
      }
    }
    if (MAP::lane(bi) == c && bi < (int)a.E) taken |= 1u << MAP::slot(bi);
#pragma unroll
    for (int jj = 0; jj < 8; ++jj)
      if (jj == j) {
        selv[jj] = bv;
        seli[jj] = bi;
      }
  }
  // affinities of the selected experts
  float affk[8];
  if (a.pre_norm) {
    float ssum = 0.f;
#pragma unroll
    for (int n = 0; n < NT; ++n) ssum += ((taken >> n) & 1u) ? fullv[n] : 0.f;
    ssum = row16_sum(ssum);
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      float o = fullv[n];
      if (a.norm_topk) o = ((taken >> n) & 1u) ? fullv[n] / ssum : 0.f;
      else if (a.mask_to_topk) o = ((taken >> n) & 1u) ? fullv[n] : 0.f;
      fullv[n] = o;
    }
  } else {
    // activate the k selected logits only
    float mx = selv[0], sum = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (j < a.k) {
        affk[j] = (a.act_fn == 1) ? expf(selv[j] - mx) : 1.0f / (1.0f + expf(-selv[j]));
        sum += affk[j];
      }
#pragma unroll
    for (int n = 0; n < NT; ++n) fullv[n] = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (j < a.k) {
        if (a.act_fn == 1) affk[j] = affk[j] / sum;
        if (MAP::lane(seli[j]) == c) {
#pragma unroll
          for (int n = 0; n < NT; ++n)
            if (n == MAP::slot(seli[j])) fullv[n] = affk[j];
        }
      }
  }
  if (live) {
#pragma unroll
    for (int n = 0; n < NT; ++n)
      if (MAP::expert(n, c) < a.E) store_val(a.aff_out, a.aff_dtype, t * a.E + MAP::expert(n, c), fullv[n]);
    if (c == 0) {
      for (int j = 0; j < a.k; ++j) {
        if (a.index_out) a.index_out[t * a.k + j] = seli[j];
      }
    }
    if (a.topk_aff_out) {
      // the lane that owns the selected expert knows its final affinity
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (j < a.k && MAP::lane(seli[j]) == c) {
#pragma unroll
          for (int n = 0; n < NT; ++n)
            if (n == MAP::slot(seli[j])) a.topk_aff_out[t * a.k + j] = fullv[n];
        }
    }
  }
}

template <int NT, int MT, bool PIPE>
__global__ __launch_bounds__(RT_THREADS) void router_kernel(const RouterArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  uint16_t* sW = (uint16_t*)smem;  // [16*NT][RT_PITCH]
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int c = lane & 15, g = lane >> 4;
  const int64_t t0 = (int64_t)blockIdx.x * (64 * MT) + w * (16 * MT);
  constexpr int EP = 16 * NT;  // experts covered by this instantiation (>= a.E)

  v4f acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[m][n] = (v4f){0.f, 0.f, 0.f, 0.f};

  const int nsteps = (int)(a.H / RT_K);
  if constexpr (!PIPE) {
  // A rows: lane (c, g) of row tile m reads token t0 + 16m + c, K elements 8g .. 8g+7 of each 32-wide step
  const uint16_t* xr[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    int64_t t = t0 + 16 * m + c;
    if (t >= a.T) t = a.T - 1;  // rows past the end repeat the last token; nothing is written for them
    xr[m] = a.x + t * a.H + 8 * g;
  }
  for (int s = 0; s < nsteps; ++s) {
    const int64_t k0 = (int64_t)s * RT_K;
    __syncthreads();
    // stage wt[:, k0 .. k0+63]: 16*NT rows of 128 bytes, 8 chunks of 16 bytes each
    for (int i = tid; i < EP * 8; i += RT_THREADS) {
      const int e = i >> 3, ch = i & 7;
      v4i v = {0, 0, 0, 0};
      if (e < a.E) v = *(const v4i*)(a.wt + (int64_t)e * a.H + k0 + ch * 8);
      *(v4i*)(sW + e * RT_PITCH + ch * 8) = v;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      v8bf af[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) af[m] = *(const v8bf*)(xr[m] + k0 + kk * 32);
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const v8bf bf = *(const v8bf*)(sW + (n * 16 + c) * RT_PITCH + kk * 32 + 8 * g);
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[m], bf, acc[m][n], 0, 0, 0);
      }
    }
  }
  } else {
    static_assert(MT == 1, "the pipelined loop handles one row tile per wave");
    constexpr int STAGE = EP * 128;       // bytes of one K slice of wt in LDS (row pitch 128 bytes)
    constexpr int NI = EP * 8 / RT_THREADS;  // 16-byte pieces of a slice per thread
    constexpr int NL = NI + 2;            // loads per step and wave: NI weight pieces + 2 token fragments
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
    const int wu = rt_uni(w);
    // weight pieces: wave instruction i covers 8 rows x 128 bytes; lane l fills slot l&7 of row 8(NI w + i) + (l>>3)
    // with the global chunk slot ^ (row & 7)
    uint32_t w_voff[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      int row = 8 * (NI * w + i) + (lane >> 3);
      const int ch = (lane & 7) ^ ((row >> 1) & 7);
      if (row >= a.E) row = (int)a.E - 1;  // padding rows repeat the last expert; their logits are never used
      w_voff[i] = (uint32_t)(row * a.H * 2 + ch * 16);
    }
    int64_t t = t0 + c;
    if (t >= a.T) t = a.T - 1;  // rows past the end repeat the last token; nothing is written for them
    const uint32_t x_voff = (uint32_t)(t * a.H * 2 + g * 16);
    const v4i rw_ = rt_rsrc(a.wt, (uint32_t)(a.E * a.H * 2)), rx_ = rt_rsrc(a.x, (uint32_t)(a.T * a.H * 2));
    // rings: three LDS stages of wt (loads two steps ahead, L2 hits), RA register sets of token fragments
    // (loads RA-1 steps ahead: this is the stream that comes from HBM, and what is in flight bounds its rate)
    constexpr int RA = 6;
    v4i af[RA][2];
#pragma unroll
    for (int u = 0; u < RA; ++u) af[u][0] = af[u][1] = (v4i){0, 0, 0, 0};
    // descriptors of zero records past the end: no traffic, zeros
    auto issue_w = [&](int s, int stage) {
      v4i rw;
      rw[0] = rt_uni(rw_[0]); rw[1] = rt_uni(rw_[1]); rw[2] = rt_uni(s < nsteps ? rw_[2] : 0); rw[3] = rt_uni(rw_[3]);
      const int koff = rt_uni(s * RT_K * 2);
      const uint32_t lds = rt_uni((int)(lds0 + (uint32_t)stage * STAGE + (uint32_t)(NI * wu) * 1024));
#pragma unroll
      for (int i = 0; i < NI; ++i) rt_ld_lds(lds + i * 1024, w_voff[i], rw, koff);
    };
    auto issue_a = [&](int s, v4i& f0, v4i& f1) {
      v4i rx;
      rx[0] = rt_uni(rx_[0]); rx[1] = rt_uni(rx_[1]); rx[2] = rt_uni(s < nsteps ? rx_[2] : 0); rx[3] = rt_uni(rx_[3]);
      const int koff = rt_uni(s * RT_K * 2);
      rt_ld(f0, x_voff, rx, koff);
      rt_ld(f1, x_voff, rx, koff + 64);
    };
    const int rd0 = c * 128;  // fragment reads: row n*16 + c, chunk 4 kk + g, swizzled
    auto step = [&](auto u_, int s) {
      constexpr int U = decltype(u_)::value, stage = U % 3;
      // out at most: the fragments issued in step s-2 and everything of step s-1
      asm volatile("s_waitcnt vmcnt(%0)" : : "n"(NI + 4) : "memory");
      asm volatile("" : "+v"(af[U][0]), "+v"(af[U][1]));
      __syncthreads();  // every wave's pieces of this step are in; every wave has left step s-1
      // into the stage and the registers that step s-1 read
      issue_w(s + 2, (stage + 2) % 3);
      issue_a(s + RA - 1, af[(U + RA - 1) % RA][0], af[(U + RA - 1) % RA][1]);
      const v8bf a0 = __builtin_bit_cast(v8bf, af[U][0]), a1 = __builtin_bit_cast(v8bf, af[U][1]);
      const uint8_t* base = smem + stage * STAGE + rd0;
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const v8bf b0 = *(const v8bf*)(base + n * 16 * 128 + ((g ^ ((c >> 1) & 7)) * 16));
        const v8bf b1 = *(const v8bf*)(base + n * 16 * 128 + (((4 + g) ^ ((c >> 1) & 7)) * 16));
        acc[0][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b0, acc[0][n], 0, 0, 0);
        acc[0][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b1, acc[0][n], 0, 0, 0);
      }
      // instruction order of the step: 8 fragment reads ahead, then 2 reads per 2 MFMAs, so that no
      // MFMA waits for the LDS round trip of its own operand (one wave per SIMD has no other cover)
      __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
#pragma unroll
      for (int i = 0; i < NT - 4; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
    };
    // prologue in the order the steps before the first would have issued
    issue_a(0, af[0][0], af[0][1]);
    issue_a(1, af[1][0], af[1][1]);
    issue_a(2, af[2][0], af[2][1]);
    issue_w(0, 0);
    issue_a(3, af[3][0], af[3][1]);
    issue_w(1, 1);
    issue_a(4, af[4][0], af[4][1]);
    int s = 0;
    for (; s + RA <= nsteps; s += RA)
      rt_static_for<0, RA>([&](auto u) { step(u, s + decltype(u)::value); });
    rt_static_for<0, RA - 1>([&](auto u) {
      if (s + decltype(u)::value < nsteps) step(u, s + decltype(u)::value);
    });
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // the loads past the end still arrive (as zeros): their registers stay reserved until here
#pragma unroll
    for (int u = 0; u < RA; ++u) asm volatile("" : : "v"(af[u][0]), "v"(af[u][1]));
  }

  // ---- epilogue: per token (row tile m, row 4g + r); the lane's experts are n*16 + c --------------
  float bias[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) bias[n] = expert_bias(a, ColsOf16::expert(n, c));
#pragma unroll
  for (int m = 0; m < MT; ++m) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t t = t0 + 16 * m + 4 * g + r;
      float v[NT];
#pragma unroll
      for (int n = 0; n < NT; ++n) v[n] = acc[m][n][r] + bias[n];
      select_and_store<NT, ColsOf16>(a, t, t < a.T, c, v);  // (t < T: uniform over the 16 lanes of the row)
    }
  }
}

template <int NT, int MT, bool PIPE>
static int launch_router(const RouterArgs& a, hipStream_t s) {
  const unsigned grid = (unsigned)((a.T + 64 * MT - 1) / (64 * MT));
  const size_t lds = PIPE ? (size_t)3 * 16 * NT * 128 : (size_t)16 * NT * RT_PITCH * 2;
  if (allow_lds<&router_kernel<NT, MT, PIPE>>((int)lds) != hipSuccess) return MOE_E_LAUNCH;
  hipLaunchKernelGGL((router_kernel<NT, MT, PIPE>), dim3(grid), dim3(RT_THREADS), lds, s, a);
  MOE_CHECK_LAUNCH();
  return MOE_OK;
}

// ---- K split over workgroups -----------------------------------------------------------------------------------
//
// Copy of w in the order router_split_kernel's fragment reads want it: for expert group b (EP experts), K step s, 16
// experts n, half step kk and lane g * 16 + c the 16 bytes of expert b * EP + 16 n + c, K = 64 s + 32 kk + 8 g .. + 7, at
// ((((b * nsteps + s) * EP / 16 + n) * 2 + kk) * 64 + lane) * 16.  Experts past E are zeros.  A workgroup turns 64 K x 64
// experts.  The padding token's row of the affinity table (pad_bytes at pad) is cleared on the side.
__global__ __launch_bounds__(256) void router_pack_w_kernel(const uint16_t* __restrict__ w, uint8_t* __restrict__ dst,
                                                            int64_t H, int64_t E, int EP, uint8_t* __restrict__ pad,
                                                            int64_t pad_bytes) {
  __shared__ __attribute__((aligned(16))) uint16_t tile[64][72];
  const int64_t s = blockIdx.x, e0 = (int64_t)blockIdx.y * 64, nsteps = H / RT_K;
  const int tid = threadIdx.x;
  if (E % 8 == 0 && ((uintptr_t)w & 15) == 0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = i * 32 + (tid >> 3), x = (tid & 7) * 8;
      v4i v = {0, 0, 0, 0};
      if (e0 + x < E) v = *(const v4i*)(w + (s * RT_K + r) * E + e0 + x);
      *(v4i*)&tile[r][x] = v;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = i * 4 + (tid >> 6), x = tid & 63;
      tile[r][x] = (e0 + x < E) ? w[(s * RT_K + r) * E + e0 + x] : (uint16_t)0;
    }
  }
  if (s == 0 && e0 == 0)
    for (int64_t i = tid; i < pad_bytes; i += 256) pad[i] = 0;
  __syncthreads();
  const int64_t b = e0 / EP;
  uint8_t* out = dst + ((b * nsteps + s) * EP + (e0 - b * EP)) * (RT_K * 2);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int piece = i * 256 + tid, lane = piece & 63, kk = (piece >> 6) & 1, n = piece >> 7;
    const int k0 = kk * 32 + (lane >> 4) * 8, x = n * 16 + (lane & 15);
    v4i v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = (int)((uint32_t)tile[k0 + 2 * j][x] | ((uint32_t)tile[k0 + 2 * j + 1][x] << 16));
    *(v4i*)(out + (int64_t)piece * 16) = v;
  }
}

struct RouterSplitArgs {
  const uint16_t* x;   // bf16 [T, H], 16-byte aligned
  const uint8_t* w;    // the copy above
  float* part;         // [nsplit][T][pitch] fp32
  int64_t T, H, pitch;
  int nsplit, egroups; // K parts, groups of EP experts
};

// Partial logits of M tokens x EP = 64 EG experts over one of nsplit parts of K: 8 waves, EG of them side by side in the
// experts (64 each), the others in the tokens (16 TW each), operands through a ring of RING LDS stages that the loads of
// RING - 1 steps are under way to.
template <int EG, int TW, int RING>
__global__ __launch_bounds__(512) void router_split_kernel(const RouterSplitArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  constexpr int EP = 64 * EG, TG = 8 / EG, M = 16 * TW * TG;
  constexpr int A_BYTES = M * 128, STAGE = A_BYTES + EP * 128;
  constexpr int NA = M / 64, NW = EG, NL = NA + NW;  // loads of a wave per step: 1 KB pieces of the tokens, of w
  const int tid = threadIdx.x, lane = tid & 63, w = rt_uni(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  // (workgroup ids go round the 8 XCDs: consecutive ids are the parts of one tile, so that an XCD keeps few parts of w)
  const int split = (int)(blockIdx.x % a.nsplit);
  const int tile = (int)(blockIdx.x / a.nsplit);
  const int64_t b = tile % a.egroups, t0 = (int64_t)(tile / a.egroups) * M;
  const int nsteps = (int)(a.H / RT_K);
  const int s0 = (int)((int64_t)nsteps * split / a.nsplit), s1 = (int)((int64_t)nsteps * (split + 1) / a.nsplit);

  const int n = s1 - s0;

  // token rows past T lie behind the end of the descriptor: zeros, and nothing is stored for them
  const int64_t rows = a.T - t0 < M ? a.T - t0 : M;
  const v4i rx = rt_rsrc(a.x + t0 * a.H, (uint32_t)(rows * a.H * 2));
  const v4i rw = rt_rsrc(a.w + b * nsteps * (int64_t)(EP * 128), (uint32_t)((int64_t)nsteps * EP * 128));
  // a token piece is 8 rows x 128 bytes: lane l fills slot l & 7 of row l >> 3 with chunk slot ^ ((row >> 1) & 7)
  uint32_t x_voff[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int row = 8 * (NA * w + i) + (lane >> 3);
    x_voff[i] = (uint32_t)(row * a.H * 2 + (((lane & 7) ^ ((row >> 1) & 7)) * 16));
  }
  const uint32_t w_voff = (uint32_t)(lane * 16);
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
  auto issue = [&](int s, uint32_t stage) {  // (steps past the end: descriptors of no records, no traffic)
    v4i dx = rx, dw = rw;
    dx[2] = rt_uni(s < n ? rx[2] : 0);
    dw[2] = rt_uni(s < n ? rw[2] : 0);
    const int kx = rt_uni((s0 + s) * (RT_K * 2)), kw = rt_uni((s0 + s) * (EP * 128));
    const uint32_t l = rt_uni((int)(lds0 + stage));
#pragma unroll
    for (int i = 0; i < NA; ++i) rt_ld_lds(l + (uint32_t)(NA * w + i) * 1024, x_voff[i], dx, kx);
#pragma unroll
    for (int i = 0; i < NW; ++i)
      rt_ld_lds(l + A_BYTES + (uint32_t)(NW * w + i) * 1024, w_voff, dw, kw + (NW * w + i) * 1024);
  };

  v4f acc[TW][4];
#pragma unroll
  for (int m = 0; m < TW; ++m)
#pragma unroll
    for (int n = 0; n < 4; ++n) acc[m][n] = (v4f){0.f, 0.f, 0.f, 0.f};

  const int eg = w % EG, tg = w / EG;
  const int row0 = tg * TW * 16 + c;  // (rows 16 apart have the same swizzle)
  const int sw = (c >> 1) & 7;
  const uint8_t* pa[2];
  pa[0] = smem + row0 * 128 + ((g ^ sw) * 16);
  pa[1] = smem + row0 * 128 + (((4 + g) ^ sw) * 16);
  const uint8_t* pw = smem + A_BYTES + eg * 8192 + lane * 16;

#pragma unroll
  for (int i = 0; i < RING - 1; ++i) issue(i, (uint32_t)(i * STAGE));
  uint32_t rd = 0, wr = (RING - 1) * STAGE;
  for (int s = 0; s < n; ++s) {
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"((RING - 2) * NL) : "memory");  // this wave's pieces of step s are in
    __syncthreads();  // everybody's are; everybody has left the stage of step s - 1
    issue(s + RING - 1, wr);
    wr = wr == (RING - 1) * STAGE ? 0 : wr + STAGE;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      v8bf fw[4], fx[TW];
#pragma unroll
      for (int n = 0; n < 4; ++n) fw[n] = *(const v8bf*)(pw + rd + (n * 2 + kk) * 1024);
#pragma unroll
      for (int m = 0; m < TW; ++m) fx[m] = *(const v8bf*)(pa[kk] + rd + m * 2048);
      // (experts are the rows of the result: a lane ends up with four neighbouring experts of one token)
#pragma unroll
      for (int m = 0; m < TW; ++m)
#pragma unroll
        for (int n = 0; n < 4; ++n) acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[n], fx[m], acc[m][n], 0, 0, 0);
    }
    rd = rd == (RING - 1) * STAGE ? 0 : rd + STAGE;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the empty loads past the end

#pragma unroll
  for (int m = 0; m < TW; ++m) {
    const int64_t t = t0 + row0 + 16 * m;
    if (t < a.T) {
      float* p = a.part + ((int64_t)split * a.T + t) * a.pitch + b * EP + eg * 64 + 4 * g;
#pragma unroll
      for (int n = 0; n < 4; ++n) *(v4f*)(p + 16 * n) = acc[m][n];
    }
  }
}

// Moves within the 16 lanes of a token: lane ^ 1, lane ^ 2, and the mirrors of 8 and of 16 lanes, which stand for ^ 4
// and ^ 8 once the lanes of a quad (of 8) agree.
template <int CTRL>
__device__ __forceinline__ int dpp(int v) { return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false); }
constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E, DPP_MIRROR8 = 0x141, DPP_MIRROR16 = 0x140;
template <class F>
__device__ __forceinline__ int row16_all(int v, F&& f) {
  v = f(v, dpp<DPP_XOR1>(v));
  v = f(v, dpp<DPP_XOR2>(v));
  v = f(v, dpp<DPP_MIRROR8>(v));
  return f(v, dpp<DPP_MIRROR16>(v));
}

// Sums the parts and selects, 16 lanes per token, four neighbouring experts per lane and 16-byte load.  Where the table
// is zero outside the selected experts (every form but the plain activation of all experts) lane j of a token carries
// the j-th selected expert: one activation per lane instead of one per expert, maxima over the lanes without LDS
// round trips, and the row goes out through LDS.  T = 8192, E = 256, top-8, four parts: 19.0 -> 13.1 us.
template <int NT>
__global__ __launch_bounds__(256) void router_select_kernel(const RouterArgs a, const float* __restrict__ part, int64_t pitch,
                                                            int nsplit) {
  __shared__ __attribute__((aligned(16))) float s_row[16][16 * NT];
  const int c = threadIdx.x & 15, row = threadIdx.x >> 4;
  const int64_t t = (int64_t)blockIdx.x * 16 + row;
  const bool live = t < a.T;
  const float* p = part + (live ? t : 0) * pitch + c * 4;
  const int64_t step = a.T * pitch;
  float v[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) v[n] = 0.f;
#pragma unroll 4
  for (int i = 0; i < nsplit; ++i) {
#pragma unroll
    for (int j = 0; j < NT / 4; ++j) {
      const v4f q = *(const v4f*)(p + i * step + j * 64);
#pragma unroll
      for (int r = 0; r < 4; ++r) v[4 * j + r] += q[r];
    }
  }
#pragma unroll
  for (int n = 0; n < NT; ++n) v[n] += expert_bias(a, ColsOf4::expert(n, c));
  if (a.pre_norm && !a.norm_topk && !a.mask_to_topk) {  // (uniform)
    select_and_store<NT, ColsOf4>(a, t, live, c, v);
    return;
  }
  const float NEG = -__builtin_inff();
#pragma unroll
  for (int n = 0; n < NT; ++n)
    if (ColsOf4::expert(n, c) >= a.E) v[n] = NEG;
#pragma unroll
  for (int j = 0; j < NT / 4; ++j) *(v4f*)&s_row[row][j * 64 + c * 4] = (v4f){0.f, 0.f, 0.f, 0.f};
  if (a.logits_out && live) {
#pragma unroll
    for (int n = 0; n < NT; ++n)
      if (ColsOf4::expert(n, c) < a.E) store_val(a.logits_out, a.logits_dtype, t * a.E + ColsOf4::expert(n, c), v[n]);
  }
  float mx = 0.f, sum = 0.f;
  if (a.pre_norm && a.act_fn == 1) {  // softmax over all experts: its largest value and its sum
    mx = NEG;
#pragma unroll
    for (int n = 0; n < NT; ++n) mx = fmaxf(mx, v[n]);
    mx = row16_max(mx);
#pragma unroll
    for (int n = 0; n < NT; ++n) sum += (v[n] == NEG) ? 0.f : expf(v[n] - mx);
    sum = row16_sum(sum);
  }
  // k rounds: the largest value left, the lowest expert that has it; its lane retires it and lane j keeps it
  float my_v = 0.f;
  int my_i = 0;
  for (int j = 0; j < a.k; ++j) {
    float bv = NEG;
#pragma unroll
    for (int n = 0; n < NT; ++n) bv = fmaxf(bv, v[n]);
    bv = __int_as_float(row16_all(__float_as_int(bv), [](int x, int y) {
      return __float_as_int(fmaxf(__int_as_float(x), __int_as_float(y)));
    }));
    int bn = 0x7fffffff;  // (nothing above -inf is left: no expert, as in select_and_store)
#pragma unroll
    for (int n = NT - 1; n >= 0; --n) bn = (v[n] == bv && bv != NEG) ? n : bn;
    const int mine = bn == 0x7fffffff ? bn : ColsOf4::expert(bn, c);
    const int bi = row16_all(mine, [](int x, int y) { return x < y ? x : y; });
    if (mine == bi) {
#pragma unroll
      for (int n = 0; n < NT; ++n) v[n] = n == bn ? NEG : v[n];
    }
    my_v = c == j ? bv : my_v;
    my_i = c == j ? bi : my_i;
  }
  const bool has = c < a.k;
  float aff = 0.f;
  if (a.pre_norm) {
    if (a.act_fn == 1) aff = (my_v == NEG) ? 0.f : expf(my_v - mx) / sum;
    else aff = 1.0f / (1.0f + expf(-my_v));
    if (!has || my_i >= (int)a.E) aff = 0.f;
    if (a.norm_topk) {
      const float ssum = row16_sum(aff);
      aff = aff / ssum;
    }
  } else {  // activation of the k selected logits only
    const float top = __shfl(my_v, threadIdx.x & 48, 64);
    aff = (a.act_fn == 1) ? expf(my_v - top) : 1.0f / (1.0f + expf(-my_v));
    if (a.act_fn == 1) {
      const float ssum = row16_sum(has ? aff : 0.f);
      aff = aff / ssum;
    }
  }
  __syncthreads();
  if (has && my_i < (int)a.E) s_row[row][my_i] = aff;
  if (has && live) {
    if (a.index_out) a.index_out[t * a.k + c] = my_i;
    if (a.topk_aff_out && my_i < (int)a.E) a.topk_aff_out[t * a.k + c] = aff;
  }
  __syncthreads();
  // the 16 rows of the workgroup are neighbours in the table
  const int64_t t0 = (int64_t)blockIdx.x * 16;
  const int rows = (int)(a.T - t0 < 16 ? a.T - t0 : 16), E = (int)a.E;
  if (a.aff_dtype == MOE_DT_BF16 && E % 4 == 0 && ((uintptr_t)a.aff_out & 7) == 0) {
    const int per = E / 4;  // 8-byte pieces of a row
    uint2* out = (uint2*)((uint16_t*)a.aff_out + t0 * E);
    for (int r = threadIdx.x / 64; r < rows; r += 4)
      for (int i = threadIdx.x & 63; i < per; i += 64) {
        const v4f q = *(const v4f*)&s_row[r][i * 4];
        out[r * per + i] = make_uint2((uint32_t)f32_to_bf16_bits(q[0]) | ((uint32_t)f32_to_bf16_bits(q[1]) << 16),
                                      (uint32_t)f32_to_bf16_bits(q[2]) | ((uint32_t)f32_to_bf16_bits(q[3]) << 16));
      }
  } else {
    for (int r = threadIdx.x / 64; r < rows; r += 4)
      for (int i = threadIdx.x & 63; i < E; i += 64) store_val(a.aff_out, a.aff_dtype, (t0 + r) * E + i, s_row[r][i]);
  }
}

// Tiling of a call: experts in groups of 64, 128 or 256, tokens in tiles of 64 or 128, K in as many parts as fill the
// 256 CUs, 16 at most (each part adds a write and a read of the logits).  Tiles of 128 tokens bring w into the CUs half
// as often but need twice the parts for the same number of workgroups: 63 against 71 us at T = 8192, H = 7168, E = 256,
// 42 against 38 at T = 2048, H = 4096, E = 256, 32 against 29.5 at T = 8192, H = 2048, E = 128, 90 against 113 at
// T = 20000, H = 4096, E = 160 (times of a pass before the selection below was written).
struct RouterTiling {
  int EP, M, nsplit;
  int64_t tiles, egroups, pitch;
  size_t w_bytes, part_bytes;
};
static RouterTiling router_tiling(int64_t T, int64_t H, int64_t E) {
  RouterTiling r;
  r.EP = E <= 64 ? 64 : E <= 128 ? 128 : 256;
  r.M = T > (r.EP == 64 ? 0 : r.EP == 128 ? 8192 : 4096) ? 128 : 64;
  r.egroups = (E + r.EP - 1) / r.EP;
  r.pitch = r.egroups * r.EP;
  r.tiles = (T + r.M - 1) / r.M * r.egroups;
  const int64_t nsteps = H / RT_K;
  int64_t n = r.tiles ? 256 / r.tiles : 1;
  if (n > 16) n = 16;
  if (n > nsteps / 2) n = nsteps / 2;
  r.nsplit = (int)(n < 1 ? 1 : n);
  r.w_bytes = (size_t)r.pitch * H * 2;
  r.part_bytes = (size_t)r.nsplit * T * r.pitch * 4;
  return r;
}
// (byte offsets of one tile's rows and of one expert group's weights are kept in 32 bits, grid sizes too)
static bool router_split_ok(int64_t T, int64_t H) { return H <= ((int64_t)1 << 20) && T < ((int64_t)1 << 31); }

template <int EG, int TW, int RING>
static int launch_router_split(const RouterSplitArgs& a, int64_t tiles, hipStream_t s) {
  constexpr int M = 16 * TW * (8 / EG);
  const size_t lds = (size_t)RING * (M + 64 * EG) * 128;
  if (allow_lds<&router_split_kernel<EG, TW, RING>>((int)lds) != hipSuccess) return MOE_E_LAUNCH;
  hipLaunchKernelGGL((router_split_kernel<EG, TW, RING>), dim3((unsigned)(tiles * a.nsplit)), dim3(512), lds, s, a);
  MOE_CHECK_LAUNCH();
  return MOE_OK;
}

static int launch_router_split_path(const RouterArgs& r, const void* w, const RouterTiling& q, int64_t pad_bytes, void* ws,
                                    hipStream_t s) {
  RouterSplitArgs a;
  a.x = r.x; a.w = (const uint8_t*)ws; a.part = (float*)((uint8_t*)ws + q.w_bytes);
  a.T = r.T; a.H = r.H; a.pitch = q.pitch; a.nsplit = q.nsplit; a.egroups = (int)q.egroups;
  uint8_t* pad = (uint8_t*)r.aff_out + r.T * pad_bytes;
  hipLaunchKernelGGL(router_pack_w_kernel, dim3((unsigned)(r.H / RT_K), (unsigned)(q.pitch / 64)), dim3(256), 0, s,
                     (const uint16_t*)w, (uint8_t*)ws, r.H, r.E, q.EP, pad, pad_bytes);
  MOE_CHECK_LAUNCH();
  int rc;
  if (q.EP == 256) rc = q.M == 128 ? launch_router_split<4, 4, 3>(a, q.tiles, s) : launch_router_split<4, 2, 4>(a, q.tiles, s);
  else if (q.EP == 128) rc = q.M == 128 ? launch_router_split<2, 2, 4>(a, q.tiles, s) : launch_router_split<2, 1, 6>(a, q.tiles, s);
  else rc = launch_router_split<1, 1, 6>(a, q.tiles, s);
  if (rc != MOE_OK) return rc;
  const dim3 grid((unsigned)((r.T + 15) / 16));
  if (q.pitch == 64) hipLaunchKernelGGL(router_select_kernel<4>, grid, dim3(256), 0, s, r, a.part, q.pitch, q.nsplit);
  else if (q.pitch == 128) hipLaunchKernelGGL(router_select_kernel<8>, grid, dim3(256), 0, s, r, a.part, q.pitch, q.nsplit);
  else if (q.pitch == 256) hipLaunchKernelGGL(router_select_kernel<16>, grid, dim3(256), 0, s, r, a.part, q.pitch, q.nsplit);
  else hipLaunchKernelGGL(router_select_kernel<32>, grid, dim3(256), 0, s, r, a.part, q.pitch, q.nsplit);
  MOE_CHECK_LAUNCH();
  return MOE_OK;
}

}  // namespace moe

using namespace moe;

extern "C" size_t moe_router_topk_workspace_bytes(int64_t H, int64_t E) { return (size_t)(H * E * 2 + 256); }

extern "C" size_t moe_router_topk_workspace_bytes_for(int64_t T, int64_t H, int64_t E) {
  const size_t least = moe_router_topk_workspace_bytes(H, E);
  if (T <= 0 || H <= 0 || E <= 0 || E > 512 || H % RT_K != 0 || !router_split_ok(T, H)) return least;
  const RouterTiling q = router_tiling(T, H, E);
  const size_t n = q.w_bytes + q.part_bytes;
  return n > least ? n : least;
}

extern "C" int moe_router_topk(const void* x, const void* w, const void* w_bias, int bias_dtype, int64_t T, int64_t H,
                               int64_t E, int k, int act_fn, int router_pre_norm, int norm_topk_prob, int mask_to_topk,
                               int pad_row, void* router_logits, int logits_dtype, int32_t* expert_index,
                               void* expert_affinities, int aff_dtype, float* topk_affinities, void* workspace,
                               size_t workspace_bytes, void* stream) {
  if (!x || !w || !expert_affinities || !workspace) return MOE_E_BAD_ARG;
  if (T < 0 || H <= 0 || E <= 0 || k <= 0 || k > 8 || k > E) return MOE_E_BAD_ARG;
  if (act_fn != 0 && act_fn != 1) return MOE_E_BAD_ARG;
  if (H % RT_K != 0 || E > 512) return MOE_E_BAD_SHAPE;
  if (aff_dtype != MOE_DT_BF16 && aff_dtype != MOE_DT_FP32) return MOE_E_BAD_ARG;
  if (router_logits && logits_dtype != MOE_DT_BF16 && logits_dtype != MOE_DT_FP32) return MOE_E_BAD_ARG;
  if (w_bias && bias_dtype != MOE_DT_BF16 && bias_dtype != MOE_DT_FP32 && bias_dtype != MOE_DT_FP16) return MOE_E_BAD_ARG;
  if (workspace_bytes < moe_router_topk_workspace_bytes(H, E)) return MOE_E_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  RouterArgs a;
  a.x = (const uint16_t*)x; a.wt = (const uint16_t*)workspace; a.bias = w_bias; a.bias_dtype = bias_dtype;
  a.T = T; a.H = H; a.E = E; a.k = k; a.act_fn = act_fn; a.pre_norm = router_pre_norm; a.norm_topk = norm_topk_prob;
  a.mask_to_topk = mask_to_topk;
  a.logits_out = router_logits; a.logits_dtype = logits_dtype; a.index_out = expert_index;
  a.aff_out = expert_affinities; a.aff_dtype = aff_dtype; a.topk_aff_out = topk_affinities;
  const int64_t pad_bytes = E * (aff_dtype == MOE_DT_BF16 ? 2 : 4);
  if (T > 0 && router_split_ok(T, H) && ((uintptr_t)x & 15) == 0 && ((uintptr_t)workspace & 15) == 0) {
    const RouterTiling q = router_tiling(T, H, E);
    if (workspace_bytes >= q.w_bytes + q.part_bytes)
      return launch_router_split_path(a, w, q, pad_row ? pad_bytes : 0, workspace, s);
  }
  if (pad_row) {
    // row T of the affinity table is the padding token's: zeros (E elements)
    hipLaunchKernelGGL(fill_zero_bytes_kernel, dim3(1), dim3(256), 0, s,
                       (uint8_t*)expert_affinities + T * pad_bytes, pad_bytes);
    MOE_CHECK_LAUNCH();
  }
  if (T == 0) return MOE_OK;
  hipLaunchKernelGGL(transpose_w_kernel, dim3((unsigned)((H + 31) / 32), (unsigned)((E + 31) / 32)), dim3(256), 0, s,
                     (const uint16_t*)w, (uint16_t*)workspace, H, E);
  MOE_CHECK_LAUNCH();
  // the pipelined kernel addresses x and wt with 32-bit byte offsets
  const bool small = T * H * 2 < ((int64_t)1 << 31) && E * H * 2 < ((int64_t)1 << 31);
  if (E <= 128) return small ? launch_router<8, 1, true>(a, s) : launch_router<8, 2, false>(a, s);
  if (E <= 256) return small ? launch_router<16, 1, true>(a, s) : launch_router<16, 2, false>(a, s);
  return launch_router<32, 2, false>(a, s);
}
