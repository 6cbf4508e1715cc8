// fused_moe_gfx950.hip -- MI355X (gfx950, CDNA4) kernels and C-ABI of the
// fused mixture-of-experts op of track 03 (include/fused_moe.h).
//
// Math (track-03/reference/reference.py:10-35), per token t: fp32 softmax of
// the bf16 router scores, the topk largest (lower expert index first on
// ties), optional renormalisation, bf16 weights; per selected expert e:
// x = bf16(h . w1[e]^T), u = bf16(x[N:] * bf16(silu(x[:N]))),
// y = bf16(u . w2[e]^T); out[t] = bf16 running sum over the selected experts
// in ascending order of bf16(y * w_e). Every bf16 rounding sits where the
// reference's bf16 tensors round, so the HIP path differs from the oracle
// only by the order of the fp32 sums inside the two GEMMs.
//
// Kernels of one call
// -------------------
// fm_route_kernel   one wave per token: softmax over E, top-k by repeated
//   wave-wide argmax on (weight, lower index), ids and bf16 weights written
//   in ascending expert order (the order of the final sum), and each
//   work-group's pairs counted per expert.
// fm_plan_kernel    as many work-groups: pairs (t, slot) listed by expert,
//   tiles of up to `tile_rows` pairs of one expert. Up to 16 tokens both are
//   one work-group's work (fm_route_plan_kernel).
// fm_gemm_kernel<gated>   (prefill, and decode over few experts) a tile of up
//   to 256 pairs x 256 weight rows (wide) or 64 (narrow) per work-group, K in
//   64-wide stages through LDS rings filled by LDS-DMA (1 KiB per wave
//   instruction, XOR-swizzled so the MFMA fragment reads are free of bank
//   conflicts), 32x32x16 bf16 MFMA, fp32 accumulation. gated: w1 rows j (gate)
//   and N + j (up) sit in the same lane and register, so silu(gate) * up is
//   formed in the epilogue. Otherwise (w2): the epilogue multiplies by the
//   pair's routing weight.
// fm_skinny_kernel<gated, PB>  (few tokens per expert: decode) the weights
//   are the streamed operand: each wave loads its 32 weight rows' MFMA
//   fragments straight from HBM into registers (8 k-steps, 24-32 KiB, in
//   flight per wave), the 16 * PB pairs' fragments likewise (L2-resident),
//   and the 4 waves of a work-group split K and add their partial sums
//   through LDS. 16x16x32 bf16 MFMA.
// fm_reduce_kernel  out[t] = bf16 running sum of the token's topk weighted
//   expert outputs, ascending expert order. Not launched when topk <= 2, N % 256
//   == 0 and experts have few pairs (decode): the routing launch clears out, and the
//   down GEMM adds each weighted row into it with packed bf16 atomics (the
//   two-term bf16 sum does not depend on the order).
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "fm_plan.h"
#include "fused_moe.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) uint8_t lds_u8_t;

using namespace fm;  // fm_plan.h

constexpr int kBK = 64;           // k per LDS stage
constexpr int kRowBytes = kBK * 2;

// ---------------------------------------------------------------------------
// device helpers
// ---------------------------------------------------------------------------
__device__ __forceinline__ float bf16r(float x) {  // round to the nearest bf16
  return static_cast<float>(static_cast<__bf16>(x));
}

// silu in fp32, as torch's bf16 silu computes it before its rounding
__device__ __forceinline__ float silu(float x) { return x / (1.f + expf(-x)); }

__device__ __forceinline__ float wave_max(float x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x = fmaxf(x, __shfl_xor(x, o));
  return x;
}

__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
  return x;
}

// Largest of the 64 lanes' values, in every lane: DPP moves within the rows of
// 16 lanes, then across them (six dependent VALU steps; a 64-bit shuffle
// butterfly took two LDS round trips per step).
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t x) {
#define FM_DPP_MAX(ctrl, rows) \
  x = max(x, uint32_t(__builtin_amdgcn_update_dpp(int(x), int(x), ctrl, rows, 0xf, false)))
  FM_DPP_MAX(0x111, 0xf);  // row_shr:1, 2, 4, 8: lane 15 of a row holds the row's maximum
  FM_DPP_MAX(0x112, 0xf);
  FM_DPP_MAX(0x114, 0xf);
  FM_DPP_MAX(0x118, 0xf);
  FM_DPP_MAX(0x142, 0xa);  // row_bcast:15 into rows 1 and 3
  FM_DPP_MAX(0x143, 0xc);  // row_bcast:31 into rows 2 and 3
#undef FM_DPP_MAX
  return uint32_t(__builtin_amdgcn_readlane(int(x), 63));
}

// LDS-DMA of 16 bytes per lane from SGPR base + 32-bit lane offset into
// LDS bytes lds_addr + 16 * lane. The LDS address is handed to the compiler
// as the M0 operand; s_nop 0 covers the wait state after its write. The
// compiler does not see the LDS write: the caller waits (vmcnt) and
// synchronizes before the data is read.
__device__ __forceinline__ void lds_dma(const void* base, uint32_t lane_off, uint32_t lds_addr) {
  asm volatile(
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %0, %1"
      :
      : "v"(lane_off), "s"(base), "{m0}"(lds_addr)
      : "memory");
}

// Work-group barrier that orders LDS traffic only (lgkmcnt = 0, then
// s_barrier): LDS-DMA loads issued earlier keep flying across it, where
// __syncthreads() would drain every outstanding global load.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);  // vmcnt = max, expcnt = max, lgkmcnt = 0
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// s_waitcnt vmcnt(n) for a wave-uniform n known only at run time.
__device__ __forceinline__ void wait_vmcnt(int n) {  // n uniform, 0..24
  switch (n) {
    case 0: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
    case 1: asm volatile("s_waitcnt vmcnt(1)" ::: "memory"); break;
    case 2: asm volatile("s_waitcnt vmcnt(2)" ::: "memory"); break;
    case 3: asm volatile("s_waitcnt vmcnt(3)" ::: "memory"); break;
    case 4: asm volatile("s_waitcnt vmcnt(4)" ::: "memory"); break;
    case 5: asm volatile("s_waitcnt vmcnt(5)" ::: "memory"); break;
    case 6: asm volatile("s_waitcnt vmcnt(6)" ::: "memory"); break;
    case 7: asm volatile("s_waitcnt vmcnt(7)" ::: "memory"); break;
    case 8: asm volatile("s_waitcnt vmcnt(8)" ::: "memory"); break;
    case 9: asm volatile("s_waitcnt vmcnt(9)" ::: "memory"); break;
    case 10: asm volatile("s_waitcnt vmcnt(10)" ::: "memory"); break;
    case 11: asm volatile("s_waitcnt vmcnt(11)" ::: "memory"); break;
    case 12: asm volatile("s_waitcnt vmcnt(12)" ::: "memory"); break;
    case 13: asm volatile("s_waitcnt vmcnt(13)" ::: "memory"); break;
    case 14: asm volatile("s_waitcnt vmcnt(14)" ::: "memory"); break;
    case 15: asm volatile("s_waitcnt vmcnt(15)" ::: "memory"); break;
    case 16: asm volatile("s_waitcnt vmcnt(16)" ::: "memory"); break;
    case 17: asm volatile("s_waitcnt vmcnt(17)" ::: "memory"); break;
    case 18: asm volatile("s_waitcnt vmcnt(18)" ::: "memory"); break;
    case 19: asm volatile("s_waitcnt vmcnt(19)" ::: "memory"); break;
    case 20: asm volatile("s_waitcnt vmcnt(20)" ::: "memory"); break;
    case 21: asm volatile("s_waitcnt vmcnt(21)" ::: "memory"); break;
    case 22: asm volatile("s_waitcnt vmcnt(22)" ::: "memory"); break;
    case 23: asm volatile("s_waitcnt vmcnt(23)" ::: "memory"); break;
    default: asm volatile("s_waitcnt vmcnt(24)" ::: "memory"); break;
  }
}

// ============================================================================
// routing
// ============================================================================
struct RouteParams {
  const __bf16* score;
  int64_t s_score;
  int32_t* ids;     // [M, topk] ascending expert ids; bits 8..31: see fm_route_kernel
  float* wts;       // [M, topk] bf16-rounded weights (as fp32)
  int32_t* hist;    // [work-groups, E] pairs per expert of a work-group's tokens
  int64_t M;
  int tokens_per_wg;
  int E, topk, renormalize;
  // when the down GEMM adds into the output itself: the rows to clear
  __bf16* zero_out;
  int64_t s_out;
  int K;
};

// Clears output row t (K bf16, 16-byte aligned) by one wave.
__device__ __forceinline__ void clear_out_row(const RouteParams& p, int64_t t, int lane) {
  __bf16* row = p.zero_out + t * p.s_out;
  bf16x8 z;
#pragma unroll
  for (int e = 0; e < 8; ++e) z[e] = static_cast<__bf16>(0.f);
  for (int k = 8 * lane; k < p.K; k += 8 * 64) *reinterpret_cast<bf16x8*>(row + k) = z;
}

// Routing of token t by one wave; lane l holds experts l + 64 i, i < kPer
// (kPer = 1 for E <= 64, else 4). `raw` are the token's scores as loaded (bf16
// widened; -inf past E). `id(slot, e)` takes the selected experts in ascending
// order of e, one call by the lane that holds e.
template <int kPer>
__device__ __forceinline__ void load_scores(const RouteParams& p, int64_t t, int lane,
                                            float (&raw)[kPer]) {
  const __bf16* srow = p.score + t * p.s_score;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int e = lane + 64 * i;
    raw[i] = e < p.E ? static_cast<float>(srow[e]) : -INFINITY;
  }
}

template <int kPer, typename Id>
__device__ __forceinline__ void route_token(const RouteParams& p, int64_t t, int lane,
                                            const float (&raw)[kPer], Id id) {
  float v[kPer];
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    v[i] = raw[i];
    mx = fmaxf(mx, v[i]);
  }
  mx = wave_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    v[i] = (lane + 64 * i) < p.E ? expf(v[i] - mx) : 0.f;
    sum += v[i];
  }
  sum = wave_sum(sum);
#pragma unroll
  for (int i = 0; i < kPer; ++i) v[i] = v[i] / sum;  // softmax weight (>= 0)
  // top-k: repeated argmax over (weight, lower index). A weight's bits order
  // like its value (weights are >= 0); among equal ones the lowest lane of the
  // lowest i is the lowest expert.
  bool sel[kPer] = {};
  float tot = 0.f;  // sum of the selected weights, in selection order
  for (int r = 0; r < p.topk; ++r) {
    uint32_t key = 0u;
#pragma unroll
    for (int i = 0; i < kPer; ++i)
      if (!sel[i] && lane + 64 * i < p.E) key = max(key, __float_as_uint(v[i]));
    key = wave_max_u32(key);
    tot += __uint_as_float(key);
    bool found = false;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const unsigned long long m =
          __ballot(!sel[i] && lane + 64 * i < p.E && __float_as_uint(v[i]) == key);
      if (!found && m != 0ull) {
        found = true;
        if (lane == __builtin_ctzll(m)) sel[i] = true;
      }
    }
  }
  // ascending-expert slot of each selected expert: ballots in expert order
  int before = 0;
  const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const unsigned long long m = __ballot(sel[i]);
    if (sel[i]) {
      const int slot = before + __popcll(m & below);
      const float w = p.renormalize ? v[i] / tot : v[i];
      id(slot, lane + 64 * i);
      p.wts[t * p.topk + slot] = bf16r(w);
    }
    before += __popcll(m);
  }
}

// One wave per token, 16 at a time per work-group. Besides its expert a pair
// gets its rank among the work-group's pairs of that expert (bits 8..31 of the
// id), and the work-group's counts go to `hist`: the plan then needs no
// atomics over all pairs.
constexpr int kRouteWaves = 16;
template <int kPer>
__global__ void __launch_bounds__(64 * kRouteWaves) fm_route_kernel(const RouteParams p) {
  __shared__ int s_cnt[kMaxExperts];
  const int lane = threadIdx.x & 63;
  const int64_t t0 = int64_t(blockIdx.x) * p.tokens_per_wg;
  const int64_t t1 = t0 + p.tokens_per_wg < p.M ? t0 + p.tokens_per_wg : p.M;
  for (int e = threadIdx.x; e < p.E; e += 64 * kRouteWaves) s_cnt[e] = 0;
  __syncthreads();
  for (int64_t t = t0 + (threadIdx.x >> 6); t < t1; t += kRouteWaves) {
    float raw[kPer];
    load_scores(p, t, lane, raw);
    route_token(p, t, lane, raw, [&](int slot, int e) {
      p.ids[t * p.topk + slot] = e | atomicAdd(&s_cnt[e], 1) << 8;
    });
    if (p.zero_out != nullptr) clear_out_row(p, t, lane);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < p.E; e += 64 * kRouteWaves)
    p.hist[int64_t(blockIdx.x) * p.E + e] = s_cnt[e];
}

// ============================================================================
// plan: pairs by expert, tiles
// ============================================================================
struct PlanParams {
  const int32_t* ids;   // fm_route_kernel's
  const int32_t* hist;
  int32_t* sorted;    // [P] pair ids (t * topk + slot) grouped by expert
  int32_t* tiles;     // [0] = tile count, [1] = tiles before the narrow ones, then
                      // int4 (expert, start, rows, 0) per tile
  int64_t P;
  int wgs, pairs_per_wg;  // of fm_route_kernel
  int E, tile_rows;
  int narrow_rows;    // tiles of at most this many pairs are listed last (narrow tiles)
};

struct PlanSmem {
  int cnt[kMaxExperts];
  int off[kMaxExperts + 1];
  int toff[kMaxExperts + 1];
  int soff[kMaxExperts + 1];
  int cur[kMaxExperts];
};

// Tiles of an expert with n pairs (tile_rows is a power of two), and how many
// of them (the last one, or all) are narrow.
__device__ __forceinline__ int tiles_of(const PlanParams& p, int n) {
  return (n + p.tile_rows - 1) >> __builtin_ctz(p.tile_rows);
}
__device__ __forceinline__ int narrow_of(const PlanParams& p, int n) {
  const int nt = tiles_of(p, n);
  return p.tile_rows <= p.narrow_rows ? nt
                                      : n > 0 && n - (nt - 1) * p.tile_rows <= p.narrow_rows;
}

// Exclusive scans over the experts, by wave 0, from their counts: first sorted
// position, first wide and first narrow tile.
__device__ __forceinline__ void plan_scan(const PlanParams& p, PlanSmem& sm) {
  const int lane = threadIdx.x;
  int carry = 0, tcarry = 0, scarry = 0;
  for (int e0 = 0; e0 < p.E; e0 += 64) {
    const int e = e0 + lane;
    const int v = e < p.E ? sm.cnt[e] : 0;
    const int sv = narrow_of(p, v);
    const int tv = tiles_of(p, v) - sv;
    int incl = v, tincl = tv, sincl = sv;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int a = __shfl_up(incl, o);
      const int b = __shfl_up(tincl, o);
      if (lane >= o) {
        incl += a;
        tincl += b;
      }
    }
    if (p.narrow_rows > 0) {
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int d = __shfl_up(sincl, o);
        if (lane >= o) sincl += d;
      }
    }
    if (e < p.E) {
      sm.off[e] = carry + incl - v;
      sm.toff[e] = tcarry + tincl - tv;
      sm.soff[e] = scarry + sincl - sv;
    }
    carry += __shfl(incl, 63);
    tcarry += __shfl(tincl, 63);
    scarry += __shfl(sincl, 63);
  }
  if (lane == 0) {
    sm.toff[p.E] = tcarry;
    sm.soff[p.E] = scarry;
  }
}

// The tile table, by the 1024 threads of one work-group, after the scan.
__device__ __forceinline__ void plan_tiles(const PlanParams& p, const PlanSmem& sm) {
  const int tid = threadIdx.x;
  if (tid == 0) {
    p.tiles[0] = sm.toff[p.E] + sm.soff[p.E];
    p.tiles[1] = sm.toff[p.E];
  }
  // 4 threads per expert: its tiles k, k + 4, ...
  for (int i = tid; i < 4 * p.E; i += 1024) {
    const int e = i >> 2;
    const int n = sm.cnt[e];
    const int wide = tiles_of(p, n) - narrow_of(p, n);
    for (int k = i & 3; k * p.tile_rows < n; k += 4) {
      const int at = k < wide ? sm.toff[e] + k : sm.toff[p.E] + sm.soff[e] + k - wide;
      *reinterpret_cast<int4*>(p.tiles + 4 + 4 * at) =
          make_int4(e, sm.off[e] + k * p.tile_rows, min(p.tile_rows, n - k * p.tile_rows), 0);
    }
  }
}

// One work-group per work-group of fm_route_kernel, placing that one's pairs.
// Each adds up the counts of all (they are few: 256 x E at most) for the
// experts' totals and, over the work-groups before it, its own offsets; the
// first also writes the tile table. Against one work-group that counted all
// pairs by LDS atomics: M = 4001, E = 64, topk = 6 21 -> 5 us, M = 4096, E = 8,
// topk = 2 8.5 -> 4.9 us (rocprof).
__global__ void __launch_bounds__(1024) fm_plan_kernel(const PlanParams p) {
  __shared__ PlanSmem sm;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int b = blockIdx.x;
  // this work-group's first pairs, loaded ahead of the counts
  const int64_t i0 = int64_t(b) * p.pairs_per_wg;
  const int64_t i1 = i0 + p.pairs_per_wg < p.P ? i0 + p.pairs_per_wg : p.P;
  const int32_t first = i0 + tid < i1 ? p.ids[i0 + tid] : 0;
  for (int e = tid; e < kMaxExperts; e += 1024) {
    sm.cnt[e] = 0;
    sm.cur[e] = 0;
  }
  __syncthreads();
  // thread (g, e): the work-groups g, g + G, ... of expert e
  const int le = p.E <= 1 ? 0 : 32 - __builtin_clz(p.E - 1);  // log2 of E, rounded up
  const int e = tid & ((1 << le) - 1);
  int tot = 0, pre = 0;
  if (e < p.E) {
    const int step = 1024 >> le;
    for (int w0 = tid >> le; w0 < p.wgs; w0 += 16 * step) {
      int v[16];  // all loads of a batch in flight
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int w = w0 + j * step;
        v[j] = w < p.wgs ? p.hist[w * p.E + e] : 0;
      }
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        tot += v[j];
        pre += w0 + j * step < b ? v[j] : 0;
      }
    }
  }
  for (int o = 1 << le; o < 64; o <<= 1) {
    tot += __shfl_xor(tot, o);
    pre += __shfl_xor(pre, o);
  }
  if (e < p.E && lane >> le == 0) {
    atomicAdd(&sm.cnt[e], tot);
    atomicAdd(&sm.cur[e], pre);
  }
  __syncthreads();
  if (tid < 64) plan_scan(p, sm);
  __syncthreads();
  auto place = [&](int64_t i, int32_t id) {
    const int x = id & 255;
    p.sorted[sm.off[x] + sm.cur[x] + (id >> 8)] = int32_t(i);
  };
  if (i0 + tid < i1) place(i0 + tid, first);
  for (int64_t i = i0 + tid + 1024; i < i1; i += 1024) place(i, p.ids[i]);
  if (b == 0) plan_tiles(p, sm);
}

// Few tokens (decode): routing and plan in one work-group, one launch fewer,
// the ids kept in LDS. Wave w routes token w. M = 1, E = 8, topk = 2: 5.6 ->
// 3.8 us with the DPP argmax and without the ids' way through memory.
template <int kPer>
__global__ void __launch_bounds__(1024) fm_route_plan_kernel(const RouteParams rp,
                                                             const PlanParams pp) {
  __shared__ PlanSmem sm;
  __shared__ int s_id[kFusedTokens * kMaxTopk];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  if (tid < kMaxExperts) sm.cnt[tid] = 0;
  static_assert(kFusedTokens <= 16, "one token per wave");
  float raw[kPer];
  if (wave < rp.M) load_scores(rp, wave, lane, raw);
  __syncthreads();
  if (wave < rp.M) {
    route_token(rp, wave, lane, raw, [&](int slot, int e) {
      s_id[wave * rp.topk + slot] = e | atomicAdd(&sm.cnt[e], 1) << 8;
    });
    if (rp.zero_out != nullptr) clear_out_row(rp, wave, lane);
  }
  __syncthreads();
  if (tid < 64) plan_scan(pp, sm);
  __syncthreads();
  for (int i = tid; i < int(pp.P); i += 1024) {
    const int id = s_id[i];
    pp.sorted[sm.off[id & 255] + (id >> 8)] = i;
  }
  plan_tiles(pp, sm);
}

// ============================================================================
// GEMMs
// ============================================================================
// GEMM 1 (gated): A row r of a tile = hidden[token of pair sorted[start + r]],
//   weight rows = w1[e] rows j (gate) and N + j (up); output u to
//   inter[start + r, j] (sorted pair order).
// GEMM 2: A row r = inter[start + r], weight rows = w2[e] rows f (features);
//   output bf16(bf16(y) * w_pair) to yw[pair, f] (pair = t * topk + slot).
struct GemmParams {
  const __bf16* a;       // hidden or inter
  int64_t a_stride;      // elements per A row
  const __bf16* w;       // w1 or w2
  int64_t w_estride;     // elements per expert
  const int32_t* sorted;
  const int32_t* tiles;  // [0] = count, then int4 per tile
  const float* wts;      // routing weights by pair (GEMM 2)
  __bf16* out;           // inter [P, N] or yw [P, K]
  int64_t out_stride;    // elements per output row
  int kin;               // reduction length: K (GEMM 1) or N (GEMM 2)
  int nout;              // GEMM 1: N (gate rows; up rows follow); GEMM 2: K
  int topk;
  int col_tiles;         // output-column tiles per pair tile
  int narrow_cols;       // ... of a narrow tile (fm_gemm_kernel)
  int ct_per_wg;         // column tiles one work-group runs (fm_stream_kernel)
  // GEMM 2 with topk <= 2 (decode): add each pair's bf16 row into the token's
  // output row instead of writing yw (null: write yw)
  __bf16* fsum;
  int64_t fsum_stride;
};

// out[0..1] += (a0, a1) as one packed bf16 atomic add at agent scope (sc1:
// performed where every XCD sees it; the two addends of an element may come
// from work-groups on different XCDs). Each element gets at most two addends
// onto the cleared 0, so the result is bf16(x + y): the reference's ascending
// running sum, whose two-term form does not depend on the order.
__device__ __forceinline__ void add_bf16x2(__bf16* out, __bf16 a0, __bf16 a1) {
  const uint32_t v = uint32_t(__builtin_bit_cast(uint16_t, a0)) |
                     uint32_t(__builtin_bit_cast(uint16_t, a1)) << 16;
  asm volatile("global_atomic_pk_add_bf16 %0, %1, off sc1" : : "v"(out), "v"(v) : "memory");
}

// ---- fm_gemm_kernel ----------------------------------------------------------------
// Work-group of a wide tile: 256 pairs x 256 weight rows, 8 waves, two per
// SIMD. Wave w takes the 32-pair row blocks of parity w >> 2 against weight
// quarter w & 3 (64 rows, 2 column blocks): 4 x 2 accumulator blocks when the
// tile is full. The blocks alternate between the two wave halves, so a tile of
// n pairs costs ceil(n / 64) block rows of MFMA time whatever n is. A narrow
// tile has 64 weight rows and wave w takes row block w: four times the
// work-groups, each with a short stage (24 or 40 KiB) and so six or four of
// them in LDS. They fill the chip where wide tiles are too few, and run an
// expert's short last tile in a third of the time (8 against 20 us).
// K streams in 64-wide stages (128 bytes of each row: a 64-byte piece costs L2
// and the vector cache as much as a whole 128-byte line, 17 against 31 TB/s
// measured): the pairs' rows (A, from L2) through two LDS buffers of 32 KiB,
// the weights (B, first touched by the launch, so from HBM) through three.
// Row r's 16-byte chunk c sits at swz(r, c): a 32x32x16 fragment read (lanes
// 0..15 = 16 consecutive rows, one chunk) then covers all 64 banks once; each
// lane of an LDS-DMA loads the chunk that belongs at its position. Wave w moves
// the 8-row DMA groups w + 8 g of A and of B; groups of A past the tile's last
// pair are skipped. Every form runs the same MFMA sequence per output element,
// so they agree bit for bit.
// What bounds it: MFMA issue (a full tile is 32 x 2 MFMAs of 32 cycles per
// SIMD and stage against 774 cycles of LDS reads) and the latency of the
// weights, so the loop reads the fragments of a 16-wide k step between the
// MFMAs of the one before, the stage barrier sits between two MFMA batches,
// and the DMAs ride between MFMAs, two stages ahead for the weights.
// Gate-up / down at K = 2048, N = 1024 (rocprof medians), against 32-wide
// stages in pairs, the row blocks of one half per wave half, 2-byte stores and
// wide tiles only: M = 4096, E = 8, topk = 2 123 / 69 -> 78 / 44 us; M = 4001,
// E = 64, topk = 6 317 / 176 -> 258 / 146 us. A full wide gate-up tile takes
// 2.9 us to its first stage, 49 us for its 32 stages (1.40 PFLOP/s over 256
// CUs; without its loads 41 us) and 3.9 us for its epilogue.
enum TileForm { kWide, kNarrow128, kNarrow256 };  // narrow: up to 128 or 256 pairs

__device__ __forceinline__ int swz(int row, int chunk) { return chunk ^ ((row >> 1) & 7); }

template <TileForm kForm>
struct TileShape {  // wide
  static constexpr int kWq = 4;                 // 64-row weight parts, one per wave
  static constexpr int kRows = kTileRows;       // pairs
  static constexpr int kABufs = 2, kBBufs = 3;  // stages of A and B in LDS
};
template <>
struct TileShape<kNarrow128> {
  static constexpr int kWq = 1, kRows = 128, kABufs = 6, kBBufs = 6;
};
template <>
struct TileShape<kNarrow256> {
  static constexpr int kWq = 1, kRows = 256, kABufs = 4, kBBufs = 4;
};
template <TileForm kForm>
struct TileLds : TileShape<kForm> {
  using S = TileShape<kForm>;
  static constexpr int kPh = 8 / S::kWq;             // waves that share a weight part
  static constexpr int kCols = 64 * S::kWq;          // weight rows
  static constexpr int kA = S::kRows * kRowBytes;    // bytes of one stage of A, of B
  static constexpr int kB = kCols * kRowBytes;
  static constexpr int kBytes = S::kABufs * kA + S::kBBufs * kB;
  static constexpr int kAGroups = S::kRows / 64;     // DMA groups per wave and stage
  static constexpr int kBGroups = kCols / 64;
};
constexpr int kGemmLds = TileLds<kWide>::kBytes;  // 160 KiB
static_assert(TileLds<kNarrow128>::kBytes <= kGemmLds && TileLds<kNarrow256>::kBytes <= kGemmLds,
              "narrow stages fit");
// epilogue: each wave passes its outputs through LDS lines of its own
constexpr int kPitchGated = 64 + 16;              // 32 outputs of a pair, padded
constexpr int kPitchDown = 128 + 16;              // 64 outputs of a pair, padded
constexpr int kPairsOff = 8 * 128 * kPitchDown;   // then the waves' pair ids (128 each)
static_assert(kPairsOff + 8 * 128 * 4 <= kGemmLds, "the epilogue fits");

// silu in fp32 with the hardware exponential and reciprocal: exp(-x) as
// 2^(t + r), t + r = -x log2(e) to about 2^-48, and x / (1 + exp(-x)) corrected
// by its remainder. Divisor and dividend are an eighth of theirs, so that the
// reciprocal (the hardware's flushes subnormal results) stays normal up to the
// largest finite 1 + exp(-x). Over every finite bf16 x above -88.7 within 1.77
// ulp of the exact value (silu() above: 1.75), and rounded to bf16 the same bits
// as silu() for all of them; below, the exponential overflows and both are -0.
__device__ __forceinline__ float silu_fast(float x) {
  const float t = x * -1.44269504f;
  const float r = __builtin_fmaf(x, -1.92596299e-8f, __builtin_fmaf(x, -1.44269504f, -t));
  float e = __builtin_amdgcn_exp2f(t);
  // (elsewhere r may not be finite, and e is 0, inf or NaN)
  const bool in = __builtin_fabsf(t) < 128.f;
  e = in ? __builtin_fmaf(e, r * 0.693147181f, e) : e;
  const float d = __builtin_fmaf(e, 0.125f, 0.125f), n = 0.125f * x;
  const float q = __builtin_amdgcn_rcpf(d);
  const float y = n * q;
  return in ? __builtin_fmaf(-__builtin_fmaf(y, d, -n), q, y) : y;
}

// Work item (pair tile, column tile) of a work-group. Work-group b
// runs on XCD b % 8 (dispatch is round-robin over the XCDs, in order of b).
// The items, pair tile by pair tile, are cut into 8 equal runs, one per XCD: a
// pair tile's gathered rows and an expert's weight rows then go to one L2 (two
// at a cut). The narrow tiles come last in the table (tiles[1] = the number
// before them), and each XCD takes its run of their items after its run of the
// wide ones, so that what starts last is short. At M = 4096, E = 8, topk = 2
// each XCD then holds one expert's four full tiles. False: no item for this
// work-group.
__device__ __forceinline__ bool gemm_item(const GemmParams& p, int& tile, int& ct, bool& narrow) {
  const int nt = p.tiles[0], nb = p.tiles[1];
  const int x = int(blockIdx.x) % kXcds;
  int s = int(blockIdx.x) / kXcds;
  const int ib = nb * p.col_tiles, is = (nt - nb) * p.narrow_cols;
  const int b0 = x * ib / kXcds, bn = (x + 1) * ib / kXcds - b0;
  narrow = s >= bn;
  if (!narrow) {
    s += b0;
    tile = s / p.col_tiles;
    ct = s % p.col_tiles;
    return true;
  }
  const int s0 = x * is / kXcds;
  s += s0 - bn;
  tile = nb + s / p.narrow_cols;
  ct = s % p.narrow_cols;
  return s < (x + 1) * is / kXcds;
}

// The K loop and epilogue of one wave's share of a tile; NRB = its 32-pair
// row blocks holding pairs (0: DMAs and barriers only).
template <bool kGated, TileForm kForm, int NRB>
__device__ __forceinline__ void gemm_tile(const GemmParams& p, uint8_t* s_buf, int e, int start,
                                         int rows, int ct) {
  using L = TileLds<kForm>;
  constexpr int kWq = L::kWq, kPh = L::kPh;
  constexpr int kCols = L::kCols;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ph = wave / kWq;  // the wave's row blocks: kPh * i + ph
  const int wq = wave % kWq;  // weight part
  const int l32 = lane & 31;
  const int hi = lane >> 5;
  const int nst = p.kin / kBK;
  constexpr int kRB = NRB > 0 ? NRB : 1;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(
      uint32_t(reinterpret_cast<uintptr_t>((lds_u8_t*)s_buf)));
  const uint8_t* abase = reinterpret_cast<const uint8_t*>(p.a);
  const uint8_t* wbase = reinterpret_cast<const uint8_t*>(p.w + int64_t(e) * p.w_estride);

  // Per-lane DMA sources: instruction g of this wave moves LDS rows
  // 8 * (wave + 8 * g) + lane / 8, lane & 7 being the chunk position there.
  const int sub = lane >> 3;
  const int pos = lane & 7;
  uint32_t a_off[L::kAGroups], b_off[L::kBGroups];
  int64_t arow[L::kAGroups];
#pragma unroll
  for (int g = 0; g < L::kAGroups; ++g) {
    const int r = 8 * (wave + 8 * g) + sub;
    const int at = start + (r < rows ? r : 0);
    arow[g] = kGated ? int64_t(p.sorted[at]) : int64_t(at);
  }
#pragma unroll
  for (int g = 0; g < L::kAGroups; ++g) {
    const int r = 8 * (wave + 8 * g) + sub;
    if (kGated) arow[g] = uint32_t(arow[g]) / uint32_t(p.topk);
    // the chunk whose swizzled position is `pos`
    a_off[g] = uint32_t(arow[g] * p.a_stride * 2 + swz(r, pos) * 16);
  }
#pragma unroll
  for (int g = 0; g < L::kBGroups; ++g) {
    const int r = 8 * (wave + 8 * g) + sub;
    // weight row of LDS row r: weight part r >> 6, column block (r >> 5) & 1
    int wrow;
    if (kGated)  // gate rows j, up rows N + j, j = ct * kCols / 2 + 32 * (r >> 6) + (r & 31)
      wrow = (((r >> 5) & 1) ? p.nout : 0) + ct * (kCols / 2) + 32 * (r >> 6) + (r & 31);
    else         // features f = ct * kCols + r
      wrow = ct * kCols + r;
    b_off[g] = uint32_t(int64_t(wrow) * p.kin * 2 + swz(r, pos) * 16);
  }
  // A instructions of this wave that hold a pair
  const int na = max(0, min(L::kAGroups, (rows - 8 * wave + 63) / 64));
  // DMAs of a stage: A group g into A buffer `ab`, B group g into B buffer `bb`
  auto dma_a = [&](int st, int ab, int g) {
    if (g < na)
      lds_dma(abase + int64_t(st) * kRowBytes, a_off[g],
              lds0 + uint32_t(ab * L::kA + (wave + 8 * g) * 1024));
  };
  auto dma_b = [&](int st, int bb, int g) {
    lds_dma(wbase + int64_t(st) * kRowBytes, b_off[g],
            lds0 + uint32_t(L::kABufs * L::kA + bb * L::kB + (wave + 8 * g) * 1024));
  };

  // the pairs of this lane's accumulator columns and their weights
  int pair[kRB];
  float wt[kRB];
  if constexpr (!kGated && NRB > 0) {
#pragma unroll
    for (int rb = 0; rb < NRB; ++rb)
      pair[rb] = p.sorted[start + min(32 * (kPh * rb + ph) + l32, rows - 1)];
#pragma unroll
    for (int rb = 0; rb < NRB; ++rb) wt[rb] = p.wts[pair[rb]];
  }

  f32x16 acc[kRB][2];
#pragma unroll
  for (int rb = 0; rb < kRB; ++rb)
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[rb][cb][i] = 0.f;

  // fragment f of one 16-wide k step: the 2 weight blocks, then the row blocks
  struct Frags {
    bf16x8 b[2], a[kRB];
  };
  auto read1 = [&](const uint8_t* sa, const uint8_t* sb, int kk, int f, Frags& fr) {
    const int pos = swz(l32, 2 * kk + hi) * 16;
    if (f < 2)
      fr.b[f] = *reinterpret_cast<const bf16x8*>(sb + (64 * wq + 32 * f + l32) * kRowBytes + pos);
    else if (f - 2 < NRB)
      fr.a[f - 2] = *reinterpret_cast<const bf16x8*>(
          sa + (32 * (kPh * (f - 2) + ph) + l32) * kRowBytes + pos);
  };
  // The MFMAs of step (fr), with the reads of the next step (sa, sb, kk) into
  // `nx` between them unless kk < 0; `after(i)` runs after MFMA pair i.
  auto step = [&](const Frags& fr, const uint8_t* sa, const uint8_t* sb, int kk, Frags& nx,
                  auto after) {
#pragma unroll
    for (int rb = 0; rb < NRB; ++rb) {
#pragma unroll
      for (int cb = 0; cb < 2; ++cb)
        acc[rb][cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr.b[cb], fr.a[rb], acc[rb][cb], 0, 0, 0);
      // all reads within the first NRB - 1 pairs (or the only one)
      constexpr int kSlots = NRB > 1 ? NRB - 1 : 1;
      if (kk >= 0 && rb < kSlots) {
#pragma unroll
        for (int f = rb * (NRB + 2) / kSlots; f < (rb + 1) * (NRB + 2) / kSlots; ++f)
          read1(sa, sb, kk, f, nx);
      }
      after(rb);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto nothing = [](int) {};

  // nst >= 2: validate() requires K % 256 == 0 and N % 128 == 0
#pragma unroll
  for (int i = 0; i < L::kBBufs; ++i) {
    if (i > 1 && i >= nst) break;
    if (i < L::kABufs) {
#pragma unroll
      for (int g = 0; g < L::kAGroups; ++g) dma_a(i, i, g);
    }
#pragma unroll
    for (int g = 0; g < L::kBGroups; ++g) dma_b(i, i, g);
  }
  // DMAs of this wave issued after those of stage s when `ahead` stages of B
  // follow it (fewer at the end): what may still fly once stage s has landed
  auto later = [&](int s, int ahead) {
    const int n = max(0, min(ahead, nst - 1 - s));
    return n * (L::kABufs == L::kBBufs ? na + L::kBGroups : L::kBGroups);
  };
  // (the wide tile's counts, in the loop: 4 or 0)
  auto wait_stage = [&](int s) {
    if constexpr (kForm != kWide) {
      wait_vmcnt(later(s, L::kBBufs - 2));
    } else {
      if (s + 1 < nst)
        wait_vmcnt(L::kBGroups);
      else
        wait_vmcnt(0);
    }
  };
  // (wide: A of stage 1 too)
  wait_vmcnt(later(0, L::kBBufs - 1) + (L::kABufs < L::kBBufs ? na : 0));
  lds_barrier();
  const uint8_t* const sb0 = s_buf + L::kABufs * L::kA;
  Frags f0, f1;
#pragma unroll
  for (int f = 0; f < NRB + 2; ++f) read1(s_buf, sb0, 0, f, f0);
  int ab = 0, bb = 0;  // the buffers of stage st
  for (int st = 0; st < nst; ++st) {
    const uint8_t* sa = s_buf + ab * L::kA;
    const uint8_t* sb = sb0 + bb * L::kB;
    const int na1 = ab == L::kABufs - 1 ? 0 : ab + 1, nb1 = bb == L::kBBufs - 1 ? 0 : bb + 1;
    step(f0, sa, sb, 1, f1, nothing);
    step(f1, sa, sb, 2, f0, nothing);
    step(f0, sa, sb, 3, f1, nothing);
    // stage st + 1 has landed, then it has for every wave, and every wave has
    // read stage st (the last pass reads a stale stage ahead, unused)
    wait_stage(st + 1);
    lds_barrier();
    // the DMAs into stage st's buffers
    const bool ma = st + L::kABufs < nst, mb = st + L::kBBufs < nst;
    auto dmas = [&](int rb) {
      constexpr int kN = L::kAGroups + L::kBGroups;
#pragma unroll
      for (int d = rb * kN / kRB; d < (rb + 1) * kN / kRB; ++d) {
        if (d < L::kAGroups) {
          if (ma) dma_a(st + L::kABufs, ab, d);
        } else {
          if (mb) dma_b(st + L::kBBufs, bb, d - L::kAGroups);
        }
      }
    };
    if constexpr (NRB == 0) dmas(0);
    step(f1, s_buf + na1 * L::kA, sb0 + nb1 * L::kB, 0, f0, dmas);
    ab = na1;
    bb = nb1;
  }

  // epilogue: the lane holds, for pair row 32 * (kPh * rb + ph) + l32, weight
  // rows 8 * a + 4 * hi + i of each column block in register 4 * a + i. The outputs
  // go through this wave's own LDS lines, so that global stores write 64
  // (gated) or 128 contiguous bytes of a row by 16 bytes per lane: 2 us instead
  // of 5 for 2-byte stores straight from the accumulators.
  lds_barrier();  // every wave's reads are done
  if constexpr (NRB > 0) {
    constexpr int kPitch = kGated ? kPitchGated : kPitchDown;
    constexpr int kOuts = kGated ? 32 : 64;        // outputs per pair row and wave
    constexpr int kLanes = kOuts / 8;              // lanes per row of a 16-byte store
    uint8_t* const sw = s_buf + wave * (128 * kPitchDown);
    int* const sp = reinterpret_cast<int*>(s_buf + kPairsOff) + 128 * wave;
#pragma unroll
    for (int rb = 0; rb < NRB; ++rb) {
      uint8_t* line = sw + (32 * rb + l32) * kPitch + 8 * hi;
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        if constexpr (kGated) {
          bf16x4 o;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float g = bf16r(silu_fast(bf16r(acc[rb][0][4 * a + i])));
            o[i] = static_cast<__bf16>(bf16r(acc[rb][1][4 * a + i]) * g);
          }
          *reinterpret_cast<bf16x4*>(line + 16 * a) = o;
        } else {
#pragma unroll
          for (int cb = 0; cb < 2; ++cb) {
            bf16x4 o;
#pragma unroll
            for (int i = 0; i < 4; ++i)
              o[i] = static_cast<__bf16>(bf16r(acc[rb][cb][4 * a + i]) * wt[rb]);
            *reinterpret_cast<bf16x4*>(line + 64 * cb + 16 * a) = o;
          }
        }
      }
      if constexpr (!kGated) sp[32 * rb + l32] = pair[rb];  // both halves: the same value
    }
    asm volatile("" ::: "memory");  // one wave: its LDS operations run in order
    const int c = lane % kLanes;
#pragma unroll
    for (int i = 0; i < 32 * NRB / (64 / kLanes); ++i) {
      const int lr = i * (64 / kLanes) + lane / kLanes;     // row within the wave's
      const int r = 32 * (kPh * (lr >> 5) + ph) + (lr & 31);  // row of the tile
      if (r >= rows) continue;
      const bf16x8 v = *reinterpret_cast<const bf16x8*>(sw + lr * kPitch + 16 * c);
      if constexpr (kGated) {
        __bf16* dst = p.out + int64_t(start + r) * p.out_stride + ct * (kCols / 2) + 32 * wq;
        *reinterpret_cast<bf16x8*>(dst + 8 * c) = v;
      } else {
        const int f = ct * kCols + 64 * wq + 8 * c;
        if (p.fsum != nullptr) {
          __bf16* dst = p.fsum + int64_t(uint32_t(sp[lr]) / uint32_t(p.topk)) * p.fsum_stride + f;
#pragma unroll
          for (int j = 0; j < 8; j += 2) add_bf16x2(dst + j, v[j], v[j + 1]);
        } else {
          *reinterpret_cast<bf16x8*>(p.out + int64_t(sp[lr]) * p.out_stride + f) = v;
        }
      }
    }
  }
}

template <bool kGated>
__global__ void __launch_bounds__(512, 1) fm_gemm_kernel(const GemmParams p) {
  __shared__ __attribute__((aligned(1024))) uint8_t s_buf[kGemmLds];
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  int tile, ct;
  bool narrow;
  if (!gemm_item(p, tile, ct, narrow)) return;
  const int32_t* tl = p.tiles + 4 + 4 * tile;
  const int e = __builtin_amdgcn_readfirstlane(tl[0]);
  const int start = __builtin_amdgcn_readfirstlane(tl[1]);
  const int rows = __builtin_amdgcn_readfirstlane(tl[2]);
  if (narrow) {  // wave w: row block w
    if (rows <= 128) {
      if (32 * wave < rows)
        gemm_tile<kGated, kNarrow128, 1>(p, s_buf, e, start, rows, ct);
      else
        gemm_tile<kGated, kNarrow128, 0>(p, s_buf, e, start, rows, ct);
    } else {
      if (32 * wave < rows)
        gemm_tile<kGated, kNarrow256, 1>(p, s_buf, e, start, rows, ct);
      else
        gemm_tile<kGated, kNarrow256, 0>(p, s_buf, e, start, rows, ct);
    }
    return;
  }
  // 32-pair row blocks 2 i + (wave >> 2) that hold pairs
  switch (max(0, min(4, (rows - 32 * (wave >> 2) + 63) / 64))) {
    case 0: gemm_tile<kGated, kWide, 0>(p, s_buf, e, start, rows, ct); break;
    case 1: gemm_tile<kGated, kWide, 1>(p, s_buf, e, start, rows, ct); break;
    case 2: gemm_tile<kGated, kWide, 2>(p, s_buf, e, start, rows, ct); break;
    case 3: gemm_tile<kGated, kWide, 3>(p, s_buf, e, start, rows, ct); break;
    default: gemm_tile<kGated, kWide, 4>(p, s_buf, e, start, rows, ct); break;
  }
}

// ---- skinny tiles (few pairs per expert) ------------------------------------------
// Work-group: one tile of up to 16 * PB pairs x 16 output rows (gated: 16
// gate rows j and the 16 up rows N + j; else 32 features in two blocks).
// Wave w takes k-steps w, w + 4, ... (32 k each): 16x16x32 MFMA with the
// weight rows as A (lane: row l % 16, k 8 * (l / 16)..+7 of the step) and the
// pairs as B, both loaded straight into registers, 8 k-steps per batch.
// D[weight row][pair]: lane holds pair l % 16, rows 4 * (l / 16) + i.
constexpr int kSkBatch = 8;

template <bool kGated, int PB>
__global__ void __launch_bounds__(256) fm_skinny_kernel(const GemmParams p) {
  __shared__ f32x4 s_red[4][2][PB][64];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int li = lane & 15;
  const int lg = lane >> 4;

  const int tile = int(blockIdx.x) / p.col_tiles;
  const int ct = int(blockIdx.x) % p.col_tiles;
  if (tile >= p.tiles[0]) return;
  const int32_t* tl = p.tiles + 4 + 4 * tile;
  const int e = tl[0];
  const int start = tl[1];
  const int rows = tl[2];

  // weight rows of this lane's A fragments (block 0 and 1)
  const __bf16* w = p.w + int64_t(e) * p.w_estride;
  const __bf16* wr[2];
  if (kGated) {
    wr[0] = w + int64_t(16 * ct + li) * p.kin;              // gate j
    wr[1] = w + int64_t(p.nout + 16 * ct + li) * p.kin;     // up j
  } else {
    wr[0] = w + int64_t(32 * ct + li) * p.kin;
    wr[1] = w + int64_t(32 * ct + 16 + li) * p.kin;
  }
  // pair rows of this lane's B fragments
  const __bf16* ar[PB];
#pragma unroll
  for (int q = 0; q < PB; ++q) {
    const int r = 16 * q + li;
    const int rr = r < rows ? r : 0;
    const int64_t arow = kGated ? int64_t(p.sorted[start + rr] / p.topk) : int64_t(start + rr);
    ar[q] = p.a + arow * p.a_stride;
  }

  f32x4 acc[2][PB];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int q = 0; q < PB; ++q) acc[b][q] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int nsteps = p.kin / 32;
  for (int s0 = wave; s0 < nsteps; s0 += 4 * kSkBatch) {
    bf16x8 wf[kSkBatch][2];
    bf16x8 af[kSkBatch][PB];
#pragma unroll
    for (int u = 0; u < kSkBatch; ++u) {
      const int s = s0 + 4 * u;
      if (s < nsteps) {
        const int k = 32 * s + 8 * lg;
#pragma unroll
        for (int b = 0; b < 2; ++b) wf[u][b] = *reinterpret_cast<const bf16x8*>(wr[b] + k);
#pragma unroll
        for (int q = 0; q < PB; ++q) af[u][q] = *reinterpret_cast<const bf16x8*>(ar[q] + k);
      }
    }
#pragma unroll
    for (int u = 0; u < kSkBatch; ++u) {
      if (s0 + 4 * u < nsteps) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int q = 0; q < PB; ++q)
            acc[b][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u][b], af[u][q], acc[b][q], 0,
                                                                 0, 0);
      }
    }
  }
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int q = 0; q < PB; ++q) s_red[wave][b][q][lane] = acc[b][q];
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int q = 0; q < PB; ++q) {
      f32x4 s = s_red[0][b][q][lane];
#pragma unroll
      for (int v = 1; v < 4; ++v) s += s_red[v][b][q][lane];  // fixed order: deterministic
      acc[b][q] = s;
    }
  // epilogue: pair r = 16 q + li, output rows 4 * lg + i
#pragma unroll
  for (int q = 0; q < PB; ++q) {
    const int r = 16 * q + li;
    if (r >= rows) continue;
    if (kGated) {
      bf16x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float g = bf16r(silu(bf16r(acc[0][q][i])));
        o[i] = static_cast<__bf16>(bf16r(acc[1][q][i]) * g);
      }
      *reinterpret_cast<bf16x4*>(p.out + int64_t(start + r) * p.out_stride + 16 * ct + 4 * lg) = o;
    } else {
      const int pair = p.sorted[start + r];
      const float wt = p.wts[pair];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        bf16x4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = static_cast<__bf16>(bf16r(acc[b][q][i]) * wt);
        *reinterpret_cast<bf16x4*>(p.out + int64_t(pair) * p.out_stride + 32 * ct + 16 * b +
                                   4 * lg) = o;
      }
    }
  }
}

// ---- streamed-weight tiles (decode) -------------------------------------------------
// Same work-group tile as fm_skinny_kernel (16 * PB pairs x 32 weight rows),
// but every operand reaches the MFMAs through LDS, filled by LDS-DMA in
// stages of 256 k: one instruction moves two rows' 512 contiguous bytes, so
// each weight row streams from HBM in long runs. Stages go through a ring of
// 3 or 4 buffers (all but one in flight); all waits are explicit (no
// compiler-tracked load shares the vmcnt counter with the DMAs). Pair rows
// past the tile's last pair are not loaded. Row r's 16-byte chunk c sits
// at position c ^ (r & 15) of its 512-byte line, so the 16 rows of a 16x16x32
// fragment read hit 16 distinct bank groups. The 4 waves split each stage's
// 8 k-steps (2 each) and add their partial sums through LDS at the end.
constexpr int kStK = 256;                 // k per stage
constexpr int kStLine = kStK * 2;         // 512 bytes per row per stage

template <bool kGated, int PB>
__global__ void __launch_bounds__(256, 1) fm_stream_kernel(const GemmParams p) {
  constexpr int kRowsW = 32;                        // weight rows per column tile
  constexpr int kRowsP = 16 * PB;                   // pair rows
  constexpr int kBuf = (kRowsW + kRowsP) * kStLine; // one stage
  constexpr int kDmaW = kRowsW / 2 / 4;             // weight DMAs per wave per stage (4)
  constexpr int kDmaP = kRowsP / 2 / 4;             // pair DMAs per wave per stage (2 PB)
  // ring depth: two work-groups per CU with three stages of one pair block
  // each, whose starts and partial-sum barriers overlap the other's loads (one
  // with six before: M = 64, E = 64, topk = 6 161 -> 151 us per call, M = 4
  // 69 -> 60); else one with four or three
  constexpr int kStBufs = PB == 1 ? 3 : (144 * 1024) / kBuf;
  static_assert(kStBufs >= 3 && 4 * 2 * PB * 64 * 16 <= kBuf, "ring and reduction fit");
  __shared__ __attribute__((aligned(1024))) uint8_t s_buf[kStBufs * kBuf];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15;
  const int lg = lane >> 4;

  // work-group: column tiles ct0 .. ct0 + p.ct_per_wg - 1 of one pair tile,
  // in one continuous stage pipeline
  const int wgs_per_tile = (p.col_tiles + p.ct_per_wg - 1) / p.ct_per_wg;
  const int tile = int(blockIdx.x) / wgs_per_tile;
  const int ct0 = (int(blockIdx.x) % wgs_per_tile) * p.ct_per_wg;
  if (tile >= p.tiles[0]) return;
  const int nct = min(p.ct_per_wg, p.col_tiles - ct0);
  const int32_t* tl = p.tiles + 4 + 4 * tile;
  const int e = __builtin_amdgcn_readfirstlane(tl[0]);
  const int start = __builtin_amdgcn_readfirstlane(tl[1]);
  const int rows = __builtin_amdgcn_readfirstlane(tl[2]);

  // DMA instruction g of a stage moves rows 2g, 2g + 1 (lane / 32 picks the
  // row, lane % 32 its chunk position); this wave issues weight instructions
  // kDmaW * wave + i and pair instructions kDmaP * wave + i. Offsets are for
  // column tile ct0; a later column tile moves the weight base.
  const int half = lane >> 5;
  const int posn = lane & 31;
  uint32_t w_off[kDmaW];
#pragma unroll
  for (int i = 0; i < kDmaW; ++i) {
    const int r = 2 * (kDmaW * wave + i) + half;  // weight row of the column tile, 0..31
    int wrow;
    if (kGated)  // rows 0..15: gate j = 16 ct + r; rows 16..31: up N + 16 ct + r - 16
      wrow = (r < 16 ? 0 : p.nout - 16) + 16 * ct0 + r;
    else
      wrow = 32 * ct0 + r;
    w_off[i] = uint32_t(int64_t(wrow) * p.kin * 2 + ((posn ^ (r & 15)) * 16));
  }
  uint32_t p_off[kDmaP];
#pragma unroll
  for (int i = 0; i < kDmaP; ++i) {
    const int r = 2 * (kDmaP * wave + i) + half;  // pair row of the tile, 0..16 PB - 1
    const int rr = r < rows ? r : 0;
    const int64_t arow = kGated ? int64_t(p.sorted[start + rr] / p.topk) : int64_t(start + rr);
    p_off[i] = uint32_t(arow * p.a_stride * 2 + ((posn ^ (r & 15)) * 16));
  }
  // pair instructions of this wave that hold a pair (rows 2 (kDmaP wave + i) ..)
  const int npd = max(0, min(kDmaP, (rows + 1) / 2 - kDmaP * wave));
  const int ndma = kDmaW + npd;  // DMAs of this wave per stage
  const uint8_t* wbase = reinterpret_cast<const uint8_t*>(p.w + int64_t(e) * p.w_estride);
  const uint8_t* abase = reinterpret_cast<const uint8_t*>(p.a);
  // bytes between the weight rows of consecutive column tiles
  const int64_t ct_step = int64_t(kGated ? 16 : 32) * p.kin * 2;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(
      uint32_t(reinterpret_cast<uintptr_t>((lds_u8_t*)s_buf)));
  const int nst = p.kin / kStK;   // stages per column tile
  const int total = nct * nst;    // stages of the work-group
  auto issue = [&](int fs) {      // flat stage fs = column tile * nst + stage
    const int c = fs / nst, st = fs - c * nst;
    const uint32_t b = lds0 + uint32_t((fs % kStBufs) * kBuf);
    const uint8_t* wb = wbase + int64_t(c) * ct_step + int64_t(st) * kStLine;
    const uint8_t* ab = abase + int64_t(st) * kStLine;
#pragma unroll
    for (int i = 0; i < kDmaW; ++i)
      lds_dma(wb, w_off[i], b + uint32_t((kDmaW * wave + i) * 2 * kStLine));
#pragma unroll
    for (int i = 0; i < kDmaP; ++i)
      if (i < npd)
        lds_dma(ab, p_off[i], b + uint32_t(kRowsW * kStLine + (kDmaP * wave + i) * 2 * kStLine));
  };

  f32x4 acc[2][PB];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int q = 0; q < PB; ++q) acc[b][q] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int fs = 0; fs < total && fs < kStBufs - 1; ++fs) issue(fs);
  for (int fs = 0; fs < total; ++fs) {
    // this wave's DMAs of stage fs are complete (those of up to two later
    // stages may fly), then every wave's are
    wait_vmcnt(ndma * min(kStBufs - 2, total - 1 - fs));
    lds_barrier();
    if (fs + kStBufs - 1 < total) issue(fs + kStBufs - 1);  // into the buffer of stage fs - 1
    const uint8_t* bw = s_buf + (fs % kStBufs) * kBuf;
    const uint8_t* bp = bw + kRowsW * kStLine;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int c = (2 * wave + u) * 4 + lg;  // 16-byte chunk of this lane's k within the line
      bf16x8 wf[2], pf[PB];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int r = 16 * b + li;
        wf[b] = *reinterpret_cast<const bf16x8*>(bw + r * kStLine + ((c ^ (r & 15)) * 16));
      }
#pragma unroll
      for (int q = 0; q < PB; ++q) {
        const int r = 16 * q + li;
        pf[q] = *reinterpret_cast<const bf16x8*>(bp + r * kStLine + ((c ^ (r & 15)) * 16));
      }
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int q = 0; q < PB; ++q)
          acc[b][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[b], pf[q], acc[b][q], 0, 0, 0);
    }
    if (fs % nst != nst - 1) continue;
    // ---- last stage of a column tile: add the waves' partial sums (fixed
    // order: deterministic); wave b < 2 finishes output block b
    const int ct = ct0 + fs / nst;
    // the partial sums go through this stage's buffer: every wave is done
    // with its operands (the barrier below), and the next DMA into it is
    // issued only after the next stage's barrier
    lds_barrier();
    f32x4(*s_red)[2][PB][64] = reinterpret_cast<f32x4(*)[2][PB][64]>(s_buf + (fs % kStBufs) * kBuf);
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int q = 0; q < PB; ++q) {
        s_red[wave][b][q][lane] = acc[b][q];
        acc[b][q] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    lds_barrier();
    if (wave < 2) {
      const int b = wave;
#pragma unroll
      for (int q = 0; q < PB; ++q) {
        f32x4 sum = s_red[0][b][q][lane];
#pragma unroll
        for (int v = 1; v < 4; ++v) sum += s_red[v][b][q][lane];
        // pair r = 16 q + li, output rows 4 * lg + i of block b
        const int r = 16 * q + li;
        if (r >= rows) continue;
        if (kGated) {
          // block 0 holds the gate rows, block 1 the up rows of the same j:
          // wave 0 reads the up partials as well and writes u
          if (b == 1) continue;
          f32x4 up = s_red[0][1][q][lane];
#pragma unroll
          for (int v = 1; v < 4; ++v) up += s_red[v][1][q][lane];
          bf16x4 o;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float g = bf16r(silu(bf16r(sum[i])));
            o[i] = static_cast<__bf16>(bf16r(up[i]) * g);
          }
          *reinterpret_cast<bf16x4*>(p.out + int64_t(start + r) * p.out_stride + 16 * ct +
                                     4 * lg) = o;
        } else {
          const int pair = p.sorted[start + r];
          const float wt = p.wts[pair];
          bf16x4 o;
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] = static_cast<__bf16>(bf16r(sum[i]) * wt);
          if (p.fsum != nullptr) {
            __bf16* fo = p.fsum + int64_t(pair / p.topk) * p.fsum_stride + 32 * ct + 16 * b + 4 * lg;
            add_bf16x2(fo, o[0], o[1]);
            add_bf16x2(fo + 2, o[2], o[3]);
          } else {
            *reinterpret_cast<bf16x4*>(p.out + int64_t(pair) * p.out_stride + 32 * ct + 16 * b +
                                       4 * lg) = o;
          }
        }
      }
    }
    // the buffer is next written by the DMA of a later stage, issued after
    // a barrier that every wave reaches only after reading it here
  }
}

// ============================================================================
// final sum over each token's experts
// ============================================================================
struct ReduceParams {
  const __bf16* yw;   // [M * topk, K]
  __bf16* out;
  int64_t s_out;
  int64_t M;
  int K, topk;
};

// One thread per 8 consecutive outputs of a token: the running bf16 sum over
// slots 0..topk-1 (ascending experts), rounded after every add like the
// reference's final_out += (reference.py:35).
__global__ void __launch_bounds__(256) fm_reduce_kernel(const ReduceParams p) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  const int per = p.K / 8;
  if (i >= p.M * per) return;
  const int64_t t = i / per;
  const int k = int(i % per) * 8;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  const __bf16* y = p.yw + t * p.topk * int64_t(p.K) + k;
  for (int j = 0; j < p.topk; ++j) {
    const bf16x8 v = *reinterpret_cast<const bf16x8*>(y + int64_t(j) * p.K);
#pragma unroll
    for (int c = 0; c < 8; ++c) acc[c] = bf16r(acc[c] + static_cast<float>(v[c]));
  }
  bf16x8 o;
#pragma unroll
  for (int c = 0; c < 8; ++c) o[c] = static_cast<__bf16>(acc[c]);
  *reinterpret_cast<bf16x8*>(p.out + t * p.s_out + k) = o;
}

int forward(const fm_args* a, hipStream_t stream, void* const* events, uint32_t* launched) {
  const int rc = validate(a);
  if (rc != FM_OK) return rc;
  if (a->M == 0) return FM_OK;
  const Plan pl = make_plan(a);
  if (a->workspace == nullptr || a->workspace_bytes < pl.bytes) return FM_EWORKSPACE;
  // Launches kernel k (FM_KERNEL_*). With the caller's events, through
  // hipExtLaunchKernel: events[2k] and events[2k+1] take the dispatch's own
  // start and end timestamps.
  auto run = [&](int k, const void* fn, dim3 grid, dim3 block, void** kargs) -> bool {
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (events != nullptr) {
      e0 = static_cast<hipEvent_t>(events[2 * k]);
      e1 = static_cast<hipEvent_t>(events[2 * k + 1]);
    }
    const hipError_t err =
        (e0 != nullptr || e1 != nullptr)
            ? hipExtLaunchKernel(fn, grid, block, kargs, 0, stream, e0, e1, 0)
            : hipLaunchKernel(fn, grid, block, kargs, 0, stream);
    if (err != hipSuccess || hipGetLastError() != hipSuccess) return false;
    if (launched != nullptr) *launched |= 1u << k;
    return true;
  };
  auto fn = [](auto kernel) { return reinterpret_cast<const void*>(kernel); };
  uint8_t* ws = static_cast<uint8_t*>(a->workspace);
  int32_t* ids = reinterpret_cast<int32_t*>(ws + pl.ids_off);
  float* wts = reinterpret_cast<float*>(ws + pl.wts_off);
  int32_t* hist = reinterpret_cast<int32_t*>(ws + pl.hist_off);
  int32_t* sorted = reinterpret_cast<int32_t*>(ws + pl.sorted_off);
  int32_t* tiles = reinterpret_cast<int32_t*>(ws + pl.tiles_off);
  __bf16* inter = reinterpret_cast<__bf16*>(ws + pl.inter_off);
  __bf16* yw = reinterpret_cast<__bf16*>(ws + pl.y_off);

  RouteParams rp{};
  rp.score = static_cast<const __bf16*>(a->score);
  rp.s_score = a->s_score;
  rp.ids = ids;
  rp.wts = wts;
  rp.hist = hist;
  rp.tokens_per_wg = pl.tokens_per_wg;
  rp.M = a->M;
  rp.E = int(a->E);
  rp.topk = int(a->topk);
  rp.renormalize = a->renormalize ? 1 : 0;
  // With at most two experts per token and N a multiple of kStK, the down GEMM
  // of streamed tiles, or of up to 24 pairs per expert, adds into the output
  // itself and the routing launch clears it: no final-sum launch.
  const bool streamed = !pl.gemm && a->N % kStK == 0;  // (K % 256 == 0 always holds)
  const bool fsum = a->topk <= 2 && (a->flags & FM_FLAG_ORDERED_SUM) == 0 &&
                    (streamed || (pl.gemm && a->N % kStK == 0 && pl.P <= 24 * a->E));
  if (fsum) {
    rp.zero_out = static_cast<__bf16*>(a->out);
    rp.s_out = a->s_out;
    rp.K = int(a->K);
  }
  PlanParams pp{};
  pp.ids = ids;
  pp.hist = hist;
  pp.wgs = pl.route_wgs;
  pp.pairs_per_wg = pl.tokens_per_wg * int(a->topk);
  pp.sorted = sorted;
  pp.tiles = tiles;
  pp.P = pl.P;
  pp.E = int(a->E);
  pp.tile_rows = pl.tile_rows;
  pp.narrow_rows = pl.narrow_rows;
  const bool e64 = a->E <= 64;
  if (pl.route_wgs == 0) {  // one launch, reported as the plan's
    void* ka[] = {&rp, &pp};
    if (!run(FM_KERNEL_PLAN, e64 ? fn(fm_route_plan_kernel<1>) : fn(fm_route_plan_kernel<4>),
             dim3(1), dim3(1024), ka))
      return FM_EHIP;
  } else {
    const dim3 grid(unsigned(pl.route_wgs));
    void* kr[] = {&rp};
    if (!run(FM_KERNEL_ROUTE, e64 ? fn(fm_route_kernel<1>) : fn(fm_route_kernel<4>), grid,
             dim3(64 * kRouteWaves), kr))
      return FM_EHIP;
    void* kp[] = {&pp};
    if (!run(FM_KERNEL_PLAN, fn(fm_plan_kernel), grid, dim3(1024), kp)) return FM_EHIP;
  }

  GemmParams g1{};
  g1.a = static_cast<const __bf16*>(a->hidden);
  g1.a_stride = a->s_hidden;
  g1.w = static_cast<const __bf16*>(a->w1);
  g1.w_estride = 2 * a->N * a->K;
  g1.sorted = sorted;
  g1.tiles = tiles;
  g1.wts = wts;
  g1.out = inter;
  g1.out_stride = a->N;
  g1.kin = int(a->K);
  g1.nout = int(a->N);
  g1.topk = int(a->topk);
  GemmParams g2 = g1;
  g2.a = inter;
  g2.a_stride = a->N;
  g2.w = static_cast<const __bf16*>(a->w2);
  g2.w_estride = a->K * a->N;
  g2.out = yw;
  g2.out_stride = a->K;
  g2.kin = int(a->N);
  g2.nout = int(a->K);
  if (pl.gemm) {
    g1.col_tiles = int(a->N / (kTileCols / 2));
    g2.col_tiles = int(a->K / kTileCols);
    g1.narrow_cols = int(a->N / (kNarrowCols / 2));
    g2.narrow_cols = int(a->K / kNarrowCols);
  } else {
    g1.col_tiles = int(a->N / 16);
    g2.col_tiles = int(a->K / 32);
  }
  // small tiles stream their weights through LDS when both reductions are
  // whole 256-wide stages, else straight into registers
  if (fsum) {
    g2.fsum = static_cast<__bf16*>(a->out);
    g2.fsum_stride = a->s_out;
  }
  g1.ct_per_wg = g2.ct_per_wg = 1;
  if (streamed) {
    // A streaming work-group runs several column tiles in one pipeline, so its
    // start (tile table -> pair list -> first DMA), about four stages' time,
    // is paid once per several: as many as make the rounds of work-groups (half
    // a round more for their spread) times a work-group's time least, for the
    // expected number of tiles. E = 64, topk = 6, us per call, 1 / 2 / 4 / 8
    // gate-up column tiles: M = 64 162 / 152 / 151 / 155, M = 128 171 / 158 /
    // 168 / -.
    const double used = double(a->E) * (1.0 - pow(1.0 - double(a->topk) / double(a->E), double(a->M)));
    const double mean = double(pl.P) / used;
    const double est = used * (1.0 + 0.5 * erfc((pl.tile_rows + 0.5 - mean) / sqrt(2.0 * mean)));
    const double slots = pl.pb == 1 ? 2.0 * kCus : kCus;
    for (GemmParams* g : {&g1, &g2}) {
      double best = 0.0;
      for (int c = 1; c <= g->col_tiles; c *= 2) {
        const double wgs = est * ((g->col_tiles + c - 1) / c);
        const double t = (ceil(wgs / slots) + 0.5) * (4 + c * (g->kin / kStK));
        if (c == 1 || t < best) {
          best = t;
          g->ct_per_wg = c;
        }
      }
    }
  }
  auto grid_of = [&](const GemmParams& g) {
    if (pl.gemm) {  // gemm_item: an XCD has at most 1 / 8 of the items of each kind, rounded up
      const bool all = pl.tile_rows <= pl.narrow_rows;  // every tile is narrow
      const int64_t narrow = all ? pl.max_tiles : pl.narrow_rows > 0 ? pl.nonempty : 0;
      // (a wide tile holds more than narrow_rows pairs)
      const int64_t wide =
          all ? 0 : std::min<int64_t>(pl.max_tiles, pl.P / (pl.narrow_rows + 1));
      return unsigned(kXcds * ((wide * g.col_tiles + narrow * g.narrow_cols) / kXcds + 2));
    }
    return unsigned(pl.max_tiles * ((g.col_tiles + g.ct_per_wg - 1) / g.ct_per_wg));
  };
  const unsigned grid1 = grid_of(g1);
  const unsigned grid2 = grid_of(g2);
  // the GEMM kernel of this plan, gated (gate-up) or not (down)
  auto gemm = [&](auto gated) -> const void* {
    constexpr bool G = decltype(gated)::value;
    if (pl.gemm) return fn(fm_gemm_kernel<G>);
    if (streamed)
      return pl.pb == 1 ? fn(fm_stream_kernel<G, 1>)
                        : pl.pb == 2 ? fn(fm_stream_kernel<G, 2>) : fn(fm_stream_kernel<G, 4>);
    return pl.pb == 1 ? fn(fm_skinny_kernel<G, 1>) : fn(fm_skinny_kernel<G, 2>);
  };
  const dim3 gemm_block(pl.gemm ? 512 : 256);
  void* k1[] = {&g1};
  if (!run(FM_KERNEL_GATEUP, gemm(std::true_type{}), dim3(grid1), gemm_block, k1)) return FM_EHIP;
  void* k2[] = {&g2};
  if (!run(FM_KERNEL_DOWN, gemm(std::false_type{}), dim3(grid2), gemm_block, k2)) return FM_EHIP;

  if (fsum) return FM_OK;
  ReduceParams rd{};
  rd.yw = yw;
  rd.out = static_cast<__bf16*>(a->out);
  rd.s_out = a->s_out;
  rd.M = a->M;
  rd.K = int(a->K);
  rd.topk = int(a->topk);
  const int64_t threads = a->M * (a->K / 8);
  void* kd[] = {&rd};
  return run(FM_KERNEL_REDUCE, fn(fm_reduce_kernel), dim3(unsigned((threads + 255) / 256)),
             dim3(256), kd) ? FM_OK : FM_EHIP;
}

}  // namespace

extern "C" {

int fm_abi_version(void) { return FM_ABI_VERSION; }

const char* fm_strerror(int code) {
  switch (code) {
    case FM_OK: return "ok";
    case FM_EINVAL: return "invalid argument (null pointer, size, stride, alignment or flags)";
    case FM_EUNSUPPORTED:
      return "unsupported shape (needs K % 256 == 0, N % 128 == 0, E <= 256, topk <= 32 and "
             "sizes within 32-bit offsets)";
    case FM_EWORKSPACE: return "workspace missing or too small";
    case FM_EHIP: return "HIP runtime error";
    default: return "unknown error";
  }
}

int fm_workspace_bytes(const fm_args* a, size_t* out_bytes) {
  if (out_bytes == nullptr) return FM_EINVAL;
  const int rc = validate(a);
  if (rc != FM_OK) return rc;
  *out_bytes = a->M == 0 ? 0 : make_plan(a).bytes;
  return FM_OK;
}

int fm_forward(const fm_args* a, void* hip_stream) {
  return forward(a, static_cast<hipStream_t>(hip_stream), nullptr, nullptr);
}

int fm_forward_events(const fm_args* a, void* hip_stream, void* const* events,
                      uint32_t* launched) {
  if (launched != nullptr) *launched = 0u;
  return forward(a, static_cast<hipStream_t>(hip_stream), events, launched);
}

}  // extern "C"
