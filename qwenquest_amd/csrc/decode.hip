// One Quest decode layer for a batch, as QuestOnlyBackend.forward_decode does it
// (reference src/qwenquest/attention/quest_only.py:132-159): store the new
// token's K/V, select the positions, gather through req_to_token and attend.
//
// Fused path (bf16, D = 128, 4 KV heads - 1, 2, 4 or 8 through qq_quest_layer_step -,
// page 64, at most 64 selected pages, at most 8192 pages per request, top_k <= 4096,
// and a zeroed sync buffer from the caller): two launches.
//   1. page scores of every long request (score_pages_fast_kernel in select.hip,
//      one 256-thread block per (request, 32 candidate pages), all resident at
//      once) and the new token's K/V (set_kv_buffer, memory.py:114-120).
//   2. attention (quest_attend_unit_kernel): the layout's slots come in units of
//      64 (a selected page, the recent window, or 64 slots of the dense layout).
//      One block of W waves per (request, KV head, part); unit_shape sizes the
//      grid to one round of resident blocks (batch 16 x top_k 2048: 8-wave blocks,
//      4 parts per (request, KV head), 256 blocks, one unit per wave).  Every
//      block first selects its request's pages from the scores (select_ranked in
//      qq_quest_dev.h; the blocks of a request compute the same list, so no block
//      waits on another).  Each wave then resolves its unit's 64 rows itself
//      (lane l: slot -> position -> req_to_token; the KV-head-0 blocks store the
//      positions), issues all 32 16-byte loads of the unit's K and V slices at
//      once (32 KiB per wave, 216 VGPRs, two waves per SIMD), computes
//      S^T = K Q^T (v_mfma_f32_16x16x32_bf16), one softmax over the 64 rows folded
//      into its running (M, L), and P V (v_mfma_f32_16x16x16bf16_1k, V transposed
//      in registers).  The W waves combine in LDS; the parts' (m, l, o) partials go
//      out with agent-scope stores, and the block that completes a (request, KV
//      head) count merges them into the output.
// The counters return to zero before the launch ends, so the next call (or a
// graph replay) starts clean.  quest_hisparse's attention over its hot-buffer
// rows runs the same kernel (its rows mode), in the same unit order, so both
// backends compute the same partials in the same order.
//
// Other shapes: four launches on one stream, each consuming the previous one's
// output: score (all CUs) -> select + new-token store (one block per request)
// -> chunk attention (MFMA) -> merge.
#include <algorithm>
#include <mutex>

#include "qq_quest_dev.h"
#include "qq_rules.h"

namespace qq {
namespace {

constexpr int kStepMaxG = 16;
constexpr int kMaxSelFused = 64;
constexpr int kStepMaxTopK = 4096;
constexpr int kDenseWaves = 8;       // dense decode: 8-wave blocks (two waves per SIMD)
constexpr int kPlanReqs = 1024;      // requests whose words the dense plan keeps in LDS at once
// The selection of a 4-wave block of the Quest step's attention (quest_attend_unit_kernel)
// holds up to 32 scores per thread (8192 pages; its LDS, 68 KiB, still lets two
// blocks share a CU).
constexpr int kUnitMinWaves = 4;
using rules::dense_all_whole;
using rules::dense_candidate;
using rules::dense_cost;
using rules::dense_first;
using rules::dense_part_begin;
using rules::dense_parts;
using rules::dense_range;
using rules::dense_units;
using rules::kDenseKV;
using rules::kDenseParts;
using rules::kUnitParts;
using rules::unit_first;
using rules::UnitShape;

struct StepArgs {
  SelectArgs s;            // scoring, selection, positions, new token
  const uint16_t* k;       // this layer's pool [kv_rows, KV, 128]
  const uint16_t* v;
  int64_t kv_rows;
  const int32_t* r2t;
  int64_t r2t_stride, r2t_rows;
  float sl2;               // scale * log2(e)
  uint16_t* out;           // [bs, H * 128] bf16
  float* part_o;           // [bs, KV, parts, G, 128] attention partials (workspace)
  float* part_ml;          // [bs, KV, parts, G, 2] (m in log2 units, l)
  uint32_t* sync;
  int bs, G;
  int kv_shift;            // log2 of the KV heads
  int parts;               // attention blocks per (request, KV head)
  const int64_t* rows_in;  // rows given [bs, rows_stride] (attention over given rows)
  int64_t rows_stride;
  const int32_t* actual;   // [bs] attended slots (attention over given rows)
};

// sync: one counter per (request, KV head), each on its own 128-byte line.
__device__ inline uint32_t* attn_count(const StepArgs& a, int bh) { return a.sync + bh * 32; }

__device__ inline bool needs_selection(const SelectArgs& sa, int64_t s) { return s > sa.top_k && sa.k_sel > 0; }

// One wave's 64 rows of one KV head (lane l: the pool row of token l, the first
// `valid` of them real), folded into its running softmax: M, L per head lo (log2
// units), o[e][i] per (head 4hi + i, channel 8lo + e).
__device__ inline void attend_unit(int r32, int valid, const uint16_t* kb, const uint16_t* vb, int row_shift,
                                   const bf16x8_t (&qb)[4], float sl2, float& M, float& L, float4_t (&o)[8]) {
  const int lane = threadIdx.x & 63;
  const int lo = lane & 15, hi = lane >> 4;
  // every K and V load of the unit in flight at once
  bf16x8_t ka[4][4];
  uint4 vr[4][4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const uint16_t* kp = kb + ((int64_t)__shfl(r32, t * 16 + lo, 64) << row_shift) + hi * 8;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) ka[t][ks] = *reinterpret_cast<const bf16x8_t*>(kp + ks * 32);
  }
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      vr[t][j] = *reinterpret_cast<const uint4*>(vb + ((int64_t)__shfl(r32, t * 16 + hi * 4 + j, 64) << row_shift) + lo * 8);
  __builtin_amdgcn_sched_barrier(0);  // all 32 loads go out before the first use of any
  // S^T[token 16t + 4hi + i][head lo] in acc[t][i]
  float4_t acc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    acc[t] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[t][ks], qb[ks], acc[t], 0, 0, 0);
  }
  float mx = -INFINITY;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float x = (t * 16 + hi * 4 + i) < valid ? acc[t][i] * sl2 : -INFINITY;
      acc[t][i] = x;
      mx = fmaxf(mx, x);
    }
  mx = fmaxf(mx, lane_xor16(mx, lane));
  mx = fmaxf(mx, lane_xor32(mx, lane));
  const float Mn = fmaxf(M, mx);
  const float alpha = M == -INFINITY ? 0.0f : exp2f(M - Mn);  // rescale of the running sums
  const float Mb = fmaxf(Mn, -3.402823466e38f);  // every score so far -inf: weights of 0, not of NaN
  float sum = 0.0f;
  short4_t pa[4];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // v_exp_f32 as it is (exp2f adds a rescale for results below 2^-126, which only
      // the weights of rows 126 binary orders under the maximum reach) and the hardware's
      // round-to-nearest-even bf16 conversion, equal to f2bf for every value that is not NaN
      const uint16_t pbits = __builtin_bit_cast(uint16_t, (__bf16)__builtin_amdgcn_exp2f(acc[t][i] - Mb));
      sum += bf2f(pbits);
      pa[t][i] = (short)pbits;
    }
  sum += lane_xor16(sum, lane);
  sum += lane_xor32(sum, lane);
  L = L * alpha + sum;
  M = Mn;
  // o rows are heads 4hi + i: their scale factors live in lanes 4hi + i
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float ai = __shfl(alpha, hi * 4 + i, 64);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e][i] *= ai;
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    short4_t vbv[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint4 w = vr[t][j];
      const uint32_t wv[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        vbv[2 * x][j] = (short)(wv[x] & 0xFFFFu);
        vbv[2 * x + 1][j] = (short)(wv[x] >> 16);
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(pa[t], vbv[e], o[e], 0, 0, 0);
  }
}

template <int W>
struct CombineSmem {
  float m[W][kStepMaxG];
  float l[W][kStepMaxG];
  float o[W][kStepMaxG][kMfmaDim];
};

// The end of an attention block: its W waves' (M, L, o) (o[e][i]: head 4hi + i,
// channel 8lo + e) combined in LDS, and either the output (`single`: nothing else
// attends for this (request, KV head)) or the (m, l, o) partial part_idx (agent
// scope).  poison: the output becomes NaN.
template <int W>
__device__ inline void combine_block(const StepArgs& a, int bh, bool single, int64_t part_idx, float M, float L,
                                     const float4_t (&o)[8], bool poison, float (*sm_m)[kStepMaxG],
                                     float (*sm_l)[kStepMaxG], float (*sm_o)[kStepMaxG][kMfmaDim]) {
  constexpr int kThreads = 64 * W;
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int lo = lane & 15, hi = lane >> 4;
  const int b = bh >> a.kv_shift, h = bh - (b << a.kv_shift);
  const int G = a.G;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int head = hi * 4 + i;
    if (head < G) {
      float* dst = &sm_o[wave][head][lo * 8];
      *reinterpret_cast<float4*>(dst) = make_float4(o[0][i], o[1][i], o[2][i], o[3][i]);
      *reinterpret_cast<float4*>(dst + 4) = make_float4(o[4][i], o[5][i], o[6][i], o[7][i]);
    }
  }
  if (hi == 0 && lo < G) {
    sm_m[wave][lo] = M;
    sm_l[wave][lo] = poison ? __builtin_nanf("") : L;  // NaN survives every weight of the merge
  }
  __syncthreads();
  uint16_t* outp = a.out + (int64_t)b * a.s.H * kMfmaDim + (int64_t)h * G * kMfmaDim;
  const __amdgpu_buffer_rsrc_t po =
      agent_rsrc(a.part_o + part_idx * G * kMfmaDim, (uint32_t)(G * kMfmaDim * sizeof(float)));
  // each thread one head x 4 channels: the waves' (m, l, o) weighted in wave order
  for (int grp = tid; grp < G * (kMfmaDim / 4); grp += kThreads) {
    const int head = grp >> 5, d4 = (grp & 31) * 4;
    // every LDS read first (one wait instead of a chain of them), then the sums
    float mw[W], lw[W];
    float4 ov[W];
#pragma unroll
    for (int w = 0; w < W; ++w) {
      mw[w] = sm_m[w][head];
      lw[w] = sm_l[w][head];
      ov[w] = *reinterpret_cast<const float4*>(&sm_o[w][head][d4]);
    }
    float Mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < W; ++w) Mx = fmaxf(Mx, mw[w]);
    float Ls = 0.0f;
    float4 Os = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float wgt = mw[w] == -INFINITY ? 0.0f : exp2f(mw[w] - Mx);
      Ls += wgt * lw[w];
      Os.x += wgt * ov[w].x;
      Os.y += wgt * ov[w].y;
      Os.z += wgt * ov[w].z;
      Os.w += wgt * ov[w].w;
    }
    if (single) {
      const bool any = !(Ls <= 0.0f);  // NaN (a poisoned part) stays NaN
      const uint32_t lo2 = (uint32_t)f2bf(any ? Os.x / Ls : 0.0f) | ((uint32_t)f2bf(any ? Os.y / Ls : 0.0f) << 16);
      const uint32_t hi2 = (uint32_t)f2bf(any ? Os.z / Ls : 0.0f) | ((uint32_t)f2bf(any ? Os.w / Ls : 0.0f) << 16);
      *reinterpret_cast<uint2*>(outp + head * kMfmaDim + d4) = make_uint2(lo2, hi2);
    } else {
      st_agent_x4(po, (uint32_t)((head * kMfmaDim + d4) * sizeof(float)), Os);
      if (d4 == 0) {
        st_agent(a.part_ml + (part_idx * G + head) * 2, Mx);
        st_agent(a.part_ml + (part_idx * G + head) * 2 + 1, Ls);
      }
    }
  }
}

// Counts this block's partial of a (request, KV head); true, in every thread, for the
// block that completes `parts` of them (the counter is then 0 again).
__device__ inline bool last_part(const StepArgs& a, int bh, int parts, uint32_t* s_last) {
  wait_memory();
  __syncthreads();
  if (threadIdx.x == 0) *s_last = add_agent(attn_count(a, bh), 1u) == (uint32_t)(parts - 1);
  __syncthreads();
  if (!*s_last) return false;
  if (threadIdx.x == 0) st_agent(attn_count(a, bh), 0u);
  return true;
}

// combine_block, then the merge of a.parts <= MG parts by the block that completes
// them (in part order: the maximum of the parts' m first, then the weighted sums),
// each thread one head x 4 channels, all loads in flight at once.
template <int W, int MG>
__device__ inline void finish_block(const StepArgs& a, int bh, int part, float M, float L, const float4_t (&o)[8],
                                    bool poison, float (*sm_m)[kStepMaxG], float (*sm_l)[kStepMaxG],
                                    float (*sm_o)[kStepMaxG][kMfmaDim], uint32_t* s_last) {
  constexpr int kThreads = 64 * W;
  const int tid = threadIdx.x;
  const int parts = a.parts, G = a.G;
  combine_block<W>(a, bh, parts == 1, (int64_t)bh * parts + part, M, L, o, poison, sm_m, sm_l, sm_o);
  if (parts == 1 || !last_part(a, bh, parts, s_last)) return;
  const int b = bh >> a.kv_shift, h = bh - (b << a.kv_shift);
  uint16_t* outp = a.out + (int64_t)b * a.s.H * kMfmaDim + (int64_t)h * G * kMfmaDim;
  const int64_t part0 = (int64_t)bh * parts;
  const __amdgpu_buffer_rsrc_t ro =
      agent_rsrc(a.part_o + part0 * G * kMfmaDim, (uint32_t)(parts * G * kMfmaDim * sizeof(float)));
  const uint64_t* ml64 = reinterpret_cast<const uint64_t*>(a.part_ml) + part0 * G;
  for (int grp = tid; grp < G * (kMfmaDim / 4); grp += kThreads) {
    const int head = grp >> 5, d4 = (grp & 31) * 4;
    float Mx = -INFINITY;
    float Ls = 0.0f;
    float4 Os = make_float4(0.f, 0.f, 0.f, 0.f);
    float4 ov[MG];
    uint64_t mlv[MG];
#pragma unroll
    for (int j = 0; j < MG; ++j) {
      if (j < parts) {
        ov[j] = ld_agent_x4(ro, (uint32_t)(((j * G + head) * kMfmaDim + d4) * sizeof(float)));
        mlv[j] = ld_agent(ml64 + j * G + head);
      }
    }
#pragma unroll
    for (int j = 0; j < MG; ++j)
      if (j < parts) Mx = fmaxf(Mx, __uint_as_float((uint32_t)mlv[j]));
#pragma unroll
    for (int j = 0; j < MG; ++j) {
      if (j < parts) {
        const float mj = __uint_as_float((uint32_t)mlv[j]);
        const float wgt = mj == -INFINITY ? 0.0f : exp2f(mj - Mx);
        Ls += wgt * __uint_as_float((uint32_t)(mlv[j] >> 32));
        Os.x += wgt * ov[j].x;
        Os.y += wgt * ov[j].y;
        Os.z += wgt * ov[j].z;
        Os.w += wgt * ov[j].w;
      }
    }
    const bool any = !(Ls <= 0.0f);  // NaN (a poisoned part) stays NaN
    const uint32_t lo2 = (uint32_t)f2bf(any ? Os.x / Ls : 0.0f) | ((uint32_t)f2bf(any ? Os.y / Ls : 0.0f) << 16);
    const uint32_t hi2 = (uint32_t)f2bf(any ? Os.z / Ls : 0.0f) | ((uint32_t)f2bf(any ? Os.w / Ls : 0.0f) << 16);
    *reinterpret_cast<uint2*>(outp + head * kMfmaDim + d4) = make_uint2(lo2, hi2);
  }
}

// ------------------------------------------------------------- dense decode
// Every request attends its whole context (attention/dense.py:26-42).  A (request, KV
// head) pair's 64-row units are split into equal parts, one to a block, of a length that
// keeps the CUs alike busy: one long request, many ragged ones, or one long one among
// many (dense_range and dense_cost in qq_rules.h).  The lengths are on the device, so the
// division is made there, by one more block of the launch that stores the new tokens (it hides
// behind that launch, and the attention's blocks each read one entry instead of the
// batch's lengths).
struct DenseItem {
  int bh;           // pair, or -1: no work for this block
  int u0, u1;       // its units
  int part, parts;  // of the pair; its parts are consecutive blocks
  int rows;         // context
  int req;          // table row, or -1: outside the table
  int queued;       // 0, or the entries of the plan, where there are more of them than blocks
};

// Where the plan has more entries than the grid has blocks, every block goes on with the
// next one that no block has.
struct DenseQueue {
  uint32_t next;
  uint32_t pad[7];
};

struct DenseSmem {
  union {
    CombineSmem<kDenseWaves> comb;
    struct {
      float w[kStepMaxG][kDenseParts];  // weight of each part
      float l[kStepMaxG];
      float4 red[64 * kDenseWaves];
    } merge;
  };
  uint32_t last;
  uint32_t next[2];  // the part after this one, in turn
};

__device__ inline int dense_rows(const StepArgs& a, int b) {
  return (int)min(max(a.s.seq[b], (int64_t)0), (int64_t)a.s.top_k);
}
// dense_parts(units, len) with 1 / len at hand: the quotient by the inverse, then put right.
__device__ inline int dense_parts_inv(int units, int len, float inv) {
  const int x = units + len - 1;
  int parts = (int)((float)x * inv);
  const int rest = x - parts * len;
  parts += rest >= len ? 1 : rest < 0 ? -1 : 0;
  return units <= rules::kDenseWhole ? 1 : min(parts, kDenseParts);
}

// The division of a batch that one round of blocks takes (dense_one_round: at most 24
// requests): a lane per request, every wave for itself, without LDS and barriers.  The
// shortest of the lengths that fit is the cheapest.
__device__ inline void plan_one_round(const StepArgs& a, DenseItem* plan, int fit, int round, int grid) {
  const int bs = a.bs, tid = threadIdx.x, lane = tid & 63;
  int rows = 0, units = 0, req = -1;
  if (lane < bs) {
    const int64_t r = a.s.rpi[lane];
    rows = dense_rows(a, lane);
    units = dense_units(rows);
    req = r >= 0 && r < a.r2t_rows ? (int)r : -1;
  }
  int total = units, longest = max(units, 1);
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    total += __shfl_xor(total, d, 64);
    longest = max(longest, __shfl_xor(longest, d, 64));
  }
  int len = 1 << 30;  // nothing is split
  if (fit > bs) {
    const int cand = dense_candidate(dense_range(min(total, rules::kDenseMaxTotal), longest, bs, fit, round), lane);
    const float inv = 1.0f / (float)cand;
    int count = 0;
    for (int b = 0; b < bs; ++b) count += dense_parts_inv(__builtin_amdgcn_readlane(units, b), cand, inv);
    const uint64_t ok = __ballot(count <= fit);
    if (ok) len = __builtin_amdgcn_readlane(cand, __builtin_ctzll(ok));
  }
  const int parts = lane < bs ? dense_parts(units, len) : 0;
  int first = parts;  // parts (per KV head) up to this request's, then before it
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int y = __shfl_up(first, d, 64);
    if (lane >= d) first += y;
  }
  const int all = __builtin_amdgcn_readlane(first, 63) * kDenseKV;
  first -= parts;
  for (int e0 = 0; e0 < grid; e0 += 256) {
    const int e = e0 + tid;
    // blocks of a request: its parts of KV head 0, then of head 1, ...
    int b = -1;
    for (int i = 0; i < bs; ++i) b += __builtin_amdgcn_readlane(first, i) * kDenseKV <= e ? 1 : 0;
    const int p = __shfl(parts, b, 64), u = __shfl(units, b, 64);
    const int at = e - __shfl(first, b, 64) * kDenseKV;
    const int h = at / p, part = at - h * p;
    const DenseItem it = {b * kDenseKV + h, dense_part_begin(u, part, p), dense_part_begin(u, part + 1, p), part,
                          p, __shfl(rows, b, 64), __shfl(req, b, 64), 0};
    if (e < grid) plan[e] = e < all ? it : DenseItem{-1, 0, 0, 0, 1, 0, -1, 0};
  }
}

// Block 0: the division of the batch, `fit` parts per KV head at most; blocks 1 .. bs:
// the new tokens (memory.py:114-120), and the parts' counters.  64 part lengths are tried, one per lane, the waves
// sharing the requests (dense_range, dense_cost), and every entry finds its request.  The
// requests' words are kept in LDS, kPlanReqs of them at a time.
__global__ __launch_bounds__(256) void dense_store_plan_kernel(StepArgs a, DenseItem* plan, DenseQueue* queue, int fit,
                                                               int round, int grid) {
  const int bs = a.bs, tid = threadIdx.x;
  if (blockIdx.x > 0) {
    const int b = blockIdx.x - 1;
    if (tid < kDenseKV) *attn_count(a, b * kDenseKV + tid) = 0u;
    store_new_token(a.s, b);
    return;
  }
  if (gridDim.x == 1)  // no blocks of new tokens
    for (int i = tid; i < bs * kDenseKV; i += 256) *attn_count(a, i) = 0u;
  if (rules::dense_one_round(bs, round)) {
    plan_one_round(a, plan, fit, round, grid);
    return;
  }
  if (tid == 0) queue->next = (uint32_t)grid;
  __shared__ int s_first[kPlanReqs + 1];  // parts (per KV head) before each request
  __shared__ int s_rows[kPlanReqs], s_req[kPlanReqs];
  __shared__ int64_t s_sum[4];
  __shared__ int s_tmp[4], s_count[4][64];
  const int wave = tid >> 6, lane = tid & 63;
  int64_t total = 0;
  int longest = 1;
  auto load_request = [&](int b) -> int {
    const int64_t req = a.s.rpi[b];
    const int rows = dense_rows(a, b);
    s_rows[b & (kPlanReqs - 1)] = rows;
    s_req[b & (kPlanReqs - 1)] = req >= 0 && req < a.r2t_rows ? (int)req : -1;
    return rows;
  };
  for (int b = tid; b < bs; b += 256) {
    const int u = dense_units(load_request(b));
    total += u;
    longest = max(longest, u);
  }
  // the words of requests c0 ... of a batch that LDS does not keep whole
  auto load_requests = [&](int c0) {
    if (bs <= kPlanReqs) return;
    __syncthreads();
    for (int b = c0 + tid; b < min(c0 + kPlanReqs, bs); b += 256) load_request(b);
    __syncthreads();
  };
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    total += __shfl_xor((long long)total, d, 64);
    longest = max(longest, __shfl_xor(longest, d, 64));
  }
  if (lane == 0) {
    s_sum[wave] = total;
    s_tmp[wave] = longest;
  }
  __syncthreads();
  const int total32 = (int)min(s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3], (int64_t)rules::kDenseMaxTotal);
  longest = max(max(s_tmp[0], s_tmp[1]), max(s_tmp[2], s_tmp[3]));
  if (fit <= bs || dense_all_whole(total32, longest, bs, round)) {
    for (int c0 = 0; c0 < bs; c0 += kPlanReqs) {
      load_requests(c0);
      for (int e = c0 * kDenseKV + tid; e < min(c0 + kPlanReqs, bs) * kDenseKV; e += 256) {
        const int r = e / kDenseKV - c0;
        plan[e] = {e, 0, dense_units(s_rows[r]), 0, 1, s_rows[r], s_req[r], 0};
      }
    }
    for (int e = bs * kDenseKV + tid; e < grid; e += 256) plan[e] = {-1, 0, 0, 0, 1, 0, -1, 0};
    return;
  }
  const int cand = dense_candidate(dense_range(total32, longest, bs, fit, round), lane);
  const float inv = 1.0f / (float)cand;
  int count = 0;
  for (int c0 = 0; c0 < bs; c0 += kPlanReqs) {
    load_requests(c0);
#pragma unroll 4
    for (int b = wave; b < min(kPlanReqs, bs - c0); b += 4)
      count += dense_parts_inv(dense_units(s_rows[b]), cand, inv);
  }
  s_count[wave][lane] = count;
  __syncthreads();
  count = s_count[0][lane] + s_count[1][lane] + s_count[2][lane] + s_count[3][lane];
  const float cost = dense_cost(total32, count, cand, fit, round);
  float least_cost = cost;
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) least_cost = fminf(least_cost, __shfl_xor(least_cost, d, 64));
  const int best = __builtin_ctzll(__ballot(cost == least_cost));
  const bool fits = least_cost < rules::kDenseNoFit;
  const int len = fits ? __shfl(cand, best, 64) : 1 << 30;
  const int parts_all = fits ? __shfl(count, best, 64) : bs;
  const int classes = parts_all > round ? 2 : 1;
  const int queued = parts_all * kDenseKV > grid ? parts_all * kDenseKV : 0;
  int base = 0;  // parts so far
  for (int cls = 0; cls < classes; ++cls)
    for (int c0 = 0; c0 < bs; c0 += kPlanReqs) {
      load_requests(c0);
      const int n = min(kPlanReqs, bs - c0), base0 = base;
      // parts before each request: a prefix sum, 256 requests at a time
      for (int b0 = 0; b0 < n; b0 += 256) {
        const int b = b0 + tid;
        int mine = 0;
        if (b < n) {
          const int u = dense_units(s_rows[b]);
          mine = dense_parts(u, len);
          if (classes > 1 && dense_first(u, mine, len) != (cls == 0)) mine = 0;
        }
        int x = mine;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
          const int y = __shfl_up(x, d, 64);
          if (lane >= d) x += y;
        }
        __syncthreads();
        if (lane == 63) s_tmp[wave] = x;
        __syncthreads();
        int before = base;
        for (int w = 0; w < wave; ++w) before += s_tmp[w];
        if (b < n) s_first[b] = before + x - mine;
        base += s_tmp[0] + s_tmp[1] + s_tmp[2] + s_tmp[3];
      }
      if (tid == 0) s_first[n] = base;
      __syncthreads();
      // blocks of a request: its parts of KV head 0, then of head 1, ...
      for (int e = base0 * kDenseKV + tid; e < base * kDenseKV; e += 256) {
        int b = 0, b_end = n;  // the last request whose first block is <= e
        while (b_end - b > 1) {
          const int mid = (b + b_end) >> 1;
          if (s_first[mid] * kDenseKV <= e) b = mid;
          else b_end = mid;
        }
        const int parts = s_first[b + 1] - s_first[b];
        const int at = e - s_first[b] * kDenseKV;
        const int h = at / parts, part = at - h * parts;
        const int units = dense_units(s_rows[b]);
        plan[e] = {(c0 + b) * kDenseKV + h, dense_part_begin(units, part, parts), dense_part_begin(units, part + 1, parts),
                   part, parts, s_rows[b], s_req[b], queued};
      }
      __syncthreads();  // s_first is free
    }
  for (int e = base * kDenseKV + tid; e < grid; e += 256) plan[e] = {-1, 0, 0, 0, 1, 0, -1, 0};
}

// The parts of a pair added up by a whole block: the weights e^(m - max) of every
// part in LDS, a wave per head and a lane per part, then each thread one head x 4
// channels of every ng-th part, 32 loads in flight.
__device__ inline void merge_dense(const StepArgs& a, int bh, int64_t part0, int parts, DenseSmem& sm) {
  constexpr int kThreads = 64 * kDenseWaves;
  constexpr int kPer = (kDenseParts + 63) / 64;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int G = a.G;
  const uint64_t* ml64 = reinterpret_cast<const uint64_t*>(a.part_ml) + part0 * G;
  const __amdgpu_buffer_rsrc_t ro =
      agent_rsrc(a.part_o + part0 * G * kMfmaDim, (uint32_t)((int64_t)parts * G * kMfmaDim * sizeof(float)));
  const int items = G * (kMfmaDim / 4);  // (head, 4 channels): up to 512
  const int ng = max(kThreads / items, 1);
  const int grp = items <= kThreads ? tid / items : 0;
  // the first kBatch parts' sums go out before the weights are known; past the last
  // part they are zeros, from beyond the resource
  constexpr int kBatch = 32;
  float4 ov[kBatch];
  auto load_parts = [&](int at, int p0) {
#pragma unroll
    for (int u = 0; u < kBatch; ++u)
      ov[u] = ld_agent_x4(ro, (uint32_t)(((p0 + u * ng) * G * kMfmaDim + at * 4) * (int)sizeof(float)));
  };
  load_parts(tid - grp * items, grp);
  for (int head = wave; head < G; head += kDenseWaves) {
    uint64_t ml[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int p = lane + 64 * i;
      ml[i] = p < parts ? ld_agent(ml64 + (int64_t)p * G + head) : (uint64_t)0xFF800000u;  // (-inf, 0)
    }
    float Mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < kPer; ++i) Mx = fmaxf(Mx, __uint_as_float((uint32_t)ml[i]));
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) Mx = fmaxf(Mx, __shfl_xor(Mx, d, 64));
    float Ls = 0.0f;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const float m = __uint_as_float((uint32_t)ml[i]);
      const float w = m == -INFINITY ? 0.0f : exp2f(m - Mx);
      if (lane + 64 * i < parts) sm.merge.w[head][lane + 64 * i] = w;
      Ls += w * __uint_as_float((uint32_t)(ml[i] >> 32));
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) Ls += __shfl_xor(Ls, d, 64);
    if (lane == 0) sm.merge.l[head] = Ls;
  }
  __syncthreads();
  if (ng == 1 && grp > 0) return;  // threads past the items
  const int b = bh / kDenseKV, h = bh - b * kDenseKV;
  uint16_t* outp = a.out + (int64_t)b * a.s.H * kMfmaDim + (int64_t)h * G * kMfmaDim;
  const int at0 = tid - grp * items;
  for (int at = at0; at < items; at += kThreads) {  // once, for every thread, where ng > 1
    const int head = at >> 5, d4 = (at & 31) * 4;
    float4 Os = make_float4(0.f, 0.f, 0.f, 0.f);
    if (grp < ng) {
      for (int p0 = grp; p0 < parts; p0 += kBatch * ng) {
        if (at != at0 || p0 != grp) load_parts(at, p0);
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          const float w = sm.merge.w[head][min(p0 + u * ng, parts - 1)];
          Os.x += w * ov[u].x;
          Os.y += w * ov[u].y;
          Os.z += w * ov[u].z;
          Os.w += w * ov[u].w;
        }
      }
    }
    if (ng > 1) {  // block-uniform
      sm.merge.red[tid] = Os;
      __syncthreads();
      if (grp != 0) return;
      for (int g = 1; g < ng; ++g) {
        const float4 x = sm.merge.red[tid + g * items];
        Os.x += x.x;
        Os.y += x.y;
        Os.z += x.z;
        Os.w += x.w;
      }
    }
    const float Ls = sm.merge.l[head];
    const bool any = !(Ls <= 0.0f);
    const uint32_t lo2 = (uint32_t)f2bf(any ? Os.x / Ls : 0.0f) | ((uint32_t)f2bf(any ? Os.y / Ls : 0.0f) << 16);
    const uint32_t hi2 = (uint32_t)f2bf(any ? Os.z / Ls : 0.0f) | ((uint32_t)f2bf(any ? Os.w / Ls : 0.0f) << 16);
    *reinterpret_cast<uint2*>(outp + head * kMfmaDim + d4) = make_uint2(lo2, hi2);
  }
}

// One part of a pair: wave w takes units u0 + w, u0 + w + 8, ..., each with all of its
// 32 KiB of K and V in flight at once; one block per CU.
//
// Bound: HBM.  Attention and store, per layer at 32 / 4 heads, against blocks of 4096
// rows each, as many per pair as the table's width holds: one request of 8000 rows
// 49 -> 17 us, of 100000 83 -> 52; 16 ragged requests of 2000 .. 65000 in a
// 131072-wide table 480 -> 106 (4.6 TB/s); 16 of 131000 785 -> 745 (5.8 TB/s); 64 of
// 3000 84 -> 77.  4-wave blocks, two per CU: 64 of 3000 87 us, one of 100000 63 (twice
// the parts to merge), one of 8000 16.9.
// QUEUE: batches whose plan may have more parts than the grid has blocks.  Against one
// round of parts as the limit (a pair per block from 64 requests on): 100000 rows and 63
// x 2000 1175 -> 103 us, 2 x 100000 and 126 x 300 1171 -> 107, 8 x 30000 and 48 x 500
// 207 -> 137, 70 x 10000 342 -> 311; 128 x 3000 143 -> 145, 64 x 3000 76.5 -> 77.  A
// block per entry instead of the queue, 512 more of them, costs those 5 us.
// A kernel's first argument, read anew from its argument block: kept in scalar registers
// over a loop, the arguments would be spilt there.
__device__ inline StepArgs reread_args(const StepArgs&) {
  typedef const __attribute__((address_space(4))) char* arg_ptr_t;
  arg_ptr_t p = (arg_ptr_t)__builtin_amdgcn_kernarg_segment_ptr();
  __asm__ volatile("" : "+s"(p));
  StepArgs a;
  __builtin_memcpy(&a, (const void*)p, sizeof(a));
  return a;
}

template <bool QUEUE>
__global__ __launch_bounds__(64 * kDenseWaves, 2) void dense_attend_kernel(StepArgs args, const DenseItem* plan,
                                                                        DenseQueue* queue) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  DenseSmem& sm = *reinterpret_cast<DenseSmem*>(smem_raw);
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lo = lane & 15, hi = lane >> 4;
  for (int e = blockIdx.x, turn = 0;; turn ^= 1) {
    const StepArgs a = QUEUE ? reread_args(args) : args;
    const SelectArgs& sa = a.s;
    const int G = a.G;
    const DenseItem it = plan[e];
    if (it.bh < 0) return;
    uint32_t next = 0;
    if (QUEUE && it.queued && tid == 0)
      next = __hip_atomic_fetch_add(&queue->next, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int n = it.rows;
    const int b = it.bh / kDenseKV, h = it.bh - b * kDenseKV;
    const int32_t* rt = a.r2t + (int64_t)max(it.req, 0) * a.r2t_stride;
    // units with rows: a request without any has one unit and no rows
    const int u_end = min(it.u1, (n + 63) / 64);
    // lane l: the pool row of token l of a unit, as the table has it (row 0 past the
    // context); looked at a unit later, so that it is loaded under the unit before
    auto table_row = [&](int j) -> int {
      const int slot = j * 64 + lane;
      return (j < u_end && slot < n && it.req >= 0) ? rt[slot] : 0;
    };
    int row = table_row(it.u0 + wave);
    bf16x8_t qb[4];
    {
      const uint16_t* qp = static_cast<const uint16_t*>(sa.q) + (int64_t)b * sa.q_bstride +
                           (int64_t)(h * G + lo) * kMfmaDim + hi * 8;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        if (lo < G) {
          qb[ks] = *reinterpret_cast<const bf16x8_t*>(qp + ks * 32);
        } else {
          qb[ks] = __builtin_bit_cast(bf16x8_t, u32x4_t{0u, 0u, 0u, 0u});
        }
      }
    }
    const uint16_t* kb = a.k + h * kMfmaDim;
    const uint16_t* vb = a.v + h * kMfmaDim;
    float M = -INFINITY, L = 0.0f;
    float4_t o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = float4_t{0.f, 0.f, 0.f, 0.f};
    // the row and the query are in; the compiler then knows that a unit's row, loaded
    // under the unit before, needs no wait, which would be one for the next row too
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    if (QUEUE && tid == 0) sm.next[turn] = next;  // read after this part's barriers
    for (int j = it.u0 + wave; j < u_end; j += kDenseWaves) {
      const int row_next = table_row(j + kDenseWaves);
      attend_unit(row >= 0 && row < a.kv_rows ? row : 0, min(n - j * 64, 64), kb, vb, 9, qb, a.sl2, M, L, o);
      row = row_next;
    }
    combine_block<kDenseWaves>(a, it.bh, it.parts == 1, e, M, L, o, false, sm.comb.m, sm.comb.l, sm.comb.o);
    if (it.parts > 1 && last_part(a, it.bh, it.parts, &sm.last))
      merge_dense(a, it.bh, (int64_t)e - it.part, it.parts, sm);
    if (!QUEUE || !it.queued) return;
    __syncthreads();  // this part's LDS is free
    e = __builtin_amdgcn_readfirstlane((int)sm.next[turn]);
    if (e >= it.queued) return;
  }
}

// ------------------------------------------------------- per-page-unit attention
// The Quest step's attention (after the score launch; and over given rows for
// quest_hisparse, so that both compute the same partials in the same order):
// one block of W waves per (request, KV head, part), blockIdx = (request, KV head) *
// parts + part.  The layout's slots come in units of 64 (a selected page, or the
// recent window, or 64 slots of the dense layout); wave w of part p takes units
// w*parts + p, w*parts + p + W*parts, ...  (unit_shape).  Per unit a
// wave resolves its 64 rows itself (lane l: slot 64u + l -> position ->
// req_to_token), shuffles them into the MFMA lane layouts and issues all 32
// loads of the unit's K and V slices (32 KiB per wave) at once, then
// S^T = K Q^T (v_mfma_f32_16x16x32_bf16, K rows as the A operand, 16 B per
// lane), one softmax over the 64 rows folded into the wave's running (M, L),
// P (bf16) straight from the S^T accumulator into v_mfma_f32_16x16x16bf16_1k
// with V transposed in registers.  The block first selects its request's pages
// (select_pages_wave: every wave ends with the page list in its lanes).
template <int KPT, int W>
struct UnitSmem {
  union {
    RankSelectSmem<(KPT > 0 ? KPT : 1), 64 * W> sel;
    CombineSmem<W> comb;
  };
};

template <bool ROWS, int KPT, int W>
__global__ __launch_bounds__(64 * W, 8 / W) void quest_attend_unit_kernel(StepArgs a) {
  constexpr int NT = 64 * W;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ uint32_t s_last;
  UnitSmem<KPT, W>& sm = *reinterpret_cast<UnitSmem<KPT, W>*>(smem_raw);
  const SelectArgs& sa = a.s;
  int parts = a.parts;
  // the score buffer, its width and the limit array are read with the block's
  // coordinates (an empty asm ties them to `parts`), so that the score and limit
  // loads below go out with the request's words instead of one round trip after them
  if constexpr (!ROWS && KPT > 0) __asm__("" : "+s"(parts) : "s"(sa.scores), "s"(sa.MP), "s"(sa.limit));
  const int bh = blockIdx.x / parts, part = blockIdx.x - bh * parts;
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int lo = lane & 15, hi = lane >> 4;
  const int b = bh >> a.kv_shift, h = bh - (b << a.kv_shift);
  const int64_t s = ROWS ? 0 : sa.seq[b];
  const int64_t req = ROWS ? 0 : sa.rpi[b];
  const int top_k = sa.top_k, k = sa.k_sel;
  constexpr int P = 64;
  const int G = a.G;
  // Q^T as the B operand: query head lo (zero past G), channels 8hi + 32ks
  bf16x8_t qb[4];
  {
    const uint16_t* qp = static_cast<const uint16_t*>(sa.q) + (int64_t)b * sa.q_bstride +
                         (int64_t)(h * G + lo) * kMfmaDim + hi * 8;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (lo < G) {
        qb[ks] = *reinterpret_cast<const bf16x8_t*>(qp + ks * 32);
      } else {
        qb[ks] = __builtin_bit_cast(bf16x8_t, u32x4_t{0u, 0u, 0u, 0u});
      }
    }
  }
  // the scores go out with the request's words (their addresses do not wait for
  // them): entries past the table re-read its last one and are masked below.  The
  // scheduling barrier keeps every use of the request's words after these loads, so
  // that the wait for the words does not come before them, and both branches below
  // read the scores, so that the loads are not moved into the selecting one
  float sv[KPT > 0 ? KPT : 1];
  int lim_raw = 0;
  if constexpr (KPT > 0) {
    const float* sc = sa.scores + (int64_t)b * sa.MP;
#pragma unroll
    for (int i = 0; i < KPT; ++i) sv[i] = sc[min(tid + NT * i, sa.MP - 1)];
    lim_raw = sa.limit[b];
    __builtin_amdgcn_sched_barrier(0);
  }
  const bool long_b = !ROWS && needs_selection(sa, s);
  // actual_lens (quest.py:345)
  const int n = ROWS ? min(max(a.actual[b], 0), top_k) : (int)min(max(s, (int64_t)0), (int64_t)top_k);
  const bool r2t_ok = !ROWS && req >= 0 && req < a.r2t_rows;
  int my_rank = -1, my_page = -1, my_row0 = -1;  // lane s: a survivor's rank, page, first pool row
  if constexpr (KPT > 0) {
    if (long_b) {  // block-uniform
      const int lim = (req >= 0 && req < sa.R) ? min(lim_raw, sa.MP) : 0;
      select_ranked<KPT, NT>(sv, lim, max(lim, k), k, sm.sel, nullptr, sa.MP, my_rank, my_page, my_row0);
    } else {
#pragma unroll
      for (int i = 0; i < KPT; ++i) __asm__ volatile("" ::"v"(sv[i]));
    }
  }
  const int units = top_k / P;
  const int stride_units = parts * W;
  const int64_t recent0 = max(s - P, (int64_t)0);
  int32_t* pos_out = !ROWS && h == 0 && sa.positions ? sa.positions + (int64_t)b * top_k : nullptr;
  const uint16_t* kb = a.k + h * kMfmaDim;
  const uint16_t* vb = a.v + h * kMfmaDim;
  const int row_shift = a.kv_shift + 7;  // KV * 128 channels per pool row
  float M = -INFINITY, L = 0.0f;
  float4_t o[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = float4_t{0.f, 0.f, 0.f, 0.f};
  bool bad = false;
  for (int u = unit_first(wave, part, parts); u < units; u += stride_units) {  // wave-uniform
    const int slot = u * P + lane;
    const int valid = min(n - u * P, P);  // real slots of this unit
    int64_t row = 0;
    if constexpr (ROWS) {
      if (lane < valid) {
        row = a.rows_in[(int64_t)b * a.rows_stride + slot];
        bad |= row < 0;
      }
    } else {
      int64_t p;
      if (!long_b)
        p = s <= top_k ? min((int64_t)slot, max(s - 1, (int64_t)0)) : min(recent0 + slot, s - 1);
      else if (u < k)
        p = (int64_t)__builtin_amdgcn_readlane(my_page, __builtin_ctzll(__ballot(my_rank == u))) * P + lane;
      else
        p = min(recent0 + (slot - k * P), s - 1);
      if (lane < valid && r2t_ok && p >= 0 && p < a.r2t_stride) row = a.r2t[req * a.r2t_stride + p];
      if (pos_out) pos_out[slot] = (int32_t)p;  // after the row load: waiting for the row does not wait for it
    }
    if (valid <= 0) continue;
    const int r32 = (row >= 0 && row < a.kv_rows) ? (int)row : 0;
    attend_unit(r32, valid, kb, vb, row_shift, qb, a.sl2, M, L, o);
  }
  bool poison = false;
  if constexpr (ROWS) poison = __syncthreads_or(bad ? 1 : 0) != 0;  // a failed swap-in: NaN output
  else lds_barrier();  // the selection's LDS is free before the combine reuses it
  finish_block<W, kUnitParts>(a, bh, part, M, L, o, poison, sm.comb.m, sm.comb.l, sm.comb.o, &s_last);
}

}  // namespace
}  // namespace qq

using namespace qq;

extern "C" int64_t qq_quest_layer_step_sync_bytes(int bs, int kv_heads) {
  if (bs <= 0 || kv_heads <= 0) return 0;
  return (int64_t)bs * kv_heads * 32 * (int64_t)sizeof(uint32_t);
}

// Compute units of the current device (cached per device).
static int device_cu_count() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cached[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cached[dev] = n;
  }
  return cached[dev];
}

// LDS of the dense attention kernel (above the 64 KiB default: opted in once per
// device).
template <bool QUEUE>
static size_t dense_smem_bytes() {
  static bool opted[64] = {false};
  int dev = 0;
  if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < 64 && !opted[dev]) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&dense_attend_kernel<QUEUE>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(DenseSmem));
    opted[dev] = true;
  }
  return sizeof(DenseSmem);
}

// LDS of a unit-attention instance: the wave combine, or the selection that
// aliases it (above the 64 KiB default for 8-wave blocks: opted in once per device).
template <bool ROWS, int KPT, int W>
static size_t unit_smem_bytes() {
  constexpr size_t kSmem = sizeof(UnitSmem<KPT, W>);
  static_assert(kSmem <= 160 * 1024, "within the CU's LDS");
  if constexpr (kSmem > 64 * 1024) {
    static bool opted[64] = {false};
    int dev = 0;
    if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < 64 && !opted[dev]) {
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&quest_attend_unit_kernel<ROWS, KPT, W>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSmem);
      opted[dev] = true;
    }
  }
  return kSmem;
}

template <bool ROWS, int KPT, int W>
static void launch_unit(const StepArgs& a, hipStream_t s) {
  const int blocks = (a.bs << a.kv_shift) * a.parts;
  quest_attend_unit_kernel<ROWS, KPT, W><<<blocks, 64 * W, unit_smem_bytes<ROWS, KPT, W>(), s>>>(a);
}

// The selection's scores per thread for n_max candidate pages (up to 8192: 32 per
// thread at W = 4, 16 at W = 8).
template <int W>
static void launch_attend_select(const StepArgs& a, int n_max, hipStream_t s) {
  constexpr int kT = 64 * W;
  constexpr int kMaxKpt = W == 4 ? 32 : 24;
  if (n_max <= 2 * kT) launch_unit<false, 2, W>(a, s);
  else if (n_max <= 4 * kT) launch_unit<false, 4, W>(a, s);
  else if (n_max <= 5 * kT) launch_unit<false, 5, W>(a, s);  // contexts up to 128K + a few pages at W = 8
  else if (n_max <= 6 * kT) launch_unit<false, 6, W>(a, s);
  else if (n_max <= 8 * kT) launch_unit<false, 8, W>(a, s);
  else if (n_max <= 9 * kT) launch_unit<false, 9, W>(a, s);  // contexts just past 128K at W = 4
  else if (n_max <= 12 * kT) launch_unit<false, 12, W>(a, s);
  else if (n_max <= 16 * kT) launch_unit<false, 16, W>(a, s);
  else if (n_max <= 24 * kT) launch_unit<false, 24, W>(a, s);
  else launch_unit<false, kMaxKpt, W>(a, s);  // contexts past 384K tokens at W = 4
}

// log2 of the KV heads for the unit attention, -1 for counts it does not take: the
// powers of two up to 8 (a pool row is KV * 128 channels, the page scores hold at
// most 1024), so that the kernel splits (request, KV head) and addresses rows with
// shifts.
static int kv_shift_of(int kv_heads) {
  return kv_heads == 1 ? 0 : kv_heads == 2 ? 1 : kv_heads == 4 ? 2 : kv_heads == 8 ? 3 : -1;
}

// Shapes the fused layer step takes (bf16, D = 128, 1, 2, 4 or 8 KV heads, G <= 16,
// page 64, at most 64 selected pages, top_k <= 4096, at most 8192 pages per request).
// new_dtype < 0: no new token.
// Per layer-step against the four launches: 8 KV heads at batch 8 x 32K 38.9 -> 29.3 us,
// 2 KV heads at batch 16 x 64K 32.3 -> 23.5 us; 4 KV heads are as with constants in the
// place of the shifts (35.5 us at batch 16 x 128K).
static bool layer_step_shape(int q_dtype, int kv_dtype, int new_dtype, int num_q_heads, int kv_heads, int head_dim,
                             int page_size, int top_k, int max_pages) {
  if (kv_shift_of(kv_heads) < 0 || head_dim != kMfmaDim || num_q_heads % kv_heads != 0 || page_size != 64 ||
      top_k <= 0 || top_k % page_size != 0)
    return false;
  return q_dtype == QQ_DTYPE_BF16 && kv_dtype == QQ_DTYPE_BF16 && (new_dtype < 0 || new_dtype == QQ_DTYPE_BF16) &&
         num_q_heads / kv_heads <= kStepMaxG && top_k / page_size - 1 <= kMaxSelFused && top_k <= kStepMaxTopK &&
         max_pages <= 32 * 64 * kUnitMinWaves;
}

// Those of qq_quest_forward_decode and its variants: the same at 4 KV heads.  Their
// callers pair them with qq_decode_attention_rows by qq_quest_fused_step, so the head
// counts at which they fuse are fixed; qq_quest_layer_step takes the others.
static bool fused_shape(int q_dtype, int kv_dtype, int new_dtype, int num_q_heads, int kv_heads, int head_dim,
                        int page_size, int top_k, int max_pages) {
  return kv_heads == 4 && layer_step_shape(q_dtype, kv_dtype, new_dtype, num_q_heads, kv_heads, head_dim, page_size,
                                           top_k, max_pages);
}

static UnitShape unit_shape(int bs, int kv_heads, int top_k) {
  return rules::unit_shape(device_cu_count(), bs, kv_heads, top_k);
}

extern "C" int qq_quest_fused_step(int q_dtype, int kv_dtype, int new_dtype, int num_q_heads, int kv_heads,
                                   int head_dim, int page_size, int top_k, int max_pages) {
  return fused_shape(q_dtype, kv_dtype, new_dtype, num_q_heads, kv_heads, head_dim, page_size, top_k, max_pages)
             ? 1
             : 0;
}

extern "C" int qq_quest_layer_step_fused(int q_dtype, int kv_dtype, int new_dtype, int num_q_heads, int kv_heads,
                                         int head_dim, int page_size, int top_k, int max_pages) {
  if (kv_heads <= 0) return 0;
  return layer_step_shape(q_dtype, kv_dtype, new_dtype, num_q_heads, kv_heads, head_dim, page_size, top_k, max_pages)
             ? 1
             : 0;
}

// The fused attention over given rows (one launch of quest_attend_unit_kernel in its rows mode);
// QQ_OK when launched, 1 when the shape or the buffers do not allow it.
int qq::attend_rows_fused(const void* q, int64_t q_bstride, int num_q_heads, const void* k_layer, const void* v_layer,
                      int64_t kv_rows, int kv_heads, const int64_t* rows, int64_t slots, const int32_t* actual, int bs, float scale,
                      void* out, void* workspace, int64_t workspace_bytes, void* sync, int64_t sync_bytes,
                      hipStream_t s) {
  if (kv_shift_of(kv_heads) < 0 || !sync || sync_bytes < qq_quest_layer_step_sync_bytes(bs, kv_heads) || slots <= 0 ||
      slots > kStepMaxTopK || slots % 64 != 0 || num_q_heads % kv_heads != 0 || num_q_heads / kv_heads > kStepMaxG ||
      !workspace)
    return 1;
  const int top_k = (int)slots;
  const int G = num_q_heads / kv_heads;
  const UnitShape us = unit_shape(bs, kv_heads, top_k);
  const int W = us.W, parts = us.parts;
  const int64_t part_bytes = (int64_t)bs * kv_heads * parts * G * (kMfmaDim + 2) * (int64_t)sizeof(float);
  if (parts > 1 && workspace_bytes < part_bytes) return 1;
  StepArgs a{};
  a.s.q = q;
  a.s.q_dtype = QQ_DTYPE_BF16;
  a.s.q_bstride = q_bstride;
  a.s.H = num_q_heads;
  a.s.top_k = top_k;
  a.s.P = 64;
  a.k = static_cast<const uint16_t*>(k_layer);
  a.v = static_cast<const uint16_t*>(v_layer);
  a.kv_rows = kv_rows;
  a.sl2 = scale * kLog2e;
  a.out = static_cast<uint16_t*>(out);
  a.part_o = static_cast<float*>(workspace);
  a.part_ml = a.part_o + (int64_t)bs * kv_heads * parts * G * kMfmaDim;
  a.kv_shift = kv_shift_of(kv_heads);
  a.parts = parts;
  a.sync = static_cast<uint32_t*>(sync);
  a.bs = bs;
  a.G = G;
  a.rows_in = rows;
  a.rows_stride = slots;
  a.actual = actual;
  if (W == 8)
    launch_unit<true, 0, 8>(a, s);
  else
    launch_unit<true, 0, 4>(a, s);
  return QQ_OK;
}

// Parts that the plan holds, at most.
static int64_t dense_entries(int bs, int64_t max_rows) {
  return rules::dense_fit(device_cu_count(), bs, max_rows) * kDenseKV;
}

extern "C" int64_t qq_dense_decode_workspace_bytes(int bs, int64_t max_rows, int num_q_heads, int kv_heads) {
  if (bs <= 0 || max_rows <= 0 || kv_heads <= 0 || num_q_heads <= 0) return 0;
  // the parts' counters, the queue, the division of the batch, then the parts' (m, l, o)
  return qq_quest_layer_step_sync_bytes(bs, kDenseKV) + (int64_t)sizeof(DenseQueue) + dense_entries(bs, max_rows) *
         (int64_t)(sizeof(DenseItem) + (num_q_heads / kv_heads) * (kMfmaDim + 2) * sizeof(float));
}

extern "C" int qq_dense_forward_decode(const void* q, int q_dtype, int64_t q_batch_stride, int num_q_heads,
                                       const void* k_new, const void* v_new, int new_dtype,
                                       const int64_t* out_cache_loc, void* k_layer, void* v_layer, int kv_dtype,
                                       int64_t kv_rows, int kv_heads, int head_dim, const int64_t* req_pool_indices,
                                       const int64_t* seq_lens, int bs, const int32_t* req_to_token,
                                       int64_t req_to_token_stride, int64_t req_to_token_rows, float scale,
                                       void* out, void* workspace, int64_t workspace_bytes, void* sync,
                                       int64_t sync_bytes, void* stream) {
  const char* what = "qq_dense_forward_decode";
  QQ_REQUIRE(q_dtype == QQ_DTYPE_BF16 && kv_dtype == QQ_DTYPE_BF16 && (!k_new || new_dtype == QQ_DTYPE_BF16) &&
                 kv_heads == kDenseKV && head_dim == kMfmaDim && num_q_heads % kv_heads == 0 &&
                 num_q_heads / kv_heads <= kStepMaxG,
             "%s: the HIP dense decode takes bf16 queries and K/V, %d KV heads x %d, at most %d query heads "
             "per KV head", what, kDenseKV, kMfmaDim, kStepMaxG);
  QQ_REQUIRE(bs >= 0 && req_to_token_stride > 0 && req_to_token_stride <= (int64_t)1 << 30, "%s: bad sizes", what);
  QQ_REQUIRE(!k_new || (v_new && out_cache_loc), "%s: new K without V or locations", what);
  if (bs == 0) return QQ_OK;
  QQ_REQUIRE(q && k_layer && v_layer && req_pool_indices && seq_lens && req_to_token && out, "%s: null pointer", what);
  QQ_REQUIRE(sync && sync_bytes >= qq_quest_layer_step_sync_bytes(bs, kv_heads), "%s: sync buffer too small", what);
  const int64_t need = qq_dense_decode_workspace_bytes(bs, req_to_token_stride, num_q_heads, kv_heads);
  QQ_REQUIRE(need == 0 || (workspace && workspace_bytes >= need), "%s: workspace %lld bytes < %lld needed", what,
             (long long)workspace_bytes, (long long)need);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int top_k = (int)req_to_token_stride;  // every context fits: seq_len <= the table's width
  const int G = num_q_heads / kv_heads;
  const int64_t entries = dense_entries(bs, top_k);
  const int round = rules::dense_round(device_cu_count());
  // a block for every (request, KV head), or as many as are resident at once
  const int64_t grid = std::min(entries, std::max<int64_t>((int64_t)bs * kDenseKV, round * kDenseKV));
  QQ_REQUIRE(entries < (int64_t)1 << 31 && req_to_token_rows < (int64_t)1 << 31, "%s: bad sizes", what);
  StepArgs a{};
  a.s.q = q;
  a.s.q_dtype = QQ_DTYPE_BF16;
  a.s.q_bstride = q_batch_stride;
  a.s.H = num_q_heads;
  a.s.rpi = req_pool_indices;
  a.s.seq = seq_lens;
  a.s.top_k = top_k;
  a.s.P = 64;
  a.s.k_sel = 0;  // no selection: positions 0 .. seq_len - 1
  a.k = static_cast<const uint16_t*>(k_layer);
  a.v = static_cast<const uint16_t*>(v_layer);
  a.kv_rows = kv_rows;
  a.r2t = req_to_token;
  a.r2t_stride = req_to_token_stride;
  a.r2t_rows = req_to_token_rows;
  a.sl2 = scale * kLog2e;
  a.out = static_cast<uint16_t*>(out);
  // everything of the call lies in its workspace: calls on several streams share nothing
  a.sync = static_cast<uint32_t*>(workspace);
  DenseQueue* queue = reinterpret_cast<DenseQueue*>(static_cast<unsigned char*>(workspace) +
                                                    qq_quest_layer_step_sync_bytes(bs, kDenseKV));
  DenseItem* plan = reinterpret_cast<DenseItem*>(queue + 1);
  a.part_o = reinterpret_cast<float*>(plan + entries);
  a.part_ml = a.part_o + entries * G * kMfmaDim;
  a.bs = bs;
  a.G = G;
  a.kv_shift = kv_shift_of(kDenseKV);
  // set_kv_buffer (memory.py:114-120) before the attention reads the pool: in 16-byte
  // pieces by the plan's launch, else by the general scatter
  const uintptr_t align = reinterpret_cast<uintptr_t>(k_new) | reinterpret_cast<uintptr_t>(v_new) |
                          reinterpret_cast<uintptr_t>(k_layer) | reinterpret_cast<uintptr_t>(v_layer);
  const bool store = k_new && align % 16 == 0;
  if (k_new && !store) {
    const int st = qq_kv_scatter(k_layer, v_layer, kv_dtype, kv_rows, k_new, v_new, new_dtype, out_cache_loc, bs,
                                 (int64_t)kv_heads * head_dim, stream);
    if (st != QQ_OK) return st;
  }
  a.s.C = kDenseKV * kMfmaDim;
  a.s.new_k = k_new;
  a.s.new_v = v_new;
  a.s.new_dtype = QQ_DTYPE_BF16;
  a.s.new_locs = out_cache_loc;
  a.s.k_pool = k_layer;
  a.s.v_pool = v_layer;
  a.s.pool_dtype = QQ_DTYPE_BF16;
  a.s.pool_rows = kv_rows;
  dense_store_plan_kernel<<<store ? bs + 1 : 1, 256, 0, s>>>(a, plan, queue, (int)(entries / kDenseKV), round,
                                                             (int)grid);
  if (entries > grid)
    dense_attend_kernel<true><<<(int)grid, 64 * kDenseWaves, dense_smem_bytes<true>(), s>>>(a, plan, queue);
  else
    dense_attend_kernel<false><<<(int)grid, 64 * kDenseWaves, dense_smem_bytes<false>(), s>>>(a, plan, queue);
  return check_launch(what);
}

static int forward_decode(
    const void* q, int q_dtype, int64_t q_batch_stride, int num_q_heads, const void* k_new,
    const void* v_new, int new_dtype, const int64_t* out_cache_loc, void* k_layer, void* v_layer,
    int kv_dtype, int64_t kv_rows, const uint16_t* page_k_bounds, int layer,
    const int64_t* req_pool_indices, const int64_t* seq_lens, const int32_t* candidate_limit,
    const int32_t* actual_lens, int bs, int max_reqs, int max_pages, int kv_heads, int head_dim,
    int page_size, int top_k, const int32_t* req_to_token, int64_t req_to_token_stride,
    int64_t req_to_token_rows, float scale, float* scores_ws, int32_t* positions, void* out,
    void* workspace, int64_t workspace_bytes, void* sync, int64_t sync_bytes,
    bool any_heads, int phase, hipStream_t s, const char* what) {
  QQ_REQUIRE(dtype_ok(q_dtype) && dtype_ok(kv_dtype) && dtype_ok(new_dtype), "%s: unsupported dtype",
             what);
  QQ_REQUIRE(kv_heads > 0 && head_dim > 0 && num_q_heads > 0 && num_q_heads % kv_heads == 0,
             "%s: q_heads %d not divisible by kv_heads %d", what, num_q_heads, kv_heads);
  QQ_REQUIRE(page_size > 0 && top_k > 0 && top_k % page_size == 0,
             "%s: top_k %d must be a positive multiple of page_size %d", what, top_k, page_size);
  const int C = kv_heads * head_dim;
  const int k_sel = top_k / page_size - 1;
  QQ_REQUIRE(C <= 1024, "%s: kv_heads*head_dim %d exceeds 1024", what, C);
  QQ_REQUIRE(k_sel <= 1024, "%s: %d selected pages exceed 1024", what, k_sel);
  QQ_REQUIRE(bs >= 0 && bs <= max_reqs && layer >= 0, "%s: bad batch/layer", what);
  QQ_REQUIRE(q && k_layer && v_layer && page_k_bounds && req_pool_indices && seq_lens &&
                 candidate_limit && actual_lens && req_to_token && scores_ws && positions && out,
             "%s: null pointer", what);
  QQ_REQUIRE(!k_new || (v_new && out_cache_loc), "%s: new K without V or locations", what);
  QQ_REQUIRE(phase >= 1 && phase <= 3, "%s: phase %d is not 1, 2 or 3", what, phase);
  if (bs == 0) return QQ_OK;

  SelectArgs sa{};
  sa.q = q;
  sa.q_dtype = q_dtype;
  sa.q_bstride = q_batch_stride;
  sa.H = num_q_heads;
  sa.bounds_layer =
      reinterpret_cast<const uint32_t*>(page_k_bounds) + (int64_t)layer * max_reqs * max_pages * C;
  sa.rpi = req_pool_indices;
  sa.seq = seq_lens;
  sa.limit = candidate_limit;
  sa.R = max_reqs;
  sa.MP = max_pages;
  sa.KV = kv_heads;
  sa.D = head_dim;
  sa.C = C;
  sa.m = (C + 63) / 64;
  sa.P = page_size;
  sa.top_k = top_k;
  sa.k_sel = k_sel;
  sa.ppb = 32;
  sa.scores = scores_ws;
  sa.positions = positions;
  sa.new_k = k_new;
  sa.new_v = v_new;
  sa.new_dtype = new_dtype;
  sa.new_locs = out_cache_loc;
  sa.k_pool = k_layer;
  sa.v_pool = v_layer;
  sa.pool_dtype = kv_dtype;
  sa.pool_rows = kv_rows;

  const int G = num_q_heads / kv_heads;
  const UnitShape us = unit_shape(bs, kv_heads, top_k);
  const int W = us.W, parts = us.parts;
  const int64_t part_bytes = (int64_t)bs * kv_heads * parts * G * (kMfmaDim + 2) * (int64_t)sizeof(float);
  const bool fused = sync && sync_bytes >= qq_quest_layer_step_sync_bytes(bs, kv_heads) &&
                     (any_heads ? layer_step_shape : fused_shape)(q_dtype, kv_dtype, k_new ? new_dtype : -1, num_q_heads,
                                                                  kv_heads, head_dim, page_size, top_k, max_pages) &&
                     workspace && workspace_bytes >= (parts > 1 ? part_bytes : 0);
  if (fused) {
    // 1. scores of the candidate pages (+ the new token's K/V), all CUs
    if (phase & 1) {
      const int st = launch_score(sa, bs, true, s);
      if (st != QQ_OK || !(phase & 2)) return st;
    }
    // 2. per (request, KV head, part): the request's selection, layout, attention, merge
    StepArgs a{};
    a.s = sa;
    a.k = static_cast<const uint16_t*>(k_layer);
    a.v = static_cast<const uint16_t*>(v_layer);
    a.kv_rows = kv_rows;
    a.r2t = req_to_token;
    a.r2t_stride = req_to_token_stride;
    a.r2t_rows = req_to_token_rows;
    a.sl2 = scale * kLog2e;
    a.out = static_cast<uint16_t*>(out);
    a.part_o = static_cast<float*>(workspace);
    a.part_ml = a.part_o + (int64_t)bs * kv_heads * parts * G * kMfmaDim;
    a.kv_shift = kv_shift_of(kv_heads);
    a.parts = parts;
    a.sync = static_cast<uint32_t*>(sync);
    a.bs = bs;
    a.G = G;
    const int n_max = max(max_pages, k_sel);
    if (W == 8)
      launch_attend_select<8>(a, n_max, s);
    else
      launch_attend_select<4>(a, n_max, s);
    return check_launch(what);
  }

  if (phase & 1) {
    const int st = launch_retrieve(sa, bs, s);
    if (st != QQ_OK || !(phase & 2)) return st;
  }

  AttnArgs aa;
  aa.q = q;
  aa.q_dtype = q_dtype;
  aa.q_bstride = q_batch_stride;
  aa.H = num_q_heads;
  aa.k = k_layer;
  aa.v = v_layer;
  aa.kv_rows = kv_rows;
  aa.KV = kv_heads;
  aa.D = head_dim;
  aa.r2t = req_to_token;
  aa.r2t_stride = req_to_token_stride;
  aa.r2t_rows = req_to_token_rows;
  aa.rpi = req_pool_indices;
  aa.positions = positions;
  aa.rows = nullptr;
  aa.pos_stride = top_k;
  aa.actual = actual_lens;
  aa.scale = scale;
  aa.out = out;
  return launch_attention(aa, kv_dtype, bs, workspace_bytes, workspace, s, what);
}

extern "C" int qq_quest_forward_decode(
    const void* q, int q_dtype, int64_t q_batch_stride, int num_q_heads, const void* k_new,
    const void* v_new, int new_dtype, const int64_t* out_cache_loc, void* k_layer, void* v_layer,
    int kv_dtype, int64_t kv_rows, const uint16_t* page_k_bounds, int layer,
    const int64_t* req_pool_indices, const int64_t* seq_lens, const int32_t* candidate_limit,
    const int32_t* actual_lens, int bs, int max_reqs, int max_pages, int kv_heads, int head_dim,
    int page_size, int top_k, const int32_t* req_to_token, int64_t req_to_token_stride,
    int64_t req_to_token_rows, float scale, float* scores_ws, int32_t* positions, void* out,
    void* workspace, int64_t workspace_bytes, void* sync, int64_t sync_bytes, void* stream) {
  return forward_decode(q, q_dtype, q_batch_stride, num_q_heads, k_new, v_new, new_dtype, out_cache_loc, k_layer, v_layer,
      kv_dtype, kv_rows, page_k_bounds, layer, req_pool_indices, seq_lens, candidate_limit, actual_lens, bs,
      max_reqs, max_pages, kv_heads, head_dim, page_size, top_k, req_to_token, req_to_token_stride,
      req_to_token_rows, scale, scores_ws, positions, out, workspace, workspace_bytes, sync, sync_bytes, false, 3, static_cast<hipStream_t>(stream), "qq_quest_forward_decode");
}

extern "C" int qq_quest_forward_decode_phase(
    const void* q, int q_dtype, int64_t q_batch_stride, int num_q_heads, const void* k_new,
    const void* v_new, int new_dtype, const int64_t* out_cache_loc, void* k_layer, void* v_layer,
    int kv_dtype, int64_t kv_rows, const uint16_t* page_k_bounds, int layer,
    const int64_t* req_pool_indices, const int64_t* seq_lens, const int32_t* candidate_limit,
    const int32_t* actual_lens, int bs, int max_reqs, int max_pages, int kv_heads, int head_dim,
    int page_size, int top_k, const int32_t* req_to_token, int64_t req_to_token_stride,
    int64_t req_to_token_rows, float scale, float* scores_ws, int32_t* positions, void* out,
    void* workspace, int64_t workspace_bytes, void* sync, int64_t sync_bytes, int phase, void* stream) {
  return forward_decode(q, q_dtype, q_batch_stride, num_q_heads, k_new, v_new, new_dtype, out_cache_loc, k_layer, v_layer,
      kv_dtype, kv_rows, page_k_bounds, layer, req_pool_indices, seq_lens, candidate_limit, actual_lens, bs,
      max_reqs, max_pages, kv_heads, head_dim, page_size, top_k, req_to_token, req_to_token_stride,
      req_to_token_rows, scale, scores_ws, positions, out, workspace, workspace_bytes, sync, sync_bytes, false, phase, static_cast<hipStream_t>(stream), "qq_quest_forward_decode_phase");
}

extern "C" int qq_quest_layer_step(
    const void* q, int q_dtype, int64_t q_batch_stride, int num_q_heads, const void* k_new,
    const void* v_new, int new_dtype, const int64_t* out_cache_loc, void* k_layer, void* v_layer,
    int kv_dtype, int64_t kv_rows, const uint16_t* page_k_bounds, int layer,
    const int64_t* req_pool_indices, const int64_t* seq_lens, const int32_t* candidate_limit,
    const int32_t* actual_lens, int bs, int max_reqs, int max_pages, int kv_heads, int head_dim,
    int page_size, int top_k, const int32_t* req_to_token, int64_t req_to_token_stride,
    int64_t req_to_token_rows, float scale, float* scores_ws, int32_t* positions, void* out,
    void* workspace, int64_t workspace_bytes, void* sync, int64_t sync_bytes, int phase, void* stream) {
  return forward_decode(q, q_dtype, q_batch_stride, num_q_heads, k_new, v_new, new_dtype, out_cache_loc, k_layer, v_layer,
      kv_dtype, kv_rows, page_k_bounds, layer, req_pool_indices, seq_lens, candidate_limit, actual_lens, bs,
      max_reqs, max_pages, kv_heads, head_dim, page_size, top_k, req_to_token, req_to_token_stride,
      req_to_token_rows, scale, scores_ws, positions, out, workspace, workspace_bytes, sync, sync_bytes, true, phase, static_cast<hipStream_t>(stream), "qq_quest_layer_step");
}

// ------------------------------------------------------------ no allocation
// qq_quest_forward_decode_noalloc: the same layer with its scratch (page
// scores, attention partials, hand-off counters) in one file-scope device
// array instead of caller workspaces, for callers that cannot allocate.  Each
// device holds its own copy; its address is looked up once per device and the
// counter region is cleared there, after which every call leaves it cleared.
namespace {

constexpr int64_t kScratchBytes = 16ll << 20;
constexpr int64_t kScratchSyncBytes = 64ll << 10;             // [0, 64 KiB): counters
constexpr int64_t kScratchScoreBytes = (4ll << 20) - kScratchSyncBytes;  // [64 KiB, 4 MiB): page scores
constexpr int64_t kScratchWorkOffset = 4ll << 20;              // [4 MiB, 16 MiB): attention partials
constexpr int64_t kScratchWorkBytes = kScratchBytes - kScratchWorkOffset;

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
unsigned char* g_scratch_ptr[kMaxDevices] = {nullptr};

__global__ void zero_words_kernel(uint32_t* p, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0u;
}

// The current device's scratch address (looked up, and its counters cleared
// on `s`, on the first call on that device); nullptr with the error recorded.
unsigned char* device_scratch(hipStream_t s) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    set_error(QQ_EHIP, "qq_quest_forward_decode_noalloc: no current HIP device (or device id >= %d)", kMaxDevices);
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev]) return g_scratch_ptr[dev];
  void* p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !p) {
    set_error(QQ_EHIP, "qq_quest_forward_decode_noalloc: hipGetSymbolAddress(scratch) failed: %s",
              hipGetErrorString(e));
    return nullptr;
  }
  zero_words_kernel<<<64, 256, 0, s>>>(static_cast<uint32_t*>(p), kScratchSyncBytes / 4);
  if (check_launch("qq_quest_forward_decode_noalloc (scratch clear)") != QQ_OK) return nullptr;
  g_scratch_ptr[dev] = static_cast<unsigned char*>(p);
  return g_scratch_ptr[dev];
}

}  // namespace

extern "C" int64_t qq_quest_forward_decode_noalloc_max_bytes(void) { return kScratchBytes; }

extern "C" int qq_quest_forward_decode_noalloc(
    const void* q, int q_dtype, int64_t q_batch_stride, int num_q_heads, const void* k_new,
    const void* v_new, int new_dtype, const int64_t* out_cache_loc, void* k_layer, void* v_layer,
    int kv_dtype, int64_t kv_rows, const uint16_t* page_k_bounds, int layer,
    const int64_t* req_pool_indices, const int64_t* seq_lens, const int32_t* candidate_limit,
    const int32_t* actual_lens, int bs, int max_reqs, int max_pages, int kv_heads, int head_dim,
    int page_size, int top_k, const int32_t* req_to_token, int64_t req_to_token_stride,
    int64_t req_to_token_rows, float scale, int32_t* positions, void* out, void* stream) {
  const char* what = "qq_quest_forward_decode_noalloc";
  QQ_REQUIRE(bs >= 0 && max_pages > 0 && kv_heads > 0 && head_dim > 0 && num_q_heads > 0, "%s: bad sizes", what);
  if (bs == 0) return QQ_OK;
  // the hand-off counters are read only by the fused layer step; other shapes take the
  // four-launch path, which needs none
  const bool fused = fused_shape(q_dtype, kv_dtype, k_new ? new_dtype : -1, num_q_heads, kv_heads, head_dim,
                                 page_size, top_k, max_pages);
  const int64_t sync_need = fused ? qq_quest_layer_step_sync_bytes(bs, kv_heads) : 0;
  const int64_t score_need = (int64_t)bs * max_pages * (int64_t)sizeof(float);
  const int64_t work_need = qq_decode_attention_workspace_bytes(bs, top_k, num_q_heads, head_dim);
  QQ_REQUIRE(sync_need <= kScratchSyncBytes && score_need <= kScratchScoreBytes && work_need <= kScratchWorkBytes,
             "%s: batch %d x %d pages x top_k %d needs %lld B of counters, %lld B of scores and %lld B of "
             "partials; the fixed scratch holds %lld, %lld and %lld",
             what, bs, max_pages, top_k, (long long)sync_need, (long long)score_need, (long long)work_need,
             (long long)kScratchSyncBytes, (long long)kScratchScoreBytes, (long long)kScratchWorkBytes);
  hipStream_t s = static_cast<hipStream_t>(stream);
  unsigned char* base = device_scratch(s);
  if (!base) return QQ_EHIP;
  return forward_decode(q, q_dtype, q_batch_stride, num_q_heads, k_new, v_new, new_dtype, out_cache_loc, k_layer,
                        v_layer, kv_dtype, kv_rows, page_k_bounds, layer, req_pool_indices, seq_lens, candidate_limit,
                        actual_lens, bs, max_reqs, max_pages, kv_heads, head_dim, page_size, top_k, req_to_token,
                        req_to_token_stride, req_to_token_rows, scale,
                        reinterpret_cast<float*>(base + kScratchSyncBytes), positions, out, base + kScratchWorkOffset,
                        kScratchWorkBytes, base, kScratchSyncBytes, false, 3, s, what);
}
