// Causal prefill attention of a batch in one launch (reference
// src/qwenquest/attention/base.py:65-93 and attention/ops.py:18-45): request i's
// n_i new tokens attend positions 0 .. prefix_i + t of its own rows
// req_to_token[req_i, :seq_i], with no host read of the lengths.
//
// bf16 queries and K/V, head_dim 128.  Scores, softmax weights and sums are fp32
// as in the general path (scaled_dot_product_attention in float32): the score
// product is exact in bf16 MFMA with fp32 accumulation, and a weight goes into
// the value product as three bf16 pieces whose sum is the fp32 weight exactly
// (8 + 8 + 8 significand bits by truncation), not as one rounded bf16.
//
// extend_kernel: a block of 4 waves takes 128 query rows of one KV head, a row
// being (token, query head of the group) in token order, so any group size fills
// the tile and the causal edge of a tile is only 128 / G tokens long.  Each wave
// holds 32 rows: S^T = K Q^T and O^T = V^T P^T with v_mfma_f32_32x32x16_bf16, so
// that a lane owns one query row throughout (its maximum, sum and rescale need no
// shuffles beyond one half-wave swap) and the S^T accumulator is the P^T operand
// as it stands (V's tokens are read in that order).  K and V tiles of 64 tokens go
// global -> LDS directly (16 B per lane, two buffers, one barrier per tile), their
// 16-byte pieces permuted in each 256-byte row so that neither K's row reads nor
// V's transposing reads (ds_read_b64_tr_b16) meet in an LDS bank; 64 KiB of LDS
// and under 256 VGPRs, so two blocks share a CU and one wave's softmax runs under
// the other's MFMAs.
//
// Bound: the matrix cores.  8192 new tokens behind 8192 cached ones, 32 / 4 heads:
// 27.5 ms with scaled_dot_product_attention in float32 over gathered rows, 2.7 to 2.8
// ms here; with the three value products that is 1180 to 1220 TFLOP/s of bf16 MFMA,
// where a library product of 8192^3 reaches 1234 on the card.  (Two pieces per weight take
// 2.2 ms, with an error against float64 that is larger in the fifth digit: the third
// piece is the weight bits that the general path keeps.)
// 600 new tokens, where a chain of ten K/V tiles per block is what counts: 26 us in the
// kernel, 30 us a call, 430 before.  The products are ordered so that neighbours have different accumulators
// (2.83 -> 2.78 ms).
#include <type_traits>

#include "qq_quest_dev.h"
#include "qq_rules.h"

namespace qq {
namespace {

typedef float float16_t __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) short4_t lds_short4_t;

constexpr int kExtWaves = 4;
using rules::extend_request_tiles;
using rules::extend_splits;
using rules::extend_tiles;
using rules::kExtMaxSplits;
using rules::kExtRows;
using rules::kExtTile;
using rules::split_chunk;
static_assert(kExtRows == 32 * kExtWaves && kExtMaxSplits <= 32, "a wave's rows; the merge's lanes");
constexpr int kTileElems = kExtTile * kMfmaDim;
constexpr int kPieces = 3;  // bf16 pieces of an fp32 weight

struct ExtendArgs {
  const uint16_t* q;  // [n, H, 128]
  int H, KV, G;
  const uint16_t* k;
  const uint16_t* v;
  int64_t kv_rows;
  const int32_t* r2t;
  int64_t r2t_stride, r2t_rows;
  const int64_t* rpi;
  const int64_t* seq;
  const int64_t* prefix;
  const int64_t* ext;
  int bs, n;
  int tiles;   // query tiles the grid holds (an upper bound of the requests' tiles), one more at its end
  int splits;  // K/V splits the grid holds
  float sl2;   // scale * log2(e)
  uint16_t* out;
  float* part_o;   // [splits, KV, tiles, 128 rows, 128]
  float* part_ml;  // [splits, KV, tiles, 128 rows, 2]
  int64_t* verdict;  // nullptr, or where the first block reports on the lengths
};

// What a block works on: request, first query row of its tile, the request's rows.
struct ExtendTile {
  int b;         // request, or -1: a tile past the requests' rows
  int tile;      // tile of the request
  int q0;        // the request's first row in q (tokens); b == -1: first token past every request
  int n;         // the request's new tokens
  int past;      // b == -1: tiles past the last request's
  int req;       // table row, or -1: outside the table
  int kv_len;    // context, cut to the table's width
  int prefix;
};

// Tiles are numbered request after request, as many as each request's rows need.
// Every wave finds the tile's request by itself: 64 requests at a time, a prefix
// sum over the lanes.
__device__ inline ExtendTile find_tile(const ExtendArgs& a, int t) {
  const int lane = threadIdx.x & 63;
  int tok = 0, tile = 0;  // tokens and tiles of the requests before this group of 64
  for (int b0 = 0; b0 < a.bs; b0 += 64) {
    const int b = b0 + lane;
    // the request's four words go out together
    const int64_t len = b < a.bs ? a.ext[b] : 0;
    const int64_t req = b < a.bs ? a.rpi[b] : 0;
    const int64_t seq = b < a.bs ? a.seq[b] : 0;
    const int64_t prefix = b < a.bs ? a.prefix[b] : 0;
    int n = (int)min(max(len, (int64_t)0), (int64_t)a.n);
    int nt = 0, sn = n;  // inclusive sums over the lanes
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int u = __shfl_up(sn, d, 64);
      if (lane >= d) sn = min(sn + u, a.n);
    }
    // q holds a.n rows: a request past them has what is left
    const int before = __shfl_up(sn, 1, 64);
    const int first = min(tok + (lane > 0 ? before : 0), a.n);
    n = min(n, a.n - first);
    const int mine = extend_request_tiles(n, a.G);
    nt = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int u = __shfl_up(nt, d, 64);
      if (lane >= d) nt += u;
    }
    const uint64_t hit = __ballot(b < a.bs && t < tile + nt);
    if (hit) {
      const int src = __builtin_ctzll(hit);
      ExtendTile r;
      r.b = b0 + src;
      r.tile = t - (tile + __shfl(nt, src, 64) - __shfl(mine, src, 64));
      r.q0 = __shfl(first, src, 64);
      r.n = __shfl(n, src, 64);
      r.past = 0;
      const int64_t row = req < 0 ? req + a.r2t_rows : req;  // a negative index counts from the table's end
      r.req = __shfl(row >= 0 && row < a.r2t_rows ? (int)row : -1, src, 64);
      const int kv = (int)min(max(seq, (int64_t)0), a.r2t_stride);
      r.kv_len = r.req >= 0 ? __shfl(kv, src, 64) : 0;  // wave-uniform branch
      r.prefix = __shfl((int)min(max(prefix, -(int64_t)(1 << 30)), (int64_t)(1 << 30)), src, 64);
      return r;
    }
    tok = min(tok + __shfl(sn, 63, 64), a.n);
    tile += __shfl(nt, 63, 64);
  }
  return {-1, 0, tok, 0, t - tile, -1, 0, 0};
}

// qq_extend_attention_checked's verdict, by one wave: one word of host memory, stored at
// system scope (nothing else is handed over with it, so no cache is written back).
__device__ inline void report_lengths(const ExtendArgs& a) {
  const int lane = threadIdx.x & 63;
  int64_t total = 0;
  bool irregular = false;
  for (int b = lane; b < a.bs; b += 64) {
    const int64_t req = a.rpi[b], n = a.ext[b], s = a.seq[b], p = a.prefix[b];
    irregular |= req < -a.r2t_rows || req >= a.r2t_rows || n < 0 || (n > 0 && (s < 1 || p < 0));
    total += n;
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) total += __shfl_xor((long long)total, d, 64);
  const bool any = __any(irregular);
  if (lane == 0)
    __hip_atomic_store(a.verdict, any ? 1 : total * 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ inline uint32_t pack_hi16(float even, float odd) {  // the high halves: truncation to bf16
  return __builtin_amdgcn_perm(__float_as_uint(odd), __float_as_uint(even), 0x07060302u);
}
__device__ inline float trunc_bf(float x) { return __uint_as_float(__float_as_uint(x) & 0xFFFF0000u); }

// The finite ones of eight bf16 values, 0 for the others.
__device__ inline bf16x8_t finite_only(bf16x8_t v) {
  u32x4_t w = __builtin_bit_cast(u32x4_t, v);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if ((w[i] & 0x7F80u) == 0x7F80u) w[i] &= 0xFFFF0000u;
    if ((w[i] & 0x7F800000u) == 0x7F800000u) w[i] &= 0xFFFFu;
  }
  return __builtin_bit_cast(bf16x8_t, w);
}

// 64 lanes x 16 bytes from per-lane global addresses to LDS byte address `lds` + 16 *
// lane.  In inline asm (it writes no register; tile_barrier waits for it), since the
// compiler would wait for the builtin's pending LDS write before the other buffer's
// reads, that is for the next tile before this one's products.  (M0 has no other use
// in these kernels.)
__device__ inline void load_lds16(const void* g, uint32_t lds) {
  __asm__ volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(g) : "memory");
}

// This wave's tile loads have landed, then every wave's: one block barrier per tile.
// (The builtin wait also tells the compiler that its own loads have landed.)
__device__ inline void wait_vm() { __builtin_amdgcn_s_waitcnt(0x0F70); }  // vmcnt(0)
__device__ inline void tile_barrier() {
  wait_vm();
  __asm__ volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

__global__ __launch_bounds__(64 * kExtWaves, 2) void extend_kernel(ExtendArgs a) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  uint16_t* sm = reinterpret_cast<uint16_t*>(smem_raw);  // [buffer][K, V][64][128]
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)smem_raw;
  // block -> (KV head, tile, split): heads fastest, so that an XCD (blocks round
  // robin) keeps to KV / 8 of the heads and its L2 to their rows; the last tiles
  // of the requests, which attend the most, first
  const int h = blockIdx.x % a.KV;
  const int rest = blockIdx.x / a.KV;
  const bool tail = rest >= a.tiles * a.splits;  // the grid's last tile, past every request's
  const int t_lin = tail ? a.tiles : a.tiles - 1 - rest % a.tiles;
  const int split = tail ? 0 : rest / a.tiles;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lo = lane & 31, hf = lane >> 5;
  if (a.verdict && blockIdx.x == 0 && wave == 0) report_lengths(a);
  const ExtendTile et = find_tile(a, t_lin);
  const int64_t row_out = (int64_t)a.H * kMfmaDim;
  if (et.b < 0) {
    // rows of q past the requests' tokens have no answer (normally there are none): NaN, in
    // 8-byte pieces, shared by the tiles past the requests' - the grid's last one always is
    const int past_tiles = a.tiles + 1 - (t_lin - et.past);
    const int pieces = a.G * kMfmaDim / 4;  // of a row, per KV head
    if (split == 0)
      for (int64_t i = et.past * 64 * kExtWaves + tid; i < (int64_t)(a.n - et.q0) * pieces;
           i += (int64_t)past_tiles * 64 * kExtWaves)
        *reinterpret_cast<uint2*>(a.out + (et.q0 + i / pieces) * row_out + ((int64_t)h * pieces + i % pieces) * 4) =
            make_uint2(0x7FC07FC0u, 0x7FC07FC0u);
    return;
  }
  const int kv_len = et.kv_len, prefix = et.prefix;
  // this lane's query row
  const int rows_n = et.n * a.G;
  const int r0 = et.tile * kExtRows;
  const int r = min(r0 + wave * 32 + lo, rows_n - 1);
  const int tok = r / a.G;
  const uint16_t* qp = a.q + (int64_t)(et.q0 + tok) * row_out + (int64_t)(h * a.G + r - tok * a.G) * kMfmaDim;
  const int lim = min(kv_len, prefix + tok + 1);  // attended positions of this row
  const int tok_first = r0 / a.G, tok_last = (min(r0 + kExtRows, rows_n) - 1) / a.G;
  const int lim_full = min(kv_len, prefix + tok_first + 1);
  const int lim_blk = min(kv_len, prefix + tok_last + 1);
  // K/V tiles of this split
  const int nt_all = lim_blk > 0 ? (lim_blk + kExtTile - 1) / kExtTile : 0;
  const int chunk = split_chunk(nt_all, a.splits);
  const bool whole = nt_all <= chunk;  // one split does it all and writes the output
  const int j_begin = split * chunk, j_end = min(nt_all, j_begin + chunk);
  if (j_begin >= j_end && !(split == 0)) return;

  bf16x8_t qb[8];
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) qb[ks] = *reinterpret_cast<const bf16x8_t*>(qp + ks * 16 + hf * 8);

  const int32_t* rt = a.r2t + (int64_t)max(et.req, 0) * a.r2t_stride;
  const int row_kv = a.KV * kMfmaDim;
  const uint16_t* kh = a.k + h * kMfmaDim;
  const uint16_t* vh = a.v + h * kMfmaDim;
  bool bad = et.req < 0;
  int rows[4];  // pool rows of this lane's tokens of the next tile: wave * 16 + 4 i + lane / 16
  auto load_rows = [&](int j) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      rows[i] = rt[min(j * kExtTile + wave * 16 + i * 4 + (lane >> 4), lim_blk - 1)];  // none past the block's limit
  };
  auto load_tile = [&](int buf) {
    // this wave's 16 tokens of the buffer's K tile (bytes)
    const uint32_t base = lds0 + (uint32_t)(buf * 2 * kTileElems + wave * 16 * kMfmaDim) * 2u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = wave * 16 + i * 4 + (lane >> 4);  // token of the tile
      int64_t row = rows[i];
      row += row < 0 ? a.kv_rows : 0;
      const bool ok = row >= 0 && row < a.kv_rows;
      bad |= !ok;
      row = ok ? row : 0;
      const int ck = (lane & 15) ^ (t & 15);        // which 16-byte piece lands in this lane's place
      const int cv = (lane & 15) ^ ((t & 3) << 2);
      load_lds16(kh + row * row_kv + ck * 8, base + i * 4 * kMfmaDim * 2);
      load_lds16(vh + row * row_kv + cv * 8, base + (kTileElems + i * 4 * kMfmaDim) * 2);
    }
  };
  float16_t o[4];
  float M, L;

  // K operand pieces 2 ks + hf of row lo (+ 32); V operand: token 4 hf + l16 / 4, channels 16 (g & 1) + 4 (l16 % 4)
  const int l16 = lane & 15;
  const int v_row = 4 * hf + (l16 >> 2);
  int k_off[8], v_off[4];
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) k_off[ks] = lo * kMfmaDim + (((2 * ks + hf) ^ (lo & 15)) << 3);
#pragma unroll
  for (int c = 0; c < 4; ++c)
    v_off[c] = v_row * kMfmaDim + ((c ^ (l16 >> 2)) << 5) + ((lane >> 4) & 1) * 16 + (l16 & 3) * 4;

  // the block's K/V tiles; finite: the lower pieces of a weight meet only finite values
  auto attend = [&](auto finite) {
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[c][i] = 0.0f;
    M = -INFINITY;
    L = 0.0f;
    if (j_begin < j_end) {
      load_rows(j_begin);
      load_tile(0);
      if (j_begin + 1 < j_end) load_rows(j_begin + 1);
    }
    int buf = 0;
    for (int j = j_begin; j < j_end; ++j) {
      tile_barrier();
      if (j + 1 < j_end) {
        load_tile(buf ^ 1);
        if (j + 2 < j_end) load_rows(j + 2);
      }
      const uint16_t* sk = sm + buf * 2 * kTileElems;
      const uint16_t* sv = sk + kTileElems;
      buf ^= 1;
      // S^T[token 32 t + 8 (i / 4) + 4 hf + i % 4][row lo] in s[t][i]
      float16_t s[2];
      {
        bf16x8_t ka[2][8];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
          for (int ks = 0; ks < 8; ++ks)
            ka[t][ks] = *reinterpret_cast<const bf16x8_t*>(sk + t * 32 * kMfmaDim + k_off[ks]);
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
          for (int i = 0; i < 16; ++i) s[t][i] = 0.0f;
#pragma unroll
          for (int ks = 0; ks < 8; ++ks)
            s[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[t][ks], qb[ks], s[t], 0, 0, 0);
        }
        // the first 32 tokens' reads, then the others' under their products
        __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x8, 8, 0);
      }
      if ((j + 1) * kExtTile > lim_full) {  // block-uniform: some row's limit is inside this tile
        const int left = lim - j * kExtTile - 4 * hf;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            s[t][i] = (t * 32 + 8 * (i / 4) + i % 4) < left ? s[t][i] : -INFINITY;
      }
      float mx = s[0][0];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[t][i]);
      mx = fmaxf(mx, lane_xor32(mx, lane));
      if (__any(mx > M)) {
        const float Mn = fmaxf(M, mx);
        const float alpha = M == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((M - Mn) * a.sl2);
        L *= alpha;
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[c][i] *= alpha;
        M = Mn;
      }
      const float mb = M == -INFINITY ? 0.0f : -M * a.sl2;  // nothing attended yet: weights of 0
      float sum = 0.0f;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t][i], a.sl2, mb));
          s[t][i] = p;
          sum += p;
        }
      L += sum;
      // O^T += V^T P^T, 16 tokens at a time, P in bf16 pieces
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        u32x4_t pw[kPieces];
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          float e = s[u >> 1][(u & 1) * 8 + 2 * x], f = s[u >> 1][(u & 1) * 8 + 2 * x + 1];
#pragma unroll
          for (int c = 0; c < kPieces; ++c) {
            pw[c][x] = pack_hi16(e, f);
            e -= trunc_bf(e);
            f -= trunc_bf(f);
          }
        }
        bf16x8_t va[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          uint16_t* vp = const_cast<uint16_t*>(sv) + v_off[c] + u * 16 * kMfmaDim;
          const short4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)vp);
          const short4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)(vp + 8 * kMfmaDim));
          va[c] = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
        }
        bf16x8_t vl[4];  // for the weights' lower pieces
#pragma unroll
        for (int c = 0; c < 4; ++c) vl[c] = decltype(finite)::value ? finite_only(va[c]) : va[c];
#pragma unroll
        for (int x = 0; x < kPieces; ++x)
#pragma unroll
          for (int c = 0; c < 4; ++c)  // independent accumulators one after the other
            o[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x == 0 ? va[c] : vl[c],
                                                           __builtin_bit_cast(bf16x8_t, pw[x]), o[c], 0, 0, 0);
      }
    }
    L += lane_xor32(L, lane);
  };
  attend(std::false_type{});
  // An infinite value times a weight is infinite (or NaN, for a weight of 0), but times a
  // lower piece that happens to be 0 it is NaN: where a sum is NaN and its weights are not,
  // the block goes over its tiles again with the infinities left to the upper pieces.
  bool again = false;
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int i = 0; i < 16; ++i) again |= o[c][i] != o[c][i];
  again &= L == L;
  if (__syncthreads_or(bad || again)) {
    if (__syncthreads_or(again)) attend(std::true_type{});
    if (__syncthreads_or(bad)) L = __builtin_nanf("");  // a row outside the pool: no answer
  }
  const bool mine = r0 + wave * 32 + lo < rows_n;
  if (whole) {
    if (!mine) return;
    uint16_t* op = a.out + (qp - a.q) + 4 * hf;
    const float inv = 1.0f / L;
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const uint32_t w0 = (uint32_t)f2bf(o[c][4 * g] * inv) | ((uint32_t)f2bf(o[c][4 * g + 1] * inv) << 16);
        const uint32_t w1 = (uint32_t)f2bf(o[c][4 * g + 2] * inv) | ((uint32_t)f2bf(o[c][4 * g + 3] * inv) << 16);
        *reinterpret_cast<uint2*>(op + c * 32 + g * 8) = make_uint2(w0, w1);
      }
    return;
  }
  const int64_t pr = (((int64_t)split * a.KV + h) * a.tiles + t_lin) * kExtRows + wave * 32 + lo;
  float* po = a.part_o + pr * kMfmaDim + 4 * hf;
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<float4*>(po + c * 32 + g * 8) =
          make_float4(o[c][4 * g], o[c][4 * g + 1], o[c][4 * g + 2], o[c][4 * g + 3]);
  if (hf == 0) *reinterpret_cast<float2*>(a.part_ml + pr * 2) = make_float2(M * a.sl2, L);
}

// Adds up a tile's splits: one block per (tile, KV head, 8 rows), 32 threads a row.
__global__ __launch_bounds__(256) void extend_merge_kernel(ExtendArgs a) {
  const int h = blockIdx.y, t_lin = blockIdx.x;
  const ExtendTile et = find_tile(a, t_lin);
  if (et.b < 0) return;
  const int kv_len = et.kv_len, prefix = et.prefix;
  const int rows_n = et.n * a.G, r0 = et.tile * kExtRows;
  const int tok_last = (min(r0 + kExtRows, rows_n) - 1) / a.G;
  const int lim_blk = min(kv_len, prefix + tok_last + 1);
  const int nt_all = lim_blk > 0 ? (lim_blk + kExtTile - 1) / kExtTile : 0;
  const int chunk = split_chunk(nt_all, a.splits);
  if (nt_all <= chunk) return;
  const int parts = (nt_all + chunk - 1) / chunk;
  const int i = blockIdx.z * 8 + (threadIdx.x >> 5), d4 = (threadIdx.x & 31) * 4;
  const int r = r0 + i;
  if (r >= rows_n) return;  // all 32 lanes of the row
  const int64_t step = (int64_t)a.KV * a.tiles * kExtRows;
  const int64_t pr = ((int64_t)h * a.tiles + t_lin) * kExtRows + i;
  // lane p of the row's 32 holds part p's (m, l): parts <= kExtMaxSplits
  const int p = threadIdx.x & 31;
  const float2 ml = p < parts ? *reinterpret_cast<const float2*>(a.part_ml + (pr + p * step) * 2)
                              : make_float2(-INFINITY, 0.0f);
  float Mx = ml.x;
#pragma unroll
  for (int d = 1; d < 32; d <<= 1) Mx = fmaxf(Mx, __shfl_xor(Mx, d, 32));
  const float w = ml.x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ml.x - Mx);
  float Ls = w * ml.y;
#pragma unroll
  for (int d = 1; d < 32; d <<= 1) Ls += __shfl_xor(Ls, d, 32);
  float4 Os = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int p0 = 0; p0 < parts; p0 += 8) {
    float4 ov[8];  // a group's loads go out together; past the last part they re-read it
#pragma unroll
    for (int u = 0; u < 8; ++u)
      ov[u] = *reinterpret_cast<const float4*>(a.part_o + (pr + min(p0 + u, parts - 1) * step) * kMfmaDim + d4);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float wu = __shfl(w, p0 + u, 32);  // p0 + u < 32
      if (p0 + u >= parts) break;  // block-uniform; a weight of 0 would make NaN of an infinite sum
      Os.x += wu * ov[u].x;
      Os.y += wu * ov[u].y;
      Os.z += wu * ov[u].z;
      Os.w += wu * ov[u].w;
    }
  }
  const float inv = 1.0f / Ls;
  const int tok = r / a.G;
  uint16_t* op = a.out + ((int64_t)(et.q0 + tok) * a.H + h * a.G + r - tok * a.G) * kMfmaDim + d4;
  *reinterpret_cast<uint2*>(op) = make_uint2((uint32_t)f2bf(Os.x * inv) | ((uint32_t)f2bf(Os.y * inv) << 16),
                                             (uint32_t)f2bf(Os.z * inv) | ((uint32_t)f2bf(Os.w * inv) << 16));
}

}  // namespace
}  // namespace qq

using namespace qq;

// Waits for a launch's verdict: it reports as it begins; a stream that is done, or in
// error, has nothing to wait for.
static int wait_verdict(const int64_t* verdict, hipStream_t s, const char* what) {
  for (;;) {
    for (int spin = 0; spin < 4096; ++spin) {
      if (__atomic_load_n(verdict, __ATOMIC_ACQUIRE) >= 0) return QQ_OK;
      __builtin_ia32_pause();
    }
    const hipError_t e = hipStreamQuery(s);
    if (e == hipErrorNotReady) continue;
    if (e == hipSuccess && __atomic_load_n(verdict, __ATOMIC_ACQUIRE) >= 0) return QQ_OK;
    set_error(QQ_EHIP, "%s: no verdict: %s", what, hipGetErrorString(e));
    return QQ_EHIP;
  }
}

extern "C" int64_t qq_extend_attention_workspace_bytes(int64_t n, int bs, int num_q_heads, int kv_heads,
                                                       int64_t max_rows) {
  if (n <= 0 || bs <= 0 || kv_heads <= 0 || num_q_heads < kv_heads) return 0;
  const int64_t tiles = extend_tiles(n, bs, num_q_heads / kv_heads);
  const int splits = extend_splits(tiles, kv_heads, max_rows);
  return splits > 1 ? splits * kv_heads * tiles * kExtRows * (kMfmaDim + 2) * (int64_t)sizeof(float) : 0;
}

extern "C" int qq_extend_attention(const void* q, int num_q_heads, const void* k_layer, const void* v_layer,
                                   int64_t kv_rows, int kv_heads, int head_dim, const int32_t* req_to_token,
                                   int64_t req_to_token_stride, int64_t req_to_token_rows,
                                   const int64_t* req_pool_indices, const int64_t* seq_lens,
                                   const int64_t* prefix_lens, const int64_t* extend_lens, int bs, int64_t n,
                                   float scale, void* out, void* workspace, int64_t workspace_bytes, void* stream) {
  return qq_extend_attention_checked(q, num_q_heads, k_layer, v_layer, kv_rows, kv_heads, head_dim, req_to_token,
                                     req_to_token_stride, req_to_token_rows, req_pool_indices, seq_lens, prefix_lens,
                                     extend_lens, bs, n, scale, out, workspace, workspace_bytes, nullptr, stream);
}

extern "C" int qq_extend_attention_checked(const void* q, int num_q_heads, const void* k_layer, const void* v_layer,
                                           int64_t kv_rows, int kv_heads, int head_dim, const int32_t* req_to_token,
                                           int64_t req_to_token_stride, int64_t req_to_token_rows,
                                           const int64_t* req_pool_indices, const int64_t* seq_lens,
                                           const int64_t* prefix_lens, const int64_t* extend_lens, int bs, int64_t n,
                                           float scale, void* out, void* workspace, int64_t workspace_bytes,
                                           int64_t* verdict, void* stream) {
  const char* what = "qq_extend_attention";
  QQ_REQUIRE(kv_heads > 0 && num_q_heads > 0 && num_q_heads % kv_heads == 0,
             "%s: q_heads %d not divisible by kv_heads %d", what, num_q_heads, kv_heads);
  QQ_REQUIRE(head_dim == kMfmaDim, "%s: head_dim %d is not %d", what, head_dim, kMfmaDim);
  QQ_REQUIRE(scale > 0.0f, "%s: the scale must be positive", what);
  QQ_REQUIRE(bs >= 0 && n >= 0 && n * (num_q_heads / kv_heads) < (int64_t)1 << 30 && req_to_token_stride > 0 &&
                 req_to_token_stride < (int64_t)1 << 30 && kv_rows > 0 &&
                 req_to_token_rows < (int64_t)1 << 31,
             "%s: bad sizes", what);
  if (verdict) *verdict = bs == 0 || n == 0 ? 0 : -1;
  if (bs == 0 || n == 0) return QQ_OK;
  QQ_REQUIRE(q && k_layer && v_layer && req_to_token && req_pool_indices && seq_lens && prefix_lens &&
                 extend_lens && out, "%s: null pointer", what);
  const int64_t need =
      qq_extend_attention_workspace_bytes(n, bs, num_q_heads, kv_heads, req_to_token_stride);
  QQ_REQUIRE(need == 0 || (workspace && workspace_bytes >= need), "%s: workspace %lld bytes < %lld needed", what,
             (long long)workspace_bytes, (long long)need);
  ExtendArgs a{};
  a.q = static_cast<const uint16_t*>(q);
  a.H = num_q_heads;
  a.KV = kv_heads;
  a.G = num_q_heads / kv_heads;
  a.k = static_cast<const uint16_t*>(k_layer);
  a.v = static_cast<const uint16_t*>(v_layer);
  a.kv_rows = kv_rows;
  a.r2t = req_to_token;
  a.r2t_stride = req_to_token_stride;
  a.r2t_rows = req_to_token_rows;
  a.rpi = req_pool_indices;
  a.seq = seq_lens;
  a.prefix = prefix_lens;
  a.ext = extend_lens;
  a.bs = bs;
  a.n = (int)n;
  const int64_t tiles = extend_tiles(n, bs, a.G);
  a.splits = extend_splits(tiles, kv_heads, req_to_token_stride);
  const int64_t grid = (tiles * a.splits + 1) * kv_heads;
  QQ_REQUIRE(grid < (int64_t)1 << 31, "%s: too many query rows", what);
  a.tiles = (int)tiles;
  a.sl2 = scale * kLog2e;
  a.out = static_cast<uint16_t*>(out);
  a.part_o = static_cast<float*>(workspace);
  a.part_ml = a.part_o ? a.part_o + a.splits * kv_heads * tiles * kExtRows * kMfmaDim : nullptr;
  a.verdict = verdict;
  hipStream_t s = static_cast<hipStream_t>(stream);
  constexpr size_t kSmem = 4 * kTileElems * sizeof(uint16_t);  // 64 KiB: two buffers of K and V
  extend_kernel<<<(int)grid, 64 * kExtWaves, kSmem, s>>>(a);
  if (a.splits > 1)
    extend_merge_kernel<<<dim3(a.tiles, kv_heads, kExtRows / 8), 256, 0, s>>>(a);
  const int st = check_launch(what);
  return st == QQ_OK && verdict ? wait_verdict(verdict, s, what) : st;
}
