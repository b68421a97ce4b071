// What the bf16 decode attention's own kernels share with the launch that takes the keys every step attends to beside the
// retrieval's query side, and with the top-k that goes on to attend to what it selected: places of keys, the step over 32 keys on
// the matrix cores, the merge of the waves.
#pragma once

#include "pkv_common.h"

#if defined(__HIPCC__)

// Fused multiply-add is welcome in every function here (the rest of the library forbids it because integer results are
// derived from its float steps; the attention's only contract is its tolerance).
#define PKV_ATT_CONTRACT _Pragma("clang fp contract(fast)")

constexpr float kNegBig = -1.0e30f;

// Segments that share one K and one V tensor (the cache's rows in HBM: sink, selected rows, local window), at most one of
// them indexed: a key is a 32-bit byte offset into the (b, h) slab.  Half of a launch over a few hundred keys used to go
// into finding addresses (1.2 us to pick a 64-bit pointer out of four for each of a lane's ten rows, after 1 us for a
// 300-byte argument block); here that is one lane exchange per row.
struct AttOne {
  const char *k, *v;
  int64_t stride_b, stride_h;           // bytes
  uint32_t end[PKV_ATTN_MAX_SEGMENTS];  // exclusive ends in the concatenated key order; unused: 2^32 - 1
  int32_t delta[PKV_ATTN_MAX_SEGMENTS]; // row - concatenated key
  const int64_t *idx;                   // of the indexed segment, keys [idx_lo, idx_hi)
  int64_t idx_stride, idx_limit;
  uint32_t idx_lo, idx_hi, idx_row0;
};

// One key's place: a byte offset into the slab (AttOne), or the addresses of its K and V rows.
template <bool ONE>
struct AttPlace {
  uint32_t off;
  __device__ __forceinline__ AttPlace from(int lane) const { return {(uint32_t)__shfl((int)off, lane, PKV_WAVE)}; }
};
template <>
struct AttPlace<false> {
  uint64_t k, v;
  __device__ __forceinline__ const char *k_from(int lane) const { return (const char *)pull(k, lane); }
  __device__ __forceinline__ const char *v_from(int lane) const { return (const char *)pull(v, lane); }
  static __device__ __forceinline__ uint64_t pull(uint64_t x, int lane) {
    return ((uint64_t)(uint32_t)__shfl((int)(x >> 32), lane, PKV_WAVE) << 32) | (uint32_t)__shfl((int)(uint32_t)x, lane, PKV_WAVE);
  }
};

// ROW: bytes of a row.
template <bool INDEXED, uint32_t ROW>
__device__ __forceinline__ AttPlace<true> att_place(const AttOne &a, int row, int, int, uint32_t jj) {
  int32_t d = a.delta[0];
#pragma unroll
  for (int t = 1; t < PKV_ATTN_MAX_SEGMENTS; ++t) d = jj >= a.end[t - 1] ? a.delta[t] : d;
  uint32_t r = jj + (uint32_t)d;
  if (INDEXED && jj >= a.idx_lo && jj < a.idx_hi) {
    const int64_t x = a.idx[(int64_t)row * a.idx_stride + (jj - a.idx_lo)];
    r = a.idx_row0 + (uint32_t)(x < 0 ? 0 : (x >= a.idx_limit ? a.idx_limit - 1 : x));
  }
  return {r * ROW};
}

// Partial results layout: ws[((row * n_splits + split) * G + g) * 130 + {0: max, 1: sum, 2..129: output}].
constexpr int kPartStride = 130;

// ---- bf16 inputs: a partial result on the matrix cores ----
//
// Each wave: 32 keys per step, v_mfma_f32_16x16x32_bf16 throughout.
//   scores:  S^T[key][head] = K[key][dim] . Q^T[dim][head]: A = 16 keys x 32 dims (lane (r, j) holds dims
//            32c + 8j .. +7 of key r: one 128-bit load), B = the query heads (zero columns past `group`),
//            4 instructions per 16 keys.  Lane (n, j) receives the scores of head n for keys 4j .. 4j+3 of the
//            tile - which is exactly where the next product wants the probabilities, so nothing is moved.
//   output:  O[head][dim] += P[head][key] . V[key][dim] over the 32 keys of two tiles: lane (n, j) supplies its
//            8 probabilities as A; for B it loads dims 8n .. 8n+7 of its 8 keys (rows read whole, 16 lanes per
//            row) and regroups them with byte permutes so that instruction m covers the dims 8n + m.
// The running maximum of head n lives in the lanes n, n+16, n+32, n+48; the output rows of head h live in lanes
// with j == h / 4.  group <= 16, all heads of the KV head in one pass.
typedef __bf16 pkv_bf16x8 __attribute__((ext_vector_type(8)));
typedef float pkv_f32x4 __attribute__((ext_vector_type(4)));
constexpr int kMfmaStepKeys = 32;

__device__ __forceinline__ pkv_f32x4 mfma_bf16(pkv_u32x4 a, pkv_u32x4 b, pkv_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(pkv_bf16x8, a), __builtin_bit_cast(pkv_bf16x8, b), c,
                                                 0, 0, 0);
}

// A score is rounded before the maximum is taken from it, whatever the compiler could fuse around a call.
__device__ __forceinline__ float att_scaled(float score, float scale) {
#pragma clang fp contract(off)
  return score * scale;
}

__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  return (uint32_t)pkv_f32_to_bf16_bits(lo) | ((uint32_t)pkv_f32_to_bf16_bits(hi) << 16);
}

constexpr int kMfmaWaves = 4;  // waves per workgroup: each takes a quarter of the split, merged through LDS

// Keys jb .. jb + 31 (of them those below j1) into the running maximum, the lane's share of the sum and the output of a wave.
// Lane in_block + i of `mine` holds the place of key jb + i.  FIRST: nothing has run yet.
template <bool ONE, bool FIRST>
__device__ __forceinline__ void att_step_mfma(const char *kbase, const char *vbase, const AttPlace<ONE> &mine, int in_block, int64_t jb,
                                              int64_t j1, const pkv_u32x4 (&qb)[4], float scale_log2e, float &m_run, float &l_part,
                                              pkv_f32x4 (&o)[8]) {
  PKV_ATT_CONTRACT
  const int lane = threadIdx.x & (PKV_WAVE - 1), n = lane & 15, j = lane >> 4;
  // K: two tiles of 16 keys, lane (n, j) reads dims 32c + 8j .. +7 of key jb + 16t + n.  Two instructions share a 128-byte line:
  // plain loads, as a streaming load gives it up after the first.  V rows are read whole.  Attention, us, K streaming / plain:
  // 8 rows x 700 keys 7.4 / 7.1, 64 x 887 11.4 / 10.6, by index 12.3 / 11.6, 64 x 2000 18.7 / 18.1, by index 21.5 / 19.0,
  // 512 x 900 52.2 / 49.2, by index 61.1 / 49.7, 1024 x 2000 207.7 / 188.1.
  pkv_u32x4 ka[2][4], vr[8];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const char *kp;
    if constexpr (ONE) kp = kbase + (uint64_t)(mine.from(in_block + 16 * t + n).off + 16u * (uint32_t)j);
    else kp = mine.k_from(in_block + 16 * t + n) + 16 * j;
#pragma unroll
    for (int c = 0; c < 4; ++c) ka[t][c] = *(const pkv_u32x4 *)(kp + 64 * c);
  }
  // V: dims 8n .. 8n+7 of the 8 keys whose probabilities this lane will hold
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int at = in_block + 16 * (e >> 2) + 4 * j + (e & 3);
    const char *vp;
    if constexpr (ONE) vp = vbase + (uint64_t)(mine.from(at).off + 16u * (uint32_t)n);
    else vp = mine.v_from(at) + 16 * n;
    vr[e] = __builtin_nontemporal_load((const pkv_u32x4 *)vp);
  }

  pkv_f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    s0 = mfma_bf16(ka[0][c], qb[c], s0);
    s1 = mfma_bf16(ka[1][c], qb[c], s1);
  }
  float sc[8];
  bool valid[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    valid[e] = jb + 16 * (e >> 2) + 4 * j + (e & 3) < j1;
    const float raw = (e < 4) ? s0[e & 3] : s1[e & 3];
    sc[e] = valid[e] ? att_scaled(raw, scale_log2e) : kNegBig;
  }
  float mx = sc[0];
#pragma unroll
  for (int e = 1; e < 8; ++e) mx = fmaxf(mx, sc[e]);
  mx = pkv_pair_max<32>(pkv_pair_max<16>(mx));
  const float m_new = fmaxf(m_run, mx);
  // the hardware's exp2: exp2f but for results below 2^-126, which are zero; nothing beside the largest weight, which is 1
  const float corr = __builtin_amdgcn_exp2f(m_run - m_new);
  m_run = m_new;
  float p[8], psum = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    p[e] = valid[e] ? __builtin_amdgcn_exp2f(sc[e] - m_new) : 0.f;
    psum += p[e];
  }
  l_part = fmaf(l_part, corr, psum);
  const pkv_u32x4 pa = {pack_bf16x2(p[0], p[1]), pack_bf16x2(p[2], p[3]), pack_bf16x2(p[4], p[5]),
                        pack_bf16x2(p[6], p[7])};
  // the output rows of this lane belong to heads 4j .. 4j+3: fetch their correction factors
  float cr[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) cr[i] = __shfl(corr, 4 * j + i, PKV_WAVE);
#pragma unroll
  for (int m = 0; m < 8; ++m) {
    // element m of each of the eight V vectors: dword m/2, half m%2
    const uint32_t sel = (m & 1) ? 0x07060302u : 0x05040100u;
    pkv_u32x4 bm;
    bm.x = __builtin_amdgcn_perm(vr[1][m >> 1], vr[0][m >> 1], sel);
    bm.y = __builtin_amdgcn_perm(vr[3][m >> 1], vr[2][m >> 1], sel);
    bm.z = __builtin_amdgcn_perm(vr[5][m >> 1], vr[4][m >> 1], sel);
    bm.w = __builtin_amdgcn_perm(vr[7][m >> 1], vr[6][m >> 1], sel);
    pkv_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (!FIRST) acc = o[m], acc.x *= cr[0], acc.y *= cr[1], acc.z *= cr[2], acc.w *= cr[3];
    o[m] = mfma_bf16(pa, bm, acc);
  }
}

// a value for a later launch, or (HANDED) for another workgroup of this one, whatever die that runs on
template <bool HANDED>
__device__ __forceinline__ void att_put(float *p, float v) {
  if (HANDED) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = v;
}

// Merge of the waves of a workgroup: every wave leaves (max, sum, output) of its keys in LDS, then the workgroup's 256 threads
// combine them, one (head, dim) pair at a time.  group <= 8.
// ml / out: of head 0; the next head's lie ml_stride / out_stride floats on.  HANDED: another workgroup of the launch reads them.
template <bool HANDED = false>
__device__ __forceinline__ void att_merge_waves(int group, float m_run, float l_part, const pkv_f32x4 (&o)[8], float *ml, int ml_stride,
                                                float *out, int out_stride) {
  PKV_ATT_CONTRACT
  const int lane = threadIdx.x & (PKV_WAVE - 1), wave = threadIdx.x / PKV_WAVE, n = lane & 15, j = lane >> 4;
  __shared__ float s_m[kMfmaWaves][8], s_l[kMfmaWaves][8];
  __shared__ alignas(16) float s_o[kMfmaWaves][8][128 + 4];  // written by 128 bits
  if (j == 0 && n < group) s_m[wave][n] = m_run, s_l[wave][n] = l_part;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int head = 4 * j + i;
    if (head < group) {
      *(float4 *)&s_o[wave][head][8 * n] = float4{o[0][i], o[1][i], o[2][i], o[3][i]};
      *(float4 *)&s_o[wave][head][8 * n + 4] = float4{o[4][i], o[5][i], o[6][i], o[7][i]};
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < group * 128; e += kMfmaWaves * PKV_WAVE) {
    const int g = e >> 7, d = e & 127;
    float mn = s_m[0][g];
#pragma unroll
    for (int w = 1; w < kMfmaWaves; ++w) mn = fmaxf(mn, s_m[w][g]);
    float ls = 0.f, os = 0.f;
#pragma unroll
    for (int w = 0; w < kMfmaWaves; ++w) {
      const float c = exp2f(s_m[w][g] - mn);
      ls = fmaf(s_l[w][g], c, ls);
      os = fmaf(s_o[w][g][d], c, os);
    }
    att_put<HANDED>(out + g * out_stride + d, os);
    if (d == 0) att_put<HANDED>(ml + g * ml_stride, mn), att_put<HANDED>(ml + g * ml_stride + 1, ls);
  }
}
// ---- a decode step's attention in two parts ----
//
// The sink and local rows are known before the retrieval starts, and a third of a short step went into the two launches behind
// its top-k (4.9 + 2.7 of 26.5 us at 8 rows x 4096 keys), so: workgroups beside the query side of the retrieval, on an otherwise
// idle chip, take the keys that are not selected, and the top-k's workgroups go on with those that are.  The sums are those of the
// one-piece attention, bit for bit: the same blocks of 32 keys (a wave's), merged by fours into splits and the splits into the
// output in the same order, with the fused form of each a * b + c written out on both sides.
constexpr int kSelBlocks = 8;   // most blocks of a selecting workgroup
constexpr int kSelSplits = 12;  // one more than a row's splits may be where the selecting workgroup merges
constexpr int kSelSlots = 32;   // partial results of a row there: splits in 0 .. 11, single blocks in 12 .. 19

struct PkvSplitAttn {
  AttOne segs;
  uint32_t total;
  int n_splits;               // of 128 keys
  int blk_lo, blk_hi;         // blocks of 32 keys that hold a selected one; the top-k's workgroups take these ...
  int sel_wgs, splits_per_wg; // ... sel_wgs == 1: one workgroup a row, which also merges; else whole splits, so many to a workgroup
  uint32_t slots;             // sel_wgs == 1: the partial results that the first launch leaves
  int n_dense, dense_a, dense_skip;  // workgroups of the first launch: splits 0 .. dense_a - 1, then from dense_a + dense_skip on
  int n_kv_heads, group;
  const void *q;
  float scale_log2e;
  float *ws;                  // sel_wgs == 1: outputs [row][20][group][128], then at ws_ml (max, sum) [row][group][kSelSlots]; else
  float *ws_ml;               // partial results of the splits as the one-piece attention leaves them
  void *out;
};

// sel_wgs == 1: a split with selected keys in some of its blocks leaves its other blocks one by one: the first such split in slots
// 12 .. 15, another (the last) in 16 .. 19.
__host__ __device__ __forceinline__ int att_block_slot(const PkvSplitAttn &a, int block) {
  return kSelSplits + (block & 3) + (block / 4 == a.blk_lo / 4 ? 0 : 4);
}
__device__ __forceinline__ float *att_slot_o(const PkvSplitAttn &a, int row, int slot, int head) {
  return a.ws + (uint32_t)(((row * 20 + slot) * a.group + head) * 128);
}
__device__ __forceinline__ float *att_slot_ml(const PkvSplitAttn &a, int row, int slot, int head) {
  return a.ws_ml + (uint32_t)(((row * a.group + head) * kSelSlots + slot) * 2);
}

// The arguments arrive in 64-byte lines when first read.  Read here, behind the caller's own loads, they are there when the attention
// starts instead of after a trip to memory of its own.
__device__ __forceinline__ void att_arguments(const PkvSplitAttn &a) {
  const uint64_t k = (uint64_t)a.segs.k, idx = (uint64_t)a.segs.idx_limit, q = (uint64_t)a.q;
  const int blk = a.blk_lo;
  asm volatile("" ::"s"(k), "s"(idx), "s"(q), "s"(blk));
}

__device__ __forceinline__ void att_load_q(const PkvSplitAttn &a, int row, pkv_u32x4 (&qb)[4]) {
  const int lane = pkv_lane(), n = lane & 15, j = lane >> 4;
  const pkv_u32x4 zero4 = {0u, 0u, 0u, 0u};
  const pkv_u32x4 *qp = (const pkv_u32x4 *)((const uint16_t *)a.q + ((int64_t)row * a.group + (n < a.group ? n : 0)) * 128 + 8 * j);
#pragma unroll
  for (int c = 0; c < 4; ++c) qb[c] = qp[4 * c];
  if (n >= a.group) qb[0] = qb[1] = qb[2] = qb[3] = zero4;
}

// Workgroup x of a row's n_dense: 256 threads.
__device__ __forceinline__ void att_dense_part(const PkvSplitAttn &a, int x, int row) {
  const int split = x < a.dense_a ? x : x + a.dense_skip;
  const int lane = pkv_lane(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PKV_WAVE), n = lane & 15, j = lane >> 4;
  const int b = row / a.n_kv_heads, h = row % a.n_kv_heads, block = 4 * split + wave;
  const bool mixed = 4 * split + 3 >= a.blk_lo && 4 * split <= a.blk_hi;
  const uint32_t j0 = 32u * (uint32_t)block, j1 = j0 + 32u < a.total ? j0 + 32u : a.total;
  const bool has = j0 < a.total && !(block >= a.blk_lo && block <= a.blk_hi);
  float m_run = kNegBig, l_part = 0.f;
  pkv_f32x4 o[8];
#pragma unroll
  for (int m = 0; m < 8; ++m) o[m] = pkv_f32x4{0.f, 0.f, 0.f, 0.f};
  if (has) {
    const int64_t slab = (int64_t)b * a.segs.stride_b + (int64_t)h * a.segs.stride_h;
    const uint32_t key = j0 + (uint32_t)(lane & 31);
    const AttPlace<true> mine = att_place<false, 256>(a.segs, row, b, h, key < j1 ? key : j1 - 1);
    pkv_u32x4 qb[4];
    att_load_q(a, row, qb);
    att_step_mfma<true, true>(a.segs.k + slab, a.segs.v + slab, mine, 0, j0, j1, qb, a.scale_log2e, m_run, l_part, o);
  }
  l_part = pkv_pair_add<32>(pkv_pair_add<16>(l_part));
  if (!mixed) {
    if (a.sel_wgs == 1) {
      att_merge_waves(a.group, m_run, l_part, o, att_slot_ml(a, row, split, 0), 2 * kSelSlots, att_slot_o(a, row, split, 0), 128);
    } else {
      float *part = a.ws + ((int64_t)row * a.n_splits + split) * a.group * kPartStride;
      att_merge_waves(a.group, m_run, l_part, o, part, kPartStride, part + 2, kPartStride);
    }
  } else if (has) {
    const int slot = att_block_slot(a, block);
    if (lane < a.group) *(float2 *)att_slot_ml(a, row, slot, n) = float2{m_run, l_part};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int head = 4 * j + i;
      if (head < a.group) {
        float *dst = att_slot_o(a, row, slot, head) + 8 * n;
        *(float4 *)dst = float4{o[0][i], o[1][i], o[2][i], o[3][i]};
        *(float4 *)(dst + 4) = float4{o[4][i], o[5][i], o[6][i], o[7][i]};
      }
    }
  }
}

constexpr int kSelThreadsAtt = 1024;  // threads of the selecting workgroup
constexpr int kSelWaves = kSelThreadsAtt / PKV_WAVE;

// What a merging workgroup needs beside its own keys, as requested.  The last waves merge (two to a head, the first head's the
// last), the first ones take blocks: lane s of a merging wave the maximum and sum in slot s, its thread the outputs at its dim.
struct AttSelRequests {
  float2 ml;
  float o[kSelSplits + 8];
};

__device__ __forceinline__ void att_request(const PkvSplitAttn &a, int row, AttSelRequests &p) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PKV_WAVE), g = (kSelWaves - 1 - wave) >> 1, lane = pkv_lane();
  p.ml = float2{kNegBig, 0.f};
#pragma unroll
  for (int s = 0; s < kSelSplits + 8; ++s) p.o[s] = 0.f;
  if (g >= a.group) return;
  if (lane < kSelSlots && ((a.slots >> (lane & 31)) & 1u)) p.ml = *(const float2 *)(att_slot_ml(a, row, 0, g) + 2 * lane);
  const float *base = att_slot_o(a, row, 0, g);
  const uint32_t d = threadIdx.x & 127;
#pragma unroll
  for (int s = 0; s < kSelSplits + 8; ++s)
    if ((a.slots >> s) & 1u) p.o[s] = (base + (uint32_t)(s * a.group * 128))[d];
}

__device__ __forceinline__ float att_lane(float x, int lane) {
  return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(x), lane));
}

// LDS of the selecting workgroups: the blocks of the splits that hold selected keys, the first of these splits first.
struct alignas(16) AttSelSmem {  // read and written by 128 bits
  float m[8][16], l[8][16], o[kSelSplits][8][128 + 4];
};
static_assert(offsetof(AttSelSmem, l) % 16 == 0 && offsetof(AttSelSmem, o) % 16 == 0 && (128 + 4) * sizeof(float) % 16 == 0, "128-bit rows");

// Clears (max, sum) of the blocks; a barrier lies between this and att_selected.
__device__ __forceinline__ void att_clear(AttSelSmem &sm) {
  if (threadIdx.x < 128) (&sm.m[0][0])[threadIdx.x] = kNegBig, (&sm.l[0][0])[threadIdx.x] = 0.f;
}

// The attention over the blocks with selected keys: ids s_sel[0 .. k) of row `row`, in LDS, made visible by the caller.  All 1024
// threads, a block to a wave.  MERGE: all of them, merged with what the first launch left, into the output; else splits
// wg * splits_per_wg .. of those with selected keys, each merged into a partial result of its own.  Bound by the instructions of
// the waves on the one CU (each costs 16 cycles where all 16 waves run it) and one round trip to memory.
template <bool MERGE>
__device__ __forceinline__ void att_selected(const PkvSplitAttn &a, int row, const uint32_t *s_sel, int wg, AttSelSmem &sm,
                                             const AttSelRequests &req) {
  PKV_ATT_CONTRACT
  const int tid = threadIdx.x, lane = tid & (PKV_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(tid / PKV_WAVE);
  const int split0 = a.blk_lo / 4 + (MERGE ? 0 : wg * a.splits_per_wg), splits = MERGE ? a.blk_hi / 4 - split0 + 1 : a.splits_per_wg;
  const int block = MERGE ? a.blk_lo + wave : 4 * split0 + wave, local = block - 4 * split0;
  const uint32_t j0 = 32u * (uint32_t)block, j1 = j0 + 32u < a.total ? j0 + 32u : a.total;
  if ((MERGE ? block <= a.blk_hi : local < 4 * splits && block / 4 <= a.blk_hi / 4) && j0 < a.total) {
    const int n = lane & 15, j = lane >> 4, b = row / a.n_kv_heads, h = row % a.n_kv_heads;
    const int64_t slab = (int64_t)b * a.segs.stride_b + (int64_t)h * a.segs.stride_h;
    uint32_t key = j0 + (uint32_t)(lane & 31);
    key = key < j1 ? key : j1 - 1;
    AttPlace<true> mine = att_place<false, 256>(a.segs, row, b, h, key);
    if (key >= a.segs.idx_lo && key < a.segs.idx_hi) {
      const uint32_t id = s_sel[key - a.segs.idx_lo], limit = (uint32_t)a.segs.idx_limit;
      mine.off = (a.segs.idx_row0 + (id < limit ? id : limit - 1)) * 256u;
    }
    pkv_u32x4 qb[4];
    att_load_q(a, row, qb);
    float m_run = kNegBig, l_part = 0.f;
    pkv_f32x4 o[8];
    att_step_mfma<true, true>(a.segs.k + slab, a.segs.v + slab, mine, 0, j0, j1, qb, a.scale_log2e, m_run, l_part, o);
    l_part = pkv_pair_add<32>(pkv_pair_add<16>(l_part));
    if (lane < a.group) sm.m[n][local] = m_run, sm.l[n][local] = l_part;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int head = 4 * j + i;
      if (head < a.group) {
        *(float4 *)&sm.o[local][head][8 * n] = float4{o[0][i], o[1][i], o[2][i], o[3][i]};
        *(float4 *)&sm.o[local][head][8 * n + 4] = float4{o[4][i], o[5][i], o[6][i], o[7][i]};
      }
    }
  }
  const int g = (kSelWaves - 1 - wave) >> 1, d = tid & 127;
  if (MERGE && g < a.group) {  // the other blocks of these splits
    const int slot = lane - kSelSplits;
    if (slot >= 0 && slot < 8 && ((a.slots >> lane) & 1u) && (tid & 64)) {
      const int at = slot < 4 ? slot : 4 * (splits - 1) + slot - 4;
      sm.m[g][at] = req.ml.x, sm.l[g][at] = req.ml.y;
    }
#pragma unroll
    for (int t = 0; t < 8; ++t)
      if ((a.slots >> (kSelSplits + t)) & 1u) sm.o[t < 4 ? t : 4 * (splits - 1) + t - 4][g][d] = req.o[kSelSplits + t];
  }
  __syncthreads();
  if constexpr (!MERGE) {
    for (int e = tid; e < splits * a.group * 128; e += kSelThreadsAtt) {
      const int sub = (e >> 7) / a.group, gg = (e >> 7) % a.group, dd = e & 127, w0 = 4 * sub, split = split0 + sub;
      if (split > a.blk_hi / 4) break;
      float mn = sm.m[gg][w0];
#pragma unroll
      for (int w = 1; w < 4; ++w) mn = fmaxf(mn, sm.m[gg][w0 + w]);
      float ls = 0.f, os = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float c = exp2f(sm.m[gg][w0 + w] - mn);
        ls = fmaf(sm.l[gg][w0 + w], c, ls);
        if (32u * (uint32_t)(4 * split + w) < a.total) os = fmaf(sm.o[w0 + w][gg][dd], c, os);
      }
      float *part = a.ws + (((int64_t)row * a.n_splits + split) * a.group + gg) * kPartStride;
      part[2 + dd] = os;
      if (dd == 0) part[0] = mn, part[1] = ls;
    }
  } else {
    if (g >= a.group) return;
    // lane = split: its maximum and sum; cw: the weights of the blocks of a split that holds selected keys
    const bool own = lane >= split0 && lane < split0 + splits;
    const float4 mw = *(const float4 *)&sm.m[g][own ? 4 * (lane - split0) : 0], lw = *(const float4 *)&sm.l[g][own ? 4 * (lane - split0) : 0];
    const float mx = fmaxf(fmaxf(mw.x, mw.y), fmaxf(mw.z, mw.w));
    const float cw[4] = {exp2f(mw.x - mx), exp2f(mw.y - mx), exp2f(mw.z - mx), exp2f(mw.w - mx)};
    // in the order of the one-piece merge, which the compiler may otherwise turn round (a b + c d has two fused forms)
    const float ls = fmaf(lw.w, cw[3], fmaf(lw.z, cw[2], fmaf(lw.y, cw[1], lw.x * cw[0])));
    const bool split_lane = lane < kSelSplits;  // the lanes behind hold single blocks
    const float mi = own ? mx : split_lane ? req.ml.x : kNegBig, li = own ? ls : split_lane ? req.ml.y : 0.f;
    const float c = exp2f(mi - pkv_wave_max(mi));
    const float two = fmaf(li, c, pkv_lane_xor_f<1>(li * c));  // the order, and the fused first step, of the merge kernel
    const float tot = pkv_pair_add<32>(pkv_pair_add<16>(pkv_pair_add<8>(pkv_pair_add<4>(pkv_pair_add<2>(two)))));
    const float weight = c / tot;
    float os = 0.f;
#pragma unroll
    for (int s = 0; s < kSelSplits; ++s) {
      if (s < a.n_splits) {  // the same in the whole workgroup, as the next
        float x = req.o[s];
        if (s >= split0 && s < split0 + splits) {
          x = 0.f;
#pragma unroll
          for (int w = 0; w < 4; ++w)
            if (32u * (uint32_t)(4 * s + w) < a.total) x = fmaf(sm.o[4 * (s - split0) + w][g][d], att_lane(cw[w], s), x);
        }
        os = fmaf(x, att_lane(weight, s), os);
      }
    }
    ((uint16_t *)a.out)[((int64_t)row * a.group + g) * 128 + d] = pkv_f32_to_bf16_bits(os);
  }
}

// The merge of a row's splits (where sel_wgs > 1).
PKV_INTERNAL int pkv_launch_attn_merge(const PkvSplitAttn &a, int rows, hipStream_t s);
// Whether pkv_decode_step's attention over `attn` can be taken in two parts around a top-k of k ids into out_ids, the retrieval
// working in `ws`; fills `out`.
PKV_INTERNAL bool pkv_plan_split_attention(const pkv_retrieve_args *r, const void *ws, const pkv_attn_args *attn, PkvSplitAttn *out);

#endif  // __HIPCC__
