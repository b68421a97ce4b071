// Vote table of one (row, subspace) pair: GQA group mean of the query, normalise, SRHT rotate, rank the 256 sign
// centroids, turn the ranking plus the cluster sizes into votes per centroid.
//
// Reference: cache_hub/polar_cache.py:1027-1031, 905-922, 1216-1222 and
// cache_hub/collision_fused/collision.cu:71-151 (convert_to_bits).
//
// Shared by the query-prep kernel (one workgroup per (row, subspace)) and by the fused table + scan kernel.
#pragma once

#include "pkv_common.h"

#if defined(__HIPCC__)

struct PkvLutSmem {
  float y[128];
  __attribute__((aligned(16))) uint32_t key[256];
  int id[256];
  int cc[256];
  int wave_tot[4];
};

// Exclusive prefix of the ranked cluster sizes -> tier weight, one thread per rank (256 threads).
__device__ __forceinline__ int pkv_tier_weight_from_rank(int my_count, const PkvTiers &tiers, int *s_wave_tot) {
  int total;
  int prefix = pkv_block_excl_scan<256>(my_count, s_wave_tot, total);
  int w = 0;
#pragma unroll
  for (int t = 0; t < PKV_MAX_TIERS; ++t)
    if (t < tiers.n && (uint32_t)prefix < tiers.t[t]) ++w;
  return w;
}

// Votes of one subspace from the rotated query in sm.y (all 128 dims, written and made visible by the caller:
// a barrier lies between that write and this call).  Called by all 256 threads of a workgroup; contains barriers.
//   cc_sub      cluster sizes of this (row, subspace): 256 ints in global memory
//   lut_out     256 bytes (global or LDS): votes per centroid id
//   sorted_out  int64[256] or null: centroid ids in ranked order
__device__ __forceinline__ void pkv_lut_rank_subspace(int dtype, const int32_t *__restrict__ cc_sub, const PkvTiers &tiers,
                                                      int sub, PkvLutSmem &sm, uint8_t *lut_out, int64_t *sorted_out);

// Called by all 256 threads of a workgroup (contains barriers; `sm` may be reused after the call once the
// caller has passed a barrier).  The rotation runs in the first wave only (two dims per lane, lane exchanges, no
// barriers); the 256 threads then score, rank and weigh the 256 centroids.
//   cc_sub      cluster sizes of this (row, subspace): 256 ints in global memory
//   lut_out     256 bytes (global or LDS): votes per centroid id
//   qhat_out    float[128] of the row or null; qnorm_out likewise (written when non-null)
//   sorted_out  int64[256] or null: centroid ids in ranked order
__device__ __forceinline__ void pkv_lut_build_subspace(const void *__restrict__ q, int dtype, int b, int h, int n_kv_heads,
                                                       int group, const float *__restrict__ signs,
                                                       const int32_t *__restrict__ cc_sub, const PkvTiers &tiers, int sub,
                                                       PkvLutSmem &sm, uint8_t *lut_out, float *qhat_out, float *qnorm_out,
                                                       int64_t *sorted_out) {
  const int tid = threadIdx.x;
  // cluster sizes by centroid id; issued first so that the latency overlaps the rotation
  const int my_cc = cc_sub[tid];

  if (tid < PKV_WAVE) {
    float y_lo, y_hi;
    const float n = pkv_query_mean_rotate_wave(q, dtype, b, h, n_kv_heads, group, signs, y_lo, y_hi);
    sm.y[tid] = y_lo, sm.y[tid + 64] = y_hi;
    if (qhat_out) qhat_out[tid] = y_lo, qhat_out[tid + 64] = y_hi;
    if (qnorm_out && tid == 0) *qnorm_out = n;
  }
  sm.cc[tid] = my_cc;
  __syncthreads();
  pkv_lut_rank_subspace(dtype, nullptr, tiers, sub, sm, lut_out, sorted_out);
}

__device__ __forceinline__ void pkv_lut_rank_subspace(int dtype, const int32_t *__restrict__ cc_sub, const PkvTiers &tiers,
                                                      int sub, PkvLutSmem &sm, uint8_t *lut_out, int64_t *sorted_out) {
  const int tid = threadIdx.x;
  if (cc_sub) sm.cc[tid] = cc_sub[tid];  // read again only after the barriers below

  // rank = number of centroids ahead of this one under (score desc, id asc).  The sign codebook is antipodal (score[255-c] ==
  // -score[c] exactly), hence rank[255-c] = 255 - rank[c], and of each such pair the member whose score is not negative (of two
  // zeros the smaller id) is ahead of every member that is not of its kind: its rank is the number of pairs whose own such member
  // is ahead of it, by magnitude and then id.  Threads 2c and 2c + 1 count for pair c over every other group of four pairs, 64
  // comparisons each and no exchange through LDS (128 comparisons each, against all 256 centroids: 64 rows x 65536 keys, 2 layers,
  // 101.3 / 99.9 us a step, adaptive 24 x 41003, 2 layers, 87.8 / 86.0).
  const int c = tid >> 1, half = tid & 1;
  float acc = 0.f;  // score of centroid c: sum_j (+-) qhat_sub[j], sequential j
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float v = sm.y[8 * sub + j];
    const float t = ((c >> j) & 1) ? v : -v;
    acc = (j == 0) ? t : acc + t;
  }
  const uint32_t bits = __float_as_uint(pkv_rdt(acc + 0.0f, dtype)), magnitude = bits & 0x7fffffffu;
  const int front = (bits >> 31) ? 255 - c : c;
  int ahead = 0, ahead1 = 0, ahead2 = 0, ahead3 = 0;  // four chains of dependent adds (one: +0.3 us per launch)
  if (dtype == PKV_DTYPE_BF16) {
    // bf16 magnitudes occupy 15 bits: fold the tie rule (smaller id first) into one 32-bit key
    const uint32_t mine = ((magnitude >> 16) << 8) | (uint32_t)(255 - front);
    if (!half) sm.key[c] = mine;
    __syncthreads();
    const pkv_u32x4 *k4 = (const pkv_u32x4 *)sm.key + half;
#pragma unroll 8
    for (int i = 0; i < 16; ++i) {
      const pkv_u32x4 k = k4[2 * i];
      ahead += (k.x > mine), ahead1 += (k.y > mine), ahead2 += (k.z > mine), ahead3 += (k.w > mine);
    }
  } else {
    uint64_t *s_key = (uint64_t *)sm.key;
    const uint64_t mine = ((uint64_t)magnitude << 8) | (uint64_t)(255 - front);
    if (!half) s_key[c] = mine;
    __syncthreads();
    const uint64_t *k = s_key + 2 * half;
#pragma unroll 8
    for (int i = 0; i < 32; i += 2) {
      ahead += (k[4 * i] > mine), ahead1 += (k[4 * i + 1] > mine), ahead2 += (k[4 * i + 4] > mine), ahead3 += (k[4 * i + 5] > mine);
    }
  }
  ahead += ahead1 + ahead2 + ahead3;
  ahead += (int)pkv_lane_xor<1>((uint32_t)ahead);
  sm.id[half ? 255 - ahead : ahead] = half ? 255 - front : front;
  __syncthreads();
  const int id = sm.id[tid];
  const int w = pkv_tier_weight_from_rank(sm.cc[id], tiers, sm.wave_tot);
  lut_out[id] = (uint8_t)w;
  if (sorted_out) sorted_out[tid] = id;
}

#endif  // __HIPCC__
