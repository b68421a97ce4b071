// Collision vote: cnt[key] = sum over the 16 subspaces of lut[subspace][code].
//
// Reference: cache_hub/collision_fused/collision.cu:163-229
// (update_cache_cnt_kernel: 16 byte loads at stride kv_len and 6 LDS bit tests
// per subspace).  Here the six tier bitsets are one 4 KB byte table per row held
// in LDS, a key's 16 codes are one 128-bit load (key-major storage), and the
// same pass also builds the per-chunk histogram that the candidate select needs,
// so the counts are never re-read to find the threshold.
//
// HBM-bound: 16 B read + 1 B written per key.
#include "pkv_common.h"
#include "pkv_attn.h"

namespace {

constexpr int kScanThreads = 256;
constexpr int kHistCopies = 16;  // replicated LDS histogram: copy = lane & 15

__device__ __forceinline__ int lut_sum16(const uint8_t *__restrict__ l8, pkv_u32x4 v) {
  int c = 0;
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int d = 0; d < 4; ++d) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t code = (w[d] >> (8 * k)) & 0xffu;
      c += l8[(4 * d + k) * 256 + code];
    }
  }
  return c;
}

__device__ __forceinline__ void load_lut(uint32_t *s_lut, const uint8_t *__restrict__ lut, int row) {
  // 4 KB = one 128-bit load per thread
  const pkv_u32x4 *g = (const pkv_u32x4 *)(lut + (int64_t)row * 4096);
  ((pkv_u32x4 *)s_lut)[threadIdx.x] = g[threadIdx.x];
}

// The row's vote table from a ranking that the caller supplies, built by each workgroup of the row for itself: one wave takes four
// subspaces, a lane four ranks of each.  s_max: 16 x 256 words.  Contains barriers, the last one behind the table's last word.
struct ScanRanking {
  const int64_t *ids;
  int64_t si_b, si_h, si_sub;
  const int32_t *cc;
  int64_t cc_b, cc_h, cc_sub;
  PkvTiers tiers;
};
__device__ __forceinline__ void lut_from_ranking(const ScanRanking &r, int b, int h, uint32_t *s_max, uint32_t *s_lut) {
  const int tid = threadIdx.x, lane = pkv_lane(), sub0 = 4 * (tid / PKV_WAVE);
  const int64_t *ids = r.ids + (int64_t)b * r.si_b + (int64_t)h * r.si_h + (int64_t)sub0 * r.si_sub + 4 * lane;
  const int32_t *cc = r.cc + (int64_t)b * r.cc_b + (int64_t)h * r.cc_h + (int64_t)sub0 * r.cc_sub;
  int id[4][4], n[4][4];
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int e = 0; e < 4; ++e) id[s][e] = (int)ids[s * r.si_sub + e] & 255;
  for (int i = tid; i < 1024; i += kScanThreads) ((pkv_u32x4 *)s_max)[i] = pkv_u32x4{0u, 0u, 0u, 0u};
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int e = 0; e < 4; ++e) n[s][e] = cc[s * r.cc_sub + id[s][e]];
  __syncthreads();
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int mine = n[s][0] + n[s][1] + n[s][2] + n[s][3];
    int before = pkv_wave_incl_scan(mine) - mine;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t votes = 0;
#pragma unroll
      for (int t = 0; t < PKV_MAX_TIERS; ++t) votes += t < r.tiers.n && (uint32_t)before < r.tiers.t[t] ? 1u : 0u;
      if (votes) atomicMax(&s_max[(sub0 + s) * 256 + id[s][e]], votes);  // an id named twice keeps its best rank
      before += n[s][e];
    }
  }
  __syncthreads();
  pkv_u32x4 packed;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const pkv_u32x4 v = ((const pkv_u32x4 *)s_max)[4 * tid + d];
    packed[d] = v.x | v.y << 8 | v.z << 16 | v.w << 24;
  }
  ((pkv_u32x4 *)s_lut)[tid] = packed;
  __syncthreads();
}

// KPT * 256 whole keys from key k0 on, in the form the retrieval runs (one-byte counts out, histogram kept): every
// load of the thread is issued before the first table lookup, and nothing in between is conditional, so the waits
// of the in-order memory counter name exact counts and the lookups of one key run while the codes of the others are
// still on their way.  Four keys per thread in flight, as in the general loop: with 8 or 16 the launch is slower at
// a full grid (config 3: 36.8 us per step with 4, 38.0 with 8, 40.1 with 16; 37.2 with the general loop), faster
// only where the grid leaves most of the chip idle.
template <int KPT>
__device__ __forceinline__ void scan_whole_keys(const pkv_u32x4 *__restrict__ base, int64_t k0, const uint8_t *l8,
                                                uint8_t *__restrict__ out8, uint32_t *s_hist, int copy) {
  const int64_t i0 = k0 + threadIdx.x;
  pkv_u32x4 v[KPT];
#pragma unroll
  for (int u = 0; u < KPT; ++u) v[u] = __builtin_nontemporal_load(base + i0 + u * kScanThreads);
#pragma unroll
  for (int u = 0; u < KPT; ++u) {
    const int c = lut_sum16(l8, v[u]);
    out8[i0 + u * kScanThreads] = (uint8_t)c;
    atomicAdd(&s_hist[c * kHistCopies + copy], 1u);
  }
}

// Key-major codes ([key][16] bytes, 16-byte aligned).  grid (n_chunks, R).
// sub_blocks = 1: workgroup c scans keys [c * chunk_keys, +chunk_keys) and leaves one suffix histogram.
// sub_blocks = S > 1: the chunk is S pieces of chunk_keys / S keys spread over the row, workgroup c scans pieces
// c, c + n_chunks, c + 2 n_chunks, ... (numbered in key order) and leaves one suffix histogram per piece, in the
// bin-major table chunk_suf[row][bin][chunk][piece of the chunk] (S = 4): the candidate select that follows works on the same pieces, so that where candidates
// bunch along the row (keys whose mean drifts) every workgroup gets a share of the crowded and of the sparse parts.
__device__ __forceinline__ void scan_keymajor(
    const uint8_t *__restrict__ codes, int64_t cs_b, int64_t cs_h, int n_kv_heads, int64_t n_keys,
    const uint8_t *__restrict__ lut, uint8_t *__restrict__ cnt_u8, int64_t cnt_u8_stride,
    int32_t *__restrict__ cnt_i32, uint32_t *__restrict__ row_suf, uint16_t *__restrict__ chunk_suf, int chunk_keys,
    int sub_blocks, int n_chunks) {
  const int row = blockIdx.y;
  // Workgroups go to the eight dies in turn.  Rows start at another chunk each, so that the chunks that hold most of the
  // candidates (the ones near the queries, the same in every row) do not all meet on one die: 64 rows x 16 chunks, two layers,
  // 115.8 -> 114.6 us with the select + rerank doing the same.
  const int chunk = (int)((blockIdx.x + blockIdx.y) % (uint32_t)n_chunks);
  const int b = row / n_kv_heads, h = row % n_kv_heads;
  const int tid = threadIdx.x;

  __shared__ __attribute__((aligned(16))) uint32_t s_lut[1024];
  __shared__ uint32_t s_hist[128 * kHistCopies];  // also reused for the compacted histogram
  load_lut(s_lut, lut, row);
  for (int i = tid; i < 128 * kHistCopies; i += kScanThreads) s_hist[i] = 0;
  __syncthreads();
  const uint8_t *l8 = (const uint8_t *)s_lut;
  const int copy = tid & (kHistCopies - 1);

  const pkv_u32x4 *base = (const pkv_u32x4 *)(codes + (int64_t)b * cs_b + (int64_t)h * cs_h);
  uint8_t *out8 = cnt_u8 ? cnt_u8 + (int64_t)row * cnt_u8_stride : nullptr;
  int32_t *out32 = cnt_i32 ? cnt_i32 + (int64_t)row * n_keys : nullptr;
  const int piece_keys = chunk_keys / sub_blocks;
  uint64_t piece_bins = 0;  // sub_blocks == 4: this thread's bin of the four pieces' suffix histograms, 16 bits each
  uint32_t bin_total = 0;

  for (int j = 0; j < sub_blocks; ++j) {
    const int64_t piece = (int64_t)chunk + (int64_t)j * n_chunks;
    const int64_t k0 = piece * piece_keys < n_keys ? piece * piece_keys : n_keys;
    const int64_t k1 = (k0 + piece_keys < n_keys) ? k0 + piece_keys : n_keys;
    int64_t kc = k0;
    if (out8 && !out32 && chunk_suf) {  // uniform: the retrieval's form; whole runs of 1024, then 512 and 256 keys first
      for (; kc + 4 * kScanThreads <= k1; kc += 4 * kScanThreads) scan_whole_keys<4>(base, kc, l8, out8, s_hist, copy);
      if (kc + 2 * kScanThreads <= k1) scan_whole_keys<2>(base, kc, l8, out8, s_hist, copy), kc += 2 * kScanThreads;
      if (kc + kScanThreads <= k1) scan_whole_keys<1>(base, kc, l8, out8, s_hist, copy), kc += kScanThreads;
    }
    for (int64_t i0 = kc + tid; i0 < k1; i0 += 4 * kScanThreads) {
      pkv_u32x4 v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t i = i0 + u * kScanThreads;
        v[u] = (i < k1) ? __builtin_nontemporal_load(base + i) : pkv_u32x4{0u, 0u, 0u, 0u};
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t i = i0 + u * kScanThreads;
        if (i < k1) {
          const int c = lut_sum16(l8, v[u]);
          if (out8) out8[i] = (uint8_t)c;
          if (out32) out32[i] = c;
          if (chunk_suf) atomicAdd(&s_hist[c * kHistCopies + copy], 1u);
        }
      }
    }
    if (chunk_suf) {
      __syncthreads();
      uint32_t sum = 0;
      if (tid < 128) {
#pragma unroll
        for (int c = 0; c < kHistCopies; ++c) sum += s_hist[tid * kHistCopies + c];
      }
      __syncthreads();
      if (tid < 128) s_hist[tid] = sum;  // compacted histogram in the first 128 words
      __syncthreads();
      if (sub_blocks == 1) {
        pkv_store_suffix_hist(s_hist, &s_hist[128], row_suf + (int64_t)row * 128,
                              chunk_suf + ((int64_t)row * n_chunks + chunk) * 128);
      } else {
        // suffix sums of this piece; thread t owns bin 127 - t and keeps its pieces' values until the last one
        int incl = 0;
        if (tid < 128) {
          incl = pkv_wave_incl_scan((int)s_hist[127 - tid]);
          if (tid == PKV_WAVE - 1) s_hist[128] = (uint32_t)incl;
        }
        __syncthreads();
        if (tid < 128) {
          if (tid >= PKV_WAVE) incl += (int)s_hist[128];
          piece_bins |= (uint64_t)(uint32_t)incl << (16 * j);
          bin_total += (uint32_t)incl;
        }
      }
      if (j + 1 < sub_blocks) {  // the next piece starts from an empty histogram
        __syncthreads();
        for (int i = tid; i < 128 * kHistCopies; i += kScanThreads) s_hist[i] = 0;
        __syncthreads();
      }
    }
  }
  // several pieces: the bin-major table [row][bin][chunk][piece of the chunk] takes the chunk's four values of a bin
  // as one 8-byte store, and the row totals one addition per bin
  if (chunk_suf && sub_blocks > 1 && tid < 128) {
    uint16_t *dst = chunk_suf + ((int64_t)row * 128 + (127 - tid)) * n_chunks * sub_blocks + (int64_t)chunk * sub_blocks;
    *(uint64_t *)dst = piece_bins;
    if (bin_total) atomicAdd(&row_suf[(int64_t)row * 128 + 127 - tid], bin_total);
  }
}

__global__ __launch_bounds__(kScanThreads) void pkv_scan_keymajor_kernel(
    const uint8_t *__restrict__ codes, int64_t cs_b, int64_t cs_h, int n_kv_heads, int64_t n_keys,
    const uint8_t *__restrict__ lut, uint8_t *__restrict__ cnt_u8, int64_t cnt_u8_stride,
    int32_t *__restrict__ cnt_i32, uint32_t *__restrict__ row_suf, uint16_t *__restrict__ chunk_suf, int chunk_keys,
    int sub_blocks) {
  scan_keymajor(codes, cs_b, cs_h, n_kv_heads, n_keys, lut, cnt_u8, cnt_u8_stride, cnt_i32, row_suf, chunk_suf, chunk_keys, sub_blocks,
                (int)gridDim.x);
}

// The retrieval's form beside the part of the step's attention that waits for nothing (workgroups n_chunks and up of a row, see
// PkvSplitAttn): for steps whose query side was another kernel's work, so that there is no launch of it to ride with.  A model's 16
// tokens over four layers, 16 rows x 12000 keys, top 100: 10.97 -> 10.55 ms (top-k 5.1 + attention 5.7 + merge 2.6 us a layer before).
__global__ __launch_bounds__(kScanThreads, 4) void pkv_scan_attend_kernel(
    const uint8_t *__restrict__ codes, int64_t cs_b, int64_t cs_h, int n_kv_heads, int64_t n_keys,
    const uint8_t *__restrict__ lut, uint8_t *__restrict__ cnt_u8, int64_t cnt_u8_stride, uint32_t *__restrict__ row_suf,
    uint16_t *__restrict__ chunk_suf, int chunk_keys, int sub_blocks, int n_chunks, PkvSplitAttn attn) {
  if ((int)blockIdx.x >= n_chunks) {
    att_dense_part(attn, (int)blockIdx.x - n_chunks, blockIdx.y);
    return;
  }
  scan_keymajor(codes, cs_b, cs_h, n_kv_heads, n_keys, lut, cnt_u8, cnt_u8_stride, nullptr, row_suf, chunk_suf, chunk_keys, sub_blocks,
                n_chunks);
}

// Any byte strides.  RUNS: a subspace's codes lie side by side (cs_key = 1, the reference's subspace-major [16][kv_len]
// tensor): a thread takes four keys, sixteen 4-byte loads in flight, at any alignment (rows of odd length).  Bound by the
// latency of that one round trip at the sizes such a call has: 16 rows x 20011 keys 4.4 us; 6.9 us with one key and sixteen
// byte loads per thread and pass.
// RANKED: from a caller's ranking, counts only; the table is built here instead of by a launch before this one.
template <bool RUNS, bool RANKED>
__global__ __launch_bounds__(kScanThreads) void pkv_scan_strided_kernel(
    const uint8_t *__restrict__ codes, int64_t cs_b, int64_t cs_h, int64_t cs_key, int64_t cs_sub, int n_kv_heads,
    int64_t n_keys, const uint8_t *__restrict__ lut, uint8_t *__restrict__ cnt_u8, int64_t cnt_u8_stride,
    int32_t *__restrict__ cnt_i32, uint32_t *__restrict__ row_suf, uint16_t *__restrict__ chunk_suf, int chunk_keys,
    ScanRanking ranking) {
  const int row = blockIdx.y;
  const int chunk = blockIdx.x;
  const int b = row / n_kv_heads, h = row % n_kv_heads;
  const int tid = threadIdx.x;

  __shared__ __attribute__((aligned(16))) uint32_t s_lut[1024];
  __shared__ __attribute__((aligned(16))) uint32_t s_hist[RANKED ? 4096 : 128 * kHistCopies];  // also reused for the compacted histogram
  if (RANKED) {
    lut_from_ranking(ranking, b, h, s_hist, s_lut);
    chunk_suf = nullptr;
  } else {
    load_lut(s_lut, lut, row);
    if (chunk_suf)
      for (int i = tid; i < 128 * kHistCopies; i += kScanThreads) s_hist[i] = 0;
    __syncthreads();
  }
  const uint8_t *l8 = (const uint8_t *)s_lut;
  const int copy = tid & (kHistCopies - 1);

  const uint8_t *base = codes + (int64_t)b * cs_b + (int64_t)h * cs_h;
  const int64_t k0 = (int64_t)chunk * chunk_keys;
  const int64_t k1 = (k0 + chunk_keys < n_keys) ? k0 + chunk_keys : n_keys;
  uint8_t *out8 = cnt_u8 ? cnt_u8 + (int64_t)row * cnt_u8_stride : nullptr;
  int32_t *out32 = cnt_i32 ? cnt_i32 + (int64_t)row * n_keys : nullptr;

  int64_t rest = k0;
  if (RUNS) {
    rest = k0 + (k1 - k0) / 4 * 4;
    for (int64_t i = k0 + 4 * tid; i < rest; i += 4 * kScanThreads) {
      uint32_t w[16], c[4] = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int s = 0; s < 16; ++s) __builtin_memcpy(&w[s], base + i + s * cs_sub, 4);
#pragma unroll
      for (int s = 0; s < 16; ++s)
#pragma unroll
        for (int e = 0; e < 4; ++e) c[e] += l8[s * 256 + ((w[s] >> (8 * e)) & 255u)];
      if (out8) {  // low bytes: a caller's table may hold entries that add up to more than the retrieval's 127 votes
        const uint32_t c8 = (c[0] & 255u) | (c[1] & 255u) << 8 | (c[2] & 255u) << 16 | c[3] << 24;
        __builtin_memcpy(out8 + i, &c8, 4);
      }
      if (out32) __builtin_memcpy(out32 + i, c, 16);
      if (chunk_suf)
        for (int e = 0; e < 4; ++e) atomicAdd(&s_hist[c[e] * kHistCopies + copy], 1u);
    }
  }
  for (int64_t i = rest + tid; i < k1; i += kScanThreads) {
    int c = 0;
#pragma unroll
    for (int s = 0; s < 16; ++s) c += l8[s * 256 + base[i * cs_key + s * cs_sub]];
    if (out8) out8[i] = (uint8_t)c;
    if (out32) out32[i] = c;
    if (chunk_suf) atomicAdd(&s_hist[c * kHistCopies + copy], 1u);
  }
  if (chunk_suf) {
    __syncthreads();
    uint32_t sum = 0;
    if (tid < 128) {
#pragma unroll
      for (int c = 0; c < kHistCopies; ++c) sum += s_hist[tid * kHistCopies + c];
    }
    __syncthreads();
    if (tid < 128) s_hist[tid] = sum;  // compacted histogram in the first 128 words
    __syncthreads();
    pkv_store_suffix_hist(s_hist, &s_hist[128], row_suf + (int64_t)row * 128,
                          chunk_suf + ((int64_t)row * gridDim.x + chunk) * 128);
  }
}

// Legacy int32 codebook [rows][16][n_keys]; codes outside [0,255] get no vote.
__global__ __launch_bounds__(kScanThreads) void pkv_scan_i32_codes_kernel(const int32_t *__restrict__ codebook,
                                                                          int64_t n_keys,
                                                                          const uint8_t *__restrict__ lut,
                                                                          int32_t *__restrict__ cnt) {
  const int row = blockIdx.y;
  __shared__ __attribute__((aligned(16))) uint32_t s_lut[1024];
  load_lut(s_lut, lut, row);
  __syncthreads();
  const uint8_t *l8 = (const uint8_t *)s_lut;
  const int64_t i = (int64_t)blockIdx.x * kScanThreads + threadIdx.x;
  if (i >= n_keys) return;
  const int32_t *base = codebook + (int64_t)row * 16 * n_keys;
  int c = 0;
#pragma unroll
  for (int s = 0; s < 16; ++s) {
    const int32_t code = base[(int64_t)s * n_keys + i];
    if ((uint32_t)code < 256u) c += l8[s * 256 + code];
  }
  cnt[(int64_t)row * n_keys + i] = c;
}

}  // namespace

static int launch_scan_impl(const uint8_t *codes, int64_t cs_b, int64_t cs_h, int64_t cs_key, int64_t cs_sub, int bs,
                            int n_kv_heads, int64_t n_keys, const uint8_t *lut, uint8_t *cnt_u8,
                            int64_t cnt_u8_stride, int32_t *cnt_i32, uint32_t *row_suf, uint16_t *chunk_suf,
                            int chunk_keys, hipStream_t s, hipEvent_t ev_start, hipEvent_t ev_stop, int sub_blocks = 1) {
  PKV_REQUIRE(chunk_keys >= 256 && chunk_keys % 256 == 0 && chunk_keys <= 32768,
              "chunk_keys must be a multiple of 256 in [256,32768], got %d", chunk_keys);
  const int64_t n_chunks = (n_keys + chunk_keys - 1) / chunk_keys;
  PKV_REQUIRE(n_chunks >= 1 && n_chunks <= 65535 * 16, "too many chunks (%lld)", (long long)n_chunks);
  PKV_REQUIRE(pkv_aligned(lut, 4), "lut must be 4-byte aligned");
  dim3 grid((unsigned)n_chunks, (unsigned)(bs * n_kv_heads));
  const bool keymajor = cs_sub == 1 && cs_key == 16 && pkv_aligned(codes, 16) && cs_b % 16 == 0 && cs_h % 16 == 0;
  PKV_REQUIRE((sub_blocks == 1 || (sub_blocks == 4 && keymajor && chunk_suf)) && (sub_blocks == 1 || chunk_keys % (sub_blocks * 1024) == 0),
              "a chunk of %d keys cannot be scanned as %d strided pieces", chunk_keys, sub_blocks);
  if (keymajor) {
    // the ext launch ties the two events to this dispatch's own begin/end timestamps
    hipExtLaunchKernelGGL(pkv_scan_keymajor_kernel, grid, dim3(kScanThreads), 0, s, ev_start, ev_stop, 0, codes, cs_b,
                          cs_h, n_kv_heads, n_keys, lut, cnt_u8, cnt_u8_stride, cnt_i32, row_suf, chunk_suf, chunk_keys,
                          sub_blocks);
    PKV_LAUNCH_CHECK("pkv_scan_keymajor_kernel");
  } else {
#define PKV_SCAN_STRIDED(RUNS)                                                                                           \
  hipExtLaunchKernelGGL((pkv_scan_strided_kernel<RUNS, false>), grid, dim3(kScanThreads), 0, s, ev_start, ev_stop, 0, codes, cs_b, \
                        cs_h, cs_key, cs_sub, n_kv_heads, n_keys, lut, cnt_u8, cnt_u8_stride, cnt_i32, row_suf,          \
                        chunk_suf, chunk_keys, ScanRanking())
    if (cs_key == 1) PKV_SCAN_STRIDED(true); else PKV_SCAN_STRIDED(false);
#undef PKV_SCAN_STRIDED
    PKV_LAUNCH_CHECK("pkv_scan_strided_kernel");
  }
  return PKV_OK;
}

int pkv_launch_scan(const uint8_t *codes, int64_t cs_b, int64_t cs_h, int64_t cs_key, int64_t cs_sub, int bs,
                    int n_kv_heads, int64_t n_keys, const uint8_t *lut, uint8_t *cnt_u8, int64_t cnt_u8_stride,
                    int32_t *cnt_i32, uint32_t *row_suf, uint16_t *chunk_suf, int chunk_keys, hipStream_t s, int sub_blocks) {
  return launch_scan_impl(codes, cs_b, cs_h, cs_key, cs_sub, bs, n_kv_heads, n_keys, lut, cnt_u8, cnt_u8_stride, cnt_i32,
                          row_suf, chunk_suf, chunk_keys, s, nullptr, nullptr, sub_blocks);
}

int pkv_launch_scan_attend(const uint8_t *codes, int64_t cs_b, int64_t cs_h, int bs, int n_kv_heads, int64_t n_keys, const uint8_t *lut,
                           uint8_t *cnt_u8, int64_t cnt_u8_stride, uint32_t *row_suf, uint16_t *chunk_suf, int chunk_keys,
                           int sub_blocks, const PkvSplitAttn &attn, hipStream_t s) {
  const int n_chunks = (int)((n_keys + chunk_keys - 1) / chunk_keys);
  PKV_REQUIRE(cs_b % 16 == 0 && cs_h % 16 == 0 && pkv_aligned(codes, 16) && pkv_aligned(lut, 16), "pkv_scan_attend: unaligned operands");
  hipLaunchKernelGGL(pkv_scan_attend_kernel, dim3((unsigned)(n_chunks + attn.n_dense), (unsigned)(bs * n_kv_heads)),
                     dim3(kScanThreads), 0, s, codes, cs_b, cs_h, n_kv_heads, n_keys, lut, cnt_u8, cnt_u8_stride, row_suf, chunk_suf,
                     chunk_keys, sub_blocks, n_chunks, attn);
  PKV_LAUNCH_CHECK("pkv_scan_attend_kernel");
  return PKV_OK;
}

// Votes of subspace-major codes from a caller's ranking in one launch.  Every workgroup builds its row's table, 0.6 to 1.4 us more
// than the launch before the scan took on the GPU; a call waits for the host time of its launches, 3.4 us each, while its keys are
// few.  us, GPU alone and call by itself, two launches / one: 8 rows x 3000 4.7, 15.6 / 5.4, 11.7; 16 x 20011 5.8, 15.4 / 7.0, 11.8;
// 8 x 80001 6.8, 15.7 / 8.3, 11.7; not taken: 24 x 80001 10.3, 15.6 / 13.1, 12.7; 64 x 80000 21.4, 20.9 / 23.6, 23.3.  Codes requested
// before the table is built: 16 x 20011 7.7.  A captured call has no host time to save (in a graph, 8 x 3000 5.2 / 5.7, 64 x 3000 6.3 / 8.8).
constexpr int64_t kRankedKeys = 1 << 20;
bool pkv_scan_takes_ranking(int64_t cs_key, int rows, int64_t n_keys, hipStream_t s) {
  return cs_key == 1 && rows * n_keys <= kRankedKeys && !pkv_capturing(s);
}

int pkv_launch_scan_ranked(const uint8_t *codes, int64_t cs_b, int64_t cs_h, int64_t cs_sub, int bs, int n_kv_heads, int64_t n_keys,
                           const int64_t *ids, int64_t si_b, int64_t si_h, int64_t si_sub, const int32_t *cc, int64_t cc_b,
                           int64_t cc_h, int64_t cc_sub, const PkvTiers &tiers, int32_t *cnt, hipStream_t s) {
  const int chunk_keys = pkv_pick_chunk_keys(bs * n_kv_heads, n_keys);
  const dim3 grid((unsigned)((n_keys + chunk_keys - 1) / chunk_keys), (unsigned)(bs * n_kv_heads));
  hipLaunchKernelGGL((pkv_scan_strided_kernel<true, true>), grid, dim3(kScanThreads), 0, s, codes, cs_b, cs_h, (int64_t)1, cs_sub,
                     n_kv_heads, n_keys, (const uint8_t *)nullptr, (uint8_t *)nullptr, (int64_t)0, cnt, (uint32_t *)nullptr,
                     (uint16_t *)nullptr, chunk_keys, ScanRanking{ids, si_b, si_h, si_sub, cc, cc_b, cc_h, cc_sub, tiers});
  PKV_LAUNCH_CHECK("pkv_scan_strided_kernel");
  return PKV_OK;
}

int pkv_launch_scan_i32_codes(const int32_t *codebook, int rows, int64_t n_keys, const uint8_t *lut, int32_t *cnt,
                              hipStream_t s) {
  dim3 grid((unsigned)((n_keys + kScanThreads - 1) / kScanThreads), (unsigned)rows);
  hipLaunchKernelGGL(pkv_scan_i32_codes_kernel, grid, dim3(kScanThreads), 0, s, codebook, n_keys, lut, cnt);
  PKV_LAUNCH_CHECK("pkv_scan_i32_codes_kernel");
  return PKV_OK;
}

extern "C" int pkv_scan_chunk_keys(int rows, int64_t n_keys) { return pkv_pick_chunk_keys(rows, n_keys); }

extern "C" int pkv_collision_scan(const uint8_t *codes, int64_t cs_b, int64_t cs_h, int64_t cs_key, int64_t cs_sub,
                                  int bs, int n_kv_heads, int64_t n_keys, const uint8_t *lut, uint8_t *cnt_u8,
                                  int32_t *cnt_i32, uint32_t *row_suf, uint16_t *chunk_suf, int chunk_keys,
                                  void *stream) {
  PKV_REQUIRE(codes && lut && (cnt_u8 || cnt_i32), "pkv_collision_scan: null pointer");
  PKV_REQUIRE(bs > 0 && n_kv_heads > 0 && (int64_t)bs * n_kv_heads <= 65535 && n_keys > 0 &&
                  n_keys <= PKV_MAX_KEYS_PER_ROW,
              "bad shape bs=%d kv_heads=%d n_keys=%lld", bs, n_kv_heads, (long long)n_keys);
  PKV_REQUIRE((row_suf == nullptr) == (chunk_suf == nullptr), "row_suf and chunk_suf go together");
  return pkv_launch_scan(codes, cs_b, cs_h, cs_key, cs_sub, bs, n_kv_heads, n_keys, lut, cnt_u8, n_keys, cnt_i32,
                         row_suf, chunk_suf, chunk_keys, (hipStream_t)stream);
}

extern "C" int pkv_collision_scan_timed(const uint8_t *codes, int64_t cs_b, int64_t cs_h, int64_t cs_key,
                                        int64_t cs_sub, int bs, int n_kv_heads, int64_t n_keys, const uint8_t *lut,
                                        uint8_t *cnt_u8, int64_t cnt_u8_stride, uint32_t *row_suf, uint16_t *chunk_suf,
                                        int chunk_keys, float *kernel_us, void *stream) {
  PKV_REQUIRE(codes && lut && cnt_u8 && kernel_us, "pkv_collision_scan_timed: null pointer");
  PKV_REQUIRE(bs > 0 && n_kv_heads > 0 && (int64_t)bs * n_kv_heads <= 65535 && n_keys > 0 &&
                  n_keys <= PKV_MAX_KEYS_PER_ROW && cnt_u8_stride >= n_keys,
              "bad shape bs=%d kv_heads=%d n_keys=%lld", bs, n_kv_heads, (long long)n_keys);
  hipEvent_t e0, e1;
  PKV_HIP(hipEventCreate(&e0));
  PKV_HIP(hipEventCreate(&e1));
  int rc = launch_scan_impl(codes, cs_b, cs_h, cs_key, cs_sub, bs, n_kv_heads, n_keys, lut, cnt_u8, cnt_u8_stride,
                            nullptr, row_suf, chunk_suf, chunk_keys, (hipStream_t)stream, e0, e1);
  if (rc == PKV_OK) {
    float ms = 0.f;
    hipError_t e = hipEventSynchronize(e1);
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
    if (e != hipSuccess) {
      pkv_set_error("event timing failed: %s", hipGetErrorString(e));
      rc = PKV_EHIP;
    }
    *kernel_us = ms * 1000.f;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return rc;
}
