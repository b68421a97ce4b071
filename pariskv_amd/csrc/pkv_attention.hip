// Dense decode attention over the gathered key set: softmax(q k^T * scale) v for ONE
// query token per sequence, GQA (the G query heads of a KV head share its keys), over
// up to four row segments of head_dim 128 (sink | update buffer | gathered top-k |
// local window), non-causal.
//
// Reference: cache_hub/polar_cache.py:1084-1105 (torch.cat of the segments, then
// flash_attn_func on [bs, S, H, D]); here the segments are read where they lie.
//
// HBM-bound: 512 B (one K row + one V row, bf16) per key and KV head, read once for
// all G query heads.  Split over the key axis (flash-decoding): grid (n_splits, R);
// every split keeps a running (max, sum, output) per query head and the partial
// results are merged by a second small launch.
//   bf16: four waves per split on the matrix cores (v_mfma_f32_16x16x32_bf16), merged through LDS, see pkv_attn.h.
//   fp32: 256 threads per split, every 16 lanes own one key at a time (a wave
//         instruction moves four whole rows), fp32 FMA and lane-exchange reductions.
//
// Arithmetic: products and sums in fp32 (bf16 path: bf16 x bf16 products accumulated in
// fp32, probabilities rounded to bf16 before P.V as flash-attn does), exp2 with the scale
// folded in; the output is rounded to the input dtype.  Not bit-reproducible against another summation order -
// the tolerance of this row is 2e-2 absolute in bf16.
#include "pkv_attn.h"

// Fused multiply-add is welcome here (the rest of the library forbids it because integer results are
// derived from its float steps; this kernel's only contract is the 2e-2 tolerance).
#pragma clang fp contract(fast)

namespace {

constexpr int kAttThreads = 256;
constexpr int kAttKeysPerIter = kAttThreads / 16;  // 16 keys per workgroup step
// A call whose caller keeps counters takes one launch, the last workgroup of a row merging, up to this many splits a row and
// workgroups in all, unless it is captured: a replayed graph has no host time to save, and would count in one half of the counters for
// good.  A decode step over a short context waits for its launches' host time (3.4 us each), not for the GPU: 8 rows x
// 1500 keys, append and attention, 14.1 us a step where two launches for the attention took 16.7.  Back to back and with nothing else
// to launch, us, one / two launches: 8 rows x 300 keys 7.0 / 9.7, 1600 8.0 / 9.9, 16 rows x 1600 9.0 / 9.6, 32 x 1600 10.1 / 9.3,
// 8 x 2500 9.7 / 9.7, 4000 11.0 / 9.9; the GPU alone, without the host, 6.7 / 6.2, 7.7 / 6.5, 8.9 / 6.8, 10.2 / 8.5, 9.6 / 7.7, 11.0 / 7.7.
// In a replayed graph 8 x 300 6.8 / 6.5, 8 x 1500 7.8 / 6.9 (eight heads 10.0 / 7.8), 16 x 1600 9.0 / 7.2, 32 x 1000 8.3 / 7.2; a call whose host
// runs ahead of the GPU loses as much, and cannot be told from one that waits for its host.
// fp32 loses there as well (12 rows x 865 keys, 7 heads, 11.5 / 10.7) and keeps its two launches.
constexpr int kWholeSplits = 16, kWholeWorkgroups = 256;
constexpr int kAttUnroll = 2;                      // keys per 16-lane group per step

struct AttSegs {
  const void *k[PKV_ATTN_MAX_SEGMENTS];
  const void *v[PKV_ATTN_MAX_SEGMENTS];
  int64_t stride_b[PKV_ATTN_MAX_SEGMENTS], stride_h[PKV_ATTN_MAX_SEGMENTS];
  int64_t row0[PKV_ATTN_MAX_SEGMENTS];
  int64_t end[PKV_ATTN_MAX_SEGMENTS];  // exclusive end of the segment in the concatenated key order
  const int64_t *idx[PKV_ATTN_MAX_SEGMENTS];  // per segment: selected rows (relative to row0) or nullptr
  int64_t idx_stride[PKV_ATTN_MAX_SEGMENTS], idx_limit[PKV_ATTN_MAX_SEGMENTS];
  int n;
};

// A field of a segment as a value in scalar registers.  Without this a field picked by a lane's segment number becomes a pick among
// the fields' addresses, for which the compiler lays the whole argument out in scratch memory: 168 and 264 bytes a lane.  Keys in
// two tensors, us with that / without: 8 rows x 1600 8.1 / 6.7, 64 x 1600 21.6 / 14.5, 8 x 8000 18.2 / 13.0, fp32 32 x 1600 24.8 / 19.8.
template <typename T>
__device__ __forceinline__ T att_field(T v) {
  asm("" : "+s"(v));
  return v;
}

// Row (inside the (b, h) slab of its segment, row0 included) and segment of concatenated key jj, packed as
// row | segment << 29.  Indexed segments cost one dependent 8-byte load.
__device__ __forceinline__ uint32_t att_resolve_row(const AttSegs &segs, int row, uint32_t jj) {
  int s = 0;
  uint32_t first = 0;
#pragma unroll
  for (int t = 1; t < PKV_ATTN_MAX_SEGMENTS; ++t)
    if (t < segs.n && jj >= (uint32_t)segs.end[t - 1]) s = t, first = (uint32_t)segs.end[t - 1];
  const int64_t *ip = att_field(segs.idx[0]);
  int64_t stride = att_field(segs.idx_stride[0]), limit = att_field(segs.idx_limit[0]), row0 = att_field(segs.row0[0]);
#pragma unroll
  for (int t = 1; t < PKV_ATTN_MAX_SEGMENTS; ++t) {
    const int64_t *const ip_t = att_field(segs.idx[t]);
    const int64_t stride_t = att_field(segs.idx_stride[t]), limit_t = att_field(segs.idx_limit[t]), row0_t = att_field(segs.row0[t]);
    if (s == t) ip = ip_t, stride = stride_t, limit = limit_t, row0 = row0_t;
  }
  int64_t r = jj - first;
  if (ip) {
    r = ip[(int64_t)row * stride + r];
    r = r < 0 ? 0 : (r >= limit ? limit - 1 : r);
  }
  return (uint32_t)(r + row0) | ((uint32_t)s << 29);
}

// Keys row `row` attends to: all `total`, its own row_keys[row], or with uniform > 0 the largest of row_keys[0 .. uniform)
// (the dense form of the adaptive-k step, where a launch of its own for the maximum took 4.5 us at 24 rows).
__device__ __forceinline__ int64_t att_row_total(int64_t total, const int32_t *__restrict__ row_keys, int row, int uniform) {
  if (!row_keys) return total;
  int64_t rk;
  if (uniform > 0) {
    int m = 0;
    for (int r = pkv_lane(); r < uniform; r += PKV_WAVE) m = max(m, row_keys[r]);
#define PKV_ATT_MAX(M) { const int o = (int)pkv_lane_xor<M>((uint32_t)m); m = max(m, o); }
    PKV_ATT_MAX(1) PKV_ATT_MAX(2) PKV_ATT_MAX(4) PKV_ATT_MAX(8) PKV_ATT_MAX(16) PKV_ATT_MAX(32)
#undef PKV_ATT_MAX
    rk = __builtin_amdgcn_readfirstlane(m);
  } else {
    rk = row_keys[row];
  }
  return rk < total ? (rk > 0 ? rk : 1) : total;
}

// The addresses of key jj's K and V rows; ROW: bytes of a row.
template <bool INDEXED, uint32_t ROW>
__device__ __forceinline__ AttPlace<false> att_place(const AttSegs &a, int row, int b, int h, uint32_t jj) {
  int s = 0;
  uint32_t first = 0;
#pragma unroll
  for (int t = 1; t < PKV_ATTN_MAX_SEGMENTS; ++t)
    if (t < a.n && jj >= (uint32_t)a.end[t - 1]) s = t, first = (uint32_t)a.end[t - 1];
  const char *k = (const char *)att_field(a.k[0]), *v = (const char *)att_field(a.v[0]);
  int64_t sb = att_field(a.stride_b[0]), sh = att_field(a.stride_h[0]), row0 = att_field(a.row0[0]);
#pragma unroll
  for (int t = 1; t < PKV_ATTN_MAX_SEGMENTS; ++t) {
    const char *const k_t = (const char *)att_field(a.k[t]), *const v_t = (const char *)att_field(a.v[t]);
    const int64_t sb_t = att_field(a.stride_b[t]), sh_t = att_field(a.stride_h[t]), row0_t = att_field(a.row0[t]);
    if (s == t) k = k_t, v = v_t, sb = sb_t, sh = sh_t, row0 = row0_t;
  }
  const int64_t r = INDEXED ? (int64_t)(att_resolve_row(a, row, jj) & 0x1fffffffu) : row0 + (int64_t)(jj - first);
  const int64_t off = ((int64_t)b * sb + (int64_t)h * sh) * (ROW / 128) + r * ROW;
  return {(uint64_t)(k + off), (uint64_t)(v + off)};
}

// Eight consecutive elements as loaded.  Kept apart from their use so that a load can be issued a whole step before its data is
// touched.
struct Raw8 {
  pkv_u32x4 a, b;
};

// Queries and K and V rows.  Plain loads: two instructions share every 128-byte line of a row, and a streaming load gives the line up
// after the first.  Attention, us, streaming / plain: 12 rows x 865 keys, 7 heads, 13.0 / 11.6, by index 13.4 / 11.8; 64 x 2000
// 35.9 / 33.3, by index 39.8 / 32.3; 256 x 900 52.4 / 51.4, by index 57.1 / 52.3; 768 x 900 140.7 / 136.3.  Slower only
// where 512 or 1024 KV heads' keys are read in order: 512 x 900 91.0 / 93.2 (by index 96.4 / 93.0), 1024 x 900 183.0 / 188.9.
__device__ __forceinline__ void load_raw8(const void *base, int64_t elem_off, Raw8 &r) {
  r.a = *(const pkv_u32x4 *)((const float *)base + elem_off);
  r.b = *(const pkv_u32x4 *)((const float *)base + elem_off + 4);
}

__device__ __forceinline__ void expand8(const Raw8 &r, float (&x)[8]) {
  x[0] = __uint_as_float(r.a.x), x[1] = __uint_as_float(r.a.y), x[2] = __uint_as_float(r.a.z), x[3] = __uint_as_float(r.a.w);
  x[4] = __uint_as_float(r.b.x), x[5] = __uint_as_float(r.b.y), x[6] = __uint_as_float(r.b.z), x[7] = __uint_as_float(r.b.w);
}

__device__ __forceinline__ void load8(const void *base, int64_t elem_off, float (&x)[8]) {
  Raw8 r;
  load_raw8(base, elem_off, r);
  expand8(r, x);
}

// WHOLE launches: the splits of a row are merged, as pkv_attn_merge_kernel merges them and to the same bits, by the workgroup
// that stores its partial result last.  gridDim.x workgroups of a row come here with their partial results stored for other
// dies (att_put); *arrived is zero before the first of them and after the last.  Nobody waits: a workgroup that is not the last
// one ends.  *spare, the next launch's counter, is zero as well unless launches that share the workspace ran at once, which spoils
// their results: it is cleared here, so that it spoils no later ones.  One chain of store acknowledgement, count and dependent loads, so every load is requested before the weights are
// known; see kWholeSplits for what it costs and saves.
__device__ __forceinline__ void att_last_merges(const float *ws, int row, int group, uint32_t *arrived, uint32_t *spare, uint16_t *out) {
  constexpr int kThreads = kMfmaWaves * PKV_WAVE;
  const int tid = threadIdx.x, n_splits = gridDim.x, lane = tid & (PKV_WAVE - 1);
  __shared__ uint32_t s_before;
  __shared__ float s_w[8][PKV_WAVE];  // weight of split s for head g, already divided by the total
  if (blockIdx.x == 0 && tid == 0) __hip_atomic_store(spare, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  pkv_wait_vmem();
  __syncthreads();
  if (tid == 0) s_before = __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (s_before != (uint32_t)n_splits - 1) return;  // uniform
  if (tid == 0) __hip_atomic_store(arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const float *rowp = ws + (int64_t)row * n_splits * group * kPartStride;
  const int next = group * kPartStride;
  auto get = [](const float *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
  // a thread's (head, dim) pairs, two at a time: four heads take one turn
  for (int base = 0; base < group * 128; base += 2 * kThreads) {
    float part[2][kWholeSplits];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int e = base + u * kThreads + tid < group * 128 ? base + u * kThreads + tid : tid & 127;
      const float *po = rowp + (e >> 7) * kPartStride + 2 + (e & 127);
#pragma unroll
      for (int s = 0; s < kWholeSplits; ++s) part[u][s] = s < n_splits ? get(po + s * next) : 0.f;  // uniform
    }
    if (base == 0) {
      for (int g = tid / PKV_WAVE; g < group; g += kMfmaWaves) {  // one wave per head: lane = split
        const bool live = lane < n_splits;
        const float *p = rowp + (live ? lane : 0) * next + g * kPartStride;
        const float m0 = get(p), l0 = get(p + 1);
        const float mi = live ? m0 : kNegBig, li = live ? l0 : 0.f;
        const float c = exp2f(mi - pkv_wave_max(mi));
        const float two = fmaf(li, c, pkv_lane_xor_f<1>(li * c));
        const float tot = pkv_pair_add<32>(pkv_pair_add<16>(pkv_pair_add<8>(pkv_pair_add<4>(pkv_pair_add<2>(two)))));
        s_w[g][lane] = c / tot;
      }
      __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int e = base + u * kThreads + tid;
      if (e >= group * 128) break;
      const int g = e >> 7, d = e & 127;
      float os = 0.f;
#pragma unroll
      for (int s = 0; s < kWholeSplits; ++s) os = fmaf(part[u][s], s < n_splits ? s_w[g][s] : 0.f, os);
      out[((int64_t)row * group + g) * 128 + d] = pkv_f32_to_bf16_bits(os);
    }
  }
}

// Splits are of 64 keys while the key set allows: a launch is one chain of dependent loads with some 1000 instructions behind
// it, not bandwidth.  Places of keys as in the bf16 kernel below.  Decode step, us, with a 64-bit pointer picked out of four for
// each row / with places: 12 rows x 865 attended keys, 7 heads (2 layers) 74.6 / 70.0, 8 rows x 696 (2 layers) 66.5 / 61.0,
// 32 rows x 896 48.6 / 45.2.
//
// grid (splits, rows, query heads by G)
template <int G, bool INDEXED, typename SEGS>
__global__ __launch_bounds__(kAttThreads) void pkv_attn_partial_kernel(const void *__restrict__ q, int n_kv_heads,
                                                                       int group, SEGS segs, int64_t total,
                                                                       const int32_t *__restrict__ row_keys, int uniform,
                                                                       int64_t per_split, float scale_log2e,
                                                                       float *__restrict__ ws) {
  // blockIdx.z: query heads g0 .. g0 + g_count - 1 of the KV head (more than four would not fit the registers)
  const int g0 = blockIdx.z * G, g_count = group - g0 < G ? group - g0 : G;
  const int split = blockIdx.x, row = blockIdx.y;
  const int b = row / n_kv_heads, h = row % n_kv_heads;
  const int tid = threadIdx.x;
  const int lane16 = tid & 15;        // owns dims 8*lane16 .. +7
  const int grp = tid >> 4;           // 16 key slots per workgroup step

  total = att_row_total(total, row_keys, row, uniform);  // ragged rows
  const int64_t j0 = (int64_t)split * per_split;
  const int64_t j1 = (j0 + per_split < total) ? j0 + per_split : total;
  constexpr bool ONE = __is_same(SEGS, AttOne);
  constexpr uint32_t kRow = 512;
  const int lane = tid & (PKV_WAVE - 1), wave = tid / PKV_WAVE;
  const char *kbase = nullptr, *vbase = nullptr;
  if constexpr (ONE) {
    const int64_t slab = (int64_t)b * segs.stride_b + (int64_t)h * segs.stride_h;
    kbase = segs.k + slab, vbase = segs.v + slab;
  }
  // K/V rows of the step after the current one are requested before the current one is consumed
  float kx[kAttUnroll][8], vx[kAttUnroll][8];
  Raw8 kn[kAttUnroll], vn[kAttUnroll];
  AttPlace<ONE> mine;
  auto fetch = [&](int64_t jb, Raw8 (&kd)[kAttUnroll], Raw8 (&vd)[kAttUnroll]) {
    // four turns (64 keys) at a time: lane 4 t + i (mod 16) finds the place of the key that the wave's lanes 16 i .. 16 i + 15
    // read in turn t
    static_assert(4 % kAttUnroll == 0 && kAttKeysPerIter == 16, "a wave reads four keys in a turn");
    const int turn = ((int)(jb - j0) / kAttKeysPerIter) & 3;
    if (turn == 0) {
      const int64_t key = jb + ((lane >> 2) & 3) * kAttKeysPerIter + 4 * wave + (lane & 3);
      mine = att_place<INDEXED, kRow>(segs, row, b, h, (uint32_t)(key < j1 ? key : j1 - 1));  // fewer than 2^24 keys
    }
#pragma unroll
    for (int u = 0; u < kAttUnroll; ++u) {
      const int at = 4 * (turn + u) + (lane >> 4);
      const char *kp, *vp;
      if constexpr (ONE) {
        const uint64_t off = mine.from(at).off + (kRow / 16) * (uint32_t)lane16;
        kp = kbase + off, vp = vbase + off;
      } else {
        kp = mine.k_from(at) + (kRow / 16) * lane16, vp = mine.v_from(at) + (kRow / 16) * lane16;
      }
      load_raw8(kp, 0, kd[u]);
      load_raw8(vp, 0, vd[u]);
    }
  };
  if (j0 < j1) fetch(j0, kn, vn);  // before the queries: nothing here waits for them

  float qv[G][8];
#pragma unroll
  for (int g = 0; g < G; ++g) {  // surplus slots idle
    load8(q, ((int64_t)row * group + g0 + (g < g_count ? g : 0)) * 128 + 8 * lane16, qv[g]);
#pragma unroll
    for (int d = 0; d < 8; ++d) qv[g][d] *= scale_log2e;  // scores come out in units of log2(e)
  }
  float m[G], l[G], o[G][8];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    m[g] = kNegBig, l[g] = 0.f;
#pragma unroll
    for (int d = 0; d < 8; ++d) o[g][d] = 0.f;
  }

  for (int64_t jb = j0; jb < j1; jb += kAttKeysPerIter * kAttUnroll) {
    bool valid[kAttUnroll];
#pragma unroll
    for (int u = 0; u < kAttUnroll; ++u) {
      valid[u] = jb + u * kAttKeysPerIter + grp < j1;
      expand8(kn[u], kx[u]);
      expand8(vn[u], vx[u]);
    }
    if (jb + kAttKeysPerIter * kAttUnroll < j1) fetch(jb + kAttKeysPerIter * kAttUnroll, kn, vn);
    float s[G][kAttUnroll];
#pragma unroll
    for (int g = 0; g < G; ++g) {
#pragma unroll
      for (int u = 0; u < kAttUnroll; ++u) {
        float acc = qv[g][0] * kx[u][0];
#pragma unroll
        for (int d = 1; d < 8; ++d) acc += qv[g][d] * kx[u][d];
        acc += pkv_lane_xor_f<1>(acc);
        acc += pkv_lane_xor_f<2>(acc);
        acc += pkv_lane_xor_f<4>(acc);
        acc += pkv_lane_xor_f<8>(acc);
        s[g][u] = valid[u] ? acc : kNegBig;
      }
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float mn = m[g];
#pragma unroll
      for (int u = 0; u < kAttUnroll; ++u) mn = fmaxf(mn, s[g][u]);
      const float corr = exp2f(m[g] - mn);
      m[g] = mn;
      float p[kAttUnroll], psum = 0.f;
#pragma unroll
      for (int u = 0; u < kAttUnroll; ++u) {
        p[u] = valid[u] ? exp2f(s[g][u] - mn) : 0.f;
        psum += p[u];
      }
      l[g] = l[g] * corr + psum;
#pragma unroll
      for (int d = 0; d < 8; ++d) {
        float acc = o[g][d] * corr;
#pragma unroll
        for (int u = 0; u < kAttUnroll; ++u) acc += p[u] * vx[u][d];
        o[g][d] = acc;
      }
    }
  }

  // merge the 16 key slots of the workgroup through LDS
  __shared__ float s_m[16][G], s_l[16][G];
  __shared__ alignas(16) float s_o[16][G][128 + 4];  // written by 128 bits
#pragma unroll
  for (int g = 0; g < G; ++g) {
    if (lane16 == 0) s_m[grp][g] = m[g], s_l[grp][g] = l[g];
    *(float4 *)&s_o[grp][g][8 * lane16] = float4{o[g][0], o[g][1], o[g][2], o[g][3]};
    *(float4 *)&s_o[grp][g][8 * lane16 + 4] = float4{o[g][4], o[g][5], o[g][6], o[g][7]};
  }
  __syncthreads();
  float *part = ws + (((int64_t)row * gridDim.x + split) * group + g0) * kPartStride;
  for (int e = tid; e < g_count * 128; e += kAttThreads) {
    const int g = e >> 7, d = e & 127;
    float mn = s_m[0][g];
#pragma unroll
    for (int w = 1; w < 16; ++w) mn = fmaxf(mn, s_m[w][g]);
    float ls = 0.f, os = 0.f;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      const float c = exp2f(s_m[w][g] - mn);
      ls += s_l[w][g] * c;
      os += s_o[w][g][d] * c;
    }
    part[g * kPartStride + 2 + d] = os;
    if (d == 0) part[g * kPartStride] = mn, part[g * kPartStride + 1] = ls;
  }
}

// grid (splits, KV heads, batch).  Decode step, us, with four-way pointer selection per row / with places by lane exchange:
// 8 rows x 693 attended keys 30.2 / 27.7, 8 x 1188 (4 layers) 136.5 / 124.2, 64 x 887 (2 layers) 133.4 / 122.8.
template <bool INDEXED, typename SEGS, bool WHOLE>
__global__ __launch_bounds__(kMfmaWaves * PKV_WAVE) void pkv_attn_partial_mfma_kernel(
    const void *__restrict__ q, int group, SEGS segs, int64_t total, const int32_t *__restrict__ row_keys, int uniform,
    int64_t per_split, float scale_log2e, float *__restrict__ ws, uint32_t *arrivals, uint32_t *spares, void *out) {
  const int split = blockIdx.x, h = blockIdx.y, b = blockIdx.z, row = b * (int)gridDim.y + h;
  constexpr bool ONE = __is_same(SEGS, AttOne);
  const int lane = threadIdx.x & (PKV_WAVE - 1), wave = threadIdx.x / PKV_WAVE;
  const int n = lane & 15, j = lane >> 4;
  total = att_row_total(total, row_keys, row, uniform);
  const int64_t per_wave = per_split / kMfmaWaves;  // a multiple of the 32 keys of one step
  const int64_t j0 = (int64_t)split * per_split + (int64_t)wave * per_wave;
  const int64_t j1 = (j0 + per_wave < total) ? j0 + per_wave : total;  // j1 <= j0: nothing left for this wave

  // Lane l holds the place of key blk0 + l of the current block of 64 keys (two steps; keys past j1 repeat the last one);
  // the lanes that read a row get it from there, so that a place is found once per key and wave.
  AttPlace<ONE> mine;
  const char *kbase = nullptr, *vbase = nullptr;
  if constexpr (ONE) {
    const int64_t slab = (int64_t)b * segs.stride_b + (int64_t)h * segs.stride_h;
    kbase = segs.k + slab, vbase = segs.v + slab;
  }
  auto place_block = [&](int64_t jb) {
    const int64_t key = jb + lane;
    mine = att_place<INDEXED, 256>(segs, row, b, h, (uint32_t)(key < j1 ? key : j1 - 1));
  };
  if (j0 < j1) place_block(j0);  // before the queries: the indices' latency is the longer one

  const pkv_u32x4 zero4 = {0u, 0u, 0u, 0u};
  pkv_u32x4 qb[4];
#pragma unroll
  for (int c = 0; c < 4; ++c)
    qb[c] = n < group ? *(const pkv_u32x4 *)((const uint16_t *)q + ((int64_t)row * group + n) * 128 + 32 * c + 8 * j) : zero4;

  float m_run = kNegBig, l_part = 0.f;
  pkv_f32x4 o[8];
#pragma unroll
  for (int m = 0; m < 8; ++m) o[m] = pkv_f32x4{0.f, 0.f, 0.f, 0.f};

  if (j0 < j1) att_step_mfma<ONE, true>(kbase, vbase, mine, 0, j0, j1, qb, scale_log2e, m_run, l_part, o);
  for (int64_t jb = j0 + kMfmaStepKeys; jb < j1; jb += kMfmaStepKeys) {
    const int in_block = (int)(jb - j0) & (PKV_WAVE - 1);
    if (in_block == 0) place_block(jb);
    att_step_mfma<ONE, false>(kbase, vbase, mine, in_block, jb, j1, qb, scale_log2e, m_run, l_part, o);
  }

  l_part = pkv_pair_add<32>(pkv_pair_add<16>(l_part));
  float *part = ws + ((int64_t)row * gridDim.x + split) * group * kPartStride;
  att_merge_waves<WHOLE>(group, m_run, l_part, o, part, kPartStride, part + 2, kPartStride);
  if (WHOLE) att_last_merges(ws, row, group, arrivals + row, spares + row, (uint16_t *)out);
}

// grid R, G*128 threads: merge the splits (at most 64) and normalise.
template <bool BF16>
__global__ void pkv_attn_merge_kernel(const float *__restrict__ ws, int n_splits, int G, void *__restrict__ out) {
  const int row = blockIdx.x;
  const int tid = threadIdx.x;
  const int g = tid >> 7, d = tid & 127;
  __shared__ float s_w[8][64];   // weight of split s for head g, already divided by the total
  const float *rowp = ws + (int64_t)row * n_splits * G * kPartStride;
  // the first 16 splits' partial outputs are requested before the weights are known: one memory round trip
  // instead of two for the usual case (a few thousand keys)
  constexpr int kEarly = 16;
  const float *po = rowp + (int64_t)g * kPartStride + 2 + d;
  float early[kEarly];
#pragma unroll
  for (int s = 0; s < kEarly; ++s) early[s] = s < n_splits ? po[(int64_t)s * G * kPartStride] : 0.f;
  if (d < PKV_WAVE) {  // one wave per head: lane = split
    const bool live = d < n_splits;
    const float *p = rowp + ((int64_t)(live ? d : 0) * G + g) * kPartStride;
    const float mi = live ? p[0] : kNegBig, li = live ? p[1] : 0.f;
    const float c = exp2f(mi - pkv_wave_max(mi));
    const float two = fmaf(li, c, pkv_lane_xor_f<1>(li * c));
    const float tot = pkv_pair_add<32>(pkv_pair_add<16>(pkv_pair_add<8>(pkv_pair_add<4>(pkv_pair_add<2>(two)))));
    s_w[g][d] = c / tot;
  }
  __syncthreads();
  float os = 0.f;
#pragma unroll
  for (int s = 0; s < kEarly; ++s) os = fmaf(early[s], s < n_splits ? s_w[g][s] : 0.f, os);
#pragma unroll 8
  for (int s = kEarly; s < n_splits; ++s) os = fmaf(po[(int64_t)s * G * kPartStride], s_w[g][s], os);
  const int64_t oi = ((int64_t)row * G + g) * 128 + d;
  if (BF16)
    ((uint16_t *)out)[oi] = pkv_f32_to_bf16_bits(os);
  else
    ((float *)out)[oi] = os;
}

// rows: times the workgroups that a KV head's query heads take (two for five to eight heads).
int pick_splits(int rows, int64_t total) {
  // One round of workgroups: with four query heads the kernel holds 3 workgroups per CU (768 on the chip); more would run as
  // a second round.  us with the second four heads' workgroups left out of this count / with them, 8 heads:
  // 32 rows x 1600 keys 31.7 / 26.6, 64 x 800 30.8 / 26.6, 256 x 800 80.8 / 75.2, 24 x 1600 22.5 / 22.4, 8 x 6000 27.7 / 25.6.
  int64_t s = 768 / rows;
  const int64_t max_by_len = (total + 63) / 64;  // at least 64 keys per split
  if (s > max_by_len) s = max_by_len;
  if (s > 64) s = 64;
  if (s < 1) s = 1;
  return (int)s;
}

// Matrix-core path: four waves per workgroup, one 32-key step per wave while that keeps the split count within
// the 64 the merge kernel takes (every load of the workgroup is then in flight at once); longer key sets give
// each wave more steps.
int pick_splits_mfma(int rows, int64_t total) {
  (void)rows;
  int64_t s = (total + kMfmaWaves * kMfmaStepKeys - 1) / (kMfmaWaves * kMfmaStepKeys);
  if (s > 64) s = 64;
  if (s < 1) s = 1;
  return (int)s;
}

// The segments as offsets into one (b, h) slab: false where they lie in different tensors, more than one is indexed or a
// row's byte offset would not fit 32 bits (2^24 rows of 256 bytes, 2^23 of 512).
bool as_one_tensor(const AttSegs &sg, int es, AttOne &one) {
  memset(&one, 0, sizeof one);
  one.k = (const char *)sg.k[0], one.v = (const char *)sg.v[0];
  one.stride_b = sg.stride_b[0] * es, one.stride_h = sg.stride_h[0] * es;
  for (int i = 0; i < PKV_ATTN_MAX_SEGMENTS; ++i) one.end[i] = 0xffffffffu;
  int64_t first = 0;
  for (int i = 0; i < sg.n; ++i) {
    if (sg.k[i] != sg.k[0] || sg.v[i] != sg.v[0] || sg.stride_b[i] != sg.stride_b[0] || sg.stride_h[i] != sg.stride_h[0])
      return false;
    const int64_t n = sg.end[i] - first, rows = sg.row0[i] + (sg.idx[i] ? sg.idx_limit[i] : n);
    if (rows > ((int64_t)1 << 32) / (128 * es)) return false;
    one.end[i] = (uint32_t)sg.end[i];
    one.delta[i] = (int32_t)(sg.row0[i] - first);
    if (sg.idx[i]) {
      if (one.idx) return false;
      one.idx = sg.idx[i], one.idx_stride = sg.idx_stride[i], one.idx_limit = sg.idx_limit[i];
      one.idx_lo = (uint32_t)first, one.idx_hi = (uint32_t)sg.end[i], one.idx_row0 = (uint32_t)sg.row0[i];
    }
    first = sg.end[i];
  }
  return true;
}

}  // namespace

// One CU fetches scattered rows at 35 to 40 GB/s, 2.7 us for 200 of them and as much as the merge's launch: up to six blocks of 32
// are one workgroup's, which then merges; more go to a workgroup per split of 128, each selecting anew, or per two or three where
// that would be more workgroups than CUs; there up to eight blocks are one workgroup's as well.  More than 8192 candidates
// take longer to select from: only the first form (several workgroups a row gain 0.6 of 43.5 us at 16 rows x 131072, top 1024, and
// 1.7 of 55.4 at 200000: not built).
// Decode step, us, attention after the top-k / in two parts, by one workgroup a row: 8 rows x 4096 keys, top 100, 25.5 / 23.5;
// 32 x 16000, 8 heads, top 100, 31.6 / 30.8; 64 x 65536, top 100, 60.0 / 56.8; 256 x 8000, top 100, 74.0 / 66.0, top 256 80.3 / 70.8;
// more than 8192 candidates, where their selection took three launches: 8 x 100000, top 100, 47.2 / 45.7, 64 x 100000 96.7 / 94.2.
// By several: 8 x 32768, top 512, 28.6 / 28.4; 32 x 16000, 8 heads, top 512, 33.6 / 32.8; 64 x 40000, top 512, 52.6 / 51.4, top 1024 57.0 / 55.2.
// After the top-k / by one / by several, 40000 keys, 4000 candidates: six blocks, 8 rows 31.3 / 29.7 / 30.9, 32 rows 38.0 / 36.5 / 38.0,
// 64 rows 51.4 / 49.0 / 49.8; eight, 16 rows 33.5 / 34.4 / 33.8, 64 rows 51.9 / 50.3 / 50.2.  After the top-k / by one, 100000 keys,
// 9000 candidates (selected in three launches): six blocks, 8 rows 47.2 / 45.9, 64 rows 94.6 / 93.0; eight, 16 rows 52.6 / 53.7.
constexpr int kSplitWorkgroups = 256, kMergeBlocks = 6;
constexpr int64_t kSplitMaxSelected = 1024;

extern "C" size_t pkv_decode_attention_ws_bytes(int bs, int n_kv_heads, int group, int64_t total_keys) {
  if (bs <= 0 || n_kv_heads <= 0 || group <= 0 || total_keys <= 0) return 256;
  // room for the largest split count either path uses (64), whatever the key count and dtype
  return pkv_align_up((size_t)bs * n_kv_heads * 64 * group * kPartStride * sizeof(float), 256);
}

// The segments that have rows, checked, one behind the other.
static int collect_segments(int dtype, const pkv_attn_segment *segments, int n_segments, AttSegs &sg, int64_t &total, bool &indexed) {
  const int64_t vec = dtype == PKV_DTYPE_BF16 ? 8 : 4;
  memset(&sg, 0, sizeof sg);
  total = 0;
  indexed = false;
  for (int i = 0; i < n_segments; ++i) {
    const pkv_attn_segment &s = segments[i];
    PKV_REQUIRE(s.n_rows >= 0 && s.row0 >= 0, "segment %d: negative extent", i);
    if (s.n_rows == 0) continue;
    PKV_REQUIRE(s.k && s.v, "segment %d: null K/V", i);
    PKV_REQUIRE(pkv_aligned(s.k, 16) && pkv_aligned(s.v, 16) && s.stride_b % vec == 0 && s.stride_h % vec == 0,
                "segment %d: K/V must be 16-byte aligned with 16-byte-multiple strides", i);
    sg.k[sg.n] = s.k, sg.v[sg.n] = s.v;
    sg.stride_b[sg.n] = s.stride_b, sg.stride_h[sg.n] = s.stride_h;
    sg.row0[sg.n] = s.row0;
    if (s.idx) {
      PKV_REQUIRE(pkv_aligned(s.idx, 8) && s.idx_stride >= s.n_rows && s.idx_limit > 0 &&
                      s.row0 + s.idx_limit < ((int64_t)1 << 29),
                  "segment %d: indexed rows need idx_stride >= n_rows and 0 < idx_limit (row0 + idx_limit < 2^29)", i);
      sg.idx[sg.n] = s.idx, sg.idx_stride[sg.n] = s.idx_stride, sg.idx_limit[sg.n] = s.idx_limit;
      indexed = true;
    }
    total += s.n_rows;
    sg.end[sg.n] = total;
    ++sg.n;
  }
  return PKV_OK;
}

static int decode_attention(const void *q, int dtype, int bs, int n_kv_heads, int group, const pkv_attn_segment *segments,
                            int n_segments, const int32_t *row_keys, int uniform, float scale, void *out, void *ws,
                            size_t ws_bytes, uint32_t *arrivals, uint32_t *spares, void *stream) {
  PKV_REQUIRE(q && segments && out && ws, "pkv_decode_attention: null pointer");
  PKV_REQUIRE(dtype == PKV_DTYPE_F32 || dtype == PKV_DTYPE_BF16, "unknown dtype %d", dtype);
  PKV_REQUIRE(bs > 0 && n_kv_heads > 0 && (int64_t)bs * n_kv_heads <= 65535, "bad shape bs=%d kv_heads=%d", bs,
              n_kv_heads);
  PKV_REQUIRE(group >= 1 && group <= 8, "GQA group must be in [1, 8] (got %d)", group);
  PKV_REQUIRE(n_segments >= 1 && n_segments <= PKV_ATTN_MAX_SEGMENTS, "1..%d key segments", PKV_ATTN_MAX_SEGMENTS);
  PKV_REQUIRE(pkv_aligned(q, 16) && pkv_aligned(out, 4), "q must be 16-byte aligned");
  AttSegs sg;
  int64_t total;
  bool indexed;
  const int rc = collect_segments(dtype, segments, n_segments, sg, total, indexed);
  if (rc) return rc;
  PKV_REQUIRE(total > 0, "pkv_decode_attention: no keys");
  PKV_REQUIRE(total < ((int64_t)1 << 23), "pkv_decode_attention: at most 2^23 - 1 keys (got %lld)", (long long)total);
  const int rows = bs * n_kv_heads;
  const bool bf = dtype == PKV_DTYPE_BF16;
  const int heads_per_wg = group == 1 ? 1 : group == 2 ? 2 : 4;  // fp32 kernel
  const int head_wgs = (group + heads_per_wg - 1) / heads_per_wg;
  const int n_splits = bf ? pick_splits_mfma(rows, total) : pick_splits(rows * head_wgs, total);
  const size_t need = (size_t)rows * n_splits * group * kPartStride * sizeof(float);
  if (ws_bytes < need || !pkv_aligned(ws, 16)) {
    pkv_set_error("pkv_decode_attention: workspace of %zu bytes required, got %zu", need, ws_bytes);
    return PKV_ENOMEM;
  }
  const int step = bf ? kMfmaWaves * kMfmaStepKeys : kAttKeysPerIter * kAttUnroll;
  int64_t per_split = (total + n_splits - 1) / n_splits;
  per_split = (per_split + step - 1) / step * step;
  const float scale_log2e = scale * 1.4426950408889634f;
  hipStream_t s = (hipStream_t)stream;
  dim3 grid((unsigned)n_splits, (unsigned)rows);
  AttOne one;
  const bool is_one = as_one_tensor(sg, bf ? 2 : 4, one);
  const bool whole = arrivals && bf && n_splits <= kWholeSplits && rows * n_splits <= kWholeWorkgroups && !pkv_capturing(s);
  if (bf) {
    const dim3 grid3((unsigned)n_splits, (unsigned)n_kv_heads, (unsigned)bs);
#define PKV_ATT_MFMA_W(IDX, S, WHOLE)                                                                                           \
  hipLaunchKernelGGL((pkv_attn_partial_mfma_kernel<IDX, decltype(S), WHOLE>), grid3, dim3(kMfmaWaves * PKV_WAVE), 0, s, q, group, S, \
                     total, row_keys, uniform, per_split, scale_log2e, (float *)ws, arrivals, spares, out)
#define PKV_ATT_MFMA(IDX, S)                                                         \
  do {                                                                               \
    if (whole) PKV_ATT_MFMA_W(IDX, S, true); else PKV_ATT_MFMA_W(IDX, S, false);     \
  } while (0)
    if (is_one) {
      if (indexed) PKV_ATT_MFMA(true, one); else PKV_ATT_MFMA(false, one);
    } else {
      if (indexed) PKV_ATT_MFMA(true, sg); else PKV_ATT_MFMA(false, sg);
    }
#undef PKV_ATT_MFMA
#undef PKV_ATT_MFMA_W
  } else {
    // The KV head's other query heads in workgroups beside the first four's, in one launch: 12 rows x 865 keys, seven
    // heads, 2 x 8.0 us as two launches one after the other; the decode step around it (9001 keys) 48.3 -> 43 us.
    grid.z = (unsigned)head_wgs;
#define PKV_ATT(GG, IDX, S)                                                                                               \
  hipLaunchKernelGGL((pkv_attn_partial_kernel<GG, IDX, decltype(S)>), grid, dim3(kAttThreads), 0, s, q, n_kv_heads, group, \
                     S, total, row_keys, uniform, per_split, scale_log2e, (float *)ws)
#define PKV_ATT_G(IDX, S)                     \
  do {                                        \
    if (heads_per_wg == 1) PKV_ATT(1, IDX, S);      \
    else if (heads_per_wg == 2) PKV_ATT(2, IDX, S); \
    else PKV_ATT(4, IDX, S);                  \
  } while (0)
    if (is_one) {
      if (indexed) PKV_ATT_G(true, one); else PKV_ATT_G(false, one);
    } else {
      if (indexed) PKV_ATT_G(true, sg); else PKV_ATT_G(false, sg);
    }
#undef PKV_ATT_G
#undef PKV_ATT
  }
  PKV_LAUNCH_CHECK("pkv_attn_partial_kernel");
  if (whole) return PKV_OK;
  if (bf)
    hipLaunchKernelGGL(pkv_attn_merge_kernel<true>, dim3((unsigned)rows), dim3(group * 128), 0, s, (const float *)ws,
                       n_splits, group, out);
  else
    hipLaunchKernelGGL(pkv_attn_merge_kernel<false>, dim3((unsigned)rows), dim3(group * 128), 0, s, (const float *)ws,
                       n_splits, group, out);
  PKV_LAUNCH_CHECK("pkv_attn_merge_kernel");
  return PKV_OK;
}

extern "C" int pkv_decode_attention(const void *q, int dtype, int bs, int n_kv_heads, int group,
                                    const pkv_attn_segment *segments, int n_segments, const int32_t *row_keys,
                                    float scale, void *out, void *ws, size_t ws_bytes, void *stream) {
  return decode_attention(q, dtype, bs, n_kv_heads, group, segments, n_segments, row_keys, 0, scale, out, ws, ws_bytes, nullptr, nullptr, stream);
}

extern "C" int pkv_decode_attention_run(const void *q, int dtype, int bs, int n_kv_heads, int group, const pkv_attn_args *a,
                                        void *stream) {
  PKV_REQUIRE(a != nullptr, "pkv_decode_attention: null args");
  return decode_attention(q, dtype, bs, n_kv_heads, group, a->segments, a->n_segments, a->row_keys,
                          a->row_keys_uniform ? bs * n_kv_heads : 0, a->scale, a->out, a->ws, a->ws_bytes, nullptr, nullptr, stream);
}

extern "C" int pkv_decode_attention_counted(const void *q, int dtype, int bs, int n_kv_heads, int group, const pkv_attn_args *a,
                                            uint32_t *arrivals, int turn, void *stream) {
  PKV_REQUIRE(a != nullptr && arrivals != nullptr, "pkv_decode_attention_counted: null pointer");
  PKV_REQUIRE(pkv_aligned(arrivals, 4) && (turn == 0 || turn == 1), "arrivals must be 4-byte aligned, turn 0 or 1");
  const int64_t rows = (int64_t)bs * n_kv_heads;  // checked before they are used
  return decode_attention(q, dtype, bs, n_kv_heads, group, a->segments, a->n_segments, a->row_keys,
                          a->row_keys_uniform ? bs * n_kv_heads : 0, a->scale, a->out, a->ws, a->ws_bytes, arrivals + turn * rows,
                          arrivals + (1 - turn) * rows, stream);
}

bool pkv_plan_split_attention(const pkv_retrieve_args *r, const void *ws, const pkv_attn_args *at, PkvSplitAttn *out) {
  // What the general path would refuse is left to it.
  if (r->dtype != PKV_DTYPE_BF16 || !r->q || !pkv_aligned(r->q, 16) || !at->out || !pkv_aligned(at->out, 4) || !at->ws ||
      !pkv_aligned(at->ws, 16) || r->bs <= 0 || r->n_kv_heads <= 0 || (int64_t)r->bs * r->n_kv_heads > 65535 || r->group < 1 ||
      r->group > 8 || at->n_segments < 1 || at->n_segments > PKV_ATTN_MAX_SEGMENTS)
    return false;
  // Launches of this call's own, for the dense part to run beside: the query side's, or the scan's where that is already done.
  if (r->launch_plan != PKV_PLAN_SEPARATE) return false;
  // The selection: in any order, of one workgroup a row, into the list that the attention reads, nothing gathered.
  if (!r->out_ids || !r->any_order || r->src_k || r->n_cand == r->n_keys || at->row_keys || r->k > kSplitMaxSelected ||
      !pkv_topk_attends(r->n_cand, r->k))
    return false;
  for (int i = 0; i < at->n_segments; ++i) {
    const pkv_attn_segment &s = at->segments[i];
    if (s.n_rows < 0 || s.row0 < 0) return false;
    if (s.n_rows == 0) continue;
    if (!s.k || !s.v || !pkv_aligned(s.k, 16) || !pkv_aligned(s.v, 16) || s.stride_b % 8 || s.stride_h % 8) return false;
    if (s.idx && (s.idx != r->out_ids || s.idx_stride != r->k || s.n_rows != r->k || s.idx_limit <= 0 ||
                  s.row0 + s.idx_limit >= ((int64_t)1 << 29)))
      return false;
  }
  AttSegs sg;
  int64_t total;
  bool indexed;
  if (collect_segments(r->dtype, at->segments, at->n_segments, sg, total, indexed) || !indexed || total >= ((int64_t)1 << 23)) return false;
  memset(out, 0, sizeof *out);
  if (!as_one_tensor(sg, 2, out->segs)) return false;  // also: one indexed segment at most
  const int rows = r->bs * r->n_kv_heads;
  out->n_splits = pick_splits_mfma(rows, total);
  constexpr int kSplitKeys = kMfmaWaves * kMfmaStepKeys;
  if (total > (int64_t)out->n_splits * kSplitKeys) return false;  // a wave would take several blocks
  out->total = (uint32_t)total;
  out->blk_lo = (int)(out->segs.idx_lo / kMfmaStepKeys), out->blk_hi = (int)((out->segs.idx_hi - 1) / kMfmaStepKeys);
  const int lo = out->blk_lo / kMfmaWaves, hi = out->blk_hi / kMfmaWaves, n_sel = hi - lo + 1;  // splits with selected keys
  const int blocks = out->blk_hi - out->blk_lo + 1;
  if (out->n_splits < kSelSplits && (blocks <= kMergeBlocks || (blocks <= kSelBlocks && (int64_t)rows * n_sel > kSplitWorkgroups))) {
    out->sel_wgs = 1;
    // the splits between the first and the last one's own blocks have nothing else to do
    const int last_block = (int)((total - 1) / kMfmaStepKeys);
    out->dense_a = (out->blk_lo + kMfmaWaves - 1) / kMfmaWaves;
    const int from = out->blk_hi == last_block ? out->n_splits : (out->blk_hi + 1) / kMfmaWaves;
    out->dense_skip = from > out->dense_a ? from - out->dense_a : 0;
    for (int i = 0; i <= last_block; ++i) {
      const bool mixed = i / kMfmaWaves >= lo && i / kMfmaWaves <= hi;
      if (i < out->blk_lo || i > out->blk_hi) out->slots |= 1u << (mixed ? att_block_slot(*out, i) : i / kMfmaWaves);
    }
    if ((int64_t)rows * 20 * r->group * 128 >= ((int64_t)1 << 31)) return false;
    out->ws_ml = (float *)at->ws + (int64_t)rows * 20 * r->group * 128;
  } else if (r->n_cand > kTopkMaxSort) {
    return false;
  } else {
    do {
      out->sel_wgs = (n_sel + ++out->splits_per_wg - 1) / out->splits_per_wg;
    } while (out->splits_per_wg < kSelSplits / 4 && (int64_t)rows * out->sel_wgs > kSplitWorkgroups);
    if (out->sel_wgs == 1) return false;  // few selected keys among very many others
    // A second round of workgroups selects once more for every row: never with eight candidates to a thread, and with fewer where
    // the last round is less than 3/8 full.  Decode step, us, attention after the top-k / by several workgroups a row: 128 rows,
    // 8192 candidates, top 1024 (384 workgroups) 94.3 / 102.5, 192 rows, 5000, top 512 (384) 105.9 / 110.4; 4096 candidates: 96 rows,
    // top 1024 (288) 59.9 / 61.6, 136, top 700 (272) 72.2 / 74.0, 192, top 1024 (576) 101.3 / 105.0; 176, top 512 (352) 85.7 / 83.5,
    // 160, top 1024 (480) 90.1 / 86.8, 256, top 512 (512) 113.3 / 106.2.
    const int64_t all = (int64_t)rows * out->sel_wgs, last = all % kSplitWorkgroups;
    if (all > kSplitWorkgroups && (r->n_cand > kTopkMaxSort / 2 || (last && last < kSplitWorkgroups * 3 / 8))) return false;
    out->dense_a = lo, out->dense_skip = n_sel;
  }
  out->n_dense = out->n_splits - out->dense_skip;
  const size_t row_floats = out->sel_wgs == 1 ? (size_t)20 * r->group * 128 + (size_t)r->group * kSelSlots * 2
                                              : (size_t)out->n_splits * r->group * kPartStride;
  const size_t at_bytes = (size_t)rows * row_floats * sizeof(float), out_bytes = (size_t)rows * r->group * 256;
  if (at->ws_bytes < at_bytes) return false;
  // Partial results and output are written while the retrieval still works, not after it: where they would lie in its workspace,
  // queries or results, the attention waits.  (An output in place of the queries is fine: a row's are read before it is written.)
  const size_t r_bytes = pkv_retrieve_ws_bytes(rows, r->n_keys, r->n_cand, r->k);
  const struct {
    const void *p;
    size_t n;
  } busy[] = {{ws, r_bytes}, {r->out_ids, (size_t)rows * r->k * 8}, {r->out_scores, (size_t)rows * r->k * 4}, {r->q, out_bytes}};
  for (const auto &u : busy)
    if (pkv_meets(at->ws, at_bytes, u.p, u.n) || (pkv_meets(at->out, out_bytes, u.p, u.n) && !(u.p == r->q && at->out == r->q))) return false;
  if (pkv_meets(at->out, out_bytes, at->ws, at_bytes)) return false;
  out->n_kv_heads = r->n_kv_heads, out->group = r->group, out->q = r->q;
  out->scale_log2e = at->scale * 1.4426950408889634f;
  out->ws = (float *)at->ws, out->out = at->out;
  return true;
}

int pkv_launch_attn_merge(const PkvSplitAttn &a, int rows, hipStream_t s) {
  hipLaunchKernelGGL(pkv_attn_merge_kernel<true>, dim3((unsigned)rows), dim3(a.group * 128), 0, s, (const float *)a.ws, a.n_splits, a.group,
                     a.out);
  PKV_LAUNCH_CHECK("pkv_attn_merge_kernel");
  return PKV_OK;
}
