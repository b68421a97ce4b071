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

// grid (splits, rows, query heads by G)
template <bool BF16, int G, bool INDEXED, typename SEGS>
__global__ __launch_bounds__(kAttThreads) void pkv_attn_partial_kernel(const void *__restrict__ q, int n_kv_heads,
                                                                       int group, SEGS segs, int64_t total,
                                                                       const int32_t *__restrict__ row_keys, int uniform,
                                                                       int64_t per_split, float scale_log2e,
                                                                       float *__restrict__ ws) {
  att_partial_vector<BF16, G, INDEXED>(q, n_kv_heads, group, segs, total, row_keys, uniform, per_split, scale_log2e, ws,
                                       (int)gridDim.x, (int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z);
}

// grid (splits, KV heads, batch).  Decode step, us, with four-way pointer selection per row / with places by lane exchange:
// 8 rows x 693 attended keys 30.2 / 27.7, 8 x 1188 (4 layers) 136.5 / 124.2, 64 x 887 (2 layers) 133.4 / 122.8.
template <bool INDEXED, typename SEGS>
__global__ __launch_bounds__(kMfmaWaves * PKV_WAVE) void pkv_attn_partial_mfma_kernel(
    const void *__restrict__ q, int group, SEGS segs, int64_t total, const int32_t *__restrict__ row_keys, int uniform,
    int64_t per_split, float scale_log2e, float *__restrict__ ws) {
  const int h = blockIdx.y, b = blockIdx.z;
  att_partial_mfma<INDEXED>(q, group, segs, total, row_keys, uniform, per_split, scale_log2e, ws, (int)gridDim.x,
                            (int)blockIdx.x, b * (int)gridDim.y + h, b, h);
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
// that would be more workgroups than CUs; there up to eight blocks are one workgroup's as well.  Where the selection takes several
// launches (more than 8192 candidates), only the first form: its last launch is too long to be run by several workgroups a row
// (16 rows x 131072, top 200, 52.0 / 52.5).
// Decode step, us, attention after the top-k / in two parts, by one workgroup a row: 8 rows x 4096 keys, top 100, 25.5 / 23.5;
// 32 x 16000, 8 heads, top 100, 31.6 / 30.8; 64 x 65536, top 100, 60.0 / 56.8; 256 x 8000, top 100, 74.0 / 66.0, top 256 80.3 / 70.8;
// more than 8192 candidates: 8 x 100000, top 100, 47.2 / 45.7, 64 x 100000 96.7 / 94.2.  By several: 8 x 32768, top 512, 28.6 / 28.4;
// 32 x 16000, 8 heads, top 512, 33.6 / 32.8; 64 x 40000, top 512, 52.6 / 51.4, top 1024 57.0 / 55.2.
// After the top-k / by one / by several, 40000 keys, 4000 candidates: six blocks, 8 rows 31.3 / 29.7 / 30.9, 32 rows 38.0 / 36.5 / 38.0,
// 64 rows 51.4 / 49.0 / 49.8; eight, 16 rows 33.5 / 34.4 / 33.8, 64 rows 51.9 / 50.3 / 50.2.  After the top-k / by one, 100000 keys,
// 9000 candidates: six blocks, 8 rows 47.2 / 45.9, 64 rows 94.6 / 93.0; eight, 16 rows 52.6 / 53.7.
constexpr int kSplitWorkgroups = 256, kMergeBlocks = 6;
constexpr int64_t kSplitMaxSelected = 1024, kSplitMaxCand = 8192;

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
                            size_t ws_bytes, void *stream) {
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
  if (bf) {
    const dim3 grid3((unsigned)n_splits, (unsigned)n_kv_heads, (unsigned)bs);
#define PKV_ATT_MFMA(IDX, S)                                                                                                    \
  hipLaunchKernelGGL((pkv_attn_partial_mfma_kernel<IDX, decltype(S)>), grid3, dim3(kMfmaWaves * PKV_WAVE), 0, s, q, group, S, total, \
                     row_keys, uniform, per_split, scale_log2e, (float *)ws)
    if (is_one) {
      if (indexed) PKV_ATT_MFMA(true, one); else PKV_ATT_MFMA(false, one);
    } else {
      if (indexed) PKV_ATT_MFMA(true, sg); else PKV_ATT_MFMA(false, sg);
    }
#undef PKV_ATT_MFMA
  } else {
    // The KV head's other query heads in workgroups beside the first four's, in one launch: 12 rows x 865 keys, seven
    // heads, 2 x 8.0 us as two launches one after the other; the decode step around it (9001 keys) 48.3 -> 43 us.
    grid.z = (unsigned)head_wgs;
#define PKV_ATT(GG, IDX, S)                                                                                               \
  hipLaunchKernelGGL((pkv_attn_partial_kernel<false, GG, IDX, decltype(S)>), grid, dim3(kAttThreads), 0, s, q, n_kv_heads, group, \
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
  return decode_attention(q, dtype, bs, n_kv_heads, group, segments, n_segments, row_keys, 0, scale, out, ws, ws_bytes, stream);
}

extern "C" int pkv_decode_attention_run(const void *q, int dtype, int bs, int n_kv_heads, int group, const pkv_attn_args *a,
                                        void *stream) {
  PKV_REQUIRE(a != nullptr, "pkv_decode_attention: null args");
  return decode_attention(q, dtype, bs, n_kv_heads, group, a->segments, a->n_segments, a->row_keys,
                          a->row_keys_uniform ? bs * n_kv_heads : 0, a->scale, a->out, a->ws, a->ws_bytes, stream);
}

static bool meets(const void *a, size_t a_bytes, const void *b, size_t b_bytes) {
  return a && b && (uintptr_t)a < (uintptr_t)b + b_bytes && (uintptr_t)b < (uintptr_t)a + a_bytes;
}

bool pkv_plan_split_attention(const pkv_retrieve_args *r, const void *ws, const pkv_attn_args *at, PkvSplitAttn *out) {
  // What the general path would refuse is left to it.
  if (r->dtype != PKV_DTYPE_BF16 || !r->q || !pkv_aligned(r->q, 16) || !at->out || !pkv_aligned(at->out, 4) || !at->ws ||
      !pkv_aligned(at->ws, 16) || r->bs <= 0 || r->n_kv_heads <= 0 || (int64_t)r->bs * r->n_kv_heads > 65535 || r->group < 1 ||
      r->group > 8 || at->n_segments < 1 || at->n_segments > PKV_ATTN_MAX_SEGMENTS)
    return false;
  // The query side: a launch of this call's own, for the dense part to run beside.
  if (r->launch_plan != PKV_PLAN_SEPARATE || r->table_ready) return false;
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
  } else if (r->n_cand > kSplitMaxCand) {
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
    if (all > kSplitWorkgroups && (r->n_cand > kSplitMaxCand / 2 || (last && last < kSplitWorkgroups * 3 / 8))) return false;
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
    if (meets(at->ws, at_bytes, u.p, u.n) || (meets(at->out, out_bytes, u.p, u.n) && !(u.p == r->q && at->out == r->q))) return false;
  if (meets(at->out, out_bytes, at->ws, at_bytes)) return false;
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
