// Attention over the paged cache, one block per (row, query head): the true
// 32-bit path, and the path of the bf16 engine for sizes its MFMA kernels
// refuse.
//
// Formula: /root/reference/core/src/nn/attention.cpp:26-105 and :121-181 —
// query head h reads kv head h / group; s_j = dot(q, k_j) * scale; a key is
// visible when j <= p and (window == 0 or p - j < window); softmax with the
// maximum subtracted; a row without visible keys is zero.  With `chunk` > 0 (no
// window then) the keys of position p's own stretch of that many positions are
// visible, [chunk * (p / chunk), p].
//
// The cache holds keys as [page][kv head][position][d] and values transposed,
// [page][kv head][d][position].
//
// Keys are taken 64 at a time in chunks at absolute positions [64c, 64c+64),
// lane l owning key 64c+l.  A chunk's maximum, sum and mix are made by one wave from
// nothing, in ascending key; the chunks' results are joined one after the other in
// ascending c, so the arithmetic of a row is a function of its position and
// window alone: it does not change with the batch, with the cut of the prompt
// into steps, with the physical pages or with the waves that share the chunks.
//
// It is bound by latency: a chunk is two dependent reads (the page's number, then its
// keys and values).  The block's waves take a chunk each, and a wave asks for a chunk's values
// before it reads its keys, sixteen bytes a load.  Measured with 14 heads of 64 in float32: one token of 3
// sequences of 40 to 260 keys 31.4 us with one wave a row and head and an element a load, 8.5 now; the
// prompts of 40, 220 and 260 rows 145 and 59.  Behind it stay calls of a few rows on a few keys, which the longer code costs
// (a prompt of 3 rows, 12 heads of 128: 7.2 and 9.0), and many rows of heads of 16 (1,000, a window of 100: 28 and 33).  Loads of
// all eight groups of values, the hidden ones aimed at a visible one's place, cost more (32 prompts of 10 rows 12.4 and 19.5),
// loads that leave the hidden ones out by a descriptor's end as much (13.7).
#include "common.h"

namespace {

constexpr int kMaxHeadDim = 256;

// Eight consecutive elements (the caches keep groups of eight together).
__device__ __forceinline__ void ld_eight(const float *p, float (&v)[8]) {
  const float4 a = *reinterpret_cast<const float4 *>(p), b = *reinterpret_cast<const float4 *>(p + 4);
  v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}
__device__ __forceinline__ void ld_eight(const bf16_t *p, float (&v)[8]) {
  const uint4 a = *reinterpret_cast<const uint4 *>(p);
  const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) v[2 * i] = __uint_as_float(w[i] << 16), v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
}

// EIGHTS: head_dim % 8 == 0, and keys are read a group of eight at a time.
template <typename TA, typename TC, int WAVES, bool EIGHTS>
__global__ void __launch_bounds__(64 * WAVES)
attention_plain_kernel(TA *__restrict__ out, const TA *__restrict__ q, int q_stride,
                       const TC *__restrict__ k_cache, const TC *__restrict__ v_cache,
                       const int32_t *__restrict__ page_table, int max_pages, int n_pages_total,
                       const int32_t *__restrict__ row_pos, const int32_t *__restrict__ row_seq,
                       int heads_q, int heads_kv, int head_dim, float scale, int window, int v_dim,
                       float softcap, int sink, const float *__restrict__ sink_scores,
                       const float *__restrict__ gate, int gate_stride, int gate_per_head, int chunk) {
  constexpr int kThreads = 64 * WAVES, kDims = (kMaxHeadDim + kThreads - 1) / kThreads;
  __shared__ float qs[kMaxHeadDim];
  __shared__ float ps[WAVES][64];
  __shared__ float part_m[WAVES], part_l[WAVES];
  __shared__ float part_o[WAVES][kMaxHeadDim];
  const int row = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int pos = row_pos[row], seq = row_seq[row];
  const int kvh = h / (heads_q / heads_kv);
  for (int d = tid; d < head_dim; d += kThreads) qs[d] = ld_f(q, size_t(row) * q_stride + size_t(h) * head_dim + d);
  __syncthreads();

  const int lo = chunk > 0 ? pos - pos % chunk : (window > 0 && pos >= window) ? pos - window + 1 : 0;
  const float neg_inf = -__builtin_inff();
  // a sink is one more key that has no value, of score 0 or, with sink_scores, of the head's own
  // number (as it is: no scale, no cap): the running maximum starts at its score and the running
  // sum at its weight
  float m = sink ? (sink_scores ? sink_scores[h] : 0.0f) : neg_inf, l = sink ? 1.0f : 0.0f;
  float o[kDims];
#pragma unroll
  for (int i = 0; i < kDims; ++i) o[i] = 0.0f;

  const int c_end = pos / SB_PAGE + 1;
  for (int c0 = lo / SB_PAGE; c0 < c_end; c0 += WAVES) {
    const int c = c0 + wave;
    const int page = c < c_end && c < max_pages ? page_table[size_t(seq) * max_pages + c] : -1;
    const bool live = page >= 0 && page < n_pages_total;      // uniform over the wave
    if (live) {
      const TC *kp = k_cache + (size_t(page) * heads_kv + kvh) * SB_PAGE * head_dim;
      const TC *vp = v_cache + (size_t(page) * heads_kv + kvh) * SB_PAGE * v_dim;
      const int j = c * SB_PAGE + lane;
      const bool visible = j >= lo && j <= pos;
      // (keys outside the window are left out by their place, not by a weight of zero: what the
      // cache holds there is anything)
      const int j0 = max(lo - c * SB_PAGE, 0), j1 = min(pos - c * SB_PAGE, SB_PAGE - 1);
      const auto seen = [&](int jg) { return 8 * jg <= j1 && 8 * jg + 7 >= j0; };      // some key of eight; uniform
      // the values of this lane's first dimension, asked for ahead of the keys
      float v[8][8];
      if (lane < v_dim) {
#pragma unroll
        for (int jg = 0; jg < 8; ++jg)
          if (seen(jg)) ld_eight(vp + sb_value_index(lane, 8 * jg), v[jg]);
      }
      float s = neg_inf;
      if (visible) {
        float dot = 0.0f;
        if constexpr (EIGHTS) {
#pragma unroll 8
          for (int d = 0; d < head_dim; d += 8) {
            float k8[8];
            ld_eight(kp + sb_key_index(lane, d, head_dim), k8);
#pragma unroll
            for (int e = 0; e < 8; ++e) dot = fmaf(qs[d + e], k8[e], dot);
          }
        } else {
          for (int d = 0; d < head_dim; ++d) dot = fmaf(qs[d], ld_f(kp, sb_key_index(lane, d, head_dim)), dot);
        }
        s = dot * scale;
        if (softcap > 0.0f) s = softcap * tanhf(s / softcap);
      }
      const float cm = wave_max(s);
      // (a score that ran out of the range weighs nothing, also in a chunk that holds no other: the join goes by the
      // maximum over all chunks)
      const float p = visible && s != neg_inf ? expf(s - cm) : 0.0f;
      const float cl = wave_sum(p);
      ps[wave][lane] = p;
      if (lane == 0) part_m[wave] = cm, part_l[wave] = cl;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      for (int d = lane; d < v_dim; d += 64) {
        if (d >= 64) {
#pragma unroll
          for (int jg = 0; jg < 8; ++jg)
            if (seen(jg)) ld_eight(vp + sb_value_index(d, 8 * jg), v[jg]);
        }
        float acc = 0.0f;
#pragma unroll
        for (int jg = 0; jg < 8; ++jg) {
          if (!seen(jg)) continue;
#pragma unroll
          for (int e = 0; e < 8; ++e)
            acc = fmaf(ps[wave][8 * jg + e], 8 * jg + e >= j0 && 8 * jg + e <= j1 ? v[jg][e] : 0.0f, acc);
        }
        part_o[wave][d] = acc;
      }
    } else if (lane == 0) {
      part_l[wave] = -1.0f;                      // no such chunk
    }
    __syncthreads();
    for (int w = 0; w < WAVES; ++w) {
      const float cl = part_l[w];
      if (cl < 0.0f) continue;                   // (a sum that is not a number goes on)
      const float cm = part_m[w], m_new = fmaxf(m, cm);
      const float alpha = expf(m - m_new), beta = expf(cm - m_new);      // alpha 0 for the first chunk
      l = l * alpha + cl * beta;
#pragma unroll
      for (int i = 0; i < kDims; ++i) {
        const int d = tid + kThreads * i;
        if (d < v_dim) o[i] = o[i] * alpha + part_o[w][d] * beta;
      }
      m = m_new;
    }
    __syncthreads();
  }
  const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
  for (int i = 0; i < kDims; ++i) {
    const int d = tid + kThreads * i;
    if (d < v_dim) {
      float r = o[i] * inv;
      // an output gate: the result times the sigmoid of the gate's number at the same place of the row, or of the head's one
      if (gate) r = r * (1.0f / (1.0f + expf(-gate[size_t(row) * gate_stride + (gate_per_head ? size_t(h) : size_t(h) * v_dim + d)])));
      st_f(out, size_t(row) * heads_q * v_dim + size_t(h) * v_dim + d, r);
    }
  }
}

template <typename TA, typename TC, int WAVES, typename... A>
void launch_waves(dim3 grid, int head_dim, hipStream_t s, A... a) {
  if (head_dim % 8 == 0) attention_plain_kernel<TA, TC, WAVES, true><<<grid, 64 * WAVES, 0, s>>>(a...);
  else attention_plain_kernel<TA, TC, WAVES, false><<<grid, 64 * WAVES, 0, s>>>(a...);
}

// Waves of a block: four, each a chunk of 64 keys at a time; eight where the blocks alone leave SIMDs idle; no more than
// there are chunks that a row can see (`most`), since a wave without one only holds its block's place.
template <typename TA, typename TC, typename... A>
void launch_attention(dim3 grid, int head_dim, int most, hipStream_t s, A... a) {
  if (most <= 1) launch_waves<TA, TC, 1>(grid, head_dim, s, a...);
  else if (most <= 2) launch_waves<TA, TC, 2>(grid, head_dim, s, a...);
  else if (most <= 4 || (long long)grid.x * grid.y > 512) launch_waves<TA, TC, 4>(grid, head_dim, s, a...);
  else launch_waves<TA, TC, 8>(grid, head_dim, s, a...);
}

}  // namespace

extern "C" int sb_attention_chunked(void *out, const void *q, int act_dtype, int q_stride, const void *k_cache,
                                    const void *v_cache, int cache_dtype, const int32_t *page_table,
                                    int max_pages, int n_pages_total, const int32_t *row_pos,
                                    const int32_t *row_seq, int n_rows, int heads_q, int heads_kv,
                                    int head_dim, int v_dim, float scale, int window, float softcap, int sink,
                                    const float *sink_scores, const float *gate, int gate_stride, int gate_per_head, int chunk,
                                    void *stream);

// The same with values of another size than the keys (v_dim; the cache then holds values
// [page][kv head][v_dim][position] and out is [rows, heads_q * v_dim]), scores capped as
// softcap * tanh(s / softcap) when softcap > 0, and with `sink` one more key of score 0 without a
// value in every row's softmax: weights exp(s_j) / (1 + sum exp(s_j)).
extern "C" int sb_attention_capped(void *out, const void *q, int act_dtype, int q_stride, const void *k_cache,
                                   const void *v_cache, int cache_dtype, const int32_t *page_table,
                                   int max_pages, int n_pages_total, const int32_t *row_pos,
                                   const int32_t *row_seq, int n_rows, int heads_q, int heads_kv,
                                   int head_dim, int v_dim, float scale, int window, float softcap, int sink,
                                   void *stream);

extern "C" int sb_attention(void *out, const void *q, int act_dtype, int q_stride, const void *k_cache,
                            const void *v_cache, int cache_dtype, const int32_t *page_table,
                            int max_pages, int n_pages_total, const int32_t *row_pos,
                            const int32_t *row_seq, int n_rows, int heads_q, int heads_kv,
                            int head_dim, float scale, int window, void *stream) {
  return sb_attention_capped(out, q, act_dtype, q_stride, k_cache, v_cache, cache_dtype, page_table, max_pages,
                             n_pages_total, row_pos, row_seq, n_rows, heads_q, heads_kv, head_dim, head_dim, scale,
                             window, 0.0f, 0, stream);
}

extern "C" int sb_attention_sink(void *out, const void *q, int act_dtype, int q_stride, const void *k_cache,
                                 const void *v_cache, int cache_dtype, const int32_t *page_table,
                                 int max_pages, int n_pages_total, const int32_t *row_pos,
                                 const int32_t *row_seq, int n_rows, int heads_q, int heads_kv,
                                 int head_dim, int v_dim, float scale, int window, float softcap, int sink,
                                 const float *sink_scores, const float *gate, int gate_stride, int gate_per_head, void *stream);

extern "C" int sb_attention_capped(void *out, const void *q, int act_dtype, int q_stride, const void *k_cache,
                                   const void *v_cache, int cache_dtype, const int32_t *page_table,
                                   int max_pages, int n_pages_total, const int32_t *row_pos,
                                   const int32_t *row_seq, int n_rows, int heads_q, int heads_kv,
                                   int head_dim, int v_dim, float scale, int window, float softcap, int sink,
                                   void *stream) {
  return sb_attention_sink(out, q, act_dtype, q_stride, k_cache, v_cache, cache_dtype, page_table, max_pages, n_pages_total,
                           row_pos, row_seq, n_rows, heads_q, heads_kv, head_dim, v_dim, scale, window, softcap, sink,
                           nullptr, nullptr, 0, 0, stream);
}

// The same with a sink whose score is a number of the query head's own, sink_scores f32 [heads_q]
// (NULL: 0): weights exp(s_j) / (exp(sink_h) + sum exp(s_j)); and with an output gate (or NULL): the
// result [rows, heads_q * v_dim] times sigmoid(gate[row * gate_stride + i]), number by number, or with
// gate_per_head every number of head h times sigmoid(gate[row * gate_stride + h]).
extern "C" int sb_attention_sink(void *out, const void *q, int act_dtype, int q_stride, const void *k_cache,
                                 const void *v_cache, int cache_dtype, const int32_t *page_table,
                                 int max_pages, int n_pages_total, const int32_t *row_pos,
                                 const int32_t *row_seq, int n_rows, int heads_q, int heads_kv,
                                 int head_dim, int v_dim, float scale, int window, float softcap, int sink,
                                 const float *sink_scores, const float *gate, int gate_stride, int gate_per_head, void *stream) {
  return sb_attention_chunked(out, q, act_dtype, q_stride, k_cache, v_cache, cache_dtype, page_table, max_pages, n_pages_total, row_pos,
                              row_seq, n_rows, heads_q, heads_kv, head_dim, v_dim, scale, window, softcap, sink, sink_scores, gate,
                              gate_stride, gate_per_head, 0, stream);
}

// The same where, with chunk > 0 (and window 0), position p sees the keys from chunk * (p / chunk) on.
extern "C" int sb_attention_chunked(void *out, const void *q, int act_dtype, int q_stride, const void *k_cache,
                                    const void *v_cache, int cache_dtype, const int32_t *page_table,
                                    int max_pages, int n_pages_total, const int32_t *row_pos,
                                    const int32_t *row_seq, int n_rows, int heads_q, int heads_kv,
                                    int head_dim, int v_dim, float scale, int window, float softcap, int sink,
                                    const float *sink_scores, const float *gate, int gate_stride, int gate_per_head, int chunk,
                                    void *stream) {
  SB_REQUIRE(chunk >= 0 && (chunk == 0 || window == 0), "sb_attention: a window and a chunk at once");
  SB_REQUIRE(!sink_scores || sink, "sb_attention: scores of a sink that is switched off");
  SB_REQUIRE(!gate || gate_stride >= heads_q * (gate_per_head ? 1 : v_dim), "sb_attention: the gate's rows of %d are too short", gate_stride);
  SB_REQUIRE(out && q && k_cache && v_cache && page_table && row_pos && row_seq,
             "sb_attention: null pointer");
  SB_REQUIRE(n_rows >= 0 && heads_q > 0 && heads_kv > 0 && head_dim > 0 && max_pages > 0 &&
                 n_pages_total > 0 && window >= 0,
             "sb_attention: bad sizes rows=%d heads_q=%d heads_kv=%d head_dim=%d", n_rows, heads_q,
             heads_kv, head_dim);
  SB_REQUIRE(heads_q % heads_kv == 0, "sb_attention: %d query heads are not a multiple of %d kv heads",
             heads_q, heads_kv);
  SB_REQUIRE(q_stride >= heads_q * head_dim, "sb_attention: query stride %d shorter than %d", q_stride,
             heads_q * head_dim);
  SB_REQUIRE(sb::valid_dtype(act_dtype) && sb::valid_dtype(cache_dtype), "sb_attention: unknown dtype");
  SB_SUPPORT(head_dim <= kMaxHeadDim && v_dim > 0 && v_dim <= kMaxHeadDim,
             "sb_attention: head sizes %d and %d must be positive and at most %d", head_dim, v_dim, kMaxHeadDim);
  SB_REQUIRE(softcap >= 0.0f, "sb_attention: the cap of the scores must not be negative");
  SB_SUPPORT(heads_q <= 65535, "sb_attention: more than 65535 query heads");
  if (n_rows == 0) return SB_OK;
  hipStream_t s = (hipStream_t)stream;
  dim3 grid(n_rows, heads_q);
  const int reach = window > 0 ? window : chunk;             // keys from the first that a row sees to itself
  const int most = reach > 0 ? min(max_pages, (reach - 1 + SB_PAGE - 1) / SB_PAGE + 1) : max_pages;
#define SB_GO(TA, TC)                                                                           \
  launch_attention<TA, TC>(grid, head_dim, most, s,                                              \
      (TA *)out, (const TA *)q, q_stride, (const TC *)k_cache, (const TC *)v_cache, page_table,  \
      max_pages, n_pages_total, row_pos, row_seq, heads_q, heads_kv, head_dim, scale, window, v_dim,  \
      softcap, sink, sink_scores, gate, gate_stride, gate_per_head, chunk)
  if (act_dtype == SB_F32 && cache_dtype == SB_F32) SB_GO(float, float);
  else if (act_dtype == SB_BF16 && cache_dtype == SB_BF16) SB_GO(bf16_t, bf16_t);
  else if (act_dtype == SB_F32 && cache_dtype == SB_BF16) SB_GO(float, bf16_t);
  else SB_GO(bf16_t, float);
#undef SB_GO
  return sb::check_launch("sb_attention");
}
