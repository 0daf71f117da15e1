// bf16 matrix products of a decode step of few rows whose block owns 16 output features whole, K cut over its waves:
// Y[t,n] = sum_k X[t,k] W[n,k].
//
// Between attention and the feed-forward of such a step stood a pass over whole rows (add the product's K slices to the
// stream, norm it), 4 to 5 us of which hardly any is work.  Because a block here ends with finished features, it rides in the
// two products on either side:
//   join:  x[t,n] += Y[t,n] (+ bias), the residual stream, and x[t,n] * weight[n] in bfloat16 and the sum of the squares of
//          the block's sixteen x[t,n].  The norm's factor of a row, 1 / sqrt(mean square + eps), is the same for all of its
//          columns, so it can be multiplied in after the next product: (x w inv) W^T = inv (x w) W^T.
//   gated: act(inv g) * (inv u), the factor made by every block from the sums of squares that the joining product's blocks
//          left, parts added in a fixed order.
// The squares are float products added up in double, and the mean is rounded once, as every RMS norm here does it
// (embed_norm.hip).  The weighted rows are rounded to bfloat16 before the factor and not after it: the same relative error.
// Measured (us, replayed graphs, weights cold; one and eight rows): the joining product with its norm against K slices and
// the pass, width 896 6.2 -> 3.7 and 6.6 -> 4.0, 1,536 7.4 -> 4.6 and 7.8 -> 5.1, 2,048 8.6 -> 6.1 and 8.9 -> 6.5, 3,584
// 11.1 -> 8.1 and 11.5 -> 8.4; the gated one against the kernel that streams weights, 9,728 x 896 7.3 -> 7.6 and 7.7 -> 7.8,
// 17,920 x 1,536 14.3 -> 15.5 and 14.3 -> 16.2, 22,016 x 2,048 20.9 -> 21.0 and 20.8 -> 22.0, 37,888 x 3,584 52.1 -> 49.9 and
// 51.6 -> 52.8.  With more rows the gated one falls behind by more than the other gains.  The gated product of up to eight rows
// goes on to gemm_skinny.hip or gemm_rows.hip where these take the sizes (gemm_rows.h); here stay less than 512 k and rows that
// do not fit LDS.
//
// W is packed (16 x 32 tiles of 1 KB in fragment order, the tiles of a row block consecutive in k), so
// a wave reads one contiguous stream, a ring of registers ahead; X's fragments come from L2 (every block
// reads all of X).  The waves' sums meet in LDS and are added in wave order.
//
// MFMA roles: A = 16 rows of W, B = 16 rows of X, D[n][t]; a lane holds four consecutive n of one t.
#include "gemm_rows.h"
#include "mfma.h"

namespace {

struct SplitArgs {
  int n_rows, n_out, n_in;
  // gated: the row's factor of X, an unfinished norm: ssq [ssq_parts][n_rows]
  const double *ssq;
  int ssq_parts;
  float eps;
  bf16_t *y;            // gated: [n_rows][n_out]
  int gate;             // gated: an sb_gate
  const void *bias;     // join, or NULL
  int bias_dtype;
  float *resid;         // join: [n_rows][n_out], added to in place
  bf16_t *xw;           // join: x * norm_w, and
  double *ssq_out;      // [tiles][n_rows]
  const void *norm_w;   // (NULL: ones)
  int norm_dtype;
};

constexpr int kMaxRows = 16;

template <bool GATED, int W>
__global__ void __launch_bounds__(64 * W)
gemm_split_kernel(const bf16_t *__restrict__ x, const bf16_t *__restrict__ w, SplitArgs a) {
  constexpr int G = GATED ? 2 : 1;
  constexpr int kAhead = 8;
  constexpr int kGroups = 64 * W / kMaxRows;     // threads a row that add its sums of squares
  __shared__ floatx4_t red[W * G * 64];
  __shared__ double row_part[kGroups * kMaxRows];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int tile = blockIdx.x, tiles = (a.n_out + 15) / 16;
  const int n_steps = (a.n_in + 31) / 32, per = (n_steps + W - 1) / W;
  const int s0 = min(wave * per, n_steps), s1 = min(s0 + per, n_steps);

  __amdgpu_buffer_rsrc_t rsrc_w[G];
#pragma unroll
  for (int g = 0; g < G; ++g)
    rsrc_w[g] = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t *>(w) + size_t(g * tiles + tile) * n_steps * 512, 0,
                                                  uint32_t(s1) * 1024u, 0x00020000);
  // rows past the last one lie past the descriptor's end and read as zeros
  const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16_t *>(x), 0, uint32_t(size_t(a.n_rows) * a.n_in * 2), 0x00020000);
  constexpr uint32_t kOutside = 0x80000000u;
  const uint32_t x_off = r < a.n_rows ? uint32_t((size_t(r) * a.n_in + 8 * q) * 2) : kOutside;

  uint4 rw[kAhead][G], rx[kAhead];
  auto ask = [&](int slot, int step) {
#pragma unroll
    for (int g = 0; g < G; ++g)
      rw[slot][g] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_w[g], lane * 16 + step * 1024, 0, kReadOnce));
    const bool in = step < s1 && step * 32 + 8 * q < a.n_in;          // (n_in is a multiple of 8)
    rx[slot] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(
        rsrc_x, int(in ? x_off + uint32_t(step) * 64u : kOutside), 0, 0));
  };
#pragma unroll
  for (int u = 0; u < kAhead; ++u) ask(u, s0 + u);

  // what the epilogue (the first wave's) reads, asked for ahead of the stream's rest
  const int unit_n = tile * 16 + 4 * q;
  const bool unit_live = wave == 0 && r < a.n_rows && unit_n < a.n_out;
  float old[4] = {0.f, 0.f, 0.f, 0.f}, nw[4] = {1.f, 1.f, 1.f, 1.f}, bias[4] = {0.f, 0.f, 0.f, 0.f};
  if constexpr (GATED) {
    const int row = tid % kMaxRows, grp = tid / kMaxRows;
    double s = 0.0;
    if (row < a.n_rows) {
#pragma unroll 4
      for (int p = grp; p < a.ssq_parts; p += kGroups) s += a.ssq[size_t(p) * a.n_rows + row];
    }
    row_part[grp * kMaxRows + row] = s;
  } else if (unit_live) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (unit_n + e >= a.n_out) continue;
      old[e] = a.resid[size_t(r) * a.n_out + unit_n + e];
      if (a.norm_w) nw[e] = ld_dyn(a.norm_w, a.norm_dtype, unit_n + e);
      if (a.bias) bias[e] = ld_dyn(a.bias, a.bias_dtype, unit_n + e);
    }
  }

  floatx4_t acc[G];
#pragma unroll
  for (int g = 0; g < G; ++g) acc[g] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](int slot) {
#pragma unroll
    for (int g = 0; g < G; ++g) acc[g] = mfma16(as_bf16x8(rw[slot][g]), as_bf16x8(rx[slot]), acc[g]);
  };
  int step = s0;
  for (; step + kAhead <= s1; step += kAhead) {
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      multiply(u);
      ask(u, step + kAhead + u);
    }
  }
#pragma unroll
  for (int u = 0; u < kAhead; ++u)
    if (step + u < s1) multiply(u);

#pragma unroll
  for (int g = 0; g < G; ++g) red[(wave * G + g) * 64 + lane] = acc[g];
  __syncthreads();
  if (wave != 0) return;                         // no barrier follows
  floatx4_t v[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    v[g] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < W; ++k) v[g] = v[g] + red[(k * G + g) * 64 + lane];
  }
  if constexpr (GATED) {
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < kGroups; ++k) s += row_part[k * kMaxRows + r];
    const float inv = 1.0f / sqrtf(float(s / double(a.n_in)) + a.eps);
    if (!unit_live) return;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (unit_n + e < a.n_out)
        a.y[size_t(r) * a.n_out + unit_n + e] = f32_to_bf16(gate_act(v[0][e] * inv, a.gate) * (v[G - 1][e] * inv));
  } else {
    float now[4];
    double sq = 0.0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      now[e] = old[e] + (v[0][e] + bias[e]);
      sq += double(now[e] * now[e]);             // (columns and rows past the last one are zeros)
    }
    if (unit_live) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (unit_n + e >= a.n_out) continue;
        const size_t idx = size_t(r) * a.n_out + unit_n + e;
        a.resid[idx] = now[e];
        a.xw[idx] = f32_to_bf16(now[e] * nw[e]);
      }
    }
    sq += __shfl_xor(sq, 16, 64);
    sq += __shfl_xor(sq, 32, 64);
    if (q == 0 && r < a.n_rows) a.ssq_out[size_t(tile) * a.n_rows + r] = sq;
  }
}

int check(const char *what, const void *x, const void *w, int n_rows, int n_out, int n_in) {
  SB_REQUIRE(x && w, "%s: null pointer", what);
  SB_REQUIRE(n_rows >= 0 && n_out > 0 && n_in > 0, "%s: bad sizes rows=%d out=%d in=%d", what, n_rows, n_out, n_in);
  SB_SUPPORT(n_rows <= kMaxRows, "%s: %d rows, at most %d", what, n_rows, kMaxRows);
  SB_SUPPORT(n_in % 8 == 0, "%s: inner size %d is not a multiple of 8", what, n_in);
  SB_SUPPORT((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) % 16 == 0, "%s: operands must be 16-byte aligned", what);
  // 32-bit byte offsets into X and into a stream of W
  SB_SUPPORT((unsigned long long)(n_rows + 1) * n_in * 2 < (1ull << 31) && (unsigned long long)n_in * 32 < (1ull << 31),
             "%s: inner size %d is too large", what, n_in);
  return SB_OK;
}

}  // namespace

extern "C" int sb_gemm_split_join_bf16(float *resid, void *xw, double *ssq, const void *norm_w, int norm_dtype, const void *x,
                                       const void *w, const void *bias, int bias_dtype, int n_rows, int n_out, int n_in,
                                       void *stream) {
  const int rc = check("sb_gemm_split_join_bf16", x, w, n_rows, n_out, n_in);
  if (rc != SB_OK) return rc;
  SB_REQUIRE(resid && xw && ssq, "sb_gemm_split_join_bf16: null pointer");
  SB_REQUIRE((!norm_w || sb::valid_dtype(norm_dtype)) && (!bias || sb::valid_dtype(bias_dtype)),
             "sb_gemm_split_join_bf16: unknown dtype");
  if (n_rows == 0) return SB_OK;
  SplitArgs a{};
  a.n_rows = n_rows, a.n_out = n_out, a.n_in = n_in, a.bias = bias, a.bias_dtype = bias_dtype;
  a.resid = resid, a.xw = (bf16_t *)xw, a.ssq_out = ssq, a.norm_w = norm_w, a.norm_dtype = norm_dtype;
  // eight waves of a block share a row block's k-steps, four where those are few (896: 3.7 us with four, 4.0 with eight;
  // 1,536: 5.0 and 4.6)
  const int blocks = (n_out + 15) / 16;
  if (n_in <= 1024)
    gemm_split_kernel<false, 4><<<blocks, 256, 0, (hipStream_t)stream>>>((const bf16_t *)x, (const bf16_t *)w, a);
  else
    gemm_split_kernel<false, 8><<<blocks, 512, 0, (hipStream_t)stream>>>((const bf16_t *)x, (const bf16_t *)w, a);
  return sb::check_launch("sb_gemm_split_join_bf16");
}

extern "C" int sb_gemm_split_gated_bf16(void *y, const void *x, const double *ssq, int ssq_parts, float eps, const void *w,
                                        int n_rows, int n_out, int n_in, int gate, void *stream) {
  const int rc = check("sb_gemm_split_gated_bf16", x, w, n_rows, n_out, n_in);
  if (rc != SB_OK) return rc;
  SB_REQUIRE(y && ssq && ssq_parts > 0, "sb_gemm_split_gated_bf16: null pointer");
  SB_SUPPORT(gate > SB_GATE_NONE && gate <= SB_GATE_RELU, "sb_gemm_split_gated_bf16: unknown gate activation %d", gate);
  if (n_rows == 0) return SB_OK;
  if (sb::tile_gated_pays(n_rows, n_out, n_in))
    return sb::tile_gated(y, x, ssq, ssq_parts, eps, w, n_rows, n_out, n_in, gate, stream);
  if (sb::rows_whole(n_rows, n_out, n_in, 1))          // blocks that keep the rows in LDS, where these fit
    return sb::rows_gated(y, x, ssq, ssq_parts, eps, w, n_rows, n_out, n_in, gate, stream);
  SplitArgs a{};
  a.n_rows = n_rows, a.n_out = n_out, a.n_in = n_in, a.ssq = ssq, a.ssq_parts = ssq_parts, a.eps = eps;
  a.y = (bf16_t *)y, a.gate = gate;
  gemm_split_kernel<true, 4><<<(n_out + 15) / 16, 256, 0, (hipStream_t)stream>>>((const bf16_t *)x, (const bf16_t *)w, a);
  return sb::check_launch("sb_gemm_split_gated_bf16");
}
