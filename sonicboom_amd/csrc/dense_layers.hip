// A prompt step through a run of like decoder layers in one call: pre-norm blocks of grouped-query
// attention with biases on q, k and v and a gated dense feed-forward, packed bfloat16 weights.
//
// Nothing here computes: it launches the kernels that the layers' parts launch one by one, with the
// same choices, in the same order, so the results have the same bits.  What it takes away is the
// host's share: a launch from Python costs 10 to 12 us with its checks, its allocation and the passing
// of twenty arguments, nine launches a layer, and a step of up to a few hundred rows took longer to
// launch than to run (0.5B sizes, 288 rows: 2.13 ms against 1.5 of kernels).
#include "common.h"

namespace {

constexpr int kFewRows = 64;            // rows that the weight-streaming kernels take in K slices
constexpr int kStreamMaxRows = 128;
// Blocks of four waves that a matrix must give the stream kernel.  A block streams its share of W at
// what one CU pulls, whatever the count of blocks, so fewer blocks than CUs only pay while the
// other kernel, which spreads K over the whole GPU, has more bytes to move than a block's share
// takes: gate/up pairs of 8,960 x 1,536 (140 blocks) 13 to 18 us against 18 to 29 at up to 64 rows,
// 11,008 x 2,048 (172 blocks) 19 to 25 against 25 to 34; 8,192 x 2,048 (128 blocks) 18 against 16,
// and 4,864 x 896 (76 blocks) 4 % slower in a whole decode step.  (Measured with four waves a block and more; matrices of 544 to 768
// tiles take three now, and are on this side of the line either way.)
constexpr int kStreamMinBlocks = 136;
constexpr int kStreamMinBlocksMoreRows = 192;        // for 65 to 128 rows

enum Product { kStream = 0, kSkinny = 1, kTiled = 2 };

}  // namespace

// The kernel that a whole bf16 product takes: 0 the one whose waves split the output features and share the rows
// through LDS (a wide packed matrix, up to 128 rows), 1 the one whose waves split K and which can cut K over the grid as
// well (up to 64 rows), 2 the tiled one.
extern "C" int sb_gemm_bf16_kernel(int n_rows, int n_out, int gated, int packed) {
  const long long wave_units = gated ? (n_out + 15) / 16 : (n_out + 31) / 32;
  Product which = packed && wave_units >= 4 * kStreamMinBlocks ? kStream : kSkinny;
  if (n_rows > kFewRows && which == kStream) {
    // 65 to 128 rows: the tiled kernel's 128 x 128 tiles do as well or better unless the
    // matrix is wide and their count leaves the last round over the 256 CUs nearly empty
    // (8,960 x 1,536 and 11,008 x 2,048 at 96 rows: 21 and 26 us tiled, 25 and 34 streamed)
    const int per = gated ? 64 : 128;
    const double rounds = ((n_out + per - 1) / per) / 256.0;
    const double whole = double((long long)rounds) < rounds ? double((long long)rounds + 1) : rounds;
    if (wave_units < 4 * kStreamMinBlocksMoreRows || whole / rounds < 1.4) which = kTiled;
  }
  if (n_rows <= kStreamMaxRows && which == kStream) return kStream;
  return n_rows <= kFewRows && which != kTiled ? kSkinny : kTiled;
}

namespace {

int whole_product(void *y, int y_dtype, const void *x, const void *w, const void *bias, const float *resid, int n_rows, int n_out,
                  int n_in, int gated, float *scratch, size_t scratch_floats, void *stream) {
  switch (sb_gemm_bf16_kernel(n_rows, n_out, gated, 1)) {
    case kStream: return sb_gemm_stream_bf16(y, y_dtype, x, w, bias, SB_F32, resid, n_rows, n_out, n_in, gated, 0, stream);
    case kSkinny:
      return sb_gemm_skinny_bf16(y, y_dtype, x, w, bias, SB_F32, resid, n_rows, n_out, n_in, gated, 1, scratch, scratch_floats, stream);
    default: return sb_gemm_mfma_bf16(y, y_dtype, x, w, bias, SB_F32, resid, n_rows, n_out, n_in, gated, 1, -1, stream);
  }
}

// K slices that the raw product of these sizes comes in (0: none of the kernels that cut K takes it)
int raw_slices(int n_rows, int n_out, int n_in) {
  if (n_rows <= kFewRows) return sb_gemm_stream_slices(n_rows, n_out, n_in, 0);
  const int s = sb_gemm_mfma_slices(n_rows, n_out, n_in, 1);
  return s > 1 ? s : 0;
}
int raw_product(float *part, const void *x, const void *w, int n_rows, int n_out, int n_in, void *stream) {
  if (n_rows <= kFewRows) return sb_gemm_stream_partial_bf16(part, x, w, n_rows, n_out, n_in, 0, stream);
  return sb_gemm_mfma_partial_bf16(part, x, w, n_rows, n_out, n_in, 1, stream);
}

#define SB_TRY(call)               \
  do {                             \
    const int rc_ = (call);        \
    if (rc_ != SB_OK) return rc_;  \
  } while (0)

// x += a w^T; then h = rmsnorm(x) * norm_w, where there is a norm
int join(const sb_dense_step &st, const void *a, const void *w, int n_in, const void *norm_w, int norm_dtype, float eps, void *stream) {
  const int t = st.n_rows, n = st.width, slices = raw_slices(t, n, n_in);
  if (slices && n % 4 == 0 && n <= sb_reduce_resid_norm_max_width()) {
    SB_TRY(raw_product(st.part, a, w, t, n, n_in, stream));
    return sb_reduce_resid_norm(norm_w ? st.h : nullptr, SB_BF16, st.x, st.part, slices, nullptr, 0, norm_w, norm_dtype, t, n, eps,
                                norm_w ? 1 : 0, stream);
  }
  SB_TRY(whole_product(st.x, SB_F32, a, w, nullptr, st.x, t, n, n_in, 0, st.part, st.part_floats, stream));
  return norm_w ? sb_rmsnorm(st.h, SB_BF16, st.x, norm_w, norm_dtype, nullptr, t, n, eps, stream) : SB_OK;
}

}  // namespace

// Floats that `part` of a step of these sizes must hold.
extern "C" size_t sb_dense_layers_floats(int n_rows, int width, int qkv_width, int q_width, int inner) {
  const size_t t = size_t(n_rows > 0 ? n_rows : 0);
  const auto sliced = [&](int n_out, int n_in) {
    const int s = raw_slices(n_rows, n_out, n_in);
    return size_t(s > 1 ? s : 1) * t * n_out;
  };
  // (whole products of few rows cut K for themselves: the gated one, and those that join rows wider than one block norms)
  const auto whole = [&](int n_out, int n_in, int gated) {
    return n_rows <= kFewRows ? sb_gemm_skinny_scratch(n_rows, n_out, n_in, gated) : size_t(0);
  };
  size_t most = sliced(qkv_width, width);
  const size_t others[5] = {sliced(width, q_width), sliced(width, inner), whole(inner, width, 1), whole(width, q_width, 0),
                            whole(width, inner, 0)};
  for (size_t o : others) most = o > most ? o : most;
  return most;
}

// The layers one after the other: x (the residual stream) in place, h = the first layer's norm of x on entry.
extern "C" int sb_dense_layers(const sb_dense_step *step, const sb_dense_layer *layers, int n_layers, void *stream) {
  SB_REQUIRE(step && (layers || n_layers == 0) && n_layers >= 0, "sb_dense_layers: null pointer");
  const sb_dense_step &st = *step;
  SB_REQUIRE(st.x && st.h && st.part && st.q && st.att && st.mid && st.attention && st.attention_error && st.row_pos && st.row_seq &&
                 st.page_table && st.tiles,
             "sb_dense_layers: null pointer");
  SB_REQUIRE(st.n_rows >= 0 && st.width > 0 && st.inner > 0 && st.heads_q > 0 && st.heads_kv > 0 && st.head_dim > 0 &&
                 st.heads_q % st.heads_kv == 0,
             "sb_dense_layers: bad sizes");
  const int t = st.n_rows, q_width = st.heads_q * st.head_dim, qkv_width = q_width + 2 * st.heads_kv * st.head_dim;
  SB_REQUIRE(st.part_floats >= sb_dense_layers_floats(t, st.width, qkv_width, q_width, st.inner), "sb_dense_layers: the workspace is too small");
  if (t == 0) return SB_OK;
  for (int i = 0; i < n_layers; ++i) {
    const sb_dense_layer &L = layers[i];
    SB_REQUIRE(L.qkv_w && L.out_w && L.gate_up_w && L.down_w && L.norm_w && L.k_cache && L.v_cache, "sb_dense_layers: null pointer");
    int slices = raw_slices(t, qkv_width, st.width);
    const float *bias = L.qkv_bias;
    if (slices) {
      SB_TRY(raw_product(st.part, st.h, L.qkv_w, t, qkv_width, st.width, stream));
    } else {
      SB_TRY(whole_product(st.part, SB_F32, st.h, L.qkv_w, bias, nullptr, t, qkv_width, st.width, 0, nullptr, 0, stream));
      slices = 1, bias = nullptr;
    }
    SB_TRY(sb_rope_kv_store_sized(st.q, SB_BF16, st.part, SB_F32, qkv_width, slices, bias, L.inv_freq, L.freq_factors, L.rot_dims,
                                  st.row_pos, st.row_seq, L.k_cache, L.v_cache, SB_BF16, st.page_table, st.max_pages, st.n_pages, t,
                                  st.heads_q, st.heads_kv, st.head_dim, st.head_dim, 1.0f, stream));
    const int rc = st.attention(st.att, st.q, L.k_cache, L.v_cache, st.page_table, st.max_pages, st.n_pages, st.row_pos, st.tiles,
                                st.n_tiles, st.heads_q, st.heads_kv, L.scale, L.window, st.tile_rows, st.row_groups, st.group_pages, 0, stream);
    if (rc != SB_OK) return sb::fail(rc, "%s", st.attention_error());
    SB_TRY(join(st, st.att, L.out_w, q_width, L.norm_w, L.norm_dtype, L.norm_eps, stream));
    SB_TRY(whole_product(st.mid, SB_BF16, st.h, L.gate_up_w, nullptr, nullptr, t, st.inner, st.width, L.gate, st.part, st.part_floats,
                         stream));
    SB_TRY(join(st, st.mid, L.down_w, st.inner, L.next_w, L.next_dtype, L.next_eps, stream));
  }
  return SB_OK;
}
