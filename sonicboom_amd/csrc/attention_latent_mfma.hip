// Latent attention on the matrix cores (bfloat16): the per-head products that carry queries into
// the latent space and results out of it, and attention over the cached latent rows.
//
// sb_head_product_bf16: out[t, a, :] = W[a] in[t, a, :], W[a] [n_out, n_in] (output-major).  A wave
// takes 16 rows of one head and 64 outputs; both operands go from global memory straight into
// MFMA 16x16x32 fragments (a lane's eight k are 16 consecutive bytes on either side), the result
// lands as four consecutive outputs of one row per lane.
//
// sb_latent_attention_bf16: all query heads read the same cached rows [c | r], so a block stages
// them once in LDS for 64 query columns.
// A decode step (a column is a head of the one row): half a page, 32 rows, at a time in two buffers that take turns,
// twice over: as it lies (a key's numbers consecutive: the A operand of S^T = K Q^T) and with the latent part turned (a
// number's keys consecutive: the A operand of O^T = C^T P^T).  Its eight waves run four tiles of 16 columns against it,
// two waves a tile.  The next half's rows are asked of memory before the current half's products start, wait in
// registers and go into the other buffer afterwards.  Softmax runs in the result layout of S^T (a lane holds 8 keys of
// one column; column maximum and sum over the four lane groups), P goes
// back in as the B operand of the second product without leaving registers: the keys of a
// 32-key step are taken in the order the first product left them, by V's fragment reads.
// A prompt step (a column is one of up to 16 consecutive rows of a head, four heads a block) has a kernel of its own below:
// measured against the form above on prompt rows, 16 heads, rows of 512 + 64 (us): 300 rows 66 -> 41, 1,000 223 -> 109,
// 4,001 1,129 -> 406 (690 TFLOP/s of the products it cannot do without), with a window of 512 327 -> 140; 20 heads of 256 + 32 at 4,001 rows
// 823 -> 340; 3 heads of 128 + 64 114 -> 64.
#include "mfma.h"

namespace {

constexpr int kThreads = 256;      // of the per-head product
constexpr int kAttnThreads = 512;  // of attention: eight waves,
constexpr int kColGroups = 4;      // four tiles of 16 query columns,
constexpr int kParts = 2;          // two waves a tile
constexpr int kPadK = 8;     // bf16 a key row is padded by in LDS
constexpr int kHalf = 32;    // keys of a step
constexpr int kVtStride = kHalf + 8;
constexpr float kLazy = 8.0f;   // how far (in powers of two) a score may pass the running maximum before it moves

template <bool GATED>
__global__ void __launch_bounds__(kThreads)
head_product_mfma_kernel(bf16_t *__restrict__ out, int out_stride, int out_hstride, const bf16_t *__restrict__ in,
                         int in_stride, int in_hstride, const bf16_t *__restrict__ w, const float *__restrict__ gate,
                         int gate_stride, int n_rows, int n_in, int n_out, int gate_per_head) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int a = blockIdx.y;
  const int t = blockIdx.x * 64 + wave * 16 + (lane & 15);      // this lane's row (B operand's column)
  const int o0 = blockIdx.z * 64;
  const int g = lane >> 4;
  const bf16_t *xin = in + size_t(min(t, n_rows - 1)) * in_stride + size_t(a) * in_hstride;
  const bf16_t *wa = w + size_t(a) * n_out * n_in;
  floatx4_t acc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  // four steps of 32 k at a time: their twenty loads go out together, then the sixteen products
  for (int k0 = 0; k0 < n_in; k0 += 128) {
    uint4 b[4], av[4][4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = k0 + 32 * u + 8 * g;
      const bool kin = k < n_in;                                 // n_in is a multiple of 8
      b[u] = ld16(xin + (kin ? k : 0), kin && t < n_rows);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int o = o0 + 16 * j + (lane & 15);
        av[u][j] = ld16(wa + size_t(min(o, n_out - 1)) * n_in + (kin ? k : 0), kin && o < n_out);
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] = mfma16(as_bf16x8(av[u][j]), as_bf16x8(b[u]), acc[j]);
  }
  if (t >= n_rows) return;
  // a lane holds four neighbouring outputs of its row: one 8-byte store where the row's layout allows
  const bool wide = (out_stride % 4 == 0) && (out_hstride % 4 == 0) && (reinterpret_cast<uintptr_t>(out) % 8 == 0);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int ob = o0 + 16 * j + 4 * g;
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] = acc[j][i];
      if (GATED && ob + i < n_out) {
        const float gv = gate[size_t(t) * gate_stride + (gate_per_head ? size_t(a) : size_t(a) * n_out + ob + i)];
        v[i] = v[i] * (1.0f / (1.0f + expf(-gv)));
      }
    }
    bf16_t *dst = out + size_t(t) * out_stride + size_t(a) * out_hstride + ob;
    if (wide && ob + 3 < n_out) {
      *reinterpret_cast<uint2 *>(dst) = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (ob + i < n_out) dst[i] = f32_to_bf16(v[i]);
    }
  }
}

// The same for many rows: a wave takes 16 RT rows against its 64 outputs, so that a fragment of W feeds RT products and one
// of the rows four (above: one and four, and W came in again for every 16 rows), 64 k a stage, the next stage's
// fragments asked for ahead of this one's products.  The same bits.
// What bounds it: the waves in flight (82 MB in 44 us are 0.4 of a copy's rate).  With RT 4 a stage is 32 k, so that with the next
// one's fragments a wave stays at 208 registers and a SIMD holds two; with 64 k a stage and its loads behind branches it took 348, one
// a SIMD.  Measured, 16 heads, rows of 16, 32 and 64 a wave (the first the kernel above), us: 128 to 512 numbers, 4,001 rows 79.7, 58.6, 43.8 (348
// registers: 51.4), 1,000 rows 22.8, 14.3, 14.0, 500 rows 12.7, 10.5, 8.4; 512 to 128 with a gate, 4,001 rows 92.7, 59.4, 44.7 (54.8),
// 3,000 rows 69.6, 48.9, 42.9, 2,000 rows with 32 31.3, with 64 27.3, 1,000 rows 26.5, 19.4, 27.4, 500 rows 15.5, 17.0, 24.1.
// (Alone, operands cold.  In a prompt of 4,001 rows, traced, 63 -> 54.9 and 54.7.)
template <bool GATED, int RT>
__global__ void __launch_bounds__(kThreads, 2)
head_product_rows_kernel(bf16_t *__restrict__ out, int out_stride, int out_hstride, const bf16_t *__restrict__ in,
                         int in_stride, int in_hstride, const bf16_t *__restrict__ w, const float *__restrict__ gate,
                         int gate_stride, int n_rows, int n_in, int n_out, int gate_per_head) {
  constexpr int kSteps = RT == 4 ? 1 : 2;    // of 32 k a stage
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int a = blockIdx.y, o0 = blockIdx.z * 64, g = lane >> 4;
  const int t0 = (blockIdx.x * 4 + wave) * (16 * RT) + (lane & 15);
  if ((blockIdx.x * 4 + wave) * (16 * RT) >= n_rows) return;      // uniform over the wave; no barrier in this kernel
  // Through descriptors (of the block's rows of this head, and of the head's W) rows, outputs and k past the last read as zeros on both
  // sides without a branch, and a load's address is one register.
  const int row0 = blockIdx.x * 4 * (16 * RT), rows_here = min(n_rows - row0, 4 * 16 * RT);
  const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16_t *>(in) + size_t(row0) * in_stride + size_t(a) * in_hstride, 0,
      (uint32_t(rows_here - 1) * uint32_t(in_stride) + uint32_t(n_in)) * 2u, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t *>(w) + size_t(a) * n_out * n_in, 0,
                                                                          uint32_t(n_out) * uint32_t(n_in) * 2u, 0x00020000);
  constexpr uint32_t kOutside = 0x80000000u;
  uint32_t x_at[RT], w_at[4];
#pragma unroll
  for (int i = 0; i < RT; ++i) x_at[i] = t0 + 16 * i < n_rows ? (uint32_t(t0 + 16 * i - row0) * uint32_t(in_stride) + 8u * g) * 2u : kOutside;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int o = o0 + 16 * j + (lane & 15);
    w_at[j] = o < n_out ? (uint32_t(o) * uint32_t(n_in) + 8u * g) * 2u : kOutside;
  }
  floatx4_t acc[RT][4];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  uint4 fx[2][kSteps][RT], fw[2][kSteps][4];
  auto ask = [&](int set, int k0) {
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
      const int k = k0 + 32 * u;
      const bool kin = k + 8 * g < n_in;     // n_in is a multiple of 8
#pragma unroll
      for (int i = 0; i < RT; ++i)
        fx[set][u][i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_x, int(kin ? x_at[i] + 2u * k : kOutside), 0, 0));
#pragma unroll
      for (int j = 0; j < 4; ++j)
        fw[set][u][j] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_w, int(kin ? w_at[j] + 2u * k : kOutside), 0, 0));
    }
  };
  auto multiply = [&](int set) {
#pragma unroll
    for (int u = 0; u < kSteps; ++u)
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = mfma16(as_bf16x8(fw[set][u][j]), as_bf16x8(fx[set][u][i]), acc[i][j]);
  };
  constexpr int kStage = 32 * kSteps;
  ask(0, 0);
  for (int k0 = 0; k0 < n_in; k0 += 2 * kStage) {
    if (k0 + kStage < n_in) ask(1, k0 + kStage);
    __builtin_amdgcn_sched_barrier(0);
    multiply(0);
    if (k0 + kStage >= n_in) break;
    if (k0 + 2 * kStage < n_in) ask(0, k0 + 2 * kStage);
    __builtin_amdgcn_sched_barrier(0);
    multiply(1);
  }
  const bool wide = (out_stride % 4 == 0) && (out_hstride % 4 == 0) && (reinterpret_cast<uintptr_t>(out) % 8 == 0);
  const bool gate4 = !gate_per_head && gate_stride % 4 == 0 && n_out % 4 == 0 && reinterpret_cast<uintptr_t>(gate) % 16 == 0;
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int t = t0 + 16 * i;
    if (t >= n_rows) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int ob = o0 + 16 * j + 4 * g;
      if (ob >= n_out) continue;
      float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
      if constexpr (GATED) {
        const float *gp = gate + size_t(t) * gate_stride + (gate_per_head ? size_t(a) : size_t(a) * n_out + ob);
        float gv[4];
        if (gate4) {
          const float4 four = *reinterpret_cast<const float4 *>(gp);
          gv[0] = four.x, gv[1] = four.y, gv[2] = four.z, gv[3] = four.w;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) gv[e] = gp[gate_per_head || ob + e >= n_out ? 0 : e];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] * (1.0f / (1.0f + expf(-gv[e])));
      }
      bf16_t *dst = out + size_t(t) * out_stride + size_t(a) * out_hstride + ob;
      if (wide && ob + 3 < n_out) {
        *reinterpret_cast<uint2 *>(dst) = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (ob + e < n_out) dst[e] = f32_to_bf16(v[e]);
      }
    }
  }
}

// KQ: steps of 32 over a latent row that the unrolled loops cover; NV: tiles of 16 over the latent part.
// A page is worked on in two halves of kHalf keys; LDS holds two halves at a time (the one the
// waves read and the one being written), each as key rows [kHalf][lk] and as turned latent rows
// [nv * 16][kVtStride].  Eight waves: a tile of 16 query columns belongs to two waves, which both
// work out its scores and weights and take half of the latent part's tiles each in the second
// product, so that a wave's accumulators and fragments leave room for two waves a SIMD.
template <int KQ, int NV>
__global__ void __launch_bounds__(kAttnThreads)
latent_attention_mfma_kernel(bf16_t *__restrict__ out, const bf16_t *__restrict__ q, const bf16_t *__restrict__ cache,
                             const int32_t *__restrict__ page_table, int max_pages, int n_pages_total,
                             const int32_t *__restrict__ row_pos, const int32_t *__restrict__ tiles, int heads, int rank,
                             int rot_dim, float scale, int window, int n_splits, float *__restrict__ part_o,
                             float *__restrict__ part_ml, int n_rows) {
  extern __shared__ __align__(16) unsigned char lds[];
  const int latent = rank + rot_dim;
  const int kq = (latent + 31) / 32, nv = (rank + 15) / 16;
  const int lk = kq * 32 + kPadK;                    // bf16 per staged key row
  const int ks_size = kHalf * lk, vt_size = nv * 16 * kVtStride;
  bf16_t *ks_base = reinterpret_cast<bf16_t *>(lds); // [2][kHalf][lk]
  bf16_t *vt_base = ks_base + 2 * ks_size;           // [2][nv * 16][kVtStride]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 15, g = lane >> 4;
  const int tile = int(gridDim.x) - 1 - int(blockIdx.x);
  const int row = tiles[4 * tile], seq = tiles[4 * tile + 2];
  const int group = wave / kParts, part = wave % kParts;       // the wave's tile of columns, and its share of the latent part
  const int nv_part = (nv + kParts - 1) / kParts;
  const int head = (blockIdx.y * kColGroups + group) * 16 + col;
  const bool wave_works = (blockIdx.y * kColGroups + group) * 16 < heads;
  const bool valid = head < heads;
  const int pos = row_pos[row];
  const int lo = (window > 0 && pos >= window) ? pos - window + 1 : 0;

  // the pads that staging never writes must not hold what multiplies to NaN
  for (int i = tid; i < 2 * kHalf * (lk - latent); i += kAttnThreads) {
    const int key = i / (lk - latent), e = i - key * (lk - latent);
    ks_base[key * lk + latent + e] = 0;
  }
  for (int b = 0; b < 2; ++b)
    for (int i = tid; i < (nv * 16 - rank) * kVtStride; i += kAttnThreads) vt_base[b * vt_size + rank * kVtStride + i] = 0;

  // this lane's query fragments: column (head), k = 32 kk + 8 g .. + 7
  uint4 qf[KQ];
  const bf16_t *qrow = q + (size_t(row) * heads + min(head, heads - 1)) * latent;
#pragma unroll
  for (int kk = 0; kk < KQ; ++kk) {
    const int k = 32 * kk + 8 * g;
    qf[kk] = ld16(qrow + (k < latent ? k : 0), valid && k < latent);      // latent is a multiple of 8
  }

  const float neg_inf = -__builtin_inff();
  const float scale2 = scale * 1.4426950408889634f;     // scores in units of ln 2: the weights are exp2
  float m_run = neg_inf, l_run = 0.0f;
  constexpr int NVP = (NV + kParts - 1) / kParts;
  floatx4_t o[NVP];
#pragma unroll
  for (int v = 0; v < NVP; ++v) o[v] = floatx4_t{0.f, 0.f, 0.f, 0.f};

  // staging: a half is kHalf rows of latent / 8 chunks of 16 bytes; thread (key = idx % kHalf, chunk = idx / kHalf)
  const int chunks = latent / 8;
  constexpr int kMaxStage = (KQ * 32 / 8 * kHalf + kAttnThreads - 1) / kAttnThreads;
  uint4 set_a[kMaxStage], set_b[kMaxStage];      // two halves on their way from memory to LDS
  int h_first = lo / kHalf, h_last = pos / kHalf;                       // halves count from the sequence's start
  if (n_splits > 1) {                                                   // this block's share of them
    const int per = (h_last - h_first + n_splits) / n_splits;
    h_first += int(blockIdx.z) * per;
    h_last = min(h_last, h_first + per - 1);
  }
  auto page_of = [&](int h) -> int {
    const int c = h / (SB_PAGE / kHalf);
    const int p = c < max_pages ? page_table[size_t(seq) * max_pages + c] : -1;
    return (p >= 0 && p < n_pages_total) ? p : -1;
  };
  auto load_half = [&](int h, uint4 (&staged)[kMaxStage]) {
    const int page = page_of(h);
    const bf16_t *src = cache + (size_t(max(page, 0)) * SB_PAGE + (h % (SB_PAGE / kHalf)) * kHalf) * latent;
#pragma unroll
    for (int it = 0; it < kMaxStage; ++it) {
      const int idx = tid + it * kAttnThreads;
      const int key = idx % kHalf, chunk = idx / kHalf;
      // (keys that the row does not see are staged as zeros: their slots may hold what another sequence left there, and a
      // weight of zero does not keep a NaN out of the sums)
      const int j = h * kHalf + key;
      staged[it] = ld16(src + size_t(key) * latent + 8 * min(chunk, chunks - 1), page >= 0 && chunk < chunks && j >= lo && j <= pos);
    }
  };
  // A thread holds eight numbers of one key; the turned copy wants a number's keys side by side.
  // Neighbouring lanes hold neighbouring keys of the same chunk, so a pair of lanes swaps half of
  // what it holds (two DPP moves inside the quad) and each writes four whole 32-bit words, (even
  // key, odd key) of one number each: the even lane numbers 0 to 3 of the chunk, the odd lane 4 to 7.
  // (Written as single 16-bit stores, two lanes a word, this step took as long as all the products.)
  auto store_half = [&](int b, const uint4 (&staged)[kMaxStage]) {
    bf16_t *ks = ks_base + b * ks_size;
    uint32_t *vt32 = reinterpret_cast<uint32_t *>(vt_base + b * vt_size);
    const bool even = (lane & 1) == 0;
#pragma unroll
    for (int it = 0; it < kMaxStage; ++it) {
      const int idx = tid + it * kAttnThreads;
      const int key = idx % kHalf, chunk = idx / kHalf;
      const uint4 st = staged[it];
      const uint32_t send0 = even ? st.z : st.x, send1 = even ? st.w : st.y;
      const uint32_t recv0 = uint32_t(__builtin_amdgcn_update_dpp(0, int(send0), 0xB1, 0xF, 0xF, true));   // quad_perm [1,0,3,2]
      const uint32_t recv1 = uint32_t(__builtin_amdgcn_update_dpp(0, int(send1), 0xB1, 0xF, 0xF, true));
      if (chunk >= chunks) continue;
      *reinterpret_cast<uint4 *>(ks + key * lk + 8 * chunk) = st;
      if (8 * chunk < rank) {                       // rank is a multiple of 8: a chunk lies inside or outside
        const uint32_t mine0 = even ? st.x : st.z, mine1 = even ? st.y : st.w;
        const uint32_t lo0 = even ? mine0 : recv0, hi0 = even ? recv0 : mine0;   // the even key's numbers, the odd key's
        const uint32_t lo1 = even ? mine1 : recv1, hi1 = even ? recv1 : mine1;
        const int d = 8 * chunk + (even ? 0 : 4);
        uint32_t *dst = vt32 + (d * kVtStride + (key & ~1)) / 2;
        dst[0 * (kVtStride / 2)] = (lo0 & 0xffffu) | (hi0 << 16);
        dst[1 * (kVtStride / 2)] = (lo0 >> 16) | (hi0 & 0xffff0000u);
        dst[2 * (kVtStride / 2)] = (lo1 & 0xffffu) | (hi1 << 16);
        dst[3 * (kVtStride / 2)] = (lo1 >> 16) | (hi1 & 0xffff0000u);
      }
    }
  };

  // Halves h (being worked on, in LDS buffer buf), h1 (on its way, in the set `held`) and h2 (asked for
  // now, into the set `free`): a half's loads go out two steps before its rows are stored, so that
  // they have a whole step of products and a step of stores to land.
  auto next_half = [&](int h) -> int {
    ++h;
    while (h <= h_last && page_of(h) < 0) ++h;        // pages that are not there hold no visible key
    return h;
  };
  int h = next_half(h_first - 1), h1 = h_last + 1;
  int buf = 0;
  if (h <= h_last) {
    load_half(h, set_a);
    store_half(0, set_a);
    h1 = next_half(h);
    if (h1 <= h_last) load_half(h1, set_a);
  }
  __syncthreads();                                    // the pads and the first half are written
  auto step = [&](uint4 (&held)[kMaxStage], uint4 (&free)[kMaxStage]) {
    const int h2 = h1 <= h_last ? next_half(h1) : h1;
    if (h2 <= h_last) load_half(h2, free);

    if (wave_works) {
      const bf16_t *ks = ks_base + buf * ks_size, *vt = vt_base + buf * vt_size;
      floatx4_t s[2] = {floatx4_t{0.f, 0.f, 0.f, 0.f}, floatx4_t{0.f, 0.f, 0.f, 0.f}};
      const bf16_t *kr = ks + col * lk + 8 * g;
#pragma unroll
      for (int kk = 0; kk < KQ; ++kk) {
        if (kk >= kq) continue;
#pragma unroll
        for (int t = 0; t < 2; ++t)
          s[t] = mfma16(as_bf16x8(*reinterpret_cast<const uint4 *>(kr + 16 * t * lk + 32 * kk)), as_bf16x8(qf[kk]), s[t]);
      }
      // s[t][i] = score of key kHalf h + 16 t + 4 g + i for this lane's column, in units of ln 2
      float mx = neg_inf;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int j = h * kHalf + 16 * t + 4 * g + i;
          const bool vis = valid && j >= lo && j <= pos;
          s[t][i] = vis ? s[t][i] * scale2 : neg_inf;
          mx = fmaxf(mx, s[t][i]);
        }
      mx = max_over_lane_groups(mx);
      // the maximum the sums are relative to moves only when a score passes it by kLazy (2^kLazy in
      // the weights, which float32 sums and bfloat16 weights carry easily): most steps then leave
      // the accumulators alone
      if (__any(mx > m_run + kLazy)) {
        const float m_new = fmaxf(m_run, mx);
        const float alpha = m_new == neg_inf ? 1.0f : __builtin_amdgcn_exp2f(m_run - m_new);   // 0 while nothing has been seen
        l_run *= alpha;
#pragma unroll
        for (int v = 0; v < NVP; ++v)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[v][i] *= alpha;
        m_run = m_new;
      }
      const float m_safe = m_run == neg_inf ? 0.0f : m_run;
      float sum = 0.0f;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s[t][i] = __builtin_amdgcn_exp2f(s[t][i] - m_safe);
          sum += s[t][i];
        }
      l_run += sum;
      const uint4 pf = make_uint4(pack_bf16(s[0][0], s[0][1]), pack_bf16(s[0][2], s[0][3]),
                                  pack_bf16(s[1][0], s[1][1]), pack_bf16(s[1][2], s[1][3]));
#pragma unroll
      for (int v = 0; v < NVP; ++v) {
        const int vg = part * nv_part + v;
        if (v >= nv_part || vg >= nv) continue;
        const bf16_t *vr = vt + (16 * vg + col) * kVtStride + 4 * g;
        const uint2 lo8 = *reinterpret_cast<const uint2 *>(vr);
        const uint2 hi8 = *reinterpret_cast<const uint2 *>(vr + 16);
        o[v] = mfma16(as_bf16x8(make_uint4(lo8.x, lo8.y, hi8.x, hi8.y)), as_bf16x8(pf), o[v]);
      }
    }
    // nobody reads the other buffer any more: its readers passed the barrier that ended the step before
    if (h1 <= h_last) store_half(buf ^ 1, held);
    __syncthreads();
    buf ^= 1;
    h = h1;
    h1 = h2;
  };
  while (h <= h_last) {
    step(set_a, set_b);
    if (h > h_last) break;
    step(set_b, set_a);
  }

  if (!wave_works) return;
  float l_tot = l_run + __shfl_xor(l_run, 16, 64);
  l_tot += __shfl_xor(l_tot, 32, 64);
  if (!valid) return;
  if (n_splits > 1) {               // unnormalized sums, with the maximum they are relative to, for the merge
    const size_t column = size_t(blockIdx.z) * n_rows * heads + size_t(row) * heads + head;
    float *po = part_o + column * rank;
#pragma unroll
    for (int v = 0; v < NVP; ++v) {
      const int vg = part * nv_part + v;
      if (v >= nv_part || vg >= nv) continue;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (16 * vg + 4 * g + i < rank) po[16 * vg + 4 * g + i] = o[v][i];
    }
    if (g == 0 && part == 0) {
      part_ml[2 * column] = m_run;
      part_ml[2 * column + 1] = l_tot;
    }
    return;
  }
  const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
  bf16_t *orow = out + (size_t(row) * heads + head) * rank;
#pragma unroll
  for (int v = 0; v < NVP; ++v) {
    const int vg = part * nv_part + v;
    if (v >= nv_part || vg >= nv) continue;
    const int d = 16 * vg + 4 * g;
    if (d + 3 < rank) {
      *reinterpret_cast<uint2 *>(orow + d) = make_uint2(pack_bf16(o[v][0] * inv, o[v][1] * inv),
                                                        pack_bf16(o[v][2] * inv, o[v][3] * inv));
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (d + i < rank) orow[d + i] = f32_to_bf16(o[v][i] * inv);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Prompt steps: a block takes a tile of up to 16 rows and four heads, 64 query columns, and a page of 64 keys a step.
// LDS is what bounds it: with 16 columns a wave every 1 KB that a wave reads of it feeds one product.  Here a wave has 32:
//   scores:  wave (cg, kt, kh) multiplies half kh of the numbers of keys 32 kt .. with the 32 columns of half cg of the
//            block, and hands half of the partial scores to the wave with the other numbers, whose sums it gets;
//   sums:    it adds up a quarter of the latent part, all 64 keys, for those 32 columns.
// The weights pass between the four waves of a half through LDS, relative to a maximum that they share.  Every page
// lies in LDS once, as it comes (a key's chunks of 16 bytes in an order in which neither reading meets a bank twice,
// loaded straight into LDS): the second product's operand, numbers by keys, is read with ds_read_b64_tr_b16, which hands a
// group of 16 lanes a block of four keys by 16 numbers turned.  Two pages take turns in two buffers.
// (The wave split by numbers, not by keys, keeps the queries in 72 registers instead of 144.  LDS is read through a
// vector type: reads of a struct type make the compiler wait for the next page's loads before the first of them.)
typedef short shortx4_t __attribute__((ext_vector_type(4)));
constexpr int kPageThreads = 512;

// The order of a key's chunks within each run of eight: bits 1, 2 and 3 of the key choose among the eight places, bit 0
// the half of the banks (a key is an odd number of runs long).  Sixteen keys read at one chunk, and four keys read at
// four neighbouring ones, all lie in different banks.
__device__ __forceinline__ int key_turn(int key) { return ((key & 2) << 1) | ((key & 4) >> 1) | ((key & 8) >> 3); }

// What the four waves of a half exchange lies in four regions of 2 KB (one a wave): first the partial scores a wave hands
// over, all of its region; then the column maxima of the wave that has read them, in its second half; then the weights of
// columns 8 w .. 8 w + 7 in its first (64 keys of a column, the chunks of eight keys turned by the column).
constexpr int kRegion = 2048;
template <int KQ>
constexpr int latent_pages_lds() { return 2 * SB_PAGE * KQ * 64 + 8 * kRegion; }

template <int KQ, int ND>
__global__ void __launch_bounds__(kPageThreads, 2)
latent_attention_pages_kernel(bf16_t *__restrict__ out, const bf16_t *__restrict__ q, const bf16_t *__restrict__ cache,
                              const int32_t *__restrict__ page_table, int max_pages, int n_pages_total,
                              const int32_t *__restrict__ row_pos, const int32_t *__restrict__ tiles, int heads, int rank,
                              int rot_dim, float scale, int window, int n_splits, float *__restrict__ part_o,
                              float *__restrict__ part_ml, int n_rows) {
  typedef __attribute__((address_space(3))) bf16x8_t *lds_ptr_t;
  typedef __attribute__((address_space(3))) shortx4_t *lds_tr_t;
  constexpr int CH = 4 * KQ;                          // chunks of a key in LDS (those past the row's end hold zeros)
  constexpr int kBuf = SB_PAGE * CH;
  extern __shared__ bf16x8_t lds_latent[];            // [2][SB_PAGE][CH], then the eight regions
  const int latent = rank + rot_dim;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cg = wave >> 2, kw = wave & 3, kt = kw & 1, kh = kw >> 1;
  const int c32 = lane & 31, r16 = lane & 15, h = lane >> 5;
  unsigned char *regions = reinterpret_cast<unsigned char *>(lds_latent + 2 * kBuf) + cg * 4 * kRegion;
  // the last tiles of a prompt see the most keys: they go first, so that the short ones fill the end
  const int tile = int(gridDim.x) - 1 - int(blockIdx.x);
  const int r0 = tiles[4 * tile], n_tile = tiles[4 * tile + 1], seq = tiles[4 * tile + 2];
  const int head = blockIdx.y * 4 + cg * 2 + (c32 >> 4);       // this lane's column: a head, and row r16 of the tile
  const bool valid = r16 < n_tile && head < heads;
  const int row = r0 + min(r16, n_tile - 1);
  const int pos0 = row_pos[r0];
  const int pos = pos0 + min(r16, n_tile - 1);        // a tile's rows are consecutive positions of one sequence
  const int lo = (window > 0 && pos >= window) ? pos - window + 1 : 0;
  const int lo_blk = (window > 0 && pos0 >= window) ? pos0 - window + 1 : 0;
  const int hi_blk = pos0 + n_tile - 1;
  const int lo_last = (window > 0 && hi_blk >= window) ? hi_blk - window + 1 : 0;      // the first key that every row sees

  bf16x8_t qf[KQ];
  const bf16_t *qrow = q + (size_t(row) * heads + min(head, heads - 1)) * latent;
#pragma unroll
  for (int i = 0; i < KQ; ++i) {
    const int k = 16 * (kh * KQ + i) + 8 * h;
    qf[i] = as_bf16x8(ld16(qrow + (k < latent ? k : 0), valid && k < latent));      // latent is a multiple of 8
  }
  const float neg_inf = -__builtin_inff();
  const float scale2 = scale * 1.4426950408889634f;
  float m_run = neg_inf, l_run = 0.f;
  floatx16_t o[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[d][i] = 0.f;

  int pg_first = lo_blk / SB_PAGE, pg_last = min(hi_blk / SB_PAGE, max_pages - 1);
  if (n_splits > 1) {
    const int per = (pg_last - pg_first + n_splits) / n_splits;
    pg_first += int(blockIdx.z) * per;
    pg_last = min(pg_last, pg_first + per - 1);
  }
  const int32_t *pt = page_table + size_t(seq) * max_pages;
  auto next_page = [&](int pg) {
    while (pg <= pg_last) {
      const int page = pt[pg];
      if (page >= 0 && page < n_pages_total) break;
      ++pg;
    }
    return pg;
  };
  const uint32_t page_bytes = uint32_t(SB_PAGE) * latent * 2;
  auto bring = [&](int pg, int buf) {
    // keys that no row of the tile sees come as zeros: their slots may hold what another sequence left there, and a weight
    // of zero does not keep a NaN out of the sums
    const int first_key = lo_blk - pg * SB_PAGE, last_key = hi_blk - pg * SB_PAGE;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16_t *>(cache + size_t(pt[pg]) * SB_PAGE * latent), 0, page_bytes, 0x00020000);
#pragma unroll
    for (int i = 0; i < CH / 8; ++i) {
      const int at = (wave * (CH / 8) + i) * 64;
      const int slot = at + lane, key = slot / CH, place = slot - key * CH;
      const int chunk = place ^ key_turn(key);                   // CH is a multiple of 8: the exchange stays in its run
      const bool in = 8 * chunk < latent && key >= first_key && key <= last_key;
      const uint32_t off = in ? uint32_t(key * latent + 8 * chunk) * 2 : page_bytes;      // past the end: zeros
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)(lds_latent) + buf * kBuf + at, 16, int(off), 0, 0, 0);
    }
  };
  auto met = [&]() {                     // what the waves have written to LDS is there for all of them, what they read is read
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto landed = [&]() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    met();
  };

  // where this lane reads: a key's chunk 2 (kh KQ + i) + h for the scores, four keys' halves of chunks for the sums (eight
  // chunks on a key's place repeats, so a few places do for all of them)
  const int key_s = 32 * kt + c32, key_v = 8 * h + ((lane >> 2) & 3);                 // of the first four of a group's eight keys
  const int chunk_v = 4 * ND * kw + 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);
  int at_s[4], at_v[2][2];
#pragma unroll
  for (int p = 0; p < 4; ++p) at_s[p] = key_s * CH + ((2 * (kh * KQ + p) + h) ^ key_turn(key_s));
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int p = 0; p < 2; ++p)
      at_v[t][p] = 2 * ((key_v + 4 * t) * CH + ((chunk_v + 4 * p) ^ key_turn(key_v + 4 * t))) + (lane & 1);
  float *give = reinterpret_cast<float *>(regions + kw * kRegion) + 4 * lane;
  float *take = reinterpret_cast<float *>(regions + (kw ^ 2) * kRegion) + 4 * lane;
  float *max_out = reinterpret_cast<float *>(regions + (kw ^ 2) * kRegion + 1024) + c32;
  const float *max_in = reinterpret_cast<float *>(regions + 1024) + c32;
  unsigned char *column = regions + (c32 >> 3) * kRegion + (c32 & 7) * 128;           // this lane's column of weights

  int pg = next_page(pg_first), buf = 0;
  if (pg <= pg_last) bring(pg, 0);
  landed();
  while (pg <= pg_last) {
    const int pg_next = next_page(pg + 1);
    if (pg_next <= pg_last) bring(pg_next, buf ^ 1);
    const bf16x8_t *page = lds_latent + buf * kBuf;

    floatx16_t part;
#pragma unroll
    for (int i = 0; i < 16; ++i) part[i] = 0.f;
#pragma unroll
    for (int i = 0; i < KQ; ++i) part = mfma32(page[at_s[i & 3] + 8 * (i >> 2)], qf[i], part);
    // part[i]: half the numbers of key 32 kt + 8 (i / 4) + 4 h + i % 4; of its 16 a lane keeps eight, keys 16 kh .. + 15
    floatx4_t keep[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const floatx4_t first = {part[4 * u], part[4 * u + 1], part[4 * u + 2], part[4 * u + 3]};
      const floatx4_t second = {part[8 + 4 * u], part[9 + 4 * u], part[10 + 4 * u], part[11 + 4 * u]};
      keep[u] = kh ? second : first;
      *reinterpret_cast<floatx4_t *>(give + 256 * u) = kh ? first : second;
    }
    met();
    float s[8];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const floatx4_t other = *reinterpret_cast<const floatx4_t *>(take + 256 * u);
#pragma unroll
      for (int i = 0; i < 4; ++i) s[4 * u + i] = (keep[u][i] + other[i]) * scale2;
    }
    if (!(pg * SB_PAGE + SB_PAGE - 1 <= pos0 && pg * SB_PAGE >= lo_last)) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int j = pg * SB_PAGE + 32 * kt + 16 * kh + 8 * (i >> 2) + 4 * h + (i & 3);
        s[i] = j >= lo && j <= pos ? s[i] : neg_inf;
      }
    }
    float mx = fmaxf(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])), fmaxf(fmaxf(s[4], s[5]), fmaxf(s[6], s[7])));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    *max_out = mx;                       // both halves of the wave write the same
    met();
    mx = fmaxf(fmaxf(max_in[0], max_in[kRegion / 4]), fmaxf(max_in[2 * kRegion / 4], max_in[3 * kRegion / 4]));
    // the maximum the sums are relative to moves only when a score passes it by kLazy (2^kLazy in the weights, which
    // float32 sums and bfloat16 weights carry easily); the four waves of a half see the same numbers
    const bool move = mx > m_run + kLazy;
    if (__any(move)) {
      const float alpha = move ? __builtin_amdgcn_exp2f(m_run - mx) : 1.f;      // 0 while nothing has been seen
      m_run = move ? mx : m_run;
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[d][i] *= alpha;
    }
    const float m_safe = m_run == neg_inf ? 0.f : m_run;
    float p[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) p[i] = __builtin_amdgcn_exp2f(s[i] - m_safe);
    l_run += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
#pragma unroll
    for (int u = 0; u < 2; ++u)
      *reinterpret_cast<shortx4_t *>(column + (((4 * kt + 2 * kh + u) ^ ((c32 >> 1) & 7)) * 16 + 8 * h)) =
          __builtin_bit_cast(shortx4_t, make_uint2(pack_bf16(p[4 * u], p[4 * u + 1]), pack_bf16(p[4 * u + 2], p[4 * u + 3])));
    met();
#pragma unroll
    for (int ks = 0; ks < SB_PAGE / 16; ++ks) {
      const bf16x8_t w = *reinterpret_cast<const bf16x8_t *>(column + ((2 * ks + h) ^ ((c32 >> 1) & 7)) * 16);
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        shortx4_t v[2];
#pragma unroll
        for (int t = 0; t < 2; ++t)
          v[t] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (lds_tr_t)(reinterpret_cast<shortx4_t *>(lds_latent) + 2 * buf * kBuf + at_v[t][d & 1] + 32 * ks * CH + 16 * (d >> 1)));
        const uint2 v0 = __builtin_bit_cast(uint2, v[0]), v1 = __builtin_bit_cast(uint2, v[1]);
        o[d] = mfma32(as_bf16x8(make_uint4(v0.x, v0.y, v1.x, v1.y)), w, o[d]);
      }
    }
    landed();
    pg = pg_next;
    buf ^= 1;
  }

  // the columns' sums of weights, over the halves of a wave and the four waves
  l_run += __shfl_xor(l_run, 32, 64);
  reinterpret_cast<float *>(regions + kw * kRegion)[c32] = l_run;
  met();
  const float *l4 = reinterpret_cast<float *>(regions) + c32;
  const float l_tot = (l4[0] + l4[kRegion / 4]) + (l4[2 * kRegion / 4] + l4[3 * kRegion / 4]);
  if (!valid) return;
  const float inv = n_splits > 1 ? 1.0f : l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
  const size_t to = size_t(row) * heads + head;
  const size_t split_to = size_t(blockIdx.z) * n_rows * heads + to;
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int at = 32 * (ND * kw + d) + 8 * u + 4 * h;       // four consecutive numbers; rank is a multiple of 8
      if (at >= rank) continue;
      const float v0 = o[d][4 * u] * inv, v1 = o[d][4 * u + 1] * inv, v2 = o[d][4 * u + 2] * inv, v3 = o[d][4 * u + 3] * inv;
      if (n_splits > 1) *reinterpret_cast<float4 *>(part_o + split_to * rank + at) = make_float4(v0, v1, v2, v3);
      else *reinterpret_cast<uint2 *>(out + to * rank + at) = make_uint2(pack_bf16(v0, v1), pack_bf16(v2, v3));
    }
  if (n_splits > 1 && kw == 0 && h == 0) {
    part_ml[2 * split_to] = m_run;
    part_ml[2 * split_to + 1] = l_tot;
  }
}

// out[column, :] = sum_s o_s 2^(m_s - M) / sum_s l_s 2^(m_s - M), M the largest m_s: the shares of
// a column's keys that n_splits blocks worked on, put together.  A block a column; the shares'
// weights 2^(m_s - M) wait in LDS, and a thread asks for eight shares of its numbers at a time.
constexpr int kMaxSplits = 512;

__global__ void __launch_bounds__(256)
latent_merge_kernel(bf16_t *__restrict__ out, const float *__restrict__ part_o, const float *__restrict__ part_ml,
                    int n_splits, size_t n_columns, int rank) {
  __shared__ float weight[kMaxSplits];
  __shared__ float wave_l[4];
  const size_t column = blockIdx.x;
  const int tid = threadIdx.x;
  float m = -__builtin_inff();
  for (int s = tid; s < n_splits; s += 256) m = fmaxf(m, part_ml[2 * (size_t(s) * n_columns + column)]);
  m = wave_max(m);
  if ((tid & 63) == 0) wave_l[tid >> 6] = m;
  __syncthreads();
  m = fmaxf(fmaxf(wave_l[0], wave_l[1]), fmaxf(wave_l[2], wave_l[3]));
  __syncthreads();
  float l = 0.0f;
  for (int s = tid; s < n_splits; s += 256) {
    const float ms = part_ml[2 * (size_t(s) * n_columns + column)];
    const float ws = ms > -__builtin_inff() ? exp2f(ms - m) : 0.0f;
    weight[s] = ws;
    l += part_ml[2 * (size_t(s) * n_columns + column) + 1] * ws;
  }
  l = wave_sum(l);
  if ((tid & 63) == 0) wave_l[tid >> 6] = l;
  __syncthreads();
  l = (wave_l[0] + wave_l[1]) + (wave_l[2] + wave_l[3]);
  const float inv = l > 0.0f ? 1.0f / l : 0.0f;
  for (int d = tid; d < rank; d += 256) {
    float acc = 0.0f;
    for (int s0 = 0; s0 < n_splits; s0 += 8) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        v[u] = part_o[(size_t(min(s0 + u, n_splits - 1)) * n_columns + column) * rank + d];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (s0 + u < n_splits) acc += v[u] * weight[s0 + u];
    }
    out[column * rank + d] = f32_to_bf16(acc * inv);
  }
}

template <int KQ, int NV>
int launch_attention(bf16_t *out, const bf16_t *q, const bf16_t *cache, const int32_t *page_table, int max_pages,
                     int n_pages_total, const int32_t *row_pos, const int32_t *tiles, int n_tiles, int heads, int rank,
                     int rot_dim, float scale, int window, int tile_rows, int n_splits, float *part_o, float *part_ml,
                     int n_rows, hipStream_t s) {
  const int latent = rank + rot_dim;
  if (tile_rows == 16) {
    constexpr int ND = NV / 8, lds_pages = latent_pages_lds<KQ>();
    static bool raised_pages = false;
    if (!raised_pages) {
      if (hipFuncSetAttribute((const void *)latent_attention_pages_kernel<KQ, ND>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              lds_pages) != hipSuccess)
        (void)hipGetLastError();
      raised_pages = true;
    }
    latent_attention_pages_kernel<KQ, ND><<<dim3(n_tiles, (heads + 3) / 4, n_splits), kPageThreads, lds_pages, s>>>(
        out, q, cache, page_table, max_pages, n_pages_total, row_pos, tiles, heads, rank, rot_dim, scale, window, n_splits,
        part_o, part_ml, n_rows);
    if (n_splits > 1)
      latent_merge_kernel<<<unsigned(size_t(n_rows) * heads), 256, 0, s>>>(out, part_o, part_ml, n_splits,
                                                                           size_t(n_rows) * heads, rank);
    return sb::check_launch("sb_latent_attention_bf16");
  }
  const int kq = (latent + 31) / 32, nv = (rank + 15) / 16;
  const size_t lds = 2 * (size_t(kHalf) * (kq * 32 + kPadK) + size_t(nv) * 16 * kVtStride) * sizeof(bf16_t);
  static bool raised = false;              // once per kernel of this shape: more dynamic LDS than the default allows
  if (!raised) {
    if (hipFuncSetAttribute((const void *)latent_attention_mfma_kernel<KQ, NV>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) != hipSuccess)
      (void)hipGetLastError();
    raised = true;
  }
  dim3 grid(n_tiles, (heads + kColGroups * 16 - 1) / (kColGroups * 16), n_splits);
  latent_attention_mfma_kernel<KQ, NV><<<grid, kAttnThreads, lds, s>>>(out, q, cache, page_table, max_pages, n_pages_total,
                                                                   row_pos, tiles, heads, rank, rot_dim, scale, window,
                                                                   n_splits, part_o, part_ml, n_rows);
  if (n_splits > 1)
    latent_merge_kernel<<<unsigned(size_t(n_rows) * heads), 256, 0, s>>>(out, part_o, part_ml, n_splits,
                                                                         size_t(n_rows) * heads, rank);
  return sb::check_launch("sb_latent_attention_bf16");
}

}  // namespace

// 1 when sb_head_product_bf16 takes these sizes and strides (all in elements).
extern "C" int sb_head_product_bf16_ok(int out_stride, int out_hstride, int in_stride, int in_hstride, int n_in) {
  (void)out_stride; (void)out_hstride;
  return n_in % 8 == 0 && in_stride % 8 == 0 && in_hstride % 8 == 0;
}

// out[t, a, o] = sum_i W[a][o][i] in[t, a, i] on the matrix cores; everything bfloat16, gate f32 or NULL
// (times sigmoid(gate[t * gate_stride + a * n_out + o])); in and W 16-byte aligned.
extern "C" int sb_head_product_gated_bf16(void *out, int out_stride, int out_hstride, const void *in, int in_stride,
                                          int in_hstride, const void *w, const float *gate, int gate_stride,
                                          int gate_per_head, int n_rows, int heads, int n_in, int n_out, void *stream);
extern "C" int sb_head_product_bf16(void *out, int out_stride, int out_hstride, const void *in, int in_stride,
                                    int in_hstride, const void *w, const float *gate, int gate_stride, int n_rows,
                                    int heads, int n_in, int n_out, void *stream) {
  return sb_head_product_gated_bf16(out, out_stride, out_hstride, in, in_stride, in_hstride, w, gate, gate_stride, 0, n_rows,
                                    heads, n_in, n_out, stream);
}

// The same with gate_per_head: the gate holds one number a head, gate[t * gate_stride + a], for all of the
// head's outputs.
extern "C" int sb_head_product_gated_bf16(void *out, int out_stride, int out_hstride, const void *in, int in_stride,
                                          int in_hstride, const void *w, const float *gate, int gate_stride,
                                          int gate_per_head, int n_rows, int heads, int n_in, int n_out, void *stream) {
  SB_REQUIRE(out && in && w, "sb_head_product_bf16: null pointer");
  SB_REQUIRE(n_rows >= 0 && heads > 0 && n_in > 0 && n_out > 0, "sb_head_product_bf16: bad sizes");
  SB_SUPPORT(sb_head_product_bf16_ok(out_stride, out_hstride, in_stride, in_hstride, n_in),
             "sb_head_product_bf16: inner size and strides must be multiples of 8");
  SB_SUPPORT((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(w)) % 16 == 0,
             "sb_head_product_bf16: operands must be 16-byte aligned");
  SB_SUPPORT(heads <= 65535 && (n_out + 63) / 64 <= 65535, "sb_head_product_bf16: too many heads or outputs");
  if (n_rows == 0) return SB_OK;
  const unsigned out_tiles = (n_out + 63) / 64;
  hipStream_t s = (hipStream_t)stream;
#define SB_HEAD_PRODUCT(KERNEL, ROWS)                                                                                             \
  KERNEL<<<dim3((n_rows + ROWS - 1) / ROWS, heads, out_tiles), kThreads, 0, s>>>((bf16_t *)out, out_stride, out_hstride,          \
                                                                                 (const bf16_t *)in, in_stride, in_hstride,       \
                                                                                 (const bf16_t *)w, gate, gate_stride, n_rows,    \
                                                                                 n_in, n_out, gate_per_head)
  // rows of a wave: the most (64, 32, 16) that give a block for every CU (see the kernel's figures)
  const auto blocks = [&](int rows) { return (long long)((n_rows + rows - 1) / rows) * heads * out_tiles; };
  // (those kernels address a block's rows and a head's W with 32-bit byte offsets)
  const bool reach = (long long)in_stride * 256 * 2 < (1ll << 31) && (long long)n_out * n_in * 2 < (1ll << 31);
  const int rt = !reach ? 1 : blocks(256) >= sb::cu_count() ? 4 : blocks(128) >= sb::cu_count() ? 2 : 1;
  if (gate) {
    if (rt == 4) SB_HEAD_PRODUCT((head_product_rows_kernel<true, 4>), 256);
    else if (rt == 2) SB_HEAD_PRODUCT((head_product_rows_kernel<true, 2>), 128);
    else SB_HEAD_PRODUCT(head_product_mfma_kernel<true>, 64);
  } else {
    if (rt == 4) SB_HEAD_PRODUCT((head_product_rows_kernel<false, 4>), 256);
    else if (rt == 2) SB_HEAD_PRODUCT((head_product_rows_kernel<false, 2>), 128);
    else SB_HEAD_PRODUCT(head_product_mfma_kernel<false>, 64);
  }
#undef SB_HEAD_PRODUCT
  return sb::check_launch("sb_head_product_bf16");
}

// The height of the runs of rows (`tiles`) that a prompt step's launch takes.
extern "C" int sb_latent_attention_tile_rows(void) { return 16; }

// 1 when sb_latent_attention_bf16 takes these sizes.
extern "C" int sb_latent_attention_bf16_ok(int rank, int rot_dim) {
  return rank > 0 && rot_dim >= 0 && rank % 8 == 0 && rot_dim % 8 == 0 && rank + rot_dim <= 576 && rank <= 512;
}

// Attention over cached latent rows on the matrix cores, everything bfloat16 (see the head of the
// file).  tiles int32 [n_tiles, 4] = (first row, rows, sequence, 0): runs of up to tile_rows
// consecutive rows of one sequence; tile_rows 16 for a prompt step, 1 for a step of single rows
// (a wave then takes 16 heads of a row).  out [n_rows, heads, rank], q [n_rows, heads, rank + rot_dim].
// n_splits > 1: the keys of every tile are shared out over that many blocks, whose unnormalized sums
// go through part_o (f32 [n_splits, n_rows, heads, rank]) and part_ml (f32 [n_splits, n_rows, heads, 2])
// and are put together by a second kernel: for steps of few rows over many keys.
extern "C" int sb_latent_attention_bf16(void *out, const void *q, const void *cache, const int32_t *page_table,
                                        int max_pages, int n_pages_total, const int32_t *row_pos, const int32_t *tiles,
                                        int n_tiles, int heads, int rank, int rot_dim, float scale, int window,
                                        int tile_rows, int n_splits, float *part_o, float *part_ml, int n_rows,
                                        void *stream) {
  SB_REQUIRE(out && q && cache && page_table && row_pos && tiles, "sb_latent_attention_bf16: null pointer");
  SB_REQUIRE(n_tiles >= 0 && heads > 0 && max_pages > 0 && n_pages_total > 0 && window >= 0,
             "sb_latent_attention_bf16: bad sizes");
  SB_REQUIRE(tile_rows == 16 || tile_rows == 1, "sb_latent_attention_bf16: tiles of 16 rows or of one");
  SB_REQUIRE(n_splits >= 1 && n_splits <= kMaxSplits && n_rows >= 0 && (n_splits == 1 || (part_o && part_ml)),
             "sb_latent_attention_bf16: shares of the keys need their scratch");
  SB_SUPPORT(sb_latent_attention_bf16_ok(rank, rot_dim), "sb_latent_attention_bf16: a latent row of %d + %d is not taken",
             rank, rot_dim);
  SB_SUPPORT((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(cache) | reinterpret_cast<uintptr_t>(out)) % 16 == 0,
             "sb_latent_attention_bf16: operands must be 16-byte aligned");
  if (n_tiles == 0) return SB_OK;
  hipStream_t s = (hipStream_t)stream;
  const int kq = (rank + rot_dim + 31) / 32, nv = (rank + 15) / 16;
#define SB_GO(KQ, NV)                                                                                              \
  return launch_attention<KQ, NV>((bf16_t *)out, (const bf16_t *)q, (const bf16_t *)cache, page_table, max_pages,    \
                                  n_pages_total, row_pos, tiles, n_tiles, heads, rank, rot_dim, scale, window, tile_rows,  \
                                  n_splits, part_o, part_ml, n_rows, s)
  if (kq <= 6 && nv <= 8) SB_GO(6, 8);
  if (kq <= 10 && nv <= 16) SB_GO(10, 16);
  SB_GO(18, 32);
#undef SB_GO
}
