// Latent attention of prompts with keys and values built (bfloat16).
//
// In the latent's space (attention_latent_mfma.hip) a pair of positions costs 2 rank + rot_dim multiply-adds a head; with a
// head's key [W_uk c | r] and value W_uv c built it costs dim + rot_dim + vdim (512, 64, 128, 128: 1,088 against 320), and
// building them dim + vdim times rank a key and head, once a step.  A step with many rows a key is far ahead with them:
//   sb_built_gather   the latents c of the pages that the step's rows see, side by side as rows of a product;
//   (the tiled product with [W_uk; W_uv] stacked: a row per key, all heads' keys, then all heads' values)
//   sb_built_attention  softmax attention of the queries' plain and rotated parts over [built key | r of the cached row]
//                       and the built values, times the sigmoid of the output gate.
// Nothing of it is kept after the step's layer.  Measured, 16 heads, 4,001 rows (us): per-head products and attention in the latent's space
// 455, here 165 (gathering 8, building 29, attention 118), 2,048 rows 203 and 79, 300 rows 60.7 and 29.3; a prompt of 4,001 rows of the
// second design 5,490 -> 4,236.
#include "mfma.h"

namespace {

constexpr int kRows = 128;          // rows of a tile: four waves of 32
constexpr float kLazyMax = 8.0f;    // how far (in powers of two) a score may pass the running maximum before it moves

// pages int32 [n][4] = (sequence, page of the sequence, first key, end of the keys): block p writes the 64 rows p * 64 ..
// of out [n * 64][rank], keys outside [first, end) and pages that are not there as zeros.
__global__ void __launch_bounds__(256)
built_gather_kernel(bf16_t *__restrict__ out, const bf16_t *__restrict__ cache, const int32_t *__restrict__ page_table, int max_pages,
                    int n_pages_total, const int32_t *__restrict__ pages, int rank, int latent) {
  const int seq = pages[4 * blockIdx.x], pg = pages[4 * blockIdx.x + 1];
  const int first = pages[4 * blockIdx.x + 2], end = pages[4 * blockIdx.x + 3];
  const int page = pg < max_pages ? page_table[size_t(seq) * max_pages + pg] : -1;
  const bool there = page >= 0 && page < n_pages_total;
  const bf16_t *src = cache + size_t(there ? page : 0) * SB_PAGE * latent;
  bf16_t *dst = out + size_t(blockIdx.x) * SB_PAGE * rank;
  const int chunks = rank / 8;
  for (int i = threadIdx.x; i < SB_PAGE * chunks; i += 256) {
    const int key = i / chunks, c = i - key * chunks;
    const uint4 v = ld16(src + size_t(key) * latent + 8 * c, there && key >= first && key < end);
    *reinterpret_cast<uint4 *>(dst + size_t(i) * 8) = v;
  }
}

// Where chunk `chunk` (16 bytes) of key `key` lies among the key's CH chunks in LDS.  Keys and rotated parts are read sixteen
// keys at one chunk, which meet every bank once; a value chunk four keys at four neighbouring ones (ds_read_b64_tr_b16).
template <int CH>
__device__ __forceinline__ constexpr int key_turned(int key) {
  return CH == 16 ? key & 15 : (key >> 1) & 7;
}
__device__ __forceinline__ constexpr int value_turned(int key) { return (key & 3) << 2; }

// Whether eight bfloat16 numbers are finite: one to the lowest bit of an exponent of ones carries into the sign's place.
__device__ __forceinline__ bool finite(bf16x8_t v) {
  const uint4 w = __builtin_bit_cast(uint4, v);
  const auto past = [](uint32_t u) { return (u & 0x7f807f80u) + 0x00800080u; };
  return ((past(w.x) | past(w.y) | past(w.z) | past(w.w)) & 0x80008000u) == 0;
}

struct BuiltArgs {
  bf16_t *out;                      // [rows][heads][VD]
  const bf16_t *q_plain;            // [rows][heads][DP]
  const bf16_t *q_rot;              // rotated part of row r, head a at (r * heads + a) * q_rot_stride
  int q_rot_stride;
  const bf16_t *built;              // [keys][built_stride]: keys of head a at a * DP, values at heads * DP + a * VD
  int built_stride;
  const bf16_t *cache;              // rows [c | r]: r behind the first `rank` numbers
  int rank, latent;
  const int32_t *page_table;
  int max_pages, n_pages_total;
  const int32_t *tiles;             // [n][8] = (first row, rows <= 128, sequence, built row of the sequence's key 0, position of the first row, ..)
  int heads;
  float scale2;                     // scale * log2(e): scores in units of ln 2
  int window;
  const float *gate;                // f32 or NULL
  int gate_stride, gate_per_head;
};

// A block takes a tile of up to 128 consecutive rows of one sequence and one head; four waves, 32 rows each, take every second
// page of 64 keys, four the others, and their sums meet in LDS.  A page: S^T = K Q^T and O^T = V^T P with MFMA 32x32x16, a lane holding one row's scores.  The order in which the first product
// leaves a lane its keys is the order in which the second one asks for values, so P stays in registers.  Keys, rotated parts
// and values of a page lie in LDS once, loaded straight into it, two buffers in turn (for either half of the waves); the values,
// rows of a key each, are read turned.
// What bounds it: a turn of two pages takes 2.6 to 2.9 us, its products 1.2 of them; fragments from LDS (320 KB a turn) and the
// exponentials fall between the products of the waves that share a SIMD instead of beside them, and a block costs some 8 us beside
// its turns.  4,001 rows of 16 heads 118 us (695 TFLOP/s), 2,048 rows 55, 300 rows 15.4 (14.6 without the look at values on the diagonal), 8,000
// rows of 32 heads 750 (875).  Blocks of four waves that take every page, two a CU: 142, 75, 18.5 and 621 where these took 125, 54, 15.5 and
// 640, as a long run's pages come one after the other.
// Which blocks: the block number counts heads fastest, so that a multiple of eight heads has a head's blocks on one die, whose
// L2 then holds its keys and values.
template <int DP, int RD, int VD>
__global__ void __launch_bounds__(512, 2)
built_attention_kernel(BuiltArgs a) {
  typedef __attribute__((address_space(3))) bf16x8_t *lds_ptr_t;
  typedef short shortx4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) shortx4_t *lds_tr_t;
  constexpr int CK = DP / 8, CR = RD / 8, CV = VD / 8;           // chunks of a key
  constexpr int kK = SB_PAGE * CK, kR = SB_PAGE * CR, kV = SB_PAGE * CV, kBuf = kK + kR + kV;
  constexpr int kSteps = (DP + RD) / 16, DT = VD / 32;
  static_assert(DT % 2 == 0 && (DT * 8 + 2) * 2 * 256 * 4 <= 4 * kBuf * 16, "halves to exchange, and room for them");
  static_assert((CK == 8 || CK == 16) && (CR == 8 || CR == 16) && CV == 16, "sizes that the orders in LDS know");
  extern __shared__ bf16x8_t lds_built[];                        // [2 halves of the waves][2][keys | rotated parts | values]
  const int lane = threadIdx.x & 63, wave8 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = wave8 >> 2, wave = wave8 & 3;
  const int tile = int(blockIdx.x) / a.heads, head = int(blockIdx.x) - tile * a.heads;
  const int row0 = a.tiles[8 * tile], n_tile = a.tiles[8 * tile + 1], seq = a.tiles[8 * tile + 2], key0 = a.tiles[8 * tile + 3];
  const int n = lane & 31, h = lane >> 5;
  const int n_wave = min(n_tile - 32 * wave, 32);                // this wave's rows (none: it only loads)
  const bool col_ok = n < n_wave;
  const int row = row0 + (col_ok ? 32 * wave + n : 0);
  // a tile's rows are consecutive positions
  const int pos_first = a.tiles[8 * tile + 4], pos_last = pos_first + n_tile - 1;
  const int lo_of_first = (a.window > 0 && pos_first >= a.window) ? pos_first - a.window + 1 : 0;
  const int lo_of_last = (a.window > 0 && pos_last >= a.window) ? pos_last - a.window + 1 : 0;      // the first key that every row sees
  const int wave_first = pos_first + 32 * wave, wave_last = wave_first + n_wave - 1;
  const int wave_lo = (a.window > 0 && wave_first >= a.window) ? wave_first - a.window + 1 : 0;
  const int wave_lo_last = (a.window > 0 && wave_last >= a.window) ? wave_last - a.window + 1 : 0;
  const int pos = wave_first + n;
  const int col_pos = col_ok ? pos : -1;
  const int col_lo = (a.window > 0 && pos >= a.window) ? pos - a.window + 1 : 0;

  bf16x8_t qf[kSteps];
  {
    const bf16_t *qp = a.q_plain + (size_t(row) * a.heads + head) * DP, *qr = a.q_rot + (size_t(row) * a.heads + head) * a.q_rot_stride;
#pragma unroll
    for (int s = 0; s < kSteps; ++s)
      qf[s] = as_bf16x8(ld16(16 * s < DP ? qp + 16 * s + 8 * h : qr + 16 * s - DP + 8 * h, col_ok));
  }
  floatx16_t o[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[d][i] = 0.f;
  float m_run = -__builtin_inff(), l_run = 0.f;

  const int32_t *pt = a.page_table + size_t(seq) * a.max_pages;
  const int pg_lo = lo_of_first / SB_PAGE, pg_hi = min(pos_last / SB_PAGE, a.max_pages - 1);
  auto there = [&](int pg) {                       // (uniform over a wave; pages that are not there hold no visible key)
    if (pg > pg_hi) return false;
    const int page = pt[pg];
    return page >= 0 && page < a.n_pages_total;
  };
  // A wave's loads of a page (64 chunks each): every fourth of the keys', rotated parts' and values'.  The turn of a lane's
  // key is the same for all of its loads of a kind, which lie a constant count of keys apart.
  const uint32_t row_bytes = uint32_t(a.built_stride) * 2, latent_bytes = uint32_t(a.latent) * 2;
  uint32_t off_k, off_r, off_v;
  {
    const int kk = wave * (64 / CK) + lane / CK, kr = wave * (64 / CR) + lane / CR, kv = wave * (64 / CV) + lane / CV;
    off_k = uint32_t(kk) * row_bytes + uint32_t((lane % CK) ^ key_turned<CK>(kk)) * 16 + uint32_t(head * DP) * 2;
    off_r = uint32_t(kr) * latent_bytes + uint32_t((lane % CR) ^ key_turned<CR>(kr)) * 16 + uint32_t(a.rank) * 2;
    off_v = uint32_t(kv) * row_bytes + uint32_t((lane % CV) ^ value_turned(kv)) * 16 + uint32_t(a.heads * DP + head * VD) * 2;
  }
  auto bring = [&](int pg, int buf) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16_t *>(a.built + size_t(key0 + pg * SB_PAGE) * a.built_stride), 0, SB_PAGE * row_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_c = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16_t *>(a.cache + size_t(pt[pg]) * SB_PAGE * a.latent), 0, SB_PAGE * latent_bytes, 0x00020000);
    lds_ptr_t to = (lds_ptr_t)(lds_built) + (2 * half + buf) * kBuf + wave * 64;
#pragma unroll
    for (int i = 0; i < CK / 4; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, to + 256 * i, 16, int(off_k), int(uint32_t(i * (256 / CK)) * row_bytes), 0, 0);
#pragma unroll
    for (int i = 0; i < CR / 4; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_c, to + kK + 256 * i, 16, int(off_r), int(uint32_t(i * (256 / CR)) * latent_bytes), 0, 0);
#pragma unroll
    for (int i = 0; i < CV / 4; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, to + kK + kR + 256 * i, 16, int(off_v), int(uint32_t(i * (256 / CV)) * row_bytes), 0, 0);
  };
  auto landed = [&]() __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // where this lane reads: key n of a score tile, chunk 2 s + h; keys 4 h + .. of a value quartet, in units of 8 bytes
  const int at_k = n * CK + (h ^ key_turned<CK>(n)), at_r = kK + n * CR + (h ^ key_turned<CR>(n));
  const int key_v = 4 * h + ((lane >> 2) & 3);
  const int at_v = 2 * (kK + kR + key_v * CV + ((2 * ((lane >> 4) & 1) + ((lane >> 1) & 1)) ^ value_turned(key_v))) + (lane & 1);

  int buf = 0;
  bool have = there(pg_lo + half);
  if (have) bring(pg_lo + half, 0);
  landed();
  for (int pg0 = pg_lo; pg0 <= pg_hi; pg0 += 2) {            // the same count of turns for all waves
    const int pg = pg0 + half;
    const bool have_next = there(pg + 2);
    if (have_next) bring(pg + 2, buf ^ 1);
    const int page_pos = pg * SB_PAGE;
    bf16x8_t *page = lds_built + (2 * half + buf) * kBuf;
    if ((pg0 + 2) * SB_PAGE - 1 > pos_first || pg0 * SB_PAGE < lo_of_last) {
      // (the pages on the diagonal and at a window's edge) a weight of zero does not keep a NaN or an infinity out of the sums.
      // Values of keys that no row of the tile sees go to zero; so do those of a key that some rows see and that hold a number that is not
      // finite, and the key becomes a NaN, which the weights of the rows that see it take on.
      const bf16x8_t zero = as_bf16x8(make_uint4(0u, 0u, 0u, 0u));
      for (int i = threadIdx.x & 255; have && i < kV; i += 256) {
        const int key = i / CV, j = page_pos + key;
        if (j > pos_last || j < lo_of_first) {
          page[kK + kR + i] = zero;
        } else if ((j > pos_first || j < lo_of_last) && !finite(page[kK + kR + i])) {
          page[kK + kR + i] = zero;
          page[key * CK] = as_bf16x8(make_uint4(0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u));
        }
      }
      __syncthreads();
    }
    if (have && page_pos <= wave_last && page_pos + SB_PAGE - 1 >= wave_lo && n_wave > 0) {
      floatx16_t s[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        floatx16_t acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
        for (int k = 0; k < kSteps; ++k)
          acc = mfma32(16 * k < DP ? page[(at_k ^ (2 * k)) + 32 * t * CK]
                                   : page[kK + ((at_r - kK) ^ (2 * (k - DP / 16))) + 32 * t * CR], qf[k], acc);
        s[t] = acc;
      }
      __builtin_amdgcn_sched_group_barrier(0x100, kSteps, 0);
#pragma unroll
      for (int k = 0; k < kSteps; ++k) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, kSteps, 0);
      __builtin_amdgcn_sched_barrier(0);
      // s[t][8 j + 4 u + e]: key 32 t + 16 j + 8 u + 4 h + e of the page
      if (!(page_pos + SB_PAGE - 1 <= wave_first && page_pos >= wave_lo_last)) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int j = page_pos + 32 * t + 8 * (i >> 2) + 4 * h + (i & 3);
            s[t][i] = (j <= col_pos && j >= col_lo) ? s[t][i] : -__builtin_inff();
          }
      }
      float mx = -__builtin_inff();
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[t][i]);
      {
        const uint32_t u = __builtin_bit_cast(uint32_t, mx);
        const auto p = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        const uint32_t p0 = p[0], p1 = p[1];
        mx = fmaxf(__builtin_bit_cast(float, p0), __builtin_bit_cast(float, p1)) * a.scale2;
      }
      // the maximum the sums are relative to moves only when a score passes it by kLazyMax
      const bool move = mx > m_run + kLazyMax;
      const float m_new = move ? mx : m_run;
      const float m_use = m_new == -__builtin_inff() ? 0.f : m_new;
      const float alpha = move ? __builtin_amdgcn_exp2f(m_run - m_use) : 1.f;      // m_run = -inf gives 0
      float sum = 0.f;
      uint4 pb[2][2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        float p[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          p[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t][i], a.scale2, -m_use));
          sum += p[i];
        }
#pragma unroll
        for (int j = 0; j < 2; ++j)
          pb[t][j] = make_uint4(pack_bf16(p[8 * j + 0], p[8 * j + 1]), pack_bf16(p[8 * j + 2], p[8 * j + 3]),
                                pack_bf16(p[8 * j + 4], p[8 * j + 5]), pack_bf16(p[8 * j + 6], p[8 * j + 7]));
      }
      l_run = l_run * alpha + sum;
      m_run = m_new;
      if (__any(move)) {
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[d][i] *= alpha;
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        floatx16_t acc = o[d];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            shortx4_t v[2];
#pragma unroll
            for (int u = 0; u < 2; ++u)
              v[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                  (lds_tr_t)(reinterpret_cast<shortx4_t *>(lds_built) + 2 * (2 * half + buf) * kBuf + ((at_v - 2 * (kK + kR)) ^ (8 * d)) + 2 * (kK + kR) +
                             2 * (32 * t + 16 * j + 8 * u) * CV));
            const uint2 v0 = __builtin_bit_cast(uint2, v[0]), v1 = __builtin_bit_cast(uint2, v[1]);
            acc = mfma32(as_bf16x8(make_uint4(v0.x, v0.y, v1.x, v1.y)), as_bf16x8(pb[t][j]), acc);
          }
        o[d] = acc;
      }
    }
    landed();
    have = have_next;
    buf ^= 1;
  }
  float l = l_run;
  {
    const uint32_t u = __builtin_bit_cast(uint32_t, l);
    const auto p = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    const uint32_t p0 = p[0], p1 = p[1];
    l = __builtin_bit_cast(float, p0) + __builtin_bit_cast(float, p1);
  }
  // the gate of the numbers that this lane will finish, asked for ahead of the exchange
  const int d0 = half * (DT / 2) * 32 + 4 * h;
  const float *grow = a.gate ? a.gate + size_t(row) * a.gate_stride + (a.gate_per_head ? head : head * VD + d0) : nullptr;
  const bool gate4 = !a.gate_per_head && a.gate_stride % 4 == 0 && reinterpret_cast<uintptr_t>(a.gate) % 16 == 0;
  floatx4_t gate[DT / 2 * 4];
  if (a.gate) {
#pragma unroll
    for (int u = 0; u < DT / 2 * 4; ++u) {
      if (gate4) gate[u] = *reinterpret_cast<const floatx4_t *>(grow + 8 * u);
      else
#pragma unroll
        for (int e = 0; e < 4; ++e) gate[u][e] = grow[a.gate_per_head ? 0 : 8 * u + e];
    }
  }
  // the two halves of the waves: each gives the other half of its tiles of numbers and finishes the rest
  constexpr int DH = DT / 2;
  float *mine = reinterpret_cast<float *>(lds_built) + half * (DH * 16 + 2) * 256 + (threadIdx.x & 255);
  const float *other = reinterpret_cast<float *>(lds_built) + (half ^ 1) * (DH * 16 + 2) * 256 + (threadIdx.x & 255);
#pragma unroll
  for (int d = 0; d < DH; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) mine[(16 * d + i) * 256] = half ? o[d][i] : o[DH + d][i];
  mine[DH * 16 * 256] = m_run;
  mine[(DH * 16 + 1) * 256] = l;
  __syncthreads();
  const float m_other = other[DH * 16 * 256], m_all = fmaxf(m_run, m_other);
  const float f_mine = m_run == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(m_run - m_all);
  const float f_other = m_other == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(m_other - m_all);
  l = half ? other[(DH * 16 + 1) * 256] * f_other + l * f_mine : l * f_mine + other[(DH * 16 + 1) * 256] * f_other;
  floatx16_t sum[DH];
#pragma unroll
  for (int d = 0; d < DH; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float own = (half ? o[DH + d][i] : o[d][i]) * f_mine, got = other[(16 * d + i) * 256] * f_other;
      sum[d][i] = half ? got + own : own + got;
    }
  if (!col_ok) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  bf16_t *orow = a.out + (size_t(row) * a.heads + head) * VD;
#pragma unroll
  for (int u = 0; u < DH * 4; ++u) {
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = sum[u >> 2][4 * (u & 3) + e] * inv;
    if (a.gate) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = v[e] * (1.0f / (1.0f + expf(-gate[u][e])));
    }
    *reinterpret_cast<uint2 *>(orow + d0 + 8 * u) = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
  }
}

template <int DP, int RD, int VD>
int launch_built(const BuiltArgs &a, int n_tiles, hipStream_t s) {
  constexpr int lds_bytes = 4 * SB_PAGE * (DP + RD + VD) * 2;
  static bool raised = false;     // per instantiation; harmless if repeated
  if (!raised) {
    const hipError_t e = hipFuncSetAttribute((const void *)built_attention_kernel<DP, RD, VD>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    SB_REQUIRE(e == hipSuccess, "sb_built_attention: cannot reserve %d bytes of LDS: %s", lds_bytes, hipGetErrorString(e));
    raised = true;
  }
  built_attention_kernel<DP, RD, VD><<<unsigned(n_tiles) * unsigned(a.heads), 512, lds_bytes, s>>>(a);
  return sb::check_launch("sb_built_attention");
}

}  // namespace

// 1 when sb_built_attention takes these sizes.
extern "C" int sb_built_attention_ok(int dim, int rot_dim, int vdim, int rank) {
  return dim == 128 && rot_dim == 64 && vdim == 128 && rank > 0 && rank % 8 == 0;
}

extern "C" int sb_built_tile_rows(void) { return kRows; }

extern "C" int sb_built_gather(void *out, const void *cache, const int32_t *page_table, int max_pages, int n_pages_total,
                               const int32_t *pages, int n_pages, int rank, int rot_dim, void *stream) {
  SB_REQUIRE(out && cache && page_table && pages, "sb_built_gather: null pointer");
  SB_REQUIRE(n_pages >= 0 && max_pages > 0 && n_pages_total > 0 && rank > 0 && rot_dim >= 0, "sb_built_gather: bad sizes");
  SB_SUPPORT(rank % 8 == 0 && rot_dim % 8 == 0, "sb_built_gather: a latent row of %d + %d is not taken", rank, rot_dim);
  SB_SUPPORT((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(cache)) % 16 == 0, "sb_built_gather: operands must be 16-byte aligned");
  if (n_pages == 0) return SB_OK;
  built_gather_kernel<<<n_pages, 256, 0, (hipStream_t)stream>>>((bf16_t *)out, (const bf16_t *)cache, page_table, max_pages, n_pages_total,
                                                                pages, rank, rank + rot_dim);
  return sb::check_launch("sb_built_gather");
}

extern "C" int sb_built_attention(void *out, const void *q_plain, const void *q_rot, int q_rot_stride, const void *built, int built_stride,
                                  const void *cache, const int32_t *page_table, int max_pages, int n_pages_total,
                                  const int32_t *tiles, int n_tiles, int heads, int dim, int rot_dim, int vdim, int rank, float scale,
                                  int window, const float *gate, int gate_stride, int gate_per_head, void *stream) {
  SB_REQUIRE(out && q_plain && q_rot && built && cache && page_table && tiles, "sb_built_attention: null pointer");
  SB_REQUIRE(n_tiles >= 0 && heads > 0 && max_pages > 0 && n_pages_total > 0 && window >= 0, "sb_built_attention: bad sizes");
  SB_SUPPORT(scale > 0.0f, "sb_built_attention: a scale of %g is not taken", double(scale));
  SB_SUPPORT(sb_built_attention_ok(dim, rot_dim, vdim, rank), "sb_built_attention: heads of %d + %d numbers and %d values are not taken", dim,
             rot_dim, vdim);
  SB_SUPPORT((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(q_plain) | reinterpret_cast<uintptr_t>(q_rot) |
              reinterpret_cast<uintptr_t>(built) | reinterpret_cast<uintptr_t>(cache)) % 16 == 0 &&
                 q_rot_stride % 8 == 0 && built_stride % 8 == 0,
             "sb_built_attention: operands must be 16-byte aligned");
  SB_REQUIRE(built_stride >= heads * (dim + vdim), "sb_built_attention: rows of built keys and values are too short");
  SB_SUPPORT((long long)built_stride * 2 * SB_PAGE < (1ll << 31) && (long long)n_tiles * heads < (1ll << 31), "sb_built_attention: too large");
  if (n_tiles == 0) return SB_OK;
  BuiltArgs a;
  a.out = (bf16_t *)out; a.q_plain = (const bf16_t *)q_plain; a.q_rot = (const bf16_t *)q_rot; a.q_rot_stride = q_rot_stride;
  a.built = (const bf16_t *)built; a.built_stride = built_stride; a.cache = (const bf16_t *)cache; a.rank = rank; a.latent = rank + rot_dim;
  a.page_table = page_table; a.max_pages = max_pages; a.n_pages_total = n_pages_total; a.tiles = tiles;
  a.heads = heads; a.scale2 = scale * 1.4426950408889634f; a.window = window;
  a.gate = gate; a.gate_stride = gate_stride; a.gate_per_head = gate_per_head;
  return launch_built<128, 64, 128>(a, n_tiles, (hipStream_t)stream);
}
