// The float32 matrix product  Y[t,n] = sum_k X[t,k] W[n,k] (+bias) (+resid): the true 32-bit path
// of every projection, and the fallback of the bf16 path for sizes its kernels refuse.
//
// It runs on the float32 matrix cores.  v_mfma_f32_16x16x4_f32 adds its four products to the
// accumulator one after the other in ascending k, each with one rounding: the bits of a chain of
// fmaf (checked against fmaf over 1,000 k, denormals among them).  An element is the sum of its
// chains, each from zero, added in ascending order: chains of kChain k where there are up to kSegment of them, of a segment of
// kSegment k where there are more.  That is a function of k alone, so its value does not depend on how many rows share the
// launch, on the tile or on the waves that made it.  The same (row, column) gives the same bits in a whole prompt, in a
// single-token step and in any batch.  W is [out, in] row-major, the memory of a
// projection weight (/root/reference/core/include/sonicboom/quant/quantized_matmul.h:74-77);
// the bias is added after the product and the residual after the bias
// (/root/reference/core/src/model/emit.cpp:260-261, :447).
//
// A block owns 16 CT columns of 16 TT rows.  Its WAVES waves take the segments of K between them
// (segment s goes to wave s % WAVES), or, where there is one and there are few blocks, its chains, straight from memory and without a
// barrier on the way; the sums meet in LDS.  A lane loads four consecutive k of one row, the four lane groups of
// a row 64 bytes side by side; four lane swaps turn the 4 x 4 of lane groups and registers over,
// after which register s holds k = 4 s + lane group, what step s of the matrix instruction takes.
// W that a projection keeps is packed (FORM kPacked): blocks of 16 rows x 16 k in the order that
// the lanes take, 1 KB each, consecutive in k, so that a wave reads one stream and swaps nothing.
// The loads run kAhead steps of 16 k ahead in a ring of registers.  Gated (G = 2): a column tile
// is a tile of W's first half and the same tile of the second, and Y = act(first) * second.
//
// What bounds it: with few rows a chain of products (64 of them are 1.3 us) behind the first loads and, where a CU streams much of W (the
// gated product: 304 blocks of 115 KB on 256 CUs), that; with many rows the matrix cores.  With one chain of up to 1,024 k few rows took
// longer: 3 rows against 896 x 896 8.1 us and 5.7 with a wave a chain, 1,152 x 896 8.1 and 5.7, 50 rows 12.9 and 9.1, 16 against 16,384 x
// 256 8.0 and 7.0; 130 rows against 1,152 x 896 14.1 and 14.5; and the error against 64 bits is half of what it was.  Longer products keep
// chains of a segment.  Shorter ones gave few rows 2,048 x 2,048 9.7 -> 9.0 us, but their sums cost registers or loads in flight: 3 rows
// against 3,584 x 18,944 54.8 -> 68.6, gated 17,920 x 1,536 26.2 -> 31.3, 520 rows against gated 37,888 x 3,584 1,372 -> 1,562 (with the
// registers bounded and the sums joined between products 1,454).
// The source keeps a step's loads behind its
// products and turns X's fragments over a step ahead: left to itself the compiler turned a whole ring over at once and so
// waited for the newest of its loads ahead of the round's first product.  Measured on MI355X at the 0.5B layer sizes, 3 rows,
// left to itself and so, a wave a segment: 896 x 896 8.2 and 7.7 us, the gated 9,728 x 896 16.1 and 13.5, 896 x 4,864 15.5 and 14.9, a block a
// segment (sb_gemm_f32_packed_partial) 9.7; 520 rows: the gated product 140 and 105 us (86 TFLOP/s), 896 x 4,864 75 and 69.
// Not kept for few rows: a wave for each half of the gated product (16 us), X's segment in LDS in the products' order with W's
// loads twice as far ahead (12 to 17 us gated, 8.7 to 9.5 for 896 x 896: staging X costs what it saves).
#include "mfma.h"

namespace {

constexpr int kSegment = 1024;          // k of a segment, the chain of products with more k: part of what the result's bits are
constexpr int kChain = 256;             // k of a chain of products with no more than a segment: likewise
constexpr int kChains = kSegment / kChain;
constexpr int kChainSteps = kChain / 16;

enum Form { kAny, kPacked, kPackedAny };   // W row-major; W packed, X by 16-byte loads; W packed, X element by element

__device__ __forceinline__ void swap_halves(float &a, float &b) {
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  const uint32_t p0 = p[0], p1 = p[1];
  a = __uint_as_float(p0);
  b = __uint_as_float(p1);
}
__device__ __forceinline__ void swap_rows(float &a, float &b) {
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  const uint32_t p0 = p[0], p1 = p[1];
  a = __uint_as_float(p0);
  b = __uint_as_float(p1);
}

// In: register s of lane group g holds k = 4 g + s.  Out: k = 4 s + g.
__device__ __forceinline__ void by_step(const floatx4_t &raw, float (&f)[4]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) f[e] = raw[e];
  swap_rows(f[0], f[1]);
  swap_rows(f[2], f[3]);
  swap_halves(f[0], f[2]);
  swap_halves(f[1], f[3]);
}

constexpr uint32_t kPastEnd = 0x80000000u;      // an offset past every descriptor's end: reads as zeros

// Four consecutive k of a row of T that starts at `row`; zeros where k lies at or past `end`.
template <typename T>
__device__ __forceinline__ floatx4_t load4_any(const T *row, int k, int end) {
  floatx4_t v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = k + e < end ? ld_f(row, size_t(k) + e) : 0.0f;
  return v;
}

struct PlainArgs {
  void *y;
  int y_dtype;
  const void *bias;
  int bias_dtype;
  const float *resid;
  int n_rows, n_out, n_in;
  int gate;        // the activation (an sb_gate) of the gated form
  bool vec4;       // n_out % 4 == 0, and Y and the residual start on 16 bytes
};

bool by_fours(const void *y, const float *resid, int n_out) {
  return n_out % 4 == 0 && (reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(resid)) % 16 == 0;
}

// CHAINS: kWhole: a wave's share is a segment, one chain (more than one segment); kInTurn: the one segment, its chains one after the
// other; kApart: a wave a chain of it.
enum Chains { kWhole, kInTurn, kApart };
template <typename TX, typename TW, int FORM, int TT, int CT, int G, int WAVES, Chains CHAINS>
__global__ void __launch_bounds__(64 * WAVES)
gemm_f32_kernel(const TX *__restrict__ x, const TW *__restrict__ w, PlainArgs a) {
  constexpr int kStreams = CT * G, kTiles = TT * CT, kThreads = 64 * WAVES;
  // steps in flight: as many as 192 registers hold, and a chain ends with a round of them (128 or less beside the accumulators of larger tiles
  // and the addresses of loads element by element)
  constexpr int kRegs = 4 * (kStreams + TT);
  constexpr int kAhead = FORM != kPacked ? 4 : kRegs == 8 && CHAINS == kWhole ? 24 : kRegs <= 12 ? 16 : kRegs <= 16 ? 8 : 4;
  static_assert(CHAINS == kWhole || kChainSteps % kAhead == 0, "chains end with a round of the ring");
  static_assert(CHAINS == kWhole || WAVES == (CHAINS == kApart ? kChains : 1), "a block has the segment's chains");
  constexpr int kPolicy = TT == 1 ? kReadOnce : 0;                  // up to sixteen rows: no other block reads this share of W (prompts and
                                                                    // eight tokens of the 0.5B sizes 19.7 -> 19.2 ms)
  constexpr int kUnits = (kTiles * 64 + kThreads - 1) / kThreads;   // groups of four outputs a thread
  extern __shared__ floatx4_t part[];            // [WAVES][G][kTiles][64]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const unsigned tiles_n = (a.n_out + 16 * CT - 1) / (16 * CT);
  const int n0 = int(blockIdx.x % tiles_n) * (16 * CT), t0 = int(blockIdx.x / tiles_n) * (16 * TT);
  const int w_tiles = (a.n_out + 15) / 16, w_steps = (a.n_in + 15) / 16;      // packed: of one half

  // Rows past the last one read the last one again (their outputs are not stored).
  const TX *x0 = x + size_t(t0) * a.n_in;
  const int x_rows = min(16 * TT, a.n_rows - t0);
  const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<TX *>(x0), 0, uint32_t(size_t(x_rows) * a.n_in * sizeof(TX)), 0x00020000);
  size_t x_at[TT];
#pragma unroll
  for (int j = 0; j < TT; ++j) x_at[j] = size_t(min(16 * j + r, x_rows - 1)) * a.n_in;
  const TW *w_row[kStreams];
  int w_tile[kStreams];
#pragma unroll
  for (int i = 0; i < kStreams; ++i) {           // stream i: column tile i / G, half i % G
    w_tile[i] = (i % G) * w_tiles + min(n0 / 16 + i / G, w_tiles - 1);
    if (FORM == kAny) w_row[i] = w + (size_t(i % G) * a.n_out + min(n0 + 16 * (i / G) + r, a.n_out - 1)) * a.n_in;
  }

  floatx4_t total[kUnits][G];
#pragma unroll
  for (int u = 0; u < kUnits; ++u)
#pragma unroll
    for (int q = 0; q < G; ++q) total[u][q] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  // a grid of as many layers as segments: each block one segment, whose raw sums are Y's plane of that number
  const bool split = gridDim.y > 1;
  const int n_seg = split ? int(blockIdx.y) + 1 : (a.n_in + kSegment - 1) / kSegment;
  constexpr int kShare = CHAINS == kApart ? kChain : kSegment;
  const int k_all = min(n_seg * kSegment, a.n_in);
  for (int s0 = blockIdx.y; s0 < n_seg; s0 += WAVES) {
    const int k0 = s0 * kSegment + wave * kShare;
    if (k0 < k_all) {                            // uniform over the wave
      const int k_end = min(k0 + kShare, a.n_in);
      const int steps = (k_end - k0 + 15) / 16;
      // packed: a descriptor a stream, of its tile's blocks up to the segment's end
      __amdgpu_buffer_rsrc_t rsrc_w[kStreams];
      if constexpr (FORM != kAny) {
#pragma unroll
        for (int i = 0; i < kStreams; ++i)
          rsrc_w[i] = __builtin_amdgcn_make_buffer_rsrc(
              const_cast<TW *>(w) + (size_t(w_tile[i]) * w_steps + k0 / 16) * 256, 0, uint32_t(steps) * 1024u, 0x00020000);
      }
      floatx4_t acc[kStreams][TT];
#pragma unroll
      for (int i = 0; i < kStreams; ++i)
#pragma unroll
        for (int j = 0; j < TT; ++j) acc[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
      floatx4_t rw[kAhead][kStreams], rx[kAhead][TT];
      const int k_lane = k0 + 4 * g;
      auto ask = [&](int slot, int step) {
        const int k = k_lane + 16 * step;
#pragma unroll
        for (int i = 0; i < kStreams; ++i) {
          if constexpr (FORM == kAny) rw[slot][i] = load4_any(w_row[i], k, k_end);
          else rw[slot][i] = __builtin_bit_cast(floatx4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc_w[i], lane * 16 + step * 1024, 0, kPolicy));
        }
#pragma unroll
        for (int j = 0; j < TT; ++j) {
          if constexpr (FORM == kPacked)
            rx[slot][j] = __builtin_bit_cast(floatx4_t, __builtin_amdgcn_raw_buffer_load_b128(
                rsrc_x, int(k < k_end ? uint32_t((x_at[j] + k) * 4) : kPastEnd), 0, 0));
          else rx[slot][j] = load4_any(x0 + x_at[j], k, k_end);
        }
      };
      // X's fragments are turned over a step ahead, beside the products of the step before
      float fx[2][TT][4];
      auto turn = [&](int slot, int set) {
#pragma unroll
        for (int j = 0; j < TT; ++j) by_step(rx[slot][j], fx[set][j]);
      };
      auto multiply = [&](int slot, int set) {
        float fw[kStreams][4];
#pragma unroll
        for (int i = 0; i < kStreams; ++i) {
          if constexpr (FORM == kAny) {
            by_step(rw[slot][i], fw[i]);
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) fw[i][e] = rw[slot][i][e];
          }
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int i = 0; i < kStreams; ++i)
#pragma unroll
            for (int j = 0; j < TT; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[i][s], fx[set][j][s], acc[i][j], 0, 0, 0);
      };
      static_assert(kAhead % 2 == 0, "the sets of turned fragments alternate");
      // a chain's end: its sums join the total, or wait in this lane's own places in LDS
      auto fold = [&](bool more) {
#pragma unroll
        for (int i = 0; i < kStreams; ++i)
#pragma unroll
          for (int j = 0; j < TT; ++j) {
            if constexpr (WAVES == 1) total[(i / G) * TT + j][i % G] = total[(i / G) * TT + j][i % G] + acc[i][j];
            else part[((wave * G + i % G) * kTiles + (i / G) * TT + j) * 64 + lane] = acc[i][j];
            if (more) acc[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
          }
      };
#pragma unroll
      for (int u = 0; u < kAhead; ++u) ask(u, u);
      turn(0, 0);
      int step = 0;
      for (; step + kAhead <= steps; step += kAhead) {       // whole rounds of the ring
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
          turn((u + 1) % kAhead, (u + 1) & 1);
          multiply(u, u & 1);
          ask(u, step + kAhead + u);
          // (left alone, the compiler turns a whole round over at once, waiting for the last of its loads ahead of the first product)
          __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (CHAINS == kInTurn) {
          const int done = step + kAhead;
          if (done % kChainSteps == 0 && done < steps) fold(true);
        }
      }
#pragma unroll
      for (int u = 0; u < kAhead; ++u)
        if (step + u < steps) {
          if (u + 1 < kAhead) turn(u + 1, (u + 1) & 1);
          multiply(u, u & 1);
        }
      fold(false);
    }
    if constexpr (WAVES > 1) {
      __syncthreads();
      const int here = min(WAVES, (k_all - s0 * kSegment + kShare - 1) / kShare);
#pragma unroll
      for (int u = 0; u < kUnits; ++u) {
        const int unit = tid + u * kThreads;
        if (unit < kTiles * 64)
          for (int v = 0; v < here; ++v)
#pragma unroll
            for (int q = 0; q < G; ++q) total[u][q] = total[u][q] + part[(v * G + q) * kTiles * 64 + unit];
      }
      __syncthreads();
    }
  }

  // unit (tile (i, j), lane (g, r)): columns 16 i + 4 g + 0..3 of row 16 j + r, stored together where they are aligned, and
  // their residuals (which the stores may overwrite, each its own) asked for ahead of the first store: a product of few k is
  // bound here (4,096 x 64 onto a residual stream of 4,000 rows 105 us a number at a time, 63 by fours, 57 so; 55 the LDS tiles)
  const auto place = [&](int u, int &t, int &nb) {
    const int unit = tid + u * kThreads, tile = unit >> 6, l = unit & 63;
    t = t0 + 16 * (tile % TT) + (l & 15), nb = n0 + 16 * (tile / TT) + 4 * (l >> 4);
    return unit < kTiles * 64 && t < a.n_rows && nb < a.n_out;
  };
  if (split) a.y = (float *)a.y + size_t(blockIdx.y) * a.n_rows * a.n_out;
  if (a.vec4) {
    floatx4_t old[kUnits];
    if (a.resid) {
#pragma unroll
      for (int u = 0; u < kUnits; ++u) {
        int t, nb;
        if (place(u, t, nb)) old[u] = *reinterpret_cast<const floatx4_t *>(a.resid + size_t(t) * a.n_out + nb);
      }
    }
#pragma unroll
    for (int u = 0; u < kUnits; ++u) {
      int t, nb;
      if (!place(u, t, nb)) continue;
      const size_t idx = size_t(t) * a.n_out + nb;
      floatx4_t v = total[u][0];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (G == 2) v[e] = gate_act(v[e], a.gate) * total[u][G - 1][e];
        if (a.bias) v[e] = v[e] + ld_dyn(a.bias, a.bias_dtype, nb + e);
      }
      if (a.resid) v = v + old[u];
      if (a.y_dtype == SB_F32) *reinterpret_cast<floatx4_t *>((float *)a.y + idx) = v;
      else
        *reinterpret_cast<ushort4 *>((bf16_t *)a.y + idx) =
            make_ushort4(f32_to_bf16(v[0]), f32_to_bf16(v[1]), f32_to_bf16(v[2]), f32_to_bf16(v[3]));
    }
    return;
  }
#pragma unroll
  for (int u = 0; u < kUnits; ++u) {
    int t, nb;
    if (!place(u, t, nb)) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int n = nb + e;
      if (n >= a.n_out) continue;
      float v = total[u][0][e];
      if constexpr (G == 2) v = gate_act(v, a.gate) * total[u][G - 1][e];
      if (a.bias) v = v + ld_dyn(a.bias, a.bias_dtype, n);
      const size_t idx = size_t(t) * a.n_out + n;
      if (a.resid) v = v + a.resid[idx];
      if (a.y_dtype == SB_F32) ((float *)a.y)[idx] = v;
      else ((bf16_t *)a.y)[idx] = f32_to_bf16(v);
    }
  }
}

template <typename TX, typename TW, int FORM, int TT, int CT, int G, int WAVES, Chains CHAINS = kWhole>
int launch_one(const TX *x, const TW *w, const PlainArgs &a, hipStream_t s, int layers = 1) {
  constexpr int lds_bytes = WAVES == 1 ? 0 : WAVES * TT * CT * G * 1024;
  auto kern = gemm_f32_kernel<TX, TW, FORM, TT, CT, G, WAVES, CHAINS>;
  static bool raised = false;     // per instantiation; harmless if repeated
  if (lds_bytes > 48 * 1024 && !raised) {
    const hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    SB_REQUIRE(e == hipSuccess, "sb_gemm: cannot reserve %d bytes of LDS: %s", lds_bytes, hipGetErrorString(e));
    raised = true;
  }
  const long long blocks = (long long)((a.n_out + 16 * CT - 1) / (16 * CT)) * ((a.n_rows + 16 * TT - 1) / (16 * TT));
  SB_SUPPORT(blocks <= 0x7fffffffLL, "sb_gemm: too many tiles");
  kern<<<dim3(unsigned(blocks), layers), 64 * WAVES, lds_bytes, s>>>(x, w, a);
  return sb::check_launch("sb_gemm");
}

template <int TT, int CT, int G>
int launch_packed(const float *x, const float *w, const PlainArgs &a, int n_seg, hipStream_t s) {
  if (n_seg == 1) return launch_one<float, float, kPacked, TT, CT, G, 1, kInTurn>(x, w, a, s);
  if (n_seg == 2) return launch_one<float, float, kPacked, TT, CT, G, 2>(x, w, a, s);
  if (n_seg <= 4) return launch_one<float, float, kPacked, TT, CT, G, 4>(x, w, a, s);
  return launch_one<float, float, kPacked, TT, CT, G, 8>(x, w, a, s);
}

// The tile for rows past sixteen.  One segment of K: the least price, rounds of waves over the SIMDs times a step's products and
// nine tenths of its loads (tiles of both sides), so that a last round that is nearly empty counts; on a tie the larger tile.
// 520 rows: gated 9,728 x 896 1,368 waves of 4 x 2 (tiles of both halves) 132 us, 2,736 of 4 x 1 105, 5,168 of 2 x 1 109; 1,152 x
// 896 tiles of 2 x 2 22, 2 x 1 29, 4 x 2 38; 200 rows gated 66, 69 and 55.  Several segments: the largest tile whose waves give
// most of the 1,024 SIMDs one (520 rows, 896 x 4,864: 4 x 2 71 us, 2 x 2 74, 2 x 1 108, 4 x 4 116).
template <int G>
int launch_packed_tiles(const float *x, const float *w, const PlainArgs &a, int n_seg, hipStream_t s) {
  const auto tiles = [&](int tt, int ct) {
    return (long long)((a.n_rows + 16 * tt - 1) / (16 * tt)) * ((a.n_out + 16 * ct - 1) / (16 * ct));
  };
  const auto waves = [&](int tt, int ct) { return tiles(tt, ct) * (n_seg < 8 ? n_seg : 8); };
  constexpr long long kEnough = 768;
  if (a.n_rows <= 16) {
    if (G == 1 && waves(1, 2) >= 4 * kEnough) return launch_packed<1, 2, G>(x, w, a, n_seg, s);
    // a wave a chain while there is a CU a block (gated, 304 blocks, it would be 13.6 us for 13.2)
    if (n_seg == 1 && tiles(1, 1) <= sb::cu_count()) return launch_one<float, float, kPacked, 1, 1, G, kChains, kApart>(x, w, a, s);
    return launch_packed<1, 1, G>(x, w, a, n_seg, s);
  }
  constexpr int kShapes[4][2] = {{4, 4 / G}, {4, 2 / G}, {2, 2 / G}, {2, 1}};      // (gated the last two are one)
  int pick = 3;
  if (n_seg == 1) {
    double best = 0;
    for (int v = 0; v < 4; ++v) {
      const int tt = kShapes[v][0], ct = kShapes[v][1];
      if (tt == 4 && a.n_rows <= 32) continue;
      const double price = double((waves(tt, ct) + 1023) / 1024) * (tt * ct * G + 0.9 * (tt + ct * G));
      if (best == 0 || price < best) best = price, pick = v;
    }
  } else {
    if (a.n_rows > 32 && waves(4, 4 / G) >= kEnough) pick = 0;
    else if (a.n_rows > 32 && waves(4, 2 / G) >= kEnough) pick = 1;
    else if (G == 1 && waves(2, 2) >= kEnough) pick = 2;
  }
  if (pick == 0) return launch_packed<4, 4 / G, G>(x, w, a, n_seg, s);
  if (pick == 1) return launch_packed<4, 2 / G, G>(x, w, a, n_seg, s);
  if (pick == 2) return launch_packed<2, 2 / G, G>(x, w, a, n_seg, s);
  // a wave a chain, of three or four (50 rows against 1,152 x 896, 144 blocks, 12.9 -> 9.1 us; gated, 304 and more, 20.4 and 21.0; two
  // chains, 20 rows against 6,144 x 512, 384 blocks, 9.8 and 11.1)
  if (n_seg == 1 && a.n_in > 2 * kChain && tiles(2, 1) <= (G == 1 ? 2 : 1) * sb::cu_count())
    return launch_one<float, float, kPacked, 2, 1, G, kChains, kApart>(x, w, a, s);
  return launch_packed<2, 1, G>(x, w, a, n_seg, s);
}

// The same sums with a chain a thread: 64 x 64 tiles staged in LDS, every element of X and W read once a tile.
constexpr int kTile = 64;        // rows and columns of a block's tile
constexpr int kStage = 16;       // k per stage; a segment is a whole number of stages
constexpr int kTileThreads = 256;

// The sums of chains are in registers; several segments' wait in LDS, a place a thread, but for a row of four.  The next stage is
// asked for ahead of a stage's products, at addresses that are the block's plus one number a thread: 58 registers, eight waves a SIMD (with
// an address for each load 96 and five).  Us, one chain of up to 1,024 k and no stage ahead, with an address each, so: 2,048 rows against
// 3,584 x 3,584 float32 796, 748, 698, bfloat16 714, 684, 636; 3,584 x 896 207, 206, 195 and 179, 193, 181; 4,000 rows against 2,000 x
// 1,024 246, 268, 248 and 231, 245, 228.
template <typename TX, typename TW, bool SEGMENTS>
__global__ void __launch_bounds__(kTileThreads)
gemm_tile_kernel(const TX *__restrict__ x, const TW *__restrict__ w, PlainArgs a) {
  __shared__ float xs[kStage][kTile + 4];
  __shared__ float ws[kStage][kTile + 4];
  __shared__ float total[SEGMENTS ? 12 : 1][kTileThreads];
  const unsigned tiles_n = (a.n_out + kTile - 1) / kTile;
  const int t0 = int(blockIdx.x / tiles_n) * kTile, n0 = int(blockIdx.x % tiles_n) * kTile;
  const int tid = threadIdx.x, ty = tid / 16, tx = tid % 16;
  float acc[4][4], sum[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = sum[i][j] = 0.0f;
  // a stage on its way: asked for ahead of the products of the stage before
  constexpr int kRowsApart = kTileThreads / kStage;
  const int row = tid / kStage, k_of = tid % kStage;
  const unsigned off = unsigned(row) * unsigned(a.n_in) + unsigned(k_of);      // (beside addresses that are the block's)
  TX nx[4];
  TW nw[4];
  const auto ask = [&](int k0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = t0 + i * kRowsApart, n = n0 + i * kRowsApart;
      nx[i] = t + row < a.n_rows && k0 + k_of < a.n_in ? (x + size_t(t) * a.n_in + k0)[off] : TX(0);
      nw[i] = n + row < a.n_out && k0 + k_of < a.n_in ? (w + size_t(n) * a.n_in + k0)[off] : TW(0);
    }
  };
  ask(0);
  constexpr int kLength = SEGMENTS ? kSegment : kChain;
  for (int c0 = 0; c0 < a.n_in; c0 += kLength) {
    const int c_end = min(c0 + kLength, a.n_in);
    for (int k0 = c0; k0 < c_end; k0 += kStage) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        xs[k_of][row + i * kRowsApart] = ld_f(&nx[i], 0);
        ws[k_of][row + i * kRowsApart] = ld_f(&nw[i], 0);
      }
      __syncthreads();
      ask(k0 + kStage);
#pragma unroll
      for (int k = 0; k < kStage; ++k) {
        float p[4], q[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = xs[k][ty * 4 + i];
#pragma unroll
        for (int j = 0; j < 4; ++j) q[j] = ws[k][tx * 4 + j];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(p[i], q[j], acc[i][j]);
      }
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (SEGMENTS && i < 3) total[4 * i + j][tid] = c0 > 0 ? total[4 * i + j][tid] + acc[i][j] : acc[i][j];
        else sum[i][j] = sum[i][j] + acc[i][j];
        acc[i][j] = 0.0f;
      }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = t0 + ty * 4 + i;
    if (t >= a.n_rows) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n >= a.n_out) continue;
      float v = SEGMENTS && i < 3 ? total[4 * i + j][tid] : sum[i][j];
      if (a.bias) v = v + ld_dyn(a.bias, a.bias_dtype, n);
      const size_t idx = size_t(t) * a.n_out + n;
      if (a.resid) v = v + a.resid[idx];
      if (a.y_dtype == SB_F32) ((float *)a.y)[idx] = v;
      else ((bf16_t *)a.y)[idx] = f32_to_bf16(v);
    }
  }
}

// Every type, any inner size and alignment: loads element by element.  The matrix-core form reads X and W once for every
// 32 x 16 tile, an element a lane and load, 10 to 30 segments of such a tile a microsecond; the form above walks K at
// 0.075 us a k with a tile or less a CU and 0.03 more for every tile a CU, and is ahead once there are many: float32,
// 2,048 rows against 3,584 x 3,584 0.81 ms (matrix cores 4.07), bfloat16 0.72 (4.37), one row against 151,936 x 896 254 us
// (436), 300 against 4,000 x 4,001 587 (814); behind with few: one row against 896 x 4,864 362 us (43), 64 against 4,096 x
// 20,000 2,908 (822), 300 against 900 x 1,001 123 (44).
template <typename TX, typename TW>
int launch_any(const TX *x, const TW *w, const PlainArgs &a, int n_seg, hipStream_t s) {
  const bool f32 = sizeof(TX) == 4 && sizeof(TW) == 4;
  const double tiles = double((a.n_rows + kTile - 1) / kTile) * ((a.n_out + kTile - 1) / kTile);
  const double segments = double((a.n_rows + 31) / 32) * ((a.n_out + 15) / 16) * (a.n_in / double(kSegment));
  const double tile_us = a.n_in * (0.075 + 0.03 * tiles / 256.0);
  const double mfma_us = segments / (!f32 ? 11.0 : a.n_rows <= 32 ? 30.0 : 17.0);
  const double wave_us = (f32 ? 28.0 : 65.0) * (n_seg > 1 ? 1.0 : a.n_in / double(kSegment));      // one wave's segment
  if (tile_us < (mfma_us > wave_us ? mfma_us : wave_us)) {
    const long long blocks = (long long)tiles;
    SB_SUPPORT(blocks <= 0x7fffffffLL, "sb_gemm: too many tiles");
    if (n_seg == 1) gemm_tile_kernel<TX, TW, false><<<unsigned(blocks), kTileThreads, 0, s>>>(x, w, a);
    else gemm_tile_kernel<TX, TW, true><<<unsigned(blocks), kTileThreads, 0, s>>>(x, w, a);
    return sb::check_launch("sb_gemm");
  }
  if (n_seg == 1) return launch_one<TX, TW, kAny, 2, 1, 1, 1, kInTurn>(x, w, a, s);
  return launch_one<TX, TW, kAny, 2, 1, 1, 8>(x, w, a, s);
}

}  // namespace

extern "C" int sb_gemm(void *y, int y_dtype, const void *x, int x_dtype, const void *w, int w_dtype,
                       const void *bias, int bias_dtype, const float *resid, int n_rows, int n_out,
                       int n_in, void *stream) {
  SB_REQUIRE(y && x && w, "sb_gemm: null pointer");
  SB_REQUIRE(n_rows >= 0 && n_out > 0 && n_in > 0, "sb_gemm: bad sizes rows=%d out=%d in=%d", n_rows,
             n_out, n_in);
  SB_REQUIRE(sb::valid_dtype(y_dtype) && sb::valid_dtype(x_dtype) && sb::valid_dtype(w_dtype) &&
                 (!bias || sb::valid_dtype(bias_dtype)),
             "sb_gemm: unknown dtype");
  SB_REQUIRE(!(resid && y_dtype != SB_F32 && (const void *)resid == y),
             "sb_gemm: a residual that aliases the output must be f32");
  SB_SUPPORT((n_rows + 63) / 64 <= 65535, "sb_gemm: more than %d rows in one call", 65535 * 64);
  if (n_rows == 0) return SB_OK;
  hipStream_t s = (hipStream_t)stream;
  const PlainArgs a{y, y_dtype, bias, bias_dtype, resid, n_rows, n_out, n_in, SB_GATE_NONE, by_fours(y, resid, n_out)};
  const int n_seg = (n_in + kSegment - 1) / kSegment;
  if (x_dtype == SB_F32 && w_dtype == SB_F32) return launch_any((const float *)x, (const float *)w, a, n_seg, s);
  if (x_dtype == SB_F32) return launch_any((const float *)x, (const bf16_t *)w, a, n_seg, s);
  if (w_dtype == SB_F32) return launch_any((const bf16_t *)x, (const float *)w, a, n_seg, s);
  return launch_any((const bf16_t *)x, (const bf16_t *)w, a, n_seg, s);
}

// The same for float32 X and packed float32 W (blocks of 16 rows x 16 k, consecutive in k, zero padded: the
// element of row r, k = 4 s + g of a block lies at (16 g + r) * 4 + s; gated: the two halves one after the
// other, each padded), with gated != 0: Y = act(X Wg^T) * (X Wu^T).  The bits of sb_gemm.
extern "C" int sb_gemm_f32_packed(void *y, int y_dtype, const float *x, const float *w, const void *bias, int bias_dtype,
                                  const float *resid, int n_rows, int n_out, int n_in, int gated, void *stream) {
  SB_REQUIRE(y && x && w, "sb_gemm_f32_packed: null pointer");
  SB_REQUIRE(n_rows >= 0 && n_out > 0 && n_in > 0, "sb_gemm_f32_packed: bad sizes rows=%d out=%d in=%d", n_rows, n_out, n_in);
  SB_REQUIRE(sb::valid_dtype(y_dtype) && (!bias || sb::valid_dtype(bias_dtype)), "sb_gemm_f32_packed: unknown dtype");
  SB_REQUIRE(!(resid && y_dtype != SB_F32 && (const void *)resid == y),
             "sb_gemm_f32_packed: a residual that aliases the output must be f32");
  SB_REQUIRE(!(gated && (bias || resid)), "sb_gemm_f32_packed: the gated form takes no bias or residual");
  SB_SUPPORT(gated >= SB_GATE_NONE && gated <= SB_GATE_RELU, "sb_gemm_f32_packed: unknown gate activation %d", gated);
  SB_SUPPORT((n_rows + 63) / 64 <= 65535, "sb_gemm_f32_packed: more than %d rows in one call", 65535 * 64);
  SB_SUPPORT(reinterpret_cast<uintptr_t>(w) % 16 == 0, "sb_gemm_f32_packed: the packed weights must be 16-byte aligned");
  if (n_rows == 0) return SB_OK;
  hipStream_t s = (hipStream_t)stream;
  const PlainArgs a{y, y_dtype, bias, bias_dtype, resid, n_rows, n_out, n_in, gated, by_fours(y, resid, n_out)};
  const int n_seg = (n_in + kSegment - 1) / kSegment;
  // 16-byte loads need rows of X that start on 16 bytes; offsets inside a block's rows fit 31 bits
  const bool vec = n_in % 4 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 && size_t(n_in) * 64 * 4 < (size_t(1) << 31);
  if (!vec) {
    if (gated) return n_seg == 1 ? launch_one<float, float, kPackedAny, 2, 1, 2, 1, kInTurn>(x, w, a, s)
                                 : launch_one<float, float, kPackedAny, 2, 1, 2, 8>(x, w, a, s);
    return n_seg == 1 ? launch_one<float, float, kPackedAny, 2, 1, 1, 1, kInTurn>(x, w, a, s)
                      : launch_one<float, float, kPackedAny, 2, 1, 1, 8>(x, w, a, s);
  }
  return gated ? launch_packed_tiles<2>(x, w, a, n_seg, s) : launch_packed_tiles<1>(x, w, a, n_seg, s);
}

// Segments of a row of K, the planes that sb_gemm_f32_packed_partial writes.
extern "C" int sb_gemm_f32_segments(int n_in) { return (n_in + kSegment - 1) / kSegment; }

// The raw product of float32 X and packed float32 W a segment at a time: partial float [segments][n_rows][n_out], which added
// in ascending order are the bits of sb_gemm_f32_packed.  A block a segment and sixteen columns: with few rows the whole
// product's blocks, whose waves take the segments between them, are a few dozen (3 rows against 896 x 4,864: 56 blocks and
// 15.8 us, 280 and 9.8).
extern "C" int sb_gemm_f32_packed_partial(float *partial, const float *x, const float *w, int n_rows, int n_out, int n_in, void *stream) {
  SB_REQUIRE(partial && x && w, "sb_gemm_f32_packed_partial: null pointer");
  SB_REQUIRE(n_rows >= 0 && n_out > 0 && n_in > 0, "sb_gemm_f32_packed_partial: bad sizes rows=%d out=%d in=%d", n_rows, n_out, n_in);
  SB_SUPPORT(n_rows <= 16, "sb_gemm_f32_packed_partial: %d rows, at most 16", n_rows);
  SB_SUPPORT(n_in % 4 == 0 && size_t(n_in) * 64 * 4 < (size_t(1) << 31), "sb_gemm_f32_packed_partial: inner size %d", n_in);
  SB_SUPPORT((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) % 16 == 0,
             "sb_gemm_f32_packed_partial: operands must be 16-byte aligned");
  if (n_rows == 0) return SB_OK;
  const int n_seg = sb_gemm_f32_segments(n_in);
  SB_SUPPORT(n_seg >= 2 && n_seg <= 65535, "sb_gemm_f32_packed_partial: %d segments", n_seg);
  const PlainArgs a{partial, SB_F32, nullptr, 0, nullptr, n_rows, n_out, n_in, SB_GATE_NONE, by_fours(partial, nullptr, n_out)};
  return launch_one<float, float, kPacked, 1, 1, 1, 1>(x, w, a, (hipStream_t)stream, n_seg);
}
