// bf16 matrix product for a few rows (decode):  Y[t,n] = sum_k X[t,k] W[n,k],
// t <= 64, with the epilogues the model needs (bias, residual, SiLU gate).
//
// The step is bound by reading W once from HBM.  A block owns 16*R output
// features; its four waves take a quarter each of the k-steps of the block's K
// slice, each loading W fragments straight from global
// memory into MFMA operands (16 rows x 64 bytes per load, every byte of W
// read once) and the matching X fragments from cache.  The waves' partial
// tiles are summed through shared memory in wave order, so the result does
// not depend on timing.  When the matrix has too few rows to fill the GPU, K
// is also split over the grid: slices go to a scratch buffer and a second
// kernel adds them in slice order and applies the epilogue.
//
// MFMA roles: A = 16 rows of W, B = 16 rows of X, D[n][t]; a lane then holds
// four consecutive n of one t, a 16-byte store.
#include "gemm_rows.h"
#include "mfma.h"

namespace {

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int kStepK = 32;   // k per MFMA

struct Epilogue {
  void *y;
  int y_dtype;
  const void *bias;
  int bias_dtype;
  const float *resid;
  int n_rows, n_out;
  int gated;
};


__device__ __forceinline__ void store_out(const Epilogue &e, int t, int n, float v) {
  if (e.bias) v = v + ld_dyn(e.bias, e.bias_dtype, n);
  const size_t idx = size_t(t) * e.n_out + n;
  if (e.resid) v = v + e.resid[idx];
  if (e.y_dtype == SB_F32) ((float *)e.y)[idx] = v;
  else ((bf16_t *)e.y)[idx] = f32_to_bf16(v);
}

// G = 1: plain.  G = 2: rows n and n_out + n of W are gate and up of output n.
// PACKED: W is stored tile by tile in MFMA fragment order (ops.pack_weight lays it out): the
// fragment of row tile nb and k-step ks is the 1 KB block (nb * n_steps + ks), lane l's eight
// elements at l * 8; rows and k are padded with zeros to whole tiles.
template <int R, int TT, int G, bool PACKED>
__global__ void __launch_bounds__(kThreads)
gemm_skinny_kernel(const bf16_t *__restrict__ x, const bf16_t *__restrict__ w, Epilogue ep,
                   float *__restrict__ partial, int n_in, int steps_per_slice) {
  extern __shared__ float red[];   // [kWaves][G*R*TT][64][4]
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r = lane & 15, q = lane >> 4;
  const int n0 = blockIdx.x * (16 * R);
  const int n_steps = (n_in + kStepK - 1) / kStepK;
  const int s_begin = blockIdx.y * steps_per_slice;
  const int s_end = min(s_begin + steps_per_slice, n_steps);
  const int n_w_rows = ep.n_out * G;

  floatx4_t acc[G * R][TT];
#pragma unroll
  for (int i = 0; i < G * R; ++i)
#pragma unroll
    for (int j = 0; j < TT; ++j) acc[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};

  const bf16_t *w_row[G * R];
  bool w_ok[G * R];
  const int tiles_out = (ep.n_out + 15) / 16;
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int n = n0 + i * 16 + r;
      if (PACKED) {
        const int tile = blockIdx.x * R + i;
        w_ok[g * R + i] = tile < tiles_out;
        w_row[g * R + i] = w + (size_t(g * tiles_out + min(tile, tiles_out - 1)) * n_steps) * 512 + lane * 8;
      } else {
        w_ok[g * R + i] = n < ep.n_out;
        const int row = min(g * ep.n_out + n, n_w_rows - 1);
        w_row[g * R + i] = w + size_t(row) * n_in;
      }
    }
  const bf16_t *x_row[TT];
  bool x_ok[TT];
#pragma unroll
  for (int j = 0; j < TT; ++j) {
    const int t = j * 16 + r;
    x_ok[j] = t < ep.n_rows;
    x_row[j] = x + size_t(min(t, ep.n_rows - 1)) * n_in;
  }

  // Each wave takes a contiguous quarter of the slice's k-steps, so that it streams whole
  // cache lines of every row; U steps' fragments are requested before the first MFMA, to
  // keep loads in flight.
  constexpr int U = (G * R + TT <= 4) ? 4 : 2;
  const int per_wave = (s_end - s_begin + kWaves - 1) / kWaves;
  const int w_begin = s_begin + wave * per_wave;
  const int w_end = min(w_begin + per_wave, s_end);
  for (int s = w_begin; s < w_end; s += U) {
    uint4 a[U][G * R], b[U][TT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int ss = s + u;
      const int k = ss * kStepK + q * 8;
      // n_in is a multiple of 8: a 16-byte group lies inside a row or outside as a whole
      const bool k_ok = ss < w_end && k < n_in;
#pragma unroll
      for (int i = 0; i < G * R; ++i)
        a[u][i] = PACKED ? ld16(w_row[i] + size_t(ss) * 512, ss < w_end && w_ok[i])
                         : ld16(w_row[i] + k, k_ok && w_ok[i]);
#pragma unroll
      for (int j = 0; j < TT; ++j) b[u][j] = ld16(x_row[j] + k, k_ok && x_ok[j]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < G * R; ++i)
#pragma unroll
        for (int j = 0; j < TT; ++j)
          acc[i][j] = mfma16(as_bf16x8(a[u][i]), as_bf16x8(b[u][j]), acc[i][j]);
  }

  // Sum the waves' partial tiles in wave order.
  constexpr int kTiles = G * R * TT;
#pragma unroll
  for (int i = 0; i < G * R; ++i)
#pragma unroll
    for (int j = 0; j < TT; ++j) {
      float *dst = red + ((size_t(wave) * kTiles + (i * TT + j)) * 64 + lane) * 4;
      *reinterpret_cast<floatx4_t *>(dst) = acc[i][j];
    }
  __syncthreads();

  // Thread e owns lane-quad (tile, lane) pairs: R*TT output tiles of 64 quads.
  for (int e = threadIdx.x; e < R * TT * 64; e += kThreads) {
    const int tile = e >> 6, l = e & 63;
    const int i = tile / TT, j = tile - i * TT;
    floatx4_t v[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int src_tile = (g * R + i) * TT + j;
      floatx4_t sum = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int wv = 0; wv < kWaves; ++wv)
        sum += *reinterpret_cast<const floatx4_t *>(red + ((size_t(wv) * kTiles + src_tile) * 64 + l) * 4);
      v[g] = sum;
    }
    const int t = j * 16 + (l & 15);
    const int nb = n0 + i * 16 + (l >> 4) * 4;
    if (t >= ep.n_rows) continue;
    if (partial != nullptr) {
      // grid split-K: raw sums of this slice, [slice][t][G*n_out]
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (nb + c < ep.n_out)
            partial[(size_t(blockIdx.y) * ep.n_rows + t) * n_w_rows + g * ep.n_out + nb + c] = v[g][c];
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if (nb + c >= ep.n_out) continue;
        float val = v[0][c];
        if (G == 2) val = gate_act(val, ep.gated) * v[1][c];
        store_out(ep, t, nb + c, val);
      }
    }
  }
}

__global__ void __launch_bounds__(256)
reduce_slices_kernel(const float *__restrict__ partial, Epilogue ep, int n_slices) {
  const size_t total = size_t(ep.n_rows) * ep.n_out;
  const size_t idx = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const int t = int(idx / ep.n_out), n = int(idx - size_t(t) * ep.n_out);
  const int width = ep.n_out * (ep.gated ? 2 : 1);
  float g = 0.f, u = 0.f;
  for (int s = 0; s < n_slices; ++s) {
    const float *p = partial + (size_t(s) * ep.n_rows + t) * width;
    g += p[n];
    if (ep.gated) u += p[ep.n_out + n];
  }
  store_out(ep, t, n, ep.gated ? gate_act(g, ep.gated) * u : g);
}

// Gated products of few rows against packed matrices, whole in one launch: a block keeps all S slices of K of its sixteen features
// to itself, so nothing goes through scratch and no second kernel adds and gates.  A wave takes of every slice the k-steps that
// the wave of its number takes in the kernel above, a chain of products for each, the chains step by step side by side; they
// meet in LDS and are added as there, waves within a slice and then slices: the same bits.  A ring of registers runs kAhead
// steps of every chain ahead (chains one after the other, with their ends found as the steps run, kept no load in flight across a
// step: 10.9 us for 6.8 at 4,096 x 2,048).  What bounds it: the read of W, and where blocks are few what one CU pulls.  Measured, three rows,
// us, weights cold, with scratch and the second kernel and so: 11,264 x 2,048 14.9 -> 12.5, 16,384 x 2,048 17.2 -> 14.2, 8,192 x 1,024 8.8 -> 5.8,
// 4,096 x 4,096 13.6 -> 10.5, 1,024 x 2,048 6.6 -> 4.6, 9,728 x 896 (a slice, one launch there too) 7.5 -> 6.5.
// SCALED: a row's factor that follows from its sums of squares ssq [ssq_parts][n_rows] (an unfinished norm) goes into both halves;
// they are asked for ahead of the ring and added up behind it, in the time that W's first loads take (left to the end, and by one
// wave in four, they cost 2 us at 4,096 k).
template <int S, bool SCALED>
__global__ void __launch_bounds__(kThreads)
gemm_skinny_gated_kernel(const bf16_t *__restrict__ x, const bf16_t *__restrict__ w, Epilogue ep, int n_in, int steps_per_slice,
                         const double *__restrict__ ssq, int ssq_parts, float eps) {
  constexpr int kAhead = S == 1 ? 8 : S == 2 ? 4 : S == 3 ? 3 : 2;
  constexpr int kGroups = kThreads / 8, kParts = 8;          // threads a row (of eight) that add its sums of squares; asked for ahead
  __shared__ floatx4_t chains[S * kWaves * 2 * 64];          // [slice][wave][gate, up][lane]
  __shared__ double row_part[SCALED ? kWaves * 8 : 1];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int tile = blockIdx.x, tiles = (ep.n_out + 15) / 16;
  const int n_steps = (n_in + kStepK - 1) / kStepK;
  int begin[S], end[S], longest = 0;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int lo = min(s * steps_per_slice, n_steps), hi = min(lo + steps_per_slice, n_steps), per_wave = (hi - lo + kWaves - 1) / kWaves;
    begin[s] = min(lo + wave * per_wave, hi);
    end[s] = min(begin[s] + per_wave, hi);
    longest = max(longest, end[s] - begin[s]);
  }

  __amdgpu_buffer_rsrc_t rsrc_w[2];
#pragma unroll
  for (int g = 0; g < 2; ++g)
    rsrc_w[g] = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t *>(w) + size_t(g * tiles + tile) * n_steps * 512, 0,
                                                  uint32_t(n_steps) * 1024u, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16_t *>(x), 0, uint32_t(size_t(ep.n_rows) * n_in * 2), 0x00020000);
  constexpr uint32_t kOutside = 0x80000000u;     // past a descriptor's end: reads as zeros
  const uint32_t x_off = r < ep.n_rows ? uint32_t((size_t(r) * n_in + 8 * q) * 2) : kOutside;

  const int sq_row = tid & 7, sq_group = tid >> 3;
  double parts[SCALED ? kParts : 1];
  if constexpr (SCALED) {
    typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
    const __amdgpu_buffer_rsrc_t rsrc_s = __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(ssq), 0,
                                                                            uint32_t(ssq_parts) * uint32_t(ep.n_rows) * 8u, 0x00020000);
#pragma unroll
    for (int i = 0; i < kParts; ++i) {
      const uint32_t at = uint32_t(sq_group + i * kGroups) * uint32_t(ep.n_rows) + sq_row;
      parts[i] = __builtin_bit_cast(double, __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(
          rsrc_s, int(sq_row < ep.n_rows ? at * 8u : kOutside), 0, 0)));
    }
    __builtin_amdgcn_sched_barrier(0);
  }

  uint4 rw[kAhead][S][2], rx[kAhead][S];
  const auto ask = [&](int slot, int s, int j) {             // (a step past the chain's end is zeros on both sides)
    const bool in = begin[s] + j < end[s];
    const int step = in ? begin[s] + j : n_steps;
#pragma unroll
    for (int g = 0; g < 2; ++g)
      rw[slot][s][g] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_w[g], lane * 16 + step * 1024, 0, kReadOnce));
    rx[slot][s] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(
        rsrc_x, int(in && step * kStepK + 8 * q < n_in ? x_off + uint32_t(step) * 64u : kOutside), 0, 0));    // (n_in is a multiple of 8)
  };
#pragma unroll
  for (int u = 0; u < kAhead; ++u)
#pragma unroll
    for (int s = 0; s < S; ++s) ask(u, s, u);
  float factor = 1.0f;
  if constexpr (SCALED) {
    __builtin_amdgcn_sched_barrier(0);
    double sum = 0.0;
#pragma unroll
    for (int i = 0; i < kParts; ++i) sum += parts[i];
    if (sq_row < ep.n_rows)
      for (int p = sq_group + kParts * kGroups; p < ssq_parts; p += kGroups) sum += ssq[size_t(p) * ep.n_rows + sq_row];
    sum += __shfl_xor(sum, 8, 64);
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    if (lane < 8) row_part[wave * 8 + lane] = sum;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // (a barrier for what is in LDS alone: the ring stays in flight)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const int row = (tid >> 2) & 7;                          // of this thread's number of the tile
    sum = (row_part[row] + row_part[8 + row]) + (row_part[16 + row] + row_part[24 + row]);
    factor = 1.0f / sqrtf(float(sum / double(n_in)) + eps);
  }
  floatx4_t acc[S][2];
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int g = 0; g < 2; ++g) acc[s][g] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  const auto multiply = [&](int slot, int s) {
#pragma unroll
    for (int g = 0; g < 2; ++g) acc[s][g] = mfma16(as_bf16x8(rw[slot][s][g]), as_bf16x8(rx[slot][s]), acc[s][g]);
  };
  int j = 0;
  for (; j + kAhead < longest; j += kAhead)
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
#pragma unroll
      for (int s = 0; s < S; ++s) {
        multiply(u, s);
        ask(u, s, j + kAhead + u);
      }
#pragma unroll
  for (int u = 0; u < kAhead; ++u)
#pragma unroll
    for (int s = 0; s < S; ++s) multiply(u, s);
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int g = 0; g < 2; ++g) chains[((s * kWaves + wave) * 2 + g) * 64 + lane] = acc[s][g];
  __syncthreads();

  // a thread a number of the tile, element e of lane l
  static_assert(kThreads == 256, "a thread a number of a tile of 16 x 16");
  const int l = tid >> 2, e = tid & 3, t = l & 15, n = tile * 16 + 4 * (l >> 4) + e;
  if (t >= ep.n_rows || n >= ep.n_out) return;
  const float *at = reinterpret_cast<const float *>(chains) + tid;
  float g = 0.f, u = 0.f;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    float gs = 0.f, us = 0.f;
#pragma unroll
    for (int wv = 0; wv < kWaves; ++wv) gs += at[(s * kWaves + wv) * 512], us += at[(s * kWaves + wv) * 512 + 256];
    g += gs, u += us;
  }
  if constexpr (SCALED) g *= factor, u *= factor;
  store_out(ep, t, n, gate_act(g, ep.gated) * u);
}

// Whether that kernel takes a gated product.  A block streams its share of W at what one CU pulls, whatever the count of blocks,
// so few blocks of a long K are better spread over the GPU in slices, second launch and all.  Three and eight rows, us, in slices
// and whole: 4,096 k, 16 blocks 7.7 and 7.0, 8.2 and 7.7; 32 blocks 8.9 and 8.4, 9.0 and 9.4; 128 blocks 14.0 and 11.6, 14.4 and 13.0;
// 6,144 k, 64 blocks 11.9 and 12.3, 12.1 and 13.8; 128 blocks 16.6 and 15.4, 17.2 and 18.0; 192 blocks 21.0 and 17.9, 22.1 and 18.9;
// 8,192 k, 16 blocks 9.8 and 13.3, 10.1 and 15.4; 128 blocks 21.4 and 19.1, 20.4 and 21.6; 192 blocks 25.6 and 22.1, 26.9 and 23.8;
// 320 blocks 38.5 and 41.5, 40.2 and 44.1; 512 blocks 52.6 and 50.9, 53.9 and 54.2; 16,384 k, 64 blocks 22.1 and 27.2, 22.6 and 31.9;
// 320 blocks 69.0 and 79.7, 70.1 and 86.4.
constexpr int kWholeRows = 8, kWholeSteps = 128, kWholeBlocks = 192, kWholeStepsOfMany = 256;
bool gated_whole(int n_rows, int n_out, int n_in, int n_slices, int packed) {
  const int n_steps = (n_in + kStepK - 1) / kStepK, blocks = (n_out + 15) / 16;
  return packed && n_rows <= kWholeRows &&
         (n_steps <= kWholeSteps || (blocks >= kWholeBlocks && n_steps <= kWholeStepsOfMany) || n_slices == 1) &&
         (unsigned long long)(n_rows + 1) * n_in * 2 < (1ull << 31) &&
         (unsigned long long)n_in * 32 < (1ull << 31);          // 32-bit byte offsets into X and into a stream of W
}

template <int R, int TT, int G, bool PACKED>
void launch(const bf16_t *x, const bf16_t *w, const Epilogue &ep, float *partial, int n_in,
            int n_slices, int steps_per_slice, hipStream_t s) {
  dim3 grid((ep.n_out + 16 * R - 1) / (16 * R), n_slices);
  const size_t lds = size_t(kWaves) * G * R * TT * 64 * 4 * sizeof(float);
  auto kern = gemm_skinny_kernel<R, TT, G, PACKED>;
  static bool raised = false;   // once per instantiation: allow more than the default dynamic LDS
  if (lds > 48 * 1024 && !raised) {
    (void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    raised = true;
  }
  kern<<<grid, kThreads, lds, s>>>(x, w, ep, partial, n_in, steps_per_slice);
}

template <int G, bool PACKED>
void launch_rt(int R, int TT, const bf16_t *x, const bf16_t *w, const Epilogue &ep, float *partial,
               int n_in, int n_slices, int steps_per_slice, hipStream_t s) {
#define SB_CASE(r, tt) \
  if (R == r && TT == tt) \
  return launch<r, tt, G, PACKED>(x, w, ep, partial, n_in, n_slices, steps_per_slice, s)
  SB_CASE(1, 1); SB_CASE(1, 2); SB_CASE(1, 4);
  SB_CASE(2, 1); SB_CASE(2, 2); SB_CASE(2, 4);
  if (G == 1) { SB_CASE(4, 1); SB_CASE(4, 2); SB_CASE(4, 4); }
#undef SB_CASE
}

}  // namespace

// Rows of X this kernel takes at most.
extern "C" int sb_gemm_skinny_max_rows(void) { return 64; }

// Floats of scratch the call may need (0 when it will not split K over the grid).
extern "C" size_t sb_gemm_skinny_scratch(int n_rows, int n_out, int n_in, int gated);

namespace {
struct Plan {
  int R, TT, n_slices, steps_per_slice;
};
Plan plan_for(int n_rows, int n_out, int n_in, int gated) {
  Plan p;
  p.TT = n_rows <= 16 ? 1 : (n_rows <= 32 ? 2 : 4);
  const int tiles = (n_out + 15) / 16;
  // Measured on MI355X.  Up to 16 rows: one row tile per block streams best, and K is cut
  // into slices until about a thousand blocks exist.  More rows: every X fragment a wave loads
  // must serve several row tiles (it comes from L2, and there are TT of them per W fragment), so
  // a wave takes four row tiles (two gated pairs) and fewer, fatter blocks are better.
  const int n_steps = (n_in + kStepK - 1) / kStepK;
  int want_blocks;
  if (p.TT == 1) {
    p.R = 1;
    want_blocks = 1024;
  } else {
    p.R = gated ? 2 : 4;
    want_blocks = 224;
  }
  const int blocks = (tiles + p.R - 1) / p.R;
  int slices = 1;
  if (blocks < want_blocks) {
    slices = (want_blocks + blocks - 1) / blocks;
    const int most = n_steps / (kWaves * 4);   // every wave keeps at least four steps
    if (slices > most) slices = most;
    if (slices > 8) slices = 8;     // what the kernels that add the slices take
    if (slices < 1) slices = 1;
  }
  p.steps_per_slice = (n_steps + slices - 1) / slices;
  p.n_slices = (n_steps + p.steps_per_slice - 1) / p.steps_per_slice;
  return p;
}

template <bool SCALED>
void launch_gated(const Plan &p, const bf16_t *x, const bf16_t *w, const Epilogue &ep, int n_in, const double *ssq, int ssq_parts,
                  float eps, hipStream_t s) {
  switch (p.n_slices) {
#define SB_CASE(n)                                                                                                                   \
  case n: gemm_skinny_gated_kernel<n, SCALED><<<(ep.n_out + 15) / 16, kThreads, 0, s>>>(x, w, ep, n_in, p.steps_per_slice, ssq,      \
                                                                                        ssq_parts, eps); break
    SB_CASE(1); SB_CASE(2); SB_CASE(3); SB_CASE(4); SB_CASE(5); SB_CASE(6); SB_CASE(7);
    default: SB_CASE(8);
#undef SB_CASE
  }
}
}  // namespace

namespace sb {
// A block a tile, or blocks that keep the rows (rows_gated)?  Without a staged X the first is ahead by its shorter start up to 4,096 k,
// but for more than four rows against matrices that take long or are few tiles of long k, where X's fragments from L2 cost more than
// that.  Scaled, us, weights cold, blocks that keep the rows and so, one and eight rows: 1,024 x 1,024 5.1 -> 4.1, 5.2 -> 4.2; 4,864 x 896
// 7.2 -> 6.4, 7.2 -> 6.4; 8,960 x 1,536 13.7 -> 13.2, 14.2 -> 13.9; 5,632 x 2,048 11.9 -> 11.8, 11.3 and 11.6; 11,008 x 2,048 18.1 -> 17.2, 17.6
// -> 17.2; 9,728 x 2,560 21.0 -> 20.9, 26.6 -> 21.3; 4,096 x 4,096 14.0 -> 13.8, 14.0 -> 13.3; 2,048 x 4,096 10.3 and 10.5, 10.5 and 11.3; 18,944 x
// 3,584 45.8 -> 45.0, 43.6 and 44.2.  Not scaled: 4,864 x 896 7.3 -> 5.7, 7.4 -> 6.0; 18,944 x 1,024 15.9 -> 13.5, 16.0 -> 13.8; 8,960 x 1,536
// 13.2 -> 12.4, 13.5 and 13.6; 11,008 x 2,048 18.0 -> 16.7, 17.4 -> 16.9; 14,336 x 4,096 40.5 -> 39.9, 40.4 and 41.9.
bool tile_gated_pays(int n_rows, int n_out, int n_in) {
  constexpr long long kLong = 26ll << 20;
  return n_rows > 0 && n_rows <= kWholeRows && n_out > 0 && n_in >= 512 && n_in <= kWholeSteps * kStepK && n_in % 8 == 0 &&
         (n_rows <= 4 || ((long long)n_out * n_in <= kLong && (n_in <= 2048 || n_out > 2048))) &&
         gated_whole(n_rows, n_out, n_in, plan_for(n_rows, n_out, n_in, 1).n_slices, 1);
}
int tile_gated(void *y, const void *x, const double *ssq, int ssq_parts, float eps, const void *w, int n_rows, int n_out, int n_in,
               int gate, void *stream) {
  SB_REQUIRE(tile_gated_pays(n_rows, n_out, n_in), "tile_gated: sizes that it does not take");
  const Plan p = plan_for(n_rows, n_out, n_in, 1);
  const Epilogue ep{y, SB_BF16, nullptr, 0, nullptr, n_rows, n_out, gate};
  if (ssq) launch_gated<true>(p, (const bf16_t *)x, (const bf16_t *)w, ep, n_in, ssq, ssq_parts, eps, (hipStream_t)stream);
  else launch_gated<false>(p, (const bf16_t *)x, (const bf16_t *)w, ep, n_in, nullptr, 0, 0.f, (hipStream_t)stream);
  return sb::check_launch("tile_gated");
}
}  // namespace sb

extern "C" size_t sb_gemm_skinny_scratch(int n_rows, int n_out, int n_in, int gated) {
  if (n_rows <= 0 || n_out <= 0 || n_in <= 0) return 0;
  const Plan p = plan_for(n_rows, n_out, n_in, gated);
  return p.n_slices > 1 ? size_t(p.n_slices) * n_rows * n_out * (gated ? 2 : 1) : 0;
}

// Y = X W^T (+bias) (+resid), or with gated != 0: Y = silu(X Wg^T) * (X Wu^T) where W = [Wg; Wu]
// is [2*n_out, n_in].  X [n_rows, n_in] and W are bf16; n_rows <= 64; n_in a multiple of 8.
// packed != 0: W is in the packed tile layout.
extern "C" int sb_gemm_skinny_bf16(void *y, int y_dtype, const void *x, const void *w, const void *bias,
                                   int bias_dtype, const float *resid, int n_rows, int n_out, int n_in,
                                   int gated, int packed, float *scratch, size_t scratch_floats,
                                   void *stream) {
  SB_REQUIRE(y && x && w, "sb_gemm_skinny_bf16: null pointer");
  SB_REQUIRE(n_rows >= 0 && n_out > 0 && n_in > 0, "sb_gemm_skinny_bf16: bad sizes rows=%d out=%d in=%d",
             n_rows, n_out, n_in);
  SB_REQUIRE(sb::valid_dtype(y_dtype) && (!bias || sb::valid_dtype(bias_dtype)),
             "sb_gemm_skinny_bf16: unknown dtype");
  SB_SUPPORT(n_rows <= 64, "sb_gemm_skinny_bf16: %d rows, at most 64", n_rows);
  SB_SUPPORT(n_in % 8 == 0, "sb_gemm_skinny_bf16: inner size %d is not a multiple of 8", n_in);
  SB_SUPPORT((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) % 16 == 0,
             "sb_gemm_skinny_bf16: operands must be 16-byte aligned");
  SB_REQUIRE(!(gated && (bias || resid)), "sb_gemm_skinny_bf16: the gated form takes no bias or residual");
  if (n_rows == 0) return SB_OK;
  const Plan p = plan_for(n_rows, n_out, n_in, gated);
  const size_t need = p.n_slices > 1 ? size_t(p.n_slices) * n_rows * n_out * (gated ? 2 : 1) : 0;
  SB_REQUIRE(need == 0 || (scratch && scratch_floats >= need),
             "sb_gemm_skinny_bf16: scratch of %zu floats needed, %zu given", need, scratch_floats);
  hipStream_t s = (hipStream_t)stream;
  SB_SUPPORT(gated >= SB_GATE_NONE && gated <= SB_GATE_RELU, "sb_gemm_skinny_bf16: unknown gate activation %d", gated);
  Epilogue ep{y, y_dtype, bias, bias_dtype, resid, n_rows, n_out, gated};
  float *partial = p.n_slices > 1 ? scratch : nullptr;
  const bf16_t *xb = (const bf16_t *)x, *wb = (const bf16_t *)w;
  if (gated && gated_whole(n_rows, n_out, n_in, p.n_slices, packed)) {
    launch_gated<false>(p, xb, wb, ep, n_in, nullptr, 0, 0.f, s);
    return sb::check_launch("sb_gemm_skinny_bf16");
  }
  if (gated && packed) launch_rt<2, true>(p.R, p.TT, xb, wb, ep, partial, n_in, p.n_slices, p.steps_per_slice, s);
  else if (gated) launch_rt<2, false>(p.R, p.TT, xb, wb, ep, partial, n_in, p.n_slices, p.steps_per_slice, s);
  else if (packed) launch_rt<1, true>(p.R, p.TT, xb, wb, ep, partial, n_in, p.n_slices, p.steps_per_slice, s);
  else launch_rt<1, false>(p.R, p.TT, xb, wb, ep, partial, n_in, p.n_slices, p.steps_per_slice, s);
  int rc = sb::check_launch("sb_gemm_skinny_bf16");
  if (rc != SB_OK) return rc;
  if (p.n_slices > 1) {
    const size_t total = size_t(n_rows) * n_out;
    reduce_slices_kernel<<<unsigned((total + 255) / 256), 256, 0, s>>>(scratch, ep, p.n_slices);
    rc = sb::check_launch("sb_gemm_skinny_bf16 (slice sum)");
  }
  return rc;
}

// K slices sb_gemm_skinny_partial_bf16 will produce for these sizes.
extern "C" int sb_gemm_skinny_slices(int n_rows, int n_out, int n_in) {
  if (n_rows <= 0 || n_out <= 0 || n_in <= 0) return 1;
  return plan_for(n_rows, n_out, n_in, 0).n_slices;
}

// The raw product in K slices, for a consumer that adds them (and bias, residual, ...) itself:
// partial float [slices][n_rows][n_out], slices = sb_gemm_skinny_slices(...), slice s holding
// sum over its k range of X[t,k] W[n,k].
extern "C" int sb_gemm_skinny_partial_bf16(float *partial, const void *x, const void *w, int n_rows,
                                           int n_out, int n_in, int packed, void *stream) {
  SB_REQUIRE(partial && x && w, "sb_gemm_skinny_partial_bf16: null pointer");
  SB_REQUIRE(n_rows >= 0 && n_out > 0 && n_in > 0, "sb_gemm_skinny_partial_bf16: bad sizes");
  SB_SUPPORT(n_rows <= 64, "sb_gemm_skinny_partial_bf16: %d rows, at most 64", n_rows);
  SB_SUPPORT(n_in % 8 == 0, "sb_gemm_skinny_partial_bf16: inner size %d is not a multiple of 8", n_in);
  SB_SUPPORT((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) % 16 == 0,
             "sb_gemm_skinny_partial_bf16: operands must be 16-byte aligned");
  if (n_rows == 0) return SB_OK;
  const Plan p = plan_for(n_rows, n_out, n_in, 0);
  Epilogue ep{nullptr, SB_F32, nullptr, 0, nullptr, n_rows, n_out, 0};
  const bf16_t *xb = (const bf16_t *)x, *wb = (const bf16_t *)w;
  hipStream_t s = (hipStream_t)stream;
  if (packed) launch_rt<1, true>(p.R, p.TT, xb, wb, ep, partial, n_in, p.n_slices, p.steps_per_slice, s);
  else launch_rt<1, false>(p.R, p.TT, xb, wb, ep, partial, n_in, p.n_slices, p.steps_per_slice, s);
  return sb::check_launch("sb_gemm_skinny_partial_bf16");
}
