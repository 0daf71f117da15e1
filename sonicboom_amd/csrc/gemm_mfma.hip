// bf16 matrix product for many rows (prefill):  Y[t,n] = sum_k X[t,k] W[n,k]
// on the matrix cores, with the model's epilogues fused: bias, float32
// residual, gate activation, float32 or bfloat16 output.  Five kernels: this one, of any inner size in
// eights and weights of either layout, three below it that load packed weights and rows straight into LDS, and one of gated products
// that loads rows so and keeps weights in registers.
//
// A block of 2 x NW waves owns a BM x BN tile of Y (128 x 128, 256 x 128 or
// 256 x 256) and walks K in stages of BK.  Both operand tiles go
// global -> registers -> LDS, the next stage's loads being issued before the
// current stage's MFMAs (two LDS buffers, one barrier per stage).  An LDS row
// holds BK k (BK / 8 chunks of 16 bytes); chunk c of row r is stored at chunk
// c ^ f(r), f chosen so that the 16-byte fragment reads of sixteen consecutive
// rows fall on distinct banks.  A wave owns (BM / 2) x 64: MT x 2 tiles of
// v_mfma_f32_32x32x16_bf16, A = rows of X, B = rows of W, so a lane holds one
// output column of 16 rows.  The taller tile halves the LDS reads per MFMA;
// the launcher picks the shape from the problem's sizes.
//
// Block order: consecutive block numbers go to different XCDs (each with its
// own L2).  The grid is walked so that the blocks one XCD runs at a time share
// their X rows and neighbouring W rows.
#include <type_traits>

#include "mfma.h"

namespace {

constexpr int kXcds = 8;

// The gate's activation in the epilogue of a tile: gate_act, with SiLU's exponential and division put together from the
// vector units' own exp2 and reciprocal for |g| < 87, where neither runs out of the range.  exp(-g) = 2^n 2^a, n the whole
// number nearest to the product with log2(e) and a what is left of it, log2(e) in two parts; one Newton step on the quotient
// rounds it like a division.  Against 64 bits, 2^24 numbers each of [-88.7, -80], [-80, -20], [-20, -1], [-1, 1] and [0, 120]:
// the errors are those of expf and the full division (at most 2.1, 2.3, 3.1, 2.5 and 2.0 units of 2^-24, root mean squares
// 0.61, 0.61, 0.64, 0.67 and 0.26), from which 20 of the numbers differ at all.  The compiler's expf and division cost a
// 256 x 256 tile's epilogue 8.5 us of vector instructions, 9 % of the tile at 3,584 k; this form is level with one that reduces
// nothing and was up to 4.3 units off (2,048 x 37,888 x 3,584 448 and 447 us, 16,384 rows 3.32 and 3.32 ms, 6,398 x 22,016 x
// 2,048 484 and 483 us).
// FAR: some number of the wave's tile lies outside; those take gate_act.
constexpr float kSiluRange = 87.0f;
template <int GATE, bool FAR>
__device__ __forceinline__ float tile_gate(float g) {
  if constexpr (GATE != SB_GATE_SILU) {
    return gate_act(g, GATE);
  } else {
#pragma clang fp contract(off)                   // (h - n fused into one operation would count h's rounding twice)
    constexpr float kMagic = 12582912.0f;        // 1.5 * 2^23: adding it rounds to whole numbers, n in the sum's low bits
    const float h = g * -1.44269502f, t = h + kMagic;
    const float l = fmaf(g, -1.92596303e-8f, fmaf(g, -1.44269502f, -h));
    const uint32_t e = __float_as_uint(__builtin_amdgcn_exp2f((h - (t - kMagic)) + l));
    const float d = 1.0f + __uint_as_float((__float_as_uint(t) << 23) + e);
    const float r = __builtin_amdgcn_rcpf(d), q = g * r;
    const float y = fmaf(fmaf(-d, q, g), r, q);
    if constexpr (FAR) {
      const float full = gate_act(g, SB_GATE_SILU);
      return fabsf(g) >= kSiluRange ? full : y;
    }
    return y;
  }
}
// Whether FAR holds; COUNT numbers a lane, the i-th of them number(i).  (Passes a NaN over: it is one in y already.)
template <int GATE, int COUNT, class Number>
__device__ __forceinline__ bool silu_far(Number number) {
  if constexpr (GATE != SB_GATE_SILU) return false;
  float largest = 0.0f;
#pragma unroll
  for (int i = 0; i < COUNT; ++i) largest = fmaxf(largest, fabsf(number(i)));
  return __any(largest >= kSiluRange);
}
typedef uint16_t u16x4_t __attribute__((ext_vector_type(4)));

struct Args {
  void *y;
  int y_dtype;
  const bf16_t *x, *w;
  const void *bias;
  int bias_dtype;
  const float *resid;
  float resid_scale;   // Y = resid_scale * (X W^T + bias) + resid  (1 unless a branch has a multiplier)
  int n_rows, n_out, n_in;
  int relu_sq;     // 1: Y = max(X W^T + bias, 0)^2 (no residual, whole products)
  const void *act_params; int act_dtype;      // xIELU's two numbers (kernels built for it)
  int gated;       // an sb_gate; not 0: W is [2*n_out, n_in], rows n (gate) and n_out + n (up)
  int tiles_m, tiles_n;
  int w_tiles;     // packed W: 16-row tiles of one half (ceil(n_out / 16))
  int w_steps;     // packed W: 32-wide k-steps (ceil(n_in / 32))
  // K cut over the grid (blockIdx.y): slice s multiplies stages [s * stages_per_slice, ...) and
  // writes its raw sums to partial [slice][n_rows][n_out]; NULL: one slice, the epilogues below
  float *partial;
  int stages_per_slice;
  int vec4;        // n_out % 4 == 0 and y, resid, partial 16-byte aligned: four outputs of a row at a time
};

// index (in 16-byte chunks) of chunk `chunk` of LDS row `row`, CPR chunks per row
template <class T>
constexpr int const_of() {
  if constexpr (std::is_integral<T>::value) return 0;
  else return T::value;
}

template <int CPR>
__device__ __forceinline__ int swz(int row, int chunk) {
  return row * CPR + (chunk ^ ((row / (16 / CPR)) & (CPR - 1)));
}


// Which tile of Y block number `block` of the grid owns (a block that goes on to further tiles
// asks for the numbers one grid apart).  XCD-aware order: hardware sends block b to XCD b % 8.  XCD x
// gets the contiguous run of tiles [x * per, (x + 1) * per), which share rows of X and W in that
// XCD's L2; the grid is padded to a multiple of eight blocks, and the blocks past the last tile
// get false and leave at once.  The tiles are walked in bands of kBand tiles along M: inside a
// band m runs fastest, then n, and the bands follow one another.  The thirty-odd blocks that an
// XCD runs at a time then cover a patch of kBand x 4 tiles and share their rows of X and of W in
// its L2, where one column of all M tiles would read a different piece of X for every block.
__device__ __forceinline__ bool tile_of_block(const Args &a, int block, int &tm, int &tn) {
  const int n_blocks = a.tiles_m * a.tiles_n;
  const int per_xcd = (n_blocks + kXcds - 1) / kXcds;
  const int bid = (block % kXcds) * per_xcd + block / kXcds;
  if (block / kXcds >= per_xcd || bid >= n_blocks) return false;
  constexpr int kBand = 8;
  const int band = bid / (kBand * a.tiles_n), in_band = bid - band * (kBand * a.tiles_n);
  const int band_m = min(kBand, a.tiles_m - band * kBand);       // the last band may be lower
  tn = in_band / band_m;
  tm = band * kBand + (in_band - tn * band_m);
  return true;
}

// The epilogue of a block's tile.  The matrix cores leave a lane with single elements of many
// rows (32 x 32 tiles: sixteen rows of one column), which stored as they lie would be sixty-four
// 2- or 4-byte stores a lane.  The caller has ended its last stage with a barrier, so LDS is
// free: each wave turns SLAB rows at a time through a float area of its own (`fill(i, area)` puts
// rows SLAB i .. SLAB (i + 1) - 1 of the wave's tile there, row r at area + r * PITCH, with the gate
// already applied) and takes them out again four columns a lane, whole rows side by side, for 8-
// or 16-byte loads of the residual and stores of the result.  The wave's LDS operations run in
// program order, so a fence for the compiler is all the ordering it needs.
// SLABS groups of SLAB rows (32 or 16) make a wave's rows, NW: waves along N, NC: output columns
// of a wave; `lds_f`: at least (waves of the block) * SLAB * PITCH floats.
// SWZ (PITCH = NC = 64, SLAB 16): no padding, the four quarters of row r turned round by r / 4.
template <int SLABS, int SLAB, int NW, int NC, int PITCH, bool SWZ = false, class Fill>
__device__ __forceinline__ void store_tile(const Args &a, float *lds_f, int t0, int n0, bool raw_allowed, Fill fill) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int wm = wave / NW, wn = wave % NW;
  constexpr int kLanesPerRow = NC / 4, kRowsPerPass = 64 / kLanesPerRow, kPasses = SLAB / kRowsPerPass;
  static_assert(SLAB % kRowsPerPass == 0, "whole passes");
  float *turn = lds_f + wave * (SLAB * PITCH);
  const int r_in = lane / kLanesPerRow, c4 = (lane % kLanesPerRow) * 4;
  const int n_first = n0 + wn * NC + c4;              // first of this lane's four columns
  const bool raw = raw_allowed && a.partial;          // K slices: raw sums to the slice's plane
  float *y_f = raw ? a.partial + size_t(blockIdx.y) * a.n_rows * a.n_out : (float *)a.y;
  bf16_t *y_h = (bf16_t *)a.y;
  const bool f32_out = raw || a.y_dtype == SB_F32;
  const void *bias = raw ? nullptr : a.bias;
  const float *resid = raw ? nullptr : a.resid;
#pragma unroll
  for (int i = 0; i < SLABS; ++i) {
    fill(i, turn);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
      const int r = p * kRowsPerPass + r_in;
      const int t = t0 + wm * (SLABS * SLAB) + i * SLAB + r;
      floatx4_t v = *reinterpret_cast<const floatx4_t *>(turn + r * PITCH + (SWZ ? c4 ^ (((r >> 2) & 3) * 16) : c4));
      if (t >= a.n_rows || n_first >= a.n_out) continue;
      const size_t idx = size_t(t) * a.n_out + n_first;
      if (a.vec4) {
        if (bias) {
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] = v[q] + ld_dyn(bias, a.bias_dtype, n_first + q);
        }
        if (a.relu_sq) {
#pragma unroll
          for (int q = 0; q < 4; ++q) { const float z = fmaxf(v[q], 0.0f); v[q] = z * z; }
        }
        if (resid) {
          const floatx4_t rv = *reinterpret_cast<const floatx4_t *>(resid + idx);
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] = v[q] * a.resid_scale + rv[q];
        }
        if (f32_out) {
          *reinterpret_cast<floatx4_t *>(y_f + idx) = v;
        } else {
          u16x4_t h;
#pragma unroll
          for (int q = 0; q < 4; ++q) h[q] = f32_to_bf16(v[q]);
          *reinterpret_cast<u16x4_t *>(y_h + idx) = h;
        }
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (n_first + q >= a.n_out) continue;
          float u = v[q];
          if (bias) u = u + ld_dyn(bias, a.bias_dtype, n_first + q);
          if (a.relu_sq) { const float z = fmaxf(u, 0.0f); u = z * z; }
          if (resid) u = u * a.resid_scale + resid[idx + q];
          if (f32_out) y_f[idx + q] = u;
          else y_h[idx + q] = f32_to_bf16(u);
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

// The filling of the turning area from 32 x 32 tiles: acc[i][j][e] is row 8 * (e / 4) +
// 4 * (lane / 32) + e % 4, column lane % 32 of tile (i, j).  PITCH = NC + 8: rows four apart fall on
// the other half of the banks.
template <int MT, int GATED, bool FAR>
__device__ __forceinline__ void fill_from_32(floatx16_t (&acc)[MT][2], int i, float *turn) {
  constexpr int kPitch = (GATED ? 32 : 64) + 8;
  const int lane = threadIdx.x & 63, col = lane & 31, row_base = (lane >> 5) * 4;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const int row = 8 * (e >> 2) + row_base + (e & 3);
    if (GATED) {
      turn[row * kPitch + col] = tile_gate<GATED, FAR>(acc[i][0][e]) * acc[i][1][e];   // GATED: the sb_gate, fixed at compile time
    } else {
      turn[row * kPitch + col] = acc[i][0][e];
      turn[row * kPitch + 32 + col] = acc[i][1][e];
    }
  }
}

// PACKED: W comes in the packed tile layout (1 KB blocks of 16 rows x 32 k in fragment order,
// zero padded), which makes its global loads contiguous and free of bounds checks.
// MT: 32-row tiles of a wave (the block has two waves along M), NW: waves along N (64 columns
// each), DEPTH: stages the global loads run ahead of the products.
template <int MT, int NW, int BK, int DEPTH, int GATED, bool PACKED, bool EVEN_K>
__global__ void __launch_bounds__(128 * NW)
gemm_mfma_kernel(Args a) {
  constexpr int BM = 64 * MT, BN = 64 * NW, kThreads = 128 * NW;
  constexpr int CPR = BK / 8;                       // 16-byte chunks in an LDS row
  constexpr int kLoadsA = BM * CPR / kThreads;
  constexpr int kLoadsB = BN * CPR / kThreads;
  constexpr int kLoads = kLoadsA + kLoadsB;
  constexpr int kSteps32 = BK / 32;                 // packed k-steps in a stage
  constexpr int kSteps16 = BK / 16;                 // MFMA k-steps in a stage
  constexpr int kMfmas = 2 * MT;                    // MFMAs of a wave per k-step
  // 16-byte chunks travel as first-class vectors, so the staging arrays stay in registers
  extern __shared__ bf16x8_t lds[];
  bf16x8_t *lds_a0 = lds, *lds_a1 = lds + BM * CPR;
  bf16x8_t *lds_b0 = lds + 2 * BM * CPR, *lds_b1 = lds_b0 + BN * CPR;

  int tm, tn;
  if (!tile_of_block(a, int(blockIdx.x), tm, tn)) return;
  const int t0 = tm * BM;
  const int n0 = tn * (GATED ? BN / 2 : BN);

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int wm = wave / NW, wn = wave % NW;

  // Global -> register staging: load i of a thread takes chunk id tid + kThreads * i of the
  // stage.  Buffer loads: a descriptor per operand in scalar registers, one 32-bit byte offset
  // per load, the stage's offset along K as the scalar offset; what lies past the operand's end
  // reads as zero, which covers the rows past the last one.  Chunks past the end of K inside a
  // row have to be zeroed by hand (EVEN_K: there are none).  Load i + 1 lands kThreads chunks
  // after load i in LDS (its rows are a multiple of 16 further on, so the swizzle term repeats).
  static_assert((kThreads / CPR) % 16 == 0, "rows per load must keep the swizzle term");
  // Byte offset of load i at stage 0.  With packed weights the loads of an operand lie a constant
  // stride apart (nothing is clamped: what lies past an operand's end is out of the descriptor's
  // range and reads as zero), so two offsets and two strides stand for all of them; kept as an
  // array they did not fit the registers beside 128 accumulators, and the one the compiler
  // spilled came back through a scratch load whose wait (the memory counter runs in order) also
  // waited for every global load just issued, once in every two stages.
  constexpr bool kLinear = PACKED && (kThreads / 64) % kSteps32 == 0 &&
                           (!GATED || (kThreads / 64 / kSteps32) % 4 == 0);   // see the loads of W below
  constexpr int kOffsets = kLinear ? 2 : kLoads;
  uint32_t off[kOffsets];
  uint32_t stride_a = 0, stride_b = 0;
  int kpos[kLoads];           // !EVEN_K: first k of the chunk within the stage (packed: of its k-step)
  int slot_a0, slot_b0;       // LDS chunk index of loads 0 of A and of B
  const size_t w_rows_total = size_t(GATED ? 2 : 1) * (PACKED ? size_t(a.w_tiles) * 16 : size_t(a.n_out));
  const size_t w_row_bytes = PACKED ? size_t(a.w_steps) * 64 : size_t(a.n_in) * 2;
  const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16_t *>(a.x), 0, uint32_t(size_t(a.n_rows) * a.n_in * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16_t *>(a.w), 0, uint32_t(w_rows_total * w_row_bytes), 0x00020000);
#pragma unroll
  for (int i = 0; i < kLoadsA; ++i) {
    const int id = tid + kThreads * i, row = id / CPR, c = id % CPR;
    if (kLinear) {
      // rows past the last one lie past the descriptor's end (the host has checked that their
      // offsets still fit 32 bits)
      if (i == 0) off[0] = uint32_t((size_t(t0 + row) * a.n_in + c * 8) * 2);
      stride_a = uint32_t(size_t(kThreads / CPR) * a.n_in * 2);
    } else {
      const int t = min(t0 + row, a.n_rows);          // n_rows: one past the end, reads zeros
      off[i] = uint32_t((size_t(t) * a.n_in + c * 8) * 2);
    }
    if (i == 0) slot_a0 = swz<CPR>(row, c);
    kpos[i] = c * 8;
  }
#pragma unroll
  for (int i = 0; i < kLoadsB; ++i) {
    const int id = tid + kThreads * i;
    if (PACKED) {
      // load id -> 1 KB block (id / 64) = (row tile of the LDS tile, k-step), lane id % 64
      const int blk = id >> 6, l = id & 63;
      const int rt = blk / kSteps32, j = blk % kSteps32;   // LDS rows rt * 16 .., k-step j of the stage
      if constexpr (kLinear) {
        // load i + 1 takes the block kThreads / 64 further on: the same k-step, row tile
        // rt + kThreads / 64 / kSteps32, which is a constant number of tiles of W further on
        if (i == 0) {
          int tile;
          if (GATED) {
            const int half = rt >> 2, within = rt & 3;
            tile = (within >> 1) * a.w_tiles + n0 / 16 + half * 2 + (within & 1);
          } else {
            tile = n0 / 16 + rt;
          }
          // a tile past the last: past the half's (or the matrix's) end; its columns are not stored
          off[1] = uint32_t(((size_t(tile) * a.w_steps + j) * 512 + size_t(l) * 8) * 2);
          constexpr int kTilesApart = GATED ? (kThreads / 64 / kSteps32) / 2 : kThreads / 64 / kSteps32;
          stride_b = uint32_t(size_t(kTilesApart) * a.w_steps * 1024);
        }
      } else {
        int tile;
        if (GATED) {
          const int half = rt >> 2, within = rt & 3;
          tile = (within >> 1) * a.w_tiles + min(n0 / 16 + half * 2 + (within & 1), a.w_tiles - 1);
        } else {
          tile = min(n0 / 16 + rt, a.w_tiles - 1);
        }
        off[kLoadsA + i] = uint32_t(((size_t(tile) * a.w_steps + j) * 512 + size_t(l) * 8) * 2);
      }
      if (i == 0) slot_b0 = swz<CPR>(rt * 16 + (l & 15), j * 4 + (l >> 4));
      kpos[kLoadsA + i] = j * 32;
    } else {
      const int row = id / CPR, c = id % CPR;
      int wrow;       // the row of W that feeds LDS row `row`
      if (GATED) {
        // LDS rows [0,32) gate of features n0..n0+31, [32,64) up of the same, [64,96) gate of
        // n0+32.., [96,128) up of the same: a wave's two B tiles are gate and up of 32 features.
        const int half = row >> 6, within = row & 63, is_up = within >> 5;
        wrow = is_up * a.n_out + min(n0 + half * 32 + (within & 31), a.n_out - 1);
      } else {
        wrow = min(n0 + row, a.n_out - 1);
      }
      off[kLoadsA + i] = uint32_t((size_t(wrow) * a.n_in + c * 8) * 2);
      if (i == 0) slot_b0 = swz<CPR>(row, c);
      kpos[kLoadsA + i] = c * 8;
    }
  }

  floatx16_t acc[MT][2];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // DEPTH 2, two register sets: while stage kt is multiplied out of LDS, stage kt + 1 waits in
  // one set (its loads went out a stage earlier) and the loads of stage kt + 2 go out into the
  // other.  DEPTH 1, one set: the loads of stage kt + 1 go out in the first half of stage kt.
  const int n_k_all = (a.n_in + BK - 1) / BK;
  const int kt_begin = a.partial ? int(blockIdx.y) * a.stages_per_slice : 0;
  const int n_k = a.partial ? min(kt_begin + a.stages_per_slice, n_k_all) : n_k_all;   // end of this slice
  constexpr uint32_t kPastEnd = 0xfff00000u;      // the host keeps every operand below this size
  bf16x8_t staged[DEPTH][kLoads];
  auto issue_load = [&](auto SET, int i, int kt) {
    constexpr int set = decltype(SET)::value;
    const bool is_a = i < kLoadsA;
    // uniform part of the address: the stage's offset along K
    int stage_off = (PACKED && !is_a) ? kt * (kSteps32 * 1024) : kt * (BK * 2);
    uint32_t offset;
    if constexpr (kLinear) offset = is_a ? off[0] + uint32_t(i) * stride_a : off[1] + uint32_t(i - kLoadsA) * stride_b;
    else offset = off[i];
    // a stage past the end of K (of this slice): an offset past every operand, which reads as zeros
    // (with no scalar offset on top, so that the sum cannot wrap around into the operand)
    if (DEPTH == 2 && kt >= n_k) { offset |= kPastEnd; stage_off = 0; }
    bf16x8_t v = __builtin_bit_cast(
        bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(is_a ? rsrc_x : rsrc_w, int(offset), stage_off, 0));
    if (!EVEN_K) {
      const bool ok = (PACKED && !is_a) ? (kt * BK + kpos[i] < a.w_steps * 32) : (kt * BK + kpos[i] < a.n_in);
      if (!ok) v = bf16x8_t{0, 0, 0, 0, 0, 0, 0, 0};
    }
    staged[set][i] = v;
  };
  auto store_lds = [&](auto SET, int i, int buf) {
    constexpr int set = decltype(SET)::value;
    if (i < kLoadsA) (buf ? lds_a1 : lds_a0)[slot_a0 + i * kThreads] = staged[set][i];
    else (buf ? lds_b1 : lds_b0)[slot_b0 + (i - kLoadsA) * kThreads] = staged[set][i];
  };

  using Set0 = std::integral_constant<int, 0>;
  using Set1 = std::integral_constant<int, 1>;
#pragma unroll
  for (int i = 0; i < kLoads; ++i) issue_load(Set0{}, i, kt_begin);
  if (DEPTH == 2) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) issue_load(std::integral_constant<int, DEPTH - 1>{}, i, kt_begin + 1);
  }
#pragma unroll
  for (int i = 0; i < kLoads; ++i) store_lds(Set0{}, i, 0);
  __syncthreads();

  // fragment reads: lane -> row lane % 32 of a 32-row tile, chunk 2 * ks + lane / 32 of the stage
  const int frag_row = lane & 31, frag_c = lane >> 5;
  const int frag_sw = (frag_row / (16 / CPR)) & (CPR - 1);     // swizzle term, equal for all tiles of a wave
  const int a_row0 = (wm * (32 * MT) + frag_row) * CPR, b_row0 = (wn * 64 + frag_row) * CPR;

  // One stage.  CUR: LDS buffer of this stage (and with two register sets the free one); LOAD: the
  // stage to load (kt + DEPTH) exists, STORE: stage kt + 1 exists.  The memory operations are spread between the MFMAs in the source
  // so that the matrix pipe keeps running while they issue.
  auto stage = [&](auto CUR, auto LOAD, auto STORE, int kt) {
    // CUR: a constant with two register sets (it names the set too); with one set it may be a
    // plain int, and then one copy of the stage serves both LDS buffers
    constexpr bool kFixed = !std::is_integral<decltype(CUR)>::value;
    const int cur = int(CUR);
    constexpr bool do_load = decltype(LOAD)::value, do_store = decltype(STORE)::value;
    using SetCur = std::integral_constant<int, DEPTH == 2 ? const_of<decltype(CUR)>() : 0>;          // set to load into
    using SetNext = std::integral_constant<int, DEPTH == 2 ? (const_of<decltype(CUR)>() ^ 1) : 0>;   // set to store from
    static_assert(kFixed || DEPTH == 1, "two register sets need the buffer as a constant");
    const bf16x8_t *la = cur ? lds_a1 : lds_a0, *lb = cur ? lds_b1 : lds_b0;
    bf16x8_t frag[2][MT + 2];
    auto read_frag = [&](int fs, int ks, int f) {
      const int c = (ks * 2 + frag_c) ^ frag_sw;
      frag[fs][f] = f < MT ? la[a_row0 + f * 32 * CPR + c] : lb[b_row0 + (f - MT) * 32 * CPR + c];
    };
#pragma unroll
    for (int f = 0; f < MT + 2; ++f) read_frag(0, 0, f);
    constexpr int kSlots = kSteps16 * kMfmas;           // MFMAs of the stage = places to put other work
    constexpr int kHalf = kSlots / 2;
#pragma unroll
    for (int ks = 0; ks < kSteps16; ++ks) {
#pragma unroll
      for (int m = 0; m < kMfmas; ++m) {
        const int i = m >> 1, j = m & 1, at = ks * kMfmas + m;
        acc[i][j] = mfma32(frag[ks & 1][i], frag[ks & 1][MT + j], acc[i][j]);
        // fragments of the next k-step, one read after each of the first MFMAs
        if (ks + 1 < kSteps16 && m < MT + 2) read_frag((ks + 1) & 1, ks + 1, m);
        // loads of stage kt + DEPTH over the first half of the stage
        if (do_load && at < kHalf) {
#pragma unroll
          for (int l = 0; l < kLoads; ++l)
            if (l >= at * kLoads / kHalf && l < (at + 1) * kLoads / kHalf)
              issue_load(SetCur{}, l, DEPTH == 1 ? min(kt + 1, n_k - 1) : kt + DEPTH);
        }
        // stage kt + 1 into the other LDS buffer over the second half: nobody reads that buffer
        // since the last barrier
        if (do_store && at >= kHalf) {
#pragma unroll
          for (int l = 0; l < kLoads; ++l)
            if (l >= (at - kHalf) * kLoads / kHalf && l < (at - kHalf + 1) * kLoads / kHalf)
              store_lds(SetNext{}, l, cur ^ 1);
        }
        // keep this order: left alone, the scheduler gathers the memory operations into lumps
        // and reads each fragment right before its MFMA, and the matrix pipe waits on both
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();
  };
  using Yes = std::true_type;
  using No = std::false_type;
  int kt = kt_begin;
  if constexpr (DEPTH == 2) {
    // Pairs of stages, one for each register set, and nothing peeled off at the end: with an odd
    // count the last pair's second stage multiplies zeros (its loads were aimed past the end).
    for (; kt < n_k; kt += 2) {
      stage(Set0{}, Yes{}, Yes{}, kt);
      stage(Set1{}, Yes{}, Yes{}, kt + 1);
    }
  } else {
    // One copy of the stage for every k, the LDS buffer as a variable: the accumulators stay in
    // their registers up to the epilogue (the peeled last stages made the compiler move them
    // through scratch memory).  The last stage loads itself once more instead of a stage past
    // the end, into the buffer that nobody reads.
    for (; kt < n_k; ++kt) stage((kt - kt_begin) & 1, Yes{}, Yes{}, kt);
  }

  static_assert(2 * (BM + BN) * CPR * 16 >= (kThreads / 64) * 32 * ((GATED ? 32 : 64) + 8) * 4,
                "the turning areas of the epilogue must fit the stage buffers");
  const bool far = silu_far<GATED, 16 * MT>([&](int i) { return acc[i / 16][0][i % 16]; });
  store_tile<MT, 32, NW, (GATED ? 32 : 64), (GATED ? 32 : 64) + 8>(
      a, reinterpret_cast<float *>(lds), t0, n0, !GATED,
      [&](int i, float *turn) {
        if (GATED == SB_GATE_SILU && far) fill_from_32<MT, GATED, true>(acc, i, turn);
        else fill_from_32<MT, GATED, false>(acc, i, turn);
      });
}

// ---------------------------------------------------------------------------------------------
// The same product with the operand tiles loaded from global memory straight into LDS
// (buffer_load ... lds: the 64 lanes of a wave fill 1 KB of LDS in lane order, 16 bytes each),
// for packed weights and an inner size that is a multiple of BK.  No registers hold a stage on
// its way, so the loads run NBUF - 1 whole stages ahead of the products (the register path has
// half a stage), and the LDS stores are gone.  X keeps the row-major swizzled layout of the
// register path in LDS: a lane's place in LDS is fixed by its number, so the swizzle goes into
// the source address instead: the lane that fills chunk place c' of row r loads chunk c' ^ f(r)
// of that row.  W is copied block by block as the packed layout has it (lanes that follow one
// another read memory that follows one another; aimed at swizzled rows instead, the four lanes
// that the address unit takes at a time fell on four cache lines, and the kernel was slower than
// the register path).
//
// It multiplies with v_mfma_f32_16x16x32_bf16.  With real data the chip runs at the clock its
// power allows, and for the same count of flops this instruction lets it run faster than
// 32 x 32 x 16 (measured: 2.13 against 1.88 PFLOP/s on registers alone, 2.49 with zeros).  The
// operand traffic is the same: a wave owns (16 * MT16) x 64 outputs as MT16 x 4 tiles and reads
// MT16 + 4 fragments for every 32 k.  W's 1 KB blocks are fragments of this instruction as they
// lie (lane 16 g + r: row r, k = 8 g ..), so a B fragment is one linear read of a block, free of
// bank conflicts without a swizzle.  Fragments: B for a whole k-step in two sets of registers, A
// in a ring of four tiles that runs two tiles ahead of the MFMAs.
//
// (Two waves a SIMD are asked for also where LDS holds one block of four: with 512 registers to a wave the
// compiler kept half of the accumulators in the other register file and moved 96 of them a stage.)
//
// PERSIST: the grid is one round of blocks, and a block goes on to the tile one grid further
// until the tiles end.  The last stage of a tile then loads the first stage of the next tile (not
// itself once more), so the next tile's loop starts right after the epilogue with its operands in
// LDS, the epilogue's stores drain behind the next tile's products instead of holding the CU
// until the block has left, and no block has to be started for a tile.
template <int MT16, int NW, int BK, int NBUF, int GATED, bool PERSIST>
__global__ void __launch_bounds__(128 * NW, 2)
gemm_direct16_kernel(Args a) {
  constexpr int BM = 32 * MT16, BN = 64 * NW, kThreads = 128 * NW, kWaves = kThreads / 64;
  constexpr int CPR = BK / 8;                       // 16-byte chunks in an LDS row of A
  constexpr int kRowsPerLoad = 64 / CPR;            // rows of A that one load of a wave (1 KB) fills
  constexpr int kSteps32 = BK / 32;
  constexpr int kLoadsA = BM / kRowsPerLoad / kWaves, kLoadsB = BN / 16 * kSteps32 / kWaves;
  constexpr int kLoads = kLoadsA + kLoadsB;
  constexpr int kBufChunks = (BM + BN) * CPR;       // 16-byte chunks of a stage buffer: A, then B
  constexpr int kTiles = kSteps32 * MT16;           // A tiles of a stage, in the order they are used
  static_assert((NBUF & (NBUF - 1)) == 0 && NBUF >= 2, "the buffers are counted modulo a power of two");
  static_assert(!PERSIST || NBUF == 2, "going on to the next tile is written for two buffers");
  static_assert(BM % (kRowsPerLoad * kWaves) == 0 && (BN / 16 * kSteps32) % kWaves == 0, "whole loads");
  static_assert((NBUF - 2) * kLoads < 64, "the memory counter has six bits");
  static_assert(CPR == 8 || CPR == 4, "stages of 64 or 32 k");
  static_assert(kTiles * 2 >= kLoads, "two loads go out with each A tile");
  extern __shared__ bf16x8_t lds[];
  typedef __attribute__((address_space(3))) bf16x8_t *lds_ptr_t;

  int vblock = blockIdx.x, tm, tn;
  if (!tile_of_block(a, vblock, tm, tn)) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / NW, wn = wave % NW;

  const size_t w_rows_total = size_t(GATED ? 2 : 1) * size_t(a.w_tiles) * 16;
  const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16_t *>(a.x), 0, uint32_t(size_t(a.n_rows) * a.n_in * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16_t *>(a.w), 0, uint32_t(w_rows_total * size_t(a.w_steps) * 64), 0x00020000);
  // Byte offset of each load's source at stage 0 of tile (m, n) (the stage's offset along K is
  // added as the scalar offset).  Rows and row tiles past an operand's end are past its
  // descriptor's range and read as zeros; the host has checked that their offsets fit 32 bits.
  // W's row tiles in LDS: [0,2) gate of features n0.., [2,4) up of the same, [4,6) gate of n0 + 32..,
  // and so on: a wave's four B tiles are gate and up of 32 features.
  uint32_t off[kLoads];
  auto aim_at = [&](int m, int n) {
    const int t0 = m * BM, n0 = n * (GATED ? BN / 2 : BN);
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      if (i < kLoadsA) {
        const int place = (i * kWaves + wave) * 64 + lane;
        const int row = place / CPR;
        const int c = (place % CPR) ^ ((row / (16 / CPR)) & (CPR - 1));
        off[i] = uint32_t((size_t(t0 + row) * a.n_in + c * 8) * 2);
      } else {
        const int blk = (i - kLoadsA) * kWaves + wave, rt = blk / kSteps32, j = blk % kSteps32;
        const int tile = GATED ? ((rt & 3) >> 1) * a.w_tiles + n0 / 16 + (rt >> 2) * 2 + (rt & 1) : n0 / 16 + rt;
        off[i] = uint32_t(((size_t(tile) * a.w_steps + j) * 512 + size_t(lane) * 8) * 2);
      }
    }
  };
  auto issue_load = [&](int i, int kt, int buf) {
    const bool is_a = i < kLoadsA;
    const int stage_off = is_a ? kt * (BK * 2) : kt * (kSteps32 * 1024);
    const int chunk = buf * kBufChunks + (is_a ? (i * kWaves + wave) * 64 : BM * CPR + ((i - kLoadsA) * kWaves + wave) * 64);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(is_a ? rsrc_x : rsrc_w, (lds_ptr_t)(lds) + chunk, 16, int(off[i]),
                                             stage_off, 0, 0);
  };
  // The next stage's tiles: this wave's share has landed (the loads of the NBUF - 2 stages after
  // it may still be on their way), and after the barrier everybody's.  A bare barrier between
  // two fences for the compiler: __syncthreads() carries a release fence, which for loads into
  // LDS means waiting for all of them.
  auto wait_and_meet = [&]() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NBUF - 2) * kLoads) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  const int n_k_all = a.n_in / BK;
  const int kt_begin = a.partial ? int(blockIdx.y) * a.stages_per_slice : 0;
  const int n_k = a.partial ? min(kt_begin + a.stages_per_slice, n_k_all) : n_k_all;   // end of this slice
  // A stage past the end (of the last tile, when the block goes on) is the last stage once more,
  // into a buffer that nobody reads again: the count of loads in flight stays the same in every
  // stage, which the waits rely on.
  aim_at(tm, tn);
#pragma unroll
  for (int s = 0; s < NBUF - 1; ++s)
#pragma unroll
    for (int i = 0; i < kLoads; ++i) issue_load(i, min(kt_begin + s, n_k - 1), s);
  wait_and_meet();

  // A fragment of tile i, k-step j: lane 16 g + r reads row 16 i + r, chunk 4 j + g of the stage,
  // swizzled by the row (the term depends on r alone).  B fragment of tile f, k-step j: block
  // (4 wn + f, j), lane by lane.
  const int fr = lane & 15, fg = lane >> 4;
  const int frag_sw = (fr / (16 / CPR)) & (CPR - 1);
  int a_lane[kSteps32];
#pragma unroll
  for (int j = 0; j < kSteps32; ++j) a_lane[j] = (wm * (16 * MT16) + fr) * CPR + ((4 * j + fg) ^ frag_sw);
  const int b_lane = BM * CPR + (wn * 4 * kSteps32) * 64 + lane;

  floatx4_t acc[MT16][4];
  // One stage: buffer `buf` is multiplied, the loads of stage kt_load go out (two with each of the
  // first A tiles) into buffer buf_load, which the stage before has read.
  auto stage = [&](int buf, int kt_load, int buf_load) {
    const bf16x8_t *ls = lds + buf * kBufChunks;
    bf16x8_t fa[4], fb[2][4];
    auto read_a = [&](int tile) {       // tile = j * MT16 + i, in the order of use
      const int j = tile / MT16, i = tile % MT16;
      fa[tile & 3] = ls[a_lane[j] + i * 16 * CPR];
    };
    auto read_b = [&](int j, int f) { fb[j & 1][f] = ls[b_lane + (f * kSteps32 + j) * 64]; };
#pragma unroll
    for (int f = 0; f < 4; ++f) read_b(0, f);
    read_a(0);
    read_a(1);
#pragma unroll
    for (int tile = 0; tile < kTiles; ++tile) {
      const int j = tile / MT16, i = tile % MT16;
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        acc[i][f] = mfma16(fa[tile & 3], fb[j & 1][f], acc[i][f]);
        if (f == 0 && tile + 2 < kTiles) read_a(tile + 2);
        // the next k-step's B fragments, one with each of the first A tiles of this one
        // (two tiles a k-step: two with each)
        if (f == 1 && i < 4 && j + 1 < kSteps32) {
#pragma unroll
          for (int ff = i; ff < 4; ff += MT16) read_b(j + 1, ff);
        }
        if (f >= 2 && tile * 2 + (f - 2) < kLoads) issue_load(tile * 2 + (f - 2), kt_load, buf_load);
        // keep this order: left alone, the scheduler gathers the memory operations into lumps
        // and reads each fragment right before its MFMA, and the matrix pipe waits on both
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    wait_and_meet();
  };

  // Epilogue.  acc[i][f][e]: row 4 * (lane / 16) + e, column lane % 16 of tile (i, f); gated: tiles
  // 0, 1 are the gate and 2, 3 the up projection of the same 32 features.  PITCH = NC + 4: the
  // four row groups of a store fall on four different quarters of the banks.
  constexpr int NC = GATED ? 32 : 64, kPitch = NC + 4;
  static_assert((NBUF == 2 ? 1 : NBUF) * kBufChunks * 16 >= kWaves * 16 * kPitch * 4,
                "the turning areas must fit a stage buffer (two buffers: the other one may hold the next tile)");
  auto epilogue = [&](int m, int n, int buf_free) {
    const bool far = silu_far<GATED, 8 * MT16>([&](int i) { return acc[i / 8][i % 8 / 4][i % 4]; });
    store_tile<MT16, 16, NW, NC, kPitch>(
        a, reinterpret_cast<float *>(lds + buf_free * kBufChunks), m * BM, n * (GATED ? BN / 2 : BN), !GATED,
        [&](int i, float *turn) {
          const auto fill = [&](auto FAR) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int row = 4 * fg + e;
              if constexpr (GATED != 0) {
#pragma unroll
                for (int f = 0; f < 2; ++f)
                  turn[row * kPitch + f * 16 + fr] = tile_gate<GATED, decltype(FAR)::value>(acc[i][f][e]) * acc[i][f + 2][e];
              } else {
#pragma unroll
                for (int f = 0; f < 4; ++f) turn[row * kPitch + f * 16 + fr] = acc[i][f][e];
              }
            }
          };
          if (GATED == SB_GATE_SILU && far) fill(std::true_type{});
          else fill(std::false_type{});
        });
  };

  int buf = 0;
  for (;;) {
#pragma unroll
    for (int i = 0; i < MT16; ++i)
#pragma unroll
      for (int f = 0; f < 4; ++f) acc[i][f] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    int tm_next = 0, tn_next = 0;
    const bool more = PERSIST && tile_of_block(a, vblock + int(gridDim.x), tm_next, tn_next);
    for (int kt = kt_begin; kt < n_k; ++kt) {
      int kt_load = kt + NBUF - 1;
      if (kt_load >= n_k) {
        if (PERSIST && more) {
          // (two buffers: this is the tile's last stage) from here on the loads are the next tile's
          aim_at(tm_next, tn_next);
          kt_load = kt_begin;
        } else {
          kt_load = n_k - 1;
        }
      }
      stage(buf, kt_load, (buf + NBUF - 1) & (NBUF - 1));
      buf = (buf + 1) & (NBUF - 1);
    }
    if (NBUF > 2) {
      // the last stages' loads (of the last stage again) are still writing LDS
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    }
    // two buffers: `buf` holds the next tile's first stage (or the last stage once more), the
    // other one is free for the epilogue
    epilogue(tm, tn, NBUF == 2 ? (buf ^ 1) : 0);
    if (!PERSIST || !more) break;
    // the next stage's loads go into the buffer that the epilogue has turned its rows through
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    vblock += int(gridDim.x);
    tm = tm_next;
    tn = tn_next;
  }
}


// ---------------------------------------------------------------------------------------------
// The same, 256 x 256 tiles, in stages of 32 k, the two waves of a SIMD a turn apart: while waves 0 to 3 read their
// fragments of a stage and send out loads, waves 4 to 7 keep the matrix cores busy with theirs, and at every meeting (a bare
// barrier) they change places.  A wave comes to its products with all twelve fragments in registers.
// X is loaded in whole lines of 128 bytes (64 k of a row, in three buffers), W, which lies in blocks, 32 k at a time through
// four: all 160 KB of LDS.  The loads run two to three stages ahead; a meeting promises the stage that is read after it, for the
// waves that read it next (which waited ahead of it for their own loads) and for the others.  A buffer's last readers were
// through a turn before its next loads go out.  The epilogue turns its rows through the one buffer of X that holds nothing
// (ungated: swizzled instead of padded, it is exactly as large), with both halves of the block at it.
// What bounds it: the loads.  By themselves (no fragments read, no products) they take 0.83 of the kernel's time at 16,384 x
// 3,584 x 18,944 and 0.71 at 16,384 x 37,888 x 3,584, products by themselves 0.67 and 0.70.  Half lines of X (64 bytes a row
// and stage) made that 1.0 and 0.9: L2 answers as many requests a second of either size.  Measured against the kernel that had
// one barrier a stage, both waves of a SIMD reading and multiplying at once, and half lines: 2,048 x 37,888 x 3,584 443 -> 415 us,
// 16,384 rows 3.31 -> 3.13 ms (1.42 PFLOP/s), 16,384 x 3,584 x 18,944 1.89 -> 1.72, 6,398 x 22,016 x 2,048 475 -> 454 us; of that
// the turns give 3 to 4 %.  Not kept: turns of 64 k (a wave's fragments then wait for W's loads, one stage ahead: 0.87 of
// the speed), whole lines with one barrier a stage and no turns (3 to 4 % slower), loads between the products (2 to 5 %),
// half of X's fragments read beside the products (6 to 10 %), s_setprio around the products (1 %).
template <int GATED, bool PERSIST, bool XIELU = false>
__global__ void __launch_bounds__(512)
gemm_pipe_kernel(Args a) {
  constexpr int MT16 = 8, NW = 4, BM = 256, BN = 256, kWaves = 8;
  constexpr int kRingA = 3, kRingW = 4;              // buffers of X (64 k each) and of W (32 k)
  constexpr int kBufA = BM * 8, kBufW = BN * 4;      // 16-byte chunks of a buffer
  constexpr int kFlight = 8;                         // loads that a wave has in flight across a meeting: two stages'
  extern __shared__ bf16x8_t lds[];
  typedef __attribute__((address_space(3))) bf16x8_t *lds_ptr_t;

  int vblock = blockIdx.x, tm, tn;
  if (!tile_of_block(a, vblock, tm, tn)) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / NW, wn = wave % NW;

  const size_t w_rows_total = size_t(GATED ? 2 : 1) * size_t(a.w_tiles) * 16;
  const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16_t *>(a.x), 0, uint32_t(size_t(a.n_rows) * a.n_in * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16_t *>(a.w), 0, uint32_t(w_rows_total * size_t(a.w_steps) * 64), 0x00020000);
  // sources of a wave's loads at k 0 of tile (m, n), as in the kernel above: four of X for 64 k, two of W for 32 k
  uint32_t off_a[4], off_w[2];
  auto aim_a = [&](int m) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int place = (i * kWaves + wave) * 64 + lane;
      const int row = place / 8, c = (place % 8) ^ ((row / 2) & 7);
      off_a[i] = uint32_t((size_t(m * BM + row) * a.n_in + c * 8) * 2);
    }
  };
  auto aim_w = [&](int n) {
    const int n0 = n * (GATED ? BN / 2 : BN);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int rt = i * kWaves + wave;
      const int tile = GATED ? ((rt & 3) >> 1) * a.w_tiles + n0 / 16 + (rt >> 2) * 2 + (rt & 1) : n0 / 16 + rt;
      off_w[i] = uint32_t((size_t(tile) * a.w_steps * 512 + size_t(lane) * 8) * 2);
    }
  };
  auto load_a = [&](int i, int k64, int buf) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_x, (lds_ptr_t)(lds) + buf * kBufA + (i * kWaves + wave) * 64, 16, int(off_a[i]),
                                             k64 * 128, 0, 0);
  };
  auto load_w = [&](int kt, int buf) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_w, (lds_ptr_t)(lds) + kRingA * kBufA + buf * kBufW + (i * kWaves + wave) * 64, 16,
                                               int(off_w[i]), kt * 1024, 0, 0);
  };
  auto meet = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto landed = [&]() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kFlight) : "memory"); };

  // stages of 32 k, an even count (the host: an inner size in 64s, slices of whole 64s)
  const int n_k_all = a.n_in / 32;
  const int kt_begin = a.partial ? int(blockIdx.y) * a.stages_per_slice * 2 : 0;
  const int n_k = a.partial ? min(kt_begin + a.stages_per_slice * 2, n_k_all) : n_k_all;
  // A stage past the end (of the last tile, when the block goes on) is the last stage once more, into a
  // buffer that nobody reads again, so that the count of loads in flight stays the same.
  aim_a(tm);
  aim_w(tn);
#pragma unroll
  for (int i = 0; i < 4; ++i) load_a(i, kt_begin / 2, 0);
  load_w(kt_begin, 0);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    load_a(2 * h, min(kt_begin / 2 + 1, n_k / 2 - 1), 1);
    load_a(2 * h + 1, min(kt_begin / 2 + 1, n_k / 2 - 1), 1);
    load_w(min(kt_begin + 1 + h, n_k - 1), 1 + h);
  }
  landed();
  meet();

  const int fr = lane & 15, fg = lane >> 4;
  int a_lane[2];                  // the fragment's place in each half of a buffer of X
#pragma unroll
  for (int j = 0; j < 2; ++j) a_lane[j] = (wm * (16 * MT16) + fr) * 8 + ((4 * j + fg) ^ ((fr / 2) & 7));
  const int b_lane = kRingA * kBufA + wn * 4 * 64 + lane;

  floatx4_t acc[MT16][4];
  int tm_next = 0, tn_next = 0;
  bool more = false;
  int buf_a = 0, buf_w = 0;
  // One stage, half HALF of 64 k: a wave's turn at the memories (its fragments, and its share of the loads two to three stages
  // further on, into buffers whose last reader was through a turn ago), then its turn at the matrix cores.
  auto stage = [&](auto HALF, int kt) {
    constexpr int half = decltype(HALF)::value;
    bf16x8_t fa[MT16], fb[4];
    const bf16x8_t *ls_a = lds + buf_a * kBufA + a_lane[half], *ls_w = lds + (buf_w + half) * kBufW + b_lane;
#pragma unroll
    for (int f = 0; f < 4; ++f) fb[f] = ls_w[f * 64];
#pragma unroll
    for (int i = 0; i < MT16; ++i) fa[i] = ls_a[i * 128];
    int k64 = kt / 2 + 2, kw = kt + 3;
    if (half == 0 ? kt + 4 >= n_k : kt + 3 >= n_k) {            // past the tile's end
      if (!PERSIST || !more) {
        k64 = n_k / 2 - 1;
        kw = min(kw, n_k - 1);
      } else {
        k64 = k64 - n_k / 2 + kt_begin / 2;
        if (half == 0) {
          if (kt + 4 == n_k) aim_a(tm_next);                    // from here on X's loads are the next tile's,
          if (kw >= n_k) kw = kw - n_k + kt_begin;
        } else {
          if (kt + 3 == n_k) aim_w(tn_next);                    // and from here on W's
          kw = kw - n_k + kt_begin;
        }
      }
    }
    const int to_a = buf_a == 0 ? 2 : buf_a - 1;
    load_a(2 * half, k64, to_a);
    load_a(2 * half + 1, k64, to_a);
    load_w(kw, (buf_w + half + 3) & (kRingW - 1));
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (wm) landed();
    meet();
#pragma unroll
    for (int i = 0; i < MT16; ++i)
#pragma unroll
      for (int f = 0; f < 4; ++f) acc[i][f] = mfma16(fa[i], fb[f], acc[i][f]);
    __builtin_amdgcn_sched_barrier(0);
    if (!wm) landed();
    meet();
  };

  constexpr int NC = GATED ? 32 : 64, kPitch = GATED ? NC + 4 : NC;
  static_assert(kBufA * 16 >= kWaves * 16 * kPitch * 4, "the turning areas must fit a buffer of X");
  auto epilogue = [&](int m, int n, int a_free) {
    const bool far = silu_far<GATED, 8 * MT16>([&](int i) { return acc[i / 8][i % 8 / 4][i % 4]; });
    float rise = 0.0f, bend = 0.0f;
    if constexpr (XIELU) xielu_numbers(a.act_params, a.act_dtype, rise, bend);
    store_tile<MT16, 16, NW, NC, kPitch, !GATED>(
        a, reinterpret_cast<float *>(lds + a_free * kBufA), m * BM, n * (GATED ? BN / 2 : BN), !GATED,
        [&](int i, float *turn) {
          const auto fill = [&](auto FAR) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int row = 4 * fg + e;
              if constexpr (GATED != 0) {
#pragma unroll
                for (int f = 0; f < 2; ++f)
                  turn[row * kPitch + f * 16 + fr] = tile_gate<GATED, decltype(FAR)::value>(acc[i][f][e]) * acc[i][f + 2][e];
              } else {
#pragma unroll
                for (int f = 0; f < 4; ++f) turn[row * kPitch + (f ^ fg) * 16 + fr] = XIELU ? xielu(acc[i][f][e], rise, bend) : acc[i][f][e];
              }
            }
          };
          if (GATED == SB_GATE_SILU && far) fill(std::true_type{});
          else fill(std::false_type{});
        });
  };

  for (;;) {
#pragma unroll
    for (int i = 0; i < MT16; ++i)
#pragma unroll
      for (int f = 0; f < 4; ++f) acc[i][f] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    more = PERSIST && tile_of_block(a, vblock + int(gridDim.x), tm_next, tn_next);
    if (wm) meet();               // the second four waves are a turn behind the first
    for (int kt = kt_begin; kt < n_k; kt += 2) {
      stage(std::integral_constant<int, 0>{}, kt);
      stage(std::integral_constant<int, 1>{}, kt + 1);
      buf_a = buf_a == kRingA - 1 ? 0 : buf_a + 1;
      buf_w ^= 2;
    }
    if (!wm) meet();
    if (!PERSIST || !more) {
      // the last loads (of the last stage again) are still writing LDS
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
    epilogue(tm, tn, buf_a == 0 ? 2 : buf_a - 1);       // the other buffers hold the next tile's first stages
    if (!PERSIST || !more) break;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    vblock += int(gridDim.x);
    tm = tm_next;
    tn = tn_next;
  }
}

// ---------------------------------------------------------------------------------------------
// The same in tiles of 256 x 128, a wave 64 x 64 of it, in stages of 64 k through three buffers of each side (144 KB), for
// products whose 256 x 256 tiles would leave half the CUs idle.  A wave's turn at the matrix cores is 512 cycles, as above, its
// turn at LDS sixteen fragments; the loads of a stage go out two stages ahead.  What bounds it: the loads, one and a half
// times the tile above's for a product.  Measured against four waves of 128 x 64, one a SIMD, whose tiles went through registers:
// 2,048 x 3,584 x 3,584 69 -> 57 us, 4,001 x 2,048 x 4,096 82 -> 70, 4,001 x 2,048 x 8,192 141 -> 123, 3,000 x 2,560 x 2,048 40 -> 35.
template <int GATED, bool PERSIST>
__global__ void __launch_bounds__(512)
gemm_pipe_half_kernel(Args a) {
  constexpr int MT16 = 4, NW = 2, BM = 256, BN = 128, kWaves = 8;
  constexpr int kRing = 3;                           // buffers of X and of W, 64 k each
  constexpr int kBufA = BM * 8, kBufW = BN * 8;      // 16-byte chunks of a buffer
  constexpr int kFlight = 6;                         // loads that a wave has in flight across a meeting: a stage's
  extern __shared__ bf16x8_t lds[];
  typedef __attribute__((address_space(3))) bf16x8_t *lds_ptr_t;

  int vblock = blockIdx.x, tm, tn;
  if (!tile_of_block(a, vblock, tm, tn)) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / NW, wn = wave % NW;
  const bool late = wave >= 4;                       // a turn behind the first four

  const size_t w_rows_total = size_t(GATED ? 2 : 1) * size_t(a.w_tiles) * 16;
  const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16_t *>(a.x), 0, uint32_t(size_t(a.n_rows) * a.n_in * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16_t *>(a.w), 0, uint32_t(w_rows_total * size_t(a.w_steps) * 64), 0x00020000);
  // sources of a wave's loads at k 0 of tile (m, n), as in the kernel above: four of X, two of W
  uint32_t off_a[4], off_w[2];
  auto aim_a = [&](int m) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int place = (i * kWaves + wave) * 64 + lane;
      const int row = place / 8, c = (place % 8) ^ ((row / 2) & 7);
      off_a[i] = uint32_t((size_t(m * BM + row) * a.n_in + c * 8) * 2);
    }
  };
  auto aim_w = [&](int n) {
    const int n0 = n * (GATED ? BN / 2 : BN);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int blk = i * kWaves + wave, rt = blk / 2;
      const int tile = GATED ? ((rt & 3) >> 1) * a.w_tiles + n0 / 16 + (rt >> 2) * 2 + (rt & 1) : n0 / 16 + rt;
      off_w[i] = uint32_t(((size_t(tile) * a.w_steps + blk % 2) * 512 + size_t(lane) * 8) * 2);
    }
  };
  auto load = [&](int kt, int buf) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_x, (lds_ptr_t)(lds) + buf * kBufA + (i * kWaves + wave) * 64, 16, int(off_a[i]),
                                               kt * 128, 0, 0);
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_w, (lds_ptr_t)(lds) + kRing * kBufA + buf * kBufW + (i * kWaves + wave) * 64, 16,
                                               int(off_w[i]), kt * 2048, 0, 0);
  };
  auto meet = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto landed = [&]() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kFlight) : "memory"); };

  // stages of 64 k
  const int n_k_all = a.n_in / 64;
  const int kt_begin = a.partial ? int(blockIdx.y) * a.stages_per_slice : 0;
  const int n_k = a.partial ? min(kt_begin + a.stages_per_slice, n_k_all) : n_k_all;
  // A stage past the end (of the last tile, when the block goes on) is the last stage once more, into a
  // buffer that nobody reads again, so that the count of loads in flight stays the same.
  aim_a(tm);
  aim_w(tn);
  load(kt_begin, 0);
  load(min(kt_begin + 1, n_k - 1), 1);
  landed();
  meet();

  const int fr = lane & 15, fg = lane >> 4;
  int a_lane[2];                  // the fragment's place in each half of a buffer of X
#pragma unroll
  for (int j = 0; j < 2; ++j) a_lane[j] = (wm * (16 * MT16) + fr) * 8 + ((4 * j + fg) ^ ((fr / 2) & 7));
  const int b_lane = kRing * kBufA + wn * 8 * 64 + lane;

  floatx4_t acc[MT16][4];
  int tm_next = 0, tn_next = 0;
  bool more = false;
  int buf = 0;
  // One stage: a wave's turn at the memories (its fragments, and its share of the loads two stages further on, into the
  // buffers whose last reader was through a turn ago), then its turn at the matrix cores.
  auto stage = [&](int kt) {
    bf16x8_t fa[2][MT16], fb[2][4];
    const bf16x8_t *ls_a = lds + buf * kBufA, *ls_w = lds + buf * kBufW + b_lane;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int f = 0; f < 4; ++f) fb[j][f] = ls_w[(f * 2 + j) * 64];
#pragma unroll
      for (int i = 0; i < MT16; ++i) fa[j][i] = ls_a[a_lane[j] + i * 128];
    }
    int to = kt + 2;
    if (to >= n_k) {                                            // past the tile's end
      if (!PERSIST || !more) {
        to = n_k - 1;
      } else {
        if (to == n_k) {                                        // from here on the loads are the next tile's
          aim_a(tm_next);
          aim_w(tn_next);
        }
        to = to - n_k + kt_begin;
      }
    }
    load(to, buf == 0 ? kRing - 1 : buf - 1);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (late) landed();
    meet();
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < MT16; ++i)
#pragma unroll
        for (int f = 0; f < 4; ++f) acc[i][f] = mfma16(fa[j][i], fb[j][f], acc[i][f]);
    __builtin_amdgcn_sched_barrier(0);
    if (!late) landed();
    meet();
  };

  constexpr int NC = GATED ? 32 : 64, kPitch = GATED ? NC + 4 : NC;
  static_assert(kBufA * 16 >= kWaves * 16 * kPitch * 4, "the turning areas must fit a buffer of X");
  auto epilogue = [&](int m, int n, int a_free) {
    const bool far = silu_far<GATED, 8 * MT16>([&](int i) { return acc[i / 8][i % 8 / 4][i % 4]; });
    store_tile<MT16, 16, NW, NC, kPitch, !GATED>(
        a, reinterpret_cast<float *>(lds + a_free * kBufA), m * BM, n * (GATED ? BN / 2 : BN), !GATED,
        [&](int i, float *turn) {
          const auto fill = [&](auto FAR) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int row = 4 * fg + e;
              if constexpr (GATED != 0) {
#pragma unroll
                for (int f = 0; f < 2; ++f)
                  turn[row * kPitch + f * 16 + fr] = tile_gate<GATED, decltype(FAR)::value>(acc[i][f][e]) * acc[i][f + 2][e];
              } else {
#pragma unroll
                for (int f = 0; f < 4; ++f) turn[row * kPitch + (f ^ fg) * 16 + fr] = acc[i][f][e];
              }
            }
          };
          if (GATED == SB_GATE_SILU && far) fill(std::true_type{});
          else fill(std::false_type{});
        });
  };

  for (;;) {
#pragma unroll
    for (int i = 0; i < MT16; ++i)
#pragma unroll
      for (int f = 0; f < 4; ++f) acc[i][f] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    more = PERSIST && tile_of_block(a, vblock + int(gridDim.x), tm_next, tn_next);
    if (late) meet();
    for (int kt = kt_begin; kt < n_k; ++kt) {
      stage(kt);
      buf = buf == kRing - 1 ? 0 : buf + 1;
    }
    if (!late) meet();
    if (!PERSIST || !more) {
      // the last loads (of the last stage again) are still writing LDS
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
    epilogue(tm, tn, buf == 0 ? kRing - 1 : buf - 1);       // the other buffers hold the next tile's first stages
    if (!PERSIST || !more) break;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    vblock += int(gridDim.x);
    tm = tm_next;
    tn = tn_next;
  }
}

// ---------------------------------------------------------------------------------------------
// The gated product whose tiles of 96, 128 or 192 rows make one round over the CUs: some hundred rows of wide matrices, whose weights
// are most of what there is to read, up to some thousand of narrow ones.  What bounds it in the forms above is how much of W a CU has on its way (three stages in LDS, beside X's): memory answers in some 2 us, and 48 KB in that time are
// 24 GB/s a CU.  Here W never passes through LDS: a wave owns 16 columns of either half, whose packed blocks are the matrix
// instruction's fragments as they lie, and keeps kDeep stages of 64 k of them in registers on their way.  Rows of X, which the block's four such
// waves share, are brought into LDS by two waves that do nothing else: loads return in order, so that waiting for a stage of X
// would also wait for the weights that were asked for before it.  One barrier a stage.
// us, the form taken before and this one (rows x 2 halves of W x k): 183 x 17,920 x 1,536 26.0 and 22.4 (a read of W alone 11),
// 96 rows 20.4 and 17.7, 192 x 22,016 x 2,048 32.7 and 28.4, 260 x 11,008 x 2,048 31.4 and 23.0, 288 x 9,728 x 896 12.6 and 9.2; prompts
// of 288 rows of the 0.5B sizes 1,519 -> 1,454, 183 rows of the 1.5B ones 2,614 -> 2,514; narrow matrices (2 x 512 x 2,048) 1,040 rows
// 19.2 and 14.1, 2,048 20.9 and 18.3, 3,072 35.6 and 24.5, (2 x 128 x 512) 8,208 10.4 and 7.4, 288 rows x 11,008 x 512 11.6 and 10.7.  Tiles of 96 and 192 rows straight into LDS as
// above were ahead by themselves (10.7 and 25.5) and not in whole steps.
// RT: tiles of 16 rows of a block.  The weights are the first operand, so that a lane ends up with four neighbouring
// columns of a row.
template <int RT, int GATED>
__global__ void __launch_bounds__(384)
gemm_ahead_kernel(Args a) {
  constexpr int kRows = 16 * RT, kBuf = kRows * 8, NB = 4, kDeep = 6;
  static_assert(GATED != 0 && (NB - 2) * RT < 64, "the memory counter has six bits");
  extern __shared__ bf16x8_t lds[];                    // [NB][row][8 chunks of 16 bytes, turned by the row]
  typedef __attribute__((address_space(3))) bf16x8_t *lds_ptr_t;
  int tm, tn;
  if (!tile_of_block(a, int(blockIdx.x), tm, tn)) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n_k = a.n_in / 64, t0 = tm * kRows;
  if (wave >= 4) {
    const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16_t *>(a.x), 0, uint32_t(size_t(a.n_rows) * a.n_in * 2), 0x00020000);
    uint32_t off[RT];                                  // rows past the last lie past the descriptor's end: zeros
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const int place = (2 * i + wave - 4) * 64 + lane, row = place / 8, c = (place % 8) ^ ((row / 2) & 7);
      off[i] = uint32_t((size_t(t0 + row) * a.n_in + c * 8) * 2);
    }
    const auto bring = [&](int kt) {                   // (past the end: the last stage again, into a buffer that nobody reads)
      const int from = min(kt, n_k - 1) * 128;
#pragma unroll
      for (int i = 0; i < RT; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_x, (lds_ptr_t)(lds) + (kt % NB) * kBuf + (2 * i + wave - 4) * 64, 16, int(off[i]),
                                                 from, 0, 0);
    };
#pragma unroll
    for (int s = 0; s < NB - 1; ++s) bring(s);
    for (int kt = 0; kt < n_k; ++kt) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NB - 2) * RT) : "memory");
      __builtin_amdgcn_s_barrier();                    // stage kt is there, and stage kt - 1 has been read
      asm volatile("" ::: "memory");
      bring(kt + NB - 1);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    return;
  }
  const int n_first = tn * 64 + 16 * wave;             // this wave's columns
  const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16_t *>(a.w), 0, uint32_t(size_t(2) * a.w_tiles * 16 * size_t(a.w_steps) * 64), 0x00020000);
  uint32_t w_off[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) w_off[h] = uint32_t((size_t(h * a.w_tiles + n_first / 16) * a.w_steps * 512 + size_t(lane) * 8) * 2);
  bf16x8_t w[kDeep][2][2];                             // [stage][32 k][half]
  const auto ask = [&](int slot, int kt) __attribute__((always_inline)) {
    const int from = min(kt, n_k - 1) * 2048;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        w[slot][j][h] = __builtin_bit_cast(bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc_w, int(w_off[h]), from + 1024 * j, 0));
  };
  floatx4_t acc[RT][2];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int h = 0; h < 2; ++h) acc[i][h] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < kDeep; ++s) {
    ask(s, s);
    __builtin_amdgcn_sched_barrier(0);
  }
  const int fr = lane & 15, fg = lane >> 4;
  const int x_lane[2] = {fr * 8 + (fg ^ (fr / 2)), fr * 8 + ((4 + fg) ^ (fr / 2))};
  const auto stage = [&](int u, int kt) __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const bf16x8_t *ls = lds + (kt % NB) * kBuf;
    bf16x8_t x[4];                                     // three tiles on their way out of LDS
#pragma unroll
    for (int i = 0; i < 3; ++i) x[i] = ls[x_lane[0] + i * 128];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 2 * RT; ++i) {
      if (i + 3 < 2 * RT) x[(i + 3) & 3] = ls[x_lane[(i + 3) / RT] + (i + 3) % RT * 128];
#pragma unroll
      for (int h = 0; h < 2; ++h) acc[i % RT][h] = mfma16(w[u][i / RT][h], x[i & 3], acc[i % RT][h]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int kt = 0;
  for (; kt + kDeep <= n_k; kt += kDeep) {
#pragma unroll
    for (int u = 0; u < kDeep; ++u) {
      stage(u, kt + u);
      ask(u, kt + kDeep + u);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int u = 0; u < kDeep; ++u)
    if (kt + u < n_k) stage(u, kt + u);
  // acc[i][h][e]: column n_first + 4 fg + e of row 16 i + fr
  const bool far = silu_far<GATED, 4 * RT>([&](int i) { return acc[i / 4][0][i % 4]; });
  const int n = n_first + 4 * fg;
  const auto store = [&](auto FAR) {
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const int t = t0 + 16 * i + fr;
      if (t >= a.n_rows || n >= a.n_out) continue;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = tile_gate<GATED, decltype(FAR)::value>(acc[i][0][e]) * acc[i][1][e];
      const size_t at = size_t(t) * a.n_out + n;
      if (a.y_dtype == SB_F32) *reinterpret_cast<floatx4_t *>((float *)a.y + at) = floatx4_t{v[0], v[1], v[2], v[3]};
      else *reinterpret_cast<uint2 *>((bf16_t *)a.y + at) = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
    }
  };
  if (GATED == SB_GATE_SILU && far) store(std::true_type{});
  else store(std::false_type{});
}

template <int RT, int GATED>
int launch_ahead_one(const Args &a, long long blocks, hipStream_t s) {
  constexpr int lds_bytes = 4 * 16 * RT * 128;
  static bool raised = false;     // per instantiation; harmless if repeated
  if (lds_bytes > 48 * 1024 && !raised) {
    const hipError_t e = hipFuncSetAttribute((const void *)gemm_ahead_kernel<RT, GATED>, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    SB_REQUIRE(e == hipSuccess, "sb_gemm_mfma_bf16: cannot reserve %d bytes of LDS: %s", lds_bytes, hipGetErrorString(e));
    raised = true;
  }
  gemm_ahead_kernel<RT, GATED><<<unsigned((blocks + kXcds - 1) / kXcds * kXcds), 384, lds_bytes, s>>>(a);
  return SB_OK;
}
template <int RT>
int launch_ahead(const Args &a, long long blocks, hipStream_t s) {
  switch (a.gated) {
    case 3: return launch_ahead_one<RT, 3>(a, blocks, s);
    case 2: return launch_ahead_one<RT, 2>(a, blocks, s);
    default: return launch_ahead_one<RT, 1>(a, blocks, s);
  }
}

template <int MT, int NW, int BK, int DEPTH, int GATED, bool PACKED, bool EVEN_K>
int launch_one(const Args &a, long long blocks, hipStream_t s) {
  constexpr int lds_bytes = 2 * (64 * MT + 64 * NW) * (BK / 8) * 16;
  static bool raised = false;     // per instantiation; harmless if repeated
  if (lds_bytes > 48 * 1024 && !raised) {
    const hipError_t e =
        hipFuncSetAttribute((const void *)gemm_mfma_kernel<MT, NW, BK, DEPTH, GATED, PACKED, EVEN_K>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    SB_REQUIRE(e == hipSuccess, "sb_gemm_mfma_bf16: cannot reserve %d bytes of LDS: %s", lds_bytes,
               hipGetErrorString(e));
    raised = true;
  }
  const int n_k = (a.n_in + BK - 1) / BK;
  const unsigned slices = a.partial ? unsigned((n_k + a.stages_per_slice - 1) / a.stages_per_slice) : 1u;
  gemm_mfma_kernel<MT, NW, BK, DEPTH, GATED, PACKED, EVEN_K>
      <<<dim3(unsigned((blocks + kXcds - 1) / kXcds * kXcds), slices), 128 * NW, lds_bytes, s>>>(a);
  return SB_OK;
}

template <int MT, int NW, int BK, int DEPTH, bool PLAIN_TOO>
int launch(const Args &a, long long blocks, int packed, hipStream_t s) {
  // the gate's activation is a template argument: the SiLU kernels hold no code of the others
  const int which = a.gated * 4 + (packed ? 2 : 0) + (a.n_in % BK == 0 ? 1 : 0);
  switch (which) {
    case 15: return launch_one<MT, NW, BK, DEPTH, 3, true, true>(a, blocks, s);
    case 14: return launch_one<MT, NW, BK, DEPTH, 3, true, false>(a, blocks, s);
    case 11: return launch_one<MT, NW, BK, DEPTH, 2, true, true>(a, blocks, s);
    case 10: return launch_one<MT, NW, BK, DEPTH, 2, true, false>(a, blocks, s);
    case 7: return launch_one<MT, NW, BK, DEPTH, 1, true, true>(a, blocks, s);
    case 6: return launch_one<MT, NW, BK, DEPTH, 1, true, false>(a, blocks, s);
    case 3: return launch_one<MT, NW, BK, DEPTH, 0, true, true>(a, blocks, s);
    case 2: return launch_one<MT, NW, BK, DEPTH, 0, true, false>(a, blocks, s);
    default: break;
  }
  if constexpr (PLAIN_TOO) {
    switch (which) {
      case 13: return launch_one<MT, NW, BK, DEPTH, 3, false, true>(a, blocks, s);
      case 12: return launch_one<MT, NW, BK, DEPTH, 3, false, false>(a, blocks, s);
      case 9: return launch_one<MT, NW, BK, DEPTH, 2, false, true>(a, blocks, s);
      case 8: return launch_one<MT, NW, BK, DEPTH, 2, false, false>(a, blocks, s);
      case 5: return launch_one<MT, NW, BK, DEPTH, 1, false, true>(a, blocks, s);
      case 4: return launch_one<MT, NW, BK, DEPTH, 1, false, false>(a, blocks, s);
      case 1: return launch_one<MT, NW, BK, DEPTH, 0, false, true>(a, blocks, s);
      default: return launch_one<MT, NW, BK, DEPTH, 0, false, false>(a, blocks, s);
    }
  }
  return sb::fail(SB_ERR_UNSUPPORTED, "sb_gemm_mfma_bf16: this tile shape takes packed weights only");
}

// PERSIST: one round of blocks (`round_blocks`: what the GPU runs at a time), each going from
// tile to tile
template <int MT16, int NW, int BK, int NBUF, int GATED, bool PERSIST>
int launch_direct_one(const Args &a, long long blocks, int round_blocks, hipStream_t s) {
  constexpr int lds_bytes = NBUF * (32 * MT16 + 64 * NW) * (BK / 8) * 16;
  static bool raised = false;     // per instantiation; harmless if repeated
  if (lds_bytes > 48 * 1024 && !raised) {
    const hipError_t e = hipFuncSetAttribute((const void *)gemm_direct16_kernel<MT16, NW, BK, NBUF, GATED, PERSIST>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    SB_REQUIRE(e == hipSuccess, "sb_gemm_mfma_bf16: cannot reserve %d bytes of LDS: %s", lds_bytes,
               hipGetErrorString(e));
    raised = true;
  }
  const int n_k = a.n_in / BK;
  const unsigned slices = a.partial ? unsigned((n_k + a.stages_per_slice - 1) / a.stages_per_slice) : 1u;
  long long grid = (blocks + kXcds - 1) / kXcds * kXcds;
  if (PERSIST && grid > round_blocks) grid = round_blocks;
  gemm_direct16_kernel<MT16, NW, BK, NBUF, GATED, PERSIST><<<dim3(unsigned(grid), slices), 128 * NW, lds_bytes, s>>>(a);
  return SB_OK;
}

// packed weights, n_in a multiple of BK
template <int MT16, int NW, int BK, int NBUF, bool PERSIST>
int launch_direct(const Args &a, long long blocks, int round_blocks, hipStream_t s) {
  switch (a.gated) {
    case 3: return launch_direct_one<MT16, NW, BK, NBUF, 3, PERSIST>(a, blocks, round_blocks, s);
    case 2: return launch_direct_one<MT16, NW, BK, NBUF, 2, PERSIST>(a, blocks, round_blocks, s);
    case 1: return launch_direct_one<MT16, NW, BK, NBUF, 1, PERSIST>(a, blocks, round_blocks, s);
    default: return launch_direct_one<MT16, NW, BK, NBUF, 0, PERSIST>(a, blocks, round_blocks, s);
  }
}

template <int GATED, bool PERSIST, bool HALF, bool XIELU = false>
int launch_pipe_one(const Args &a, long long blocks, hipStream_t s) {
  // (256 x 256: all that a CU has)
  constexpr int lds_bytes = HALF ? 3 * (256 + 128) * 128 : 3 * 256 * 128 + 4 * 256 * 64;
  auto kern = gemm_pipe_kernel<GATED, PERSIST, XIELU>;
  if constexpr (HALF) kern = gemm_pipe_half_kernel<GATED, PERSIST>;
  static bool raised = false;     // per instantiation; harmless if repeated
  if (!raised) {
    const hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    SB_REQUIRE(e == hipSuccess, "sb_gemm_mfma_bf16: cannot reserve %d bytes of LDS: %s", lds_bytes, hipGetErrorString(e));
    raised = true;
  }
  const int n_k = a.n_in / 64;
  const unsigned slices = a.partial ? unsigned((n_k + a.stages_per_slice - 1) / a.stages_per_slice) : 1u;
  long long grid = (blocks + kXcds - 1) / kXcds * kXcds;
  if (PERSIST && grid > sb::cu_count()) grid = sb::cu_count();        // a block a CU
  kern<<<dim3(unsigned(grid), slices), 512, lds_bytes, s>>>(a);
  return SB_OK;
}

template <bool HALF>
int launch_pipe(const Args &a, long long blocks, bool a_block_a_tile, hipStream_t s) {
  // (going on to the next tile, whose first stages are loaded in the last 128 k of this one, takes 128 k)
  if (!HALF && a.act_params) return launch_pipe_one<0, true, false, true>(a, blocks, s);      // (128 k and more)
  if (a_block_a_tile || a.n_in < 128) {
    switch (a.gated) {
      case 3: return launch_pipe_one<3, false, HALF>(a, blocks, s);
      case 2: return launch_pipe_one<2, false, HALF>(a, blocks, s);
      case 1: return launch_pipe_one<1, false, HALF>(a, blocks, s);
      default: return launch_pipe_one<0, false, HALF>(a, blocks, s);
    }
  }
  switch (a.gated) {
    case 3: return launch_pipe_one<3, true, HALF>(a, blocks, s);
    case 2: return launch_pipe_one<2, true, HALF>(a, blocks, s);
    case 1: return launch_pipe_one<1, true, HALF>(a, blocks, s);
    default: return launch_pipe_one<0, true, HALF>(a, blocks, s);
  }
}

// Tile shapes the launcher chooses from: rows x columns of Y per block.
struct Shape { int bm, bn; };
constexpr Shape kShapes[9] = {{128, 128}, {256, 128}, {256, 256}, {128, 256}, {192, 256}, {64, 128},
                              {96, 128}, {128, 128}, {192, 128}};      // (the last three: gated, weights through registers)

// The tile shape for a problem: the one with the best product of three factors.  How fast the
// shape's kernel runs on a full grid, relative to 128 x 128 (measured on MI355X at 2,048 to 16,384
// rows of Qwen2.5-7B's four products: the 256 x 256 kernel reaches 1.34 to 1.48 PFLOP/s on a full
// grid where the 128 x 128 one reaches 0.73 to 0.98; tiles of 192 rows loaded straight into LDS 1.04 to 1.12, of 256 x 128 0.92 to 1.2); the share of the tiles' rows
// that are rows of Y; and the share of the last round of tiles over the CUs that is filled.
// Some of what this decides at 2,048 rows: the output product (3,584 x 3,584) takes 256 x 128
// (224 tiles, one round: 57 us against 92 with 112 tiles of 256 x 256), the QKV product 192 x 256
// (198 tiles: 63 us against 73 with 144 of 256 x 256, 93 with 288 of 256 x 128);
// from 4,096 rows on nearly everything takes 256 x 256.  `direct_ok`: the kernel that loads
// straight into LDS takes these operands (the 192 x 256 shape has no other).
int pick_shape(int n_rows, int n_out, int n_in, int gated, bool direct_ok, double *score_out = nullptr) {
  (void)n_in;
  // (256 x 128, gated: faster by itself, but no faster beside tiles of 128 x 128, several of which share a CU: 900 rows
  // against 22,016 x 2,048 89 us and 79)
  const double speed[5] = {1.0, gated ? 1.0 : direct_ok ? 1.24 : 1.05, 1.45, 0.0, gated ? 1.11 : 1.2};
  double best = 0;
  int pick = 0;
  for (int v = 0; v < 5; ++v) {
    if (v == 3 || (v == 4 && !direct_ok)) continue;
    const int bm = kShapes[v].bm, bn = gated ? kShapes[v].bn / 2 : kShapes[v].bn;
    const long long tiles_m = (n_rows + bm - 1) / bm, tiles_n = (n_out + bn - 1) / bn;
    const long long tiles = tiles_m * tiles_n, rounds = (tiles + sb::cu_count() - 1) / sb::cu_count();
    const double score = speed[v] * (double(n_rows) / double(tiles_m * bm)) * (double(tiles) / double(rounds * sb::cu_count()));
    if (score > best) { best = score; pick = v; }
  }
  if (score_out) *score_out = best;
  return pick;
}

}  // namespace

// Y = X W^T (+bias) (+resid), or gated: Y = silu(X Wg^T) * (X Wu^T), W = [Wg; Wu].
// X [n_rows, n_in] and W bf16, n_in a multiple of 8, operands 16-byte aligned; packed != 0: W is
// in the packed tile layout.
extern "C" int sb_gemm_mfma_scaled_bf16(void *y, int y_dtype, const void *x, const void *w, const void *bias,
                                        int bias_dtype, const float *resid, float resid_scale, int n_rows, int n_out,
                                        int n_in, int gated, int packed, int tile_shape, void *stream);

namespace {
int gemm_whole(void *y, int y_dtype, const void *x, const void *w, const void *bias, int bias_dtype, const float *resid, float resid_scale,
               int n_rows, int n_out, int n_in, int gated, int relu_sq, int packed, int tile_shape, void *stream,
               const void *act_params = nullptr, int act_dtype = 0);
}

// The product with an activation of an ungated feed-forward on its way out: SB_ACT_RELU_SQ, max(z, 0)^2 of z = X W^T + bias.
extern "C" int sb_gemm_mfma_act_bf16(void *y, int y_dtype, const void *x, const void *w, const void *bias, int bias_dtype, int n_rows,
                                     int n_out, int n_in, int act, int packed, int tile_shape, void *stream) {
  SB_SUPPORT(act == SB_ACT_RELU_SQ, "sb_gemm_mfma_act_bf16: activation %d is not the square of max(z, 0)", act);
  return gemm_whole(y, y_dtype, x, w, bias, bias_dtype, nullptr, 1.0f, n_rows, n_out, n_in, 0, 1, packed, tile_shape, stream);
}

// xIELU on a product's way out: in tiles of 256 x 256, whose kernel is built for it (asked for at run time it slows every product),
// of packed weights whose product would stay whole.
// 4,001 rows against 8,192 x 2,048: 117 us and a pass of 49, together 147.
extern "C" int sb_gemm_mfma_xielu_ok(int n_rows, int n_out, int n_in) {
  return n_rows > 0 && n_out > 0 && n_in >= 128 && n_in % 64 == 0 && pick_shape(n_rows, n_out, n_in, 0, true) == 2 &&
         sb_gemm_mfma_slices(n_rows, n_out, n_in, 1) == 1;
}
extern "C" int sb_gemm_mfma_xielu_bf16(void *y, int y_dtype, const void *x, const void *w, int n_rows, int n_out, int n_in,
                                       const void *params, int params_dtype, void *stream) {
  SB_SUPPORT(sb_gemm_mfma_xielu_ok(n_rows, n_out, n_in), "sb_gemm_mfma_xielu_bf16: rows=%d out=%d in=%d are not taken", n_rows, n_out, n_in);
  SB_REQUIRE(params && sb::valid_dtype(params_dtype), "sb_gemm_mfma_xielu_bf16: xIELU takes two numbers");
  return gemm_whole(y, y_dtype, x, w, nullptr, 0, nullptr, 1.0f, n_rows, n_out, n_in, 0, 0, 1, -1, stream, params, params_dtype);
}

extern "C" int sb_gemm_mfma_bf16(void *y, int y_dtype, const void *x, const void *w, const void *bias,
                                 int bias_dtype, const float *resid, int n_rows, int n_out, int n_in,
                                 int gated, int packed, int tile_shape, void *stream) {
  return sb_gemm_mfma_scaled_bf16(y, y_dtype, x, w, bias, bias_dtype, resid, 1.0f, n_rows, n_out, n_in, gated, packed,
                                  tile_shape, stream);
}

// The same with a multiplier on the product before the residual joins: Y = resid_scale * (X W^T + bias) + resid
// (a multiplier of 1 gives the bits of the form above).
extern "C" int sb_gemm_mfma_scaled_bf16(void *y, int y_dtype, const void *x, const void *w, const void *bias,
                                        int bias_dtype, const float *resid, float resid_scale, int n_rows, int n_out,
                                        int n_in, int gated, int packed, int tile_shape, void *stream) {
  return gemm_whole(y, y_dtype, x, w, bias, bias_dtype, resid, resid_scale, n_rows, n_out, n_in, gated, 0, packed, tile_shape, stream);
}

namespace {
int gemm_whole(void *y, int y_dtype, const void *x, const void *w, const void *bias, int bias_dtype, const float *resid, float resid_scale,
               int n_rows, int n_out, int n_in, int gated, int relu_sq, int packed, int tile_shape, void *stream, const void *act_params,
               int act_dtype) {
  SB_REQUIRE(y && x && w, "sb_gemm_mfma_bf16: null pointer");
  SB_REQUIRE(n_rows >= 0 && n_out > 0 && n_in > 0, "sb_gemm_mfma_bf16: bad sizes rows=%d out=%d in=%d",
             n_rows, n_out, n_in);
  SB_REQUIRE(sb::valid_dtype(y_dtype) && (!bias || sb::valid_dtype(bias_dtype)),
             "sb_gemm_mfma_bf16: unknown dtype");
  SB_SUPPORT(n_in % 8 == 0, "sb_gemm_mfma_bf16: inner size %d is not a multiple of 8", n_in);
  SB_SUPPORT((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) % 16 == 0,
             "sb_gemm_mfma_bf16: operands must be 16-byte aligned");
  SB_REQUIRE(!(gated && (bias || resid)), "sb_gemm_mfma_bf16: the gated form takes no bias or residual");
  SB_SUPPORT(gated >= SB_GATE_NONE && gated <= SB_GATE_RELU, "sb_gemm_mfma_bf16: unknown gate activation %d", gated);
  if (n_rows == 0) return SB_OK;
  Args a;
  a.y = y; a.y_dtype = y_dtype; a.x = (const bf16_t *)x; a.w = (const bf16_t *)w;
  a.bias = bias; a.bias_dtype = bias_dtype; a.resid = resid; a.resid_scale = resid_scale;
  a.n_rows = n_rows; a.n_out = n_out; a.n_in = n_in; a.gated = gated; a.relu_sq = relu_sq;
  a.act_params = act_params; a.act_dtype = act_dtype;
  a.partial = nullptr; a.stages_per_slice = 0;
  a.vec4 = n_out % 4 == 0 && (reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(resid)) % 16 == 0;
  const bool direct_ok = packed && n_in % 64 == 0;
  int variant = pick_shape(n_rows, n_out, n_in, a.gated, direct_ok);
  // Tiles that make one round over the CUs go straight into LDS with four stages' buffers, a block a CU: a stage of 64 k then takes
  // 0.33 us in tiles of 64 x 128 and 0.55 in 128 x 128, through registers 0.65 (600 rows against 2,560 x 2,048 15.9, 21.4 and 22.6
  // us; 400 against 4,608 x 3,584 25.2, 30.0 and 33.8, 600 there, 360 tiles of 64, 46.5, 34.7 and 38.0; gated, 183 against 9,728 x 896 10.8, 13.3 and
  // 14.6, 288 there 18.1, 13.3 and 15.1).  Gated, a little over one round: 64 x 128 tiles, three to a CU (183 rows against 17,920 x
  // 1,536, 280 tiles of 128: 26.4 and 31.5).  Gated, past one round of tiles of 64 rows: the lowest of the tiles of 96, 128 and 192 whose
  // weights pass through registers that makes one round (figures at gemm_ahead_kernel; 66 to 120 rows against 11,008 x 2,048, in one round of 64 x
  // 128, 16.5 to 19.0 and 19.4 to 22.5 so).
  int path = 0;
  if (direct_ok && variant == 0) {
    const int bn = gated ? 64 : 128;
    const long long across = (n_out + bn - 1) / bn;
    const auto one_round = [&](long long tiles) { return (tiles + kXcds - 1) / kXcds * kXcds <= sb::cu_count(); };
    const long long tiles = (long long)((n_rows + 127) / 128) * across;
    if (one_round((long long)((n_rows + 63) / 64) * across)) variant = 5, path = 2;
    else if (gated && a.vec4 && one_round((long long)((n_rows + 95) / 96) * across)) variant = 6, path = 2;
    else if (gated && a.vec4 && one_round(tiles)) variant = 7, path = 2;
    else if (gated && a.vec4 && one_round((long long)((n_rows + 191) / 192) * across)) variant = 8, path = 2;
    else if (one_round(tiles)) path = 2;
    else if (gated && n_rows <= 384 && tiles <= sb::cu_count() * 3 / 2 && (n_rows + 63) / 64 * 64 < (n_rows + 127) / 128 * 128)
      variant = 5, path = 2;
  }
  // a test's or a measurement's choice: the shape (0..8) + 16 * the path (0: the launcher's, 1:
  // through registers, 2: straight into LDS)
  if (tile_shape >= 0) {
    SB_REQUIRE((tile_shape & 15) < 9 && (tile_shape >> 4) < 4, "sb_gemm_mfma_bf16: unknown tile shape %d", tile_shape);
    variant = tile_shape & 15;
    path = tile_shape >> 4;
  }
  if (!packed) variant = 0, path = 0;       // the bigger tiles are built for packed weights only
  const int bm = kShapes[variant].bm, bn = gated ? kShapes[variant].bn / 2 : kShapes[variant].bn;
  a.tiles_m = (n_rows + bm - 1) / bm;
  a.tiles_n = (n_out + bn - 1) / bn;
  const long long blocks = (long long)a.tiles_m * a.tiles_n;
  SB_SUPPORT(blocks <= 0x7fffffffLL, "sb_gemm_mfma_bf16: too many tiles");
  // the kernel addresses both operands with 32-bit byte offsets
  const unsigned long long w_rows = (unsigned long long)((n_out + 15) / 16 * 16) * (gated ? 2 : 1);
  const unsigned long long k_padded = (unsigned long long)((n_in + 31) / 32 * 32);
  // ... also for the rows and row tiles past an operand's end that a block at the edge asks for
  // (they lie past the descriptor's end and read as zero, but must not wrap around)
  SB_SUPPORT(((unsigned long long)n_rows + 257) * n_in * 2 < (1ull << 32) - (1ull << 20) &&
                 (w_rows + 512) * k_padded * 2 < (1ull << 32) - (1ull << 20),
             "sb_gemm_mfma_bf16: an operand of 4 GiB or more (rows=%d out=%d in=%d)", n_rows, n_out, n_in);
  hipStream_t s = (hipStream_t)stream;
  a.w_tiles = (n_out + 15) / 16;
  a.w_steps = (n_in + 31) / 32;
  int rc;
  SB_SUPPORT(path < 2 || direct_ok, "sb_gemm_mfma_bf16: the direct path takes packed weights and an inner size in 64s");
  // left to themselves the shapes of 192 and 256 rows go straight into LDS; the smaller tiles' stages are too
  // short for loads that run one stage ahead, and the register path, which runs two ahead, is
  // faster there unless the tiles make one round and LDS holds four stages of each (above)
  const bool direct = path >= 2 || (path == 0 && direct_ok && (variant == 1 || variant == 2 || variant == 4));
  SB_SUPPORT(variant < 6 || (gated && a.vec4 && direct), "sb_gemm_mfma_bf16: the shapes whose weights pass through registers are gated ones");
  SB_SUPPORT(variant < 3 || direct, "sb_gemm_mfma_bf16: the shapes from 128 x 256 on exist on the direct path only");
  if (direct) {
    // the shapes of four waves take as many buffers as the tiles' count leaves LDS for: four (a block a CU, three
    // stages in flight) in one round over the CUs, else two (two or three blocks a CU)
    const bool one_round = (blocks + kXcds - 1) / kXcds * kXcds <= sb::cu_count();
    if (variant == 0) rc = one_round ? launch_direct<4, 2, 64, 4, false>(a, blocks, 0, s) : launch_direct<4, 2, 64, 2, false>(a, blocks, 0, s);
    else if (variant == 1) rc = launch_pipe<true>(a, blocks, path == 3, s);
    else if (variant == 2) rc = launch_pipe<false>(a, blocks, path == 3, s);      // (path 3: a measurement's)
    else if (variant == 3) rc = launch_direct<4, 4, 64, 2, false>(a, blocks, 0, s);
    else if (variant == 4) rc = launch_direct<6, 4, 64, 2, true>(a, blocks, sb::cu_count(), s);
    else if (variant == 6) rc = launch_ahead<6>(a, blocks, s);
    else if (variant == 7) rc = launch_ahead<8>(a, blocks, s);
    else if (variant == 8) rc = launch_ahead<12>(a, blocks, s);
    else rc = one_round ? launch_direct<2, 2, 64, 4, false>(a, blocks, 0, s) : launch_direct<2, 2, 64, 2, false>(a, blocks, 0, s);
  } else {
    if (variant == 0) rc = launch<2, 2, 64, 2, true>(a, blocks, packed, s);
    else if (variant == 1) rc = launch<4, 2, 64, 2, false>(a, blocks, packed, s);
    else rc = launch<4, 4, 64, 1, false>(a, blocks, packed, s);
  }
  if (rc != SB_OK) return rc;
  return sb::check_launch("sb_gemm_mfma_bf16");
}
}  // namespace

namespace {
// K slices of the partial form, and the tiles that multiply them.  Few rows: enough blocks for
// the GPU (one 128 x 128 tile per CU and slice), every slice at least four stages of 64 long, at
// most the eight that the consumers add.  Where that gives one slice, a problem with few tiles
// of 256 x 256 (a prompt of one or two thousand rows against a matrix a few thousand wide) may
// still be faster with those tiles, loaded straight into LDS, and K cut so that the tiles and
// slices together make one round over the CUs.  Both ways are priced in microseconds from
// what was measured on MI355X with the 7B products at 768 to 2,304 rows: a shape's tile takes
// 2 bm bn K flops at its kernel's rate on a full GPU (1 standing for 0.93
// PFLOP/s over 256 CUs); a round that leaves CUs idle runs faster (0.72 of the time with up to 170
// blocks, rising to 1 at 256: the chip's clock follows its load); either kernel costs 14 us
// beside its tiles; the consumer's pass over the additional slices moves (2 slices - 2) x the
// result's bytes at 4 TB/s.  The cut is taken when it comes out under 0.9 of the best whole
// product.  The 1.05 of tiles of 256 x 128 is not that kernel's speed (1.24, pick_shape) but what places this line: the pass
// over a whole product's result is in neither price, and with 1.24 the down product of 1,536 rows and more would stay whole.
// Measured one after the other with cold weights, whole + norm against the cut taken + the pass that adds the slices, the residual and
// the norm, us: 3,584 x 18,944 at 1,024 rows 185 and 130, 1,280 226 and 157, 1,536 227 and 204, 1,792 241 and 220, 2,048 254 and 239,
// 2,304 277 and 253; 2,560 x 9,728 at 1,792 130 and 96, 2,304 138 and 122; 3,072 x 8,192 at 1,536 109 and 87, 2,048 114 and 115; 4,096 x
// 14,336 at 1,280 177 and 136, 2,048 210 and 203; 5,120 x 13,824 at 896 165 and 127, 1,536 200 and 190.  Left whole: 3,584 x 3,584 at 2,048 rows 69
// (cut in two 71); and, where the cut would be ahead, 1,152 rows of 3,584 x 18,944 181 (three 151), 1,792 and 2,048 rows of 2,048 x
// 11,008 109 and 111 (three 98 and 107), 896 rows of 4,096 x 14,336 138 (four 104).  Prices fitted to all of these (to 4 %) take those cuts as well; in
// whole prompt steps that gave 4.5 % at 1,152 rows of the 7B sizes, nothing at 1,792 of the 3B ones, and cost 1 % at 2,048 of the
// 3B sizes and at 1,800 and 2,300 of 2,048 wide layers of other designs: not taken.
//
// Some hundred rows: the same tiles of 128 x 128, or of 64 x 128, loaded straight into LDS with four
// stages' buffers, a block a CU, where tiles x slices make one round over each die's 32 CUs, or a whole product whose tiles make one.
// Prices in microseconds, fitted to 292 sizes of 96 to 3,500 rows in all their cuts (slices and the pass that adds them, the stream and its
// norm, against the whole product and the norm; replayed graphs, weights cold): a stage of 64 k 0.29 (64 rows), 0.41 (128 rows; in a whole
// product 0.525) and 0.8 (128 x 128 through registers); a slice is written and read at 3.1 TB/s, past 32 MB (what
// the dies' L2 hold) at 2.8, the stream and its norm take two and a half times as much, and a whole product one plane and 2.6 us more; past
// 1,150 rows slices through registers are never ahead.  The choice is 2.2 % behind the best on the mean (3.6 with the prices before), most where
// a whole product takes larger tiles than the price knows: 700 x 3,584 x 18,944 (rows, out, in) 120 us whole, 154 in slices.  us, the best cut / the
// choice with prices of 183 to 900 rows that changed their rate at 640 / this one: 288 x 4,096 x 14,336 60.6 / 82.3 / 60.6; 400 x 3,072 x
// 8,192 38.9 / 50.2 / 38.9; 520 x 2,560 x 9,728 46.4 / 59.9 / 46.4; 640 x 1,536 x 8,960 35.6 / 39.1 / 35.6; 1,000 x 1,152 x 896 15.0 / 19.1 / 15.0; 1,200 x
// 896 x 896 14.7 / 19.4 / 14.8; but 600 x 2,560 x 2,048 21.4 / 21.4 / 22.6.
enum PartialTile { kRegisters128, kBig, kDirect128, kDirect64 };
struct PartialPlan { int slices; PartialTile tile; };
double load_factor(long long blocks) { return blocks <= 170 ? 0.72 : 0.72 + 0.28 * double(blocks - 170) / 86.0; }
PartialPlan partial_plan(int n_rows, int n_out, int n_in, bool direct_ok) {
  const long long tiles = (long long)((n_rows + 127) / 128) * ((n_out + 127) / 128);
  const int n_k = (n_in + 63) / 64;
  long long s = (224 + tiles - 1) / tiles;
  if (s > n_k / 4) s = n_k / 4;
  if (s > 8) s = 8;
  if (s < 1) s = 1;
  const long long big = (long long)((n_rows + 255) / 256) * ((n_out + 255) / 256);
  const long long big_grid = (big + kXcds - 1) / kXcds * kXcds;       // the grid is padded to whole eights
  if (s == 1 && direct_ok && 2 * big_grid <= sb::cu_count()) {
    const double per_cu = 0.93e9 / 256.0;                                        // a CU's flops per microsecond at speed 1
    const double speed[5] = {1.0, 1.05, 1.45, 0.0, 1.2};                         // (256 x 128: see above)
    double t_whole = 0;
    for (int v = 0; v < 5; ++v) {
      if (v == 3) continue;
      const int bm = kShapes[v].bm, bn = kShapes[v].bn;
      const long long n_tiles = (long long)((n_rows + bm - 1) / bm) * ((n_out + bn - 1) / bn);
      const long long rounds = (n_tiles + sb::cu_count() - 1) / sb::cu_count(), last = n_tiles - (rounds - 1) * sb::cu_count();
      const double t = 2.0 * bm * bn * double(n_in) / (speed[v] * per_cu) * (double(rounds - 1) + load_factor(last)) + 14.0;
      if (v == 0 || t < t_whole) t_whole = t;
    }
    double t_best = 0;
    long long s_best = 0;
    for (long long s2 = 2; s2 <= 8 && s2 * big_grid <= sb::cu_count() && s2 <= n_k / 4; ++s2) {
      const int per = int((n_k + s2 - 1) / s2);
      const double t = 2.0 * 256 * 256 * (64.0 * per) / (speed[2] * per_cu) * load_factor(s2 * big_grid) + 14.0 +
                       (2.0 * s2 - 2.0) * n_rows * double(n_out) * 4.0 / 4e6;
      if (s_best == 0 || t < t_best) t_best = t, s_best = s2;
    }
    if (s_best && t_best < 0.9 * t_whole) {
      const int per = int((n_k + s_best - 1) / s_best);
      return {(n_k + per - 1) / per, kBig};
    }
  }
  if (s > 1 && direct_ok) {
    const double plane_mb = n_rows * double(n_out) * 4e-6;
    const auto pass_us = [](double mb) { return mb <= 32.0 ? 0.325 * mb : 0.325 * 32.0 + 0.36 * (mb - 32.0); };      // to write or read
    const auto cost = [&](double stage_us, long long slices) {
      return stage_us * double((n_k + slices - 1) / slices) + 2.0 * pass_us(slices * plane_mb) + 2.5 * pass_us(plane_mb);
    };
    const auto one_round = [&](long long n_tiles) { return (n_tiles + kXcds - 1) / kXcds <= sb::cu_count() / kXcds; };
    const auto tiles_of = [&](int bm) { return (long long)((n_rows + bm - 1) / bm) * ((n_out + 127) / 128); };
    double best = cost(0.8, s);
    PartialTile tile = kRegisters128;
    for (int half = 0; half < 2; ++half) {
      const long long n_tiles = tiles_of(half ? 64 : 128);
      for (long long s2 = 2; s2 <= 8 && (n_tiles + kXcds - 1) / kXcds * s2 <= sb::cu_count() / kXcds && s2 * 3 <= n_k; ++s2) {
        const double t = cost(half ? 0.29 : 0.41, s2);
        if (t < best) best = t, tile = half ? kDirect64 : kDirect128, s = s2;
      }
    }
    const double stage_whole = one_round(tiles_of(64)) ? 0.29 : one_round(tiles_of(128)) ? 0.525 : 0.0;
    if ((tile == kRegisters128 && n_rows > 1150) || (stage_whole > 0.0 && stage_whole * n_k + 3.5 * pass_us(plane_mb) + 2.6 < best))
      return {1, kRegisters128};
    const int per = int((n_k + s - 1) / s);
    return {(n_k + per - 1) / per, tile};
  }
  const int per = int((n_k + s - 1) / s);
  return {(n_k + per - 1) / per, kRegisters128};
}
}  // namespace

// Slices sb_gemm_mfma_partial_bf16 writes for these sizes.
extern "C" int sb_gemm_mfma_slices(int n_rows, int n_out, int n_in, int packed) {
  return partial_plan(n_rows, n_out, n_in, packed && n_in % 64 == 0).slices;
}

// The raw product X W^T in K slices: partial float [slices][n_rows][n_out], for a consumer that
// adds the slices itself.  For few rows against a narrow, long matrix, where one slice would not
// give the GPU enough tiles.  128 x 128 tiles, or 256 x 256 (see partial_plan).
extern "C" int sb_gemm_mfma_partial_bf16(float *partial, const void *x, const void *w, int n_rows, int n_out,
                                         int n_in, int packed, void *stream) {
  SB_REQUIRE(partial && x && w, "sb_gemm_mfma_partial_bf16: null pointer");
  SB_REQUIRE(n_rows >= 0 && n_out > 0 && n_in > 0, "sb_gemm_mfma_partial_bf16: bad sizes rows=%d out=%d in=%d",
             n_rows, n_out, n_in);
  SB_SUPPORT(n_in % 8 == 0, "sb_gemm_mfma_partial_bf16: inner size %d is not a multiple of 8", n_in);
  SB_SUPPORT((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) % 16 == 0,
             "sb_gemm_mfma_partial_bf16: operands must be 16-byte aligned");
  if (n_rows == 0) return SB_OK;
  Args a;
  a.y = nullptr; a.y_dtype = SB_F32; a.x = (const bf16_t *)x; a.w = (const bf16_t *)w;
  a.bias = nullptr; a.bias_dtype = 0; a.resid = nullptr; a.resid_scale = 1.0f;
  a.n_rows = n_rows; a.n_out = n_out; a.n_in = n_in; a.gated = 0; a.relu_sq = 0; a.act_params = nullptr; a.act_dtype = 0;
  const PartialPlan plan = partial_plan(n_rows, n_out, n_in, packed && n_in % 64 == 0);
  const int bm = plan.tile == kBig ? 256 : plan.tile == kDirect64 ? 64 : 128, bn = plan.tile == kBig ? 256 : 128;
  a.tiles_m = (n_rows + bm - 1) / bm;
  a.tiles_n = (n_out + bn - 1) / bn;
  const long long blocks = (long long)a.tiles_m * a.tiles_n;
  SB_SUPPORT(blocks <= 0x7fffffffLL, "sb_gemm_mfma_partial_bf16: too many tiles");
  const unsigned long long w_rows = (unsigned long long)((n_out + 15) / 16 * 16);
  const unsigned long long k_padded = (unsigned long long)((n_in + 31) / 32 * 32);
  // with room for the rows and row tiles past an operand's end that a block at the edge asks for
  SB_SUPPORT(((unsigned long long)n_rows + 257) * n_in * 2 < (1ull << 32) - (1ull << 20) &&
                 (w_rows + 512) * k_padded * 2 < (1ull << 32) - (1ull << 20),
             "sb_gemm_mfma_partial_bf16: an operand of 4 GiB or more");
  a.w_tiles = (n_out + 15) / 16;
  a.w_steps = (n_in + 31) / 32;
  const int slices = plan.slices;
  const int n_k = (n_in + 63) / 64;
  a.partial = partial;
  a.vec4 = n_out % 4 == 0 && reinterpret_cast<uintptr_t>(partial) % 16 == 0;
  a.stages_per_slice = (n_k + slices - 1) / slices;
  hipStream_t st = (hipStream_t)stream;
  const int rc = plan.tile == kBig         ? launch_pipe_one<0, false, false>(a, blocks, st)
                 : plan.tile == kDirect128 ? launch_direct_one<4, 2, 64, 4, 0, false>(a, blocks, 0, st)
                 : plan.tile == kDirect64  ? launch_direct_one<2, 2, 64, 4, 0, false>(a, blocks, 0, st)
                                           : launch<2, 2, 64, 2, true>(a, blocks, packed, st);
  if (rc != SB_OK) return rc;
  return sb::check_launch("sb_gemm_mfma_partial_bf16");
}

