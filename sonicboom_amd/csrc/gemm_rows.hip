// bf16 products of up to eight rows against large packed matrices (decode): Y[t,n] = sum_k X[t,k] W[n,k].
//
// They are bound by reading W once, so all that counts is that W's loads never stop.  A block keeps its share of X in LDS for
// good and goes from tile to tile (16 features, or 16 gate/up pairs); its waves take the k-steps of a tile in turn (step s is
// wave s % W's, so that a block reads whole runs of W), each with a ring of kAhead loads of every stream in flight that runs on
// into the next tile.  The waves' sums meet in LDS, two buffers in turn so that one barrier a tile is enough, and the waves take
// turns at adding them up (in wave order) and writing the result.  X and, for an unfinished norm, the sums of squares are asked
// for ahead of W's ring and put away behind it: asked for behind it, they would wait for it, and W for them.  The order of a
// step's loads and products is kept as written: left alone the compiler gathers a round's loads behind its last product.
//
// Measured (us, replayed graphs, weights cold; against the kernels that read X's fragments beside W's, one and eight rows):
// gated 18,944 x 3,584 46.6 -> 45.7, 49.1 -> 45.8 (a plain read in this order of addresses 42); 13,824 x 5,120 51.9 -> 50.4,
// 54.3 -> 49.5; 14,336 x 4,096 43.2 -> 39.2, 45.5 -> 39.3; 11,008 x 2,048 19.5 -> 17.4, 20.4 -> 17.7; 8,960 x 1,536 14.5 -> 13.7,
// 15.3 -> 14.2; 5,632 x 2,048 12.8 -> 11.2, 13.6 -> 11.2; 4,864 x 896 7.1 -> 7.2, 7.3 -> 7.2.  In K slices, against the kernel whose
// waves split the features: 3,584 x 18,944 24.9 -> 23.2, 25.4 -> 24.0; 2,048 x 11,008 10.0 -> 9.0, 10.2 -> 9.8; 1,536 x 8,960 7.5 ->
// 6.3, 7.7 -> 7.0; 896 x 4,864 4.9 -> 3.9, 5.0 -> 4.5; 4,608 x 3,584 8.5 -> 7.3, 8.7 -> 8.5; 7,168 x 5,120 15.1 -> 12.9, 15.3 -> 13.7.
// At sixteen rows X's way into LDS takes what is gained (3,584 x 18,944 26.0 and 25.7, 4,096 x 14,336 21.4 and 23.2).
//
// MFMA roles: A = 16 rows of W, B = 16 rows of X, D[n][t]; a lane holds four consecutive n of one t.
#include "gemm_rows.h"

#include "mfma.h"

namespace {

constexpr int kMaxRows = 8;
constexpr int kTile = 16;
constexpr int kAhead = 4;           // k-steps a wave has in flight of every stream
constexpr size_t kLds = 160 * 1024;

struct RowsArgs {
  int n_rows, n_out, n_in;
  int steps_per_slice, rounds;      // of K; rounds: of kAhead steps a wave that a slice takes
  const double *ssq;                // gated: [ssq_parts][n_rows], or NULL
  int ssq_parts;
  float eps;
  int gate;
  void *y;                          // gated: bf16 [n_rows][n_out]; else float [slices][n_rows][n_out]
};

// BATCH: 16-byte groups of X a thread asks for ahead of W's ring (the rest, if any, behind it).
template <bool GATED, int W, int BATCH>
__global__ void __launch_bounds__(64 * W)
gemm_rows_kernel(const bf16_t *__restrict__ x, const bf16_t *__restrict__ w, RowsArgs a) {
  constexpr int G = GATED ? 2 : 1;
  constexpr int kThreads = 64 * W, kRound = kAhead * W;
  constexpr int kGroups = kThreads / kTile;      // threads a row that add its sums of squares
  constexpr int kParts = 8;                      // sums a thread asks for ahead of W's ring
  extern __shared__ uint4 xs[];                  // [n_rows][stride]
  __shared__ floatx4_t red[2][W * G * 64];
  __shared__ double row_part[GATED ? kGroups * kTile : 1];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int tiles = (a.n_out + kTile - 1) / kTile, n_steps = (a.n_in + 31) / 32;
  const int s0 = int(blockIdx.y) * a.steps_per_slice, s1 = min(s0 + a.steps_per_slice, n_steps);
  // 16-byte groups of a staged row: whole rounds, zeros past the slice's end; one more of padding, so that a fragment's
  // sixteen rows start on distinct banks
  const int units = a.rounds * kRound * 4, stride = units + 1, x_units = a.n_rows * units;

  // what lies outside of a descriptor reads as zeros: a tile past the last, a step past the slice's end, a row past the last
  constexpr uint32_t kOutside = 0x80000000u;
  const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16_t *>(x), 0, uint32_t(size_t(a.n_rows) * a.n_in * 2), 0x00020000);
  const auto x_load = [&](int id) {
    const int row = id / units, k = s0 * 32 + (id - row * units) * 8;            // (n_in is a multiple of 8)
    const bool in = id < x_units && k < a.n_in && k < s1 * 32;
    return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(
        rsrc_x, int(in ? uint32_t((size_t(row) * a.n_in + k) * 2) : kOutside), 0, 0));
  };
  const auto x_store = [&](int id, uint4 v) {
    const int row = id / units;
    if (id < x_units) xs[row * stride + (id - row * units)] = v;
  };
  const auto stream = [&](int tile, int g) {
    const bool in = tile < tiles;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t *>(w) + size_t(g * tiles + (in ? tile : 0)) * n_steps * 512, 0,
                                             in ? uint32_t(s1) * 1024u : 0u, 0x00020000);
  };

  uint4 xb[BATCH];
#pragma unroll
  for (int i = 0; i < BATCH; ++i) xb[i] = x_load(tid + i * kThreads);
  const int sq_row = tid % kTile, sq_group = tid / kTile;
  double parts[kParts];
  if constexpr (GATED) {
    typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
    const __amdgpu_buffer_rsrc_t rsrc_s = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<double *>(a.ssq), 0, a.ssq ? uint32_t(a.ssq_parts) * uint32_t(a.n_rows) * 8u : 0u, 0x00020000);
#pragma unroll
    for (int i = 0; i < kParts; ++i) {
      const uint32_t at = uint32_t(sq_group + i * kGroups) * uint32_t(a.n_rows) + sq_row;
      const u32x2_t v = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(rsrc_s, int(sq_row < a.n_rows ? at * 8u : kOutside), 0, 0));
      parts[i] = __builtin_bit_cast(double, v);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  int tile = blockIdx.x;
  __amdgpu_buffer_rsrc_t now[G];
#pragma unroll
  for (int g = 0; g < G; ++g) now[g] = stream(tile, g);
  const int w_lane = lane * 16 + (s0 + wave) * 1024;
  uint4 ring[kAhead][G];
  const auto ask = [&](int u, int g, const __amdgpu_buffer_rsrc_t &rsrc, int from) {
    ring[u][g] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, from + u * W * 1024, 0, kReadOnce));
  };
#pragma unroll
  for (int u = 0; u < kAhead; ++u)
#pragma unroll
    for (int g = 0; g < G; ++g) ask(u, g, now[g], w_lane);
  __builtin_amdgcn_sched_barrier(0);

#pragma unroll
  for (int i = 0; i < BATCH; ++i) x_store(tid + i * kThreads, xb[i]);
  for (int id = tid + BATCH * kThreads; id < x_units; id += BATCH * kThreads) {
#pragma unroll
    for (int i = 0; i < BATCH; ++i) xb[i] = x_load(id + i * kThreads);
#pragma unroll
    for (int i = 0; i < BATCH; ++i) x_store(id + i * kThreads, xb[i]);
  }
  if constexpr (GATED) {
    double sum = 0.0;
#pragma unroll
    for (int i = 0; i < kParts; ++i) sum += parts[i];
    if (a.ssq && sq_row < a.n_rows)
      for (int p = sq_group + kParts * kGroups; p < a.ssq_parts; p += kGroups) sum += a.ssq[size_t(p) * a.n_rows + sq_row];
    row_part[sq_group * kTile + sq_row] = sum;
  }
  // a barrier for what is in LDS alone: W's loads stay in flight across it
  const auto meet = [] {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  meet();
  float factor = 1.0f;
  if constexpr (GATED) {
    if (a.ssq) {
      double sum = 0.0;
#pragma unroll
      for (int k = 0; k < kGroups; ++k) sum += row_part[k * kTile + r];
      factor = 1.0f / sqrtf(float(sum / double(a.n_in)) + a.eps);
    }
  }

  // (rows past the last one read the last one again: their columns of D are not stored)
  const uint4 *my_x = xs + min(r, a.n_rows - 1) * stride + q + wave * 4;
  int buf = 0, turn = 0;
  for (; tile < tiles; tile += gridDim.x) {
    __amdgpu_buffer_rsrc_t next[G];
    floatx4_t acc[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      next[g] = stream(tile + gridDim.x, g);
      acc[g] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    }
    for (int c = 0; c < a.rounds; ++c) {
      const bool last = c + 1 == a.rounds;
      const int from = w_lane + (last ? 0 : (c + 1) * kRound * 1024);
      const uint4 *bx = my_x + c * (kRound * 4);
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const bf16x8_t b = as_bf16x8(bx[u * W * 4]);
#pragma unroll
        for (int g = 0; g < G; ++g) acc[g] = mfma16(as_bf16x8(ring[u][g]), b, acc[g]);
#pragma unroll
        for (int g = 0; g < G; ++g) ask(u, g, last ? next[g] : now[g], from);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int g = 0; g < G; ++g) red[buf][(wave * G + g) * 64 + lane] = acc[g];
    meet();
    if (wave == turn) {
      floatx4_t v[G];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        v[g] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < W; ++k) v[g] = v[g] + red[buf][(k * G + g) * 64 + lane];
      }
      const int n = tile * kTile + 4 * q;
      if (r < a.n_rows) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (n + e >= a.n_out) continue;
          if constexpr (GATED)
            ((bf16_t *)a.y)[size_t(r) * a.n_out + n + e] = f32_to_bf16(gate_act(v[0][e] * factor, a.gate) * (v[G - 1][e] * factor));
          else ((float *)a.y)[(size_t(blockIdx.y) * a.n_rows + r) * a.n_out + n + e] = v[0][e];
        }
      }
    }
    turn = turn + 1 == W ? 0 : turn + 1;
    buf ^= 1;
#pragma unroll
    for (int g = 0; g < G; ++g) now[g] = next[g];
  }
}

// Rounds of kAhead steps a wave, of W waves, in `steps` steps; the bytes of X's share in LDS.
int rounds_of(int steps, int w) { return (steps + kAhead * w - 1) / (kAhead * w); }
size_t x_bytes(int n_rows, int steps, int w) { return size_t(n_rows) * (size_t(rounds_of(steps, w)) * kAhead * w * 4 + 1) * 16; }

// 32-bit byte offsets into X and into a stream of W
bool reach(int n_rows, int n_out, int n_in) {
  return n_rows > 0 && n_rows <= kMaxRows && n_out > 0 && n_in > 0 && n_in % 8 == 0 &&
         (unsigned long long)(n_rows + 1) * n_in * 2 < (1ull << 31) && (unsigned long long)n_in * 32 < (1ull << 31);
}

// Waves a block of the whole forms: four where a tile has few steps (2,048 k: 17.4 us of 11,008 pairs with four, 18.1 with
// eight), eight where it has more (4,096 k: 40.4 and 39.0 of 14,336 pairs, 3,072: 20.0 and 19.5 of 8,192).
constexpr int kFewSteps = 80;

// LDS of a block besides X's share: where the waves' sums meet, and the parts of the rows' sums of squares.
constexpr size_t own_bytes(bool gated, int w) {
  return sizeof(floatx4_t) * 2 * w * (gated ? 2 : 1) * 64 + sizeof(double) * (gated ? 64 * w : 1);
}

// Blocks of a whole form: at most `each` a CU, and no more than its LDS holds: one that waits for a place stages X when the others are
// done, and its share runs by itself.  Eight rows, us, three a CU where two fit and so: gated 13,824 x 2,560 28.7 -> 27.0, 20,480 x 2,560
// 39.2 -> 35.7, 27,648 x 2,560 49.6 -> 47.0; two where one fits: plain 40,000 x 3,584 48.5 -> 46.8, 152,064 x 3,584 175.3 -> 173.7, 32,000 x
// 4,096 45.1 -> 43.7, but 128,256 x 4,096 166.4 and 166.6.
int blocks_for(const RowsArgs &a, bool gated, int w, int each) {
  const int tiles = (a.n_out + kTile - 1) / kTile, fit = int(kLds / (x_bytes(a.n_rows, a.steps_per_slice, w) + own_bytes(gated, w)));
  const int most = (each < fit ? each : fit) * sb::cu_count();
  return tiles < most ? tiles : most;
}

template <bool GATED, int W, int BATCH>
int launch(const char *who, const void *x, const void *w, RowsArgs a, int blocks, int slices, hipStream_t s) {
  a.rounds = rounds_of(a.steps_per_slice, W);
  const size_t lds = x_bytes(a.n_rows, a.steps_per_slice, W);
  const auto kern = gemm_rows_kernel<GATED, W, BATCH>;
  constexpr int kMost = int(kLds - own_bytes(GATED, W));
  static bool raised = false;      // once per instantiation: X's share and the block's own LDS may be more than the default allows
  if (!raised) {
    const hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, kMost);
    SB_REQUIRE(e == hipSuccess, "%s: cannot reserve %d bytes of LDS: %s", who, kMost, hipGetErrorString(e));
    raised = true;
  }
  kern<<<dim3(blocks, slices), 64 * W, lds, s>>>((const bf16_t *)x, (const bf16_t *)w, a);
  return sb::check_launch(who);
}

// K cut over the grid: slices, and blocks that each slice's tiles are dealt out to.
struct Cut {
  int slices, steps_per_slice, blocks;
};
// The cost of a choice: what the CU with the most blocks works through (a tile: its steps, half of those that fill its last round,
// and two for its end; a block: 20 steps until it streams and 2.5 a row that it stages), and 50 where not every CU has two blocks.
// Over 36 matrices of one to eight rows, each in some 35 ways, its choice is 1.4 % behind the best one.
Cut cut_for(int n_rows, int n_out, int n_in, size_t share) {
  constexpr int kMostSteps = 240;        // (a block's steps: 2 slices of 296 steps, 3,584 x 18,944, 25.0 us where 4 take 22.2)
  const int tiles = (n_out + kTile - 1) / kTile, n_steps = (n_in + 31) / 32, n_cu = sb::cu_count();
  Cut best{0, 0, 0};
  double best_cost = 0.0;
  for (int want = 1; want <= 8; ++want) {
    const int sps = (n_steps + want - 1) / want, slices = (n_steps + sps - 1) / sps;
    if (slices != want || sps > kMostSteps || x_bytes(n_rows, sps, 8) > share) continue;
    const double tile_cost = 0.5 * rounds_of(sps, 8) * kAhead * 8 + 0.5 * sps + 2.0;
    for (int each = 1; each <= 8; ++each) {
      const int blocks = (tiles + each - 1) / each;
      const long long all = (long long)blocks * slices, rounds = (all + n_cu - 1) / n_cu;
      const double spare = 2.0 - double(all) / n_cu;
      const double cost = double(rounds) * (each * tile_cost + 20.0 + 2.5 * n_rows) + (spare > 0.0 ? 50.0 * spare : 0.0);
      if (!best.slices || cost < best_cost) best = Cut{slices, sps, blocks}, best_cost = cost;
    }
  }
  return best;
}
// X's share in LDS: 44 KB, or where no cut gives that little 50, so that a CU still holds two blocks.
Cut cut_for(int n_rows, int n_out, int n_in) {
  const Cut c = cut_for(n_rows, n_out, n_in, 44000);
  return c.slices ? c : cut_for(n_rows, n_out, n_in, 50000);
}

}  // namespace

namespace sb {

// Matrices of more than four million weights: of 2,048 x 2,048 the kernel whose waves split the features is ahead (one row 3.55 us
// and 3.64, eight 3.7 and 4.2), of 896 x 4,864 this one.
int rows_slices(int n_rows, int n_out, int n_in) {
  if (!reach(n_rows, n_out, n_in) || (long long)n_out * n_in <= (4ll << 20)) return 0;
  return cut_for(n_rows, n_out, n_in).slices;
}

int rows_partial(float *partial, const void *x, const void *w, int n_rows, int n_out, int n_in, void *stream) {
  const Cut c = cut_for(n_rows, n_out, n_in);
  SB_REQUIRE(c.slices > 0 && reach(n_rows, n_out, n_in), "rows_partial: sizes that it does not take");
  RowsArgs a{};
  a.n_rows = n_rows, a.n_out = n_out, a.n_in = n_in, a.steps_per_slice = c.steps_per_slice, a.y = partial;
  return n_rows <= 4 ? launch<false, 8, 2>("rows_partial", x, w, a, c.blocks, c.slices, (hipStream_t)stream)
                     : launch<false, 8, 4>("rows_partial", x, w, a, c.blocks, c.slices, (hipStream_t)stream);
}

// (Gated ones from 512 k: 9,001 pairs of 40 k 4.5 us in the kernel whose waves split the features and 6.0 here.)
bool rows_whole(int n_rows, int n_out, int n_in, int gated) {
  if (gated && n_in < 512) return false;
  const int steps = (n_in + 31) / 32, w = steps <= kFewSteps ? 4 : 8;
  const size_t fixed = sizeof(floatx4_t) * 2 * w * (gated ? 2 : 1) * 64 + 64 * w * sizeof(double);
  return reach(n_rows, n_out, n_in) && x_bytes(n_rows, steps, w) + fixed <= kLds;
}

int rows_gated(void *y, const void *x, const double *ssq, int ssq_parts, float eps, const void *w, int n_rows, int n_out, int n_in,
               int gate, void *stream) {
  SB_REQUIRE(rows_whole(n_rows, n_out, n_in, 1), "rows_gated: sizes that it does not take");
  RowsArgs a{};
  a.n_rows = n_rows, a.n_out = n_out, a.n_in = n_in, a.steps_per_slice = (n_in + 31) / 32;
  a.ssq = ssq, a.ssq_parts = ssq_parts, a.eps = eps, a.gate = gate, a.y = y;
  return a.steps_per_slice <= kFewSteps ? launch<true, 4, 8>("rows_gated", x, w, a, blocks_for(a, true, 4, 3), 1, (hipStream_t)stream)
                                        : launch<true, 8, 8>("rows_gated", x, w, a, blocks_for(a, true, 8, 1), 1, (hipStream_t)stream);
}

int rows_plain(float *y, const void *x, const void *w, int n_rows, int n_out, int n_in, void *stream) {
  SB_REQUIRE(rows_whole(n_rows, n_out, n_in, 0), "rows_plain: sizes that it does not take");
  RowsArgs a{};
  a.n_rows = n_rows, a.n_out = n_out, a.n_in = n_in, a.steps_per_slice = (n_in + 31) / 32, a.y = y;
  return a.steps_per_slice <= kFewSteps ? launch<false, 4, 8>("rows_plain", x, w, a, blocks_for(a, false, 4, 3), 1, (hipStream_t)stream)
                                        : launch<false, 8, 8>("rows_plain", x, w, a, blocks_for(a, false, 8, 2), 1, (hipStream_t)stream);
}

}  // namespace sb
