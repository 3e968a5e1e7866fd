// Products of many bfloat16 rows with the inner loop of tile_ring.h, for what the vendor's library does not do or does slowly:
// C = A W^T in parts of K for the norm that follows to add (few tiles, long K), and the gated product
// act(A Wg^T) * (A Wu^T) in one kernel, gate and up sums meeting in a lane's registers.
#include "common.h"
#include "splitk_reduce.h"
#include "tile_ring.h"

enum { RING_PLAIN = 0, RING_SILU = 1, RING_GELU = 2, RING_RELU = 3, RING_CAPPED = 4 };

template <int GATE>
__device__ __forceinline__ float ring_gate(float z, float u, float alpha, float limit, float shift) {
  if constexpr (GATE == RING_SILU) return z / (1.0f + __expf(-z)) * u;
  else if constexpr (GATE == RING_RELU) return fmaxf(z, 0.f) * u;
  else if constexpr (GATE == RING_CAPPED) {
    const float g = fminf(z, limit);
    return g / (1.0f + __expf(-alpha * g)) * (fminf(fmaxf(u, -limit), limit) + shift);
  } else {
    const float t = 0.7978845608028654f * (z + 0.044715f * z * z * z);
    return 0.5f * z * (2.0f - 2.0f / (1.0f + __expf(2.0f * t))) * u;        // 1 + tanh(t)
  }
}

__device__ __forceinline__ void ring_store4(float* p, const ring_floatx4& v) { *reinterpret_cast<ring_floatx4*>(p) = v; }
__device__ __forceinline__ void ring_store4(bf16_t* p, const ring_floatx4& v) {
  *reinterpret_cast<uint2*>(p) = make_uint2((uint32_t)float_to_bf16_bits(v[0]) | ((uint32_t)float_to_bf16_bits(v[1]) << 16),
                                            (uint32_t)float_to_bf16_bits(v[2]) | ((uint32_t)float_to_bf16_bits(v[3]) << 16));
}

// C[M, N] = A[M, K] W[N, K]^T (+ bias), N a multiple of 4, K of 32.  `splits` parts of K, `k_chunk` (a multiple of 64) each: part s goes to
// slab s of C (float [splits, M, N], ldc = N, no bias).  GATE: W holds `N` gate rows, then N up rows; C[M, N] is the gated result.  Weight
// rows of a gated tile lie in LDS as sixteen gate rows, the sixteen up rows of the same columns, and so on.
// Workgroups in groups of sixteen tiles of rows times all columns, equal runs of that order to the chiplets (every eighth workgroup).
template <class Ring, int BM, int BN, int GATE, typename OutT>
__global__ void __launch_bounds__(Ring::THREADS)
gemm_ring_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, const float* __restrict__ bias, OutT* __restrict__ C,
                 int M, int N, int K, int lda, int ldc, int splits, int k_chunk, float alpha, float limit, float shift) {
  constexpr int GROUP = 16, COLUMNS = GATE ? BN / 2 : BN;
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int tall = (M + BM - 1) / BM, strips = (N + COLUMNS - 1) / COLUMNS, total = tall * strips * splits, per_chiplet = (total + 7) / 8;
  const int turn = (int)(blockIdx.x >> 3), place = (int)(blockIdx.x & 7) * per_chiplet + turn;
  if (turn >= per_chiplet || place >= total) return;
  const int split = place / (tall * strips), at = place - split * tall * strips;
  const int first = at / (GROUP * strips) * GROUP, high = min(GROUP, tall - first), inside = at - first * strips;
  const int m0 = (first + inside % high) * BM, n0 = inside / high * COLUMNS;
  uint32_t a_at[Ring::LA], w_at[Ring::LB];
#pragma unroll
  for (int i = 0; i < Ring::LA; ++i)
    a_at[i] = (uint32_t)min(m0 + Ring::load_row(wave, lane, Ring::LA, i), M - 1) * lda * 2 + Ring::piece_bytes(lane);
#pragma unroll
  for (int i = 0; i < Ring::LB; ++i) {
    const int row = Ring::load_row(wave, lane, Ring::LB, i);
    const int n = GATE ? min(n0 + (row >> 5) * 16 + (row & 15), N - 1) + (row & 16 ? N : 0) : min(n0 + row, N - 1);
    w_at[i] = (uint32_t)n * K * 2 + Ring::piece_bytes(lane);
  }
  const int k_begin = split * k_chunk, k_here = min(K - k_begin, k_chunk);
  ring_floatx4 acc[Ring::MI][Ring::NI];
  Ring::run(A + k_begin, a_at, W + k_begin, w_at, k_here / 64, (k_here & 32) != 0, acc);
  const int r = lane & 15, g = lane >> 4, wm = wave / Ring::ACROSS, wn = wave % Ring::ACROSS;
  C += (size_t)split * M * ldc;
#pragma unroll
  for (int i = 0; i < Ring::MI; ++i) {
    const int m = m0 + wm * Ring::WM + 16 * i + r;
    if (m >= M) continue;
    OutT* row = C + (size_t)m * ldc;
    if constexpr (GATE != RING_PLAIN) {
#pragma unroll
      for (int j = 0; j < Ring::NI; j += 2) {
        const int n = n0 + wn * (Ring::WN / 2) + 8 * j + 4 * g;
        if (n >= N) continue;
        ring_floatx4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = ring_gate<GATE>(acc[i][j][e], acc[i][j + 1][e], alpha, limit, shift);
        ring_store4(row + n, v);
      }
    } else {
#pragma unroll
      for (int j = 0; j < Ring::NI; ++j) {
        const int n = n0 + wn * Ring::WN + 16 * j + 4 * g;
        if (n >= N) continue;
        ring_floatx4 v = acc[i][j];
        if (bias)
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += bias[n + e];
        ring_store4(row + n, v);
      }
    }
  }
}

// The q/k/v projection with bias, rotation and the store of keys and values behind the product: n_q + 2 n_kv heads of d columns (d a multiple
// of 32), q [M, n_q d]; a token's keys and values go to the place slots[m] of their pages (negative: nowhere), as rope_kv.hip lays them out.
// A head's rows lie in LDS as sixteen of its first half, the sixteen as far into its second half, and so on, so that a lane holds both
// coordinates of a turn.  Nothing is rounded before the result (the product used to be).  The angles hang on the positions, which are
// asked for ahead of the product; a block of columns' angles for all of a wave's rows at once, one trip to memory a block.
// (Library product and rotation kernel | this, us: 2,048 rows, 1,152 columns over 896 18.0 | 14.8, 2,048 over 1,536 26.6 | 20.3; 512 rows 10.2 | 7.1,
// 13.6 | 9.2.)
template <class Ring, int BM, int BN>
__global__ void __launch_bounds__(Ring::THREADS)
qkv_ring_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, const float* __restrict__ bias, bf16_t* __restrict__ q,
                const int* __restrict__ positions, const float* __restrict__ cos_sin, const int* __restrict__ slots,
                bf16_t* __restrict__ k_pages, bf16_t* __restrict__ v_pages, int M, int K, int lda, int n_q, int n_kv, int d, int page_size) {
  constexpr int GROUP = 16;
  const int lane = threadIdx.x & 63, wave = wave_index(), N = (n_q + 2 * n_kv) * d;
  const int tall = (M + BM - 1) / BM, strips = (N + BN - 1) / BN, total = tall * strips, per_chiplet = (total + 7) / 8;
  const int turn = (int)(blockIdx.x >> 3), place = (int)(blockIdx.x & 7) * per_chiplet + turn;
  if (turn >= per_chiplet || place >= total) return;
  const int first = place / (GROUP * strips) * GROUP, high = min(GROUP, tall - first), inside = place - first * strips;
  const int m0 = (first + inside % high) * BM, n0 = inside / high * BN;
  const int r = lane & 15, g = lane >> 4, wm = wave / Ring::ACROSS, wn = wave % Ring::ACROSS;
  int position[Ring::MI], slot[Ring::MI];
#pragma unroll
  for (int i = 0; i < Ring::MI; ++i) {
    const int m = min(m0 + wm * Ring::WM + 16 * i + r, M - 1);
    position[i] = positions[m];
    slot[i] = slots ? slots[m] : -1;
  }
  uint32_t a_at[Ring::LA], w_at[Ring::LB];
#pragma unroll
  for (int i = 0; i < Ring::LA; ++i)
    a_at[i] = (uint32_t)min(m0 + Ring::load_row(wave, lane, Ring::LA, i), M - 1) * lda * 2 + Ring::piece_bytes(lane);
#pragma unroll
  for (int i = 0; i < Ring::LB; ++i) {
    const int c = min(n0 + Ring::load_row(wave, lane, Ring::LB, i), N - 1), head = c / d, w = c - head * d;
    w_at[i] = (uint32_t)(head * d + ((w >> 4) & 1) * (d / 2) + (w >> 5) * 16 + (w & 15)) * K * 2 + Ring::piece_bytes(lane);
  }
  ring_floatx4 acc[Ring::MI][Ring::NI];
  Ring::run(A, a_at, W, w_at, K / 64, (K & 32) != 0, acc);
#pragma unroll
  for (int j = 0; j < Ring::NI; j += 2) {
    const int c = n0 + wn * Ring::WN + 16 * j;               // (the same for the wave, and its 32 columns are of one head)
    if (c >= N) continue;
    const int head = c / d, at = (c - head * d) / 2 + 4 * g;
    ring_floatx4 low = {0.f, 0.f, 0.f, 0.f}, high_half = low, cosine[Ring::MI], sine[Ring::MI];
    if (bias) {
      low = *reinterpret_cast<const ring_floatx4*>(bias + head * d + at);
      high_half = *reinterpret_cast<const ring_floatx4*>(bias + head * d + d / 2 + at);
    }
    const bool turned = cos_sin && head < n_q + n_kv;
    if (turned) {
#pragma unroll
      for (int i = 0; i < Ring::MI; ++i) {
        cosine[i] = *reinterpret_cast<const ring_floatx4*>(cos_sin + (size_t)position[i] * d + at);
        sine[i] = *reinterpret_cast<const ring_floatx4*>(cos_sin + (size_t)position[i] * d + d / 2 + at);
      }
    }
#pragma unroll
    for (int i = 0; i < Ring::MI; ++i) {
      const int m = m0 + wm * Ring::WM + 16 * i + r;
      if (m >= M) continue;
      ring_floatx4 x = acc[i][j], y = acc[i][j + 1];
#pragma unroll
      for (int e = 0; e < 4; ++e) { x[e] += low[e]; y[e] += high_half[e]; }
      if (turned) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float u = x[e] * cosine[i][e] - y[e] * sine[i][e], v = y[e] * cosine[i][e] + x[e] * sine[i][e];
          x[e] = u;
          y[e] = v;
        }
      }
      if (head < n_q) {
        bf16_t* to = q + ((size_t)m * n_q + head) * d + at;
        ring_store4(to, x);
        ring_store4(to + d / 2, y);
      } else if (slot[i] >= 0) {
        const int page = slot[i] / page_size, off = slot[i] % page_size;
        if (head < n_q + n_kv) {
          bf16_t* to = k_pages + (((size_t)page * n_kv + (head - n_q)) * page_size + off) * d + at;
          ring_store4(to, x);
          ring_store4(to + d / 2, y);
        } else {
          bf16_t* to = v_pages + (((size_t)page * n_kv + (head - n_q - n_kv)) * d + at) * page_size + off;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            to[(size_t)e * page_size].bits = float_to_bf16_bits(x[e]);
            to[(size_t)(e + d / 2) * page_size].bits = float_to_bf16_bits(y[e]);
          }
        }
      }
    }
  }
}

// The tiles there are, and what a product costs with each, in microseconds on a device of 256 compute units:
//   start + rounds * (fixed + steps * step), rounds of workgroups over the compute units, steps of 64 of K,
// but no less than the weights' trip from memory, and on top the result's (parts are written, and read by whoever adds them: the norm
// that follows, or a kernel of its own).
// Fitted to 5,700 timed products (17 to 4,096 rows, the Qwen2.5 models' matrices at 0.5B, 1.5B and 7B sizes, one to ten parts, plain and
// gated, weights from memory), the price of parts of more than 64 rows to 620 more of 24 matrices of widths of 512 to 5,504: the tile and parts
// with the lowest cost are on average 1.5 % slower than the fastest of all, 20 % at worst.
struct RingShape { int bm, bn; double start, fixed, step; };
static const RingShape RING_SHAPES[] = {
  {64, 64, 2.06, 0.58, 0.232}, {64, 128, 2.37, 0.62, 0.376}, {64, 256, 0.99, 3.08, 0.627}, {128, 128, 0.39, 3.73, 0.513},
  {128, 256, 1.53, 4.57, 0.793}, {256, 128, 1.05, 5.31, 0.757}, {256, 192, 1.97, 4.86, 1.153}, {256, 256, 3.26, 6.01, 1.316}};
enum { RING_SHAPE_COUNT = 8, RING_TAILED = 8, RING_MOST_PARTS = 8 };

struct RingPlan { int shape, parts; double cost; int main_strips; };

// gated: N columns of the result, 2 N weight rows.  pending: parts are left for the caller to add.  least, most: how many parts.
static RingPlan ring_plan(long M, long N, long K, bool gated, bool pending, int least, int most) {
  const int units = compute_units();
  RingPlan best = {gated ? 1 : 0, least, 1e30, 0};
  const double weights = 3.0 + (gated ? 2.0 : 1.0) * N * K * 2 / 5.2e6;
  for (int shape = gated ? 1 : 0; shape < RING_SHAPE_COUNT; ++shape) {
    const RingShape& t = RING_SHAPES[shape];
    if (M <= t.bm / 2 && t.bm > 64) continue;
    const long columns = gated ? t.bn / 2 : t.bn, tiles = (M + t.bm - 1) / t.bm * ((N + columns - 1) / columns);
    for (int s = least; s <= most; ++s) {
      if (s > 1 && least < most && (K / s < 256 || parts_of_k((int)K, s, 64) != s || (double)s * M * N > (1 << 25))) continue;
      const double rounds = (double)((tiles * s + units - 1) / units), steps = (double)((K + s - 1) / s) / 64;
      double cost = t.start + rounds * (t.fixed + steps * t.step);
      // (Where the weights' trip is what counts, the cheaper tile reads the rows less often: 65 rows x 151,936 over 1,536 133 us in 64 x 256
      // tiles, 113 in 128 x 256 ones.  Up to 64 rows of results so wide that the smallest tiles fill the chip twice read them next to never, and what
      // counts is how many workgroups stream: rows of 4 KB and more of 131,072 and 64,000 columns over 2,048, one row 104 and 53.7 us in 64 x 64 tiles,
      // 116 and 56.4 in 64 x 128, 125 and 60.9 in 64 x 256; 32,768 over 4,096 54, 63, 68; shorter ones are level or the other way, 50,256 over
      // 1,600 34.7, 32.3, 31.0; and more than 32 rows are read again often enough: 64 of 152,064 over 3,584 247, 227, 234.)
      const bool streams = M <= 64 && (N + 63) / 64 >= 2 * units && s == 1;
      if (cost >= weights) cost += 0.15 * weights;
      else if (streams) cost = weights * (K >= 2048 && t.bn > (M <= 32 ? 64 : 128) ? 1.02 : 1.0) + 0.05 * cost + (t.bn == 64 && M > 32 ? 0.02 * weights : 0.0);
      else cost = weights + 0.15 * cost;
      if (s == 1) cost += M * N * 2 / 8e6;
      else if (M <= 64) cost += s * (double)M * N / 1e6 + (pending ? 0.0 : 4.0);
      else cost += s * (double)M * N / 0.8e6 + (pending ? 1.0 : 3.0);
      if (cost < best.cost) best = {shape, s, cost, 0};
    }
  }
  // Whole rounds of 256 x 256 (128 x 256) tiles and the columns behind them in 128 x 128 (64 x 128) ones.
  if (gated && least == 1)
    for (int shape = 4; shape <= 7; shape += 3) {
      const RingShape &t = RING_SHAPES[shape], &u = RING_SHAPES[shape == 7 ? 3 : 1];
      const long tall = (M + t.bm - 1) / t.bm, strips = (N + 127) / 128, rounds = tall * strips / units, main = rounds * units / tall;
      if (rounds < 1 || main < 1 || main >= strips) continue;
      const long left = (M + u.bm - 1) / u.bm * ((N - main * 128 + 63) / 64);
      const double steps = (double)K / 64;
      double cost = t.start + rounds * (t.fixed + steps * t.step) + (double)((left + units - 1) / units) * (u.fixed + steps * u.step);
      cost = cost < weights ? weights + 0.15 * cost : cost + 0.15 * weights;
      cost += M * N * 2 / 8e6;
      if (cost < best.cost) best = {RING_TAILED + (shape == 7), 1, cost, (int)main};
    }
  return best;
}

// The gated product where rounds of large tiles would leave the last one mostly empty: `main_strips` strips of columns in the large tiles of
// Main, the columns behind them in the smaller ones of Tail, which the compute units take up as they get through with the large ones.
// Both use the same LDS: Main's stages have A and W in arrays of their own, Tail's lie in those.
// (2,048 rows x 4,864 columns over 896: 256 + 192 tiles in 44.8 us, 408 of 256 x 192 in 50.9, 304 of 256 x 256 in 54.0; 8,960 over 1,536
// 112, 119, 128; 512 rows x 18,944 over 3,584 136, 156 without.)
template <class Tile, int BM, int BN, int GATE, class ASlot, class WSlot>
__device__ __forceinline__ void gated_tile(ASlot a_slot, WSlot w_slot, int m0, int n0, const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                           bf16_t* __restrict__ C, int M, int N, int K, int lda, float alpha, float limit, float shift) {
  const int lane = threadIdx.x & 63, wave = wave_index();
  uint32_t a_at[Tile::LA], w_at[Tile::LB];
#pragma unroll
  for (int i = 0; i < Tile::LA; ++i)
    a_at[i] = (uint32_t)min(m0 + Tile::load_row(wave, lane, Tile::LA, i), M - 1) * lda * 2 + Tile::piece_bytes(lane);
#pragma unroll
  for (int i = 0; i < Tile::LB; ++i) {
    const int row = Tile::load_row(wave, lane, Tile::LB, i);
    w_at[i] = (uint32_t)(min(n0 + (row >> 5) * 16 + (row & 15), N - 1) + (row & 16 ? N : 0)) * K * 2 + Tile::piece_bytes(lane);
  }
  ring_floatx4 acc[Tile::MI][Tile::NI];
  Tile::run_in(a_slot, w_slot, A, a_at, W, w_at, K / 64, (K & 32) != 0, acc);
  const int r = lane & 15, g = lane >> 4, wm = wave / Tile::ACROSS, wn = wave % Tile::ACROSS;
#pragma unroll
  for (int i = 0; i < Tile::MI; ++i) {
    const int m = m0 + wm * Tile::WM + 16 * i + r;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < Tile::NI; j += 2) {
      const int n = n0 + wn * (Tile::WN / 2) + 8 * j + 4 * g;
      if (n >= N) continue;
      ring_floatx4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = ring_gate<GATE>(acc[i][j][e], acc[i][j + 1][e], alpha, limit, shift);
      ring_store4(C + (size_t)m * N + n, v);
    }
  }
}

// WIDE: 256 x 256 (two stages) and 128 x 128 (four); else 128 x 256 and 64 x 128 (three stages both).
template <bool WIDE, int GATE>
__global__ void __launch_bounds__(512)
gemm_ring_tailed_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, bf16_t* __restrict__ C, int M, int N, int K, int lda,
                        int main_strips, int main_blocks, float alpha, float limit, float shift) {
  constexpr int BM = WIDE ? 256 : 128, TM = BM / 2, GROUP = 16;
  __shared__ __attribute__((aligned(1024))) char wide0[32768];
  __shared__ __attribute__((aligned(1024))) char wide1[32768];
  __shared__ __attribute__((aligned(1024))) char wide2[32768];
  __shared__ __attribute__((aligned(1024))) char more0[WIDE ? 32768 : 16384];
  __shared__ __attribute__((aligned(1024))) char more1[WIDE ? 16 : 16384];
  __shared__ __attribute__((aligned(1024))) char more2[WIDE ? 16 : 16384];
  const bool main = (int)blockIdx.x < main_blocks;
  const int columns = main ? 128 : 64, height = main ? BM : TM, block = main ? blockIdx.x : blockIdx.x - main_blocks;
  const int from = main ? 0 : main_strips * 128;
  const int tall = (M + height - 1) / height, strips = main ? main_strips : (N - from + columns - 1) / columns;
  const int total = tall * strips, per_chiplet = (total + 7) / 8, turn = block >> 3, place = (block & 7) * per_chiplet + turn;
  if (turn >= per_chiplet || place >= total) return;
  const int first = place / (GROUP * strips) * GROUP, high = min(GROUP, tall - first), inside = place - first * strips;
  const int m0 = (first + inside % high) * height, n0 = from + inside / high * columns;
  if (main) {
    auto a_slot = [&](auto which) -> ring_lds {
      constexpr int j = decltype(which)::value % (WIDE ? 2 : 3);
      if constexpr (WIDE) { if constexpr (j == 0) return (ring_lds)wide0; else return (ring_lds)wide1; }
      else if constexpr (j == 0) return (ring_lds)more0; else if constexpr (j == 1) return (ring_lds)more1; else return (ring_lds)more2;
    };
    auto w_slot = [&](auto which) -> ring_lds {
      constexpr int j = decltype(which)::value % (WIDE ? 2 : 3);
      if constexpr (WIDE) { if constexpr (j == 0) return (ring_lds)wide2; else return (ring_lds)more0; }
      else if constexpr (j == 0) return (ring_lds)wide0; else if constexpr (j == 1) return (ring_lds)wide1; else return (ring_lds)wide2;
    };
    gated_tile<RingTile<BM, 256, WIDE ? 2 : 3, 2, 4>, BM, 256, GATE>(a_slot, w_slot, m0, n0, A, W, C, M, N, K, lda, alpha, limit, shift);
  } else {
    auto a_slot = [&](auto which) -> ring_lds {
      constexpr int j = decltype(which)::value % (WIDE ? 4 : 3);
      if constexpr (j == 0) return (ring_lds)wide0; else if constexpr (j == 1) return (ring_lds)wide1;
      else if constexpr (j == 2) return (ring_lds)wide2; else return (ring_lds)more0;
    };
    auto w_slot = [&](auto which) -> ring_lds { return a_slot(which) + TM * 128; };
    gated_tile<RingTile<TM, 128, WIDE ? 4 : 3, 2, 4>, TM, 128, GATE>(a_slot, w_slot, m0, n0, A, W, C, M, N, K, lda, alpha, limit, shift);
  }
}

template <int BM, int BN, int STAGES, int WM_WAVES, int WN_WAVES, int GATE, typename OutT>
static int launch_ring(const void* A, const void* W, const void* bias, void* C, int M, int N, int K, int lda, int ldc, int splits,
                       int k_chunk, float alpha, float limit, float shift, hipStream_t stream) {
  typedef RingTile<BM, BN, STAGES, WM_WAVES, WN_WAVES> Ring;
  constexpr int COLUMNS = GATE ? BN / 2 : BN;
  const long tiles = (long)((M + BM - 1) / BM) * ((N + COLUMNS - 1) / COLUMNS) * splits;
  if (tiles > 0x7ffffff0L) return -1;
  gemm_ring_kernel<Ring, BM, BN, GATE, OutT><<<(int)((tiles + 7) / 8 * 8), Ring::THREADS, 0, stream>>>(
      (const bf16_t*)A, (const bf16_t*)W, (const float*)bias, (OutT*)C, M, N, K, lda, ldc, splits, k_chunk, alpha, limit, shift);
  return LAUNCH_STATUS();
}

template <bool WIDE, int GATE>
static int launch_tailed(const void* A, const void* W, void* out, int M, int N, int K, int lda, int main_strips, float alpha, float limit,
                         float shift, hipStream_t stream) {
  const long tall = (M + (WIDE ? 255 : 127)) / (WIDE ? 256 : 128), low = (M + (WIDE ? 127 : 63)) / (WIDE ? 128 : 64);
  const long main = tall * main_strips, left = low * ((N - 128l * main_strips + 63) / 64), main_blocks = (main + 7) / 8 * 8;
  if (main_strips < 0 || 128l * main_strips >= N || main_blocks + left > 0x7ffffff0L) return -1;
  gemm_ring_tailed_kernel<WIDE, GATE><<<(int)(main_blocks + (left + 7) / 8 * 8), 512, 0, stream>>>(
      (const bf16_t*)A, (const bf16_t*)W, (bf16_t*)out, M, N, K, lda, main_strips, (int)main_blocks, alpha, limit, shift);
  return LAUNCH_STATUS();
}

// Whether the kernels of this file take the operands.
static bool ring_takes(const void* A, const void* W, const void* C, int M, long w_rows, int N, int K, int lda, int ldc) {
  return K >= 64 && K % 32 == 0 && N % 4 == 0 && lda % 8 == 0 && ldc % 4 == 0 && (((uintptr_t)A | (uintptr_t)W | (uintptr_t)C) & 15) == 0 &&
         (long)M * lda < (1l << 31) && w_rows * K < (1l << 31);
}

// How `ta_gemm_ring` cuts K: into how many parts.
extern "C" int ta_gemm_ring_parts(int M, int N, int K, int pending) {
  if (M <= 0 || N <= 0 || K < 64) return 1;
  return ring_plan(M, N, K, false, pending != 0, 1, RING_MOST_PARTS).parts;
}

// Whether the gated product of more than 64 rows (N columns of the result) is expected to be faster than the library's product and the
// activation kernel: their multiplications at 1,330 TFLOP/s, part of the weights' trip, the sums' trip to memory and back, and 18 us for what
// two launches cost.  Fitted to 314 products of 65 to 5,000 rows and matrices of 2 to 141 million elements: with the ring kernel wherever this
// says so they take 0.836 of the other way's time (the faster of the two each time: 0.833), 10 of them 3 % more and the worst 11 %; with
// it from 225 rows on, whatever the size, 0.840, 21 and 18 %.  (Us, library and activation | ring: 512 rows, inner 4,864 over 896 23.1 | 18.1;
// 2,048 rows 59 | 45, 8,960 over 1,536 138 | 112, 18,944 over 3,584 557 | 468, 11,008 over 4,096 338 | 301; and the other way 300 rows, 11,008 over
// 4,096 75 | 88, 800 rows 143 | 171, 300 rows, 13,824 over 5,120 104 | 119.)
extern "C" int ta_gemm_ring_gated_pays(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K < 64) return 0;
  const double other = 18.0 + 0.75 * 4e-9 * M * N * K + 0.4 * 4.0 * N * K / 5.2e6 + 1.5e-6 * M * N;
  return ring_plan(M, N, K, true, false, 1, 1).cost <= other;
}

// out[M, N] = act(A Wg^T) * (A Wu^T), W = [Wg; Wu] of 2 N rows.  act: 1 silu, 2 gelu_tanh, 3 relu, 4 the capped gate of (alpha, limit, shift).
// shape: a tile of RING_SHAPES, RING_TAILED for 128 x 256 and 64 x 128, + 1 for 256 x 256 and 128 x 128, or -1 for the cheapest.  -2: not these
// operands.
extern "C" int ta_gemm_ring_gated(const void* A, const void* W, void* out, int M, int N, int K, int lda, int act, float alpha, float limit,
                                  float shift, int shape, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (!ring_takes(A, W, out, M, 2l * N, N, K, lda, N)) return -2;
  int main_strips = 0;
  if (shape < 0) {
    const RingPlan best = ring_plan(M, N, K, true, false, 1, 1);
    shape = best.shape;
    main_strips = best.main_strips;
  } else if (shape >= RING_TAILED) {                        // (asked for: half of the columns in large tiles)
    main_strips = (N + 127) / 256;
  }
#define GO(BM, BN, ST, WMW, WNW, ACT) launch_ring<BM, BN, ST, WMW, WNW, ACT, bf16_t>(A, W, nullptr, out, M, N, K, lda, N, 1, K, alpha, limit, shift, stream)
#define SHAPES(ACT)                                         \
  switch (shape) {                                          \
    case 1: return GO(64, 128, 3, 2, 4, ACT);               \
    case 2: return GO(64, 256, 4, 2, 4, ACT);               \
    case 3: return GO(128, 128, 4, 2, 4, ACT);              \
    case 4: return GO(128, 256, 3, 2, 4, ACT);              \
    case 5: return GO(256, 128, 3, 4, 2, ACT);              \
    case 6: return GO(256, 192, 2, 4, 2, ACT);              \
    case 7: return GO(256, 256, 2, 2, 4, ACT);              \
    case RING_TAILED: return launch_tailed<false, ACT>(A, W, out, M, N, K, lda, main_strips, alpha, limit, shift, stream);      \
    case RING_TAILED + 1: return launch_tailed<true, ACT>(A, W, out, M, N, K, lda, main_strips, alpha, limit, shift, stream);   \
    default: return -1;                                     \
  }
  switch (act) {
    case RING_SILU: SHAPES(RING_SILU)
    case RING_GELU: SHAPES(RING_GELU)
    case RING_RELU: SHAPES(RING_RELU)
    case RING_CAPPED: SHAPES(RING_CAPPED)
    default: return -1;
  }
#undef SHAPES
#undef GO
}

// C[M, N] (rows ldc apart; bfloat16 or float) = A W^T + bias.  parts: what `ta_gemm_ring_parts` said; with more than one `partial` takes
// them, float [parts, M, N], and C may be null: whoever comes next adds them (and the bias).  shape: a tile, or -1 for the cheapest with
// these parts.  -2: not these operands.
extern "C" int ta_gemm_ring(const void* A, const void* W, const void* bias, void* C, void* partial, int M, int N, int K, int lda, int ldc,
                            int parts, int out_dtype, int shape, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (parts < 1 || (parts > 1 && !partial) || (parts == 1 && !C)) return -1;
  if (!ring_takes(A, W, parts > 1 ? partial : C, M, N, N, K, lda, parts > 1 ? N : ldc) || (C && (ldc % 4 || (uintptr_t)C % 16))) return -2;
  if (parts > 1 && parts_of_k(K, parts, 64) != parts) return -1;
  if (shape < 0) shape = ring_plan(M, N, K, false, C == nullptr, parts, parts).shape;
  const int chunk = parts == 1 ? K : ((K + parts - 1) / parts + 63) / 64 * 64;
#define GO(BM, BN, ST, WMW, WNW)                                                                                                         \
  {                                                                                                                                      \
    int status = parts > 1 ? launch_ring<BM, BN, ST, WMW, WNW, 0, float>(A, W, nullptr, partial, M, N, K, lda, N, parts, chunk, 0, 0, 0, stream) \
      : out_dtype == DT_F32 ? launch_ring<BM, BN, ST, WMW, WNW, 0, float>(A, W, bias, C, M, N, K, lda, ldc, 1, chunk, 0, 0, 0, stream)   \
                            : launch_ring<BM, BN, ST, WMW, WNW, 0, bf16_t>(A, W, bias, C, M, N, K, lda, ldc, 1, chunk, 0, 0, 0, stream); \
    if (status == 0 && parts > 1 && C) status = launch_splitk_reduce((const float*)partial, bias, C, M, N, ldc, parts, out_dtype, stream); \
    return status;                                                                                                                       \
  }
  switch (shape) {
    case 0: GO(64, 64, 4, 2, 2)
    case 1: GO(64, 128, 3, 2, 4)
    case 2: GO(64, 256, 4, 2, 4)
    case 3: GO(128, 128, 4, 2, 4)
    case 4: GO(128, 256, 3, 2, 4)
    case 5: GO(256, 128, 3, 4, 2)
    case 6: GO(256, 192, 2, 4, 2)
    case 7: GO(256, 256, 2, 2, 4)
    default: return -1;
  }
#undef GO
}

// The q/k/v projection of many rows with what follows it (see the kernel).  shape: a tile of RING_SHAPES, or -1 for the cheapest.  -2: not
// these operands.
extern "C" int ta_gemm_ring_qkv(const void* A, int lda, const void* W, const void* bias, void* q, const void* positions, const void* cos_sin,
                                const void* slots, void* k_pages, void* v_pages, int M, int K, int n_q, int n_kv, int d, int page_size,
                                int shape, hipStream_t stream) {
  if (M <= 0) return 0;
  if (n_q <= 0 || n_kv < 0 || d <= 0 || page_size <= 0 || !positions || (slots && (!k_pages || !v_pages))) return -1;
  const long N = (long)(n_q + 2 * n_kv) * d;
  if (d % 32 || N > 0x7fffffffL || !ring_takes(A, W, q, M, N, (int)N, K, lda, n_q * d) || (((uintptr_t)bias | (uintptr_t)cos_sin) & 15) ||
      (((uintptr_t)k_pages | (uintptr_t)v_pages) & 7))
    return -2;
  if (shape < 0) shape = ring_plan(M, N, K, false, false, 1, 1).shape;
#define GO(BM, BN, ST, WMW, WNW)                                                                                                          \
  {                                                                                                                                       \
    typedef RingTile<BM, BN, ST, WMW, WNW> Ring;                                                                                          \
    const long tiles = (long)((M + BM - 1) / BM) * ((N + BN - 1) / BN);                                                                   \
    if (tiles > 0x7ffffff0L) return -1;                                                                                                   \
    qkv_ring_kernel<Ring, BM, BN><<<(int)((tiles + 7) / 8 * 8), Ring::THREADS, 0, stream>>>(                                              \
        (const bf16_t*)A, (const bf16_t*)W, (const float*)bias, (bf16_t*)q, (const int*)positions, (const float*)cos_sin,                 \
        (const int*)slots, (bf16_t*)k_pages, (bf16_t*)v_pages, M, K, lda, n_q, n_kv, d, page_size);                                       \
    return LAUNCH_STATUS();                                                                                                               \
  }
  switch (shape) {
    case 0: GO(64, 64, 4, 2, 2)
    case 1: GO(64, 128, 3, 2, 4)
    case 2: GO(64, 256, 4, 2, 4)
    case 3: GO(128, 128, 4, 2, 4)
    case 4: GO(128, 256, 3, 2, 4)
    case 5: GO(256, 128, 3, 4, 2)
    case 6: GO(256, 192, 2, 4, 2)
    case 7: GO(256, 256, 2, 2, 4)
    default: return -1;
  }
#undef GO
}
