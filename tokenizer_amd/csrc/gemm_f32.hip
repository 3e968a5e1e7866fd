// C[M,N] = A[M,K] * W[N,K]^T (+ bias), everything float: the matrix products of the 32-bit path.
//
// The float matrix instructions (v_mfma_f32_32x32x2_f32, v_mfma_f32_16x16x4_f32) multiply 32-bit operands and add to 32-bit
// sums, rounding as a multiply-add does: nothing is narrower than with vector instructions, and a compute unit does 256
// operations a clock where vector multiply-adds do 128.  The kernels:
//   more than 16 rows   tiles through LDS, K cut over workgroups where the tiles alone would leave compute units idle; where pieces of
//                       sixteen bytes are aligned on the bfloat16 instructions, every operand split into three numbers of theirs
//   up to 16 rows       one pass over the weights, sixteen weight rows a workgroup whose waves share K
//   one or two rows (up to four of large wide matrices), and up to 16 whose pieces of sixteen bytes are not aligned    vector
//                       multiply-adds, four weight rows a wave
#include "splitk_reduce.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float silu_f32(float g) { return g / (1.0f + expf(-g)); }

// ---------------------------------------------------------------------------------------------------- many rows
// A workgroup of four waves makes a BM x BN tile, each wave a quarter of it in blocks of 32 x 32.  K goes in steps of 32
// floats: a row of a step is eight pieces of sixteen bytes, which lie in LDS XOR-swizzled by the row, so that the 32 rows a
// fragment read takes at one place of the step fall into all banks.  A lane of the lower half of a wave reads k..k+3 of its
// row, one of the upper half k+4..k+7: the sums run over the same k in both operands, whatever their order, so one sixteen
// byte read feeds four matrix instructions.  The next step's rows are on their way to registers while the current one is
// multiplied; two buffers in LDS, one barrier a step.
// Bound by the matrix cores: 128 x 128 x 32 are 4,096 clocks of them against 32 KB fetched and 64 KB read from LDS.
// blockIdx.x runs over tiles so that the workgroups of one chiplet (every eighth) share strips of weight rows.
// (1,280 rows at 0.5B sizes, vector multiply-adds and this: gate/up, 9,728 columns over 896, 283 us = 79 TFLOP/s and 203 = 110; down,
// 896 columns over 4,864 with K cut, 863 and 135; a layer's four products 1,480 and 415.)
// A tile's place in the launch: false where there is none.
struct F32Tile { int m0, n0, k_begin, k_end; };
template <int BM, int BN>
__device__ __forceinline__ bool f32_tile_place(F32Tile& t, int K, int k_part, int m_tiles, int n_tiles) {
  const int total = m_tiles * n_tiles, per_chiplet = (total + 7) / 8;
  const int tile = (blockIdx.x % 8) * per_chiplet + blockIdx.x / 8;
  if (tile >= total) return false;
  t.m0 = tile % m_tiles * BM;
  t.n0 = tile / m_tiles * BN;
  t.k_begin = blockIdx.y * k_part;
  t.k_end = min(K, t.k_begin + k_part);
  return true;
}

// Four floats of a row (zeros past the rows and past the part of K).
__device__ __forceinline__ f32x4 f32_piece(const float* base, int row, int rows, int stride, int k, int k_end, int vec) {
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if (row < rows) {
    const float* p = base + (size_t)row * stride + k;
    if (vec && k + 3 < k_end) {
      v = *reinterpret_cast<const f32x4*>(p);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (k + i < k_end) v[i] = p[i];
    }
  }
  return v;
}

// The sums of a tile; `lds` holds BUFFERS (BM + BN) rows of 32 floats (with one buffer a step has a barrier more).
template <int BM, int BN, int BUFFERS>
__device__ __forceinline__ void f32_tile_sums(const F32Tile& t, const float* __restrict__ A, const float* __restrict__ W, int M, int N, int K,
                                              int lda, int vec, float (&lds)[BUFFERS * (BM + BN) * 32],
                                              f32x16 (&acc)[BM / 64][BN / 64]) {
  constexpr int TK = 32, QM = BM / 64, QN = BN / 64;       // blocks of 32 x 32 a wave holds each way
  constexpr int PA = BM / 32, PW = BN / 32;                // rows a thread brings of each operand
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int row_in = threadIdx.x >> 3, piece = threadIdx.x & 7;       // 32 rows of eight pieces at a time
  f32x4 a_next[PA], w_next[PW];
  auto fetch = [&](int k0) {
    const int k = k0 + piece * 4;
#pragma unroll
    for (int i = 0; i < PA; ++i) a_next[i] = f32_piece(A, t.m0 + row_in + 32 * i, M, lda, k, t.k_end, vec);
#pragma unroll
    for (int i = 0; i < PW; ++i) w_next[i] = f32_piece(W, t.n0 + row_in + 32 * i, N, K, k, t.k_end, vec);
  };
  auto put = [&](int buffer) {
    const int at = row_in * TK + ((piece ^ (row_in & 7)) << 2);       // (rows 32 apart are swizzled alike)
#pragma unroll
    for (int i = 0; i < PA; ++i) *reinterpret_cast<f32x4*>(&lds[buffer * (BM + BN) * TK + at + 32 * TK * i]) = a_next[i];
#pragma unroll
    for (int i = 0; i < PW; ++i) *reinterpret_cast<f32x4*>(&lds[(buffer * (BM + BN) + BM) * TK + at + 32 * TK * i]) = w_next[i];
  };

#pragma unroll
  for (int i = 0; i < QM; ++i)
#pragma unroll
    for (int j = 0; j < QN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  const int wm = (wave & 1) * (BM / 2), wn = (wave >> 1) * (BN / 2);
  const int r = lane & 31, half = lane >> 5;

  fetch(t.k_begin);
  put(0);
  int buffer = 0;
  for (int k0 = t.k_begin; k0 < t.k_end; k0 += TK, buffer ^= BUFFERS - 1) {
    __syncthreads();
    const bool more = k0 + TK < t.k_end;
    if (more) fetch(k0 + TK);
#pragma unroll
    for (int s = 0; s < TK / 8; ++s) {
      const int at = r * TK + (((2 * s + half) ^ (r & 7)) << 2);
      f32x4 a[QM], w[QN];
#pragma unroll
      for (int i = 0; i < QM; ++i) a[i] = *reinterpret_cast<const f32x4*>(&lds[(buffer * (BM + BN) + wm + 32 * i) * TK + at]);
#pragma unroll
      for (int j = 0; j < QN; ++j) w[j] = *reinterpret_cast<const f32x4*>(&lds[(buffer * (BM + BN) + BM + wn + 32 * j) * TK + at]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < QM; ++i)
#pragma unroll
          for (int j = 0; j < QN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(w[j][e], a[i][e], acc[i][j], 0, 0, 0);
    }
    if (BUFFERS == 1) __syncthreads();
    if (more) put(buffer ^ (BUFFERS - 1));        // (its readers passed the barrier above)
  }
}

// Weight rows are the instruction's rows: element e of a lane is column 8 (e / 4) + 4 half + e % 4 of row r of A.
template <int BM, int BN>
__device__ __forceinline__ void f32_tile_store(const F32Tile& t, const float* __restrict__ bias, float* __restrict__ C, int M, int N, int ldc,
                                               float* __restrict__ partial, const f32x16 (&acc)[BM / 64][BN / 64]) {
  constexpr int QM = BM / 64, QN = BN / 64;
  const int lane = threadIdx.x & 63, wave = wave_index(), r = lane & 31, half = lane >> 5;
  const int wm = (wave & 1) * (BM / 2), wn = (wave >> 1) * (BN / 2), m0 = t.m0, n0 = t.n0;
  float* dst = partial ? partial + (size_t)blockIdx.y * M * N : C;
  const int stride = partial ? N : ldc;
  const bool quads = N % 4 == 0 && stride % 4 == 0 && ((uintptr_t)dst & 15) == 0;
#pragma unroll
  for (int i = 0; i < QM; ++i) {
    const int m = m0 + wm + 32 * i + r;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < QN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = n0 + wn + 32 * j + 8 * q + 4 * half;
        f32x4 v = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
        float* out = dst + (size_t)m * stride + n;
        if (quads && n < N) {
          if (bias && !partial) { v[0] += bias[n]; v[1] += bias[n + 1]; v[2] += bias[n + 2]; v[3] += bias[n + 3]; }
          *reinterpret_cast<f32x4*>(out) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < N) out[e] = v[e] + (bias && !partial ? bias[n + e] : 0.f);
        }
      }
  }
}

template <int BM, int BN>
__global__ void __launch_bounds__(256)
gemm_f32_tile_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                     float* __restrict__ C, int M, int N, int K, int lda, int ldc, int vec, int k_part, int m_tiles,
                     int n_tiles, float* __restrict__ partial) {
  __shared__ __attribute__((aligned(16))) float lds[2 * (BM + BN) * 32];
  F32Tile t;
  if (!f32_tile_place<BM, BN>(t, K, k_part, m_tiles, n_tiles)) return;
  f32x16 acc[BM / 64][BN / 64];
  f32_tile_sums<BM, BN, 2>(t, A, W, M, N, K, lda, vec, lds, acc);
  f32_tile_store<BM, BN>(t, bias, C, M, N, ldc, partial, acc);
}

// The same products on the bfloat16 instructions, sixteen times as fast as the float ones, without losing anything of the operands: a float
// is the sum of three bfloat16 numbers (its nearest one, that of the rest, that of what then is left: 8 + 8 + 8 bits and the signs), and
// of the nine products of two such sums the six largest are summed, smallest first (a1 b3, a3 b1, a2 b2, a1 b2, a2 b1, a1 b1); of the
// three left out a2 b3 and a3 b2 are at most 2^-25 of |a b| each, a3 b3 2^-34.  Products of bfloat16 numbers are exact, the sums are floats, and
// an instruction rounds a sum of sixteen products where the float one rounds after two: against 64 bits the relative error (2-norm) is
// 2.1e-7 to 7.7e-7 over 17 to 2,048 rows and K of 896 to 4,864, 10 to 20 % below the float instructions' at every size measured.
// Operands are split times 2^24 and sums stored times 2^-48: every float, down to the smallest, then is a multiple of 2^-125, so that none of
// the three numbers is too small for a bfloat16 (split as they are, operands below 2^-110 lose their last bits: rows of size 1e-36 were
// off by 2.7e-5, of 1e-38 by 2.7e-3).  The multiplication costs 1 to 3 % (1,280 rows of 9,728 columns over 896 125 -> 128 us, of
// 896 over 4,864 73.5 -> 76.5; 64 rows of 151,936 over 896 156 -> 159); ordinary operands' results are the same bits.
// A sum that is no finite number sends its workgroup back over the tile with the float instructions, whose result takes its place:
// infinities have no rest to split off, and numbers past the largest bfloat16 (times 2^24: from 2^103 on, sums from 2^79) none either.
// The splitting is done once a tile and step, on the way from registers to LDS: three planes of rows of 64 bytes, whose four pieces are
// XOR-swizzled by a quarter of the row (by half of it the reads run at 0.9 of LDS's rate, by the row itself at half).  One buffer: three workgroups share a compute unit, so that one splits while another multiplies.
// AHEAD steps' rows are on their way to registers.  Bound by the matrix cores (1,536 clocks a step of 32 at 128 x 128, six times the work of a
// bfloat16 product: 1,000 to 1,100 TFLOP/s of it) and, beside them, by the splitting's vector instructions (some 700); few tiles by a
// step's chain of load, split, LDS and multiplication, 0.8 us.
// (Float tiles | this, us: 1,280 rows of 9,728 columns over 896 208 | 130, of 896 over 4,864 129 | 80, of 1,152 over 896 37 | 25; 300 rows 69 | 52,
// 45 | 31, 17.6 | 12.5; 64 rows of 151,936 over 896 218 | 155.)
typedef __bf16 split_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 split_bf16x4 __attribute__((ext_vector_type(4)));
template <int BM, int BN, int AHEAD>
__global__ void __launch_bounds__(256, 3)
gemm_f32_split_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                      float* __restrict__ C, int M, int N, int K, int lda, int ldc, int k_part, int m_tiles, int n_tiles,
                      float* __restrict__ partial) {
  constexpr int TK = 32, ROW = 64, QM = BM / 64, QN = BN / 64, PA = BM / 32, PW = BN / 32, PLANE = (BM + BN) * ROW;
  // (The planes; a buffer of float rows, where it comes to that.)
  __shared__ __attribute__((aligned(16))) union { char planes[3 * PLANE]; float rows[(BM + BN) * 32]; } lds;
  F32Tile t;
  if (!f32_tile_place<BM, BN>(t, K, k_part, m_tiles, n_tiles)) return;
  const int lane = threadIdx.x & 63, wave = wave_index(), r = lane & 31, half = lane >> 5;
  const int wm = (wave & 1) * (BM / 2), wn = (wave >> 1) * (BN / 2);
  const int row_in = threadIdx.x >> 3, piece = threadIdx.x & 7;
  // Rows past the last read the last one (their results are not stored); pieces past the end of K read the part's first and are put
  // down as zeros.  So every load is made, and the compiler can count them.
  uint32_t a_at[PA], w_at[PW];
#pragma unroll
  for (int i = 0; i < PA; ++i) a_at[i] = ((uint32_t)min(t.m0 + row_in + 32 * i, M - 1) * lda + piece * 4) * 4;
#pragma unroll
  for (int i = 0; i < PW; ++i) w_at[i] = ((uint32_t)min(t.n0 + row_in + 32 * i, N - 1) * K + piece * 4) * 4;
  f32x4 a_next[AHEAD][PA], w_next[AHEAD][PW];
  typedef const char __attribute__((address_space(1)))* memory;
  typedef const f32x4 __attribute__((address_space(1)))* pieces;
  const int k_last = t.k_begin + (t.k_end - t.k_begin - 1) / TK * TK;
  auto fetch = [&](int k_asked, f32x4 (&a_now)[PA], f32x4 (&w_now)[PW]) {
    const int k0 = min(k_asked, k_last);                    // (past the end the last step again)
    const uint32_t back = k0 + piece * 4 < t.k_end ? 0 : piece * 16;
    memory a_base = (memory)(uintptr_t)(A + k0), w_base = (memory)(uintptr_t)(W + k0);
    asm("" : "+s"(a_base), "+s"(w_base));
#pragma unroll
    for (int i = 0; i < PA; ++i) {
      uint32_t at = a_at[i] - back;
      asm("" : "+v"(at));
      a_now[i] = *(pieces)(a_base + at);
    }
#pragma unroll
    for (int i = 0; i < PW; ++i) {
      uint32_t at = w_at[i] - back;
      asm("" : "+v"(at));
      w_now[i] = *(pieces)(w_base + at);
    }
  };
  const int put_at = row_in * ROW + (((piece >> 1) ^ ((row_in >> 2) & 3)) << 4) + (piece & 1) * 8;   // (rows 32 apart are swizzled alike)
  auto put = [&](const f32x4& v, int at) {
    f32x4 rest;
#pragma unroll
    for (int e = 0; e < 4; ++e) rest[e] = v[e] * 0x1p24f;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      split_bf16x4 near;
#pragma unroll
      for (int e = 0; e < 4; ++e) near[e] = (__bf16)rest[e];
      *reinterpret_cast<split_bf16x4*>(lds.planes + p * PLANE + at) = near;
#pragma unroll
      for (int e = 0; e < 4; ++e) rest[e] -= (float)near[e];
    }
  };
  f32x16 acc[QM][QN];
#pragma unroll
  for (int i = 0; i < QM; ++i)
#pragma unroll
    for (int j = 0; j < QN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  auto one = [&](int k0, f32x4 (&a_now)[PA], f32x4 (&w_now)[PW]) {
    if (k0 + piece * 4 >= t.k_end) {
#pragma unroll
      for (int i = 0; i < PA; ++i) a_now[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < PW; ++i) w_now[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    __syncthreads();                                        // (the step before has been read)
#pragma unroll
    for (int i = 0; i < PA; ++i) put(a_now[i], put_at + 32 * ROW * i);
#pragma unroll
    for (int i = 0; i < PW; ++i) put(w_now[i], BM * ROW + put_at + 32 * ROW * i);
    __syncthreads();
    fetch(k0 + AHEAD * TK, a_now, w_now);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int at = r * ROW + (((2 * s + half) ^ ((r >> 2) & 3)) << 4);
      split_bf16x8 a[3][QM], w[3][QN];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
#pragma unroll
        for (int i = 0; i < QM; ++i) a[p][i] = *reinterpret_cast<const split_bf16x8*>(lds.planes + p * PLANE + (wm + 32 * i) * ROW + at);
#pragma unroll
        for (int j = 0; j < QN; ++j) w[p][j] = *reinterpret_cast<const split_bf16x8*>(lds.planes + p * PLANE + (BM + wn + 32 * j) * ROW + at);
      }
      constexpr int OF_A[6] = {0, 2, 1, 0, 1, 0}, OF_W[6] = {2, 0, 1, 1, 0, 0};
#pragma unroll
      for (int p = 0; p < 6; ++p)
#pragma unroll
        for (int i = 0; i < QM; ++i)
#pragma unroll
          for (int j = 0; j < QN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[OF_W[p]][j], a[OF_A[p]][i], acc[i][j], 0, 0, 0);
    }
  };
#pragma unroll
  for (int j = 0; j < AHEAD; ++j) fetch(t.k_begin + j * TK, a_next[j], w_next[j]);
  for (int k0 = t.k_begin; k0 < t.k_end; k0 += AHEAD * TK) {
#pragma unroll
    for (int j = 0; j < AHEAD; ++j)
      if (k0 + j * TK < t.k_end) one(k0 + j * TK, a_next[j], w_next[j]);
  }
  // Only the sums that are no finite numbers are replaced, so that a row's result does not hang on what other rows of its tile hold
  // (rows that only fill a batch up may hold anything).
  uint64_t odd = 0;
#pragma unroll
  for (int i = 0; i < QM; ++i)
#pragma unroll
    for (int j = 0; j < QN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        if (!(fabsf(acc[i][j][e]) < INFINITY)) odd |= 1ull << ((i * QN + j) * 16 + e);
        acc[i][j][e] *= 0x1p-48f;
      }
  f32_tile_store<BM, BN>(t, bias, C, M, N, ldc, partial, acc);
  if (!__syncthreads_or(odd != 0)) return;
  f32_tile_sums<BM, BN, 1>(t, A, W, M, N, K, lda, 1, lds.rows, acc);
  float* dst = partial ? partial + (size_t)blockIdx.y * M * N : C;
  const int stride = partial ? N : ldc;
#pragma unroll
  for (int i = 0; i < QM; ++i)
#pragma unroll
    for (int j = 0; j < QN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = t.m0 + wm + 32 * i + r, n = t.n0 + wn + 32 * j + 8 * (e >> 2) + 4 * half + (e & 3);
        if ((odd >> ((i * QN + j) * 16 + e) & 1) && m < M && n < N)
          dst[(size_t)m * stride + n] = acc[i][j][e] + (bias && !partial ? bias[n] : 0.f);
      }
}

// ----------------------------------------------------------------------------------------------------- few rows
// Up to sixteen rows: sixteen weight rows a workgroup (GATED: eight rows of the first half of W and the eight as far into
// its second half, whose results meet in silu(first) * second), eight waves that take units of 32 floats of K in turn.
// Lane (row, g) reads the sixteen bytes g and g + 4 of a weight row's 128 byte line and the same of row `row` of A; the
// matrix instruction's sum runs over the four g.  Four sums a lane (one for each float of a piece) keep the chains of
// additions short; they and the eight waves' come together through LDS.  Bound by the weights' trip from memory: a wave
// asks for its first two pairs of units at once and for the next pair before it multiplies the current one.
// (Half lines through the caches | whole lines past them, four rows: 896 columns over 4,864 in eight parts of K 8.7 | 7.1 us, over 896 in two
// 5.6 | 4.4, 1,536 over 8,960 34 | 26; sixteen rows: gate/up of 17,920 over 1,536 45 | 30, of 37,888 over 3,584 182 | 128.  Weights that are in
// the last-level cache already, all of a model in less than its 256 MB, four rows and sixteen: 768 columns over 3,072 12.0 | 10.5 and 14.3 | 13.3.)
// LINES (K a multiple of 32): the weights come by whole cache lines, eight rows' a load (`lines_to_rows` in common.h), past the caches.
// ROPE: the product is the joined q/k/v projection; a tile is eight elements of the first half of a head and the eight half a head further
// on, which the half-split rotation pairs; bias, rotation and the store of keys and values into their pages follow in the epilogue.
struct F32Store {
  const int* positions; const float* cos_sin; const int* slots;
  float* k_pages; float* v_pages;
  int n_q, n_kv, d, page_size;
};

// PLAIN and ROPE take fewer rows a workgroup (`tile_rows` in all: down to four; of each half with ROPE: down to two) where sixteen (eight) are
// fewer workgroups than compute units.  Rows of the sixteen past them repeat the last one (lanes that read by lines load nothing for
// them): a matrix's places are all that is read, and what is made of them feeds sums that nobody reads.
// STAGE > 0 (LINES, up to four rows for one and up to eight for two): a wave brings a pair of units of A's rows in STAGE loads of sixteen
// different bytes a lane and turns them into fragments through a part of LDS of its own; a fragment straight from memory is a load
// that holds up the memory pipeline like any other though its lanes mostly ask for the same bytes.
// (Before all of this, a pair that is not there multiplied as zeros and positions fetched where they are used | so, us, weights from memory,
// four rows and eight: q/k/v of 896 with rotation 5.7 | 4.9 and 5.9 | 5.3, 896 over 896 in two parts 4.4 | 3.5 and 4.5 | 3.6, 896 over 4,864 in eight
// 7.4 | 6.3 and 7.7 | 7.0.)
enum { ROWS_PLAIN = 0, ROWS_GATED = 1, ROWS_ROPE = 2 };

// Where workgroup `block`'s weight rows lie in a matrix of n: row i (0 .. 15) of its tile, with two halves row i & 7 of the first or (i >= 8) of the second.
template <int KIND>
struct RowTile {
  int head, first_in, n0, half, limit, rows;                // (head, first_in: ROPE, the head and the tile's place in its first half)
  __host__ __device__ RowTile(int block, int n, int tile_rows, int d) : rows(tile_rows) {
    const int per_head = KIND == ROWS_ROPE ? d / 2 / rows : 1;
    head = KIND == ROWS_ROPE ? block / per_head : 0;
    first_in = KIND == ROWS_ROPE ? block % per_head * rows : 0;
    half = KIND == ROWS_ROPE ? d / 2 : n / 2;
    n0 = KIND == ROWS_ROPE ? head * d + first_in : block * rows;
    limit = KIND == ROWS_GATED ? half : n;
  }
  __host__ __device__ int place(int i) const { return KIND == ROWS_PLAIN ? i : i & 7; }
  __host__ __device__ bool there(int i) const { return place(i) < rows; }
  __host__ __device__ int row(int i) const {
    const int at = n0 + (there(i) ? place(i) : rows - 1);
    return (at < limit ? at : limit - 1) + (KIND != ROWS_PLAIN && i >= 8 ? half : 0);
  }
};

// The row of the matrix that row i of a workgroup's tile is read from (`kind`: the enumeration above), as the kernel below has it; -1 for what is no tile.
extern "C" int ta_gemm_f32_tile_row(int kind, int block, int n, int tile_rows, int d, int i) {
  if (n <= 0 || tile_rows <= 0 || tile_rows > 16 || i < 0 || i > 15 || block < 0 || (kind == ROWS_ROPE && d / 2 < tile_rows)) return -1;
  return kind == ROWS_ROPE ? RowTile<ROWS_ROPE>(block, n, tile_rows, d).row(i)
         : kind == ROWS_GATED ? RowTile<ROWS_GATED>(block, n, tile_rows, d).row(i) : RowTile<ROWS_PLAIN>(block, n, tile_rows, d).row(i);
}

// FULL: the tile has all of its rows (always with GATED), so that no load of weights stands behind a question of its lane's (151,936 columns over 896,
// sixteen rows 129 -> 126 us).
template <int KIND, bool LINES, int STAGE, bool FULL>
__global__ void __launch_bounds__(512)
gemm_f32_rows_kernel(const float* __restrict__ A, const float* __restrict__ W, uint32_t m_rows_d, int N, int K, int lda, int units_part,
                     const float* __restrict__ bias, float* __restrict__ partial, float* __restrict__ C, int ldc,
                     const F32Store store = F32Store()) {
  HELD(A, W, m_rows_d, N, K, lda, units_part, bias, partial);                // (the words that are there when a wave starts)
  constexpr int WAVES = 8, PAIR = 2, ROW_BYTES = PAIR * 128 + 16;
  static_assert(STAGE == 0 || LINES, "rows are staged line by line");
  __shared__ float sums[WAVES][16][17];
  __shared__ __attribute__((aligned(16))) char rows_s[STAGE > 0 ? WAVES * 4 * STAGE * ROW_BYTES : 16];
  const int M = m_rows_d & 0xff, tile_rows = (m_rows_d >> 8) & 0xff, d = m_rows_d >> 16;    // (d: ROPE)
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int row = lane & 15, g = lane >> 4;
  const RowTile<KIND> tile(blockIdx.x, N, tile_rows, d);
  const int head = tile.head, first_in = tile.first_in, half = tile.half, n0 = tile.n0;
  const int units = (K + 31) / 32;
  const int u_begin = blockIdx.y * units_part, u_end = min(units, u_begin + units_part);
  const int a_m = min(row, M - 1);
  const float* a_row = A + (size_t)a_m * lda;
  const float* w_row[2];
  bool w_ok[2];
  w_row[0] = W + (size_t)tile.row(LINES ? row & 7 : row) * K;
  w_row[1] = LINES ? W + (size_t)tile.row(8 + (row & 7)) * K : w_row[0];
  w_ok[0] = tile.there(LINES ? row & 7 : row);
  w_ok[1] = LINES ? tile.there(8 + (row & 7)) : w_ok[0];
  const int piece = 2 * g + (row >> 3);
  char* mine = rows_s + (STAGE > 0 ? wave * M * ROW_BYTES : 0);
  f32x4 w[2][PAIR][2], a[2][PAIR][2], staged[2][STAGE > 0 ? STAGE : 1];
  auto ask = [&](int slot, int u0) {
#pragma unroll
    for (int p = 0; p < PAIR; ++p) {
      const int u = u0 + p * WAVES;
      if constexpr (LINES) {
#pragma unroll
        for (int h = 0; h < 2; ++h) w[slot][p][h] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (STAGE == 0) a[slot][p][0] = a[slot][p][1] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (u < u_end) {                                     // (the same for the whole wave)
#pragma unroll
          for (int h = 0; h < 2; ++h)
            if (FULL || w_ok[h]) w[slot][p][h] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(w_row[h] + u * 32 + 4 * piece));
          if constexpr (STAGE == 0) {
#pragma unroll
            for (int h = 0; h < 2; ++h) a[slot][p][h] = *reinterpret_cast<const f32x4*>(a_row + u * 32 + 8 * g + 4 * h);
          }
        }
      } else {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          // (K is a multiple of four: a piece is inside a row or past its end, where the row's first piece is read and
          // multiplied by zeros.)
          const int k = u * 32 + 16 * h + 4 * g;
          const bool in = u < u_end && k < K;
          w[slot][p][h] = *reinterpret_cast<const f32x4*>(w_row[0] + (in ? k : 0));
          a[slot][p][h] = *reinterpret_cast<const f32x4*>(a_row + (in ? k : 0));
        }
      }
    }
    if (STAGE > 0 && u0 < u_end) {
      // Piece i of the pair's M * 16 is piece i % 16 of row i / 16; a unit past the end is the last one again, put down as zeros.
#pragma unroll
      for (int j = 0; j < STAGE; ++j) {
        const int i = min(j * WAVE + lane, M * 16 - 1), u = min(u0 + ((i & 15) >> 3) * WAVES, u_end - 1);
        staged[slot][j] = *reinterpret_cast<const f32x4*>(A + (size_t)(i >> 4) * lda + u * 32 + 4 * (i & 7));
      }
    }
  };
  f32x4 acc[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int first = u_begin + wave;
  ask(0, first);
  // What the epilogue needs is asked for behind the first weights, positions and slots through the scalar unit.
  const int m = threadIdx.x >> 4, at = threadIdx.x & 15;    // its thread: row m, weight row `at`; wave v has rows 4 v .. 4 v + 3
  float cosine = 1.f, sine = 0.f, bias1 = 0.f, bias2 = 0.f;
  int slot_of = -1;
  if (4 * wave < M) {
    HELD(C, ldc, store.positions, store.cos_sin, store.slots, store.k_pages, store.v_pages, store.n_q, store.n_kv, store.page_size);
    if constexpr (KIND == ROWS_ROPE) {
      const bool turned = head < store.n_q + store.n_kv && store.cos_sin;
      int position = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int of = min(4 * wave + j, M - 1);
        const int p = turned ? scalar_int(store.positions + of) : 0, s = store.slots ? scalar_int(store.slots + of) : -1;
        position = (lane >> 4) == j ? p : position;
        slot_of = (lane >> 4) == j ? s : slot_of;
      }
      if (m < M && at < tile_rows) {
        if (turned) {
          const float* cs = store.cos_sin + (size_t)position * d + first_in + at;
          cosine = cs[0];
          sine = cs[half];
        }
        if (bias) { bias1 = bias[n0 + at]; bias2 = bias[n0 + half + at]; }
      }
    } else if (KIND == ROWS_PLAIN && bias && !partial && m < M) {
      bias1 = bias[min(n0 + at, N - 1)];
    }
  }
  for (int u0 = first; u0 < u_end; u0 += 2 * PAIR * WAVES) {
#pragma unroll
    for (int slot = 0; slot < 2; ++slot) {
      const int now = u0 + slot * PAIR * WAVES;
      if (now >= u_end) break;                               // (the same for the whole wave)
      if (LINES || now + PAIR * WAVES < u_end) ask(slot ^ 1, now + PAIR * WAVES);
      if constexpr (STAGE > 0) {
#pragma unroll
        for (int j = 0; j < STAGE; ++j) {
          const int i = min(j * WAVE + lane, M * 16 - 1);
          if (now + ((i & 15) >> 3) * WAVES >= u_end) staged[slot][j] = f32x4{0.f, 0.f, 0.f, 0.f};
          *reinterpret_cast<f32x4*>(mine + (i >> 4) * ROW_BYTES + (i & 15) * 16) = staged[slot][j];
        }
        wave_exchange();
#pragma unroll
        for (int p = 0; p < PAIR; ++p)
#pragma unroll
          for (int h = 0; h < 2; ++h) a[slot][p][h] = *reinterpret_cast<const f32x4*>(mine + a_m * ROW_BYTES + p * 128 + 32 * g + 16 * h);
        wave_exchange();                                     // (the next pair's pieces are stored behind these reads)
      }
#pragma unroll
      for (int p = 0; p < PAIR; ++p) {
        if constexpr (LINES) {
          // (Units past the end are zeros in both operands.)
          line_bf16x8 b[2];
          lines_to_rows(__builtin_bit_cast(word4, w[slot][p][0]), __builtin_bit_cast(word4, w[slot][p][1]), row < 8, b[0], b[1]);
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const f32x4 wv = __builtin_bit_cast(f32x4, b[h]);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[e], a[slot][p][h][e], acc[e], 0, 0, 0);
          }
        } else {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int u = now + p * WAVES;
            const bool in = u < u_end && u * 32 + 16 * h + 4 * g < K;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              // (Both operands: the first piece of a row may hold an infinity, whose product with zero is no number.)
              const float wv = in ? w[slot][p][h][e] : 0.f, av = in ? a[slot][p][h][e] : 0.f;
              acc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv, av, acc[e], 0, 0, 0);
            }
          }
        }
      }
    }
  }
  // A lane holds weight rows 4 g .. 4 g + 3 of A's row `row`.
#pragma unroll
  for (int j = 0; j < 4; ++j) sums[wave][row][4 * g + j] = (acc[0][j] + acc[1][j]) + (acc[2][j] + acc[3][j]);
  __syncthreads();
  if (m >= M || at >= tile_rows) return;                   // (threads from the sixteenth row on leave here too)
  auto total = [&](int place) {
    float t = 0.f;
#pragma unroll
    for (int v = 0; v < WAVES; ++v) t += sums[v][m][place];
    return t;
  };
  if constexpr (KIND == ROWS_ROPE) {
    const float x1 = total(at) + bias1, x2 = total(at + 8) + bias2;
    const float v1 = x1 * cosine - x2 * sine, v2 = x2 * cosine + x1 * sine;     // cosine 1 and sine 0 where nothing turns
    const int i = first_in + at;
    if (head < store.n_q) {
      float* dst = C + (size_t)m * ldc + (size_t)head * d + i;
      st(dst, v1);
      st(dst + half, v2);
      return;
    }
    if (slot_of < 0) return;                                // this row's keys and values are not stored
    const int page = slot_of / store.page_size, off = slot_of % store.page_size;
    if (head < store.n_q + store.n_kv) {
      float* dst = store.k_pages + (((size_t)page * store.n_kv + (head - store.n_q)) * store.page_size + off) * d + i;
      st(dst, v1);
      st(dst + half, v2);
    } else {
      float* dst = store.v_pages + (((size_t)page * store.n_kv + (head - store.n_q - store.n_kv)) * d + i) * store.page_size + off;
      st(dst, v1);
      st(dst + (size_t)half * store.page_size, v2);
    }
  } else if (KIND == ROWS_GATED) {
    if (n0 + at < half) st(C + (size_t)m * ldc + n0 + at, silu_f32(total(at)) * total(at + 8));
  } else if (n0 + at < N) {
    if (partial) st(partial + ((size_t)blockIdx.y * M + m) * N + n0 + at, total(at));
    else st(C + (size_t)m * ldc + n0 + at, total(at) + bias1);
  }
}

// Launches the kernel above: `rows` weight rows a workgroup (of each half with GATED and ROPE), `d` the head size (ROPE).
template <int KIND>
static void launch_f32_rows(dim3 grid, const float* a, const float* w, const float* bias, float* c, int M, int N, int K, int lda, int ldc,
                            int units_part, float* partial, int rows, int d, const F32Store& store, hipStream_t stream) {
  const uint32_t packed = (uint32_t)M | (uint32_t)rows << 8 | (uint32_t)d << 16;
#define GO_FORM(LINES, STAGE, FULL) gemm_f32_rows_kernel<KIND, LINES, STAGE, FULL><<<grid, 512, 0, stream>>>(a, w, packed, N, K, lda, units_part, \
                                                                                                           bias, partial, c, ldc, store)
#define GO(LINES, STAGE) do { if (KIND == ROWS_GATED || rows == (KIND == ROWS_PLAIN ? 16 : 8)) GO_FORM(LINES, STAGE, true); \
                              else GO_FORM(LINES, STAGE, KIND == ROWS_GATED); } while (0)
  if (K % 32) GO_FORM(false, 0, false);
  else if (M <= 4) GO(true, 1);
  else if (M <= 8) GO(true, 2);
  else GO(true, 0);
#undef GO
#undef GO_FORM
}

// One or two rows, four of large matrices, and up to sixteen whose pieces of sixteen bytes do not lie on sixteen bytes (VEC false):
// a wave takes four weight rows (GATED: two of W's first half and the two as far into its second, whose results meet in
// silu(first) * second) and walks K sixteen bytes or an element a lane, every row of A against them.  With so little work for a
// weight the matrix instructions gain nothing, and this way more of the weights are on their way at once (figures at `vector_rows`).
// UN: pieces of 256 floats a wave asks for at once (past the caches).  Four where the workgroups are no more than the compute units, one
// where they are more, which hide each other's trips (one row, one piece | four: 896 columns over 896 4.7 | 4.1, over 4,864 14.3 | 12.5,
// 3,584 over 18,944 55.3 | 51.3, but 4,608 over 3,584 13.5 | 16.7, 151,936 over 896, three rows 84 | 98).  Past the caches, one row from memory
// and from the last-level cache, us through them | past them: 768 columns over 3,072 9.7 | 8.3 and 6.9 | 8.0, over 768 4.0 | 3.4 and 3.3 | 3.4, 896
// over 4,864 14.2 | 12.3 and 9.7 | 11.7: a model in less than the cache's 256 MB loses, which the kernel cannot know, and every other gains.
// ROWS (VEC): the rows of A are brought into LDS once for the workgroup's four waves, which otherwise ask for all of them each.  The sums over
// a wave are taken eight at a time, each where one lane stores it, the gate with it.  (Gate/up 4,864 over 896, four rows, each wave for itself
// and one lane with all gates | so: 10.1 | 8.9 us, two rows 8.4 | 8.2; 35 MB of weights are 5.7.)
template <int MR, bool VEC, bool GATED, int UN = 1, bool ROWS = false>
__global__ void __launch_bounds__(256)
gemv_f32_kernel(const float* __restrict__ A, const float* __restrict__ W, int M, int N, int K, int lda, const float* __restrict__ bias,
                float* __restrict__ C, int ldc) {
  HELD(A, W, M, N, K, lda, bias, C, ldc);
  extern __shared__ __attribute__((aligned(16))) float rows_s[];
  const int lane = threadIdx.x & 63, wave = wave_index(), half = N / 2;
  const int n0 = (blockIdx.x * 4 + wave) * (GATED ? 2 : 4);  // this wave's weight rows
  if (!ROWS && n0 >= (GATED ? half : N)) return;
  // Which of eight sums ends in this lane (see `wave_sums8`), and the bias of its weight row.
  const int s8 = (lane & 1) + 2 * ((lane >> 4) & 1) + 4 * (lane >> 5);
  float bias_here = 0.f;
  if (!GATED && bias) bias_here = bias[min(n0 + (s8 & 3), N - 1)];
  float acc[4][MR];
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int m = 0; m < MR; ++m) acc[r][m] = 0.f;
  const float* w[4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
    w[r] = W + (size_t)(GATED ? (r < 2 ? 0 : half) + min(n0 + (r & 1), half - 1) : min(n0 + r, N - 1)) * K;
  if constexpr (ROWS) {
    for (int i = threadIdx.x * 4; i < M * K; i += 256 * 4) {
      const int m = i / K;
      *reinterpret_cast<f32x4*>(rows_s + i) = *reinterpret_cast<const f32x4*>(A + (size_t)m * lda + (i - m * K));
    }
    __syncthreads();
    if (n0 >= (GATED ? half : N)) return;
  }
  if constexpr (VEC) {
    for (int k0 = lane * 4; k0 < K; k0 += UN * WAVE * 4) {
      f32x4 wv[UN][4];
#pragma unroll
      for (int u = 0; u < UN; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          wv[u][r] = f32x4{0.f, 0.f, 0.f, 0.f};
          if (k0 + u * WAVE * 4 < K) wv[u][r] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(w[r] + k0 + u * WAVE * 4));
        }
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const int k = k0 + u * WAVE * 4;
        if (k >= K) break;
#pragma unroll
        for (int m = 0; m < MR; ++m) {
          if (m >= M) break;
          const float4 a = *reinterpret_cast<const float4*>(ROWS ? rows_s + m * K + k : A + (size_t)m * lda + k);
#pragma unroll
          for (int r = 0; r < 4; ++r)
            acc[r][m] = fmaf(a.x, wv[u][r][0], fmaf(a.y, wv[u][r][1], fmaf(a.z, wv[u][r][2], fmaf(a.w, wv[u][r][3], acc[r][m]))));
        }
      }
    }
  } else {
    for (int k = lane; k < K; k += WAVE) {
      float wv[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) wv[r] = w[r][k];
#pragma unroll
      for (int m = 0; m < MR; ++m) {
        if (m >= M) break;
        const float a = A[(size_t)m * lda + k];
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r][m] = fmaf(a, wv[r], acc[r][m]);
      }
    }
  }
  // Sum i of eight: PLAIN weight row i % 4 of row i / 4, GATED weight row i % 2 of row i / 2 of both halves.
  constexpr int ROWS_IN_8 = GATED ? 4 : 2;
#pragma unroll
  for (int m0 = 0; m0 < MR; m0 += ROWS_IN_8) {
    if (m0 >= M) break;
    float v[8], up[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int m = m0 + i / (8 / ROWS_IN_8), r = i % (8 / ROWS_IN_8);
      v[i] = m < MR ? acc[r][m < MR ? m : 0] : 0.f;
      if (GATED) up[i] = m < MR ? acc[r + 2][m < MR ? m : 0] : 0.f;
    }
    const float total = wave_sums8(v, lane), second = GATED ? wave_sums8(up, lane) : 0.f;
    const int m = m0 + s8 / (8 / ROWS_IN_8), n = n0 + s8 % (8 / ROWS_IN_8);
    if ((lane & 15) > 1 || m >= M) continue;
    if constexpr (GATED) {
      if (n < half) st(C + (size_t)m * ldc + n, silu_f32(total) * second);
    } else if (n < N) {
      st(C + (size_t)m * ldc + n, total + bias_here);
    }
  }
}

// (Rows without elements have no piece that could be read: they go to the kernels that walk K an element at a time.)
static bool sixteen_bytes(const void* A, const void* W, int M, int K, int lda) {
  return K > 0 && K % 4 == 0 && (M <= 1 || lda % 4 == 0) && (((uintptr_t)A | (uintptr_t)W) & 15) == 0;
}

// Whether up to sixteen aligned rows go to the vector kernel.  K of whole lines, us, matrix instructions | vector: one row of 896 columns
// over 896 5.1 | 4.1, over 4,864 14.5 | 12.5, 9,728 over 896 11.1 | 8.2, 3,584 over 18,944 50.2 | 51.3; two of 896 over 896 5.1 | 4.9, of
// 1,536 over 8,960 24.8 | 24.6, of 3,584 over 18,944 51.1 | 55.4, of 9,728 over 896 11.0 | 8.7; four of 9,728 over 896 11.3 | 10.8, of 17,920
// over 1,536 25.0 | 21.8, of 4,608 over 3,584 22 | 18, of 3,584 over 3,584 13.3 | 16.5; eight of 3,584 over 18,944 57 | 88.  With K cut for the
// next norm, one row of 896 over 896 4.3 | 4.1, two 4.3 | 4.9, two of 3,584 over 18,944 51.9 | 55.5.
// Other K: two rows of 1,536 columns over 8,960 34.0 | 21.7, four of 17,920 over 1,536 33.7 | 24.4, eight of 3,584 over 18,944
// 96.9 | 92.0, of 1,536 over 8,960 36.6 | 38.9.
static bool vector_rows(int M, int N, int K, bool pending) {
  if (pending && N % 4 == 0 && K >= 4096 && N <= 2048) return false;
  const bool large = (long)N * K >= (8l << 20), many = (N + 15) / 16 > compute_units();
  if (K % 32 == 0) {
    if (M == 1) return true;
    if (pending && N % 4 == 0 && !many) return false;
    return M == 2 ? !large || many : M <= 4 && large && many;
  }
  return M <= 2 || (M <= 4 && (K >= 4096 || large)) || (M <= 8 && K >= 16384 && !pending);
}

// The split kernel's microseconds for tiles of 64 and 128: start, a workgroup's fixed ones, and those of a step of 32 with one, two and three
// workgroups on a compute unit (each step 16 or 32 KB from memory, and no less than the weights' trip).  Fitted to 1,070 timed products (17
// to 3,000 rows, matrices of the 0.5B and 1.5B models, one to eight parts); the choice is on average 1 % slower than the fastest, 17 % at worst.
static const double SPLIT_64[] = {6.46, -2.10, 0.797, 1.048, 1.382}, SPLIT_128[] = {7.22, -1.00, 1.632, 2.475, 3.672};

// Which kernel and into how many parts of K (at most 8): `tile` 16 (few rows), 64 or 128, 0 (vector
// multiply-adds).  Few rows: a power of two, until there are workgroups for every compute unit, each of eight units of 32 at least, and only
// where the next kernel adds them (`pending`): a reduction of its own costs as much as it saves.  Many rows: the estimate above where the
// pieces are aligned; else rounds of workgroups over the compute units, a round as long as its tile's multiplications at what the
// two float tiles reach (128 x 128: 110 to 121 of the 157 TFLOP/s there are; 64 x 64: 99 to 102 in one part, 90 in two, counted as 88); plus
// the parts' trip to memory and, where nobody else adds them, a further launch.
static void f32_choice(int M, int N, int K, bool aligned, bool pending, int* tile, int* parts) {
  const int units = compute_units();
  *tile = 0;
  *parts = 1;
  if (M <= 16) {
    if (!aligned || vector_rows(M, N, K, pending)) return;
    *tile = 16;
    if (pending && N % 4 == 0)
      while (*parts < 8 && (N + 15) / 16 * *parts < units && K / 32 / (2 * *parts) >= 8) *parts *= 2;
    return;
  }
  double best = 1e30;
  if (aligned) {
    for (int t = 64; t <= 128; t *= 2)
      for (int p = 1; p <= 8; ++p) {
        if (p > 1 && (N % 4 || K / p < 128 || parts_of_k(K, p, 32) != p)) continue;
        const long tiles = (long)((M + t - 1) / t) * ((N + t - 1) / t) * p, load = (tiles + units - 1) / units;
        const double steps = (double)(((K + p - 1) / p + 31) / 32), *c = t == 64 ? SPLIT_64 : SPLIT_128;
        double cost = c[0] + (double)(load / 3) * (c[1] + steps * c[4]) + (load % 3 ? c[1] + steps * c[1 + load % 3] : 0.0);
        const double weights = 3.0 + (double)N * K * 4 / 5.2e6;
        if (cost < weights) cost = weights;
        cost += p == 1 ? (double)M * N * 4 / 8e6 : (double)M * N * 4 * p / 4e6 + (pending ? 0.0 : 4.0);
        if (cost < best) { best = cost; *tile = t; *parts = p; }
      }
    return;
  }
  for (int t = 64; t <= 128; t *= 2)
    for (int p = 1; p <= 8; p *= 2) {
      if (p > 1 && (N % 4 || K / p < 128)) continue;
      const double tiles = (double)((M + t - 1) / t) * ((N + t - 1) / t) * p;
      const double flops = 2.0 * t * t * ((K + p - 1) / p), rate = (t == 128 ? 110e6 : 88e6) / units;   // a unit's, per us
      const double rounds = tiles <= units ? 1.0 : (double)(long)((tiles + units - 1) / units);
      double cost = rounds * flops / rate + 3.0;
      if (p > 1) cost += (double)M * N * 4 * p * 2 / 4e6 + (pending ? 0.0 : 4.0);
      if (cost < best) { best = cost; *tile = t; *parts = p; }
    }
}

// The parts of K a product is cut into where `pending` says that whoever takes it adds them; 1: it is not.
extern "C" int ta_gemm_f32_parts(const void* A, const void* W, int M, int N, int K, int lda, int pending) {
  if (M <= 0 || N <= 0 || K <= 0) return 1;
  int tile, parts;
  f32_choice(M, N, K, sixteen_bytes(A, W, M, K, lda), pending != 0, &tile, &parts);
  return parts_of_k(K, parts, 32);
}

// partial: float [ta_gemm_f32_parts][M][N] where that is more than 1, else null.  C null: the parts are left there.
extern "C" int ta_gemm_f32(const void* A, const void* W, const void* bias, void* C, int M, int N, int K,
                           int lda, int ldc, void* partial, int pending, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  const bool aligned = sixteen_bytes(A, W, M, K, lda);
  int tile = 0, parts = 1;
  f32_choice(M, N, K, aligned, pending != 0, &tile, &parts);
  parts = parts_of_k(K, parts, 32);
  if ((parts > 1) != (partial != nullptr) || (!C && parts == 1)) return -1;
  const float *a = (const float*)A, *w = (const float*)W, *b = (const float*)bias;
  float *c = (float*)C, *slabs = (float*)partial;
  const int k_part = parts > 1 ? ((K + parts - 1) / parts + 31) / 32 * 32 : K;
  if (tile == 16) {
    const int units = compute_units(), even = (int)(((long)N * parts + units - 1) / units), rows = even < 4 ? 4 : even > 16 ? 16 : even;
    launch_f32_rows<ROWS_PLAIN>(dim3((N + rows - 1) / rows, parts), a, w, b, c, M, N, K, lda, ldc, (k_part + 31) / 32, slabs, rows, 0,
                                F32Store(), stream);
  } else if (tile) {
    const int m_tiles = (M + tile - 1) / tile, n_tiles = (N + tile - 1) / tile;
    dim3 grid((m_tiles * n_tiles + 7) / 8 * 8, parts);
    const bool split = aligned && (long)M * lda < (1l << 30) && (long)N * K < (1l << 30);      // (32-bit places)
    if (split && tile == 128)
      gemm_f32_split_kernel<128, 128, 2><<<grid, 256, 0, stream>>>(a, w, b, c, M, N, K, lda, ldc, k_part, m_tiles, n_tiles, slabs);
    else if (split)
      gemm_f32_split_kernel<64, 64, 3><<<grid, 256, 0, stream>>>(a, w, b, c, M, N, K, lda, ldc, k_part, m_tiles, n_tiles, slabs);
    else if (tile == 128)
      gemm_f32_tile_kernel<128, 128><<<grid, 256, 0, stream>>>(a, w, b, c, M, N, K, lda, ldc, aligned, k_part, m_tiles,
                                                               n_tiles, slabs);
    else
      gemm_f32_tile_kernel<64, 64><<<grid, 256, 0, stream>>>(a, w, b, c, M, N, K, lda, ldc, aligned, k_part, m_tiles,
                                                             n_tiles, slabs);
  } else {
    const int blocks = (N + 15) / 16;
#define GO(MR, VEC, ...) gemv_f32_kernel<MR, VEC, false, ##__VA_ARGS__><<<blocks, 256, 0, stream>>>(a, w, M, N, K, lda, b, c, ldc)
    if (aligned && blocks <= compute_units()) { if (M <= 1) GO(1, true, 4); else if (M <= 2) GO(2, true, 4); else if (M <= 4) GO(4, true, 4); else GO(8, true, 2); }
    else if (aligned) { if (M <= 1) GO(1, true); else if (M <= 2) GO(2, true); else if (M <= 4) GO(4, true); else GO(8, true); }
    else if (M <= 1) GO(1, false); else if (M <= 2) GO(2, false); else if (M <= 4) GO(4, false);
    else if (M <= 8) GO(8, false); else GO(16, false);
#undef GO
  }
  int status = LAUNCH_STATUS();
  if (status == 0 && parts > 1 && C) status = launch_splitk_reduce(slabs, bias, C, M, N, ldc, parts, DT_F32, stream);
  return status;
}

// out[M, N/2] = silu(A W1^T) * (A W2^T), W = [W1; W2], for up to sixteen rows; -2 where the pieces are not aligned or K is 0 (the caller
// then runs the product and the gate one after the other).
extern "C" int ta_gemm_f32_silu_gate(const void* A, const void* W, void* out, int M, int N, int K, int lda, int ldc,
                                     hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (N % 2) return -1;
  if (M > 16 || !sixteen_bytes(A, W, M, K, lda)) return -2;
  const float *a = (const float*)A, *w = (const float*)W;
  const int blocks = (N / 2 + 7) / 8;
  const size_t rows_bytes = (size_t)M * K * sizeof(float);
  const bool rows_fit = M > 1 && rows_bytes <= 20 * 1024;    // (eight workgroups a compute unit)
#define GO(MR) do { if (blocks <= compute_units()) gemv_f32_kernel<MR, true, true, 4><<<blocks, 256, 0, stream>>>(a, w, M, N, K, lda, nullptr, (float*)out, ldc); \
                    else if (rows_fit) gemv_f32_kernel<MR, true, true, 1, true><<<blocks, 256, rows_bytes, stream>>>(a, w, M, N, K, lda, nullptr, (float*)out, ldc); \
                    else gemv_f32_kernel<MR, true, true><<<blocks, 256, 0, stream>>>(a, w, M, N, K, lda, nullptr, (float*)out, ldc); } while (0)
  if (!vector_rows(M, N, K, false)) {
    launch_f32_rows<ROWS_GATED>(dim3(blocks), a, w, nullptr, (float*)out, M, N, K, lda, ldc, (K + 31) / 32, nullptr, 8, 0, F32Store(), stream);
  } else if (M <= 1) GO(1); else if (M <= 2) GO(2); else if (M <= 4) GO(4); else GO(8);
#undef GO
  return LAUNCH_STATUS();
}

// The joined q/k/v projection of up to sixteen rows with bias, rotation and the cache write in its epilogue (see F32Store): x [M, K] (row
// stride lda), W [(n_q + 2 n_kv) d, K], d a multiple of 16, bias or null; queries go to q_out [M, n_q d]; cos_sin [positions, d] or null (no
// rotation); slots int32 [M] or null (nothing is stored; a negative slot skips its row).  -2: rows without pieces of sixteen bytes.
extern "C" int ta_gemm_f32_qkv_rope(const void* x, int lda, const void* W, const void* bias, void* q_out, const void* positions,
                                    const void* cos_sin, const void* slots, void* k_pages, void* v_pages, int M, int K, int n_q,
                                    int n_kv, int d, int page_size, hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > 16 || d <= 0 || d % 16 || n_q <= 0 || n_kv <= 0 || page_size <= 0 || !positions || (slots && (!k_pages || !v_pages))) return -1;
  if (!sixteen_bytes(x, W, M, K, lda)) return -2;
  const F32Store store = {(const int*)positions, (const float*)cos_sin, (const int*)slots, (float*)k_pages, (float*)v_pages,
                          n_q, n_kv, d, page_size};
  const int heads = n_q + 2 * n_kv;
  if (d > 0xffff) return -1;                                 // (what the kernel's packed arguments hold)
  int rows = 8;                                              // of each half (d / 2 is a multiple of eight)
  while (rows > 2 && heads * (d / 2 / rows) * 2 <= compute_units()) rows /= 2;
  launch_f32_rows<ROWS_ROPE>(dim3(heads * (d / 2 / rows)), (const float*)x, (const float*)W, (const float*)bias, (float*)q_out, M, heads * d, K, lda,
                             n_q * d, (K + 31) / 32, nullptr, rows, d, store, stream);
  return LAUNCH_STATUS();
}
