// C[M,N] = A[M,K] * W[N,K]^T (+ bias) for few rows (M <= 64): the decode-time product, bound by the
// one pass over the weights.  Computed transposed on the matrix cores, C^T = W A^T: sixteen weight rows are
// the M side of a 16x16x32 MFMA, up to four blocks of sixteen activation rows the N side, so every weight
// element is loaded once, 16 bytes per lane.  The waves of a workgroup split K between them and add up
// through LDS.  With GATED the kernel computes silu(A Wg^T) * (A Wu^T) for W = [Wg; Wu] in one pass.
#include "common.h"
#include "splitk_reduce.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf16x8 load8(const bf16_t* p, bool ok) {
  bf16x8 z;
  if (ok) return *reinterpret_cast<const bf16x8*>(p);
#pragma unroll
  for (int i = 0; i < 8; ++i) z[i] = (__bf16)0.0f;
  return z;
}

__device__ __forceinline__ void store4(float* p, const float* v) {
  *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ void store4(bf16_t* p, const float* v) {
  uint2 packed;
  packed.x = (uint32_t)float_to_bf16_bits(v[0]) | ((uint32_t)float_to_bf16_bits(v[1]) << 16);
  packed.y = (uint32_t)float_to_bf16_bits(v[2]) | ((uint32_t)float_to_bf16_bits(v[3]) << 16);
  *reinterpret_cast<uint2*>(p) = packed;
}
__device__ __forceinline__ void store1(float* p, float v) { *p = v; }
__device__ __forceinline__ void store1(bf16_t* p, float v) { p->bits = float_to_bf16_bits(v); }

// grid.x: tiles of 16 output columns (of N, or of N/2 with GATED).  NW waves per workgroup.
// grid.y: parts of K of `k_chunk` elements (a multiple of 32; one part with LINES) each: with more than one, a workgroup writes the
// float sums of its part into its slab of `partial` [parts, M, N] and `splitk_reduce` finishes the product.  That is
// for few output tiles and a long K (the down projection of a decode batch): every compute unit gets a share.
//
// ROPE (with GATED's two sets of weight rows): the product is the joined q/k/v projection.  A tile is sixteen
// elements of the first half of a head and the sixteen half a head further on, which the half-split rotation
// pairs; the epilogue adds the bias, rotates query and key heads by the row's position and writes queries to
// C [M, n_q * d], keys and values into their pages (values transposed inside a page).
struct RopeStore {
  const int* positions; const float* cos_sin; const int* slots;
  bf16_t* k_pages; bf16_t* v_pages;
  int n_q, n_kv, d, page_size;
};

// NB: blocks of sixteen output columns per workgroup.  Every workgroup reads all the rows of A for its part of K;
// with two blocks the rows are read half as often, which is what a product of many rows is bound by once the
// rows outweigh a tile's weights (what comes over the fabric from the caches counts like what comes from memory).
// LINES > 0: the weights are read line by line (`lines_to_rows` in common.h), K walked in steps of 64, LINES steps at a time, past the
// caches (a stream that does not come again): for products that are one long stream over a big matrix.  WHOLE: K is a multiple of 64.
template <int MB, int NW, bool GATED, typename OutT, bool ROPE = false, int NB = 1, int LINES = 0, bool WHOLE = false>
__global__ void __launch_bounds__(NW * WAVE)
skinny_gemm_kernel(const bf16_t* __restrict__ A, int lda, int k_chunk, const bf16_t* __restrict__ W,
                   OutT* __restrict__ C, int ldc, int M, int N, int K_all, float* __restrict__ partial,
                   const float* __restrict__ bias, const RopeStore rope = RopeStore(), int gate_act = 0) {
  // (What the walk over K needs stands in the first fourteen words of the arguments, which are in scalar registers
  // when a wave starts; the bias and the rotation's arguments, which the epilogue needs, lie behind.)
  HELD(A, lda, k_chunk, W, C, ldc, M, N, K_all, partial);
  static_assert(!ROPE || GATED, "the rotation uses the two sets of weight rows");
  static_assert(!ROPE || NB == 1, "the rotation pairs rows within one block");
  constexpr int HALVES = GATED ? 2 : 1;                     // gate and up rows (or the two halves of a head)
  constexpr int SETS = HALVES * NB;                         // set h * NB + b: half h, column block b
  __shared__ float red[NW][HALVES * MB * 4][WAVE];
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int col = lane & 15, g = lane >> 4;
  const int n_out = ROPE ? N : GATED ? N / 2 : N;
  // ROPE: tile t is block t % (d/32) of sixteen elements in the first half of head t / (d/32).
  const int rope_half = ROPE ? rope.d / 2 : 0;
  const int rope_head = ROPE ? blockIdx.x / (rope_half / 16) : 0;
  const int rope_first = ROPE ? (blockIdx.x % (rope_half / 16)) * 16 : 0;      // first element of the tile in its head
  const int n_first = ROPE ? rope_head * rope.d + rope_first : blockIdx.x * 16 * NB;
  const int k_lo = blockIdx.y * k_chunk;
  const int K = min(K_all, k_lo + k_chunk) - k_lo;                // this workgroup's part of K
  // grid.z: the rows in shares of MB blocks of sixteen (one share unless the launcher cut them: a small matrix
  // whose tiles would not fill the device otherwise; the weights are then read once per share).
  const int m_base = blockIdx.z * (MB * 16);
  // Rows past the end are clamped, not masked: they only feed outputs that are never stored.
  // The second half: the `up` rows when GATED, the rows half a head further on with ROPE.
  const bf16_t* wp[SETS];
#pragma unroll
  for (int h = 0; h < HALVES; ++h)
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int wrow = min(n_first + 16 * b + col, n_out - 1) + h * (ROPE ? rope_half : n_out);
      wp[h * NB + b] = W + (size_t)wrow * K_all + k_lo + 8 * g;
    }
  // Lanes of activation rows past M load nothing and hold zeros: a load costs the memory pipeline by its
  // active lanes, and with few rows most of a block's lanes are such.
  const bf16_t* a_row[MB];
  bool a_ok[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    a_ok[mb] = m_base + mb * 16 + col < M;
    a_row[mb] = A + (size_t)min(m_base + mb * 16 + col, M - 1) * lda + k_lo + 8 * g;
  }

  floatx4 acc[SETS][MB];
#pragma unroll
  for (int s = 0; s < SETS; ++s)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[s][mb] = (floatx4){0.f, 0.f, 0.f, 0.f};

  constexpr int UN = (SETS * MB > 4) ? 2 : 4;
  if constexpr (LINES > 0) {
    const int sub = col & 7, piece = 2 * g + (col >> 3);
    const bool low_lane = col < 8;
    const bf16_t* wl[SETS][2];
#pragma unroll
    for (int h = 0; h < HALVES; ++h)
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          const int wrow = min(n_first + 16 * b + 8 * hh + sub, n_out - 1) + h * (ROPE ? rope_half : n_out);
          wl[h * NB + b][hh] = W + (size_t)wrow * K_all + k_lo + 8 * piece;
        }
    const int pairs = (K + 63) / 64;                        // lines of a row; the last may be short
    constexpr int UP = LINES;
    for (int first = wave; first < pairs; first += UP * NW) {
      word4 wf[UP][SETS][2];
      bf16x8 af[UP][MB][2];
#pragma unroll
      for (int q = 0; q < UP; ++q) {
        const int pair = first + q * NW;
        const bool valid = pair < pairs;
        const int at = min(pair, pairs - 1) * 64;
        const bool mine = valid && (WHOLE || at + 8 * piece < K);        // this lane's sixteen bytes lie inside K
#pragma unroll
        for (int s = 0; s < SETS; ++s)
#pragma unroll
          for (int hh = 0; hh < 2; ++hh) {
            wf[q][s][hh] = (word4){0u, 0u, 0u, 0u};
            if (mine) wf[q][s][hh] = __builtin_nontemporal_load(reinterpret_cast<const word4*>(wl[s][hh] + at));
          }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int hh = 0; hh < 2; ++hh) {         // (`a_row` is 8 g on already)
            const int place = at + 16 * g + hh * 8;
            af[q][mb][hh] = load8(a_row[mb] + place - 8 * g, valid && a_ok[mb] && (WHOLE || place < K));
          }
      }
#pragma unroll
      for (int q = 0; q < UP; ++q) {
#pragma unroll
        for (int s = 0; s < SETS; ++s) {
          bf16x8 b0, b1;
          lines_to_rows(wf[q][s][0], wf[q][s][1], low_lane, b0, b1);
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) {
            acc[s][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b0, af[q][mb][0], acc[s][mb], 0, 0, 0);
            acc[s][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b1, af[q][mb][1], acc[s][mb], 0, 0, 0);
          }
        }
      }
    }
  } else {
  const int full_steps = K / 32;
  // UN steps at a time, all loads first, so that many are in flight per lane.  A wave's last batch may reach
  // past the end of K: such steps load nothing and multiply zeros (no matrix instruction sits behind a
  // condition), so that a wave's share of K is as few trips to memory as can be, never one trip per step.
  for (int ks = wave; ks < full_steps; ks += UN * NW) {
    bf16x8 wf[UN][SETS], af[UN][MB];
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const int step = ks + u * NW;
      const bool valid = step < full_steps;
      const int k = min(step, full_steps - 1) * 32;
#pragma unroll
      for (int s = 0; s < SETS; ++s) wf[u][s] = load8(wp[s] + k, valid);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) af[u][mb] = load8(a_row[mb] + k, valid && a_ok[mb]);
    }
#pragma unroll
    for (int u = 0; u < UN; ++u)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int s = 0; s < SETS; ++s)
          acc[s][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u][s], af[u][mb], acc[s][mb], 0, 0, 0);
  }
  if (K & 31) {
    // The tail of K (a multiple of 8), zero-filled, is one wave's; the others multiply zeros, so that no matrix
    // instruction sits behind a condition on the wave (it would run whatever a lane mask says).
    const int k = full_steps * 32;
    const bool k_ok = wave == full_steps % NW && k + 8 * g < K;
    bf16x8 wt[SETS];
#pragma unroll
    for (int s = 0; s < SETS; ++s) wt[s] = load8(wp[s] + k, k_ok);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const bf16x8 af = load8(a_row[mb] + k, k_ok && a_ok[mb]);
#pragma unroll
      for (int s = 0; s < SETS; ++s) acc[s][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wt[s], af, acc[s][mb], 0, 0, 0);
    }
  }
  }
  // One column block at a time through LDS (both halves of it), so that more blocks need no more LDS.
#pragma unroll
  for (int b = 0; b < NB; ++b) {
  const int n0 = n_first + 16 * b;
  if (b > 0) __syncthreads();                                   // the block before has been read
#pragma unroll
  for (int h = 0; h < HALVES; ++h)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wave][(h * MB + mb) * 4 + r][lane] = acc[h * NB + b][mb][r];
  __syncthreads();
  // Lane (col, g) of block mb holds C^T rows n0 + 4g + r (r = 0..3), column m = mb*16 + col.
  for (int item = threadIdx.x; item < MB * WAVE; item += NW * WAVE) {
    const int mb = item / WAVE, ln = item % WAVE;
    const int m = m_base + mb * 16 + (ln & 15);
    const int n = n0 + 4 * (ln >> 4);
    if (m >= M || n >= n_out) continue;
    float v[4], v2[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float sum0 = 0.f, sum1 = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        sum0 += red[w][mb * 4 + r][ln];
        if (GATED) sum1 += red[w][(MB + mb) * 4 + r][ln];
      }
      if (ROPE) {
        v[r] = sum0 + (bias ? bias[n + r] : 0.f);
        v2[r] = sum1 + (bias ? bias[n + rope_half + r] : 0.f);
        continue;
      }
      if (bias && !partial && n + r < n_out) sum0 += bias[n + r];
      // gate_act 1: the tanh form of GELU in place of silu; 2: max(z, 0).
      v[r] = !GATED ? sum0
             : gate_act == 2 ? fmaxf(sum0, 0.f) * sum1
             : gate_act == 1 ? 0.5f * sum0 * (1.0f + tanhf(0.7978845608028654f * (sum0 + 0.044715f * sum0 * sum0 * sum0))) * sum1
                             : sum0 / (1.0f + __expf(-sum0)) * sum1;
    }
    if constexpr (ROPE) {
      const int d = rope.d, i = rope_first + 4 * (ln >> 4);          // elements i..i+3 of the head, and i + half
      if (rope_head < rope.n_q + rope.n_kv && rope.cos_sin) {
        const float* cs = rope.cos_sin + (size_t)rope.positions[m] * d;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float c = cs[i + r], sn = cs[rope_half + i + r], x1 = v[r], x2 = v2[r];
          v[r] = x1 * c - x2 * sn;
          v2[r] = x2 * c + x1 * sn;
        }
      }
      if (rope_head < rope.n_q) {
        bf16_t* dst = reinterpret_cast<bf16_t*>(C) + (size_t)m * ldc + (size_t)rope_head * d + i;
        store4(dst, v);
        store4(dst + rope_half, v2);
        continue;
      }
      const int slot = rope.slots ? rope.slots[m] : -1;
      if (slot < 0) continue;                                     // this row's keys and values are not stored
      const int page = slot / rope.page_size, off = slot % rope.page_size;
      if (rope_head < rope.n_q + rope.n_kv) {
        bf16_t* dst = rope.k_pages + (((size_t)page * rope.n_kv + (rope_head - rope.n_q)) * rope.page_size + off) * d + i;
        store4(dst, v);
        store4(dst + rope_half, v2);
      } else {
        bf16_t* dst = rope.v_pages + (((size_t)page * rope.n_kv + (rope_head - rope.n_q - rope.n_kv)) * d + i) * rope.page_size + off;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          store1(dst + (size_t)r * rope.page_size, v[r]);
          store1(dst + (size_t)(rope_half + r) * rope.page_size, v2[r]);
        }
      }
      continue;
    }
    if (partial) {                                              // (never GATED; N is a multiple of 4)
      store4(partial + ((size_t)blockIdx.y * M + m) * n_out + n, v);
      continue;
    }
    OutT* dst = C + (size_t)m * ldc + n;
    if (n + 3 < n_out && (ldc & 3) == 0) {
      store4(dst, v);
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n + r < n_out) store1(dst + r, v[r]);
    }
  }
  }
}

// Up to sixteen rows: the same product with what a launch of that size is bound by taken out.
// * A workgroup has R <= 16 weight rows, so that a small matrix is spread over all compute units (896 columns are 224 workgroups of
//   four, not 56 of sixteen); lanes whose weight row is past R load nothing and only feed results that are never stored.  UPPER: R > 8 (LINES).
// * The epilogue is the tail that the launch waits for: a lane has one output, which it adds up in the waves' order; wave v < ceil(M / 4)
//   takes rows 4 v .. 4 v + 3, sixteen lanes the block's weight rows.  The bias is on its way beside the first weights.
// * STAGE > 0 (up to eight rows): a wave brings a trip's share of the rows in STAGE loads of sixteen different bytes a lane and turns
//   them into fragments through a part of LDS that is its own; a fragment straight from memory is a load that holds up the memory
//   pipeline like any other though its lanes mostly ask for the same bytes.
// SUMS 2 (with whole lines): a wave keeps the sums of two waves of half lines, a line's first 32 elements of K and its second, so that a
// product has the same bits whichever way its weights come.
// Which wave takes which steps of K does not hang on any of this, nor does a result.
// Us, weights from memory, sixteen rows a workgroup with four outputs a lane | so, one row, eight and sixteen: 896 over 896 3.5 | 3.0, 3.9 | 3.2
// and 4.15 | 3.6; 896 over 4,864 8.1 | 5.7, 9.7 | 5.8 and 11.2 | 8.3; 1,536 over 1,536 4.5 | 3.6, 5.1 | 3.8 and 5.6 | 4.6; 1,536 over 8,960 12.6 | 9.3,
// 15.5 | 9.4 and 18.3 | 14.2; 3,584 over 3,584 7.2 | 6.8, 8.5 | 7.5 and 9.4 | 8.7; 3,584 over 18,944 24.6 | 23.0, 30.1 | 25.0 and 35.7 | 33.8; gate/up
// 4,864 over 896 7.3 | 6.4, 7.7 | 7.0 and 8.1 | 7.25, 8,960 over 1,536 14.9 | 12.7, 15.9 | 13.9 and 17.3 | 15.6.  (A kernel that does nothing: 1.65.)
template <int NW, bool GATED, typename OutT, int LINES, bool WHOLE, int SUMS, bool UPPER, int STAGE>
__global__ void __launch_bounds__(NW * WAVE)
few_rows_gemm_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, const float* __restrict__ bias,
                     float* __restrict__ partial, int lda, int k_chunk, uint32_t m_rows_act, int N, int K_all, int ldc,
                     OutT* __restrict__ C) {
  HELD(A, W, bias, partial, lda, k_chunk, m_rows_act, N, K_all, ldc);    // (the fourteen words that are there)
  static_assert(SUMS == 1 || (SUMS == 2 && LINES > 0 && WHOLE), "two sums a wave: whole lines, a sum for each half");
  constexpr int SETS = GATED ? 2 : 1, TRIP = LINES > 0 ? LINES : 4;      // lines, or steps of 32, a trip
  constexpr int PIECES = TRIP * (LINES > 0 ? 8 : 4), ROW_BYTES = PIECES * 16 + 16;
  __shared__ float red[NW * SUMS][SETS * 4][WAVE];
  extern __shared__ __attribute__((aligned(16))) char rows_s[];
  const int M = m_rows_act & 0xff, R = (m_rows_act >> 8) & 0xff, gate_act = m_rows_act >> 16;
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int col = lane & 15, g = lane >> 4;
  const int n_out = GATED ? N / 2 : N;
  const int n_first = blockIdx.x * R;
  const int k_lo = blockIdx.y * k_chunk;
  const int K = min(K_all, k_lo + k_chunk) - k_lo;                // this workgroup's part of K
  const bool a_ok = col < M;
  const int a_m = min(col, M - 1);
  const bf16_t* a_row = A + (size_t)a_m * lda + k_lo;
  // The lane of the epilogue: weight row `er` of the block, row `em` (and, with two waves, the row eight further on).
  const int er = lane & 15, em = 4 * wave + (lane >> 4), n = n_first + er;
  const bool e_wave = 4 * wave < M;
  float bias_here;
  asm volatile("" : "=v"(bias_here));                             // (whatever it holds: only read where it was loaded)
  const bool biased = bias && !partial;
  if (e_wave && biased) bias_here = bias[min(n, n_out - 1)];
  // STAGE: piece i of the M * PIECES of a trip is piece i % PIECES of row i / PIECES.
  char* mine = rows_s + (STAGE > 0 ? (size_t)wave * M * ROW_BYTES : 0);
  word4 staged[STAGE > 0 ? STAGE : 1];
  int stage_k[STAGE > 0 ? STAGE : 1];
  auto stage_ask = [&](int first) {                               // `first`: the wave's first line, or step, of the trip
#pragma unroll
    for (int j = 0; j < STAGE; ++j) {
      const int i = min(j * WAVE + lane, M * PIECES - 1), piece = i % PIECES;
      stage_k[j] = LINES > 0 ? (first + (piece >> 3) * NW) * 64 + 8 * (piece & 7) : (first + (piece >> 2) * NW) * 32 + 8 * (piece & 3);
      staged[j] = *reinterpret_cast<const word4*>(A + (size_t)(i / PIECES) * lda + k_lo + min(stage_k[j], K - 8));
    }
  };
  auto stage_put = [&]() {                                        // (past the end of K: zeros)
#pragma unroll
    for (int j = 0; j < STAGE; ++j) {
      const int i = min(j * WAVE + lane, M * PIECES - 1);
      if (stage_k[j] >= K) staged[j] = (word4){0u, 0u, 0u, 0u};
      *reinterpret_cast<word4*>(mine + i / PIECES * ROW_BYTES + i % PIECES * 16) = staged[j];
    }
    wave_exchange();
  };
  auto fragment = [&](int byte) { return __builtin_bit_cast(bf16x8, *reinterpret_cast<const word4*>(mine + a_m * ROW_BYTES + byte)); };

  floatx4 sums[SUMS][SETS];
#pragma unroll
  for (int i = 0; i < SUMS; ++i)
#pragma unroll
    for (int s = 0; s < SETS; ++s) sums[i][s] = (floatx4){0.f, 0.f, 0.f, 0.f};

  if constexpr (LINES > 0) {
    constexpr int HH = UPPER ? 2 : 1;
    const int sub = col & 7, piece = SUMS == 2 ? g + 4 * (col >> 3) : 2 * g + (col >> 3);
    const int a_first = SUMS == 2 ? 8 * g : 16 * g, a_apart = SUMS == 2 ? 32 : 8;    // the rows' elements of the line that meet the weights'
    const bf16_t* wl[SETS][HH];
    bool w_ok[HH];
#pragma unroll
    for (int hh = 0; hh < HH; ++hh) {
      w_ok[hh] = 8 * hh + sub < R && n_first + 8 * hh + sub < n_out;
#pragma unroll
      for (int s = 0; s < SETS; ++s)
        wl[s][hh] = W + (size_t)(min(n_first + 8 * hh + sub, n_out - 1) + s * n_out) * K_all + k_lo + 8 * piece;
    }
    const int pairs = (K + 63) / 64;                        // lines of a row; the last may be short
    for (int first = wave; first < pairs; first += LINES * NW) {
      word4 wf[LINES][SETS][HH];
      bf16x8 af[LINES][2];
#pragma unroll
      for (int q = 0; q < LINES; ++q) {
        const int pair = first + q * NW;
        const bool valid = pair < pairs;
        const int at = min(pair, pairs - 1) * 64;
        const bool inside = valid && (WHOLE || at + 8 * piece < K);      // this lane's sixteen bytes lie inside K
#pragma unroll
        for (int s = 0; s < SETS; ++s)
#pragma unroll
          for (int hh = 0; hh < HH; ++hh) {
            wf[q][s][hh] = (word4){0u, 0u, 0u, 0u};
            if (inside && w_ok[hh]) wf[q][s][hh] = __builtin_nontemporal_load(reinterpret_cast<const word4*>(wl[s][hh] + at));
          }
        if constexpr (STAGE == 0) {
#pragma unroll
          for (int hh = 0; hh < 2; ++hh) {
            const int place = at + a_first + hh * a_apart;
            af[q][hh] = load8(a_row + place, valid && a_ok && (WHOLE || place < K));
          }
        }
      }
      if constexpr (STAGE > 0) {
        stage_ask(first);
        stage_put();
#pragma unroll
        for (int q = 0; q < LINES; ++q)
#pragma unroll
          for (int hh = 0; hh < 2; ++hh) af[q][hh] = fragment(q * 128 + 2 * (a_first + hh * a_apart));
        wave_exchange();                                    // (the next trip's pieces are stored behind these reads)
      }
#pragma unroll
      for (int q = 0; q < LINES; ++q) {
#pragma unroll
        for (int s = 0; s < SETS; ++s) {
          bf16x8 b0, b1;
          lines_to_rows(wf[q][s][0], wf[q][s][HH - 1], col < 8, b0, b1);
          sums[0][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b0, af[q][0], sums[0][s], 0, 0, 0);
          sums[SUMS - 1][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b1, af[q][1], sums[SUMS - 1][s], 0, 0, 0);
        }
      }
    }
  } else {
    const bool w_ok = col < R && n_first + col < n_out;
    const bf16_t* wp[SETS];
#pragma unroll
    for (int s = 0; s < SETS; ++s) wp[s] = W + (size_t)(min(n_first + col, n_out - 1) + s * n_out) * K_all + k_lo + 8 * g;
    const int full_steps = K / 32;
    // A wave's last trip may reach past the end of K: such steps load nothing and multiply zeros (no matrix instruction sits
    // behind a condition).
    for (int ks = wave; ks < full_steps; ks += TRIP * NW) {
      bf16x8 wf[TRIP][SETS], af[TRIP];
#pragma unroll
      for (int u = 0; u < TRIP; ++u) {
        const int step = ks + u * NW;
        const bool valid = step < full_steps;
        const int k = min(step, full_steps - 1) * 32;
#pragma unroll
        for (int s = 0; s < SETS; ++s) wf[u][s] = load8(wp[s] + k, valid && w_ok);
        if constexpr (STAGE == 0) af[u] = load8(a_row + k + 8 * g, valid && a_ok);
      }
      if constexpr (STAGE > 0) {
        stage_ask(ks);
        stage_put();
#pragma unroll
        for (int u = 0; u < TRIP; ++u) {
          af[u] = fragment(u * 64 + 16 * g);
          if (ks + u * NW >= full_steps) af[u] = load8(nullptr, false);   // (the tail of K has weights of its own)
        }
        wave_exchange();
      }
#pragma unroll
      for (int u = 0; u < TRIP; ++u)
#pragma unroll
        for (int s = 0; s < SETS; ++s) sums[0][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u][s], af[u], sums[0][s], 0, 0, 0);
    }
    if (K & 31) {
      // The tail of K (a multiple of 8), zero-filled, is one wave's; the others multiply zeros, so that no matrix
      // instruction sits behind a condition on the wave (it would run whatever a lane mask says).
      const int k = full_steps * 32;
      const bool k_ok = wave == full_steps % NW && k + 8 * g < K;
      const bf16x8 af = load8(a_row + k + 8 * g, k_ok && a_ok);
#pragma unroll
      for (int s = 0; s < SETS; ++s)
        sums[0][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(load8(wp[s] + k, k_ok && w_ok), af, sums[0][s], 0, 0, 0);
    }
  }
  // (A register's lanes are turned by four for every register before it, so that the epilogue's reads touch every bank once.)
#pragma unroll
  for (int i = 0; i < SUMS; ++i)
#pragma unroll
    for (int s = 0; s < SETS; ++s)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wave * SUMS + i][s * 4 + r][(lane + 4 * r) & 63] = sums[i][s][r];
  __syncthreads();
  if (!e_wave || er >= R || n >= n_out) return;
#pragma unroll
  for (int at_m = 0; at_m < 16; at_m += 4 * NW) {
    const int m = em + at_m;
    if (m >= M) return;
    const int at = (er & 3) * WAVE + (((er >> 2) * 16 + m + 4 * (er & 3)) & 63);
    float v = 0.f, up = 0.f;
#pragma unroll
    for (int w = 0; w < NW * SUMS; ++w) {
      v += (&red[w][0][0])[at];
      if (GATED) up += (&red[w][(SETS - 1) * 4][0])[at];
    }
    if (biased) v += bias_here;
    // gate_act 1: the tanh form of GELU in place of silu; 2: max(z, 0).
    if (GATED)
      v = gate_act == 2 ? fmaxf(v, 0.f) * up
          : gate_act == 1 ? 0.5f * v * (1.0f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v))) * up
                          : v / (1.0f + __expf(-v)) * up;
    if (partial) st(partial + ((size_t)blockIdx.y * M + m) * n_out + n, v);         // (never GATED)
    else st(C + (size_t)m * ldc + n, v);
  }
}

// Weight rows a workgroup: sixteen where their workgroups are as many as compute units, fewer (four at least) where they are not.
static int few_rows_a_workgroup(int n_out, int splits) {
  const int units = compute_units();
  if ((long)((n_out + 15) / 16) * splits >= units) return 16;
  const int rows = (int)(((long)n_out * splits + units - 1) / units);
  return rows < 4 ? 4 : rows > 16 ? 16 : rows;
}

template <int NW, bool GATED, typename OutT, int LINES, bool WHOLE, int SUMS, bool UPPER, int STAGE>
static int launch_few_kernel(const void* A, int lda, const void* W, const void* bias, void* C, int ldc, int M, int N, int K, int k_chunk,
                             int rows, dim3 grid, float* slabs, int gate_act, hipStream_t stream) {
  constexpr int PIECES = (LINES > 0 ? LINES * 8 : 16);
  const size_t lds = STAGE > 0 ? (size_t)NW * M * (PIECES * 16 + 16) : 0;
  auto kernel = few_rows_gemm_kernel<NW, GATED, OutT, LINES, WHOLE, SUMS, UPPER, STAGE>;
  if (lds > 24 * 1024) {                                     // (beside up to 32 KB of its own)
    const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err != hipSuccess) return (int)err;
  }
  kernel<<<grid, NW * WAVE, lds, stream>>>((const bf16_t*)A, (const bf16_t*)W, (const float*)bias, slabs, lda, k_chunk,
                                           (uint32_t)M | (uint32_t)rows << 8 | (uint32_t)gate_act << 16, N, K, ldc, (OutT*)C);
  return LAUNCH_STATUS();
}

template <int NW, bool GATED, int LINES = 0, bool WHOLE = false, int SUMS = 1, bool UPPER = true>
static int launch_few(const void* A, int lda, const void* W, const void* bias, void* C, int ldc, int M, int N, int K, int out_dtype,
                      hipStream_t stream, int splits = 1, void* partial = nullptr, int gate_act = 0) {
  const int n_out = GATED ? N / 2 : N;
  const int step = LINES > 0 ? 64 : 32;
  const int k_chunk = splits > 1 ? ((K + splits - 1) / splits + step - 1) / step * step : K;
  if (splits > 1) splits = (K + k_chunk - 1) / k_chunk;          // no part without a step of its own
  const int rows = few_rows_a_workgroup(n_out, splits);
  if (!UPPER && rows > 8) return -1;
  const dim3 grid((n_out + rows - 1) / rows, splits);
  float* slabs = splits > 1 ? (float*)partial : nullptr;
  constexpr int PIECES = (LINES > 0 ? LINES * 8 : 16), MOST = (8 * PIECES + WAVE - 1) / WAVE;
  int status;
#define RUN(T, ST) launch_few_kernel<NW, GATED, T, LINES, WHOLE, SUMS, UPPER, ST>(A, lda, W, bias, C, ldc, M, N, K, k_chunk, rows, grid, \
                                                                                 slabs, gate_act, stream)
  // Rows straight from memory as well where a wave has up to three steps, whose fragments are hardly more loads than pieces and are there
  // sooner, and, K not in whole lines, in walks of more than one trip (two over tens of thousands of columns), where a trip's pieces are
  // asked for when the one before has been multiplied.  (Staged | direct, us: eight rows of 248 over 120 2.66 | 2.33, six of 200 over 232
  // 2.69 | 2.34, three of 752 over 128 2.56 | 2.26; eight of 7,576 over 1,424 7.6 | 7.0, of 6,000 over 6,000 24.6 | 23.7, gate/up 5,176 over 2,272 15.3 | 14.3;
  // six of 34,424 over 1,064 20.1 | 19.5, eight of 31,816 over 1,240 22.1 | 21.5.)
  const bool direct = M > 8 || K < 8 || (LINES == 0 && ((NW <= 8 && k_chunk <= NW * 96) || k_chunk > NW * (NW == 4 ? 256 : 128)));
#define PICK(T) status = direct ? RUN(T, 0) : M * PIECES <= WAVE ? RUN(T, 1) : RUN(T, MOST)
  if (out_dtype == DT_F32) PICK(float); else PICK(bf16_t);
#undef PICK
#undef RUN
  if (status == 0 && splits > 1 && C) status = launch_splitk_reduce(slabs, bias, C, M, N, ldc, splits, out_dtype, stream);
  return status;
}

// Column blocks per workgroup, by the launcher's choice (`asked` 0) or the caller's (1 or 2): two once there are
// more than 32 rows and the workgroups still fill the device.
static int column_blocks(int asked, int M, int n_out, int splits) {
  if (asked == 1 || asked == 2) return asked;
  return (M > 32 && (long)((n_out + 31) / 32) * splits >= 128) ? 2 : 1;
}

// Whether products that are not cut over K read their weights line by line where that is the faster way (tests and measurements switch it).
static int g_lines = 1;
extern "C" void ta_skinny_lines(int on) { g_lines = on; }

template <int MB, int NW, bool GATED, int NB = 1, int LINES = 0, bool WHOLE = false>
static int launch_skinny(const void* A, int lda, const void* W, const void* bias, void* C, int ldc, int M, int N,
                         int K, int out_dtype, hipStream_t stream, int splits = 1, void* partial = nullptr, int gate_act = 0) {
  const int n_out = GATED ? N / 2 : N;
  const int k_chunk = splits > 1 ? ((K + splits - 1) / splits + 31) / 32 * 32 : K;
  if (splits > 1) splits = (K + k_chunk - 1) / k_chunk;          // no part without a step of its own
  const dim3 grid((n_out + 16 * NB - 1) / (16 * NB), splits);
  float* slabs = splits > 1 ? (float*)partial : nullptr;
  if (out_dtype == DT_F32)
    skinny_gemm_kernel<MB, NW, GATED, float, false, NB, LINES, WHOLE><<<grid, NW * WAVE, 0, stream>>>(
        (const bf16_t*)A, lda, k_chunk, (const bf16_t*)W, (float*)C, ldc, M, N, K, slabs, (const float*)bias, RopeStore(), gate_act);
  else
    skinny_gemm_kernel<MB, NW, GATED, bf16_t, false, NB, LINES, WHOLE><<<grid, NW * WAVE, 0, stream>>>(
        (const bf16_t*)A, lda, k_chunk, (const bf16_t*)W, (bf16_t*)C, ldc, M, N, K, slabs, (const float*)bias, RopeStore(), gate_act);
  int status = LAUNCH_STATUS();
  if (status == 0 && splits > 1 && C) status = launch_splitk_reduce(slabs, bias, C, M, N, ldc, splits, out_dtype, stream);
  return status;
}

// Lines a wave with two sums asks for at once (`waves`: how many half lines would take).  The more rows, the fewer, since each brings as
// much of its own per line; a share of K of six lines in one trip and one of seven or eight in two; a gated product's two matrices fill
// a trip with one line, or two where rows are a multiple of 4 KB apart and a line of each is too much for the same memory channels.
// (Us by lines a trip.  Sixteen sums: 3,584 over 18,944, one row, 1 to 4: 38.2, 29.4, 26.0, 26.2, eight 32.8, 29.5, 30.1, 32.7, sixteen 35.1, 36.2,
// 37.7, 37.1; 3,584 over 3,584, one row 9.9, 8.1, 7.9, 7.5.  Eight: 4,608 over 3,584, one row 14.6, 11.3, 10.8, 11.2, sixteen 14.8, 15.3, 16.4, 16.1;
// gate/up 8,960 over 1,536, eight rows, 1, 2 and 6: 15.0, 15.1, 14.2; 8,960 over 3,584, one row 26.4, 29.3, 28.6; 14,336 over 4,096
// 47.2, 40.7, 42.3.  Four: 18,944 over 3,584, one row, 1 to 3: 26.4, 22.5, 25.1, sixteen 32.9, 36.0, 35.3; gate/up 42.5, 46.7, 44.6.)
static int lines_a_trip(bool gated, int waves, int M, int K) {
  const int share = (K / 64 + waves / 2 - 1) / (waves / 2);
  if (waves == 8 && share <= 6 && (gated || M <= 8)) return 6;
  if (M > 8) return 1;
  if (gated) return waves == 16 || K % 2048 == 0 ? 2 : 1;
  if (waves == 4 || M > 4) return 2;
  return waves == 16 && (share == 7 || share == 8) ? 4 : 3;
}

template <int MB, bool GATED>
static int pick_waves(const void* A, int lda, const void* W, const void* bias, void* C, int ldc, int M, int N,
                      int K, int out_dtype, hipStream_t stream, int col_blocks = 0, int gate_act = 0) {
  if constexpr (MB >= 3) {
    if (column_blocks(col_blocks, M, GATED ? N / 2 : N, 1) == 2)
      return launch_skinny<MB, 8, GATED, 2>(A, lda, W, bias, C, ldc, M, N, K, out_dtype, stream, 1, nullptr, gate_act);
  }
  if constexpr (MB == 1 && !GATED) {
    // Up to sixteen rows against tens of thousands of output columns (the vocabulary projection of a decode
    // step): four column blocks per workgroup, or a quarter of the workgroups would each read all the rows again.
    if ((col_blocks == 0 || col_blocks == 4) && (N + 15) / 16 >= 4096 && K <= 8192) {
      // The one long stream of a decode step: its weights are read line by line (0.5B sizes, 8 rows: 61.7 -> 55.7 us;
      // 7B sizes: 229 -> 201 us, 16 rows 248 -> 211 us).
      if (g_lines && (K & 63) == 0) return launch_skinny<1, 4, false, 4, 2, true>(A, lda, W, bias, C, ldc, M, N, K, out_dtype, stream);
      if (g_lines) return launch_skinny<1, 4, false, 4, 2>(A, lda, W, bias, C, ldc, M, N, K, out_dtype, stream);
      return launch_skinny<1, 4, false, 4>(A, lda, W, bias, C, ldc, M, N, K, out_dtype, stream);
    }
  }
  // Few output tiles and a long K: more waves per tile, so that enough loads are in flight.
  const int tiles = ((GATED ? N / 2 : N) + 15) / 16;
  const int k_steps = (K + 31) / 32;
  const int waves = tiles >= 1024 || k_steps <= 8 ? 4 : tiles >= 256 || k_steps <= 32 || MB * (GATED ? 2 : 1) > 2 ? 8 : 16;
  if constexpr (MB == 1) {
    // Whole lines where a wave's share of K is more than two of them: a shorter one is two trips at most and gains nothing (896 columns over
    // 896 3.3 -> 3.4 us, gate/up 4,864 over 896 7.1 -> 7.4).  Half as many waves with two sums each, so that the result is the one of half
    // lines to the last bit.  With one workgroup a compute unit and eight sums, half lines' eight waves have more on their way: there only
    // from five rows and 4,096 elements on (4,096 over 4,096, one and eight rows 9.2 and 9.4 us, whole lines 10.2 and 10.8; over 14,336
    // 25.9 and 30.0, 28.1 and 28.8; gate/up 4,096 over 2,048 10.0 and 10.0, 10.6 and 10.9).  Lines a trip: few rows' own loads leave room
    // for more of the weights' (see `lines_a_trip`).  Us half lines | so, weights from memory, one row and sixteen: gate/up 18,944 over 3,584
    // 53.4 | 42.5 and 59.4 | 52.4, down 31.8 | 26.0 and 44.4 | 35.1, 18,944 over 3,584 28.2 | 22.5 and 41.2 | 32.9; 3,584 over 3,584 8.0 | 7.5
    // and 9.5 | 9.1; gate/up 8,960 over 1,536 15.2 | 13.9 and 17.0 | 15.6, down 13.9 | 12.7 and 20.8 | 18.0; down 4,864 to 896 8.6 | 7.8 and
    // 11.7 | 10.9; 768 over 3,072 6.2 | 6.0 and 8.0 | 7.9.  Weights that are in the last-level cache already (all of a model in less than its
    // 256 MB) lose by it, one row and eight: 768 over 3,072 5.6 | 5.9 and 6.8 | 6.9, 896 over 4,864 7.8 | 7.8 and 9.3 | 9.4, 3,584 over
    // 3,584 6.6 | 6.8 and 7.5 | 8.0; the kernel cannot know, and models of that size are the exception.
    const int lines = K / 64;
    if (g_lines && (K & 63) == 0 && lines > 2 * waves && (waves != 8 || tiles > compute_units() || (!GATED && M > 4 && K > 4096))) {
      const int up = waves == 8 && tiles <= compute_units() ? 3 : lines_a_trip(GATED, waves, M, K);
#define GO(NWV, L) return launch_few<NWV, GATED, L, true, 2>(A, lda, W, bias, C, ldc, M, N, K, out_dtype, stream, 1, nullptr, gate_act)
#define HALF(L) return launch_few<8, false, L, true, 2, false>(A, lda, W, bias, C, ldc, M, N, K, out_dtype, stream, 1, nullptr, gate_act)
#define TRIPS(NWV) if (up == 1) GO(NWV, 1); if (up == 2) GO(NWV, 2); if constexpr (!GATED && NWV > 2) { if (up == 3) GO(NWV, 3); } \
                   if constexpr (!GATED && NWV == 8) { if (up == 4) GO(NWV, 4); } if constexpr (NWV == 4) { if (up == 6) GO(NWV, 6); }
      if constexpr (!GATED) {
        // Up to eight weight rows a workgroup: a line of them is one load, so a trip has more lines.
        if (waves == 16 && few_rows_a_workgroup(N, 1) <= 8) {
          const int share = (lines + 7) / 8, trips = M > 8 ? (share + 3) / 4 : (share + 9) / 10, each = (share + trips - 1) / trips;
          if (each <= 4) HALF(4);
          if (each <= 6) HALF(6);
          if (each <= 8) HALF(8);
          HALF(10);
        }
      }
      if (waves == 4) { TRIPS(2) }
      if (waves == 8) { TRIPS(4) }
      if (waves == 16) { TRIPS(8) }
#undef TRIPS
#undef HALF
#undef GO
    }
    if (waves == 4) return launch_few<4, GATED>(A, lda, W, bias, C, ldc, M, N, K, out_dtype, stream, 1, nullptr, gate_act);
    if (waves == 8) return launch_few<8, GATED>(A, lda, W, bias, C, ldc, M, N, K, out_dtype, stream, 1, nullptr, gate_act);
    return launch_few<16, GATED>(A, lda, W, bias, C, ldc, M, N, K, out_dtype, stream, 1, nullptr, gate_act);
  } else {
    if (waves == 4) return launch_skinny<MB, 4, GATED>(A, lda, W, bias, C, ldc, M, N, K, out_dtype, stream, 1, nullptr, gate_act);
    if constexpr (MB * (GATED ? 2 : 1) <= 2)
      if (waves == 16) return launch_skinny<MB, 16, GATED>(A, lda, W, bias, C, ldc, M, N, K, out_dtype, stream, 1, nullptr, gate_act);
    return launch_skinny<MB, 8, GATED>(A, lda, W, bias, C, ldc, M, N, K, out_dtype, stream, 1, nullptr, gate_act);
  }
}

// M <= 64; K, lda multiples of 8; pointers 16-byte aligned; with `gated` N is even and C is [M, N/2]
// (gated 1: silu(gate) * up; 2: the tanh form of GELU in place of silu; 3: max(gate, 0)).
// col_blocks: blocks of sixteen output columns per workgroup, 0 = the launcher's choice (see column_blocks).
extern "C" int ta_gemm_skinny_bf16(const void* A, int lda, const void* W, const void* bias, void* C, int ldc,
                                   int M, int N, int K, int out_dtype, int gated, int col_blocks, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 64 || (K & 7) || (lda & 7) || (gated && (N & 1))) return -1;
  const int mb = (M + 15) / 16;
#define GO(MBV) (gated ? pick_waves<MBV, true>(A, lda, W, bias, C, ldc, M, N, K, out_dtype, stream, col_blocks, gated - 1) \
                       : pick_waves<MBV, false>(A, lda, W, bias, C, ldc, M, N, K, out_dtype, stream, col_blocks))
  switch (mb) {
    case 1: return GO(1);
    case 2: return GO(2);
    case 3: return GO(3);
    default: return GO(4);
  }
#undef GO
}

// The same product (not gated) with K cut into `splits` parts (at most; parts are multiples of 32, of 64 for up to sixteen rows and
// K in whole lines, which are then always read as such, one block of columns a workgroup, whatever `ta_skinny_lines` and `col_blocks`
// say: 8 rows x 1,536 over 8,960 12.2 -> 11.7 us, one row 11.0 -> 10.2) over the workgroups, the parts' float sums added afterwards in a
// fixed order.  partial: room for splits * M * N floats; N % 4 == 0; M <= 64.  With C null (and more than one part after the rounding of
// the parts' length) the sums are left in `partial` for a later kernel to add.
extern "C" int ta_gemm_skinny_bf16_splitk(const void* A, int lda, const void* W, const void* bias, void* C, int ldc,
                                          void* partial, int M, int N, int K, int out_dtype, int splits,
                                          int col_blocks, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 64 || (K & 7) || (lda & 7) || (N & 3) || splits < 1 || (splits > 1 && !partial)) return -1;
  const bool whole = M <= 16 && (K & 63) == 0;
  if (!C && parts_of_k(K, splits, whole ? 64 : 32) < 2) return -1;
  if (whole) return launch_few<8, false, 1, true>(A, lda, W, bias, C, ldc, M, N, K, out_dtype, stream, splits, partial);
#define GO(MBV, NBV) launch_skinny<MBV, 8, false, NBV>(A, lda, W, bias, C, ldc, M, N, K, out_dtype, stream, splits, partial)
  const bool two = column_blocks(col_blocks, M, N, parts_of_k(K, splits, 32)) == 2;
  switch ((M + 15) / 16) {
    case 1: return launch_few<8, false>(A, lda, W, bias, C, ldc, M, N, K, out_dtype, stream, splits, partial);
    case 2: return GO(2, 1);
    case 3: return two ? GO(3, 2) : GO(3, 1);
    default: return two ? GO(4, 2) : GO(4, 1);
  }
#undef GO
}

// The joined q/k/v projection of 17 to 64 rows with bias, rotation and the cache write in its epilogue (see
// RopeStore): x bfloat16 [M, K] (row stride lda), W [(n_q + 2 n_kv) d, K], bias float32 or null; queries go to
// q_out [M, n_q d]; cos_sin float32 [positions, d] or null (no rotation); slots int32 [M] or null (nothing is
// stored; a negative slot skips its row).  d a multiple of 32.
extern "C" int ta_gemm_skinny_qkv_rope(const void* x, int lda, const void* W, const void* bias, void* q_out,
                                       const void* positions, const void* cos_sin, const void* slots, void* k_pages,
                                       void* v_pages, int M, int K, int n_q, int n_kv, int d, int page_size,
                                       hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > 64 || (K & 7) || (lda & 7) || (d & 31) || n_q <= 0 || n_kv <= 0 || page_size <= 0 || !positions) return -1;
  if (slots && (!k_pages || !v_pages)) return -1;
  RopeStore rope;
  rope.positions = (const int*)positions; rope.cos_sin = (const float*)cos_sin; rope.slots = (const int*)slots;
  rope.k_pages = (bf16_t*)k_pages; rope.v_pages = (bf16_t*)v_pages;
  rope.n_q = n_q; rope.n_kv = n_kv; rope.d = d; rope.page_size = page_size;
  const int N = (n_q + 2 * n_kv) * d;
  const int tiles = (n_q + 2 * n_kv) * (d / 32);
  const int blocks = (M + 15) / 16;
  // Few tiles (a small model's joined matrix is a few dozen): the blocks of sixteen rows are dealt to workgroups
  // of their own, as many shares as it takes to fill the device; every share reads the matrix again.
  const int shares = min(blocks, (compute_units() + tiles - 1) / tiles);
  const int per_share = (blocks + shares - 1) / shares;
  const dim3 grid(tiles, 1, (blocks + per_share - 1) / per_share);
#define GO(MBV) skinny_gemm_kernel<MBV, 8, true, bf16_t, true><<<grid, 8 * WAVE, 0, stream>>>( \
    (const bf16_t*)x, lda, K, (const bf16_t*)W, (bf16_t*)q_out, n_q * d, M, N, K, nullptr, (const float*)bias, rope)
  switch (per_share) {
    case 1: GO(1); break;
    case 2: GO(2); break;
    case 3: GO(3); break;
    default: GO(4); break;
  }
#undef GO
  return LAUNCH_STATUS();
}
