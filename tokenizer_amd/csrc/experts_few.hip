// Routed experts of few rows (decode steps): only the experts that some row chose are read.  Two kernels: the first
// product of every chosen expert with the rows that chose it, the activation and the rows' weights in its epilogue; and
// the second product, whose results lie pick by pick (slab k holds every row's k-th pick), for whoever adds them up.
// bfloat16 operands, float sums on the matrix cores (16x16x32), computed transposed, C^T = W x^T, as the weight-streaming
// product does: sixteen weight rows are the M side, up to sixteen (row, pick) pairs of the expert the N side, the waves of a
// workgroup take turns of 64 elements of K and add up through LDS.  Bound by the chosen matrices' way from memory: they are read line
// by line (`lines_to_rows` in common.h) and past the caches, which no later workgroup asks them from.  (Sixteen rows' half lines a load |
// whole lines | whole lines past the caches, us for both products: 2 of 8 experts of 9,472 over 3,584, four rows, 197 | 177 | 160
// (6.4 TB/s); 2 of 8 of 2,240 and a shared one of 4,480 over 1,536, three rows, 42.3 | 37.3 | 34.4; half lines past the caches 215 and
// 44.8: each line then comes twice.  Weights that are in the last-level cache already, all of a model in less than its 256 MB, half lines | so,
// one row, four and sixteen: 1,024 over 1,024 7.9 | 8.3, 11.3 | 11.7, 13.9 | 13.3; 3,648 over 896 14.8 | 14.0, 23.6 | 22.7, 32.4 | 32.4; 2,736
// over 2,048 21.6 | 23.5, 31.9 | 30.6, 52.6 | 58.4.)  An expert that every row uses besides (of an inner width of its own) is one further
// expert in both grids, whose pairs are the rows; its K in the second product is cut into parts about
// as long as the others', each a slab of its own.
#include "common.h"

typedef float ef_floatx4 __attribute__((ext_vector_type(4)));

#define EF_MAX_PAIRS 256

// The pairs of this workgroup's expert, in rising order: every wave counts them for itself (the count is the same for all),
// the first wave lists them in LDS.
__device__ __forceinline__ int ef_pairs_of(const int* __restrict__ chosen, int n_pairs, int expert, int* list) {
  const int lane = threadIdx.x & (WAVE - 1);
  int count = 0;
#pragma unroll
  for (int base = 0; base < EF_MAX_PAIRS; base += WAVE) {
    if (base >= n_pairs) break;
    const int p = base + lane;
    const bool mine = p < n_pairs && chosen[p] == expert;
    const unsigned long long all = __ballot(mine);
    if (mine && threadIdx.x < WAVE) list[count + __popcll(all & ((1ull << lane) - 1))] = p;
    count += __popcll(all);
  }
  return __builtin_amdgcn_readfirstlane(count);
}

// The expert that all rows use: `inner` 0 says that there is none.  Its matrices stand behind the others'; weights null: 1.
struct EfShared { int inner; const float* weights; bf16_t* act; int parts, length; };   // K of `inner` in `parts` of `length`

// acc[h] += sixteen rows of matrix h (lane (col, g): `w_at[h][0]` is row col % 8 of them, `w_at[h][1]` row 8 + col % 8) times the
// rows of x that `row_at(i)` says for its `here` <= 16 pairs, over this wave's turns of K, UN of which are asked for at once.
// SLOTS > 0 (here * UN * 8 pieces of sixteen bytes fill no more loads): the pairs' shares of a trip come in SLOTS loads of sixteen different
// bytes a lane and become fragments through `stage`, LDS of the wave's own.  A chosen expert of a few rows has one or two pairs, and a
// fragment straight from memory is two loads a turn, as many as a matrix has, whose lanes mostly ask for nothing of their own.
#define EF_STAGE_ROWS(UN) ((UN) == 1 ? 8 : 16 / (UN))                 // pairs that are staged at most: SLOTS 1, with four turns 2 too
#define EF_STAGE_BYTES(UN) (EF_STAGE_ROWS(UN) * ((UN) * 128 + 16))
template <int NW, int HALVES, int UN, int SLOTS, typename RowAt>
__device__ __forceinline__ void ef_walk_form(const bf16_t* const (&w_at)[HALVES][2], RowAt row_at, int here, int K, int wave, char* stage,
                                             ef_floatx4 (&acc)[HALVES]) {
  const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4, piece = g + 4 * (col >> 3);
  const int turns = (K + 63) / 64;
  constexpr int PIECES = UN * 8, ROW_BYTES = PIECES * 16 + 16;
  const word4 zero = {0u, 0u, 0u, 0u};
  const bf16_t* from[SLOTS > 0 ? SLOTS : 1];
  if constexpr (SLOTS > 0) {
#pragma unroll
    for (int j = 0; j < SLOTS; ++j) from[j] = row_at(min(j * WAVE + lane, here * PIECES - 1) / PIECES);
  } else {
    from[0] = row_at(min(col, here - 1));
  }
  const bool x_ok = col < here;
  for (int first = wave; first < turns; first += UN * NW) {
    word4 wf[UN][HALVES][2], xf[UN][2], staged[SLOTS > 0 ? SLOTS : 1];
#pragma unroll
    for (int q = 0; q < UN; ++q) {
      const int turn = first + q * NW, at = min(turn, turns - 1) * 64;
      const bool w_in = turn < turns && at + 8 * piece < K;
#pragma unroll
      for (int h = 0; h < HALVES; ++h)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
          wf[q][h][hh] = w_in ? __builtin_nontemporal_load(reinterpret_cast<const word4*>(w_at[h][hh] + at + 8 * piece)) : zero;
      if constexpr (SLOTS == 0) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {                        // what the weights are after the exchange: the pieces g and 4 + g
          const bool x_in = turn < turns && at + 32 * s + 8 * g < K;
          xf[q][s] = x_in && x_ok ? *reinterpret_cast<const word4*>(from[0] + at + 32 * s + 8 * g) : zero;
        }
      }
    }
    if constexpr (SLOTS > 0) {
#pragma unroll
      for (int j = 0; j < SLOTS; ++j) {
        const int i = min(j * WAVE + lane, here * PIECES - 1) % PIECES, k = (first + (i >> 3) * NW) * 64 + 8 * (i & 7);
        staged[j] = *reinterpret_cast<const word4*>(from[j] + min(k, K - 8));
      }
#pragma unroll
      for (int j = 0; j < SLOTS; ++j) {
        const int i = min(j * WAVE + lane, here * PIECES - 1), k = (first + ((i % PIECES) >> 3) * NW) * 64 + 8 * (i & 7);
        if (k >= K) staged[j] = zero;
        *reinterpret_cast<word4*>(stage + i / PIECES * ROW_BYTES + i % PIECES * 16) = staged[j];
      }
      wave_exchange();
#pragma unroll
      for (int q = 0; q < UN; ++q)
#pragma unroll
        for (int s = 0; s < 2; ++s) xf[q][s] = *reinterpret_cast<const word4*>(stage + min(col, here - 1) * ROW_BYTES + q * 128 + s * 64 + g * 16);
      wave_exchange();                                       // (the next trip's pieces are stored behind these reads)
    }
#pragma unroll
    for (int q = 0; q < UN; ++q)
#pragma unroll
      for (int h = 0; h < HALVES; ++h) {
        line_bf16x8 part[2];
        lines_to_rows(wf[q][h][0], wf[q][h][1], col < 8, part[0], part[1]);
#pragma unroll
        for (int s = 0; s < 2; ++s)
          acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(part[s], __builtin_bit_cast(line_bf16x8, xf[q][s]), acc[h], 0, 0, 0);
      }
  }
}
template <int NW, int HALVES, int UN, bool STAGED, typename RowAt>
__device__ __forceinline__ void ef_walk(const bf16_t* const (&w_at)[HALVES][2], RowAt row_at, int here, int K, int wave, char* stage,
                                        ef_floatx4 (&acc)[HALVES]) {
  static_assert(UN == 1 || UN == 4, "");
  constexpr int ONE = 8 / UN;                                // pairs of one load
  if (!STAGED) ef_walk_form<NW, HALVES, UN, 0>(w_at, row_at, here, K, wave, stage, acc);
  else if (here <= ONE) ef_walk_form<NW, HALVES, UN, 1>(w_at, row_at, here, K, wave, stage, acc);
  else if (UN == 4 && here <= 2 * ONE) ef_walk_form<NW, HALVES, UN, 2>(w_at, row_at, here, K, wave, stage, acc);
  else ef_walk_form<NW, HALVES, UN, 0>(w_at, row_at, here, K, wave, stage, acc);
}

// x [n_rows, x_stride]; chosen int [n_rows * top], weights float [n_rows * top]; expert e's first matrix starts at
// W + e * HALVES * inner * hidden: [gate; up] of `inner` rows each (HALVES 2) or `up` alone (HALVES 1), rows of `hidden`.
// act [n_rows * top, inner]: pair p's row.  HALVES 2: weigh_input ? silu(w g) * (w u) : w * silu(g) * u; HALVES 1: w * max(u, 0)^2.
// Grid: (blocks of sixteen columns of inner, experts).
template <int NW, int HALVES, int UN, bool STAGED>
__global__ void __launch_bounds__(NW * WAVE)
experts_few_up_kernel(const bf16_t* __restrict__ x, int x_stride, const int* __restrict__ chosen, const float* __restrict__ weights,
                      int n_pairs, int top, const bf16_t* __restrict__ W, int inner, int hidden, bf16_t* __restrict__ act,
                      int weigh_input, EfShared every) {
  HELD(x, x_stride, chosen, weights, n_pairs, top, W, inner, hidden, act, weigh_input, every.inner, every.weights, every.act);
  __shared__ int list[EF_MAX_PAIRS];
  __shared__ float red[NW][HALVES * 4][WAVE];
  __shared__ __attribute__((aligned(16))) char stage_s[STAGED ? NW * EF_STAGE_BYTES(UN) : 16];
  // (The shared expert's workgroups, the ones with the most rows, come first.)
  const bool shared = every.inner > 0 && blockIdx.y == 0;
  const int expert = blockIdx.y - (every.inner > 0 ? 1 : 0), n0 = blockIdx.x * 16;
  const bf16_t* first = W + (size_t)(shared ? gridDim.y - 1 : expert) * HALVES * inner * hidden;
  int count;
  if (shared) {                                              // its pairs are the rows
    count = n_pairs / top;
    inner = every.inner;
    top = 1;
    weights = every.weights;
    act = every.act;
    for (int i = threadIdx.x; i < count; i += NW * WAVE) list[i] = i;
  } else {
    count = ef_pairs_of(chosen, n_pairs, expert, list);
  }
  if (count == 0 || n0 >= inner) return;                     // nobody's expert, or past its width: the same for the whole workgroup
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = wave_index(), col = lane & 15;
  const bf16_t* w_at[HALVES][2];
#pragma unroll
  for (int h = 0; h < HALVES; ++h)
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) w_at[h][hh] = first + ((size_t)h * inner + min(n0 + 8 * hh + (col & 7), inner - 1)) * hidden;
  for (int p0 = 0; p0 < count; p0 += 16) {
    const int here = min(count - p0, 16);
    // The weight of the pair whose sum this thread stores, asked for beside the first rows.
    float wgt = 1.f;
    if (wave < 4 && weights) wgt = weights[list[p0 + min((int)threadIdx.x >> 4, here - 1)]];
    ef_floatx4 acc[HALVES];
#pragma unroll
    for (int h = 0; h < HALVES; ++h) acc[h] = (ef_floatx4){0.f, 0.f, 0.f, 0.f};
    ef_walk<NW, HALVES, UN, STAGED>(w_at, [&](int i) { return x + (size_t)(list[p0 + i] / top) * x_stride; }, here, hidden, wave,
                            stage_s + wave * EF_STAGE_BYTES(UN), acc);
    // A matrix instruction's result may be read eight wait states behind it at the earliest.  The compiler leaves them out in front
    // of the stores below where there is one matrix (the store is the second instruction behind the last sum; with many
    // workgroups some stored a sum that was not there yet), so they are here, twice over; with two matrices it has them.
    if constexpr (HALVES == 1) asm volatile("s_nop 7\n\ts_nop 7" : "+v"(acc[0]));
#pragma unroll
    for (int h = 0; h < HALVES; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wave][h * 4 + r][lane] = acc[h][r];
    __syncthreads();
    // Lane (col, g) held rows 4 g .. 4 g + 3 of column (pair) col: thread (pair, row) gathers its own.
    for (int idx = threadIdx.x; idx < 256; idx += NW * WAVE) {
      const int c = idx >> 4, r = idx & 15;
      if (p0 + c >= count || n0 + r >= inner) continue;
      float v[HALVES];
#pragma unroll
      for (int h = 0; h < HALVES; ++h) {
        v[h] = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) v[h] += red[w][h * 4 + (r & 3)][(r >> 2) * 16 + c];
        // (Rounded as the product over all experts leaves them, so that a row is the same in either form but for the
        // order of its sums.)
        v[h] = bf16_bits_to_float(float_to_bf16_bits(v[h]));
      }
      const int p = list[p0 + c];
      float value;
      if constexpr (HALVES == 2) {
        const float before = weigh_input ? wgt : 1.f, z = before * v[0];
        value = (weigh_input ? 1.f : wgt) * (z / (1.0f + expf(-z)) * (before * v[1]));
      } else {
        const float z = fmaxf(v[0], 0.f);
        value = wgt * (z * z);
      }
      // (A pick that weighs nothing adds nothing, whatever its expert makes of the row: as the form over all experts has it.)
      if (!shared && wgt == 0.f) value = 0.f;
      st(act + (size_t)p * inner + n0 + r, value);
    }
    __syncthreads();                                         // the sums are read before the next sixteen pairs' are written
  }
}

// out [top, n_rows, hidden] float: out[p % top, p / top] = act[p] times expert chosen[p]'s second matrix, which is columns
// e * inner .. of W [hidden, ldw].  Grid: (blocks of sixteen output columns, experts).
template <int NW, bool STAGED>
__global__ void __launch_bounds__(NW * WAVE)
experts_few_down_kernel(const bf16_t* __restrict__ act, const int* __restrict__ chosen, int n_pairs, int top, int n_rows,
                        const bf16_t* __restrict__ W, int ldw, int inner, int hidden, float* __restrict__ out, EfShared every) {
  HELD(act, chosen, n_pairs, top, n_rows, W, ldw, inner, hidden, out, every.parts, every.length, every.inner, every.act);
  __shared__ int list[EF_MAX_PAIRS];
  __shared__ float red[NW][4][WAVE];
  __shared__ __attribute__((aligned(16))) char stage_s[STAGED ? NW * EF_STAGE_BYTES(4) : 16];
  const int part = blockIdx.y;                               // below every.parts: a part of the shared expert's K
  const bool shared = part < every.parts;
  const int expert = part - every.parts, n0 = blockIdx.x * 16;
  const bf16_t* columns = W + (size_t)(shared ? (int)gridDim.y - every.parts : expert) * inner;
  int count, stride = inner, slab = 0;
  if (shared) {
    const int begin = part * every.length;
    count = n_rows;
    stride = every.inner;
    inner = min(every.length, every.inner - begin);
    columns += begin;
    act = every.act + begin;
    slab = top + part;
    top = 1;
    for (int i = threadIdx.x; i < count; i += NW * WAVE) list[i] = i;
  } else {
    count = ef_pairs_of(chosen, n_pairs, expert, list);
  }
  if (count == 0) return;
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = wave_index(), col = lane & 15;
  const bf16_t* const w_at[1][2] = {{columns + (size_t)min(n0 + (col & 7), hidden - 1) * ldw,
                                     columns + (size_t)min(n0 + 8 + (col & 7), hidden - 1) * ldw}};
  for (int p0 = 0; p0 < count; p0 += 16) {
    const int here = min(count - p0, 16);
    ef_floatx4 acc[1] = {(ef_floatx4){0.f, 0.f, 0.f, 0.f}};
    ef_walk<NW, 1, 4, STAGED>(w_at, [&](int i) { return act + (size_t)list[p0 + i] * stride; }, here, inner, wave, stage_s + wave * EF_STAGE_BYTES(4), acc);
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wave][r][lane] = acc[0][r];
    __syncthreads();
    for (int idx = threadIdx.x; idx < 256; idx += NW * WAVE) {
      const int c = idx >> 4, r = idx & 15;
      if (p0 + c >= count || n0 + r >= hidden) continue;
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) v += red[w][r & 3][(r >> 2) * 16 + c];
      const int p = list[p0 + c];
      out[((size_t)(slab + p % top) * n_rows + p / top) * hidden + n0 + r] = v;
    }
    __syncthreads();
  }
}

// The shared expert's second product: K in parts about as long as the others' K, four at most, each of whole turns of 64 and none
// without one.
static int shared_part(int inner, int shared) {
  const int parts = (shared + inner - 1) / inner;
  const int most = parts < 4 ? parts : 4;
  return ((shared + most - 1) / most + 63) / 64 * 64;
}

// The parts it is left in (slabs behind the picks').
extern "C" int ta_experts_few_shared_parts(int inner, int shared) {
  if (shared <= 0 || inner <= 0) return 0;
  const int length = shared_part(inner, shared);
  return (shared + length - 1) / length;
}

// Returns -2 for sizes the kernels do not take.  halves: 2 = gate and up rows (silu), 1 = up rows alone (squared ReLU).
// shared: the inner width of the expert all rows use (0: there is none), whose matrices stand behind the others' in w_first and
// w_second; shared_weights float [n_rows] or null; act_shared [n_rows, shared].
extern "C" int ta_experts_few(const void* x, int x_stride, const void* chosen, const void* weights, int n_rows, int top,
                              int n_experts, const void* w_first, int halves, int inner, int hidden, int weigh_input, void* act,
                              const void* w_second, int ldw, void* out, int shared, const void* shared_weights, void* act_shared,
                              hipStream_t stream) {
  if (n_rows <= 0) return 0;
  const long pairs = (long)n_rows * top;
  if (top <= 0 || n_experts <= 0 || n_experts > 65535 || inner <= 0 || hidden <= 0 || (halves != 1 && halves != 2) ||
      ldw < n_experts * inner + shared || x_stride < hidden || shared < 0 || (shared > 0 && (!act_shared || weigh_input)))
    return -1;
  if (pairs > EF_MAX_PAIRS || inner % 8 || hidden % 8 || ldw % 8 || x_stride % 8 || shared % 8 ||
      (((uintptr_t)x | (uintptr_t)w_first | (uintptr_t)w_second | (uintptr_t)act | (uintptr_t)act_shared) & 15))
    return -2;
  const EfShared every = {shared, (const float*)shared_weights, (bf16_t*)act_shared, ta_experts_few_shared_parts(inner, shared),
                          shared > 0 ? shared_part(inner, shared) : 0};
  if (n_experts + every.parts > 65535) return -2;            // (a grid's second dimension)
  const dim3 up(((inner > shared ? inner : shared) + 15) / 16, n_experts + (shared > 0)),
      down((hidden + 15) / 16, n_experts + every.parts);
#define UP(NW, HH, UN, ST) experts_few_up_kernel<NW, HH, UN, ST><<<up, NW * WAVE, 0, stream>>>((const bf16_t*)x, x_stride, (const int*)chosen, \
    (const float*)weights, (int)pairs, top, (const bf16_t*)w_first, inner, hidden, (bf16_t*)act, weigh_input, every)
#define DOWN(NW, ST) experts_few_down_kernel<NW, ST><<<down, NW * WAVE, 0, stream>>>((const bf16_t*)act, (const int*)chosen, (int)pairs, top, \
    n_rows, (const bf16_t*)w_second, ldw, inner, hidden, (float*)out, every)
  // Turns asked for at once.  One of two matrices, four loads of weights a lane (two take registers that more waves a compute unit make
  // better use of: 5,504 over 2,048, four rows 52.5 | 55.0 us for both products), but four where the workgroups cannot be more than the
  // compute units, however the rows choose, and none has another to hide its trips (one | four: 1,792 over 4,096, one row 33.6 | 24.8; 1,024
  // over 1,024 10.9 | 9.4, two rows 11.4 | 9.8; 512 over 1,024, four rows 11.5 | 10.0).  Four of one matrix, eight loads.
  const long busy = (pairs < n_experts ? pairs : n_experts) * ((inner + 15) / 16) + (shared + 15) / 16;
  // Rows are staged where a wave has more than two turns of K: with fewer most of a trip's pieces are none (512 over 512, two of 8 experts, one row
  // 6.8 | 7.05 us both products, sixteen 8.3 | 8.5).
#define FOUR(HH) do { if (hidden <= 512) UP(4, HH, 4, false); else if (hidden <= 1024) UP(4, HH, 4, true); else UP(8, HH, 4, true); } while (0)
  if (halves == 1) FOUR(1);
  else if (busy <= compute_units()) FOUR(2);
  // (The staged forms' registers leave a SIMD five waves in place of seven: they pay while an expert has few pairs and long rows.  Both products, two of 8
  // experts, direct | staged: 1,536 and 2,240 beside 4,480, three rows 35.3 | 34.5, eight 41.7 | 41.9, sixteen 46.2 | 46.7; 3,584 and 9,472, four
  // rows 188.4 | 185.0; but 1,024 and 3,584, two rows 20.2 | 21.0.)
  else if (hidden <= 1024) UP(4, 2, 1, false);
  else if (pairs <= 8) UP(8, 2, 1, true);
  else UP(8, 2, 1, false);
  int status = LAUNCH_STATUS();
  if (status != 0) return status;
  if (inner <= 512) DOWN(4, false); else if (inner <= 1024) DOWN(4, true); else DOWN(8, true);
#undef FOUR
#undef UP
#undef DOWN
  return LAUNCH_STATUS();
}
