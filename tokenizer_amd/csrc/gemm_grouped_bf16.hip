// Products of a routed feed-forward over sorted tokens: every tile of BM rows belongs to one expert and is multiplied
// with that expert's matrix alone.  bfloat16 operands, float accumulation on the matrix cores
// (v_mfma_f32_32x32x16_bf16), staged through LDS as in gemm_bf16.hip; and the two small kernels around them: the one
// that sorts a step's (token, chosen expert) pairs into such tiles, and the one that adds a token's experts up.
#include "common.h"
#include "tile_ring.h"

typedef __bf16 gg_bf16x8 __attribute__((ext_vector_type(8)));
typedef float gg_floatx16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ void gg_store(float* p, float v) { *p = v; }
__device__ __forceinline__ void gg_store(bf16_t* p, float v) { p->bits = float_to_bf16_bits(v); }

typedef float gg_floatx4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void gg_store4(float* p, const gg_floatx4& v) { *reinterpret_cast<gg_floatx4*>(p) = v; }
__device__ __forceinline__ void gg_store4(bf16_t* p, const gg_floatx4& v) {
  *reinterpret_cast<uint2*>(p) = make_uint2((uint32_t)float_to_bf16_bits(v[0]) | ((uint32_t)float_to_bf16_bits(v[1]) << 16),
                                            (uint32_t)float_to_bf16_bits(v[2]) | ((uint32_t)float_to_bf16_bits(v[3]) << 16));
}

#define GG_MAX_EXPERTS 256

// chosen: int [n_entries] (entry i = token i / top, its pick i % top; a value outside 0..n_experts-1 is passed over).
// Every expert's entries get consecutive slots, the expert's run starting at a multiple of `bm` slots:
//   slot_of[i] = the entry's slot (or -1), row_of[slot] = the entry's token (or -1 for a slot that only fills a tile up),
//   tile_expert[tile] = the expert of slots tile * bm .. + bm - 1 (or -1 for a tile past the last run).
// row_of has n_tiles * bm entries, tile_expert n_tiles, n_tiles >= n_entries / bm + n_experts.  One workgroup; the
// order of an expert's entries among themselves is whatever order the counter was reached in, which no result depends on.
__global__ void __launch_bounds__(1024)
expert_slots_kernel(const int* __restrict__ chosen, int n_entries, int top, int n_experts, int bm, int n_tiles,
                    int* __restrict__ slot_of, int* __restrict__ row_of, int* __restrict__ tile_expert) {
  __shared__ int count_s[GG_MAX_EXPERTS], start_s[GG_MAX_EXPERTS];
  for (int e = threadIdx.x; e < n_experts; e += blockDim.x) count_s[e] = 0;
  for (int s = threadIdx.x; s < n_tiles * bm; s += blockDim.x) row_of[s] = -1;
  for (int t = threadIdx.x; t < n_tiles; t += blockDim.x) tile_expert[t] = -1;
  __syncthreads();
  for (int i = threadIdx.x; i < n_entries; i += blockDim.x) {
    const int e = chosen[i];
    slot_of[i] = (e >= 0 && e < n_experts) ? atomicAdd(&count_s[e], 1) : -1;      // for now: the entry's rank in its run
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int at = 0;
    for (int e = 0; e < n_experts; ++e) {
      start_s[e] = at;
      at += (count_s[e] + bm - 1) / bm * bm;
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < n_experts; e += blockDim.x)
    for (int t = start_s[e] / bm; t < (start_s[e] + count_s[e] + bm - 1) / bm; ++t) tile_expert[t] = e;
  for (int i = threadIdx.x; i < n_entries; i += blockDim.x) {
    const int e = chosen[i];
    if (e < 0 || e >= n_experts) continue;
    const int slot = start_s[e] + slot_of[i];
    slot_of[i] = slot;
    row_of[slot] = i / top;
  }
}

// C[slot, :N] = A[row_of[slot], :K] . W_e[:N, :K]^T for every slot of every tile, W_e = W + e * expert_stride elements
// with rows `ldw` apart, e = tile_expert[tile].  row_of null: A's rows are the slots themselves.  A slot that only fills
// a tile up (row_of < 0) is computed from row 0 and never read by anyone.  K, lda, ldw and expert_stride multiples
// of 8, pointers 16-byte aligned.
template <int BM, int BN, int BK, typename OutT, int AHEAD = 3>
__global__ void __launch_bounds__(256)
grouped_gemm_bf16_kernel(const bf16_t* __restrict__ A, int lda, const int* __restrict__ row_of,
                         const int* __restrict__ tile_expert, const bf16_t* __restrict__ W, long expert_stride, int ldw,
                         OutT* __restrict__ C, int ldc, int N, int K) {
  constexpr int WM = BM / 2, WN = BN / 2, TMI = WM / 32, TNI = WN / 32;
  constexpr int GB_LDS = BK + 8, CPR = BK / 8;
  constexpr int A_CHUNKS = BM * CPR / 256, W_CHUNKS = BN * CPR / 256;
  const int expert = scalar_int(tile_expert + blockIdx.y);
  if (expert < 0) return;                                   // a tile past the last run
  __shared__ __attribute__((aligned(16))) uint16_t a_s[2][BM * GB_LDS];
  __shared__ __attribute__((aligned(16))) uint16_t w_s[2][BN * GB_LDS];
  __shared__ int src_s[BM];
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_index();
  const int wm = wave >> 1, wn = wave & 1;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  for (int r = tid; r < BM; r += 256) src_s[r] = row_of ? max(row_of[m0 + r], 0) : m0 + r;
  __syncthreads();
  const bf16_t* We = W + (size_t)expert * expert_stride;
  gg_floatx16 acc[TMI][TNI];
#pragma unroll
  for (int i = 0; i < TMI; ++i)
#pragma unroll
    for (int j = 0; j < TNI; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  uint4 a_reg[AHEAD][A_CHUNKS], w_reg[AHEAD][W_CHUNKS];
  int a_row[A_CHUNKS];
#pragma unroll
  for (int i = 0; i < A_CHUNKS; ++i) a_row[i] = src_s[(tid + i * 256) / CPR];
  auto fetch = [&](int k0, uint4 (&a_now)[A_CHUNKS], uint4 (&w_now)[W_CHUNKS]) {
#pragma unroll
    for (int i = 0; i < A_CHUNKS; ++i) {
      const int c = tid + i * 256;
      const int k = min(k0 + (c % CPR) * 8, K - 8);
      a_now[i] = *reinterpret_cast<const uint4*>(A + (size_t)a_row[i] * lda + k);
    }
#pragma unroll
    for (int i = 0; i < W_CHUNKS; ++i) {
      const int c = tid + i * 256;
      const int n = min(n0 + c / CPR, N - 1), k = min(k0 + (c % CPR) * 8, K - 8);
      w_now[i] = *reinterpret_cast<const uint4*>(We + (size_t)n * ldw + k);
    }
  };
  auto stash = [&](int buf, int k0, const uint4 (&a_now)[A_CHUNKS], const uint4 (&w_now)[W_CHUNKS]) {
    const uint4 zero = make_uint4(0, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < A_CHUNKS; ++i) {
      const int c = tid + i * 256;
      uint4 v = a_now[i];
      if (k0 + (c % CPR) * 8 >= K) v = zero;
      *reinterpret_cast<uint4*>(a_s[buf] + (c / CPR) * GB_LDS + (c % CPR) * 8) = v;
    }
#pragma unroll
    for (int i = 0; i < W_CHUNKS; ++i) {
      const int c = tid + i * 256;
      uint4 v = w_now[i];
      if (k0 + (c % CPR) * 8 >= K) v = zero;
      *reinterpret_cast<uint4*>(w_s[buf] + (c / CPR) * GB_LDS + (c % CPR) * 8) = v;
    }
  };
#pragma unroll
  for (int j = 0; j < AHEAD; ++j) fetch(j * BK, a_reg[j], w_reg[j]);
  stash(0, 0, a_reg[0], w_reg[0]);
  __syncthreads();
  int buf = 0;
  for (int k_round = 0; k_round < K; k_round += AHEAD * BK) {
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
      const int k0 = k_round + j * BK;
      if (k0 < K) {
        fetch(k0 + AHEAD * BK, a_reg[j], w_reg[j]);
#pragma unroll
        for (int ks = 0; ks < BK; ks += 16) {
          gg_bf16x8 af[TMI], bf[TNI];
#pragma unroll
          for (int i = 0; i < TMI; ++i)
            af[i] = *reinterpret_cast<const gg_bf16x8*>(a_s[buf] + (wm * WM + i * 32 + (lane & 31)) * GB_LDS + ks + 8 * (lane >> 5));
#pragma unroll
          for (int jn = 0; jn < TNI; ++jn)
            bf[jn] = *reinterpret_cast<const gg_bf16x8*>(w_s[buf] + (wn * WN + jn * 32 + (lane & 31)) * GB_LDS + ks + 8 * (lane >> 5));
#pragma unroll
          for (int i = 0; i < TMI; ++i)
#pragma unroll
            for (int jn = 0; jn < TNI; ++jn)
              acc[i][jn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], bf[jn], acc[i][jn], 0, 0, 0);
        }
        if (k0 + BK < K) stash(buf ^ 1, k0 + BK, a_reg[(j + 1) % AHEAD], w_reg[(j + 1) % AHEAD]);
        __syncthreads();
        buf ^= 1;
      }
    }
  }
  // Lane l holds column l%32 and rows 8*(r/4) + 4*(l/32) + r%4 of each 32x32 tile.
#pragma unroll
  for (int i = 0; i < TMI; ++i)
#pragma unroll
    for (int j = 0; j < TNI; ++j) {
      const int n = n0 + wn * WN + j * 32 + (lane & 31);
      if (n >= N) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = m0 + wm * WM + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        gg_store(C + (size_t)m * ldc + n, acc[i][j][r]);
      }
    }
}

// The same for tiles of BM slots and BN columns with the inner loop of tile_ring.h (K a multiple of 32, from 64 on).
// Workgroups run over the tiles up to the last that has slots, in groups of sixteen tiles times all columns; the chiplets (every eighth
// workgroup) get equal runs of that order, so what is under way on one chiplet at a time are sixteen tiles of slots times a few
// strips of columns, and its L2 serves an operand's row several times for one trip from memory.
// Bound by the loads' way into LDS (128 x 256: 48 KB a step of 1,024 clocks of matrix work).  36 tiles of 128 slots over 3,584 x 18,944
// and 9,472 x 3,584: 679 + 327 us, 921 and 955 TFLOP/s; 808 + 402 with rows that went through registers on their way to LDS (256 columns,
// steps of 32), 1,094 + 500 in the kernel above.
// ACT: what becomes of the sums before they are stored.  GROUPED_SILU: an expert's W has N gate rows, then N up rows, and C[slot, :N] =
// silu(gate) * up; GROUPED_WEIGHED: silu(w gate) * (w up), w = weights[p] of the pair p with slot_of[p] = slot, one of the `top` of the
// slot's token; GROUPED_RELU2: max(z, 0)^2.  Gate and up rows lie in LDS sixteen by sixteen, so that a lane has both sums of a column.
// (Two of eight experts of 9,472 on a width of 3,584, 2,048 tokens: product and activation 654 + 30 us, as one 649; whole passes of
// that design 26.3 -> 25.5 ms.)
enum { GROUPED_PLAIN = 0, GROUPED_SILU = 1, GROUPED_WEIGHED = 2, GROUPED_RELU2 = 3 };
template <int BM, int BN, int STAGES, int WN_WAVES, int ACT, typename OutT>
__global__ void __launch_bounds__(128 * WN_WAVES)
grouped_gemm_ring_kernel(const bf16_t* __restrict__ A, int lda, const int* __restrict__ row_of,
                         const int* __restrict__ tile_expert, int n_tiles, const bf16_t* __restrict__ W, long expert_stride,
                         int ldw, OutT* __restrict__ C, int ldc, int N, int K, const int* __restrict__ slot_of,
                         const float* __restrict__ weights, int top) {
  typedef RingTile<BM, BN, STAGES, 2, WN_WAVES> Ring;
  constexpr bool GATED = ACT == GROUPED_SILU || ACT == GROUPED_WEIGHED;
  constexpr int GROUP = 16, COLUMNS = GATED ? BN / 2 : BN;
  const int lane = threadIdx.x & 63, wave = wave_index();
  // The list up to its last tile with slots.
  int used = 0;
  for (int base = 0; base < n_tiles; base += WAVE) {
    const unsigned long long has = __ballot(base + lane < n_tiles && tile_expert[min(base + lane, n_tiles - 1)] >= 0);
    if (has) used = base + WAVE - __clzll(has);
  }
  used = __builtin_amdgcn_readfirstlane(used);
  const int strips = (N + COLUMNS - 1) / COLUMNS, total = used * strips, per_chiplet = (total + 7) / 8;
  const int turn = (int)(blockIdx.x >> 3), place = (int)(blockIdx.x & 7) * per_chiplet + turn;
  if (turn >= per_chiplet || place >= total) return;
  const int first = place / (GROUP * strips) * GROUP, high = min(GROUP, used - first), inside = place - first * strips;
  const int tile = first + inside % high, m0 = tile * BM, n0 = inside / high * COLUMNS;
  const int expert = scalar_int(tile_expert + tile);
  if (expert < 0) return;                                   // (a tile without slots among the others)
  uint32_t a_at[Ring::LA], w_at[Ring::LB];
#pragma unroll
  for (int i = 0; i < Ring::LA; ++i) {
    const int slot = m0 + Ring::load_row(wave, lane, Ring::LA, i);
    a_at[i] = (uint32_t)(row_of ? max(row_of[slot], 0) : slot) * lda * 2 + Ring::piece_bytes(lane);
  }
#pragma unroll
  for (int i = 0; i < Ring::LB; ++i) {
    const int row = Ring::load_row(wave, lane, Ring::LB, i);
    const int n = GATED ? min(n0 + (row >> 5) * 16 + (row & 15), N - 1) + (row & 16 ? N : 0) : min(n0 + row, N - 1);
    w_at[i] = (uint32_t)n * ldw * 2 + Ring::piece_bytes(lane);
  }
  const int r = lane & 15, g = lane >> 4;
  float weight[Ring::MI];
  if constexpr (ACT == GROUPED_WEIGHED) {
#pragma unroll
    for (int i = 0; i < Ring::MI; ++i) {
      const int slot = m0 + wave / WN_WAVES * Ring::WM + 16 * i + r, token = row_of[slot];
      weight[i] = 0.f;                                      // (a slot that only fills the tile up)
      if (token >= 0)
        for (int k = 0; k < top; ++k)
          if (slot_of[token * top + k] == slot) weight[i] = weights[token * top + k];
    }
  }
  ring_floatx4 acc[Ring::MI][Ring::NI];
  Ring::run(A, a_at, W + (size_t)expert * expert_stride, w_at, K / 64, (K & 32) != 0, acc);
#pragma unroll
  for (int i = 0; i < Ring::MI; ++i) {
    OutT* row = C + (size_t)(m0 + wave / WN_WAVES * Ring::WM + 16 * i + r) * ldc;
#pragma unroll
    for (int j = 0; j < Ring::NI; j += GATED ? 2 : 1) {
      const int n = n0 + (GATED ? wave % WN_WAVES * (Ring::WN / 2) + 8 * j : wave % WN_WAVES * Ring::WN + 16 * j) + 4 * g;
      ring_floatx4 v = acc[i][j];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (ACT == GROUPED_SILU) v[e] = v[e] / (1.0f + __expf(-v[e])) * acc[i][j + 1][e];
        if constexpr (ACT == GROUPED_WEIGHED) {
          const float z = weight[i] * v[e];
          v[e] = z / (1.0f + __expf(-z)) * (weight[i] * acc[i][j + 1][e]);
        }
        if constexpr (ACT == GROUPED_RELU2) { const float z = fmaxf(v[e], 0.f); v[e] = z * z; }
      }
      if (n + 3 < N && (ldc & 3) == 0) gg_store4(row + n, v);
      else
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) gg_store(row + n + e, v[e]);
    }
  }
}

// out[t, :] = shared[t, :] (if given; times shared_weight[t], float, if that is given) + sum over the token's picks k of weights[t, k] * rows[slot_of[t * top + k], :]
// (a pick without a slot is passed over).  rows float [*, hidden]; shared and out of type T.
template <typename T>
__global__ void expert_combine_kernel(const float* __restrict__ rows, const int* __restrict__ slot_of,
                                      const float* __restrict__ weights, int top, const T* __restrict__ shared,
                                      T* __restrict__ out, int hidden, size_t total,
                                      const float* __restrict__ shared_weight) {
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (size_t)gridDim.x * blockDim.x) {
    const size_t t = idx / hidden;
    const int h = (int)(idx - t * hidden);
    float sum = shared ? ld(shared + idx) : 0.f;
    if (shared && shared_weight) sum *= shared_weight[t];
    for (int k = 0; k < top; ++k) {
      const int slot = slot_of[t * top + k];
      if (slot >= 0) sum = fmaf(weights ? weights[t * top + k] : 1.f, rows[(size_t)slot * hidden + h], sum);
    }
    st(out + idx, sum);
  }
}

extern "C" int ta_expert_slots(const void* chosen, int n_entries, int top, int n_experts, int bm, int n_tiles,
                               void* slot_of, void* row_of, void* tile_expert, hipStream_t stream) {
  if (n_entries <= 0) return 0;
  if (n_experts <= 0 || n_experts > GG_MAX_EXPERTS || top <= 0 || bm <= 0 || (long)n_tiles * bm < n_entries ||
      n_tiles < (n_entries + bm - 1) / bm + n_experts)
    return -1;
  expert_slots_kernel<<<1, 1024, 0, stream>>>((const int*)chosen, n_entries, top, n_experts, bm, n_tiles, (int*)slot_of,
                                              (int*)row_of, (int*)tile_expert);
  return LAUNCH_STATUS();
}

// Which width: 64 columns (tiles of 64 slots) where even those give no compute unit a second workgroup; else 256 where their
// rounds over the units, each 1.6 times as long, are fewer than those of 128.  Measured, us, 64 | 128 | 256 columns (and the general
// kernel).  64 slots a tile: 12 tiles x 896 columns over 3,648 23 | 32 | 50 (31), 24 tiles 37 | 31 | 47 (42), 40 tiles 48 | 45 | 47 (62);
// 12 tiles x 3,648 columns over 896 20 | 20 | 19 (20); 24 tiles x 3,584 columns over 9,472 261 | 215 | 243 (250), 68 tiles x 18,944
// columns over 3,584 1,178 | 955 | 908 (1,340).  128 slots, 128 | 256 columns: 36 tiles x 18,944 over 3,584 795 | 679 (1,129), 36 x
// 3,584 over 9,472 395 | 327 (502), 8 such tiles 132 | 171 (181); 36 x 896 over 3,648 42 | 58 (73); 18 x 4,480 over 1,536 61 | 62 (68).
// The general kernel is left with a K that is no multiple of 32, one of 32, and matrices past 32-bit places.
static int ring_width(int choice, int bm, int N, int expected) {
  const int units = compute_units();
  auto workgroups = [&](int width) { return (long)((N + width - 1) / width) * expected; };
  auto rounds = [&](int width) { return (double)((workgroups(width) + units - 1) / units); };
  if (choice > 0) return choice == 1 ? 256 : choice;
  return bm == 64 && workgroups(64) <= units ? 64 : rounds(256) * 1.6 < rounds(128) ? 256 : 128;
}

// bm: 64 or 128 (the tile height the slots were made for).  C has n_tiles * bm rows.  expected: about how many of the tiles will
// have slots (it only goes into the choice of kernel).  rows: how many A has.  choice: 0 = the expected fastest, -1 = the general kernel,
// 64, 128 or 256 = the ring kernel with so many columns a tile wherever it can (64 columns: tiles of 64 slots; 128 in their place at
// 128), 1 = with 256.
extern "C" int ta_grouped_gemm_bf16(const void* A, int rows, int lda, const void* row_of, const void* tile_expert, int n_tiles, int bm,
                                    const void* W, long expert_stride, int ldw, void* C, int ldc, int N, int K,
                                    int out_dtype, int expected, int choice, hipStream_t stream) {
  if (n_tiles <= 0 || N <= 0) return 0;
  if ((K & 7) || (lda & 7) || (ldw & 7) || (expert_stride & 7) || K < 8 || (((uintptr_t)A | (uintptr_t)W) & 15)) return -1;
  if (bm != 64 && bm != 128) return -1;
#define GO(BMV, BNV, BKV, TT)                                                                                          \
  grouped_gemm_bf16_kernel<BMV, BNV, BKV, TT><<<dim3((N + BNV - 1) / BNV, n_tiles), 256, 0, stream>>>(                 \
      (const bf16_t*)A, lda, (const int*)row_of, (const int*)tile_expert, (const bf16_t*)W, expert_stride, ldw, (TT*)C, ldc, N, K)
#define RING(BMV, BNV, ST, WAVES, TT) grouped_gemm_ring_kernel<BMV, BNV, ST, WAVES, 0, TT><<<blocks, 128 * WAVES, 0, stream>>>( \
    (const bf16_t*)A, lda, (const int*)row_of, (const int*)tile_expert, n_tiles, (const bf16_t*)W, expert_stride, ldw, (TT*)C, ldc, N, K, \
    nullptr, nullptr, 0)
  const bool ring = choice >= 0 && K % 32 == 0 && K >= 64 && (long)(N - 1) * ldw + K < (1l << 31) && (long)rows * lda < (1l << 31);
  const int width = ring_width(choice, bm, N, expected);
  if (width != 64 && width != 128 && width != 256) return -1;
  const int blocks = ((N + width - 1) / width * n_tiles + 7) / 8 * 8;
  const bool f32 = out_dtype == DT_F32;
  if (ring && bm == 128) {
    if (width == 256) { if (f32) RING(128, 256, 3, 4, float); else RING(128, 256, 3, 4, bf16_t); }
    else if (f32) RING(128, 128, 4, 4, float); else RING(128, 128, 4, 4, bf16_t);
  } else if (ring) {
    if (width == 256) { if (f32) RING(64, 256, 4, 4, float); else RING(64, 256, 4, 4, bf16_t); }
    else if (width == 128) { if (f32) RING(64, 128, 3, 4, float); else RING(64, 128, 3, 4, bf16_t); }
    else if (f32) RING(64, 64, 4, 2, float); else RING(64, 64, 4, 2, bf16_t);
  } else if (bm == 128) { if (f32) GO(128, 128, 32, float); else GO(128, 128, 32, bf16_t); }
  else if (f32) GO(64, 64, 64, float); else GO(64, 64, 64, bf16_t);
#undef RING
#undef GO
  return LAUNCH_STATUS();
}

extern "C" int ta_expert_combine(const void* rows, const void* slot_of, const void* weights, int n_tokens, int top,
                                 const void* shared, void* out, int hidden, int dtype, const void* shared_weight,
                                 hipStream_t stream) {
  const size_t total = (size_t)n_tokens * hidden;
  if (total == 0) return 0;
  const int blocks = (int)((total + 255) / 256 < 65535 ? (total + 255) / 256 : 65535);
  if (dtype == DT_F32)
    expert_combine_kernel<float><<<blocks, 256, 0, stream>>>((const float*)rows, (const int*)slot_of, (const float*)weights,
                                                             top, (const float*)shared, (float*)out, hidden, total,
                                                             (const float*)shared_weight);
  else
    expert_combine_kernel<bf16_t><<<blocks, 256, 0, stream>>>((const float*)rows, (const int*)slot_of, (const float*)weights,
                                                              top, (const bf16_t*)shared, (bf16_t*)out, hidden, total,
                                                              (const float*)shared_weight);
  return LAUNCH_STATUS();
}

// The first product of a routed layer and its activation: C[slot, :inner] (bfloat16) = act over A's rows and the tile's expert, W_e as the
// kernel's ACT says (1: [gate; up] rows, silu; 2: the same with weighted inputs, slot_of, weights [tokens, top] and row_of given; 3: inner rows,
// max(z, 0)^2).  The other arguments as in `ta_grouped_gemm_bf16`.  -2: not these operands (the product and the activation one by one).
extern "C" int ta_grouped_gemm_act(const void* A, int rows, int lda, const void* row_of, const void* tile_expert, int n_tiles, int bm,
                                   const void* W, long expert_stride, int ldw, void* C, int inner, int K, int act, const void* slot_of,
                                   const void* weights, int top, int expected, int choice, hipStream_t stream) {
  if (n_tiles <= 0 || inner <= 0) return 0;
  if (bm != 64 && bm != 128) return -1;
  if (act < 1 || act > 3 || (act == GROUPED_WEIGHED && (!slot_of || !weights || !row_of || top <= 0))) return -1;
  const long w_rows = (act == GROUPED_RELU2 ? 1l : 2l) * inner;
  if (choice < 0 || (K & 31) || K < 64 || (lda & 7) || (ldw & 7) || (expert_stride & 7) || (((uintptr_t)A | (uintptr_t)W | (uintptr_t)C) & 15) ||
      (w_rows - 1) * ldw + K >= (1l << 31) || (long)rows * lda >= (1l << 31) || w_rows > 0x7fffffffL)
    return -2;
  const int width = ring_width(choice, bm, (int)w_rows, expected);
  if (width != 64 && width != 128 && width != 256) return -1;
  const int columns = act == GROUPED_RELU2 ? width : width / 2, blocks = ((inner + columns - 1) / columns * n_tiles + 7) / 8 * 8;
#define RING(BMV, BNV, ST, WAVES, ACT) grouped_gemm_ring_kernel<BMV, BNV, ST, WAVES, ACT, bf16_t><<<blocks, 128 * WAVES, 0, stream>>>( \
    (const bf16_t*)A, lda, (const int*)row_of, (const int*)tile_expert, n_tiles, (const bf16_t*)W, expert_stride, ldw, (bf16_t*)C, inner, \
    inner, K, (const int*)slot_of, (const float*)weights, top)
#define WIDTHS(ACT)                                                                                              \
  {                                                                                                              \
    if (bm == 128) { if (width == 256) RING(128, 256, 3, 4, ACT); else RING(128, 128, 4, 4, ACT); }              \
    else if (width == 256) RING(64, 256, 4, 4, ACT);                                                             \
    else if (width == 128) RING(64, 128, 3, 4, ACT);                                                             \
    else RING(64, 64, 4, 2, ACT);                                                                                \
  }
  if (act == GROUPED_SILU) WIDTHS(GROUPED_SILU) else if (act == GROUPED_WEIGHED) WIDTHS(GROUPED_WEIGHED) else WIDTHS(GROUPED_RELU2)
#undef WIDTHS
#undef RING
  return LAUNCH_STATUS();
}
