// Products of a routed feed-forward over sorted tokens: every tile of BM rows belongs to one expert and is multiplied
// with that expert's matrix alone.  bfloat16 operands, float accumulation on the matrix cores
// (v_mfma_f32_32x32x16_bf16), staged through LDS as in gemm_bf16.hip; and the two small kernels around them: the one
// that sorts a step's (token, chosen expert) pairs into such tiles, and the one that adds a token's experts up.
#include "common.h"
#include <type_traits>

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

// The same for tiles of BM slots and 256 columns, K in steps of 32 (a multiple of 32 here).  A wave owns 64 columns and all the
// slots.  Three steps' rows are on their way to registers, the next step's lie in the other of two buffers in LDS, whose
// rows of 64 bytes keep their four pieces XOR-swizzled by the row (no bank is asked twice by the eight lanes that a read or
// a write serves at a time); the fragments of the next two blocks of slots are read while two are multiplied.
// Rounds of three steps run without a branch, so that the compiler counts the loads under way and waits for the oldest alone.
// Workgroups run over the tiles up to the last that has slots, in groups of sixteen tiles times all columns; the chiplets (every eighth
// workgroup) get equal runs of that order, so what is under way on one chiplet at a time are sixteen tiles of slots times a few
// strips of columns, and its L2 serves an operand's row several times for one trip from memory.
// Bound by LDS and the vector memory pipe together (12 KB of fragments and 6 KB of rows a wave for 512 clocks of matrix work).
// (2,048 tokens, two of eight experts of 9,472 on a width of 3,584: both products 958 + 482 us in the kernel above, 739 + 394
// here, 750 TFLOP/s.  The weights' fragments straight from memory, past LDS: 885 + 440, since neighbouring lanes then name
// different rows and the pipe takes such loads lane by lane.)
template <int BM, typename OutT, int AHEAD = 3>
__global__ void __launch_bounds__(256, 2)
grouped_gemm_wide_kernel(const bf16_t* __restrict__ A, int lda, const int* __restrict__ row_of,
                         const int* __restrict__ tile_expert, int n_tiles, const bf16_t* __restrict__ W, long expert_stride,
                         int ldw, OutT* __restrict__ C, int ldc, int N, int K) {
  constexpr int BN = 256, BK = 32, GROUP = 16, PA = BM / 64, BLOCKS = BM / 16;
  __shared__ __attribute__((aligned(16))) uint16_t a_s[2][BM * BK];
  __shared__ __attribute__((aligned(16))) uint16_t w_s[2][BN * BK];
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_index(), r = lane & 15, g = lane >> 4;
  // The list up to its last tile with slots.
  int used = 0;
  for (int base = 0; base < n_tiles; base += WAVE) {
    const unsigned long long has = __ballot(base + lane < n_tiles && tile_expert[min(base + lane, n_tiles - 1)] >= 0);
    if (has) used = base + WAVE - __clzll(has);
  }
  used = __builtin_amdgcn_readfirstlane(used);
  const int strips = (N + BN - 1) / BN, total = used * strips, per_chiplet = (total + 7) / 8;
  const int turn = (int)(blockIdx.x >> 3), place = (int)(blockIdx.x & 7) * per_chiplet + turn;
  if (turn >= per_chiplet || place >= total) return;
  const int first = place / (GROUP * strips) * GROUP, high = min(GROUP, used - first), inside = place - first * strips;
  const int tile = first + inside % high, m0 = tile * BM, n0 = inside / high * BN;
  const int expert = scalar_int(tile_expert + tile);
  if (expert < 0) return;                                   // (a tile without slots among the others)
  const bf16_t* We = W + (size_t)expert * expert_stride;
  // A thread brings pieces of sixteen bytes of rows tid / 4, 64 further, ...: four neighbours a row's 64 bytes.  Places are
  // 32-bit offsets from a pointer that is the same for the workgroup and moves along K.
  uint32_t a_at[PA], w_at[4];
#pragma unroll
  for (int i = 0; i < PA; ++i) {
    const int slot = m0 + (tid >> 2) + 64 * i;
    a_at[i] = ((uint32_t)(row_of ? max(row_of[slot], 0) : slot) * lda + (tid & 3) * 8) * 2;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) w_at[j] = ((uint32_t)min(n0 + (tid >> 2) + 64 * j, N - 1) * ldw + (tid & 3) * 8) * 2;
  gg_floatx4 acc[BLOCKS][4];
#pragma unroll
  for (int i = 0; i < BLOCKS; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = gg_floatx4{0.f, 0.f, 0.f, 0.f};
  word4 a_reg[AHEAD][PA], w_reg[AHEAD][4];
  const int steps = K / BK;
  typedef const char __attribute__((address_space(1)))* memory;
  typedef const word4 __attribute__((address_space(1)))* pieces;
  auto fetch = [&](int step, word4 (&a_now)[PA], word4 (&w_now)[4]) {
    // (Past the last step it is asked for again: a valid place, never used.)
    const size_t along = (size_t)min(step, steps - 1) * (2 * BK);
    memory a_base = (memory)(uintptr_t)A + along, w_base = (memory)(uintptr_t)We + along;
    asm("" : "+s"(a_base), "+s"(w_base));
#pragma unroll
    for (int i = 0; i < PA; ++i) a_now[i] = *(pieces)(a_base + a_at[i]);
#pragma unroll
    for (int j = 0; j < 4; ++j) w_now[j] = *(pieces)(w_base + w_at[j]);
  };
  const int put_at = (tid >> 2) * BK + ((tid & 3) ^ ((tid >> 3) & 3)) * 8;         // (rows 64 apart are swizzled alike)
  auto stash = [&](int buf, const word4 (&a_now)[PA], const word4 (&w_now)[4]) {
#pragma unroll
    for (int i = 0; i < PA; ++i) *reinterpret_cast<word4*>(a_s[buf] + put_at + 64 * BK * i) = a_now[i];
#pragma unroll
    for (int j = 0; j < 4; ++j) *reinterpret_cast<word4*>(w_s[buf] + put_at + 64 * BK * j) = w_now[j];
  };
#pragma unroll
  for (int j = 0; j < AHEAD; ++j) fetch(j, a_reg[j], w_reg[j]);
  stash(0, a_reg[0], w_reg[0]);
  __syncthreads();
  int buf = 0;
  const int get_at = r * BK + (g ^ ((r >> 1) & 3)) * 8;
  auto one = [&](int step, auto which) {
    constexpr int j = decltype(which)::value, next = (j + 1) % AHEAD;
    fetch(step + AHEAD, a_reg[j], w_reg[j]);
    __builtin_amdgcn_sched_barrier(0);
    stash(buf ^ 1, a_reg[next], w_reg[next]);                // (its readers passed the barrier of the step before)
    gg_bf16x8 wf[4], af[2][2];
    auto read = [&](int pair, gg_bf16x8 (&now)[2]) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
        now[i] = *reinterpret_cast<const gg_bf16x8*>(a_s[buf] + (pair * 2 + i) * 16 * BK + get_at);
    };
#pragma unroll
    for (int n = 0; n < 4; ++n) wf[n] = *reinterpret_cast<const gg_bf16x8*>(w_s[buf] + (wave * 64 + n * 16) * BK + get_at);
    read(0, af[0]);
#pragma unroll
    for (int pair = 0; pair < BLOCKS / 2; ++pair) {
      if (pair + 1 < BLOCKS / 2) read(pair + 1, af[(pair + 1) & 1]);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int n = 0; n < 4; ++n)
          acc[pair * 2 + i][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[n], af[pair & 1][i], acc[pair * 2 + i][n], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    buf ^= 1;
  };
  static_assert(AHEAD == 3);
  int step = 0;
  for (; step + AHEAD <= steps; step += AHEAD) {
    one(step, std::integral_constant<int, 0>{});
    one(step + 1, std::integral_constant<int, 1>{});
    one(step + 2, std::integral_constant<int, 2>{});
  }
  if (step < steps) one(step, std::integral_constant<int, 0>{});
  if (step + 1 < steps) one(step + 1, std::integral_constant<int, 1>{});
  // Weight rows are the instruction's rows: a lane holds columns 4 g .. 4 g + 3 of slot r of each block of sixteen.
#pragma unroll
  for (int i = 0; i < BLOCKS; ++i) {
    OutT* row = C + (size_t)(m0 + 16 * i + r) * ldc;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + wave * 64 + 16 * j + 4 * g;
      if (n + 3 < N && (ldc & 3) == 0) gg_store4(row + n, acc[i][j]);
      else
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) gg_store(row + n + e, acc[i][j][e]);
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

// bm: 64 or 128 (the tile height the slots were made for).  C has n_tiles * bm rows.  expected: about how many of the tiles will
// have slots (the launch's sizes do not depend on it).  rows: how many A has.  choice: 1 = the wide kernel wherever it can, -1 = never,
// 0 = where it is expected to be the faster one.
extern "C" int ta_grouped_gemm_bf16(const void* A, int rows, int lda, const void* row_of, const void* tile_expert, int n_tiles, int bm,
                                    const void* W, long expert_stride, int ldw, void* C, int ldc, int N, int K,
                                    int out_dtype, int expected, int choice, hipStream_t stream) {
  if (n_tiles <= 0 || N <= 0) return 0;
  if ((K & 7) || (lda & 7) || (ldw & 7) || (expert_stride & 7) || K < 8 || (((uintptr_t)A | (uintptr_t)W) & 15)) return -1;
  if (bm != 64 && bm != 128) return -1;
#define GO(BMV, BNV, BKV, TT)                                                                                          \
  grouped_gemm_bf16_kernel<BMV, BNV, BKV, TT><<<dim3((N + BNV - 1) / BNV, n_tiles), 256, 0, stream>>>(                 \
      (const bf16_t*)A, lda, (const int*)row_of, (const int*)tile_expert, (const bf16_t*)W, expert_stride, ldw, (TT*)C, ldc, N, K)
#define WIDE(BMV, TT) grouped_gemm_wide_kernel<BMV, TT><<<blocks, 256, 0, stream>>>((const bf16_t*)A, lda, (const int*)row_of, \
    (const int*)tile_expert, n_tiles, (const bf16_t*)W, expert_stride, ldw, (TT*)C, ldc, N, K)
  // Which kernel: by the rounds of workgroups that each needs over the compute units, a round of wide tiles as long as 1.65 of
  // 128 x 128 ones or 3.15 of 64 x 64 ones (for twice and four times the work).  Measured at 128 slots a tile, us, this | the wide
  // one: 36 tiles x 18,944 columns over 3,584 958 | 739, 3,584 columns over 9,472 482 | 394, 8 tiles of those 178 | 207; 36 tiles x
  // 4,480 columns over 1,536 114 | 100, 18 tiles 67 | 71; 36 tiles x 896 columns over 3,648 70 | 72.  At 64: 68 tiles x 18,944
  // columns over 3,584 1,276 | 1,018, 24 480 | 434; 24 tiles x 3,584 columns over 9,472 243 | 298.
  const int units = compute_units(), strips = (N + 255) / 256, blocks = (strips * n_tiles + 7) / 8 * 8;
  auto rounds = [&](int width) { return (int)(((long)((N + width - 1) / width) * expected + units - 1) / units); };
  const bool wide = K % 32 == 0 && (long)(N - 1) * ldw + K < (1l << 31) && (long)rows * lda < (1l << 31) &&
                    (choice > 0 || (choice == 0 && rounds(256) * (bm == 128 ? 1.65 : 3.15) < rounds(bm)));
  if (wide) {
    if (bm == 128) { if (out_dtype == DT_F32) WIDE(128, float); else WIDE(128, bf16_t); }
    else if (out_dtype == DT_F32) WIDE(64, float); else WIDE(64, bf16_t);
  } else if (bm == 128) { if (out_dtype == DT_F32) GO(128, 128, 32, float); else GO(128, 128, 32, bf16_t); }
  else if (out_dtype == DT_F32) GO(64, 64, 64, float); else GO(64, 64, 64, bf16_t);
#undef WIDE
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
