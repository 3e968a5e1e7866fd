// Attention over a cached latent: what stands between the joined down-projections and the paged attention kernels
// (the two latents' norms, the rotation of the shared key part, the write of the latent into its pages), products
// head by head with a matrix of the head's own (the query taken into the latent's space, the read-out taken out of
// it), and the rotation of the query heads' tails.
#include "common.h"

#define LT_THREADS 256

// rows: [n_tokens, row_stride].  latent_q[t, :] = rows[t, q_offset : q_offset + q_rank] / rms * q_norm.  The kept row
// of a token is [c | turned tail]: c = rows[t, kv_offset : kv_offset + kv_rank] / rms * kv_norm, and the rot
// coordinates behind it in `rows` with coordinate i < rot / 2 and coordinate i + rot / 2 (neighbours: coordinates 2 i and
// 2 i + 1) turned by the angle position * rates[i] (float).  It goes into key page [n_pages, 1, page_size, kv_rank + rot] at the token's slot and,
// transposed inside a page, into value page [n_pages, 1, kv_rank + rot, page_size].  slots null or a negative slot:
// nothing is stored; without value pages the row goes into its key page alone.
// A workgroup a token and part (blockIdx.y: the queries' latent, the keys'), or with BOTH a workgroup a token, whose first `q_threads` threads
// have the queries' latent and the others the keys'; a part is as many waves as it has elements for, four at most.  A thread keeps its
// PER elements in registers from their one load on (what lies behind PER * LT_THREADS of a longer latent is read again), norm weights,
// position and rates are asked for beside them, and the angles are the last wave's, which has the fewest elements.  (One workgroup for
// both parts one behind the other, each read twice | so, in a graph: four rows of latents of 448 and 96 3.5 | 2.4 us, of 1,792 and 192
// 4.9 | 2.7.)
template <typename T, int PER, bool BOTH>
__global__ void __launch_bounds__(2 * LT_THREADS)
latent_store_kernel(const T* __restrict__ rows, int row_stride, int q_offset, int q_rank, const float* __restrict__ q_norm,
                    int kv_offset, int kv_rank, const float* __restrict__ kv_norm, int rot, const float* __restrict__ rates,
                    float eps, const int* __restrict__ positions, const int* __restrict__ slots, T* __restrict__ k_pages,
                    T* __restrict__ v_pages, int page_size, T* __restrict__ latent_q, int neighbours, int q_threads) {
  HELD(rows, row_stride, q_offset, q_rank, q_norm, kv_offset, kv_rank, kv_norm, rot, rates, eps, positions, slots, k_pages, v_pages,
       page_size, latent_q, neighbours, q_threads);
  __shared__ float scratch[2 * LT_THREADS / WAVE];
  const int t = blockIdx.x, wave = wave_index();
  const bool keys = BOTH ? wave >= q_threads / WAVE : blockIdx.y != 0;
  const int slot = keys ? scalar_int(slots + t) : -1;         // (without slots there is no such part)
  if (!BOTH && keys && slot < 0) return;                      // (the same for every thread of the workgroup)
  const int before = BOTH && keys ? q_threads : 0;            // the part's first thread
  const int rank = keys ? kv_rank : q_rank, tid = threadIdx.x - before, threads = (BOTH && !keys ? q_threads : blockDim.x) - before;
  const T* row = rows + (size_t)t * row_stride;
  const T* from = row + (keys ? kv_offset : q_offset);
  const float* norm = keys ? kv_norm : q_norm;
  T raw[PER];
  float w[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int i = min(j * LT_THREADS + tid, rank - 1);
    raw[j] = from[i];
    w[j] = norm[i];
  }
  const int half = keys ? rot / 2 : 0, turn = tid + WAVE < threads ? tid + WAVE : tid + WAVE - threads;    // (the thread's pair of the tail)
  const T* tail = row + kv_offset + kv_rank;
  float rate = 0.f, position = 0.f;
  T one_raw = {}, other_raw = {};
  if (half > 0) {                                             // (the same for the wave)
    const int i = min(turn, half - 1);
    rate = rates[i];
    one_raw = tail[neighbours ? 2 * i : i];
    other_raw = tail[neighbours ? 2 * i + 1 : half + i];
    position = (float)scalar_int(positions + t);
  }
  float sq = 0.f;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const float v = ld(&raw[j]);
    if (j * LT_THREADS + tid < rank) sq += v * v;
  }
  for (int i = PER * LT_THREADS + tid; i < rank; i += LT_THREADS) { const float v = ld(from + i); sq += v * v; }
  sq = wave_sum(sq);
  if ((threadIdx.x & (WAVE - 1)) == 0) scratch[wave] = sq;
  __syncthreads();
  if (BOTH && keys && slot < 0) return;                       // (the same for the wave)
  float total = 0.f;                                          // (added wave by wave in their order)
#pragma unroll
  for (int j = 0; j < LT_THREADS / WAVE; ++j) total += j < threads / WAVE ? scratch[before / WAVE + j] : 0.f;
  const float inv = 1.0f / sqrtf(total / (float)rank + eps);
  if (!keys) {
    T* dst = latent_q + (size_t)t * q_rank;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int i = j * LT_THREADS + tid;
      if (i < rank) st(dst + i, ld(&raw[j]) * inv * w[j]);
    }
    for (int i = PER * LT_THREADS + tid; i < rank; i += LT_THREADS) st(dst + i, ld(from + i) * inv * norm[i]);
    return;
  }
  const int page = slot / page_size, off = slot % page_size, width = kv_rank + rot;
  T* k_row = k_pages + ((size_t)page * page_size + off) * width;
  T* v_col = v_pages + (size_t)page * width * page_size + off;
  auto put = [&](int i, float c) {
    st(k_row + i, c);
    if (v_pages) st(v_col + (size_t)i * page_size, c);
  };
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int i = j * LT_THREADS + tid;
    if (i < rank) put(i, ld(&raw[j]) * inv * w[j]);
  }
  for (int i = PER * LT_THREADS + tid; i < rank; i += LT_THREADS) put(i, ld(from + i) * inv * norm[i]);
  for (int i = turn; i < half; i += threads) {
    if (i != turn) { rate = rates[i]; one_raw = tail[neighbours ? 2 * i : i]; other_raw = tail[neighbours ? 2 * i + 1 : half + i]; }
    float s, c;
    sincosf(position * rate, &s, &c);
    const float a = ld(&one_raw), b = ld(&other_raw);
    put(kv_rank + (neighbours ? 2 * i : i), a * c - b * s);
    put(kv_rank + (neighbours ? 2 * i + 1 : half + i), b * c + a * s);
  }
}

// out[t, h * out_stride + out_offset + i] for i < rot: the rot coordinates of q[t, h * head_width + tail_offset ...]
// with coordinate i < rot / 2 and coordinate i + rot / 2 (neighbours: coordinates 2 i and 2 i + 1) turned by
// position * rates[i].
template <typename T>
__global__ void __launch_bounds__(LT_THREADS)
rotate_tails_kernel(const T* __restrict__ q, int q_stride, int heads, int head_width, int tail_offset, int rot,
                    const float* __restrict__ rates, const int* __restrict__ positions, T* __restrict__ out, int out_row,
                    int out_stride, int out_offset, int neighbours) {
  const int t = blockIdx.x, half = rot / 2;
  const float position = (float)positions[t];
  for (int idx = threadIdx.x; idx < heads * half; idx += LT_THREADS) {
    const int i = idx % half, h = idx / half;           // (threads side by side share a head and differ in the rate)
    float s, c;
    sincosf(position * rates[i], &s, &c);
    const T* src = q + (size_t)t * q_stride + (size_t)h * head_width + tail_offset;
    T* dst = out + (size_t)t * out_row + (size_t)h * out_stride + out_offset;
    const int one = neighbours ? 2 * i : i, other = neighbours ? 2 * i + 1 : half + i;
    const float a = ld(src + one), b = ld(src + other);
    st(dst + one, a * c - b * s);
    st(dst + other, b * c + a * s);
  }
}

// Products head by head: out[t, h * out_stride + out_offset + n] = sum_k x[t, h * x_stride + x_offset + k] * W[h, n, k],
// W [heads, N, K] contiguous.  Float sums in every dtype.  A workgroup owns 64 rows by 64 columns of one head's
// output; tiles of 16 elements of K go through LDS, and a thread keeps 4 by 4 sums.
#define HL_TILE 64
#define HL_K 16
template <typename T>
__global__ void __launch_bounds__(256)
head_linear_kernel(const T* __restrict__ x, int x_row, int x_stride, int x_offset, const T* __restrict__ W,
                   T* __restrict__ out, int out_row, int out_stride, int out_offset, int M, int N, int K) {
  __shared__ float a_s[HL_K][HL_TILE + 4], w_s[HL_K][HL_TILE + 4];
  const int h = blockIdx.z, m0 = blockIdx.y * HL_TILE, n0 = blockIdx.x * HL_TILE, tid = threadIdx.x;
  const T* a = x + (size_t)h * x_stride + x_offset;
  const T* w = W + (size_t)h * N * K;
  const int tm = (tid / 16) * 4, tn = (tid % 16) * 4;
  float acc[4][4] = {};
  for (int k0 = 0; k0 < K; k0 += HL_K) {
    for (int idx = tid; idx < HL_TILE * HL_K; idx += 256) {
      const int r = idx / HL_K, kk = idx % HL_K;
      const int m = m0 + r, n = n0 + r, k = k0 + kk;
      a_s[kk][r] = (m < M && k < K) ? ld(a + (size_t)m * x_row + k) : 0.f;
      w_s[kk][r] = (n < N && k < K) ? ld(w + (size_t)n * K + k) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < HL_K; ++kk) {
      float av[4], wv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) { av[i] = a_s[kk][tm + i]; wv[i] = w_s[kk][tn + i]; }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(av[i], wv[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + tm + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tn + j;
      if (n < N) st(out + (size_t)m * out_row + (size_t)h * out_stride + out_offset + n, acc[i][j]);
    }
  }
}

// The same on the matrix cores (v_mfma_f32_32x32x16_bf16) for bfloat16 operands whose rows can be read sixteen bytes at
// a time (K, the heads' offsets and the row strides multiples of eight).  A workgroup of four waves owns 64 rows by 64
// columns of a head's output, a wave a 32 by 32 quarter; steps of 32 elements of K go through LDS.
typedef __bf16 lt_bf16x8 __attribute__((ext_vector_type(8)));
typedef float lt_floatx16 __attribute__((ext_vector_type(16)));
#define HM_BK 32
#define HM_LDS (HM_BK + 8)
__global__ void __launch_bounds__(256)
head_linear_mfma_kernel(const bf16_t* __restrict__ x, int x_row, int x_stride, int x_offset, const bf16_t* __restrict__ W,
                        bf16_t* __restrict__ out, int out_row, int out_stride, int out_offset, int M, int N, int K) {
  __shared__ __attribute__((aligned(16))) uint16_t a_s[2][64 * HM_LDS], w_s[2][64 * HM_LDS];
  const int h = blockIdx.z, m0 = blockIdx.y * 64, n0 = blockIdx.x * 64, tid = threadIdx.x, lane = tid & 63;
  const int wave = wave_index(), wm = wave >> 1, wn = wave & 1;
  const bf16_t* a = x + (size_t)h * x_stride + x_offset;
  const bf16_t* w = W + (size_t)h * N * K;
  // A thread brings one piece of sixteen bytes of each tile a step: row tid / 4, piece tid % 4.
  const int r = tid >> 2, piece = (tid & 3) * 8;
  const int am = min(m0 + r, M - 1), wr = min(n0 + r, N - 1);
  lt_floatx16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
  auto fetch = [&](int k0, uint4& av, uint4& wv) {
    const int k = min(k0 + piece, K - 8);
    av = *reinterpret_cast<const uint4*>(a + (size_t)am * x_row + k);
    wv = *reinterpret_cast<const uint4*>(w + (size_t)wr * K + k);
  };
  auto stash = [&](int buf, int k0, uint4 av, uint4 wv) {
    if (k0 + piece >= K) av = wv = make_uint4(0, 0, 0, 0);
    *reinterpret_cast<uint4*>(a_s[buf] + r * HM_LDS + piece) = av;
    *reinterpret_cast<uint4*>(w_s[buf] + r * HM_LDS + piece) = wv;
  };
  uint4 av, wv;
  fetch(0, av, wv);
  stash(0, 0, av, wv);
  __syncthreads();
  int buf = 0;
  for (int k0 = 0; k0 < K; k0 += HM_BK) {
    const bool more = k0 + HM_BK < K;
    if (more) fetch(k0 + HM_BK, av, wv);
#pragma unroll
    for (int ks = 0; ks < HM_BK; ks += 16) {
      const lt_bf16x8 af = *reinterpret_cast<const lt_bf16x8*>(a_s[buf] + (wm * 32 + (lane & 31)) * HM_LDS + ks + 8 * (lane >> 5));
      const lt_bf16x8 bf = *reinterpret_cast<const lt_bf16x8*>(w_s[buf] + (wn * 32 + (lane & 31)) * HM_LDS + ks + 8 * (lane >> 5));
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, bf, acc, 0, 0, 0);
    }
    if (more) stash(buf ^ 1, k0 + HM_BK, av, wv);
    __syncthreads();
    buf ^= 1;
  }
  // Lane l holds column l % 32 and rows 8 (i / 4) + 4 (l / 32) + i % 4 of the wave's 32 by 32 tile.
  const int n = n0 + wn * 32 + (lane & 31);
  if (n < N) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int m = m0 + wm * 32 + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
      if (m < M) st(out + (size_t)m * out_row + (size_t)h * out_stride + out_offset + n, acc[i]);
    }
  }
}

// Few rows (single tokens): a wave owns one output column of one head for up to HS_ROWS rows and reads the column's
// row of W once, sixteen bytes a lane a trip, so that the head's matrix streams from memory once whatever the rows.
// GATED: row m's results, rounded, times sigmoid(gate[m gate_row + h gate_head + n gate_unit]).  The eight sums over the wave share their
// exchanges (`wave_sums8`), and a lane a row stores: eight sums through the LDS crossbar and a lane's eight stores one behind the other were
// half of the kernel, and the gate a kernel of its own.  (Us, one, four and eight rows, 14 heads of 64 over 128: 2.4, 3.3 and 4.5 without the
// gate; 2.3, 2.8 and 3.4 so, 2.6, 3.1 and 3.7 with it; each sum by itself 2.2, 2.9 and 3.7.)
// ROWS: the rows a wave asks for, all of them before the first is multiplied: one behind the other, behind a question whether there is a
// further one, each was a trip.  One behind the other | so, one row, four and eight, 14 heads of 96 over 64: 2.6 | 2.0, 3.1 | 2.35 and
// 3.8 | 2.7; 28 of 192 over 128, four rows 4.4 | 3.1, sixteen 7.1 | 5.5.  (The stores go through the chiplet's cache: a column's sixteen-bit
// values lie apart, and each past the cache by itself cost 1.3 us.)
#define HS_ROWS 8
template <bool GATED, int ROWS>
__global__ void __launch_bounds__(256)
head_linear_skinny_kernel(const bf16_t* __restrict__ x, int x_row, int x_stride, int x_offset, const bf16_t* __restrict__ W,
                          bf16_t* __restrict__ out, int out_row, int out_stride, int out_offset, int M, int N, int K,
                          const bf16_t* __restrict__ gate, int gate_row, int gate_head, int gate_unit) {
  HELD(x, x_row, x_stride, x_offset, W, out, out_row, out_stride, out_offset, M, N, K, gate, gate_row, gate_head, gate_unit);
  const int h = blockIdx.z, lane = threadIdx.x & 63, n = blockIdx.x * 4 + wave_index(), m0 = blockIdx.y * HS_ROWS;
  if (n >= N) return;
  const bf16_t* a = x + (size_t)h * x_stride + x_offset;
  const bf16_t* w = W + ((size_t)h * N + n) * K;
  const int mine = m0 + (lane & 1) + 2 * ((lane >> 4) & 1) + 4 * (lane >> 5);         // the row whose sum ends in this lane
  bf16_t z = {0};
  if (GATED) z = gate[(size_t)min(mine, M - 1) * gate_row + (size_t)h * gate_head + (size_t)n * gate_unit];
  float acc[HS_ROWS] = {};
  for (int k = lane * 8; k < K; k += 64 * 8) {
    const uint4 raw = *reinterpret_cast<const uint4*>(w + k);
    uint4 xa[ROWS];                                          // (past the last row: the last one again, whose sum nobody stores)
#pragma unroll
    for (int i = 0; i < ROWS; ++i) xa[i] = *reinterpret_cast<const uint4*>(a + (size_t)min(m0 + i, M - 1) * x_row + k);
    const uint32_t ww[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      const uint32_t xw[4] = {xa[i].x, xa[i].y, xa[i].z, xa[i].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        acc[i] = fmaf(__uint_as_float(ww[j] << 16), __uint_as_float(xw[j] << 16), acc[i]);
        acc[i] = fmaf(__uint_as_float(ww[j] & 0xffff0000u), __uint_as_float(xw[j] & 0xffff0000u), acc[i]);
      }
    }
  }
  float total = wave_sums8(acc, lane);
  if ((lane & 15) < 2 && mine < M) {
    if (GATED) total = bf16_bits_to_float(float_to_bf16_bits(total)) / (1.0f + expf(-ld(&z)));
    st(out + (size_t)mine * out_row + (size_t)h * out_stride + out_offset + n, total);
  }
}

template <bool GATED>
static int launch_head_skinny(const void* x, int x_row, int x_stride, int x_offset, const void* W, void* out, int out_row, int out_stride,
                              int out_offset, int M, int N, int K, int heads, const void* gate, int gate_row, int gate_head, int gate_unit,
                              hipStream_t stream) {
  const dim3 grid((N + 3) / 4, (M + HS_ROWS - 1) / HS_ROWS, heads);
#define GO(ROWS) head_linear_skinny_kernel<GATED, ROWS><<<grid, 256, 0, stream>>>((const bf16_t*)x, x_row, x_stride, x_offset, (const bf16_t*)W, \
    (bf16_t*)out, out_row, out_stride, out_offset, M, N, K, (const bf16_t*)gate, gate_row, gate_head, gate_unit)
  if (M <= 1) GO(1); else if (M <= 2) GO(2); else if (M <= 4) GO(4); else GO(8);
#undef GO
  return LAUNCH_STATUS();
}

extern "C" int ta_latent_store(const void* rows, int row_stride, int q_offset, int q_rank, const void* q_norm, int kv_offset,
                               int kv_rank, const void* kv_norm, int rot, const void* rates, float eps, const void* positions,
                               const void* slots, void* k_pages, void* v_pages, int page_size, void* latent_q, int n_tokens,
                               int neighbours, int dtype, hipStream_t stream) {
  if (n_tokens <= 0) return 0;
  if (q_rank <= 0 || kv_rank <= 0 || rot < 0 || (rot & 1) || (rot > 0 && !rates) || (slots && (!k_pages || !kv_norm || page_size <= 0)))
    return -1;
  const int most = q_rank > kv_rank ? q_rank : kv_rank;
  auto threads_of = [](int rank) { return rank >= LT_THREADS ? LT_THREADS : (rank + WAVE - 1) / WAVE * WAVE; };
  const int q_threads = threads_of(q_rank), k_threads = threads_of(kv_rank);
  // Many rows whose parts are of different lengths, or short: both in a workgroup, so that none is there for waves without an element.
  // (2,000 rows in bfloat16, latents of 192 and 64, a workgroup a part | one for both: 5.55 | 4.15 us, 64 and 192 6.3 | 5.2, 768 and 64
  // 6.35 | 5.6, but 1,536 and 192 8.3 | 9.0; four rows 2.4 to 3.0 | 0.1 to 0.3 more.)
  const bool both = slots && n_tokens >= 2 * compute_units() && (q_threads < LT_THREADS || k_threads <= LT_THREADS / 2);
  const int threads = both ? q_threads + k_threads : slots && k_threads > q_threads ? k_threads : q_threads;
  const dim3 grid(n_tokens, slots && !both ? 2 : 1);
#define LS_GO(TT, PER, BOTH) latent_store_kernel<TT, PER, BOTH><<<grid, threads, 0, stream>>>((const TT*)rows, row_stride, \
    q_offset, q_rank, (const float*)q_norm, kv_offset, kv_rank, (const float*)kv_norm, rot, (const float*)rates, eps, (const int*)positions, \
    (const int*)slots, (TT*)k_pages, (TT*)v_pages, page_size, (TT*)latent_q, neighbours, q_threads)
#define LS_PER(TT, PER) do { if (both) LS_GO(TT, PER, true); else LS_GO(TT, PER, false); } while (0)
#define LS(TT) do { if (most <= LT_THREADS) LS_PER(TT, 1); else if (most <= 2 * LT_THREADS) LS_PER(TT, 2); \
                    else if (most <= 4 * LT_THREADS) LS_PER(TT, 4); else LS_PER(TT, 8); } while (0)
  if (dtype == DT_F32) LS(float); else LS(bf16_t);
#undef LS
#undef LS_PER
#undef LS_GO
  return LAUNCH_STATUS();
}

extern "C" int ta_rotate_tails(const void* q, int q_stride, int heads, int head_width, int tail_offset, int rot,
                               const void* rates, const void* positions, void* out, int out_row, int out_stride,
                               int out_offset, int n_tokens, int neighbours, int dtype, hipStream_t stream) {
  if (n_tokens <= 0 || rot == 0) return 0;
  if (rot < 0 || (rot & 1) || heads <= 0 || tail_offset + rot > head_width) return -1;
#define RT(TT) rotate_tails_kernel<TT><<<n_tokens, LT_THREADS, 0, stream>>>((const TT*)q, q_stride, heads, head_width, \
    tail_offset, rot, (const float*)rates, (const int*)positions, (TT*)out, out_row, out_stride, out_offset, neighbours)
  if (dtype == DT_F32) RT(float); else RT(bf16_t);
#undef RT
  return LAUNCH_STATUS();
}

extern "C" int ta_head_linear(const void* x, int x_row, int x_stride, int x_offset, const void* W, void* out, int out_row,
                              int out_stride, int out_offset, int M, int N, int K, int heads, int dtype, hipStream_t stream) {
  if (M <= 0 || N <= 0 || heads <= 0) return 0;
  if (K <= 0 || heads > 65535) return -1;
  if (dtype == DT_BF16 && K % 8 == 0 && x_row % 8 == 0 && x_stride % 8 == 0 && x_offset % 8 == 0 &&
      (((uintptr_t)x | (uintptr_t)W) & 15) == 0) {
    if (M <= 2 * HS_ROWS)
      return launch_head_skinny<false>(x, x_row, x_stride, x_offset, W, out, out_row, out_stride, out_offset, M, N, K, heads, nullptr, 0, 0, 0,
                                       stream);
    dim3 grid((N + 63) / 64, (M + 63) / 64, heads);
    if (grid.y > 65535) return -1;
    head_linear_mfma_kernel<<<grid, 256, 0, stream>>>((const bf16_t*)x, x_row, x_stride, x_offset, (const bf16_t*)W,
                                                      (bf16_t*)out, out_row, out_stride, out_offset, M, N, K);
    return LAUNCH_STATUS();
  }
  dim3 grid((N + HL_TILE - 1) / HL_TILE, (M + HL_TILE - 1) / HL_TILE, heads);
  if (grid.y > 65535) return -1;
#define HL(TT) head_linear_kernel<TT><<<grid, 256, 0, stream>>>((const TT*)x, x_row, x_stride, x_offset, (const TT*)W, \
    (TT*)out, out_row, out_stride, out_offset, M, N, K)
  if (dtype == DT_F32) HL(float); else HL(bf16_t);
#undef HL
  return LAUNCH_STATUS();
}

// The same for up to sixteen aligned bfloat16 rows, the results times sigmoid(gate[m gate_row + h gate_head + n gate_unit]); -2 where the caller
// runs the product and the gate one behind the other.
extern "C" int ta_head_linear_gated(const void* x, int x_row, int x_stride, int x_offset, const void* W, void* out, int out_row,
                                    int out_stride, int out_offset, const void* gate, int gate_row, int gate_head, int gate_unit,
                                    int M, int N, int K, int heads, int dtype, hipStream_t stream) {
  if (M <= 0 || N <= 0 || heads <= 0) return 0;
  if (K <= 0 || heads > 65535 || !gate) return -1;
  if (dtype != DT_BF16 || M > 2 * HS_ROWS || K % 8 || x_row % 8 || x_stride % 8 || x_offset % 8 || (((uintptr_t)x | (uintptr_t)W) & 15)) return -2;
  return launch_head_skinny<true>(x, x_row, x_stride, x_offset, W, out, out_row, out_stride, out_offset, M, N, K, heads, gate, gate_row, gate_head,
                                  gate_unit, stream);
}
