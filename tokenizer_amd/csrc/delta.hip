// Gated delta rule with a decay per key channel, over a batch of portions, with the state of every request in its
// slot: the short causal convolutions in front of it (with silu) and the recurrence itself.  Unit vectors, gates,
// decays and the state are float in every dtype.  A state row is
// [heads * d * dv (S, per head [d, dv]) | (taps - 1) * channels (the convolutions' last inputs, oldest first) | ...].
#include "common.h"

#define DL_GROUP 16          // tokens whose q, k, decays (and v) are brought into LDS in one trip
#define DL_MAX_D 256
#define DL_MAX_TAPS 16

// x summed over the sixteen lanes of a row (lanes 16 i .. 16 i + 15), in every lane of the row: four rotations within the
// row, which cost no trip through LDS.
__device__ __forceinline__ float dl_row_sum16(float x) {
#define DL_ROR(n) __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x120 | (n), 0xF, 0xF, false))
  x += DL_ROR(8);
  x += DL_ROR(4);
  x += DL_ROR(2);
  x += DL_ROR(1);
#undef DL_ROR
  return x;
}

// x summed over the wave's lanes, in a scalar: the rows' sums, carried from row to row (lane 15 into the next row, lane 31 into the upper half).
__device__ __forceinline__ float dl_wave_sum(float x) {
  x = dl_row_sum16(x);
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x142, 0xA, 0xF, false));
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x143, 0xC, 0xF, false));
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}

__device__ __forceinline__ float dl_softplus(float z) { return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))); }

// Up to three runs of columns of `rows` (run i: `width[i]` columns from `offset[i]` on) are the channels, side by side.
struct ConvRuns { int offset[3]; int width[3]; };

__device__ __forceinline__ int conv_column(const ConvRuns& runs, int c) {
  if (c < runs.width[0]) return runs.offset[0] + c;
  c -= runs.width[0];
  if (c < runs.width[1]) return runs.offset[1] + c;
  return runs.offset[2] + c - runs.width[1];
}

// out[t, c] = silu(bias[c] + sum_j taps[c, j] * x[t - (n_taps - 1) + j, c]) (bias float [channels], or null): inputs before the portion's first row come from the
// entry's state row (its last n_taps - 1 inputs, oldest first), and are zeros if the portion starts at position 0.
// A thread a (token, channel); blockIdx.x is the token.
template <typename T>
__global__ void __launch_bounds__(256)
short_conv_silu_kernel(const T* __restrict__ rows, int row_stride, ConvRuns runs, int channels, const float* __restrict__ taps,
                       int n_taps, const float* __restrict__ state, size_t state_stride, int state_offset,
                       const int* __restrict__ cu_q, const int* __restrict__ first_position,
                       const int* __restrict__ state_slots, const int* __restrict__ entry_of_token, T* __restrict__ out,
                       const float* __restrict__ bias) {
  const int t = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
  if (c >= channels) return;
  const int e = entry_of_token[t];
  if (e < 0) {                                               // a token that only fills the batch up
    st(out + (size_t)t * channels + c, 0.f);
    return;
  }
  const int lo = cu_q[e];
  const bool zeros = first_position[e] == 0;
  const float* tail = state + (size_t)state_slots[e] * state_stride + state_offset;
  const int column = conv_column(runs, c);
  float y = bias ? bias[c] : 0.f;
  for (int j = 0; j < n_taps; ++j) {
    const int src = t - (n_taps - 1) + j;
    float x;
    if (src >= lo) x = ld(rows + (size_t)src * row_stride + column);
    else x = zeros ? 0.f : tail[(size_t)(src - lo + n_taps - 1) * channels + c];
    y = fmaf(taps[(size_t)c * n_taps + j], x, y);
  }
  st(out + (size_t)t * channels + c, y / (1.0f + expf(-y)));
}

// The entry's last n_taps - 1 inputs become its state row's: a thread an (entry, channel) moves what stays of the old
// ones forward (reading ahead of what it writes) and puts the portion's last rows behind them.
template <typename T>
__global__ void __launch_bounds__(256)
short_conv_keep_kernel(const T* __restrict__ rows, int row_stride, ConvRuns runs, int channels, int n_taps,
                       float* __restrict__ state, size_t state_stride, int state_offset, const int* __restrict__ cu_q,
                       const int* __restrict__ first_position, const int* __restrict__ state_slots) {
  const int e = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
  if (c >= channels) return;
  const int lo = cu_q[e], hi = cu_q[e + 1], n = hi - lo, keep = n_taps - 1;
  if (n <= 0) return;
  const bool zeros = first_position[e] == 0;
  float* tail = state + (size_t)state_slots[e] * state_stride + state_offset;
  const int column = conv_column(runs, c);
  for (int i = 0; i < keep; ++i) {
    const int at = i + n;                          // the place in [old inputs | the portion's rows]
    float x;
    if (at < keep) x = zeros ? 0.f : tail[(size_t)at * channels + c];
    else x = ld(rows + (size_t)(lo + at - keep) * row_stride + column);
    tail[(size_t)i * channels + c] = x;
  }
}

// Both for steps of about a token an entry: a thread an (entry, channel) has the entry's last inputs in registers, walks its rows and leaves the
// last inputs behind.  One kernel and two trips to memory (the entry's numbers, then all it reads) where the two above are two kernels of
// four trips and more, 5.3 + 2.6 us (896 channels, two entries) and 6.5 + 5.0 (2,688, four) where they were profiled.
template <typename T, int TAPS>
__global__ void __launch_bounds__(256)
short_conv_step_kernel(const T* __restrict__ rows, int row_stride, ConvRuns runs, int channels, const float* __restrict__ taps,
                       float* __restrict__ state, size_t state_stride, int state_offset, const int* __restrict__ cu_q,
                       const int* __restrict__ first_position, const int* __restrict__ state_slots,
                       const int* __restrict__ entry_of_token, T* __restrict__ out, const float* __restrict__ bias, int n_tokens,
                       int n_entries) {
  const int e = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
  if (e < n_tokens && c < channels && scalar_int(entry_of_token + e) < 0) st(out + (size_t)e * channels + c, 0.f);   // a token that only fills up
  if (e >= n_entries || c >= channels) return;
  const int lo = scalar_int(cu_q + e), hi = scalar_int(cu_q + e + 1), first = scalar_int(first_position + e);
  if (hi <= lo) return;
  float* tail = state + (size_t)scalar_int(state_slots + e) * state_stride + state_offset + c;
  const T* x_at = rows + conv_column(runs, c);
  const float start = bias ? bias[c] : 0.f;
  float tap[TAPS], kept[TAPS - 1];
  T raw = x_at[(size_t)lo * row_stride];
#pragma unroll
  for (int j = 0; j < TAPS; ++j) tap[j] = taps[(size_t)c * TAPS + j];
#pragma unroll
  for (int i = 0; i + 1 < TAPS; ++i) kept[i] = tail[(size_t)i * channels];
  if (first == 0) {
#pragma unroll
    for (int i = 0; i + 1 < TAPS; ++i) kept[i] = 0.f;
  }
  for (int t = lo; t < hi; ++t) {
    const float x = ld(&raw);
    if (t + 1 < hi) raw = x_at[(size_t)(t + 1) * row_stride];
    float y = start;
#pragma unroll
    for (int j = 0; j + 1 < TAPS; ++j) y = fmaf(tap[j], kept[j], y);
    y = fmaf(tap[TAPS - 1], x, y);
#pragma unroll
    for (int i = 0; i + 2 < TAPS; ++i) kept[i] = kept[i + 1];
    kept[TAPS - 2] = x;
    st(out + (size_t)t * channels + c, y / (1.0f + expf(-y)));
  }
#pragma unroll
  for (int i = 0; i + 1 < TAPS; ++i) tail[(size_t)i * channels] = kept[i];
}

// Long portions walk in blocks of DL_BLOCK tokens, counted from the portion's first, on the float matrix instructions.  With S the state before
// a block and G_i the product of the block's decays up to token i (row by row), token i's a_i = k_i . S_(i-1) decayed is
// (k_i G_i) . S + sum over j < i of c_ij u_j, where c_ij = k_i . (k_j times the decays behind j up to i), and its read-out likewise with q_i and
// D_ij (D_ii = q_i . k_i); u_i = beta_i (v_i - a_i).  So with y = v - (k G) S: u = T y, T = (1 + beta c)^(-1) beta, read-out = (q G) S + (D T) y, and the
// state behind the block is G_last S + sum_j e_j u_j, e_j = k_j times the decays behind j.  T and D T are lower triangular, a head's own and the
// same for all columns of S.  Decays are only ever multiplied: nothing is divided by them.
// This kernel makes all that does not depend on the state, for every block side by side: a wave a (block, head), a lane R rows of it.
// EACH 0: all blocks of all portions; else blocks FIRST .. FIRST + EACH - 1 of every portion, for steps whose records are more than their room.
// A block's record (number cu_q[e] / 8 + e + its number in the portion, which no two share; else EACH e + its number among those) of
// 25 DP + 128 floats, DP = d filled up to a multiple of 16 with zeros: [16 rows of DP: row 4 (a / 2) + a % 2 k G of token a, two further on its q G | e of token 2 g + s, row
// 16 b + i: place (16 g + i) DP / 8 + 2 b + s | G_last | T and D T: place 2 (16 g + row) + s, row as above with T and D T for k G and q G, column
// token 2 g + s].  Tokens past the end are zeros.
#define DL_BLOCK 8
#define DL_RECORD(dp) (25 * (dp) + 128)
template <typename T, int R>
__global__ void __launch_bounds__(4 * WAVE)
delta_blocks_kernel(const T* __restrict__ fresh, int fresh_stride, const float* __restrict__ z, const float* __restrict__ neg_rate,
                    const T* __restrict__ beta_rows, int beta_stride, int beta_offset, float* __restrict__ prep,
                    const int* __restrict__ cu_q, int n_entries, int heads, int groups, int d, int dp, float unit_eps, int first,
                    int each) {
  const int block = blockIdx.x, lane = threadIdx.x & (WAVE - 1), h = blockIdx.y * 4 + wave_index();
  int e, number;
  if (each > 0) {
    e = block / each;
    number = first + block % each;
  } else {
    int from = 0;                                            // portions whose blocks' numbers begin at this one's or before
    for (int i = lane; i < n_entries; i += WAVE) from += cu_q[i] / DL_BLOCK + i <= block ? 1 : 0;
#pragma unroll
    for (int off = WAVE / 2; off > 0; off >>= 1) from += __shfl_xor(from, off, WAVE);
    e = __builtin_amdgcn_readfirstlane(from) - 1;            // (the first portion's begin at 0)
    number = block - cu_q[e] / DL_BLOCK - e;
  }
  const int t = cu_q[e] + number * DL_BLOCK, count = min(DL_BLOCK, cu_q[e + 1] - t);
  if (count <= 0 || h >= heads) return;
  const float q_scale = 1.0f / sqrtf((float)d), rate = neg_rate[h];
  const int grp = h / (heads / groups);
  float q[DL_BLOCK][R], k[DL_BLOCK][R], g[DL_BLOCK][R], beta[DL_BLOCK];
  T raw_q[DL_BLOCK][R], raw_k[DL_BLOCK][R], raw_beta[DL_BLOCK];
#pragma unroll
  for (int i = 0; i < DL_BLOCK; ++i) {
    const size_t at = t + min(i, count - 1);                 // (every load is made, from a place inside)
    raw_beta[i] = beta_rows[at * beta_stride + beta_offset + h];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int j = min(lane + WAVE * r, d - 1);
      const T* x = fresh + at * fresh_stride + (size_t)grp * d + j;
      raw_q[i][r] = x[0];
      raw_k[i][r] = x[(size_t)groups * d];
      g[i][r] = z[at * heads * d + (size_t)h * d + j];
    }
  }
#pragma unroll
  for (int i = 0; i < DL_BLOCK; ++i) {
    beta[i] = i < count ? 1.0f / (1.0f + expf(-ld(&raw_beta[i]))) : 0.f;
    float sq = 0.f, sk = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const bool in = i < count && lane + WAVE * r < d;
      q[i][r] = in ? ld(&raw_q[i][r]) : 0.f;
      k[i][r] = in ? ld(&raw_k[i][r]) : 0.f;
      g[i][r] = in ? expf(rate * dl_softplus(g[i][r])) : 1.f;
      sq = fmaf(q[i][r], q[i][r], sq);
      sk = fmaf(k[i][r], k[i][r], sk);
    }
    sq = dl_wave_sum(sq);
    sk = dl_wave_sum(sk);
    const float inv_q = i < count ? q_scale / sqrtf(sq + unit_eps) : 0.f, inv_k = i < count ? 1.0f / sqrtf(sk + unit_eps) : 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) { q[i][r] *= inv_q; k[i][r] *= inv_k; }
  }
  float c[DL_BLOCK][DL_BLOCK], dd[DL_BLOCK][DL_BLOCK];
#pragma unroll
  for (int j = 0; j < DL_BLOCK; ++j) {
    float w[R];
#pragma unroll
    for (int r = 0; r < R; ++r) w[r] = k[j][r];
#pragma unroll
    for (int i = j; i < DL_BLOCK; ++i) {
      float kk = 0.f, qk = 0.f;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (i > j) w[r] *= g[i][r];
        kk = fmaf(k[i][r], w[r], kk);
        qk = fmaf(q[i][r], w[r], qk);
      }
      c[i][j] = i > j ? dl_wave_sum(kk) : 0.f;
      dd[i][j] = dl_wave_sum(qk);
    }
  }
  float* out = prep + ((size_t)block * heads + h) * DL_RECORD(dp);
  // Lane j: column j of T, top to bottom, and of D T.
  float x[DL_BLOCK], y[DL_BLOCK];
#pragma unroll
  for (int i = 0; i < DL_BLOCK; ++i) {
    float sum = 0.f;
#pragma unroll
    for (int l = 0; l < i; ++l) sum = fmaf(c[i][l], x[l], sum);
    x[i] = lane == i ? beta[i] : lane < i ? -beta[i] * sum : 0.f;
  }
#pragma unroll
  for (int i = 0; i < DL_BLOCK; ++i) {
    y[i] = 0.f;
#pragma unroll
    for (int l = 0; l <= i; ++l) y[i] = fmaf(dd[i][l], x[l], y[i]);
  }
  if (lane < DL_BLOCK) {
    float* numbers = out + 25 * dp + 32 * (lane >> 1) + (lane & 1);
#pragma unroll
    for (int i = 0; i < DL_BLOCK; ++i) {
      numbers[2 * (4 * (i >> 1) + (i & 1))] = x[i];
      numbers[2 * (4 * (i >> 1) + (i & 1) + 2)] = y[i];
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int j = lane + WAVE * r;                           // (rows past d are zeros, whose decays multiply nothing)
    if (j >= dp) continue;
    float product = 1.f, behind = 1.f;
#pragma unroll
    for (int i = 0; i < DL_BLOCK; ++i) {
      product *= g[i][r];
      out[(size_t)(4 * (i >> 1) + (i & 1)) * dp + j] = k[i][r] * product;
      out[(size_t)(4 * (i >> 1) + (i & 1) + 2) * dp + j] = q[i][r] * product;
    }
    out[24 * dp + j] = product;
#pragma unroll
    for (int i = DL_BLOCK - 1; i >= 0; --i) {
      out[16 * dp + (16 * (i >> 1) + (j & 15)) * (dp / 8) + 2 * (j >> 4) + (i & 1)] = k[i][r] * behind;
      behind *= g[i][r];
    }
  }
}

// The walk over a portion's blocks: a wave has sixteen columns of S to itself (S[b][r] of lane (col, g): row 16 b + 4 g + r, which is at once the
// result's place of one 16x16x4 instruction and the right operand's of the next), so that nothing is exchanged and nothing waited for but
// the records, AHEAD of which are on their way: every load is made, from a place inside, since a load behind a condition or a value
// converted where it arrives makes the wave wait for all that is under way.  Per block DP / 4 instructions for (k G, q G) S, two for
// (T, D T) y, DP / 2 for the state's update: at d = 64 26 of 32 clocks for eight tokens.  Bound by their chain: 0.9 us a block
// where token by token eight took 1.6, a chain of some two dozen dependent instructions and two sums over lanes each.
// (Both kernels, us: what had the same prepared token by token and then walked token by token | so.  One portion of 2,048 tokens, 14 heads of
// 64 395 | 234, 12 of 128 539 | 391, eight of 256 2,167 | 1,058; portions of 150 to 1,000 tokens 198 | 136, 319 | 209, 1,878 | 541; 32 portions
// of 200 tokens 169 | 105, 438 | 207, 3,078 | 546; one of 300 beside fifteen single tokens 120 | 53, 283 | 138, 2,204 | 343.)
typedef float dl_x4 __attribute__((ext_vector_type(4)));
template <typename T, int NB>
__global__ void __launch_bounds__(4 * WAVE, 1)
delta_walk_kernel(const T* __restrict__ fresh, int fresh_stride, const float* __restrict__ prep, float* __restrict__ state,
                  size_t state_stride, const int* __restrict__ cu_q, const int* __restrict__ first_position,
                  const int* __restrict__ state_slots, float* __restrict__ out, int heads, int groups, int d, int dv, int first,
                  int each) {
  constexpr int DP = 16 * NB, AHEAD = NB <= 8 ? 2 : 1;
  const int e = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & (WAVE - 1), col = lane & 15, g = lane >> 4;
  const int lo = cu_q[e], hi = cu_q[e + 1], first_col = ((int)blockIdx.z * 4 + wave_index()) * 16;
  if (hi <= lo || first_col >= dv) return;                   // (the same for the whole wave)
  const int c = first_col + col, all = (hi - lo + DL_BLOCK - 1) / DL_BLOCK, blocks = each > 0 ? min(all, first + each) : all;
  if (first >= blocks) return;                               // (its last block is behind it)
  const bool live = c < dv;
  float* mem = state + (size_t)state_slots[e] * state_stride + (size_t)h * d * dv;
  const bool from_zero = first == 0 && first_position[e] == 0;
  dl_x4 S[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = 16 * b + 4 * g + r;
      S[b][r] = (!from_zero && live && j < d) ? mem[(size_t)j * dv + c] : 0.f;
    }
  const float* mine = prep + ((size_t)(each > 0 ? each * e : lo / DL_BLOCK + e) * heads + h) * DL_RECORD(DP);
  const size_t record = (size_t)heads * DL_RECORD(DP);
  const T* values = fresh + (size_t)2 * groups * d + (size_t)h * dv + min(c, dv - 1);
  typedef float dl_x2 __attribute__((ext_vector_type(2)));
  struct Block { dl_x4 rows[NB], decay[NB]; float back[NB][2]; dl_x2 number; T v[2]; };
  auto fetch = [&](Block& x, int asked) {
    const int n = min(asked, blocks - 1);
    const float* at = mine + (n - first) * record;
#pragma unroll
    for (int b = 0; b < NB; ++b) x.rows[b] = *reinterpret_cast<const dl_x4*>(at + col * DP + 16 * b + 4 * g);
#pragma unroll
    for (int s = 0; s < 2; ++s) x.v[s] = values[(size_t)min(lo + n * DL_BLOCK + 2 * g + s, hi - 1) * fresh_stride];
    x.number = *reinterpret_cast<const dl_x2*>(at + 25 * DP + 2 * lane);
#pragma unroll
    for (int b = 0; b < NB; ++b) x.decay[b] = *reinterpret_cast<const dl_x4*>(at + 24 * DP + 16 * b + 4 * g);
    if constexpr (NB == 1) {
      const dl_x2 both = *reinterpret_cast<const dl_x2*>(at + 16 * DP + 2 * lane);
      x.back[0][0] = both[0];
      x.back[0][1] = both[1];
    } else {
#pragma unroll
      for (int b = 0; b < NB; b += 2) {
        const dl_x4 four = *reinterpret_cast<const dl_x4*>(at + 16 * DP + 2 * NB * lane + 2 * b);
#pragma unroll
        for (int i = 0; i < 4; ++i) x.back[b + (i >> 1)][i & 1] = four[i];
      }
    }
    __builtin_amdgcn_sched_barrier(0);                       // (one block's loads behind the other's: a wait for the first then leaves the second under way)
  };
  Block next[AHEAD];
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) fetch(next[i], first + i);
  for (int from = first; from < blocks; from += AHEAD)
#pragma unroll
  for (int turn = 0; turn < AHEAD; ++turn) {
    const int n = from + turn, t0 = lo + n * DL_BLOCK;
    if (n >= blocks) break;                                  // (the same for the whole wave)
    Block& x = next[turn];
    // Rows 4 g and 4 g + 1: k G S of tokens 2 g and 2 g + 1, rows 4 g + 2 and 4 g + 3 their q G S.
    dl_x4 sum[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) sum[r & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.rows[b][r], S[b][r], sum[r & 1], 0, 0, 0);
    float y[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) y[s] = (live && t0 + 2 * g + s < hi ? ld(&x.v[s]) : 0.f) - (sum[0][s] + sum[1][s]);
    dl_x4 res = {0.f, 0.f, sum[0][2] + sum[1][2], sum[0][3] + sum[1][3]};
    if (__all(fabsf(y[0]) < INFINITY && fabsf(y[1]) < INFINITY)) {
#pragma unroll
      for (int s = 0; s < 2; ++s) res = __builtin_amdgcn_mfma_f32_16x16x4f32(x.number[s], y[s], res, 0, 0, 0);
    } else {
      // A number that is not finite must not reach the tokens in front of it through the zeros above the diagonal: row by row, with the
      // tokens behind it left out.
      const dl_x4 start = res;
      for (int i = 0; i < DL_BLOCK; ++i) {
        dl_x4 row = start;
        row = __builtin_amdgcn_mfma_f32_16x16x4f32(x.number[0], 2 * g <= i ? y[0] : 0.f, row, 0, 0, 0);
        row = __builtin_amdgcn_mfma_f32_16x16x4f32(x.number[1], 2 * g + 1 <= i ? y[1] : 0.f, row, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) res[r] = 2 * g + (r & 1) == i ? row[r] : res[r];
      }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) S[b] *= x.decay[b];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int b = 0; b < NB; ++b) S[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.back[b][s], res[s], S[b], 0, 0, 0);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int t = t0 + 2 * g + s;
      if (live && t < hi) out[(size_t)t * heads * dv + (size_t)h * dv + c] = res[2 + s];
    }
    fetch(x, n + AHEAD);
  }
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = 16 * b + 4 * g + r;
      if (live && j < d) mem[(size_t)j * dv + c] = S[b][r];
    }
}

// One workgroup of four waves per (portion, head, 16 columns of S).  A wave owns four columns; its lanes are (column,
// part p = lane % 16): lane (c, p) keeps rows p PER .. p PER + PER - 1 of column c in registers.  Columns of S do not
// depend on each other: for column c, with s = g * S[:, c] (row by row), a = k . s and b = q . s (sums within a row of
// sixteen lanes), u = beta (v_c - a), the new column is s + k u and its read-out q . (s + k u) = b + (q . k) u.
// The rows of q, k (made unit vectors here; q times d^(-1/2)) and of the decays g = exp(neg_rate * softplus(z)) come
// into LDS sixteen tokens at a time; the next sixteen are asked for before the current ones are worked on.
// fresh: rows of `fresh_stride`, [groups d (q) | groups d (k) | heads dv (v)]; z: float rows [heads d]; beta's
// pre-activation at beta_rows[t, beta_offset + h].  A portion that starts at position 0 starts from zeros.
// (Steps of few rows an entry; long portions walk in blocks, see above.)
template <typename T, int PER>
__global__ void __launch_bounds__(4 * WAVE)
delta_scan_kernel(const T* __restrict__ fresh, int fresh_stride, const float* __restrict__ z, const float* __restrict__ neg_rate,
                  const T* __restrict__ beta_rows, int beta_stride, int beta_offset, float* __restrict__ state, size_t state_stride,
                  const int* __restrict__ cu_q, const int* __restrict__ first_position, const int* __restrict__ state_slots,
                  float* __restrict__ out, int heads, int groups, int d, int dv, float unit_eps) {
  constexpr int DP = 16 * PER;                     // rows of S a workgroup's lanes cover (d filled up with zeros)
  constexpr int PIECES = (DL_GROUP * DP) / (4 * WAVE);       // (token, row) pairs a thread brings: PER
  __shared__ __attribute__((aligned(16))) float q_s[DL_GROUP][DP], k_s[DL_GROUP][DP], g_s[DL_GROUP][DP];
  __shared__ float v_s[DL_GROUP][16], beta_s[DL_GROUP], qk_s[DL_GROUP];
  const int e = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & (WAVE - 1), wave = tid / WAVE;
  const int lo = cu_q[e], hi = cu_q[e + 1];
  if (hi <= lo) return;
  const int part = lane & 15, local = wave * 4 + (lane >> 4);
  const int c = blockIdx.z * 16 + local;
  const bool live = c < dv;
  const int qk_head = h / (heads / groups);
  float* mem = state + (size_t)state_slots[e] * state_stride + (size_t)h * d * dv;
  const bool from_zero = first_position[e] == 0;
  float S[PER];
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    const int j = part * PER + r;
    S[r] = (!from_zero && live && j < d) ? mem[(size_t)j * dv + c] : 0.f;
  }
  const float rate = neg_rate[h], q_scale = 1.0f / sqrtf((float)d);
  // (Every load is made, from a place inside, and nothing is converted before it is put down: see the walk in blocks.)
  T q_next[PIECES], k_next[PIECES], v_next, beta_next;
  float g_next[PIECES];
  auto fetch = [&](int t0) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int idx = i * 4 * WAVE + tid, at = min(t0 + idx / DP, hi - 1), j = min(idx % DP, d - 1);
      const T* x = fresh + (size_t)at * fresh_stride;
      q_next[i] = x[(size_t)qk_head * d + j];
      k_next[i] = x[(size_t)(groups + qk_head) * d + j];
      g_next[i] = z[(size_t)at * heads * d + (size_t)h * d + j];
    }
    v_next = fresh[(size_t)min(t0 + (tid >> 4), hi - 1) * fresh_stride + (size_t)2 * groups * d + (size_t)h * dv +
                   min(blockIdx.z * 16 + (tid & 15), (uint32_t)dv - 1)];
    beta_next = beta_rows[(size_t)min(t0 + (tid & 15), hi - 1) * beta_stride + beta_offset + h];
  };
  fetch(lo);
  for (int t0 = lo; t0 < hi; t0 += DL_GROUP) {
    __syncthreads();                                         // the group before has been worked off
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int idx = i * 4 * WAVE + tid, tok = idx / DP, j = idx % DP;
      const bool in = j < d && t0 + tok < hi;
      q_s[tok][j] = in ? ld(&q_next[i]) : 0.f;
      k_s[tok][j] = in ? ld(&k_next[i]) : 0.f;
      g_s[tok][j] = in ? expf(rate * dl_softplus(g_next[i])) : 1.f;
    }
    v_s[tid >> 4][tid & 15] = (int)blockIdx.z * 16 + (tid & 15) < dv && t0 + (tid >> 4) < hi ? ld(&v_next) : 0.f;
    if (tid < DL_GROUP) beta_s[tid] = t0 + tid < hi ? 1.0f / (1.0f + expf(-ld(&beta_next))) : 0.f;
    if (t0 + DL_GROUP < hi) fetch(t0 + DL_GROUP);
    __syncthreads();
    // Unit vectors: sixteen threads a token add up the squares (and q . k) over the rows, then scale the rows in place.
    {
      const int tok = tid >> 4, p = tid & 15;
      float sq = 0.f, sk = 0.f, qk = 0.f;
#pragma unroll
      for (int r = 0; r < PER; ++r) {
        const float qv = q_s[tok][p + 16 * r], kv = k_s[tok][p + 16 * r];
        sq = fmaf(qv, qv, sq);
        sk = fmaf(kv, kv, sk);
        qk = fmaf(qv, kv, qk);
      }
      sq = dl_row_sum16(sq);
      sk = dl_row_sum16(sk);
      qk = dl_row_sum16(qk);
      const float inv_q = q_scale / sqrtf(sq + unit_eps), inv_k = 1.0f / sqrtf(sk + unit_eps);
#pragma unroll
      for (int r = 0; r < PER; ++r) {
        q_s[tok][p + 16 * r] *= inv_q;
        k_s[tok][p + 16 * r] *= inv_k;
      }
      if (p == 0) qk_s[tok] = qk * inv_q * inv_k;
      __syncthreads();
    }
    // Token by token.  (A token past the portion's end has decay 1, beta 0 and zeros for q, k and v: it changes nothing.
    // Rows past d hold zeros in q and k and decay 1: they stay zero and add nothing.)
    float read[DL_GROUP];
#pragma unroll
    for (int tok = 0; tok < DL_GROUP; ++tok) {
      float a = 0.f, b = 0.f;
#pragma unroll
      for (int r = 0; r < PER; ++r) {
        S[r] *= g_s[tok][part * PER + r];
        a = fmaf(k_s[tok][part * PER + r], S[r], a);
        b = fmaf(q_s[tok][part * PER + r], S[r], b);
      }
      a = dl_row_sum16(a);
      b = dl_row_sum16(b);
      const float u = beta_s[tok] * (v_s[tok][local] - a);
#pragma unroll
      for (int r = 0; r < PER; ++r) S[r] = fmaf(k_s[tok][part * PER + r], u, S[r]);
      read[tok] = fmaf(qk_s[tok], u, b);
    }
    if (part == 0 && live) {
#pragma unroll
      for (int tok = 0; tok < DL_GROUP; ++tok)
        if (t0 + tok < hi) out[(size_t)(t0 + tok) * heads * dv + (size_t)h * dv + c] = read[tok];
    }
  }
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    const int j = part * PER + r;
    if (live && j < d) mem[(size_t)j * dv + c] = S[r];
  }
}

// rows: [n_tokens, row_stride]; the channels are three runs of its columns (offsets o0..o2, widths w0..w2); taps float
// [channels, n_taps]; out [n_tokens, channels].
extern "C" int ta_short_conv_silu(const void* rows, int row_stride, int o0, int w0, int o1, int w1, int o2, int w2,
                                  const void* taps, int n_taps, void* state, long state_stride, int state_offset,
                                  const void* cu_q, const void* first_position, const void* state_slots,
                                  const void* entry_of_token, void* out, int n_tokens, int n_entries, int dtype,
                                  const void* bias, hipStream_t stream) {
  if (n_tokens <= 0 || n_entries <= 0) return 0;
  const int channels = w0 + w1 + w2;
  if (channels <= 0 || w0 < 0 || w1 < 0 || w2 < 0 || n_taps < 1 || n_taps > DL_MAX_TAPS || channels > 65535 * 256 ||
      state_stride < (long)state_offset + (long)(n_taps - 1) * channels)
    return -1;
  ConvRuns runs = {{o0, o1, o2}, {w0, w1, w2}};
  dim3 per_token(n_tokens, (channels + 255) / 256), per_entry(n_entries, (channels + 255) / 256);
#define CONV(TT)                                                                                                           \
  short_conv_silu_kernel<TT><<<per_token, 256, 0, stream>>>((const TT*)rows, row_stride, runs, channels, (const float*)taps, \
      n_taps, (const float*)state, (size_t)state_stride, state_offset, (const int*)cu_q, (const int*)first_position,        \
      (const int*)state_slots, (const int*)entry_of_token, (TT*)out, (const float*)bias);                                  \
  if (n_taps > 1)                                                                                                          \
    short_conv_keep_kernel<TT><<<per_entry, 256, 0, stream>>>((const TT*)rows, row_stride, runs, channels, n_taps,          \
        (float*)state, (size_t)state_stride, state_offset, (const int*)cu_q, (const int*)first_position,                   \
        (const int*)state_slots)
#define STEP(TT, NN)                                                                                                       \
  short_conv_step_kernel<TT, NN><<<dim3(max(n_entries, n_tokens), (channels + 255) / 256), 256, 0, stream>>>((const TT*)rows, \
      row_stride, runs, channels, (const float*)taps, (float*)state, (size_t)state_stride, state_offset, (const int*)cu_q,  \
      (const int*)first_position, (const int*)state_slots, (const int*)entry_of_token, (TT*)out, (const float*)bias,        \
      n_tokens, n_entries)
#define STEPS(TT) if (n_taps == 2) { STEP(TT, 2); } else if (n_taps == 3) { STEP(TT, 3); } else { STEP(TT, 4); }
  if (n_taps >= 2 && n_taps <= 4 && n_tokens <= n_entries) {          // (several rows of one entry come one after the other there)
    if (dtype == DT_F32) { STEPS(float); } else { STEPS(bf16_t); }
    return LAUNCH_STATUS();
  }
  if (dtype == DT_F32) { CONV(float); } else { CONV(bf16_t); }
#undef STEPS
#undef STEP
#undef CONV
  return LAUNCH_STATUS();
}

// fresh: rows of `fresh_stride` elements, [groups d (q) | groups d (k) | heads dv (v)]; z float [n_tokens, heads d];
// neg_rate float [heads]; out float [n_tokens, heads dv].  prep: null, or room for `records` (at least n_entries) records of heads
// (25 d' + 128) floats, d' = d filled up to 16, 32, 64, 128 or 256: then the portions walk in blocks of eight tokens, whose share that does
// not depend on the state is made for all of them side by side first, which is what steps with long portions want.  n_tokens / 8 +
// n_entries records hold all blocks; with fewer the portions walk slice by slice, every portion's next records / n_entries blocks, and
// the state is carried in memory.
extern "C" int ta_delta_scan(const void* fresh, int fresh_stride, const void* z, const void* neg_rate, const void* beta_rows,
                             int beta_stride, int beta_offset, void* state, long state_stride, const void* cu_q,
                             const void* first_position, const void* state_slots, void* out, void* prep, int records, int n_tokens,
                             int n_entries, int heads, int groups, int d, int dv, float unit_eps, int dtype,
                             hipStream_t stream) {
  if (n_entries <= 0 || n_tokens <= 0) return 0;
  if (d < 1 || d > DL_MAX_D || dv < 1 || heads < 1 || groups < 1 || heads % groups || heads > 65535 ||
      state_stride < (long)heads * d * dv)
    return -1;
  dim3 grid(n_entries, heads, (dv + 15) / 16);
  if (grid.z > 65535) return -1;
  const int per = (d + 15) / 16;
  if (prep) {
    const int nb = per <= 1 ? 1 : per <= 2 ? 2 : per <= 4 ? 4 : per <= 8 ? 8 : 16;
    const dim3 walks(n_entries, heads, (dv + 63) / 64);
    const int all = n_tokens / DL_BLOCK + n_entries, each = records >= all ? 0 : records / n_entries;
    if (each < 1 && records < all) return -1;
#define BLOCKS(TT, RR) delta_blocks_kernel<TT, RR><<<dim3(each ? each * n_entries : all, (heads + 3) / 4), 4 * WAVE, 0, stream>>>( \
    (const TT*)fresh, fresh_stride, (const float*)z, (const float*)neg_rate, (const TT*)beta_rows, beta_stride, beta_offset,      \
    (float*)prep, (const int*)cu_q, n_entries, heads, groups, d, 16 * nb, unit_eps, first, each)
#define WALK(TT, NN) delta_walk_kernel<TT, NN><<<walks, 4 * WAVE, 0, stream>>>((const TT*)fresh, fresh_stride, (const float*)prep, \
    (float*)state, (size_t)state_stride, (const int*)cu_q, (const int*)first_position, (const int*)state_slots, (float*)out,     \
    heads, groups, d, dv, first, each)
#define BOTH(TT)                                                                                                              \
    if (nb <= 4) BLOCKS(TT, 1); else if (nb <= 8) BLOCKS(TT, 2); else BLOCKS(TT, 4);                                           \
    if (nb == 1) WALK(TT, 1); else if (nb == 2) WALK(TT, 2); else if (nb == 4) WALK(TT, 4); else if (nb == 8) WALK(TT, 8);     \
    else WALK(TT, 16)
    for (int first = 0; first * DL_BLOCK < n_tokens; first += each ? each : all) {      // (no portion is longer than the step)
      if (dtype == DT_F32) { BOTH(float); } else { BOTH(bf16_t); }
    }
#undef BOTH
#undef WALK
#undef BLOCKS
    return LAUNCH_STATUS();
  }
#define SCAN(TT, PP) delta_scan_kernel<TT, PP><<<grid, 4 * WAVE, 0, stream>>>((const TT*)fresh, fresh_stride, (const float*)z,    \
    (const float*)neg_rate, (const TT*)beta_rows, beta_stride, beta_offset, (float*)state, (size_t)state_stride,              \
    (const int*)cu_q, (const int*)first_position, (const int*)state_slots, (float*)out, heads, groups, d, dv, unit_eps)
#define SCANS(TT) if (per <= 1) SCAN(TT, 1); else if (per <= 2) SCAN(TT, 2); else if (per <= 4) SCAN(TT, 4); \
                  else if (per <= 8) SCAN(TT, 8); else SCAN(TT, 16)
  if (dtype == DT_F32) { SCANS(float); } else { SCANS(bf16_t); }
#undef SCANS
#undef SCAN
  return LAUNCH_STATUS();
}
