// Fused products for decode batches of up to 16 rows.  Each keeps the layout of the weight-streaming kernel
// (C^T = W A^T on 16x16x32 MFMAs, the waves of a workgroup split K and add up through LDS) and folds the
// neighbouring small kernels into its prologue or epilogue:
//   NORM prologue   the rows are read from the float residual stream and RMS-normalised on the fly into LDS
//                   (or, normalised already, copied there once: what a workgroup pulls in over the fabric from
//                   the caches counts like what it pulls from memory, and rows asked for again in every batch
//                   of weights would be half as many bytes again as the weights)
//   ROPE_STORE      q/k/v projection: bias, half-split rotation, keys and values written into their pages
//   GATED           silu(gate) * up
//   RESIDUAL        the product is added into the float residual stream in place
#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

enum { EPI_ROPE_STORE = 0, EPI_GATED = 1, EPI_RESIDUAL = 2 };

struct FusedArgs {
  // input rows: bfloat16 activations, or (with the NORM prologue) the float residual with norm weight and eps
  const bf16_t* a; int lda;
  const float* residual_in; const float* norm_weight; float eps;
  const bf16_t* w; const float* bias;
  int m, n, k;
  int rows;                                                // weight rows per workgroup
  // EPI_GATED / plain output (bfloat16 [m, ldc])
  bf16_t* out; int ldc;
  // EPI_RESIDUAL
  float* residual_out;
  // EPI_ROPE_STORE
  const int* positions; const float* cos_sin; const int* slots;
  bf16_t* k_pages; bf16_t* v_pages; int n_q, n_kv, d, page_size;
  float temper_coef; int temper_every;                     // temper_every > 0: query heads times 1 + coef ln(floor((p + 1) / every) + 1)
};

__device__ __forceinline__ bf16x8 fz8() {
  bf16x8 z;
#pragma unroll
  for (int i = 0; i < 8; ++i) z[i] = (__bf16)0.0f;
  return z;
}
// Registers with whatever they hold, for lanes whose load is left out and whose products are never stored (a row
// of the weights only feeds its own row of the result).  Zeros would do as well, but the compiler keeps one zero
// for many purposes, copies a loaded value over it, and waits for the load to do so, in the middle of a batch of
// loads: the batch then takes two trips to memory instead of one.
__device__ __forceinline__ bf16x8 any8() {
  bf16x8 v;
  asm volatile("" : "=v"(v));
  return v;
}

// Words between a wave's sums of one register and of the next.
__host__ __device__ constexpr int fused_sum_words(int epi, bool one) { return epi == EPI_RESIDUAL || one ? WAVE + 4 : WAVE; }

// A workgroup owns `p.rows` weight rows (output columns), in PASSES blocks of up to sixteen: the M side of the
// MFMA.  Lanes whose weight row or input row only feeds results that are never stored load nothing: a
// load costs the memory pipeline by its active lanes.  So a small matrix is spread thinly over many
// workgroups (4 rows each), and a large one is cut so that every compute unit streams the same share.
//
// UN: steps of 32 along K that a wave requests at once.  ONE: the host has checked that a wave's whole share
// of K is one such batch, so there is no loop, the batches of all passes are requested at the start, and a
// small matrix is over after one trip to memory instead of several.
//
// The arguments are all asked for at the kernel's start (`HELD`): left to itself the compiler fetches each piece
// of the argument block where it is first used, and a small kernel then begins with several trips to memory one
// after the other.  What the epilogue needs from memory is asked for before the weights where a second load hangs
// on a first one (the angle table's row on the position), and otherwise right after them and left alone until the
// epilogue: a value that is used early makes the wave wait for everything it asked for before, the weights included.
//
// The kernel takes its arguments one by one, those that every instance needs before its first load in the first
// sixteen words of the argument block: the library is compiled so that these are in scalar registers when a wave
// starts (`-amdgpu-kernarg-preload-count`; fourteen words in fact), and no instance begins with a fetch of arguments:
// m, the rows a workgroup and the head size share a word (16 bits for the head size, which the launcher checks), the two numbers of heads another (with the
// gated epilogue: whether its results go past the chiplet's caches).
// One pointer serves for the rows (bfloat16, or the float residual for the norm prologue) and one for the result (bfloat16 rows, or
// the float residual that is added to), which never occur together.  The rest lies behind; only the waves of the epilogue wait for it,
// with their weights under way.  Positions and slots come through the scalar unit there, so that the angles, which hang on the
// position, are asked for without a wait among the vector loads (q/k/v of 896, one row, weights from memory: 4.4 -> 4.1 us).
//
// The epilogue is the tail that every launch waits for, and a wave's instructions one behind the other are its length: each of its
// lanes has one output.  Wave v < ceil(M / 4) takes input rows 4 v .. 4 v + 3, sixteen lanes side by side the block's weight rows, so that a
// store is one run of the result; a lane adds the NW partial sums of its output in the waves' order.  (Four outputs a lane of one wave,
// four times the LDS reads, activations and stores behind each other, one row and eight: q/k/v of 896 5.0 -> 4.4 and 5.4 -> 5.0 us,
// out 3.15 -> 2.8 and 3.5 -> 3.2, gate/up 4,864 over 896 6.8 -> 6.15 and 7.75 -> 7.15, down 5.6 -> 5.4 and 6.9 -> 6.7; a kernel that
// does nothing is 1.65.)
//
// LINES (K a multiple of 64): the weights come by whole cache lines (`lines_to_rows` in common.h), past the caches, which hold nothing
// that comes again: a pair of steps is one line of each of a block's sixteen rows, u even its lower eight rows, u odd its upper
// eight.  For walks of several trips; where all is asked for in one trip of four steps there is nothing to stream (896 columns level).
// Us, sixteen rows' half lines a load | so, one input row and sixteen, weights from memory: gate/up 18,944 over 3,584 55.5 | 46.1
// and 68.8 | 54.0, down 18,944 to 3,584 26.4 | 25.4 and 36.2 | 34.4, q/k/v of 3,584 13.8 | 11.3 and 16.1 | 12.3, gate/up 8,960 over 1,536
// 17.8 | 17.0 and 22.6 | 18.1, down 8,960 to 1,536 11.2 | 9.7 and 15.2 | 14.2, down 4,864 to 896 6.4 | 5.8 and 9.2 | 8.7.  Weights that are in
// the last-level cache already (all of a model in less than its 256 MB, the exception): gate/up 4,096 over 2,048 12.7 | 10.7 and 16.3 | 13.3,
// 3,072 over 1,536 7.3 | 7.7 and 9.7 | 9.7, down 4,096 to 1,024 5.5 | 5.5 and 7.7 | 7.6, 8,192 to 2,048 8.9 | 9.6 and 14.2 | 13.7.
//
// STAGE (up to eight rows from memory, a share of K in one trip): a wave brings its lines of all rows in STAGE loads of sixteen
// different bytes a lane and turns them into fragments through a part of LDS that is its own, without a barrier.  A fragment loaded
// straight from memory is one of UN loads whose lanes mostly ask for the same bytes, and such a load holds up the memory pipeline
// like any other: a workgroup's weights and rows, down 4,864 to 896, were 80 loads of the one and 160 of the other.  Us, direct |
// staged, one row and eight: down 4,864 to 896 5.4 | 4.55 and 6.7 | 5.4, out 896 to 896 2.8 | 2.75 and 3.2 | 2.9 (weights alone 3.3 and 2.0).
// With more than eight rows a staged share is as many loads as the fragments are.
//
// An instance's code begins on a page of its own, so that none of up to 4 KB lies across a page's end and where it lies in the cache of instructions
// does not hang on the instances in front of it: out of 896 over 896, eight rows, had come to lie across one when others were taken out, and took 3.0 us
// for the 2.77 that the same instructions take elsewhere (eight chat turns 13.75 ms, so 13.66; on 8 KB, where all instances' starts share
// their places in that cache, 13.79).
template <int NW, int EPI, bool NORM, int UN, bool ONE, int PASSES, bool LINES, int STAGE>
__global__ void __launch_bounds__(NW * WAVE) __attribute__((aligned(4096)))
fused_decode_kernel(const bf16_t* w, const void* rows_in, const float* norm_weight, uint32_t m_rows_d, uint32_t heads,
                    int n, int k, int lda, float eps, void* result, const float* bias,
                    const int* positions, const float* cos_sin, const int* slots, bf16_t* k_pages, bf16_t* v_pages,
                    int page_size, float temper_coef, int temper_every) {
  HELD(w, rows_in, norm_weight, m_rows_d, heads, n, k, lda, eps, result);  // (the fourteen words that are there)
  const int m = m_rows_d & 0xff, rows = (m_rows_d >> 8) & 0xff, d = m_rows_d >> 16, n_q = heads & 0xffff, n_kv = heads >> 16;
  FusedArgs p;
  // (Rows with a norm weight are the float residual; without one they are bfloat16, normalised already or plain.)
  p.a = norm_weight ? nullptr : (const bf16_t*)rows_in; p.lda = lda;
  p.residual_in = norm_weight ? (const float*)rows_in : nullptr; p.norm_weight = norm_weight; p.eps = eps;
  p.w = w; p.bias = bias; p.m = m; p.n = n; p.k = k; p.rows = rows;
  p.out = (bf16_t*)result; p.ldc = EPI == EPI_GATED ? n / 2 : n_q * d;
  p.residual_out = (float*)result;
  p.positions = positions; p.cos_sin = cos_sin; p.slots = slots; p.k_pages = k_pages; p.v_pages = v_pages;
  p.n_q = n_q; p.n_kv = n_kv; p.d = d; p.page_size = page_size;
  constexpr int SETS = (EPI == EPI_RESIDUAL) ? 1 : 2;
  constexpr int HELD = ONE ? PASSES : 1;                     // batches of weights held at once
  static_assert(EPI != EPI_ROPE_STORE || PASSES == 1, "the rotation pairs rows within one block");
  // (The epilogue's reads touch every bank once: four words stand between a wave's registers.  Where long rows lie in LDS beside two sets, that
  // kilobyte can be a workgroup less on a compute unit, nine rows of 3,584 60.4 -> 69.7 us, and a register's lanes are turned by four for every
  // register before it instead, which costs short launches 0.02 to 0.1 us.)
  constexpr int RS = fused_sum_words(EPI, ONE), TURN = RS == WAVE ? 4 : 0;
  __shared__ float red[NW][SETS * 4][RS];
  extern __shared__ __attribute__((aligned(16))) uint16_t a_s[];   // NORM: the m normalised rows of K + 8 bfloat16; STAGE: the waves' pieces
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int col = lane & 15, g = lane >> 4;
  const int M = p.m, K = p.k, R = p.rows;
  const int tile = blockIdx.x;

  // Which weight rows this workgroup owns: `row0` onwards (+ `row1` onwards for the second set).
  int row0, row1 = 0;
  bool paired = true;
  if (EPI == EPI_ROPE_STORE) {
    const int half = p.d / 2, per_half = half / R;
    const int n_pair_tiles = (p.n_q + p.n_kv) * per_half;
    if (tile < n_pair_tiles) {
      const int hd = tile / per_half, j = tile % per_half;
      row0 = hd * p.d + j * R;
      row1 = row0 + half;
    } else {
      paired = false;
      row0 = (p.n_q + p.n_kv) * p.d + (tile - n_pair_tiles) * R;
      row1 = row0;
    }
  } else if (EPI == EPI_GATED) {
    row0 = tile * R;
    row1 = row0 + p.n / 2;
  } else {
    row0 = tile * R;
  }
  const int n_limit = (EPI == EPI_GATED) ? p.n / 2 : p.n;
  const bf16_t* w0[PASSES];
  const bf16_t* w1[PASSES];
  bool w_lane[PASSES], w_upper[PASSES];                     // LINES: the lane's row of the lower eight, of the upper eight
  const int piece = LINES ? g + 4 * (col >> 3) : g;
#pragma unroll
  for (int ps = 0; ps < PASSES; ++ps) {
    const int r = 16 * ps + (LINES ? col & 7 : col);
    w_lane[ps] = r < R && row0 + r < n_limit;
    w_upper[ps] = LINES && r + 8 < R && row0 + r + 8 < n_limit;
    w0[ps] = p.w + (size_t)min(row0 + r, n_limit - 1) * K + 8 * piece;
    w1[ps] = p.w + (size_t)min(row1 + r, p.n - 1) * K + 8 * piece;
  }
  const bool a_lane = col < M;
  const int a_m = min(col, M - 1);
  const int full_steps = K / 32;
  const int lds_stride = K + 8;

  // The epilogue's lanes: weight row `er` of a block, input row `em`; `e_at` is where that output stands in a wave's part of `red`.
  const int er = lane & 15, em = 4 * wave + (lane >> 4);
  const bool e_wave = 4 * wave < M;
  const int e_lane = (er >> 2) * 16 + em, e_at = (er & 3) * RS + (TURN ? (e_lane + TURN * (er & 3)) & 63 : e_lane);

  // Weight fragments come from HBM and take longest; the first batch is requested before the prologue.
  // Step j of a wave's batch: steps come in pairs (128 contiguous bytes of a weight row, one cache line),
  // pair q of the batch starting at pair `base` is pair base + q * NW.
  auto step_of = [&](int base_pair, int u) { return (base_pair + (u >> 1) * NW) * 2 + (u & 1); };
  const int pairs = (full_steps + 1) / 2;
  bf16x8 wf[HELD][UN][SETS];
  auto load_w = [&](int held, int ps, int base_pair) {
    if constexpr (LINES) {
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const int pair = base_pair + (u >> 1) * NW;
        const int at = min(pair, pairs - 1) * 64 + (u & 1) * 8 * K;      // (the upper rows' place is only used by lanes that have one)
        wf[held][u][0] = ONE ? any8() : fz8();
        if (SETS == 2) wf[held][u][SETS - 1] = ONE ? any8() : fz8();
        if ((u & 1 ? w_upper[ps] : w_lane[ps]) && (ONE || pair < pairs)) {
          wf[held][u][0] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(w0[ps] + at));
          if (SETS == 2) wf[held][u][SETS - 1] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(w1[ps] + at));
        }
      }
      return;
    }
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const int step = min(step_of(base_pair, u), max(full_steps - 1, 0));   // clamped loads are not used
      // (in the loop of the long walks the zeros stay: there the statement that leaves a register as it is would
      // stand between the loop's loads and products, which the compiler then no longer moves past each other)
      wf[held][u][0] = ONE ? any8() : fz8();
      if (SETS == 2) wf[held][u][SETS - 1] = ONE ? any8() : fz8();
      if (w_lane[ps]) {
        wf[held][u][0] = *reinterpret_cast<const bf16x8*>(w0[ps] + step * 32);
        if (SETS == 2) wf[held][u][SETS - 1] = *reinterpret_cast<const bf16x8*>(w1[ps] + step * 32);
      }
    }
  };
  load_w(0, 0, wave);
  if (ONE) {
#pragma unroll
    for (int ps = 1; ps < PASSES; ++ps) load_w(HELD - PASSES + ps, ps, wave);
  }
  // LINES: steps u and u + 1 of a pair, inside K or at its last line.
  auto a_line = [&](int base_pair, int u) { return min(base_pair + (u >> 1) * NW, pairs - 1) * 64 + 32 * (u & 1); };
  auto a_inside = [&](int base_pair, int u) { return base_pair + (u >> 1) * NW < pairs; };
  const bf16_t* ar = NORM ? nullptr : p.a + (size_t)a_m * p.lda + 8 * g;
  bf16x8 af_one[ONE ? UN : 1];
  // STAGE: piece i of the wave's M * PIECES pieces of sixteen bytes is piece i % PIECES of row i / PIECES.
  constexpr int PIECES = UN * 4, ROW_BYTES = PIECES * 16 + 16;  // (sixteen bytes on, so that the rows of a fragment lie in different banks)
  char* mine = reinterpret_cast<char*>(a_s) + (STAGE > 0 ? (size_t)wave * M * ROW_BYTES : 0);
  word4 staged[STAGE > 0 ? STAGE : 1];
  if constexpr (STAGE > 0) {
#pragma unroll
    for (int j = 0; j < STAGE; ++j) {
      const int i = min(j * WAVE + lane, M * PIECES - 1), piece = i % PIECES;
      const int k = min((wave + (piece >> 3) * NW) * 64 + 8 * (piece & 7), K - 8);   // (what lies past the end of K is not used)
      staged[j] = *reinterpret_cast<const word4*>(p.a + (size_t)(i / PIECES) * p.lda + k);
    }
  } else if (ONE && !NORM) {                               // the rows' fragments as well
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      // (every lane: a row past the end repeats the last one and only feeds columns that are never stored)
      af_one[u] = *reinterpret_cast<const bf16x8*>(ar + (LINES ? a_line(wave, u) : min(step_of(wave, u), max(full_steps - 1, 0)) * 32));
    }
  }

  // What else the epilogue needs besides the sums is requested now as well, and not touched before the epilogue.
  float pre_cos = 1.f, pre_sin = 0.f;
  int pre_slot = -1;
  if (EPI == EPI_ROPE_STORE && e_wave) {
    HELD(bias, positions, cos_sin, slots, k_pages, v_pages);
    const bool turned = p.cos_sin || temper_every > 0;
    int position = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int row = min(4 * wave + j, M - 1);
      const int at = turned ? scalar_int(positions + row) : 0, slot = slots ? scalar_int(slots + row) : -1;
      position = (lane >> 4) == j ? at : position;
      pre_slot = (lane >> 4) == j ? slot : pre_slot;
    }
    if (em < M && er < R) {
      if (paired && p.cos_sin) {
        const float* cs = p.cos_sin + (size_t)position * p.d + row0 % p.d + er;
        pre_cos = cs[0];
        pre_sin = cs[p.d / 2];
      } else if (temper_every > 0 && row0 < p.n_q * p.d) {    // the factor stands where a rotation's cosine would
        pre_cos = 1.f + temper_coef * logf((float)((position + 1) / temper_every) + 1.f);
      }
    }
  }
  float pre_a[PASSES], pre_b[PASSES];                        // the old residual and the bias; or the two halves' bias
#pragma unroll
  for (int ps = 0; ps < PASSES; ++ps) pre_a[ps] = pre_b[ps] = 0.f;
  // EPI_GATED with another activation than silu: its three numbers (alpha, limit, shift) lie where the rotation's table
  // would: g' = min(g, limit), u' = clamp(u, -limit, limit), g' sigmoid(alpha g') (u' + shift).
  float act_alpha = 1.f, act_limit = INFINITY, act_shift = 0.f;
  if (EPI == EPI_GATED && p.cos_sin) { act_alpha = p.cos_sin[0]; act_limit = p.cos_sin[1]; act_shift = p.cos_sin[2]; }
  if (EPI == EPI_RESIDUAL && e_wave) HELD(bias);
  if (e_wave && em < M) {
    if (EPI == EPI_RESIDUAL) {
#pragma unroll
      for (int ps = 0; ps < PASSES; ++ps) {
        const int local = 16 * ps + er, n = row0 + local;
        if (local < R && n < p.n) {
          pre_a[ps] = p.residual_out[(size_t)em * p.n + n];
          if (p.bias) pre_b[ps] = p.bias[n];
        }
      }
    } else if (EPI == EPI_ROPE_STORE && er < R && p.bias) {
      pre_a[0] = p.bias[row0 + er];
      pre_b[0] = p.bias[row1 + er];
    }
  }

  if (NORM && !p.residual_in) {
    // Rows that are normalised already: copied into LDS once.
    for (int m = wave; m < M; m += NW) {
      const bf16_t* x = p.a + (size_t)m * p.lda;
      uint16_t* dst = a_s + (size_t)m * lds_stride;
      for (int k = lane * 8; k < K; k += WAVE * 8)
        *reinterpret_cast<uint4*>(dst + k) = *reinterpret_cast<const uint4*>(x + k);
    }
    __syncthreads();
  } else if (NORM) {
    // Each row once: 1 / sqrt(mean(x^2) + eps), then x * that * weight rounded to bfloat16 into LDS.
    for (int m = wave; m < M; m += NW) {
      const float* x = p.residual_in + (size_t)m * K;
      uint16_t* dst = a_s + (size_t)m * lds_stride;
      if (K <= 4 * WAVE * 4) {
        // The row fits in four float4 per lane: read it (and the norm weight) once and keep it in registers.
        float4 v[4], gw[4];
        float sq = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int k = (i * WAVE + lane) * 4;
          v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
          gw[i] = v[i];
          if (k < K) {
            v[i] = *reinterpret_cast<const float4*>(x + k);          // K is a multiple of 8
            gw[i] = *reinterpret_cast<const float4*>(p.norm_weight + k);
          }
          sq += v[i].x * v[i].x + v[i].y * v[i].y + v[i].z * v[i].z + v[i].w * v[i].w;
        }
        sq = wave_sum(sq);
        const float inv = 1.0f / sqrtf(sq / (float)K + p.eps);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int k = (i * WAVE + lane) * 4;
          if (k >= K) continue;
          union { bf16x4 v; uint2 bits; } packed;
          packed.v[0] = (__bf16)(v[i].x * inv * gw[i].x); packed.v[1] = (__bf16)(v[i].y * inv * gw[i].y);
          packed.v[2] = (__bf16)(v[i].z * inv * gw[i].z); packed.v[3] = (__bf16)(v[i].w * inv * gw[i].w);
          *reinterpret_cast<uint2*>(dst + k) = packed.bits;
        }
        continue;
      }
      float sq = 0.f;
      for (int k = lane * 4; k < K; k += WAVE * 4) {
        const float4 v = *reinterpret_cast<const float4*>(x + k);
        sq += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
      }
      sq = wave_sum(sq);
      const float inv = 1.0f / sqrtf(sq / (float)K + p.eps);
      for (int k = lane * 4; k < K; k += WAVE * 4) {
        const float4 v = *reinterpret_cast<const float4*>(x + k);
        const float4 gw = *reinterpret_cast<const float4*>(p.norm_weight + k);
        union { bf16x4 v; uint2 bits; } packed;
        packed.v[0] = (__bf16)(v.x * inv * gw.x); packed.v[1] = (__bf16)(v.y * inv * gw.y);
        packed.v[2] = (__bf16)(v.z * inv * gw.z); packed.v[3] = (__bf16)(v.w * inv * gw.w);
        *reinterpret_cast<uint2*>(dst + k) = packed.bits;
      }
    }
    __syncthreads();
  }
  if constexpr (STAGE > 0) {
#pragma unroll
    for (int j = 0; j < STAGE; ++j) {
      const int i = min(j * WAVE + lane, M * PIECES - 1);
      *reinterpret_cast<word4*>(mine + i / PIECES * ROW_BYTES + i % PIECES * 16) = staged[j];
    }
    wave_exchange();
#pragma unroll
    for (int u = 0; u < UN; ++u) af_one[u] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const word4*>(mine + a_m * ROW_BYTES + u * 64 + 16 * g));
  }
  const uint16_t* as_row = a_s + (size_t)a_m * lds_stride + 8 * g;
  auto load_a = [&](int k) -> bf16x8 {
    if (NORM) return *reinterpret_cast<const bf16x8*>(as_row + k);
    return a_lane ? *reinterpret_cast<const bf16x8*>(ar + k) : fz8();
  };

#pragma unroll
  for (int ps = 0; ps < PASSES; ++ps) {
    floatx4 acc[SETS];
#pragma unroll
    for (int s = 0; s < SETS; ++s) acc[s] = (floatx4){0.f, 0.f, 0.f, 0.f};
    if constexpr (LINES) {
      auto multiply = [&](const bf16x8 (&w)[UN][SETS], const bf16x8 (&af)[UN]) {
#pragma unroll
        for (int u = 0; u < UN; u += 2)
#pragma unroll
          for (int s = 0; s < SETS; ++s) {
            bf16x8 b0, b1;
            lines_to_rows(__builtin_bit_cast(word4, w[u][s]), __builtin_bit_cast(word4, w[u + 1][s]), col < 8, b0, b1);
            acc[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b0, af[u], acc[s], 0, 0, 0);
            acc[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b1, af[u + 1], acc[s], 0, 0, 0);
          }
      };
      bf16x8 af[UN];
      if constexpr (ONE) {
#pragma unroll
        for (int u = 0; u < UN; ++u) {
          af[u] = NORM ? load_a(a_line(wave, u)) : af_one[u];
          if (!a_inside(wave, u)) af[u] = fz8();             // past the end of K: zeros, see below
        }
        multiply(wf[HELD - PASSES + ps], af);
      } else {
        // The next batch's weights, and rows that come from memory, are requested before the current one is multiplied (rows asked for with
        // their own batch would wait in line behind the weights just asked for: down 18,944 to 3,584 33 us in place of 26).
        bf16x8 next[UN];
        auto ask_rows = [&](int pair) {
#pragma unroll
          for (int u = 0; u < UN; ++u) {
            next[u] = fz8();
            if (a_lane && a_inside(pair, u)) next[u] = *reinterpret_cast<const bf16x8*>(ar + a_line(pair, u));
          }
        };
        if (!NORM) ask_rows(wave);
        for (int pair = wave; pair < pairs; pair += (UN / 2) * NW) {
          bf16x8 wc[UN][SETS];
#pragma unroll
          for (int u = 0; u < UN; ++u) {
            wc[u][0] = wf[0][u][0];
            if (SETS == 2) wc[u][SETS - 1] = wf[0][u][SETS - 1];
            if (NORM) {
              af[u] = load_a(a_line(pair, u));
              if (!a_inside(pair, u)) af[u] = fz8();
            } else {
              af[u] = next[u];
            }
          }
          if (pair + (UN / 2) * NW < pairs) {
            load_w(0, ps, pair + (UN / 2) * NW);
            if (!NORM) ask_rows(pair + (UN / 2) * NW);
          }
          multiply(wc, af);
        }
        if (ps + 1 < PASSES) load_w(0, ps + 1, wave);
      }
    } else if constexpr (ONE) {
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        // A step past the end of K is multiplied all the same, with zeros for the rows: no matrix instruction
        // sits behind a condition (it would run whatever a lane mask says, and whether the compiler masks
        // or branches here is its choice).  The weights of such a step were read from a clamped, valid place.
        const int step = step_of(wave, u);
        bf16x8 af = NORM ? load_a(min(step, max(full_steps - 1, 0)) * 32) : af_one[u];
        if (step >= full_steps) af = fz8();
#pragma unroll
        for (int s = 0; s < SETS; ++s)
          acc[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[HELD - PASSES + ps][u][s], af, acc[s], 0, 0, 0);
      }
    } else {
      // Batches of UN steps; the next batch's weights are requested before the current one is multiplied.
      for (int pair = wave; pair * 2 < full_steps; pair += (UN / 2) * NW) {
        bf16x8 wc[UN][SETS], af[UN];
#pragma unroll
        for (int u = 0; u < UN; ++u) {
          wc[u][0] = wf[0][u][0];
          if (SETS == 2) wc[u][SETS - 1] = wf[0][u][SETS - 1];
          af[u] = load_a(min(step_of(pair, u), full_steps - 1) * 32);
          if (step_of(pair, u) >= full_steps) af[u] = fz8();      // past the end of K: zeros, see above
        }
        if ((pair + (UN / 2) * NW) * 2 < full_steps) load_w(0, ps, pair + (UN / 2) * NW);
#pragma unroll
        for (int u = 0; u < UN; ++u) {
#pragma unroll
          for (int s = 0; s < SETS; ++s)
            acc[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wc[u][s], af[u], acc[s], 0, 0, 0);
        }
      }
      if (ps + 1 < PASSES) load_w(0, ps + 1, wave);          // the next block's first batch, before this one's sums
    }
    if (!LINES && (K & 31)) {                                            // tail of K (a multiple of 8): zero-filled; wave 0's
      const int k = full_steps * 32;
      const bool ok = wave == 0 && k + 8 * g < K;
      const bf16x8 af = ok ? load_a(k) : fz8();
      acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ok ? *reinterpret_cast<const bf16x8*>(w0[ps] + k) : fz8(), af, acc[0], 0, 0, 0);
      if (SETS == 2)
        acc[SETS - 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ok ? *reinterpret_cast<const bf16x8*>(w1[ps] + k) : fz8(), af, acc[SETS - 1], 0, 0, 0);
    }
    if (ps > 0) __syncthreads();                             // the block before has been read
#pragma unroll
    for (int s = 0; s < SETS; ++s)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wave][s * 4 + r][(lane + TURN * r) & 63] = acc[s][r];
    __syncthreads();
    const int local = 16 * ps + er;                          // the lane's row within the workgroup's
    if (e_wave && em < M && local < R) {
      float v0 = 0.f, v1 = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        v0 += (&red[w][0][0])[e_at];
        if (SETS == 2) v1 += (&red[w][(SETS - 1) * 4][0])[e_at];
      }
      if (EPI == EPI_RESIDUAL) {
        const int n = row0 + local;
        if (n < p.n) st_through(p.residual_out + (size_t)em * p.n + n, (pre_a[ps] + pre_b[ps]) + v0);   // old residual (+ bias) from the start
      } else if (EPI == EPI_GATED) {
        const int n = row0 + local;
        if (n < n_limit) {
          bf16_t* dst = p.out + (size_t)em * p.ldc + n;
          if (p.cos_sin) {
            const float gate = fminf(v0, act_limit), up = fminf(fmaxf(v1, -act_limit), act_limit);
            v0 = gate / (1.0f + __expf(-act_alpha * gate)) * (up + act_shift);
          } else {
            v0 = v0 / (1.0f + __expf(-v0)) * v1;
          }
          if (heads) st_through(dst, v0); else st(dst, v0);        // (the word says which, see the launcher)
        }
      } else {
        const int d = p.d, half = d / 2;
        const int slot = pre_slot;
        const int page = slot >= 0 ? slot / p.page_size : 0, off = slot >= 0 ? slot % p.page_size : 0;
        if (paired) {
          const int hd = row0 / d, i = row0 % d + er;               // element i (< half) of head hd, and i + half
          const float x1 = v0 + pre_a[0], x2 = v1 + pre_b[0];
          // cos 1, sin 0 without a rotation.  Which product is rounded before the other joins it is written down, so that it stays as it
          // is when the code around it changes (the compiler joins either; its choice in the instances of eight waves by lines is the other).
          const float r1 = fmaf(x1, pre_cos, -(x2 * pre_sin));
          const float r2 = NW == 8 && LINES ? fmaf(x2, pre_cos, x1 * pre_sin) : fmaf(x1, pre_sin, x2 * pre_cos);
          bf16_t* dst = nullptr;
          if (hd < p.n_q) dst = p.out + (size_t)em * p.ldc + (size_t)hd * d + i;
          else if (slot >= 0) dst = p.k_pages + (((size_t)page * p.n_kv + (hd - p.n_q)) * p.page_size + off) * d + i;
          if (dst) { st_through(dst, r1); st_through(dst + half, r2); }
        } else if (slot >= 0) {
          const int e = row0 - (p.n_q + p.n_kv) * d + er;           // element of the joined value heads
          const int kvh = e / d, dd = e % d;
          st_through(p.v_pages + (((size_t)page * p.n_kv + kvh) * d + dd) * p.page_size + off, v0 + pre_a[0]);
        }
      }
    }
  }
}

template <int NW, int EPI, bool NORM, int UN, bool ONE, int PASSES, bool LINES = false, int STAGE = 0>
static int launch_kernel(const FusedArgs& args, int tiles, hipStream_t stream) {
  if constexpr (ONE && !NORM && STAGE == 0) {
    constexpr int MOST = UN / 2;                             // loads for eight rows of UN / 2 lines
    const int loads = (args.m * UN * 4 + WAVE - 1) / WAVE;
    if (args.m <= 8 && args.k >= 8) {
      if (loads <= 1) return launch_kernel<NW, EPI, NORM, UN, ONE, PASSES, LINES, 1>(args, tiles, stream);
      if (loads <= 2) return launch_kernel<NW, EPI, NORM, UN, ONE, PASSES, LINES, 2>(args, tiles, stream);
      if (MOST > 2 && loads <= 3) return launch_kernel<NW, EPI, NORM, UN, ONE, PASSES, LINES, MOST < 3 ? MOST : 3>(args, tiles, stream);
      return launch_kernel<NW, EPI, NORM, UN, ONE, PASSES, LINES, MOST>(args, tiles, stream);
    }
  }
  size_t lds = NORM ? (size_t)args.m * (args.k + 8) * sizeof(uint16_t) : (size_t)(STAGE > 0 ? NW * args.m * (UN * 64 + 16) : 0);
  constexpr size_t SUMS_BYTES = NW * (EPI == EPI_RESIDUAL ? 1 : 2) * 4 * fused_sum_words(EPI, ONE) * sizeof(float);   // (the kernel's own: `red`)
  if (lds + SUMS_BYTES > 64 * 1024) {
    // More LDS than a launch has unasked: ask for it (the device has 160 KB per compute unit).
    if (lds > 140 * 1024) return -1;
    hipError_t err = hipFuncSetAttribute(
        reinterpret_cast<const void*>(&fused_decode_kernel<NW, EPI, NORM, UN, ONE, PASSES, LINES, STAGE>),
        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err != hipSuccess) return (int)err;
  }
  // The kernel tells the float residual from bfloat16 rows by whether there is a norm weight.
  const bool from_residual = args.residual_in != nullptr;
  if (from_residual != (args.norm_weight != nullptr) || (!from_residual && !args.a) || !args.w) return -1;
  if (EPI == EPI_RESIDUAL ? !args.residual_out : !args.out) return -1;
  if (args.d > 0xffff || args.n_q > 0xffff || args.n_kv > 0xffff) return -1;   // (what the packed arguments hold)
  // Gated results go past the chiplet's caches while two workgroups a compute unit are all there are: with more, the first ones' are written back
  // under the others' way (8,960 over 1,536, 747 workgroups: 17.9 us past them, 17.3 plainly, eight rows 16.0 and 14.9; 4,864 over 896, 487
  // workgroups: 6.05 and 6.19).
  const bool through = tiles <= 2 * compute_units();
  fused_decode_kernel<NW, EPI, NORM, UN, ONE, PASSES, LINES, STAGE><<<tiles, NW * WAVE, lds, stream>>>(
      args.w, from_residual ? (const void*)args.residual_in : (const void*)args.a, args.norm_weight,
      (uint32_t)args.m | (uint32_t)args.rows << 8 | (uint32_t)args.d << 16, EPI == EPI_GATED ? (uint32_t)through : (uint32_t)args.n_q | (uint32_t)args.n_kv << 16, args.n, args.k,
      args.lda, args.eps, EPI == EPI_RESIDUAL ? (void*)args.residual_out : (void*)args.out, args.bias, args.positions, args.cos_sin,
      args.slots, args.k_pages, args.v_pages, args.page_size, args.temper_coef, args.temper_every);
  return LAUNCH_STATUS();
}

template <int NW, int EPI, bool NORM, int PASSES>
static int launch_one(const FusedArgs& args, int tiles, hipStream_t stream) {
  // Steps of a wave: pairs of steps are dealt round-robin to the waves.
  const int pairs = (args.k / 32 + 1) / 2;
  const int steps_per_wave = 2 * ((pairs + NW - 1) / NW);
  const bool whole = (args.k & 63) == 0;                     // K in whole cache lines
  // (Rows straight from memory have a trip for all of a short share with the residual epilogue alone: the others' rows lie in LDS while K is short.)
  if constexpr (NORM || EPI == EPI_RESIDUAL)
    if (steps_per_wave <= 4) return launch_kernel<NW, EPI, NORM, 4, true, PASSES>(args, tiles, stream);
  if constexpr (NORM && (EPI == EPI_ROPE_STORE || PASSES == 1)) {
    // Rows in LDS: only the weights take registers, and a wave's whole share of up to eight steps is one trip
    // (rows of 1,025 to 2,048 elements at eight waves: two trips in the loop below; q/k/v at 1,536: 8.4 -> 7.5 us).
    // The gated product's matrix is several workgroups for every compute unit: it takes a whole share at once only
    // while two workgroups' registers fit a unit together, which is one block of rows and six steps (with two blocks
    // of rows 19.9 -> 22.3 us at 8,960 x 1,536, with eight steps 25.4 -> 31.3 us at 11,008 x 2,048).
    if constexpr (EPI == EPI_GATED)
      if (whole && steps_per_wave <= 6) return launch_kernel<NW, EPI, NORM, 6, true, PASSES, true>(args, tiles, stream);
    if (steps_per_wave <= 6) return launch_kernel<NW, EPI, NORM, 6, true, PASSES>(args, tiles, stream);
    if constexpr (EPI == EPI_ROPE_STORE)
      if (steps_per_wave <= 8) return launch_kernel<NW, EPI, NORM, 8, true, PASSES>(args, tiles, stream);
  }
  if constexpr (!NORM && EPI == EPI_RESIDUAL && PASSES == 1) {
    // Rows from memory: one trip for a wave's whole share if it fits the registers (128 a lane at 16 waves).
    if (steps_per_wave <= 8) return launch_kernel<NW, EPI, NORM, 8, true, 1>(args, tiles, stream);
    if (whole && steps_per_wave <= 10) return launch_kernel<NW, EPI, NORM, 10, true, 1, true>(args, tiles, stream);
    if (steps_per_wave <= 10) return launch_kernel<NW, EPI, NORM, 10, true, 1>(args, tiles, stream);
  }
  if constexpr (EPI == EPI_RESIDUAL && PASSES == 1) {
    // One set of weight rows leaves registers for three lines a trip; with more input rows the wider trip gains nothing.  Four steps |
    // six, 8 rows: down 8,960 to 1,536 11.8 | 11.1 us (one row 11.3 | 9.7), 18,944 to 3,584 28.4 | 28.7; 16 rows 14.2 | 14.2, 34.4 | 35.2.
    if (whole && args.m <= 8) return launch_kernel<NW, EPI, NORM, 6, false, PASSES, true>(args, tiles, stream);
  }
  if (whole) return launch_kernel<NW, EPI, NORM, 4, false, PASSES, true>(args, tiles, stream);
  return launch_kernel<NW, EPI, NORM, 4, false, PASSES>(args, tiles, stream);
}

// waves 0: the launcher's choice of how many waves share a workgroup's K.
template <int EPI, bool NORM>
static int launch_rows(const FusedArgs& args, int tiles, int waves, hipStream_t stream) {
  const int k_steps = (args.k + 31) / 32;
  const bool two = args.rows > 16;
  if (waves == 0) waves = (tiles >= 1024 || k_steps <= 8) ? 4 : (tiles >= 256 || k_steps <= 64 || NORM || two) ? 8 : 16;
  if (EPI != EPI_RESIDUAL && waves > 8) waves = 8;           // two sets of weight registers: no room at 16 waves
  if constexpr (EPI != EPI_ROPE_STORE) {
    if (two) {
      if (waves == 4) return launch_one<4, EPI, NORM, 2>(args, tiles, stream);
      return launch_one<8, EPI, NORM, 2>(args, tiles, stream);
    }
  }
  if (waves == 4) return launch_one<4, EPI, NORM, 1>(args, tiles, stream);
  if (waves == 8 || NORM) return launch_one<8, EPI, NORM, 1>(args, tiles, stream);
  if constexpr (EPI == EPI_RESIDUAL) return launch_one<16, EPI, false, 1>(args, tiles, stream);
  return -1;
}

// Weight rows per workgroup for the rotation epilogue, where a block pairs rows half a head apart: 16, 8 or 4.
// Every workgroup reads and normalises all m input rows before its share of the weights, so the choice weighs
// the bytes the busiest compute unit has to ask for: rounds of workgroups x (prologue + its weight rows + what a
// unit could have streamed during the trips to memory that every workgroup begins with; without that last term one
// row of 3,584 took three rounds of four weight rows, 17.7 us, where one round of sixteen takes 14.0).
static int rows_per_tile(int n_q, int n_kv, int n_v, int d, int m, int k, bool norm, int rows_override) {
  if (rows_override == 16 || rows_override == 8 || rows_override == 4) return rows_override;
  const long units = compute_units();
  const long prologue = (long)m * k * (norm ? 8 : 2);       // float rows and the norm weight per row, or bfloat16 rows
  int best = 16;
  long best_cost = -1;
  for (int r = 16; r >= 4; r /= 2) {
    const long tiles = (long)(n_q + n_kv) * (d / 2 / r) + (long)n_v * d / r;
    const long cost = ((tiles + units - 1) / units) * (prologue + 2L * r * k * 2 + 64 * 1024);
    if (best_cost < 0 || cost < best_cost) { best = r; best_cost = cost; }
  }
  return best;
}

// Weight rows per workgroup elsewhere: the matrix is cut into a multiple of the compute units' number of
// equal shares of at most 32 rows, so that every unit streams the same number of bytes; never fewer than 4.
static int rows_per_workgroup(int n_rows, int rows_override) {
  if (rows_override >= 1 && rows_override <= 32) return rows_override;
  const int units = compute_units();
  const int rounds = (n_rows + units * 32 - 1) / (units * 32);
  int rows = (n_rows + units * rounds - 1) / (units * rounds);
  // One round of 17 to 31 rows would be a block of sixteen and a nearly empty second one, one after the other:
  // two workgroups of half the rows on every compute unit, one block each, are over sooner (measured at 4,864
  // rows of 896: 19 rows 8.6 us, 10 rows 8.2 us; with two rounds, 8,960 rows of 1,536, the halves are slower).
  if (rounds == 1 && rows > 16 && rows < 32) rows = (n_rows + 2 * units - 1) / (2 * units);
  return rows < 4 ? 4 : rows;
}

// The gated product from rows in LDS: where the even shares would be two blocks of rows a workgroup (17 to 32) and
// a wave's share of K at eight waves is at most six steps, workgroups of one block whose weights are asked for at
// once are over sooner: as many rounds of workgroups as blocks of sixteen need, in equal shares (8,960 rows of 1,536:
// 18 rows in two blocks 19.9 us, 12 rows 19.3 us at eight input rows; 18.3 and 17.3 us at one).  Up to eight input
// rows: every workgroup brings all of them in first, and half as many workgroups again weigh more than they save
// at sixteen (22.9 and 24.8 us).
static int rows_per_gated_workgroup(int n_rows, int m, int k, int rows_override) {
  int rows = rows_per_workgroup(n_rows, rows_override);
  if (rows_override >= 1 && rows_override <= 32) return rows;
  const int pairs = (k / 32 + 1) / 2;
  if (rows > 16 && m <= 8 && 2 * ((pairs + 7) / 8) <= 6) {
    const int units = compute_units();
    const int rounds = (n_rows + units * 16 - 1) / (units * 16);
    rows = (n_rows + units * rounds - 1) / (units * rounds);
  }
  return rows;
}

// Rows that are normalised already go through LDS (the NORM instances, which then copy instead of normalising)
// while a workgroup's copy fits a compute unit beside its other LDS (measured at a width of 3,584: 1.06x for 8
// rows, where two workgroups' copies fit, level for 12, 1.02x for 16).
static bool stage_rows(int m, int k) { return (size_t)m * (k + 8) * sizeof(uint16_t) <= 120 * 1024; }

static int fused_qkv_rope(const FusedArgs& base, bool norm, const void* w, const void* bias, void* q_out,
                          const void* positions, const void* cos_sin, const void* slots, void* k_pages, void* v_pages,
                          int m, int k, int n_q, int n_kv, int d, int page_size, int rows, int waves, hipStream_t stream,
                          bool tied = false) {
  if (m <= 0) return 0;
  if (m > 16 || (k & 7) || (d & 31)) return -1;
  FusedArgs a = base;
  const int n_v = tied ? 0 : n_kv;                           // (values that are the keys have no rows and no pages of their own)
  a.w = (const bf16_t*)w; a.bias = (const float*)bias; a.m = m; a.n = (n_q + n_kv + n_v) * d; a.k = k;
  a.out = (bf16_t*)q_out; a.ldc = n_q * d;
  a.positions = (const int*)positions; a.cos_sin = (const float*)cos_sin; a.slots = (const int*)slots;
  a.k_pages = (bf16_t*)k_pages; a.v_pages = (bf16_t*)v_pages; a.n_q = n_q; a.n_kv = n_kv; a.d = d; a.page_size = page_size;
  a.rows = rows_per_tile(n_q, n_kv, n_v, d, m, k, norm, rows);
  const int tiles = (n_q + n_kv) * (d / 2 / a.rows) + n_v * d / a.rows;
  if (norm || stage_rows(m, k)) return launch_rows<EPI_ROPE_STORE, true>(a, tiles, waves, stream);
  return launch_rows<EPI_ROPE_STORE, false>(a, tiles, waves, stream);
}

// q/k/v projection of up to 16 rows read from the float residual (normalised on the fly): bias, rotation,
// q into `q_out` [m, n_q * d], keys and values into their pages (slots null or negative: not stored).
// rows / waves: 0 = the launcher's choice of weight rows per workgroup and waves sharing a workgroup's K.
extern "C" int ta_fused_norm_qkv_rope(const void* residual, const void* norm_weight, float eps, const void* w,
                                      const void* bias, void* q_out, const void* positions, const void* cos_sin,
                                      const void* slots, void* k_pages, void* v_pages, int m, int k, int n_q,
                                      int n_kv, int d, int page_size, int rows, int waves, hipStream_t stream) {
  FusedArgs a = {};
  a.residual_in = (const float*)residual; a.norm_weight = (const float*)norm_weight; a.eps = eps;
  return fused_qkv_rope(a, true, w, bias, q_out, positions, cos_sin, slots, k_pages, v_pages, m, k, n_q, n_kv, d,
                        page_size, rows, waves, stream);
}

// The same from rows that are normalised already: x bfloat16 [m, k] with row stride lda.  For wide models, where
// normalising all rows again in every workgroup costs more than one small kernel before this one.
extern "C" int ta_fused_qkv_rope(const void* x, int lda, const void* w, const void* bias, void* q_out,
                                 const void* positions, const void* cos_sin, const void* slots, void* k_pages,
                                 void* v_pages, int m, int k, int n_q, int n_kv, int d, int page_size, int rows,
                                 int waves, hipStream_t stream) {
  if (lda & 7) return -1;
  FusedArgs a = {};
  a.a = (const bf16_t*)x; a.lda = lda;
  return fused_qkv_rope(a, false, w, bias, q_out, positions, cos_sin, slots, k_pages, v_pages, m, k, n_q, n_kv, d,
                        page_size, rows, waves, stream);
}

// The projection of queries and of keys that are the values too, from rows that are normalised already: query heads times
// 1 + coef ln(floor((position + 1) / every) + 1) (coef 0: as they are), keys into the key pages.
extern "C" int ta_fused_qk_temper(const void* x, int lda, const void* w, void* q_out, const void* positions, float coef, int every,
                                  const void* slots, void* k_pages, int m, int k, int n_q, int n_kv, int d, int page_size,
                                  int rows, int waves, hipStream_t stream) {
  if ((lda & 7) || every < 1 || !positions) return -1;
  FusedArgs a = {};
  a.a = (const bf16_t*)x; a.lda = lda; a.temper_coef = coef; a.temper_every = coef == 0.f ? 0 : every;
  return fused_qkv_rope(a, false, w, nullptr, q_out, positions, nullptr, slots, k_pages, nullptr, m, k, n_q, n_kv, d, page_size,
                        rows, waves, stream, true);
}

// out [m, n/2] = silu(x Wg^T) * (x Wu^T), x = the normalised residual rows, W = [Wg; Wu] of shape [n, k].
// act: null for silu, else three floats on the device (alpha, limit, shift): g' = min(g, limit), u' = clamp(u, +-limit),
// out = g' sigmoid(alpha g') (u' + shift).
extern "C" int ta_fused_norm_gated(const void* residual, const void* norm_weight, float eps, const void* w,
                                   void* out, int m, int n, int k, int rows, int waves, const void* act,
                                   hipStream_t stream) {
  if (m <= 0) return 0;
  if (m > 16 || (k & 7) || (n & 1)) return -1;
  FusedArgs a = {};
  a.residual_in = (const float*)residual; a.norm_weight = (const float*)norm_weight; a.eps = eps;
  a.w = (const bf16_t*)w; a.m = m; a.n = n; a.k = k; a.out = (bf16_t*)out; a.ldc = n / 2;
  a.cos_sin = (const float*)act;
  a.rows = rows_per_gated_workgroup(n / 2, m, k, rows);
  return launch_rows<EPI_GATED, true>(a, (n / 2 + a.rows - 1) / a.rows, waves, stream);
}

// The same from rows that are normalised already: x bfloat16 [m, k] with row stride lda.
extern "C" int ta_fused_gated(const void* x, int lda, const void* w, void* out, int m, int n, int k, int rows,
                              int waves, const void* act, hipStream_t stream) {
  if (m <= 0) return 0;
  if (m > 16 || (k & 7) || (lda & 7) || (n & 1)) return -1;
  FusedArgs a = {};
  a.a = (const bf16_t*)x; a.lda = lda;
  a.w = (const bf16_t*)w; a.m = m; a.n = n; a.k = k; a.out = (bf16_t*)out; a.ldc = n / 2;
  a.cos_sin = (const float*)act;
  a.rows = stage_rows(m, k) ? rows_per_gated_workgroup(n / 2, m, k, rows) : rows_per_workgroup(n / 2, rows);
  if (stage_rows(m, k)) return launch_rows<EPI_GATED, true>(a, (n / 2 + a.rows - 1) / a.rows, waves, stream);
  return launch_rows<EPI_GATED, false>(a, (n / 2 + a.rows - 1) / a.rows, waves, stream);
}

// residual [m, n] += x W^T (+ bias), x bfloat16 [m, k] with row stride lda.
extern "C" int ta_fused_linear_residual(const void* x, int lda, const void* w, const void* bias, void* residual,
                                        int m, int n, int k, int rows, int waves, hipStream_t stream) {
  if (m <= 0) return 0;
  if (m > 16 || (k & 7) || (lda & 7)) return -1;
  FusedArgs a = {};
  a.a = (const bf16_t*)x; a.lda = lda; a.w = (const bf16_t*)w; a.bias = (const float*)bias;
  a.m = m; a.n = n; a.k = k; a.residual_out = (float*)residual;
  a.rows = rows_per_workgroup(n, rows);
  return launch_rows<EPI_RESIDUAL, false>(a, (n + a.rows - 1) / a.rows, waves, stream);
}
