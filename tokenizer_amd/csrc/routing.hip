// Routed feed-forwards and the per-layer token input: the choice of experts from float router logits, the gated
// activation of the chosen experts with their weights folded in, and the gate of the token input.
#include "common.h"

__device__ __forceinline__ float rt_gelu_tanh(float z) {
  return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}

// logits: float [n_tokens, n_experts].  For every token the `top` largest logits (the lower index of equals) in falling
// order: chosen [n_tokens, top] and weights [n_tokens, top] = softmax over those logits alone.  A wave a token.
__global__ void __launch_bounds__(256)
route_top_kernel(const float* __restrict__ logits, int n_tokens, int n_experts, int top, int* __restrict__ chosen,
                 float* __restrict__ weights) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int t = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
  if (t >= n_tokens) return;
  const float* row = logits + (size_t)t * n_experts;
  float top_value = 0.f, total = 0.f, mine = 0.f;
  int last = -1;
  float last_value = INFINITY;
  for (int k = 0; k < top; ++k) {
    // The largest logit that comes behind the one picked last in the order (value falling, index rising).
    float best = -INFINITY;
    int best_at = n_experts;
    for (int e = lane; e < n_experts; e += WAVE) {
      const float v = row[e];
      const bool behind = v < last_value || (v == last_value && e > last);
      if (behind && (v > best || (v == best && e < best_at))) { best = v; best_at = e; }
    }
#pragma unroll
    for (int off = WAVE / 2; off > 0; off >>= 1) {
      const float other = __shfl_xor(best, off, WAVE);
      const int other_at = __shfl_xor(best_at, off, WAVE);
      if (other > best || (other == best && other_at < best_at)) { best = other; best_at = other_at; }
    }
    if (k == 0) top_value = best;
    const float e = expf(best - top_value);
    total += e;
    if (lane == k) mine = e;                        // lane k keeps pick k's term
    if (lane == 0) chosen[(size_t)t * top + k] = best_at;
    last = best_at;
    last_value = best;
  }
  // Every lane holds the same total, lane k pick k's term (the launcher takes top <= 64).
  if (lane < top) weights[(size_t)t * top + lane] = mine / total;
}

// Eight bfloat16 elements (sixteen bytes) as floats, and back.
__device__ __forceinline__ void rt_unpack8(const uint4 raw, float (&v)[8]) {
  const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) { v[2 * i] = __uint_as_float(w[i] << 16); v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u); }
}
__device__ __forceinline__ uint4 rt_pack8(const float (&v)[8]) {
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = (uint32_t)float_to_bf16_bits(v[2 * i]) | ((uint32_t)float_to_bf16_bits(v[2 * i + 1]) << 16);
  return make_uint4(w[0], w[1], w[2], w[3]);
}

#define RT_MAX_EXPERTS 256
#define RT_ROW_PIECES 8        // sixteen-byte pieces of a row that a lane keeps: rows of up to 64 * 8 * 8 bfloat16 elements

template <typename T> struct RtVec;
template <> struct RtVec<bf16_t> {
  static constexpr int N = 8;
  __device__ static __forceinline__ void unpack(const uint4 raw, float (&v)[8]) { rt_unpack8(raw, v); }
};
template <> struct RtVec<float> {
  static constexpr int N = 4;
  __device__ static __forceinline__ void unpack(const uint4 raw, float (&v)[4]) {
    v[0] = __uint_as_float(raw.x); v[1] = __uint_as_float(raw.y); v[2] = __uint_as_float(raw.z); v[3] = __uint_as_float(raw.w);
  }
};

// The float sums of a row with router rows wave, wave + WAVES, ... below `count`, handed to `put(row, sum)` in every lane: a lane
// keeps its PIECES pieces of sixteen bytes of the row.  Few rows (AHEAD): the first router row's pieces are asked for beside them, so
// a wave with one row to do makes one trip to memory; many rows hide the trips of one behind the others', and a wave that holds
// half as many registers leaves room for more of them.  (Pieces past the rows' end are the row's last ones again, replaced by zeros.)
template <typename T, int PIECES, int WAVES, bool AHEAD, typename Put>
__device__ __forceinline__ void rt_row_sums(const T* __restrict__ row, const T* __restrict__ router, int hidden, int count, Put put) {
  constexpr int N = RtVec<T>::N;
  const int lane = threadIdx.x & (WAVE - 1), wave = wave_index();
  if (wave >= count) return;
  if (hidden <= 0) {                                         // rows without a piece that could be read
    for (int e = wave; e < count; e += WAVES) put(e, 0.f);
    return;
  }
  uint4 xv[PIECES], wv[PIECES];
  auto ask = [&](const T* from, uint4 (&v)[PIECES]) {
#pragma unroll
    for (int p = 0; p < PIECES; ++p) v[p] = *reinterpret_cast<const uint4*>(from + min((p * WAVE + lane) * N, hidden - N));
  };
  auto inside = [&](int p, const uint4 raw, float (&v)[N]) {        // (nothing is past the end of pieces that are full)
    const bool in = (p * WAVE + lane) * N < hidden;
    RtVec<T>::unpack(make_uint4(in ? raw.x : 0u, in ? raw.y : 0u, in ? raw.z : 0u, in ? raw.w : 0u), v);
  };
  ask(row, xv);
  if (AHEAD) ask(router + (size_t)wave * hidden, wv);
  for (int e = wave; e < count; e += WAVES) {
    float sum = 0.f;
    if (!AHEAD) ask(router + (size_t)e * hidden, wv);
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
      float x[N], w[N];
      inside(p, xv[p], x);
      inside(p, wv[p], w);
#pragma unroll
      for (int k = 0; k < N; ++k) sum = fmaf(w[k], x[k], sum);
    }
    if (AHEAD && e + WAVES < count) ask(router + (size_t)(e + WAVES) * hidden, wv);
    put(e, wave_sum(sum));
  }
}

__device__ __forceinline__ float rt_lane(float v, int lane) {          // (`lane` the same for the whole wave)
  return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), lane));
}

// A lane's place among the wave's first `count` values, one a lane: how many are larger, or as large and of a lower lane.  For values
// that are numbers that is the order in which a search for the largest one after the other finds them.
__device__ __forceinline__ int rt_place(float mine, int lane, int count) {
  int ahead = 0;
  for (int o = 0; o < count; ++o) {
    const float v = rt_lane(mine, o);
    ahead += (v > mine || (v == mine && o < lane)) ? 1 : 0;
  }
  return ahead;
}

// The `top` first of those places: `value` of each, added up in their order.
__device__ __forceinline__ float rt_sum_in_order(float value, int place, int top) {
  float total = 0.f;
  for (int k = 0; k < top; ++k) total += rt_lane(value, (int)__builtin_ctzll(__ballot(place == k)));
  return total;
}

// The router's product and the choice in one kernel, a workgroup a token: x [n_tokens, hidden] (row stride lda) and
// router [n_experts, hidden] of type T in pieces of sixteen bytes; wave w forms the logits of experts w, w + WAVES, ... as
// float sums, wave 0 then picks as route_top_kernel does.  (Three rows of 1,536 and 8 experts: 5.5 us with four waves and loads
// behind branches, 4.4 with a wave an expert; in a graph and with places
// counted in place of searches through LDS 3.7 -> 2.6, four rows of 3,584 4.6 -> 3.4.)
template <typename T, int PIECES, int WAVES>
__global__ void __launch_bounds__(WAVES * WAVE)
route_rows_kernel(const T* __restrict__ x, int lda, const T* __restrict__ router, int hidden, int n_experts, int top,
                  int* __restrict__ chosen, float* __restrict__ weights) {
  __shared__ float logit_s[RT_MAX_EXPERTS];
  const int t = blockIdx.x;
  const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
  rt_row_sums<T, PIECES, WAVES, WAVES == 8>(x + (size_t)t * lda, router, hidden, n_experts,
                                [&](int e, float sum) { if (lane == 0) logit_s[e] = sum; });
  __syncthreads();
  if (wave != 0) return;
  if (n_experts <= WAVE) {
    // An expert a lane: its place among them all is counted, not searched for (a search is twelve exchanges through LDS a pick).
    const float z = lane < n_experts ? logit_s[lane] : -INFINITY;
    if (__ballot(z != z) == 0) {                             // (what is no number has no place: those rows search)
      const int place = lane < n_experts ? rt_place(z, lane, n_experts) : n_experts;
      const float term = expf(z - rt_lane(z, (int)__builtin_ctzll(__ballot(place == 0))));
      const float sum = rt_sum_in_order(term, place, top);
      if (place < top) {
        chosen[(size_t)t * top + place] = lane;
        st(weights + (size_t)t * top + place, term / sum);
      }
      return;
    }
  }
  float top_value = 0.f, total = 0.f, mine = 0.f, last_value = INFINITY;
  int last = -1;
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY;
    int best_at = n_experts;
    for (int e = lane; e < n_experts; e += WAVE) {
      const float v = logit_s[e];
      const bool behind = v < last_value || (v == last_value && e > last);
      if (behind && (v > best || (v == best && e < best_at))) { best = v; best_at = e; }
    }
#pragma unroll
    for (int off = WAVE / 2; off > 0; off >>= 1) {
      const float other = __shfl_xor(best, off, WAVE);
      const int other_at = __shfl_xor(best_at, off, WAVE);
      if (other > best || (other == best && other_at < best_at)) { best = other; best_at = other_at; }
    }
    if (k == 0) top_value = best;
    const float term = expf(best - top_value);
    total += term;
    if (lane == k) mine = term;
    if (lane == 0) chosen[(size_t)t * top + k] = best_at;
    last = best_at;
    last_value = best;
  }
  if (lane < top) weights[(size_t)t * top + lane] = mine / total;
}

// gate_up: [n_tokens, n_experts * 2 * inner + 2 * shared], expert e's gate rows then its up rows, the shared expert
// last.  out: [n_tokens, columns] with columns >= n_experts * inner + shared: out[t, e * inner + i] =
// w * silu(gate) * up for an expert the token chose with weight w, 0 for the others; the shared expert's columns
// with weight 1 (or shared_weight[t], float, where given); columns beyond are 0.  weigh_input: silu(w * gate) * (w * up)
// instead (the expert is handed its row times w).
template <typename T>
__global__ void expert_gate_kernel(const T* __restrict__ gate_up, const int* __restrict__ chosen,
                                   const float* __restrict__ weights, int top, int n_experts, int inner, int shared,
                                   int columns, T* __restrict__ out, size_t total, const float* __restrict__ shared_weight,
                                   int weigh_input) {
  const int in_stride = n_experts * 2 * inner + 2 * shared;
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (size_t)gridDim.x * blockDim.x) {
    const size_t t = idx / columns;
    const int c = (int)(idx - t * columns);
    const T* row = gate_up + t * in_stride;
    float value = 0.f;
    if (c < n_experts * inner) {
      const int e = c / inner, i = c - e * inner;
      float w = 0.f;
      for (int k = 0; k < top; ++k)
        if (chosen[t * top + k] == e) w += weights[t * top + k];
      if (w != 0.f) {
        float g = ld(row + (size_t)e * 2 * inner + i), u = ld(row + (size_t)e * 2 * inner + inner + i);
        if (weigh_input) { g *= w; u *= w; w = 1.f; }
        value = w * (g / (1.0f + expf(-g)) * u);
      }
    } else if (c < n_experts * inner + shared) {
      const int i = c - n_experts * inner;
      const float g = ld(row + (size_t)n_experts * 2 * inner + i), u = ld(row + (size_t)n_experts * 2 * inner + shared + i);
      value = g / (1.0f + expf(-g)) * u;
      if (shared_weight) value *= shared_weight[t];
    }
    st(out + idx, value);
  }
}

// out[t, j] = gelu_tanh(gate[t, j]) * table[token_ids[t], offset + j] for j < dim, 0 for dim <= j < columns.
// gate, out: [n_tokens, columns]; table: [vocab, table_width].
template <typename T>
__global__ void side_gate_kernel(const T* __restrict__ gate, const T* __restrict__ table, int table_width,
                                 const int* __restrict__ token_ids, int offset, int dim, int columns,
                                 T* __restrict__ out, size_t total) {
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (size_t)gridDim.x * blockDim.x) {
    const size_t t = idx / columns;
    const int j = (int)(idx - t * columns);
    float value = 0.f;
    if (j < dim) value = rt_gelu_tanh(ld(gate + idx)) * ld(table + (size_t)token_ids[t] * table_width + offset + j);
    st(out + idx, value);
  }
}

template <bool RELU>
__device__ __forceinline__ float rt_gate_act(float z) { return RELU ? fmaxf(z, 0.f) : rt_gelu_tanh(z); }

// out[t, j] = act(in[t, j]) * in[t, inner + j]: gelu_tanh, or (RELU) max(z, 0).
template <typename T, bool RELU>
__global__ void named_gate_kernel(const T* __restrict__ in, T* __restrict__ out, int inner, size_t total) {
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (size_t)gridDim.x * blockDim.x) {
    const size_t t = idx / inner;
    const int j = (int)(idx - t * inner);
    st(out + idx, rt_gate_act<RELU>(ld(in + t * 2 * inner + j)) * ld(in + t * 2 * inner + inner + j));
  }
}

// expert_gate for bfloat16 with inner, shared and columns multiples of 8: a thread makes eight columns, which lie in
// one expert; the rows of experts a token did not choose are not read.
__global__ void expert_gate_vec_kernel(const bf16_t* __restrict__ gate_up, const int* __restrict__ chosen,
                                       const float* __restrict__ weights, int top, int n_experts, int inner, int shared,
                                       int columns, bf16_t* __restrict__ out, size_t total8,
                                       const float* __restrict__ shared_weight, int weigh_input) {
  const int in_stride = n_experts * 2 * inner + 2 * shared, columns8 = columns / 8;
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total8; idx += (size_t)gridDim.x * blockDim.x) {
    const size_t t = idx / columns8;
    const int c = (int)(idx - t * columns8) * 8;
    const bf16_t* row = gate_up + t * in_stride;
    const bf16_t* g_at = nullptr;
    int up_off = 0;
    float w = 0.f;
    if (c < n_experts * inner) {
      const int e = c / inner, i = c - e * inner;
      for (int k = 0; k < top; ++k)
        if (chosen[t * top + k] == e) w += weights[t * top + k];
      if (w != 0.f) { g_at = row + (size_t)e * 2 * inner + i; up_off = inner; }
    } else if (c < n_experts * inner + shared) {
      g_at = row + (size_t)n_experts * 2 * inner + (c - n_experts * inner);
      up_off = shared;
      w = shared_weight ? shared_weight[t] : 1.f;
    }
    uint4 packed = make_uint4(0, 0, 0, 0);
    if (g_at) {
      float g[8], u[8], v[8];
      rt_unpack8(*reinterpret_cast<const uint4*>(g_at), g);
      rt_unpack8(*reinterpret_cast<const uint4*>(g_at + up_off), u);
      const float before = weigh_input ? w : 1.f, behind = weigh_input ? 1.f : w;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float z = before * g[k];
        v[k] = behind * (z / (1.0f + expf(-z)) * (before * u[k]));
      }
      packed = rt_pack8(v);
    }
    *reinterpret_cast<uint4*>(out + t * columns + c) = packed;
  }
}

// The same for bfloat16 rows whose length is a multiple of 8: sixteen bytes of gate and of up per thread.
template <bool RELU>
__global__ void named_gate_vec_kernel(const bf16_t* __restrict__ in, bf16_t* __restrict__ out, int inner8, size_t total8) {
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total8; idx += (size_t)gridDim.x * blockDim.x) {
    const size_t t = idx / inner8, j = idx - t * inner8;
    const uint4* row = reinterpret_cast<const uint4*>(in) + t * 2 * inner8;
    float g[8], u[8], v[8];
    rt_unpack8(row[j], g);
    rt_unpack8(row[inner8 + j], u);
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = rt_gate_act<RELU>(g[k]) * u[k];
    reinterpret_cast<uint4*>(out)[idx] = rt_pack8(v);
  }
}

// Rows sorted by expert: gate_up [slots, 2 * inner], out [slots, inner]: for pair p (token p / top, its pick p % top) in slot
// slot_of[p], out[slot] = silu(w * gate) * (w * up) with w = weights[p].  Slots of no pair are not written.
template <typename T>
__global__ void expert_gate_slots_kernel(const T* __restrict__ gate_up, const int* __restrict__ slot_of,
                                         const float* __restrict__ weights, int inner, T* __restrict__ out, size_t total) {
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (size_t)gridDim.x * blockDim.x) {
    const size_t p = idx / inner;
    const int i = (int)(idx - p * inner);
    if (slot_of[p] < 0) continue;
    const size_t slot = slot_of[p];
    const float w = weights[p], g = w * ld(gate_up + slot * 2 * inner + i), u = w * ld(gate_up + slot * 2 * inner + inner + i);
    st(out + slot * inner + i, g / (1.0f + expf(-g)) * u);
  }
}

__global__ void expert_gate_slots_vec_kernel(const bf16_t* __restrict__ gate_up, const int* __restrict__ slot_of,
                                             const float* __restrict__ weights, int inner8, bf16_t* __restrict__ out,
                                             size_t total8) {
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total8; idx += (size_t)gridDim.x * blockDim.x) {
    const size_t p = idx / inner8, j = idx - p * inner8;
    if (slot_of[p] < 0) continue;
    const size_t slot = slot_of[p];
    const float w = weights[p];
    const uint4* row = reinterpret_cast<const uint4*>(gate_up) + slot * 2 * inner8;
    float g[8], u[8], v[8];
    rt_unpack8(row[j], g);
    rt_unpack8(row[inner8 + j], u);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float z = w * g[k];
      v[k] = z / (1.0f + expf(-z)) * (w * u[k]);
    }
    reinterpret_cast<uint4*>(out)[slot * inner8 + j] = rt_pack8(v);
  }
}

static inline int rt_blocks(size_t total) { return (int)((total + 255) / 256 < 65535 ? (total + 255) / 256 : 65535); }

extern "C" int ta_route_top(const void* logits, int n_tokens, int n_experts, int top, void* chosen, void* weights,
                            hipStream_t stream) {
  if (n_tokens <= 0) return 0;
  if (top <= 0 || top > n_experts || top > WAVE) return -1;
  route_top_kernel<<<(n_tokens + 3) / 4, 256, 0, stream>>>((const float*)logits, n_tokens, n_experts, top, (int*)chosen,
                                                           (float*)weights);
  return LAUNCH_STATUS();
}

// GO(type, pieces a lane keeps of a row, waves) for these rows: eight while there are no more rows than compute units, else four
// (2,048 rows of 1,536: 14.5 us with eight, 8.4 with four).
#define RT_PIECES(GO, TT, WW) do { const int pieces = (hidden + WAVE * piece - 1) / (WAVE * piece);                         \
    if (pieces <= 1) GO(TT, 1, WW); else if (pieces <= 2) GO(TT, 2, WW); else if (pieces <= 4) GO(TT, 4, WW);               \
    else GO(TT, 8, WW); } while (0)
#define RT_INSTANCES(GO) do { const bool wide = n_tokens <= compute_units();                       \
  if (dtype == DT_F32) { if (wide) RT_PIECES(GO, float, 8); else RT_PIECES(GO, float, 4); }                                  \
  else { if (wide) RT_PIECES(GO, bf16_t, 8); else RT_PIECES(GO, bf16_t, 4); } } while (0)

// Returns -2 for sizes the fused kernel does not take (the caller then forms the logits with a product of its own).
extern "C" int ta_route_rows(const void* x, int lda, const void* router, int n_tokens, int hidden, int n_experts, int top,
                             void* chosen, void* weights, int dtype, hipStream_t stream) {
  if (n_tokens <= 0) return 0;
  if (top <= 0 || top > n_experts || top > WAVE) return -1;
  const int piece = dtype == DT_F32 ? 4 : 8;
  if (n_experts > RT_MAX_EXPERTS || hidden % piece || lda % piece || hidden > WAVE * RT_ROW_PIECES * piece ||
      (((uintptr_t)x | (uintptr_t)router) & 15))
    return -2;
#define ROUTE(TT, PP, WW) route_rows_kernel<TT, PP, WW><<<n_tokens, WW * WAVE, 0, stream>>>((const TT*)x, lda, (const TT*)router, \
    hidden, n_experts, top, (int*)chosen, (float*)weights)
  RT_INSTANCES(ROUTE);
#undef ROUTE
  return LAUNCH_STATUS();
}

extern "C" int ta_expert_gate(const void* gate_up, const void* chosen, const void* weights, int n_tokens, int top,
                              int n_experts, int inner, int shared, int columns, void* out, int dtype,
                              const void* shared_weight, int weigh_input, hipStream_t stream) {
  const size_t total = (size_t)n_tokens * columns;
  if (total == 0) return 0;
  if (columns < n_experts * inner + shared || (weigh_input && shared)) return -1;
  if (dtype == DT_BF16 && inner % 8 == 0 && shared % 8 == 0 && columns % 8 == 0 &&
      (((uintptr_t)gate_up | (uintptr_t)out) & 15) == 0) {
    expert_gate_vec_kernel<<<rt_blocks(total / 8), 256, 0, stream>>>((const bf16_t*)gate_up, (const int*)chosen,
        (const float*)weights, top, n_experts, inner, shared, columns, (bf16_t*)out, total / 8, (const float*)shared_weight,
        weigh_input);
    return LAUNCH_STATUS();
  }
  if (dtype == DT_F32)
    expert_gate_kernel<float><<<rt_blocks(total), 256, 0, stream>>>((const float*)gate_up, (const int*)chosen,
        (const float*)weights, top, n_experts, inner, shared, columns, (float*)out, total, (const float*)shared_weight,
        weigh_input);
  else
    expert_gate_kernel<bf16_t><<<rt_blocks(total), 256, 0, stream>>>((const bf16_t*)gate_up, (const int*)chosen,
        (const float*)weights, top, n_experts, inner, shared, columns, (bf16_t*)out, total, (const float*)shared_weight,
        weigh_input);
  return LAUNCH_STATUS();
}

extern "C" int ta_expert_gate_slots(const void* gate_up, const void* slot_of, const void* weights, int n_pairs, int inner,
                                    void* out, int dtype, hipStream_t stream) {
  const size_t total = (size_t)n_pairs * inner;
  if (n_pairs <= 0 || inner <= 0) return 0;
  if (dtype == DT_BF16 && inner % 8 == 0 && (((uintptr_t)gate_up | (uintptr_t)out) & 15) == 0)
    expert_gate_slots_vec_kernel<<<rt_blocks(total / 8), 256, 0, stream>>>((const bf16_t*)gate_up, (const int*)slot_of,
        (const float*)weights, inner / 8, (bf16_t*)out, total / 8);
  else if (dtype == DT_F32)
    expert_gate_slots_kernel<float><<<rt_blocks(total), 256, 0, stream>>>((const float*)gate_up, (const int*)slot_of,
        (const float*)weights, inner, (float*)out, total);
  else
    expert_gate_slots_kernel<bf16_t><<<rt_blocks(total), 256, 0, stream>>>((const bf16_t*)gate_up, (const int*)slot_of,
        (const float*)weights, inner, (bf16_t*)out, total);
  return LAUNCH_STATUS();
}

extern "C" int ta_side_gate(const void* gate, const void* table, int table_width, const void* token_ids, int offset, int dim,
                            int columns, int n_tokens, void* out, int dtype, hipStream_t stream) {
  const size_t total = (size_t)n_tokens * columns;
  if (total == 0) return 0;
  if (dim > columns || offset < 0 || offset + dim > table_width) return -1;
  if (dtype == DT_F32)
    side_gate_kernel<float><<<rt_blocks(total), 256, 0, stream>>>((const float*)gate, (const float*)table, table_width,
        (const int*)token_ids, offset, dim, columns, (float*)out, total);
  else
    side_gate_kernel<bf16_t><<<rt_blocks(total), 256, 0, stream>>>((const bf16_t*)gate, (const bf16_t*)table, table_width,
        (const int*)token_ids, offset, dim, columns, (bf16_t*)out, total);
  return LAUNCH_STATUS();
}

template <bool RELU>
static int launch_named_gate(const void* in, void* out, int n_tokens, int inner, int dtype, hipStream_t stream) {
  const size_t total = (size_t)n_tokens * inner;
  if (total == 0) return 0;
  if (dtype == DT_BF16 && inner % 8 == 0 && (((uintptr_t)in | (uintptr_t)out) & 15) == 0) {
    named_gate_vec_kernel<RELU><<<rt_blocks(total / 8), 256, 0, stream>>>((const bf16_t*)in, (bf16_t*)out, inner / 8, total / 8);
    return LAUNCH_STATUS();
  }
  if (dtype == DT_F32)
    named_gate_kernel<float, RELU><<<rt_blocks(total), 256, 0, stream>>>((const float*)in, (float*)out, inner, total);
  else
    named_gate_kernel<bf16_t, RELU><<<rt_blocks(total), 256, 0, stream>>>((const bf16_t*)in, (bf16_t*)out, inner, total);
  return LAUNCH_STATUS();
}

extern "C" int ta_gelu_gate(const void* in, void* out, int n_tokens, int inner, int dtype, hipStream_t stream) {
  return launch_named_gate<false>(in, out, n_tokens, inner, dtype, stream);
}

extern "C" int ta_relu_gate(const void* in, void* out, int n_tokens, int inner, int dtype, hipStream_t stream) {
  return launch_named_gate<true>(in, out, n_tokens, inner, dtype, stream);
}

// ---------------------------------------------------------------------------------------------------------------
// A router of sigmoid scores with a correction and groups, and experts without a gate branch.

#define RS_MAX_EXPERTS 1024

// logits: float [n_tokens, n_experts].  s = sigmoid(logit); an expert's choice score is s + correction.  With n_groups > 0
// the experts form that many equal groups of neighbours; a group is worth the sum of its two largest choice scores (its
// one score if it has one expert), and experts outside the `keep` best groups (the lower index of equals) count as minus
// infinity.  The `top` largest choice scores (the lower index of equals) are chosen, in falling order; their weights
// are their s over the sum of the chosen s (+ 1e-20).  A wave a token; the scores of a token lie in LDS.
// The choice among one token's scores in LDS (`choice`: s + correction, `score`: s, `worth`: room for a number a group).
// Every wave that calls it for a token runs the same steps between the same barriers (waves that share a token write
// the same values); `store` says whether this wave writes the token's results.
__device__ __forceinline__ void rs_choose(float* choice, const float* score, float* worth, int lane, int n_experts,
                                          int n_groups, int keep, int top, bool store, int* __restrict__ chosen_row,
                                          float* __restrict__ weights_row, bool group_max = false, bool renormalize = true) {
  if (n_groups > 0) {
    const int per = n_experts / n_groups;
    for (int g = lane; g < n_groups; g += WAVE) {
      float first = -INFINITY, second = -INFINITY;
      for (int i = 0; i < per; ++i) {
        const float v = choice[g * per + i];
        if (v > first) { second = first; first = v; }
        else if (v > second) second = v;
      }
      worth[g] = (per > 1 && !group_max) ? first + second : first;
    }
    __syncthreads();
    for (int g = lane; g < n_groups; g += WAVE) {
      const float mine = worth[g];
      int ahead = 0;
      for (int o = 0; o < n_groups; ++o) {
        const float v = worth[o];
        ahead += (v > mine || (v == mine && o < g)) ? 1 : 0;
      }
      if (ahead >= keep)
        for (int i = 0; i < per; ++i) choice[g * per + i] = -INFINITY;
    }
    __syncthreads();
  }
  float total = 0.f, mine = 0.f;
  int last = -1;
  float last_value = INFINITY;
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY;
    int best_at = n_experts;
    for (int e = lane; e < n_experts; e += WAVE) {
      const float v = choice[e];
      const bool behind = v < last_value || (v == last_value && e > last);
      if (behind && (v > best || (v == best && e < best_at))) { best = v; best_at = e; }
    }
#pragma unroll
    for (int off = WAVE / 2; off > 0; off >>= 1) {
      const float other = __shfl_xor(best, off, WAVE);
      const int other_at = __shfl_xor(best_at, off, WAVE);
      if (other > best || (other == best && other_at < best_at)) { best = other; best_at = other_at; }
    }
    best_at = min(best_at, n_experts - 1);
    const float s = score[best_at];
    total += s;
    if (lane == k) mine = s;
    if (store && lane == 0) chosen_row[k] = best_at;
    last = best_at;
    last_value = best;
  }
  if (store && lane < top) weights_row[lane] = renormalize ? mine / (total + 1e-20f) : mine;
}

__global__ void __launch_bounds__(256)
route_sigmoid_kernel(const float* __restrict__ logits, const float* __restrict__ correction, int n_tokens, int n_experts,
                     int n_groups, int keep, int top, int* __restrict__ chosen, float* __restrict__ weights) {
  extern __shared__ float rs_scratch[];
  const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
  const int slot = blockIdx.x * (blockDim.x / WAVE) + wave;
  const bool live = slot < n_tokens;                          // (a wave past the end works on the last token and stores nothing)
  const int t = live ? slot : n_tokens - 1;
  float* choice = rs_scratch + (size_t)wave * (2 * n_experts + n_groups);
  float* score = choice + n_experts;
  float* worth = score + n_experts;
  const float* row = logits + (size_t)t * n_experts;
  for (int e = lane; e < n_experts; e += WAVE) {
    const float s = 1.0f / (1.0f + expf(-row[e]));
    score[e] = s;
    choice[e] = s + correction[e];
  }
  __syncthreads();
  rs_choose(choice, score, worth, lane, n_experts, n_groups, keep, top, live, chosen + (size_t)t * top, weights + (size_t)t * top);
}

// The same choice from scores of either kind.  logits: float rows of `stride` numbers, the experts' first.  softmax: the
// scores are the softmax over all experts (else sigmoid); correction may be null; group_max: a group is worth its
// largest choice score (else the sum of its two largest); gate (float [n_tokens] or null) gets sigmoid of the number
// behind the experts' logits in the row.  raw: the weights are the chosen scores themselves, not over their sum.  A wave a token.
__global__ void __launch_bounds__(256)
route_scores_kernel(const float* __restrict__ logits, int stride, const float* __restrict__ correction, int n_tokens,
                    int n_experts, int n_groups, int keep, int top, int softmax, int group_max, int* __restrict__ chosen,
                    float* __restrict__ weights, float* __restrict__ gate, int raw) {
  extern __shared__ float rs_scratch[];
  const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
  const int slot = blockIdx.x * (blockDim.x / WAVE) + wave;
  const bool live = slot < n_tokens;                          // (a wave past the end works on the last token and stores nothing)
  const int t = live ? slot : n_tokens - 1;
  float* choice = rs_scratch + (size_t)wave * (2 * n_experts + n_groups);
  float* score = choice + n_experts;
  float* worth = score + n_experts;
  const float* row = logits + (size_t)t * stride;
  float top_logit = -INFINITY, total = 1.f;
  if (softmax) {
    for (int e = lane; e < n_experts; e += WAVE) top_logit = fmaxf(top_logit, row[e]);
    top_logit = wave_max(top_logit);
    total = 0.f;
    for (int e = lane; e < n_experts; e += WAVE) total += expf(row[e] - top_logit);
    total = wave_sum(total);
  }
  for (int e = lane; e < n_experts; e += WAVE) {
    const float s = softmax ? expf(row[e] - top_logit) / total : 1.0f / (1.0f + expf(-row[e]));
    score[e] = s;
    // (Chosen by s alone, without groups: by the logit, whose order is the same and does not end where s rounds to 1.)
    choice[e] = correction ? s + correction[e] : (n_groups > 0 ? s : row[e]);
  }
  if (gate && live && lane == 0) gate[t] = 1.0f / (1.0f + expf(-row[n_experts]));
  __syncthreads();
  rs_choose(choice, score, worth, lane, n_experts, n_groups, keep, top, live, chosen + (size_t)t * top,
            weights + (size_t)t * top, group_max != 0, raw == 0);
}

// The router's product and the choice in one kernel, a token a workgroup (few rows: a decode step): as route_rows_kernel
// forms the logits (float sums of the row with each expert's router row, the row kept in registers), then all
// waves choose together and the first stores.  (Three rows of 896 and 8 experts in 4 groups: 6.8 us with four waves and loads
// behind branches, 5.7 with a wave an expert; in a graph, with the correction on its
// way beside the rows and places counted in registers, four rows of 896 5.05 -> 3.5, of 3,584 6.2 -> 4.5; 64 experts of 2,048 in 8 groups, one
// row, searched 13.7, every expert walked past for a group's two largest 14.0, its own members alone 8.7.)
enum : uint32_t { RS_SOFTMAX = 0x100, RS_GROUP_MAX = 0x200, RS_RAW = 0x400 };     // beside `top`, which is 64 at most
template <typename T, int PIECES, int WAVES>
__global__ void __launch_bounds__(WAVES * WAVE)
route_rows_sigmoid_kernel(const T* __restrict__ x, int lda, const T* __restrict__ router, const float* __restrict__ correction,
                          int hidden, int n_experts, uint32_t groups_keep, uint32_t top_kind, int* __restrict__ chosen,
                          float* __restrict__ weights, float* __restrict__ gate) {
  HELD(x, lda, router, correction, hidden, n_experts, groups_keep, top_kind, chosen);
  extern __shared__ float rs_scratch[];
  float* choice = rs_scratch;
  float* score = choice + n_experts;
  float* worth = score + n_experts;
  const int n_groups = groups_keep & 0xffff, keep = groups_keep >> 16, top = top_kind & 0xff;
  const bool softmax = top_kind & RS_SOFTMAX, group_max = top_kind & RS_GROUP_MAX, raw = top_kind & RS_RAW;
  const int t = blockIdx.x;
  const int lane = threadIdx.x & (WAVE - 1), wave = wave_index();
  const bool few = n_experts <= WAVE;
  float correct = 0.f;                                       // (asked for beside the rows: behind the logits it is a trip of its own)
  if (few && correction) correct = correction[min(lane, n_experts - 1)];
  // (With a gate, the router has one row more: the gate's, behind the experts'.)
  rt_row_sums<T, PIECES, WAVES, WAVES == 8>(x + (size_t)t * lda, router, hidden, n_experts + (gate ? 1 : 0), [&](int e, float sum) {
    if (lane != 0) return;
    if (e == n_experts) st(gate + t, 1.0f / (1.0f + expf(-sum)));
    else score[e] = sum;                                     // the logit, until all of them are there
  });
  __syncthreads();
  if (few) {
    // An expert a lane, every score, worth and place in registers: searches for the largest are exchanges through LDS one behind
    // the other.  Every step gives what the searches below give, in their order of sums.
    const float z = lane < n_experts ? score[lane] : -INFINITY;
    float s;
    if (softmax) {
      const float top_logit = wave_max(z), term = expf(z - top_logit);
      float total = 0.f;
      for (int e = 0; e < n_experts; ++e) total += rt_lane(term, e);
      s = term / total;
    } else {
      s = 1.0f / (1.0f + expf(-z));
    }
    float pick = lane >= n_experts ? -INFINITY : correction ? s + correct : (n_groups > 0 ? s : z);
    if (__ballot(pick != pick || z != z) == 0) {             // (what is no number has no place: those rows search)
      if (wave != 0) return;                                 // (all waves alike: the scores are the same for all)
      if (n_groups > 0) {
        const int per = n_experts / n_groups;
        int group = 0;
        for (int o = per; o < n_experts; o += per) group += lane >= o ? 1 : 0;
        // The two largest of the lane's group, from its own members alone, eight on their way at once.
        float first = -INFINITY, second = -INFINITY;
        for (int j0 = 0; j0 < per; j0 += 8) {
          float v[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) v[j] = __shfl(pick, group * per + min(j0 + j, per - 1), WAVE);
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            if (j0 + j >= per) v[j] = -INFINITY;
            second = v[j] > first ? first : fmaxf(second, v[j]);
            first = fmaxf(first, v[j]);
          }
        }
        const float value = (per > 1 && !group_max) ? first + second : first;
        int ahead = 0;
        for (int g = 0; g < n_groups; ++g) {
          const float v = rt_lane(value, g * per);
          ahead += (v > value || (v == value && g < group)) ? 1 : 0;
        }
        if (ahead >= keep) pick = -INFINITY;
      }
      const int place = lane < n_experts ? rt_place(pick, lane, n_experts) : n_experts;
      const float total = rt_sum_in_order(s, place, top);
      if (place < top) {
        chosen[(size_t)t * top + place] = lane;
        st(weights + (size_t)t * top + place, raw ? s : s / (total + 1e-20f));
      }
      return;
    }
  }
  // Every thread sums the few logits up for itself.
  float top_logit = -INFINITY, total = 0.f;
  if (softmax) {
    for (int e = 0; e < n_experts; ++e) top_logit = fmaxf(top_logit, score[e]);
    for (int e = 0; e < n_experts; ++e) total += expf(score[e] - top_logit);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < n_experts; e += WAVES * WAVE) {
    const float z = score[e], s = softmax ? expf(z - top_logit) / total : 1.0f / (1.0f + expf(-z));
    score[e] = s;
    choice[e] = correction ? s + correction[e] : (n_groups > 0 ? s : z);
  }
  __syncthreads();
  rs_choose(choice, score, worth, lane, n_experts, n_groups, keep, top, wave == 0, chosen + (size_t)t * top,
            weights + (size_t)t * top, group_max, !raw);
}

// up: [n_tokens, n_experts * inner]; out: [n_tokens, columns], columns >= n_experts * inner:
// out[t, e * inner + i] = w * max(up, 0)^2 for an expert the token chose with weight w, 0 for the others and beyond.
template <typename T>
__global__ void expert_act_kernel(const T* __restrict__ up, const int* __restrict__ chosen, const float* __restrict__ weights,
                                  int top, int n_experts, int inner, int columns, T* __restrict__ out, size_t total) {
  const int in_stride = n_experts * inner;
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (size_t)gridDim.x * blockDim.x) {
    const size_t t = idx / columns;
    const int c = (int)(idx - t * columns);
    float value = 0.f;
    if (c < in_stride) {
      const int e = c / inner;
      float w = 0.f;
      for (int k = 0; k < top; ++k)
        if (chosen[t * top + k] == e) w += weights[t * top + k];
      if (w != 0.f) {
        const float z = fmaxf(ld(up + t * in_stride + c), 0.f);
        value = w * (z * z);
      }
    }
    st(out + idx, value);
  }
}

// The same for bfloat16 rows in pieces of eight (inner and columns multiples of eight).
__global__ void expert_act_vec_kernel(const bf16_t* __restrict__ up, const int* __restrict__ chosen,
                                      const float* __restrict__ weights, int top, int n_experts, int inner, int columns,
                                      bf16_t* __restrict__ out, size_t total8) {
  const int in_stride = n_experts * inner, columns8 = columns / 8;
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total8; idx += (size_t)gridDim.x * blockDim.x) {
    const size_t t = idx / columns8;
    const int c = (int)(idx - t * columns8) * 8;
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (c < in_stride) {
      const int e = c / inner;
      float w = 0.f;
      for (int k = 0; k < top; ++k)
        if (chosen[t * top + k] == e) w += weights[t * top + k];
      if (w != 0.f) {
        rt_unpack8(*reinterpret_cast<const uint4*>(up + t * in_stride + c), v);
#pragma unroll
        for (int i = 0; i < 8; ++i) { const float z = fmaxf(v[i], 0.f); v[i] = w * (z * z); }
      }
    }
    *reinterpret_cast<uint4*>(out + idx * 8) = rt_pack8(v);
  }
}

// out = max(in, 0)^2, element by element.
template <typename T>
__global__ void relu2_kernel(const T* __restrict__ in, T* __restrict__ out, size_t total) {
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (size_t)gridDim.x * blockDim.x) {
    const float z = fmaxf(ld(in + idx), 0.f);
    st(out + idx, z * z);
  }
}

__global__ void relu2_vec_kernel(const bf16_t* __restrict__ in, bf16_t* __restrict__ out, size_t total8) {
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total8; idx += (size_t)gridDim.x * blockDim.x) {
    float v[8];
    rt_unpack8(*reinterpret_cast<const uint4*>(in + idx * 8), v);
#pragma unroll
    for (int i = 0; i < 8; ++i) { const float z = fmaxf(v[i], 0.f); v[i] = z * z; }
    *reinterpret_cast<uint4*>(out + idx * 8) = rt_pack8(v);
  }
}

extern "C" int ta_route_sigmoid(const void* logits, const void* correction, int n_tokens, int n_experts, int n_groups,
                                int keep, int top, void* chosen, void* weights, hipStream_t stream) {
  if (n_tokens <= 0) return 0;
  if (top <= 0 || top > n_experts || top > WAVE || n_experts > RS_MAX_EXPERTS || n_groups < 0) return -1;
  if (n_groups > 0 && (n_experts % n_groups || keep <= 0 || keep > n_groups || keep * (n_experts / n_groups) < top)) return -1;
  const size_t lds = (size_t)4 * (2 * n_experts + n_groups) * sizeof(float);
  route_sigmoid_kernel<<<(n_tokens + 3) / 4, 256, lds, stream>>>((const float*)logits, (const float*)correction, n_tokens,
                                                                 n_experts, n_groups, keep, top, (int*)chosen, (float*)weights);
  return LAUNCH_STATUS();
}

extern "C" int ta_route_scores(const void* logits, int stride, const void* correction, int n_tokens, int n_experts,
                               int n_groups, int keep, int top, int softmax, int group_max, void* chosen, void* weights,
                               void* gate, int raw, hipStream_t stream) {
  if (n_tokens <= 0) return 0;
  if (top <= 0 || top > n_experts || top > WAVE || n_experts > RS_MAX_EXPERTS || n_groups < 0) return -1;
  if (stride < n_experts + (gate ? 1 : 0)) return -1;
  if (n_groups > 0 && (n_experts % n_groups || keep <= 0 || keep > n_groups || keep * (n_experts / n_groups) < top)) return -1;
  const size_t lds = (size_t)4 * (2 * n_experts + n_groups) * sizeof(float);
  route_scores_kernel<<<(n_tokens + 3) / 4, 256, lds, stream>>>((const float*)logits, stride, (const float*)correction,
      n_tokens, n_experts, n_groups, keep, top, softmax, group_max, (int*)chosen, (float*)weights, (float*)gate, raw);
  return LAUNCH_STATUS();
}

// The same for scores of either kind (see route_scores_kernel): router [n_experts (+ 1 with a gate), hidden].
extern "C" int ta_route_rows_scores(const void* x, int lda, const void* router, const void* correction, int n_tokens,
                                    int hidden, int n_experts, int n_groups, int keep, int top, int softmax, int group_max,
                                    void* chosen, void* weights, void* gate, int raw, int dtype, hipStream_t stream) {
  if (n_tokens <= 0) return 0;
  if (top <= 0 || top > n_experts || top > WAVE || n_groups < 0) return -1;
  if (n_groups > 0 && (n_experts % n_groups || keep <= 0 || keep > n_groups || keep * (n_experts / n_groups) < top)) return -1;
  const int piece = dtype == DT_F32 ? 4 : 8;
  if (n_experts > RT_MAX_EXPERTS || hidden % piece || lda % piece || hidden > WAVE * RT_ROW_PIECES * piece ||
      (((uintptr_t)x | (uintptr_t)router) & 15))
    return -2;
  const size_t lds = (size_t)(2 * n_experts + n_groups) * sizeof(float);
#define ROUTE(TT, PP, WW) route_rows_sigmoid_kernel<TT, PP, WW><<<n_tokens, WW * WAVE, lds, stream>>>((const TT*)x, lda, \
    (const TT*)router, (const float*)correction, hidden, n_experts, (uint32_t)n_groups | (uint32_t)(n_groups > 0 ? keep : 0) << 16, \
    (uint32_t)top | (softmax ? RS_SOFTMAX : 0u) | (group_max ? RS_GROUP_MAX : 0u) | (raw ? RS_RAW : 0u), (int*)chosen, (float*)weights, \
    (float*)gate)
  RT_INSTANCES(ROUTE);
#undef ROUTE
  return LAUNCH_STATUS();
}

// Returns -2 for sizes the fused kernel does not take (the caller then forms the logits with a product of its own).
extern "C" int ta_route_rows_sigmoid(const void* x, int lda, const void* router, const void* correction, int n_tokens,
                                     int hidden, int n_experts, int n_groups, int keep, int top, void* chosen, void* weights,
                                     int dtype, hipStream_t stream) {
  if (n_tokens <= 0) return 0;
  if (top <= 0 || top > n_experts || top > WAVE || n_groups < 0) return -1;
  if (n_groups > 0 && (n_experts % n_groups || keep <= 0 || keep > n_groups || keep * (n_experts / n_groups) < top)) return -1;
  const int piece = dtype == DT_F32 ? 4 : 8;
  if (n_experts > RT_MAX_EXPERTS || hidden % piece || lda % piece || hidden > WAVE * RT_ROW_PIECES * piece ||
      (((uintptr_t)x | (uintptr_t)router) & 15))
    return -2;
  const size_t lds = (size_t)(2 * n_experts + n_groups) * sizeof(float);
#define ROUTE(TT, PP, WW) route_rows_sigmoid_kernel<TT, PP, WW><<<n_tokens, WW * WAVE, lds, stream>>>((const TT*)x, lda, \
    (const TT*)router, (const float*)correction, hidden, n_experts, (uint32_t)n_groups | (uint32_t)(n_groups > 0 ? keep : 0) << 16, \
    (uint32_t)top, (int*)chosen, (float*)weights, nullptr)
  RT_INSTANCES(ROUTE);
#undef ROUTE
  return LAUNCH_STATUS();
}

extern "C" int ta_expert_act(const void* up, const void* chosen, const void* weights, int n_tokens, int top, int n_experts,
                             int inner, int columns, void* out, int dtype, hipStream_t stream) {
  const size_t total = (size_t)n_tokens * columns;
  if (total == 0) return 0;
  if (columns < n_experts * inner) return -1;
  if (dtype == DT_BF16 && inner % 8 == 0 && columns % 8 == 0 && (((uintptr_t)up | (uintptr_t)out) & 15) == 0) {
    expert_act_vec_kernel<<<rt_blocks(total / 8), 256, 0, stream>>>((const bf16_t*)up, (const int*)chosen,
        (const float*)weights, top, n_experts, inner, columns, (bf16_t*)out, total / 8);
    return LAUNCH_STATUS();
  }
  if (dtype == DT_F32)
    expert_act_kernel<float><<<rt_blocks(total), 256, 0, stream>>>((const float*)up, (const int*)chosen,
        (const float*)weights, top, n_experts, inner, columns, (float*)out, total);
  else
    expert_act_kernel<bf16_t><<<rt_blocks(total), 256, 0, stream>>>((const bf16_t*)up, (const int*)chosen,
        (const float*)weights, top, n_experts, inner, columns, (bf16_t*)out, total);
  return LAUNCH_STATUS();
}

extern "C" int ta_relu2(const void* in, void* out, size_t total, int dtype, hipStream_t stream) {
  if (total == 0) return 0;
  if (dtype == DT_BF16 && total % 8 == 0 && (((uintptr_t)in | (uintptr_t)out) & 15) == 0)
    relu2_vec_kernel<<<rt_blocks(total / 8), 256, 0, stream>>>((const bf16_t*)in, (bf16_t*)out, total / 8);
  else if (dtype == DT_F32)
    relu2_kernel<float><<<rt_blocks(total), 256, 0, stream>>>((const float*)in, (float*)out, total);
  else
    relu2_kernel<bf16_t><<<rt_blocks(total), 256, 0, stream>>>((const bf16_t*)in, (bf16_t*)out, total);
  return LAUNCH_STATUS();
}
