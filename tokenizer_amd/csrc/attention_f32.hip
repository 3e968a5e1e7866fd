// Attention over paged keys and values in 32 bits, on the matrix cores' float instructions (v_mfma_f32_16x16x4_f32: 32-bit
// operands, 32-bit sums).  The conventions of tokens, pages, window, chunk, slopes, sinks, kept first keys, value heads and
// capped scores are those of attention_generic.hip, which keeps the forms this kernel has no instance for (values that are
// the keys, head sizes that are no multiples of four or beyond 256, pages that are no multiples of sixteen keys).
#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

struct F32Args {
  const float* q; int q_stride; float* out; const float* k_pages; const float* v_pages;
  const int* tiles; const int* cu_q; const int* first_position; const int* rows; const int* positions;
  const int* entry_of_token; const int* block_table; int table_stride; int n_q, n_kv, d, dv, page_size, window; float scale;
  int chunk; const float* slopes; const float* sinks; int keep_first, n_v; float softcap; int splits; float* part_o; float* part_ml;
};

// A workgroup takes sixteen queries that see the same pages: SINGLE, the heads of one key head of one token (and one part
// of its keys); else sixteen tokens of a portion under one head.  Its waves walk the blocks of sixteen keys in turn and
// bring their softmax states together through LDS at the end (eight where a single token's keys are one part and few).  With the queries as columns of S^T = K Q^T, lane (column c,
// g) gets the scores of keys 4 g .. 4 g + 3; summed over the keys in the order j, g those are, as they stand, the right
// operand of O^T = V^T P^T, and the left one, keys 4 g .. 4 g + 3 of a row of V^T, is one load of sixteen bytes from the
// value page.  No operand goes through LDS.  S: blocks of sixteen coordinates.  Bound by the matrix cores while the
// workgroups fill the device (2 S x 4 instructions of 32 clocks a block), by a block's trip from memory otherwise: the next
// block's keys and values are asked for before the current one is worked on.
// (14 / 2 heads of 64, portions of 77 to 700 tokens, 1,273 in all: 315 us with a workgroup a token and head on vector
// multiply-adds, 39 with this; four single tokens behind as many keys 28.6 and 6.7 + 3.6 for the merge.)
template <int S, bool SINGLE, int WAVES>
__global__ void __launch_bounds__(WAVES * WAVE)
attention_f32_kernel(F32Args p) {
  __shared__ float m_s[WAVES][16], l_s[WAVES][16];
  __shared__ float acc_s[WAVES][S * 16][17];
  const int lane = threadIdx.x & 63, wave = wave_index(), c = lane & 15, g = lane >> 4;
  const int group = p.n_q / p.n_kv, head_blocks = (group + 15) / 16;
  int entry, kvh, head, row, pos, first_pos, last_pos;     // head, row, pos: this column's query
  bool valid;
  if (SINGLE) {
    row = p.rows ? scalar_int(p.rows + blockIdx.z) : (int)blockIdx.z;
    if (row < 0) return;
    entry = scalar_int(p.entry_of_token + row);
    if (entry < 0) return;
    kvh = blockIdx.y / head_blocks;
    const int in_group = blockIdx.y % head_blocks * 16 + c;
    valid = in_group < group;
    head = kvh * group + min(in_group, group - 1);
    pos = first_pos = last_pos = scalar_int(p.positions + row);
  } else {
    entry = scalar_int(p.tiles + 2 * blockIdx.x);
    const int offset = scalar_int(p.tiles + 2 * blockIdx.x + 1);
    const int row0 = scalar_int(p.cu_q + entry), count = scalar_int(p.cu_q + entry + 1) - row0 - offset;
    if (count <= 0) return;                                // a tile that only fills the step up
    head = blockIdx.y;
    kvh = head / group;
    valid = c < count;
    row = row0 + offset + min(c, count - 1);
    first_pos = scalar_int(p.first_position + entry) + offset;
    pos = first_pos + min(c, count - 1);
    last_pos = first_pos + min(15, count - 1);
  }
  const int vh = kvh / (p.n_kv / p.n_v);
  const int* table = p.block_table + (size_t)entry * p.table_stride;
  auto low_of = [&](int at) {
    int lo = p.window >= 0 && at > p.window ? at - p.window : 0;
    return p.chunk > 0 ? max(lo, at / p.chunk * p.chunk) : lo;
  };
  const int lo = low_of(pos), lo_first = low_of(first_pos), lo_last = low_of(last_pos), lo_block = lo_first / 16;
  // Blocks of sixteen keys in the order they are walked: the kept first ones, then from the first any query sees.
  const int kept = min((min(p.keep_first, last_pos + 1) + 15) / 16, lo_block);
  const int blocks = kept + last_pos / 16 - lo_block + 1;
  int begin = 0, end = blocks;
  if (SINGLE) {                                            // this workgroup's part of them
    const int part = (blocks + p.splits - 1) / p.splits;
    begin = blockIdx.x * part;
    end = min(blocks, begin + part);
  }
  auto first_key = [&](int index) { return 16 * (index < kept ? index : lo_block + index - kept); };

  f32x4 q[S], k[S], v[S], k_next[S], v_next[S];
  const float* q_row = p.q + (size_t)row * p.q_stride + (size_t)head * p.d;
#pragma unroll
  for (int i = 0; i < S; ++i) {
    const int at = 16 * i + 4 * g;
    q[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (at < p.d) q[i] = *reinterpret_cast<const f32x4*>(q_row + at);
  }
  auto ask = [&](int index) {
    const int key = first_key(min(index, end - 1));        // (the last block again where there is no further one)
    const int page = scalar_int(table + key / p.page_size), off = key % p.page_size;
    const float* k_row = p.k_pages + ((size_t)(page * p.n_kv + kvh) * p.page_size + off + c) * p.d;
    const float* v_col = p.v_pages + (size_t)(page * p.n_v + vh) * p.dv * p.page_size + off + 4 * g;
#pragma unroll
    for (int i = 0; i < S; ++i) {
      // (Past a row's end its first piece, which then meets zeros of the other operand or rows that nobody stores.)
      const int at = 16 * i + 4 * g, r = 16 * i + c;
      k_next[i] = *reinterpret_cast<const f32x4*>(k_row + (at < p.d ? at : 0));
      v_next[i] = *reinterpret_cast<const f32x4*>(v_col + (size_t)(r < p.dv ? r : 0) * p.page_size);
    }
  };
  f32x4 acc[S];
#pragma unroll
  for (int i = 0; i < S; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;                            // of this column; l: this lane's keys only, until the end
  const float slope = p.slopes ? p.slopes[head] : 0.f;
  if (begin + wave < end) ask(begin + wave);
  for (int index = begin + wave; index < end; index += WAVES) {
    const int block0 = first_key(index), key0 = block0 + 4 * g;
#pragma unroll
    for (int i = 0; i < S; ++i) { k[i] = k_next[i]; v[i] = v_next[i]; }
    // Keys that some query of the workgroup does not see: a value must not meet their weight, be it zero, if it is no number
    // or infinite.
    const bool partly = block0 + 15 > first_pos || (block0 < lo_last && block0 + 15 >= p.keep_first);
    if (partly) {
      // Of keys that none sees (behind the last query, where nobody may have written, or between the kept first keys and the
      // window) nothing is used.
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int key = key0 + j;
        const bool used = key <= last_pos && (key >= lo_first || key < p.keep_first);
#pragma unroll
        for (int i = 0; i < S; ++i) v[i][j] = used ? v[i][j] : 0.f;
      }
    }
    ask(index + WAVES);
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;              // two chains of sums
#pragma unroll
    for (int i = 0; i < S; ++i) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float kv = 16 * i + 4 * g < p.d ? k[i][e] : 0.f;
        if (e & 1) s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kv, q[i][e], s1, 0, 0, 0);
        else s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kv, q[i][e], s0, 0, 0, 0);
      }
    }
    float score[4], top = -INFINITY;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int key = key0 + j;
      float s = (s0[j] + s1[j]) * p.scale - slope * (float)(pos - key);
      if (p.softcap > 0.f) s = p.softcap * tanhf(s / p.softcap);
      const bool seen = key <= pos && (key >= lo || key < p.keep_first);
      score[j] = seen ? s : -INFINITY;
      top = fmaxf(top, score[j]);
    }
    top = fmaxf(top, __shfl_xor(top, 16, WAVE));
    top = fmaxf(top, __shfl_xor(top, 32, WAVE));
    const float m_new = fmaxf(m, top), base = m_new == -INFINITY ? 0.f : m_new;
    const float keep = expf(m - base);                     // (0 on the first block)
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) { score[j] = expf(score[j] - base); sum += score[j]; }
    l = l * keep + sum;
    m = m_new;
#pragma unroll
    for (int i = 0; i < S; ++i) acc[i] *= keep;
    if (!SINGLE && partly) {
      float extremes = 0.f;                                // no number if one of the values is none, or infinite
#pragma unroll
      for (int i = 0; i < S; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) extremes = fmaf(v[i][j], 0.f, extremes);
      if (__ballot(extremes != 0.f)) {
        // Such a value goes to the queries that see its key and to no other: the block's products one key after the other.
        // Lane (c, g) holds the sums of coordinates 4 g .. 4 g + 3 of each sixteen for query c.
        for (int from = 0; from < 4; ++from)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int key = block0 + 4 * from + j;
            const float weight = __shfl(score[j], 16 * from + c, WAVE);
            const bool seen = key <= pos && (key >= lo || key < p.keep_first);
#pragma unroll
            for (int i = 0; i < S; ++i)
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const float value = __shfl(v[i][j], 16 * from + 4 * g + e, WAVE);
                if (seen) acc[i][e] = fmaf(value, weight, acc[i][e]);
              }
          }
#pragma unroll
        for (int i = 0; i < S; ++i) v[i] = f32x4{0.f, 0.f, 0.f, 0.f};      // (all of it is in the sums)
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < S; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[i][j], score[j], acc[i], 0, 0, 0);
  }
  l += __shfl_xor(l, 16, WAVE);
  l += __shfl_xor(l, 32, WAVE);
  if (g == 0) { m_s[wave][c] = m; l_s[wave][c] = l; }
#pragma unroll
  for (int i = 0; i < S; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc_s[wave][16 * i + 4 * g + j][c] = acc[i][j];
  __syncthreads();
  // Each lane keeps its column; the workgroup's sixteen groups of sixteen lanes take the coordinates in turn.
  float big = -INFINITY;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) big = fmaxf(big, m_s[w][c]);
  // (A sink joins the first part's softmax.)
  const bool with_sink = p.sinks && (!SINGLE || blockIdx.x == 0);
  if (with_sink) big = fmaxf(big, p.sinks[head]);
  const float base = big == -INFINITY ? 0.f : big;
  float weight[WAVES], total = with_sink ? expf(p.sinks[head] - base) : 0.f;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) { weight[w] = expf(m_s[w][c] - base); total += l_s[w][c] * weight[w]; }
  if (!valid) return;
  const bool whole = !SINGLE || p.splits == 1;
  const size_t item = SINGLE ? ((size_t)blockIdx.z * p.n_q + head) * p.splits + blockIdx.x : 0;
  float* dst = whole ? p.out + ((size_t)row * p.n_q + head) * p.dv : p.part_o + item * p.dv;
  const float inv = whole ? 1.0f / total : 1.0f;
  for (int i = threadIdx.x >> 4; i < p.dv; i += WAVES * 4) {
    float o = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) o += acc_s[w][i][c] * weight[w];
    dst[i] = o * inv;
  }
  if (!whole && threadIdx.x < 16) { p.part_ml[2 * item] = big; p.part_ml[2 * item + 1] = total; }
}

// out = the parts of a single token's keys under one maximum and sum; a wave a (token, head), COLS coordinates a lane, 64 apart.  Up to 64
// parts: a part a lane brings maxima and sums and makes the weights, and beside them up to 64 numbers of a lane are on their way at once: one or
// two trips to memory for what was one for every eight parts of every 64 coordinates.  (Attention and merge, us, eight parts of 64 coordinates
// a trip behind two passes over the maxima | behind one | so: one row of 12 heads of 128 on two, 3,000 keys 14.0 | 15.8 | 10.7, of 32 of 256
// on four 24.3 | 28.0 | 17.3; four rows of 28 of 128 on four, 1,500 keys 15.0 | 16.0 | 13.1, of 14 of 64 on two, 500 keys 8.0 | 8.0 | 7.5.)
template <int COLS>
__global__ void __launch_bounds__(WAVE)
attention_f32_merge_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml, const int* __restrict__ rows,
                           float* __restrict__ out, int n_q, int dv, int splits, const int* __restrict__ entry_of_token) {
  HELD(part_o, part_ml, rows, out, n_q, dv, splits, entry_of_token);
  const int item = blockIdx.x / n_q, head = blockIdx.x % n_q, lane = threadIdx.x;
  const int row = rows ? scalar_int(rows + item) : item;
  if (row < 0 || scalar_int(entry_of_token + row) < 0) return;
  const size_t base = ((size_t)item * n_q + head) * splits;
  const float2* ml = reinterpret_cast<const float2*>(part_ml) + base;
  float* dst = out + ((size_t)row * n_q + head) * dv;
  if (splits <= WAVE) {
    constexpr int RUN = 8, RUNS = WAVE / RUN / COLS;         // parts that are asked for behind one question whether there are any
    const float* from = part_o + base * dv;
    float2 stat = ml[min(lane, splits - 1)];
    float v[RUNS][RUN][COLS], o[COLS], weight = 0.f, denom = 0.f;
    int at[COLS];
#pragma unroll
    for (int c = 0; c < COLS; ++c) { at[c] = min(lane + c * WAVE, dv - 1); o[c] = 0.f; }
    for (int s0 = 0; s0 < splits; s0 += RUNS * RUN) {
#pragma unroll
      for (int r = 0; r < RUNS; ++r) {
        if (s0 + r * RUN >= splits) break;
#pragma unroll
        for (int j = 0; j < RUN; ++j)
#pragma unroll
          for (int c = 0; c < COLS; ++c) v[r][j][c] = from[min(s0 + r * RUN + j, splits - 1) * dv + at[c]];
      }
      if (s0 == 0) {
        if (lane >= splits) stat = make_float2(-INFINITY, 0.f);
        const float big = wave_max(stat.x);
        weight = lane < splits ? expf(stat.x - big) : 0.f;
        denom = wave_sum(stat.y * weight);
      }
#pragma unroll
      for (int r = 0; r < RUNS; ++r) {
        if (s0 + r * RUN >= splits) break;
#pragma unroll
        for (int j = 0; j < RUN; ++j) {
          const int s = s0 + r * RUN + j;
          const float w = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(weight), s));      // (0 past the last part)
#pragma unroll
          for (int c = 0; c < COLS; ++c) o[c] = fmaf(s < splits ? v[r][j][c] : 0.f, w, o[c]);
        }
      }
    }
#pragma unroll
    for (int c = 0; c < COLS; ++c)
      if (lane + c * WAVE < dv) dst[lane + c * WAVE] = o[c] / denom;
    return;
  }
  float big = -INFINITY;
  for (int s = lane; s < splits; s += WAVE) big = fmaxf(big, ml[s].x);
  big = wave_max(big);
  float denom = 0.f;
  for (int s = lane; s < splits; s += WAVE) denom += ml[s].y * expf(ml[s].x - big);
  denom = wave_sum(denom);
  for (int i = lane; i < dv; i += WAVE) {
    float o = 0.f;
#pragma unroll 8
    for (int s = 0; s < splits; ++s) o += part_o[(base + s) * dv + i] * expf(ml[s].x - big);
    dst[i] = o / denom;
  }
}

// tiles [n_tiles, 2]: the portions' tiles of sixteen tokens (entry, offset); rows [n_single] (null: the tokens 0 .. n_single - 1
// of a step of single tokens): the single tokens, whose keys are cut into `splits` parts (part_o float [n_single, n_q, splits,
// dv], part_ml float [.., 2] where that is more than one).  -2: no instance for this form.
extern "C" int ta_paged_attention_f32(const void* q, int q_stride, void* out, const void* k_pages, const void* v_pages,
                                      const void* tiles, int n_tiles, const void* cu_q, const void* first_position,
                                      const void* rows, int n_single, const void* positions, const void* entry_of_token,
                                      const void* block_table, int table_stride, int n_q, int n_kv, int d, int dv,
                                      int page_size, int window, float scale, int chunk, const void* slopes, const void* sinks,
                                      int keep_first, int n_v, float softcap, int splits, void* part_o, void* part_ml,
                                      hipStream_t stream) {
  if (n_kv <= 0 || n_q % n_kv || n_v <= 0 || n_kv % n_v || keep_first < 0 || splits < 1) return -1;
  if (!v_pages || d % 4 || d > 256 || dv > 256 || d <= 0 || dv <= 0 || page_size % 16 || q_stride % 4 || n_single > 65535 ||
      (((uintptr_t)q | (uintptr_t)k_pages | (uintptr_t)v_pages) & 15))
    return -2;
  if (n_single > 0 && splits > 1 && (!part_o || !part_ml)) return -1;
  const F32Args args = {(const float*)q, q_stride, (float*)out, (const float*)k_pages, (const float*)v_pages, (const int*)tiles,
                        (const int*)cu_q, (const int*)first_position, (const int*)rows, (const int*)positions,
                        (const int*)entry_of_token, (const int*)block_table, table_stride, n_q, n_kv, d, dv, page_size, window,
                        scale, chunk, (const float*)slopes, (const float*)sinks, keep_first, n_v, softcap, splits,
                        (float*)part_o, (float*)part_ml};
  const int blocks = ((d > dv ? d : dv) + 15) / 16;
  const dim3 many(n_tiles, n_q), few(splits, n_kv * ((n_q / n_kv + 15) / 16), n_single);
  // Single tokens whose keys are not cut: eight waves while workgroups are few (up to 512 keys, 128 rows of head size 64, 300 keys
  // 11.4 -> 10.4 us; 512 rows 19.3 -> 23.3, so not there) and two of them fit a unit's registers (up to 128 coordinates).
  const bool wide = splits == 1 && blocks <= 8 && (long)few.y * n_single <= 256;
#define GO(SS) do {                                                                                                  \
    if (n_tiles > 0) attention_f32_kernel<SS, false, 4><<<many, 4 * WAVE, 0, stream>>>(args);                        \
    if (n_single > 0 && wide) attention_f32_kernel<SS, true, (SS <= 8 ? 8 : 4)><<<few, (SS <= 8 ? 8 : 4) * WAVE, 0, stream>>>(args); \
    else if (n_single > 0) attention_f32_kernel<SS, true, 4><<<few, 4 * WAVE, 0, stream>>>(args);                    \
  } while (0)
  if (blocks <= 1) GO(1); else if (blocks <= 2) GO(2); else if (blocks <= 4) GO(4); else if (blocks <= 6) GO(6);
  else if (blocks <= 8) GO(8); else if (blocks <= 12) GO(12); else GO(16);
#undef GO
  int status = LAUNCH_STATUS();
  if (status == 0 && n_single > 0 && splits > 1) {
#define GO(COLS) attention_f32_merge_kernel<COLS><<<n_single * n_q, WAVE, 0, stream>>>((const float*)part_o, (const float*)part_ml, \
      (const int*)rows, (float*)out, n_q, dv, splits, (const int*)entry_of_token)
    if (dv <= 64) GO(1); else if (dv <= 128) GO(2); else GO(4);
#undef GO
    status = LAUNCH_STATUS();
  }
  return status;
}
