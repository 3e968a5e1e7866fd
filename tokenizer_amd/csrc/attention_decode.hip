// Attention of single query tokens over paged bfloat16 keys and values on the matrix cores, with the
// key range of every token split over several workgroups (partial results are merged by a second kernel).
//
// One workgroup handles one (token, kv head, block of up to 16 query heads, split).  The query heads that
// share a kv head form the N dimension of the 16x16x32 MFMA, so keys and values are read once for all of
// them.  Both products are computed transposed, S^T = K Q^T and O^T = V^T P^T, which keeps the head index
// in `lane % 16` for scores and outputs alike: the online-softmax rescaling needs no cross-lane traffic.
// Values are stored transposed inside a page ([page, kv head, d, slot]), so that the eight keys a lane
// contracts over are contiguous in memory.
#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));


__device__ __forceinline__ bf16x8 zero8() {
  bf16x8 z;
#pragma unroll
  for (int i = 0; i < 8; ++i) z[i] = (__bf16)0.0f;
  return z;
}

// D: head size (multiple of 16).  Pages: K [n_pages, n_kv, page_size, D], V^T [n_pages, n_kv, D, page_size],
// page_size a multiple of 16.  rows: the token rows to serve (null: row i = item i; a negative row is passed over).
// Token at position p sees keys max(0, p - window)..p (window < 0: from 0).
// Partials: part_o [n_items, n_q, splits, D] (unnormalised), part_ml [n_items, n_q, splits, 2] (max, sum);
// with splits == 1 the result goes straight to `out` [n_tokens, n_q * D].
// AHEAD: a wave asks for its next block of keys while it works on the current one (see below).
// EXTRA also: keep_first > 0 (with a window): keys at positions below keep_first stay visible behind the window; the
// last `kept_splits` of the `splits` workgroups of a row walk those keys (positions 0 .. min(keep_first, first key of
// the window) - 1) and leave their partial state beside the others'.  n_v < n_kv: the value pages hold n_v heads and
// key head g reads value head g / (n_kv / n_v).
// EXTRA: chunk > 0: only the keys of the token's own run of `chunk` positions (runs counted from position 0) are seen;
// slopes (float [n_q] or null): head h's score loses slopes[h] per position between token and key; softcap > 0: a
// score s (scaled, with its distance term) becomes softcap * tanh(s / softcap).
// sinks (float [n_q] or null): exp(sinks[h]) joins the softmax's denominator (it rides in the first split's partial sums).
// TIED: the values are the keys, and only the key pages are read: a wave leaves its block of keys in LDS as it came, key by
// key, and takes the eight keys of a coordinate that the second product wants from there (`transposed_keys`).
template <int D, int DEC_WAVES, bool AHEAD, bool EXTRA, bool TIED>
__global__ void __launch_bounds__(DEC_WAVES * WAVE)
decode_attention_kernel(const bf16_t* __restrict__ q, int q_stride, bf16_t* __restrict__ out,
                        const bf16_t* __restrict__ k_pages, const bf16_t* __restrict__ vt_pages,
                        const int* __restrict__ rows, const int* __restrict__ positions,
                        const int* __restrict__ entry_of_token, const int* __restrict__ block_table,
                        int table_stride, float* __restrict__ part_o, float* __restrict__ part_ml,
                        int n_q, int n_kv, int page_size, int window, float scale, int split_keys, int splits, int deal,
                        int chunk, const float* __restrict__ slopes, const float* __restrict__ sinks,
                        int keep_first, int kept_splits, int n_v, float softcap) {
  constexpr int KS = (D + 31) / 32;   // 32-wide steps over the head size for Q K^T
  constexpr int DB = D / 16;          // 16-row blocks of O^T
  HELD(q, q_stride, out, k_pages, vt_pages, rows, positions, entry_of_token, block_table, table_stride, part_o, part_ml,
       n_q, n_kv, page_size, window, scale, split_keys, splits, sinks);
  // (The waves' blocks of keys, where they are kept, lie where the waves' sums lie afterwards.)
  constexpr int SUMS = DEC_WAVES * D * 17 * 4, STAGES = TIED ? DEC_WAVES * KeyStage<D>::BYTES : 0;
  __shared__ __attribute__((aligned(16))) char shared_s[SUMS > STAGES ? SUMS : STAGES];
  float (*acc_s)[D][17] = reinterpret_cast<float (*)[D][17]>(shared_s);
  __shared__ float m_s[DEC_WAVES][16], l_s[DEC_WAVES][16];

  const int group = n_q / n_kv;
  const int head_blocks = (group + 15) / 16;
  // Chiplets get every eighth workgroup, and a chiplet's compute units take those in turn.  With an even count of parts the same
  // parts of all rows would land on the same chiplets and units, and short contexts leave the last parts empty.  So a row's
  // count starts one further for every eight workgroups in front of it, and once more for every round of the units; an odd count
  // goes round by itself.  (16 rows of 16 kv heads of size 64, contexts spread up to 8,000, four parts, three draws: counted alike
  // in all rows 66, 66 and 51 us, from a hash of the row 66, 67 and 41, so 62, 63 and 41; 32 such rows, three parts, four draws:
  // hashed 112 to 116, so 101 to 112.)  `deal` holds the two shifts and stands beside `splits`, with which it is fetched: worked out
  // here they took a branch and a further fetch at the head of the kernel, 0.2 to 0.4 % of a decode step at batch 8.
  const uint32_t row = blockIdx.y + n_kv * head_blocks * blockIdx.z;
  const uint32_t turn = (row >> (deal & 255)) + ((row * (uint32_t)splits) >> (deal >> 8));
  const int split = (int)((blockIdx.x + turn) % (uint32_t)splits);
  const int kvh = blockIdx.y / head_blocks, hb = blockIdx.y % head_blocks;
  const int item = blockIdx.z;
  const int t = rows ? scalar_int(rows + item) : item;      // the same for every lane
  if (t < 0) return;                                       // a row that only fills the list up: nothing to do
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int col = lane & 15, g = lane >> 4;
  const int heads_here = min(16, group - hb * 16);
  const int head = kvh * group + hb * 16 + col;          // valid when col < heads_here
  // entry_of_token null: every request has one token in the batch, request e is row e (one dependent load fewer).
  const int* table = block_table + (size_t)(entry_of_token ? scalar_int(entry_of_token + t) : t) * table_stride;
  // Without a window the split's first key does not hang on the position, so the pages of the wave's first block
  // are looked up beside the position rather than after it (one trip fewer before the first keys are asked for).
  // An entry past the request's pages may hold anything; it is only used for keys that exist (see load_block).
  const int early_kb = split * split_keys + wave * 32;
  int early_page0 = 0, early_page1 = 0;
  const bool from_zero = window < 0 && !(EXTRA && chunk > 0);      // the first key is key 0 whatever the position
  if (from_zero) {
    early_page0 = scalar_int(table + min(early_kb / page_size, table_stride - 1));
    early_page1 = scalar_int(table + min((early_kb + 16) / page_size, table_stride - 1));
  }
  const int pos = scalar_int(positions + t);
  int lo = (window >= 0 && pos > window) ? pos - window : 0;
  if (EXTRA && chunk > 0) lo = max(lo, pos / chunk * chunk);
  const float slope = (EXTRA && slopes && col < heads_here) ? slopes[head] : 0.f;
  int first = (lo / 32) * 32 + split * split_keys;        // first key of this split (a multiple of 32)
  int last = min(pos, first + split_keys - 1);
  int vh = kvh, n_vh = n_kv;                               // the value head this key head reads, of so many
  if (EXTRA) {
    if (n_v > 0 && n_v < n_kv) { vh = kvh / (n_kv / n_v); n_vh = n_v; }
    if (kept_splits > 0 && split >= splits - kept_splits) {       // a split over the kept first keys
      first = (split - (splits - kept_splits)) * split_keys;
      last = min(min(keep_first, lo) - 1, first + split_keys - 1);
      lo = 0;
    }
  }

  // Q^T fragments: lane holds head `col`, head-size elements ks*32 + 8g .. +7.
  bf16x8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int d0 = ks * 32 + 8 * g;
    qf[ks] = zero8();
    if (col < heads_here && d0 < D)
      qf[ks] = *reinterpret_cast<const bf16x8*>(q + (size_t)t * q_stride + (size_t)head * D + d0);
  }
  floatx4 acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) acc[db] = (floatx4){0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  // A block of 32 keys as the matrix instructions want it.  Key kb + k is index k of the second product's
  // contraction (lane group g holds k = 8g .. 8g+7), so a lane's eight values of a row of V^T are sixteen
  // contiguous bytes of one page: one load.  For that the first product's two instructions take the keys in an
  // order of their own: row r of instruction t is key kb + 8 (r / 4) + 4 t + r % 4, whose score then lands in
  // the lane group that holds that key in the second product.  Keys kb .. kb+15 lie in one page, kb+16 .. kb+31
  // in one (page sizes are multiples of 16).
  struct KeyBlock {
    bf16x8 kf[2][KS];
    union VFrag { uint4 bits; bf16x8 v; } vf[TIED ? 1 : DB];
    bool active;
    int left;                                              // this lane's eight keys of the block that exist: 0 .. left
  };
  // All loads of a block are issued together: keys, and values (whose addresses do not wait for the scores).
  // Nothing that was loaded is touched here (values of slots nobody wrote are set to zero when the block is used):
  // a value that is used makes the wave wait for all it asked for before, one trip to memory for every such use.
  auto load_block = [&](KeyBlock& blk, int kb) {
    blk.active = (kb <= last) && (kb + 31 >= lo);
    blk.left = 7;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) blk.kf[t][ks] = zero8();
    if (!TIED) {
#pragma unroll
      for (int db = 0; db < DB; ++db) blk.vf[db].bits = make_uint4(0, 0, 0, 0);
    }
    if (blk.active) {
      // The two halves of sixteen keys: a half that holds no key of the range (before `lo`: its page may have been
      // given back; after `last`: it may not exist yet) borrows the other half's page, which is a valid address;
      // what is read there never counts (scores outside lo..last are masked, such values are set to zero).  So
      // the branch is the same for the whole wave, and the addresses are a page number a lane away from scalars.
      const bool there0 = kb + 15 >= lo, there1 = kb + 16 <= last;
      int page0, page1;
      if (from_zero && kb == early_kb) {                    // (without a window the first half always holds keys)
        page0 = early_page0;
        page1 = there1 ? early_page1 : early_page0;
      } else {
        page0 = scalar_int(table + (there0 ? kb : kb + 16) / page_size);
        page1 = scalar_int(table + (there1 ? kb + 16 : kb) / page_size);
      }
      const uint32_t page_elems = (uint32_t)page_size * D;                  // same element count for K and V^T pages
      {
        const int half = col >> 3;
        const uint32_t at = ((uint32_t)(half ? page1 : page0) * n_kv + kvh) * page_elems +
                            (uint32_t)(((kb + 16 * half) % page_size) + 8 * ((col >> 2) & 1) + (col & 3)) * D + 8 * g;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int ks = 0; ks < KS; ++ks)
            if (ks * 32 + 8 * g < D) blk.kf[t][ks] = *reinterpret_cast<const bf16x8*>(k_pages + at + t * 4 * D + ks * 32);
      }
      if (!TIED) {
        const int half = g >> 1;
        const uint32_t at = ((uint32_t)(half ? page1 : page0) * n_vh + vh) * page_elems + (uint32_t)col * page_size +
                            ((kb + 16 * half) % page_size) + 8 * (g & 1);
        blk.left = (half ? there1 : there0) ? last - (kb + 8 * g) : -1;
#pragma unroll
        for (int db = 0; db < DB; ++db)
          blk.vf[db].bits = *reinterpret_cast<const uint4*>(vt_pages + at + db * 16 * page_size);
      }
    }
  };
  // One step of the online softmax over a block that has been brought in.
  auto attend = [&](KeyBlock& blk, int kb) {
    if (TIED) {
      if (kb < lo || kb + 31 > last || !blk.active) {        // (the same for the whole wave)
        // Keys outside lo .. last hold anything (slots nobody wrote, a borrowed page): as values they must be zero.
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int key = kb + 8 * (col >> 2) + 4 * t + (col & 3);
          if (key < lo || key > last) {
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) blk.kf[t][ks] = zero8();
          }
        }
      }
      char* stage = shared_s + wave * KeyStage<D>::BYTES;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          if (ks * 32 + 8 * g < D)
            *reinterpret_cast<bf16x8*>(stage + (8 * (col >> 2) + 4 * t + (col & 3)) * KeyStage<D>::ROW + (ks * 4 + g) * 16) = blk.kf[t][ks];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    if (!TIED && blk.left < 7) {                                      // slots nobody wrote may hold anything: 0 * NaN would poison the sum
      const int left = blk.left;
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        uint4 v = blk.vf[db].bits;
        if (left < 0) v.x = 0; else if (left < 1) v.x &= 0xffffu;
        if (left < 2) v.y = 0; else if (left < 3) v.y &= 0xffffu;
        if (left < 4) v.z = 0; else if (left < 5) v.z &= 0xffffu;
        if (left < 6) v.w = 0; else v.w &= 0xffffu;
        blk.vf[db].bits = v;
      }
    }
    float s[2][4];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      floatx4 st = (floatx4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        st = __builtin_amdgcn_mfma_f32_16x16x32_bf16(blk.kf[t][ks], qf[ks], st, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = kb + 8 * g + 4 * t + r;
        float score = st[r] * scale;
        if (EXTRA) score = fmaf(-slope, (float)(pos - key), score);
        if (EXTRA && softcap > 0.f) score = softcap * (1.f - 2.f / (1.f + __expf(2.f * score / softcap)));
        s[t][r] = (blk.active && key >= lo && key <= last) ? score : -INFINITY;
      }
    }
    float mx = fmaxf(fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3])),
                     fmaxf(fmaxf(s[1][0], s[1][1]), fmaxf(s[1][2], s[1][3])));
    mx = wave_max_across<32>(wave_max_across<16>(mx));
    const float m_new = fmaxf(m, mx);
    if (__all(m_new == -INFINITY)) return;                 // nothing visible yet: the same for every head, a scalar branch
    const float corr = (m_new == -INFINITY) ? 1.f : __expf(m - m_new);
    bf16x8 pf;
    float psum = 0.f;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = __expf(s[t][r] - m_new);           // exp(-inf) = 0 for masked keys
        psum += p;
        pf[t * 4 + r] = (__bf16)p;
      }
    l = l * corr + psum;
    m = m_new;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[db][r] *= corr;
      if constexpr (TIED) {
        // Keys 8g .. 8g+7 of coordinate db * 16 + col: rows 8g .. 8g+3, then 8g+4 .. 8g+7, sixteen coordinates each.
        const char* at = shared_s + wave * KeyStage<D>::BYTES + (8 * g + (col >> 2)) * KeyStage<D>::ROW + db * 32 + (col & 3) * 8;
        acc[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(transposed_keys(at, at + 4 * KeyStage<D>::ROW), pf, acc[db], 0, 0, 0);
      } else {
        acc[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(blk.vf[db].v, pf, acc[db], 0, 0, 0);
      }
    }
    if (TIED) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // (the next block is stored behind these reads)
  };
  constexpr int STRIDE = DEC_WAVES * 32;
  int kb = first + wave * 32;
  if constexpr (AHEAD) {
    // Two blocks in turn: while one is worked on, the next one's keys and values are on their way (a wave that
    // asked for them only when it got there would wait a trip to memory in every block).  That pays while a wave
    // has a few blocks; over dozens of blocks the second set of registers costs more in waves a SIMD holds
    // (measured at batch 64, head size 64: 1.03x at a context of 2,048, level at 8,192, 0.89x at 30,000).
    if (kb <= last) {
      KeyBlock one, two;
      load_block(one, kb);
      while (true) {
        const bool more = kb + STRIDE <= last;
        if (more) load_block(two, kb + STRIDE);
        attend(one, kb);
        kb += STRIDE;
        if (!more) break;
        const bool further = kb + STRIDE <= last;
        if (further) load_block(one, kb + STRIDE);
        attend(two, kb);
        kb += STRIDE;
        if (!further) break;
      }
    }
  } else {
    for (; kb <= last; kb += STRIDE) {
      KeyBlock one;
      load_block(one, kb);
      attend(one, kb);
    }
  }
  // Sum of the lane groups' partial denominators (the maximum is already common to them).
  l = wave_add_across<32>(wave_add_across<16>(l));
  // (The lane's head's sink, on its way while the waves meet: asked for behind them it is a trip of its own, and at the start, before the keys, it cost
  // kernels without sinks 0.1 us.)
  float sink_of = 0.f;
  if (sinks) sink_of = sinks[kvh * group + hb * 16 + min(col, heads_here - 1)];
  if (TIED) __syncthreads();                                // (no wave reads its keys any more)
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 4; ++r) acc_s[wave][db * 16 + 4 * g + r][col] = acc[db][r];
  if (g == 0) { m_s[wave][col] = m; l_s[wave][col] = l; }
  __syncthreads();
  // The waves' sums brought together, a wave a head: lane w of every DEC_WAVES has wave w's maximum and sum, so that each weight is
  // one exponential of one lane, read into a scalar for all; a lane has elements lane, lane + 64, .. of the head.  Attention and
  // merge, us, before (each lane of each head worked every wave's weight out, those of waves without keys too, and exchanges went
  // through LDS) and so: one row of 14 / 2 heads of 64, 16 keys 3.8 -> 3.3, 400 5.7 -> 5.4, 2,000 6.3 -> 6.2; eight rows, 2,000 keys 7.8 -> 7.55; eight
  // rows of 28 / 4 of 128, 1,300 keys 11.8 -> 11.2.
  for (int h = wave; h < heads_here; h += DEC_WAVES) {
    const int hg = kvh * group + hb * 16 + h;
    constexpr int PER = (D + WAVE - 1) / WAVE;
    const float mine = m_s[lane % DEC_WAVES][h], sum = l_s[lane % DEC_WAVES][h];
    float big = wave_max_repeated<DEC_WAVES>(mine);
    float denom = 0.f;
    if (sinks && split == 0) {
      const float sink = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(sink_of), h));
      big = fmaxf(big, sink);
      denom = __expf(sink - big);
    }
    const float weight = (mine == -INFINITY) ? 0.f : __expf(mine - big);
    float o[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) o[j] = 0.f;
    constexpr int STEP = DEC_WAVES < 4 ? DEC_WAVES : 4;
#pragma unroll
    for (int w0 = 0; w0 < DEC_WAVES; w0 += STEP) {
      if (w0 * 32 > last - first) break;                      // (the waves from here on had no keys)
      float part[PER][STEP];
#pragma unroll
      for (int j = 0; j < PER; ++j)
#pragma unroll
        for (int w = 0; w < STEP; ++w) part[j][w] = acc_s[w0 + w][min(lane + j * WAVE, D - 1)][h];
#pragma unroll
      for (int w = 0; w < STEP; ++w) {
        const float wgt = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(weight), w0 + w));
        denom += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(sum), w0 + w)) * wgt;
#pragma unroll
        for (int j = 0; j < PER; ++j) o[j] += part[j][w] * wgt;
      }
    }
    const size_t p = ((size_t)item * n_q + hg) * splits + split;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int d = lane + j * WAVE;
      if (D % WAVE != 0 && d >= D) continue;
      if (splits == 1) st_through(out + ((size_t)t * n_q + hg) * D + d, o[j] / denom);
      else st_through(part_o + p * D + d, o[j]);
    }
    if (splits != 1 && lane < 2) st_through(part_ml + p * 2 + lane, lane ? denom : big);
  }
}

// out[t, head, :] = sum_s part_o[s] * exp(m_s - M) / sum_s l_s * exp(m_s - M).  One wave per (item, head).
// LANES (16, 32 or 64: those of head sizes to 64, 128 and 256) lanes share a split's elements (a float4 each), the groups of so many
// take every 64 / LANES-th split, and all of a lane's loads are requested before the first is used: the kernel is one trip to memory.
// (With sixteen lanes for every head size longer heads were two to four trips.  Attention and merge, eight rows of 1,000
// keys: 12 heads of 128 9.1 -> 8.5 us, eight of 256 13.8 -> 11.8.)
// A separate kernel on purpose: a last-arrival merge inside the first kernel needs device-wide fences,
// which flush the L2 of every XCD and cost more than this launch.
// FIRST_TILES: the launch's workgroups are those of a prompt kernel's tiles in front (`tiled`) and of single tokens behind: one launch for
// both kinds of a step that has both.
struct MergeTiles { const float* part_o; const float* part_ml; int splits, blocks; };
template <int LANES, bool FIRST_TILES = false>
__global__ void __launch_bounds__(WAVE)
decode_attention_merge(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                       const int* __restrict__ rows, bf16_t* __restrict__ out, int n_q, int d, int splits,
                       const int* __restrict__ tiles, const int* __restrict__ cu_q, const MergeTiles tiled = MergeTiles()) {
  HELD(part_o, part_ml, rows, out, n_q, d, splits, tiles);   // (the words that are there when a wave starts)
  int block = blockIdx.x;
  if constexpr (FIRST_TILES) {
    if (block < tiled.blocks) {
      part_o = tiled.part_o; part_ml = tiled.part_ml; splits = tiled.splits; rows = nullptr;
    } else {
      block -= tiled.blocks;
      tiles = nullptr;
    }
  }
  const int item = block / n_q, head = block % n_q;
  int t = rows ? scalar_int(rows + item) : item;
  if (t < 0) return;
  if (tiles) {
    // Items are (tile, token of the tile): the output row is the tile's first row + the token; a tile's padding
    // has no row.
    const int tile = item >> 4, token = item & 15;
    const int entry = scalar_int(tiles + 2 * tile), row0 = scalar_int(cu_q + entry) + scalar_int(tiles + 2 * tile + 1);
    if (token >= scalar_int(cu_q + entry + 1) - row0) return;
    t = row0 + token;
  }
  const size_t base = ((size_t)item * n_q + head) * splits;
  constexpr int GROUPS = WAVE / LANES;
  const int lane = threadIdx.x, part = lane % LANES, grp = lane / LANES;
  const float2* ml = reinterpret_cast<const float2*>(part_ml) + base;
  constexpr int HELD = LANES == 16 ? 8 : 16;                 // splits a lane holds at once: 32 or 16 a round
  for (int e0 = 0; e0 < d; e0 += 4 * LANES) {
    const int e = e0 + 4 * part;
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    float big = -INFINITY, denom = 0.f;
    for (int s0 = 0; s0 < splits; s0 += GROUPS * HELD) {
      float4 v[HELD];
      float2 stat[HELD];
#pragma unroll
      for (int j = 0; j < HELD; ++j) {
        const int s = s0 + GROUPS * j + grp;
        v[j] = make_float4(0.f, 0.f, 0.f, 0.f);
        stat[j] = make_float2(-INFINITY, 0.f);
        if (s < splits) {
          stat[j] = ml[s];
          if (e < d) v[j] = *reinterpret_cast<const float4*>(part_o + (base + s) * d + e);
        }
      }
      float round_big = big;
#pragma unroll
      for (int j = 0; j < HELD; ++j) round_big = fmaxf(round_big, stat[j].x);
      const float keep = (big == -INFINITY) ? 0.f : __expf(big - round_big);   // this lane's sums so far, rescaled
      o.x *= keep; o.y *= keep; o.z *= keep; o.w *= keep;
      denom *= keep;
      big = round_big;
#pragma unroll
      for (int j = 0; j < HELD; ++j) {
        const float w = (stat[j].x == -INFINITY) ? 0.f : __expf(stat[j].x - big);
        o.x += v[j].x * w; o.y += v[j].y * w; o.z += v[j].z * w; o.w += v[j].w * w;
        denom += stat[j].y * w;
      }
    }
    // The lane groups hold sums over different splits under different maxima: bring them together.
    float all_big = big;
    if constexpr (LANES <= 16) all_big = wave_max_across<16>(all_big);
    if constexpr (LANES <= 32) all_big = wave_max_across<32>(all_big);
    const float w = (big == -INFINITY) ? 0.f : __expf(big - all_big);
    // (Groups of sixteen lanes: a group's own product joins the neighbour's rounded one in one rounding, as `fmaf` says.  The second
    // register of a swap of rows is the neighbour's in rows 0 and 2, which are those that group 0's sums come from.)
    auto across = [w](float x) {
      float sum = x * w;
      if constexpr (LANES <= 16) {
        float neighbour = sum;
        wave_swap16(sum, neighbour);
        sum = fmaf(x, w, neighbour);
      }
      if constexpr (LANES <= 32) sum = wave_add_across<32>(sum);
      return sum;
    };
    o.x = across(o.x); o.y = across(o.y); o.z = across(o.z); o.w = across(o.w);
    denom = across(denom);
    if (grp == 0 && e < d) {
      const float inv = 1.0f / denom;
      bf16_t* dst = out + (size_t)t * n_q * d + (size_t)head * d + e;
      union { bf16x4 v; uint2 bits; } packed;
      packed.v[0] = (__bf16)(o.x * inv); packed.v[1] = (__bf16)(o.y * inv);
      packed.v[2] = (__bf16)(o.z * inv); packed.v[3] = (__bf16)(o.w * inv);
      st_through(reinterpret_cast<uint2*>(dst), packed.bits);
    }
  }
}

template <int D>
static int launch_decode(const void* q, int q_stride, void* out, const void* k_pages, const void* vt_pages,
                         const void* rows, const void* positions, const void* entry_of_token,
                         const void* block_table, int table_stride, void* part_o, void* part_ml, int n_items,
                         int n_q, int n_kv, int page_size, int window, float scale, int split_keys, int splits,
                         int chunk, const void* slopes, const void* sinks, int keep_first, int kept_splits, int n_v,
                         float softcap, int tied, hipStream_t stream) {
  const int group = n_q / n_kv;
  dim3 grid(splits, n_kv * ((group + 15) / 16), n_items);
  // The shifts by which a row's first part moves on with the rows in front of it (31: it does not): with an even count, by the log2
  // of eight over what it shares with eight, and by that of the compute units.
  const int even = __builtin_ctz((unsigned)splits | 8u);
  const int deal = even ? (3 - even) | (31 - __builtin_clz((unsigned)compute_units())) << 8 : 31 | 31 << 8;
  constexpr int NW = D > 128 ? 2 : 4, WIDE = D <= 64 ? 16 : D <= 128 ? 8 : 4;
#define GO(WAVES, AHEAD, EE, TT) decode_attention_kernel<D, WAVES, AHEAD, EE, TT><<<grid, WAVES * WAVE, 0, stream>>>( \
      (const bf16_t*)q, q_stride, (bf16_t*)out, (const bf16_t*)k_pages, (const bf16_t*)vt_pages, (const int*)rows, \
      (const int*)positions, (const int*)entry_of_token, (const int*)block_table, table_stride, (float*)part_o, \
      (float*)part_ml, n_q, n_kv, page_size, window, scale, split_keys, splits, deal, chunk, (const float*)slopes, \
      (const float*)sinks, keep_first, kept_splits, n_v, softcap)
  const bool few = split_keys <= 32 * NW * 8;              // up to eight blocks a wave
  // Workgroups of sixteen (eight, four) waves where they are few and each has many keys: the keys are on their way at once, and
  // fewer parts do.  64 tokens, 2 kv heads, 1,000 keys, two parts and their merge: head size 64 12.3 us in nine parts of four
  // waves, 10.5 so; 128 21.0 and 17.9; of 500 keys, in one part without a merge, 9.2 -> 7.1 and 14.6 -> 10.4; one token, 256, eight
  // heads on one, 16.2 (two waves) and 13.5.  Many workgroups are better off with four waves (1,024 of 500 keys, size 64: 22.7 us,
  // 28.5 with sixteen); 512 is a measured line, two for each of 256 compute units.
  const bool wide = split_keys >= (D > 128 ? 128 : 288) && split_keys <= 2048 &&
                    (long)splits * n_kv * ((group + 15) / 16) * n_items < 512;
  const bool extra = chunk > 0 || slopes || kept_splits > 0 || softcap > 0.f || (n_v > 0 && n_v < n_kv);
  if (extra && !vt_pages) return -1;
  if (extra) { if (wide) GO(WIDE, true, true, false); else if (few) GO(NW, true, true, false); else GO(NW, false, true, false); }
  else if (tied || !vt_pages) { if (few) GO(NW, true, false, true); else GO(NW, false, false, true); }
  else if (wide) GO(WIDE, true, false, false);
  else if (few) GO(NW, true, false, false); else GO(NW, false, false, false);
#undef GO
  int status = LAUNCH_STATUS();
  if (status == 0 && splits > 1 && out) {
    decode_attention_merge<D <= 64 ? 16 : D <= 128 ? 32 : 64><<<n_items * n_q, 64, 0, stream>>>(
                                                             (const float*)part_o, (const float*)part_ml, (const int*)rows, (bf16_t*)out, n_q, D, splits,
                                                             nullptr, nullptr);
    status = LAUNCH_STATUS();
  }
  return status;
}

// The same merge for the prompt kernel whose tiles' keys were cut over workgroups: items are (tile, token of the
// tile), part_o float [n_tiles * 16, n_q, splits, d], part_ml float [n_tiles * 16, n_q, splits, 2].
extern "C" int ta_attention_merge_tiles(const void* part_o, const void* part_ml, const void* tiles, int n_tiles,
                                        const void* cu_q, void* out, int n_q, int d, int splits, hipStream_t stream) {
  if (n_tiles <= 0) return 0;
  if ((long)n_tiles * 16 * n_q > 0x7fffffffL || d % 4 || splits < 1) return -1;
#define GO(LANES) decode_attention_merge<LANES><<<n_tiles * 16 * n_q, 64, 0, stream>>>((const float*)part_o, (const float*)part_ml, nullptr, \
      (bf16_t*)out, n_q, d, splits, (const int*)tiles, (const int*)cu_q)
  if (d <= 64) GO(16); else if (d <= 128) GO(32); else GO(64);
#undef GO
  return LAUNCH_STATUS();
}

// Both merges of a step that has prompt tiles and single tokens, whose kernels have left their parts (out null): one launch.
extern "C" int ta_attention_merge_both(const void* tiles_o, const void* tiles_ml, const void* tiles, int n_tiles, const void* cu_q,
                                       int tiles_splits, const void* part_o, const void* part_ml, const void* rows, int n_items,
                                       int splits, void* out, int n_q, int d, hipStream_t stream) {
  const long in_tiles = (long)n_tiles * 16 * n_q, blocks = in_tiles + (long)n_items * n_q;
  if (n_tiles <= 0 || n_items <= 0 || blocks > 0x7fffffffL || d % 4 || tiles_splits < 1 || splits < 1) return -1;
  const MergeTiles tiled = {(const float*)tiles_o, (const float*)tiles_ml, tiles_splits, (int)in_tiles};
#define GO(LANES) decode_attention_merge<LANES, true><<<(unsigned)blocks, WAVE, 0, stream>>>((const float*)part_o, (const float*)part_ml, \
      (const int*)rows, (bf16_t*)out, n_q, d, splits, (const int*)tiles, (const int*)cu_q, tiled)
  if (d <= 64) GO(16); else if (d <= 128) GO(32); else GO(64);
#undef GO
  return LAUNCH_STATUS();
}

// tied: the value pages hold what the key pages hold, and only the keys are read; vt_pages may then be null.  out null with more than one
// part: the parts are left where they are.
// Returns -2 for a head size this kernel has no instance for (the caller then uses the generic kernel).
extern "C" int ta_decode_attention_bf16(const void* q, int q_stride, void* out, const void* k_pages,
                                        const void* vt_pages, const void* rows, const void* positions,
                                        const void* entry_of_token, const void* block_table, int table_stride,
                                        void* part_o, void* part_ml, int n_items, int n_q, int n_kv, int d,
                                        int page_size, int window, float scale, int split_keys, int splits,
                                        int chunk, const void* slopes, const void* sinks, int keep_first,
                                        int kept_splits, int n_v, float softcap, int tied, hipStream_t stream) {
  if (n_items <= 0) return 0;
  if (n_kv <= 0 || n_q % n_kv || page_size % 16 || split_keys % 32 || splits < 1 || (!out && splits < 2)) return -1;
  if (n_v <= 0) n_v = n_kv;
  if (n_kv % n_v || keep_first < 0 || kept_splits < 0 || kept_splits >= splits || (keep_first > 0) != (kept_splits > 0) ||
      (long)kept_splits * split_keys < keep_first || (keep_first > 0 && (window < 0 || chunk > 0)))
    return -1;
#define CASE(DD) case DD: return launch_decode<DD>(q, q_stride, out, k_pages, vt_pages, rows, positions, entry_of_token, \
    block_table, table_stride, part_o, part_ml, n_items, n_q, n_kv, page_size, window, scale, split_keys, splits, chunk, \
    slopes, sinks, keep_first, kept_splits, n_v, softcap, tied, stream);
  switch (d) {
    CASE(16) CASE(32) CASE(48) CASE(64) CASE(80) CASE(96) CASE(112) CASE(128) CASE(160) CASE(192) CASE(224) CASE(256)
    default: return -2;
  }
#undef CASE
}
