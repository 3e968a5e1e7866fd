// The inner loop of the products over many rows: a tile of BM rows by BN weight rows, K in steps of 64, both operands
// straight from memory into a ring of STAGES buffers in LDS (`global_load_lds_dwordx4`: no register and no LDS write
// instruction in between), from there into fragments of v_mfma_f32_16x16x32_bf16, float sums.
//
// A step: the fragments of its second half are read while its first half is multiplied; then a wait for the next step's loads
// and for the wave's own reads, one barrier, the loads of the step STAGES ahead into the buffer that the barrier has freed, and
// the first fragments of the next step are read while the second half is multiplied.  So no matrix instruction waits for a read
// that was asked for right before it, and a load has STAGES - 1 steps to arrive.
//
// The buffers are arrays of their own, each named where it is used (the steps are unrolled by STAGES): the compiler then knows
// that a read of one does not touch the loads on their way into another.  With one array for all it waits for every such load
// before every read, which is what made loads into LDS lose to registers in a product before.
// A row's 128 bytes are eight pieces; piece p of row r lies at place p ^ (r % 8), so that the lanes that a read serves at a time
// find their pieces in different banks; as a load writes LDS in the order of its lanes, the lanes ask for the pieces in that order.
//
// Square 256 tiles, two buffers, eight waves: 8,192 cubed at 1,360 TFLOP/s (the vendor's library 1,480 on the same card), 4,096 x 18,944
// over 3,584 470 us (library 530).  128 x 256, three buffers: 540; 128 x 128, four buffers: 630; four waves instead of eight:
// 5 to 20 % slower; v_mfma_f32_32x32x16: level to 10 % slower; raised wave priority around the matrix instructions: 5 to 8 % slower.
// Bound by the loads' way into LDS: 50 to 60 GB/s a compute unit at 128 x 128, where the matrix cores idle half the time.
#pragma once
#include "common.h"
#include <type_traits>

typedef __bf16 ring_bf16x8 __attribute__((ext_vector_type(8)));
typedef float ring_floatx4 __attribute__((ext_vector_type(4)));
typedef const char __attribute__((address_space(1)))* ring_memory;
typedef char __attribute__((address_space(3)))* ring_lds;

// Waits until at most VM of the wave's loads are on their way and none of its LDS reads.
template <int VM>
__device__ __forceinline__ void ring_wait() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((VM & 15) | (7 << 4) | ((VM >> 4) << 14));
  asm volatile("" ::: "memory");
}
__device__ __forceinline__ void ring_barrier() {
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// WM_WAVES x WN_WAVES waves share the tile.  `run` wants, per wave, the byte places of the pieces that its lanes bring: load i
// of A covers rows `a_row(i)` = (wave * LA + i) * 8 + lane / 8, load i of W likewise with LB; the piece within the row is
// `piece(row)`.  Places are unsigned 32-bit offsets from pointers that are the same for the whole workgroup.
// acc[i][j]: weight rows are the instruction's rows, so lane (r = lane % 16, g = lane / 16) holds columns 4 g .. 4 g + 3 of block j
// of row r of block i (row wm * WM + 16 i + r, column wn * WN + 16 j + 4 g).
template <int BM, int BN, int STAGES, int WM_WAVES, int WN_WAVES>
struct RingTile {
  static constexpr int WAVES = WM_WAVES * WN_WAVES, ACROSS = WN_WAVES, THREADS = WAVES * WAVE, ROW = 128;
  static constexpr int WM = BM / WM_WAVES, WN = BN / WN_WAVES, MI = WM / 16, NI = WN / 16;
  static constexpr int LA = BM / 8 / WAVES, LB = BN / 8 / WAVES, LOADS = LA + LB, STAGE = (BM + BN) * ROW;
  static_assert(BM % (8 * WAVES) == 0 && BN % (8 * WAVES) == 0 && STAGES >= 2 && STAGES <= 4 && STAGES * STAGE <= 160 * 1024);

  static __device__ __forceinline__ int load_row(int wave, int lane, int loads, int i) { return (wave * loads + i) * 8 + (lane >> 3); }
  static __device__ __forceinline__ uint32_t piece_bytes(int lane) { return ((lane & 7) ^ (lane >> 3)) * 16; }

  // A, W: where the tile's K starts; K of `steps` * 64 and, if `half`, 32 more.
  static __device__ __forceinline__ void run(const void* A, const uint32_t (&a_at)[LA], const void* W, const uint32_t (&w_at)[LB],
                                             int steps, bool half, ring_floatx4 (&acc)[MI][NI]) {
    __shared__ __attribute__((aligned(1024))) char ring0[STAGE];
    __shared__ __attribute__((aligned(1024))) char ring1[STAGE];
    __shared__ __attribute__((aligned(1024))) char ring2[STAGES > 2 ? STAGE : 16];
    __shared__ __attribute__((aligned(1024))) char ring3[STAGES > 3 ? STAGE : 16];
    auto slot = [&](auto which) -> ring_lds {
      constexpr int j = decltype(which)::value % STAGES;
      if constexpr (j == 0) return (ring_lds)ring0;
      else if constexpr (j == 1) return (ring_lds)ring1;
      else if constexpr (j == 2) return (ring_lds)ring2;
      else return (ring_lds)ring3;
    };
    run_in(slot, [&](auto which) -> ring_lds { return slot(which) + BM * ROW; }, A, a_at, W, w_at, steps, half, acc);
  }

  // The same in buffers of the caller's: `a_slot(j)`, `w_slot(j)` (j an integral constant, to be taken modulo STAGES) give the places of
  // BM and BN rows, in arrays of their own for every j.
  template <class ASlot, class WSlot>
  static __device__ __forceinline__ void run_in(ASlot a_slot, WSlot w_slot, const void* A, const uint32_t (&a_at)[LA], const void* W,
                                                const uint32_t (&w_at)[LB], int steps, bool half, ring_floatx4 (&acc)[MI][NI]) {
    const int lane = threadIdx.x & 63, wave = wave_index(), r = lane & 15, g = lane >> 4;
    const int wm = wave / WN_WAVES, wn = wave % WN_WAVES;
    // `keep`: the bits of a place that count.  A step past the last one asks for the first piece again and again: one line, so
    // that the loads under way stay countable and cost next to nothing.
    auto bring = [&](ring_lds to_a, ring_lds to_w, ring_memory a, ring_memory w, uint32_t keep, uint32_t back) {
      asm("" : "+s"(a), "+s"(w));
      uint32_t av[LA], wv[LB];
#pragma unroll
      for (int i = 0; i < LA; ++i) { av[i] = (a_at[i] - back) & keep; asm("" : "+v"(av[i])); }
#pragma unroll
      for (int i = 0; i < LB; ++i) { wv[i] = (w_at[i] - back) & keep; asm("" : "+v"(wv[i])); }
#pragma unroll
      for (int i = 0; i < LA; ++i)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(a + av[i]),
                                         (__attribute__((address_space(3))) void*)(to_a + (wave * LA + i) * 1024), 16, 0, 0);
#pragma unroll
      for (int i = 0; i < LB; ++i)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(w + wv[i]),
                                         (__attribute__((address_space(3))) void*)(to_w + (wave * LB + i) * 1024), 16, 0, 0);
    };
    auto fetch = [&](int step, auto which) {
      const bool past = step >= steps;
      const size_t along = past ? 0 : (size_t)step * ROW;
      bring(a_slot(which), w_slot(which), (ring_memory)(uintptr_t)A + along, (ring_memory)(uintptr_t)W + along, past ? 0u : ~0u, 0u);
    };
    uint32_t a_get[2], w_get[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      a_get[ks] = (wm * WM + r) * ROW + (((ks * 4 + g) ^ (r & 7)) * 16);
      w_get[ks] = (wn * WN + r) * ROW + (((ks * 4 + g) ^ (r & 7)) * 16);
    }
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) acc[i][j] = ring_floatx4{0.f, 0.f, 0.f, 0.f};
    ring_bf16x8 af[2][MI], wf[2][NI];
    auto read = [&](auto which, auto half_step) {
      constexpr int ks = decltype(half_step)::value;
      const ring_lds from_a = a_slot(which) + a_get[ks], from_w = w_slot(which) + w_get[ks];
#pragma unroll
      for (int j = 0; j < NI; ++j) wf[ks][j] = *(const ring_bf16x8 __attribute__((address_space(3)))*)(from_w + j * 16 * ROW);
#pragma unroll
      for (int i = 0; i < MI; ++i) af[ks][i] = *(const ring_bf16x8 __attribute__((address_space(3)))*)(from_a + i * 16 * ROW);
    };
    auto multiply = [&](auto half_step) {
      constexpr int ks = decltype(half_step)::value;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[ks][j], af[ks][i], acc[i][j], 0, 0, 0);
      // A read, then the matrix instructions that last about as long, and so on.
#pragma unroll
      for (int i = 0; i < MI + NI; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, MI * NI / (MI + NI), 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    const std::integral_constant<int, 0> first{};
    const std::integral_constant<int, 1> second{};
    auto one = [&](int step, auto which) {
      const std::integral_constant<int, decltype(which)::value + 1> next{};
      read(which, second);
      multiply(first);
      ring_wait<(STAGES - 2) * LOADS>();
      ring_barrier();
      fetch(step + STAGES, which);                          // (every wave has its fragments of this buffer)
      read(next, first);
      multiply(second);
    };
    fetch(0, std::integral_constant<int, 0>{});
    fetch(1, std::integral_constant<int, 1>{});
    if constexpr (STAGES > 2) fetch(2, std::integral_constant<int, 2>{});
    if constexpr (STAGES > 3) fetch(3, std::integral_constant<int, 3>{});
    ring_wait<(STAGES - 1) * LOADS>();
    ring_barrier();
    read(first, first);
    int step = 0;
    for (; step + STAGES <= steps; step += STAGES) {
      one(step, std::integral_constant<int, 0>{});
      one(step + 1, std::integral_constant<int, 1>{});
      if constexpr (STAGES > 2) one(step + 2, std::integral_constant<int, 2>{});
      if constexpr (STAGES > 3) one(step + 3, std::integral_constant<int, 3>{});
    }
    if (step < steps) one(step, std::integral_constant<int, 0>{});
    if constexpr (STAGES > 2) { if (step + 1 < steps) one(step + 1, std::integral_constant<int, 1>{}); }
    if constexpr (STAGES > 3) { if (step + 2 < steps) one(step + 2, std::integral_constant<int, 2>{}); }
    ring_wait<0>();                                         // (what was asked for past the end has arrived too)
    if (half) {
      // The last 32 of K: pieces 4 .. 7 of a row are not there and ask for pieces 0 .. 3 again; only the first half is used.
      ring_barrier();
      const size_t along = (size_t)steps * ROW;
      const uint32_t back = (((lane & 7) ^ (lane >> 3)) & 4) * 16;
      bring(a_slot(first), w_slot(first), (ring_memory)(uintptr_t)A + along, (ring_memory)(uintptr_t)W + along, ~0u, back);
      ring_wait<0>();
      ring_barrier();
      read(first, first);
      multiply(first);
      ring_wait<0>();
    }
  }
};
