// What the products in tiles share (gemm_tiles.hip, moe_grouped.hip): operands of 64 k a stage straight from memory into a ring of
// stages in LDS, and the matrix instructions that read them from there.
//
// What bounds such products is the chain request -> arrival -> LDS -> matrix instruction of a workgroup that lives for a few
// dozen steps of k, far more than bytes or operations.  So a workgroup's waves share a tile of BM rows of X and BN rows of W,
// brought by requests that go straight into LDS (16 bytes a lane a request, no register on the way) through STAGES stages:
// STAGES - 1 are on their way while one is multiplied, a wave waits for its own requests of the oldest stage only (vmcnt counts the
// younger ones), and one barrier a step tells everybody that the stage is whole and the one before it is free.  The requests are
// inline assembly, and the barrier with its wait too: the compiler would make every LDS read wait for all requests that are on
// their way.  (A request has no output register; its two address operands are read when it is issued.)  A stage's rows are unpadded,
// their eight 16-byte pieces permuted by the row (piece p of row r lies at place p ^ (r % 8)), so that a fragment's rows meet no bank
// twice.
//
// The products are transposed (W's rows are the matrix instruction's first operand): a lane then holds four neighbouring columns of
// one row of the result, stored as one piece, and, where gate and up rows alternate sixteen at a time, gate and up of the same columns.
#pragma once
#include "common.h"

namespace kvcm {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 ring_bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float ring_f32x4;

union RingFrag {
  uint4 u;
  ring_bf16x8 v;
};

constexpr int kStepK = 64;      // k of a stage: 128 bytes a row

// results may begin at any element: the hardware takes 8- and 16-byte stores there
typedef float any_f32x4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float any_f32x2 __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t any_u32x2 __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t any_u32x4 __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t any_u32 __attribute__((aligned(2)));

__device__ __forceinline__ uint32_t two_bf16(float a, float b) { return uint32_t(float_to_bf16_bits(a)) | uint32_t(float_to_bf16_bits(b)) << 16; }

// All but this wave's N youngest requests have arrived, its LDS reads too, and everybody else's.
template <int N>
__device__ __forceinline__ void ring_arrived() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// 16 bytes a lane from base + offset (the lane's) into LDS: lane l's go to `to` + 16 l
__device__ __forceinline__ void ring_bring16(uint32_t offset, uint64_t base, uint32_t to) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(offset), "s"(base) : "memory", "m0");
}

// The same where offsets do not fit 32 bits: every lane has an address of its own.
__device__ __forceinline__ void ring_bring16(uint64_t offset, uint64_t base, uint32_t to) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(to), "v"(base + offset) : "memory", "m0");
}

// Rows this many elements apart or more need offsets of 64 bits: a tile has up to 256 of them.
constexpr int kFarRows = 1 << 22;

// Workgroups go to the eight XCDs in turn: each XCD takes a contiguous stretch of the numbers, so that neighbours, which read the
// same rows of W, meet in one L2.
__device__ __forceinline__ int neighbours_on_one_xcd() {
  const int per = gridDim.x / 8, more = gridDim.x % 8, xcd = blockIdx.x % 8;
  return xcd * per + (xcd < more ? xcd : more) + blockIdx.x / 8;
}

// The waves are WM x WN, each with BM / WM rows of X and BN / WN rows of W.
template <int BM, int BN, int WM, int WN, int STAGES>
struct TileRing {
  static constexpr int NW = WM * WN, TM = BM / WM / 16, TN = BN / WN / 16;
  static constexpr int kRequests = (BM + BN) / 8, R = (kRequests + NW - 1) / NW;      // a request of a wave: 64 k of eight rows
  static constexpr int kStage = (BM + BN) * kStepK * 2, kBytes = STAGES * kStage;
  static_assert(kBytes <= 160 * 1024, "LDS");
  static_assert(BM % (WM * 16) == 0 && BN % (WN * 16) == 0 && STAGES >= 2 && STAGES <= 8 && (STAGES - 2) * R <= 63, "tile");

  // The q-th request of this wave: rows 8 req .. + 7 of the tile (X's first).  A wave without one in the last turn repeats the
  // stage's last.
  static __device__ __forceinline__ int request_of(int q, int wave) { return q * NW + wave < kRequests ? q * NW + wave : kRequests - 1; }
  // Lane l of a request brings, of row l / 8, the piece (of eight elements) that belongs at place l % 8.
  static __device__ __forceinline__ int piece_of(int lane) { return (lane % 8) ^ (lane / 8); }

  // acc += X W^T over `steps` steps of k.  offset[q] (uint32_t, or uint64_t for far rows): bytes from base(request) to the lane's piece
  // at the first k; base: the same for the whole wave; the steps are walked from step `phase` on and wrap around.  left < 64 (with phase 0): the last step has that many
  // k (a multiple of 8), the lanes whose pieces lie beyond bring the row's first piece of the step, which is not multiplied.
  // between: done once while the first stages are on their way.  works: this wave has rows (else it only brings operands).
  template <class Offset, class Base, class Between>
  static __device__ __forceinline__ void multiply(unsigned char* ring, const Offset (&offset)[R], Base base, int steps, int phase, int left,
                                                  int wave, int lane, ring_f32x4 (&acc)[TN][TM], Between between, bool works = true) {
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(
        reinterpret_cast<uintptr_t>(reinterpret_cast<__attribute__((address_space(3))) void*>(reinterpret_cast<uintptr_t>(ring)))));
    const int piece = piece_of(lane);
    auto request = [&](int t, int stage) {
      const int k = t + phase < steps ? t + phase : t + phase - steps;
      const uint64_t along = static_cast<uint64_t>(k) * 128;
      const uint32_t back = t == steps - 1 && piece * 8 >= left ? static_cast<uint32_t>(piece) * 16u : 0u;
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int req = request_of(q, wave);
        ring_bring16(offset[q] - back, base(req) + along, lds0 + stage * kStage + req * 1024);
      }
    };
    const int wm = wave % WM, wn = wave / WM, frow = lane % 16, fk = lane / 16;
    auto step = [&](int stage, int k_left) {
      if (!works) return;
      const unsigned char* xs = ring + stage * kStage + (wm * TM * 16 + frow) * 128;
      const unsigned char* ws = ring + stage * kStage + (BM + wn * TN * 16 + frow) * 128;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const int at = ((ks * 4 + fk) ^ (frow % 8)) * 16;      // (rows 16 apart have the same permutation)
        RingFrag x[TM], w[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) x[i].u = *reinterpret_cast<const uint4*>(xs + i * 2048 + at);
#pragma unroll
        for (int j = 0; j < TN; ++j) w[j].u = *reinterpret_cast<const uint4*>(ws + j * 2048 + at);
        if (k_left < kStepK) {
          const bool in = ks * 32 + fk * 8 < k_left;
#pragma unroll
          for (int i = 0; i < TM; ++i) x[i].u = in ? x[i].u : uint4{0u, 0u, 0u, 0u};
#pragma unroll
          for (int j = 0; j < TN; ++j) w[j].u = in ? w[j].u : uint4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int i = 0; i < TM; ++i) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j].v, x[i].v, acc[j][i], 0, 0, 0);
      }
    };
#pragma unroll
    for (int t = 0; t < STAGES - 1; ++t)
      if (t < steps) request(t, t);
    between();
    int stage = 0, fill = STAGES - 1, t = 0;
    for (; t < steps - (STAGES - 1); ++t) {
      ring_arrived<(STAGES - 2) * R>();
      request(t + STAGES - 1, fill);      // into the stage that everybody has read by now
      step(stage, kStepK);
      fill = fill + 1 == STAGES ? 0 : fill + 1;
      stage = stage + 1 == STAGES ? 0 : stage + 1;
    }
    // the last STAGES - 1 steps (or all, where there are fewer): LEFT younger stages are on their way
#define KVCM_RING_LAST(LEFT)                              \
  if constexpr ((LEFT) <= STAGES - 2) {                   \
    if ((LEFT) < steps) {                                 \
      ring_arrived<(LEFT) * R>();                         \
      step(stage, (LEFT) == 0 ? left : kStepK);           \
      stage = stage + 1 == STAGES ? 0 : stage + 1;        \
    }                                                     \
  }
    KVCM_RING_LAST(6) KVCM_RING_LAST(5) KVCM_RING_LAST(4) KVCM_RING_LAST(3) KVCM_RING_LAST(2) KVCM_RING_LAST(1) KVCM_RING_LAST(0)
#undef KVCM_RING_LAST
  }
};

}  // namespace kvcm
