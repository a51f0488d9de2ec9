// The matrix half of products in large tiles (gemm_tiles.hip, moe_grouped.hip): operands in a ring of stages in LDS as in
// tile_ring.h, four waves with a quarter of the tile each, and fragments that are read while the ones before them are multiplied.
//
// What bounds a tile of 128 x 128 and more is LDS, not the matrix cores: a fragment goes to every wave that has its rows, so that eight
// waves of 128 x 64 read a half more of a stage of 256 x 256 than four of 128 x 128 do, and a wave that reads in front of every
// product waits a trip to LDS per 32 k.  Four waves, one a SIMD, have 512 registers each: 256 sums, and two sets of
// fragments.  A step of 64 k is two halves of 32: while a half is multiplied, the next one's fragments are read, one read between two
// or three matrix instructions (the order is the source's: the compiler would gather them), and in the second half the requests of
// the stage that has just become free go out the same way.  One barrier a step, between the halves: by then everybody has the
// stage's last fragments, and the next stage is whole.
//
// us, the eight to twelve waves of tile_ring.h / this (launches one after the other, weights from memory): 2048 x 2048 x 5632 54.4 / 51.8
// (128 x 128), 2048 x 2560 x 2048 30.6 / 22.8, gate and up of 5632 x 2048, 2,048 rows 95.1 / 88.9, 32,768 rows 1,382 / 1,118, 8192^3 1,133 / 752.
// With weights that are in the memory-side cache 2048 x 2048 x 5632 takes 44 us; more stages do not help (three to five: the same).
// Tried and taken back: W's fragments read one block of columns ahead instead of a half (registers for 256 x 352; 5 to 10 % slower at the
// same tile), matrix instructions of 32 x 32 (1,474 TFLOP/s of registers alone, these 1,703: random operands are bound by power, zeros reach 2,205).
#pragma once
#include <type_traits>

#include "tile_ring.h"

namespace kvcm {

// The waves are WM x WN, each with BM / WM rows of X and BN / WN rows of W.
template <int BM, int BN, int WM, int WN, int STAGES>
struct TilePipe {
  static constexpr int NW = WM * WN, TM = BM / WM / 16, TN = BN / WN / 16;
  static constexpr int kRequests = (BM + BN) / 8, R = (kRequests + NW - 1) / NW;      // a request of a wave: 64 k of eight rows
  static constexpr int kStage = (BM + BN) * kStepK * 2, kBytes = STAGES * kStage;
  static constexpr int NF = TM + TN, NM = TM * TN;      // fragments and matrix instructions of a half
  static_assert(kBytes <= 160 * 1024, "LDS");
  static_assert(BM % (WM * 16) == 0 && BN % (WN * 16) == 0 && STAGES >= 2 && (STAGES - 1) * R <= 63, "tile");

  // (as in TileRing)
  static __device__ __forceinline__ int request_of(int q, int wave) { return q * NW + wave < kRequests ? q * NW + wave : kRequests - 1; }
  static __device__ __forceinline__ int piece_of(int lane) { return (lane % 8) ^ (lane / 8); }

  // acc += X W^T over `steps` steps of k; offset, base, phase, left and works as in TileRing::multiply.
  template <class Offset, class Base, class Between>
  static __device__ __forceinline__ void multiply(unsigned char* ring, const Offset (&offset)[R], Base base, int steps, int phase, int left,
                                                  int wave, int lane, ring_f32x4 (&acc)[TN][TM], Between between, bool works = true) {
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(
        reinterpret_cast<uintptr_t>(reinterpret_cast<__attribute__((address_space(3))) void*>(reinterpret_cast<uintptr_t>(ring)))));
    const int piece = piece_of(lane);
    auto request = [&](int q, int t, int stage) {
      const int req = request_of(q, wave), k = t + phase < steps ? t + phase : t + phase - steps;
      const uint32_t back = t == steps - 1 && piece * 8 >= left ? static_cast<uint32_t>(piece) * 16u : 0u;
      ring_bring16(offset[q] - back, base(req) + static_cast<uint64_t>(k) * 128, lds0 + stage * kStage + req * 1024);
    };
    const int wm = wave % WM, wn = wave / WM, frow = lane % 16, fk = lane / 16;
    const unsigned char* xs = ring + (wm * TM * 16 + frow) * 128;
    const unsigned char* ws = ring + (BM + wn * TN * 16 + frow) * 128;
    const int at0 = (fk ^ (frow % 8)) * 16, at1 = ((4 + fk) ^ (frow % 8)) * 16;      // of the two halves
    RingFrag xa[TM], wa[TN], xb[TM], wb[TN];
    auto read = [&](RingFrag(&x)[TM], RingFrag(&w)[TN], int f, int stage, int at) {
      if (f < TN) w[f].u = *reinterpret_cast<const uint4*>(ws + stage * kStage + f * 2048 + at);
      else x[f - TN].u = *reinterpret_cast<const uint4*>(xs + stage * kStage + (f - TN) * 2048 + at);
    };
    // multiplies (x, w); READS: the fragments of (rstage, rat) meanwhile; REQUESTS: those of step rt into qstage
    auto half = [&](RingFrag(&x)[TM], RingFrag(&w)[TN], RingFrag(&nx)[TM], RingFrag(&nw)[TN], auto reads, int rstage, int rat, auto requests,
                    int rt, int qstage) {
      int f = 0, q = 0;
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        const int j = m / TM, i = m % TM;
        acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j].v, x[i].v, acc[j][i], 0, 0, 0);
        // the reads over the first three quarters, the requests over the whole half
        if constexpr (decltype(reads)::value)
          if (f < NF && (m + 1) * NF * 4 >= (f + 1) * NM * 3) read(nx, nw, f++, rstage, rat);
        if constexpr (decltype(requests)::value)
          if (q < R && (m + 1) * R >= (q + 1) * NM) request(q++, rt, qstage);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (decltype(reads)::value) {
#pragma unroll
        for (; f < NF; ++f) read(nx, nw, f, rstage, rat);
      }
      if constexpr (decltype(requests)::value) {
#pragma unroll
        for (; q < R; ++q) request(q, rt, qstage);
      }
    };
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    auto after = [](int stage) { return stage + 1 == STAGES ? 0 : stage + 1; };
#pragma unroll
    for (int t = 0; t < STAGES; ++t) {
      if (t < steps) {
#pragma unroll
        for (int q = 0; q < R; ++q) request(q, t, t);
      }
    }
    between();
    if (steps >= STAGES) ring_arrived<(STAGES - 1) * R>();
    else ring_arrived<0>();
    int stage = 0, t = 0;
    if (!works) {      // (the same barriers and requests)
      for (; t < steps - STAGES; ++t) {
        ring_arrived<(STAGES - 2) * R>();
#pragma unroll
        for (int q = 0; q < R; ++q) request(q, t + STAGES, stage);
        stage = after(stage);
      }
      for (; t < steps - 1; ++t) ring_arrived<0>();
      return;
    }
#pragma unroll
    for (int f = 0; f < NF; ++f) read(xa, wa, f, 0, at0);
    for (; t < steps - STAGES; ++t) {
      const int next = after(stage);
      half(xa, wa, xb, wb, yes, stage, at1, no, 0, 0);
      ring_arrived<(STAGES - 2) * R>();
      half(xb, wb, xa, wa, yes, next, at0, yes, t + STAGES, stage);
      stage = next;
    }
    for (; t < steps - 1; ++t) {
      const int next = after(stage);
      half(xa, wa, xb, wb, yes, stage, at1, no, 0, 0);
      ring_arrived<0>();
      half(xb, wb, xa, wa, yes, next, at0, no, 0, 0);
      stage = next;
    }
    // the last step may have fewer than 64 k
    auto cut = [&](RingFrag(&x)[TM], RingFrag(&w)[TN], bool in) {
#pragma unroll
      for (int i = 0; i < TM; ++i) x[i].u = in ? x[i].u : uint4{0u, 0u, 0u, 0u};
#pragma unroll
      for (int j = 0; j < TN; ++j) w[j].u = in ? w[j].u : uint4{0u, 0u, 0u, 0u};
    };
    if (left < kStepK) cut(xa, wa, fk * 8 < left);
    half(xa, wa, xb, wb, yes, stage, at1, no, 0, 0);
    if (left < kStepK) cut(xb, wb, 32 + fk * 8 < left);
    half(xb, wb, xa, wa, no, 0, 0, no, 0, 0);
  }
};

// Neighbouring numbers are tiles of one XCD (neighbours_on_one_xcd): the 32 workgroups that run side by side there take a few row blocks of
// a few columns, so that both operands' rows are shared in its L2.  us, row blocks of all rows first / eight / four: 32,768 x 2048 x 5632 643 /
// 556 / 553 (256 x 256), 32,768 rows gate and up of 5632 x 2048 1,382 / 1,190 / 1,118; 2048 x 2048 x 5632 (128 x 128) 55.3 / 51.7 / 53.1.
template <int BM>
__device__ __forceinline__ void tile_of(int id, int tiles_m, int tiles_n, int& tm, int& tn) {
  constexpr int kRowBlocks = BM >= 192 ? 4 : 8;
  const int group = id / (kRowBlocks * tiles_n), first = group * kRowBlocks, rows = tiles_m - first < kRowBlocks ? tiles_m - first : kRowBlocks;
  id -= group * kRowBlocks * tiles_n;
  tm = first + id % rows;
  tn = id / rows;
}

// Which row of W (or of a pair of gate and up rows) of a wave lies at row a of its block (of 16) b of `blocks`: blocks are paired
// so that a lane, which holds rows 4 q .. 4 q + 3 of each, has eight neighbours of a pair, 16 bytes of a bfloat16 result, and the four lanes of
// a row 64 (as blocks lie: 32 bytes a row and store).
__device__ __forceinline__ constexpr int paired_row(int b, int a, int blocks) {
  return b / 2 * 2 + 1 < blocks ? b / 2 * 32 + a / 4 * 8 + b % 2 * 4 + a % 4 : b * 16 + a;
}

}  // namespace kvcm
