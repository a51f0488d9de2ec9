// Products of a few to a few thousand rows, bfloat16: Y[M,N] = X[M,K] * W[N,K]^T, 32-bit sums, the result stored (bfloat16 or
// 32-bit), left as partial sums of S slices of K ([S][M][N], the consumer adds them in slice order), or, SWIGLU, made into
// act[M,I] = silu(X W_gate^T) * (X W_up^T), or with relu in silu's place, of a fused [gate (I rows) | up (I rows)] matrix.
//
// A workgroup of 2 to 6 waves owns a tile of BM rows x BN columns and a slice of K, its operands in a ring of stages in LDS
// (tile_ring.h, which says what bounds such products and why the ring); from 96 rows on four waves that read ahead (tile_pipe.h).
//
// Measured (us, weights from memory, one launch after the other in a graph; the kernel that shared only X through LDS and streamed
// W into registers, its own trips double-buffered / this one):
//   64 rows   2560 x 2048 7.5 / 5.1   2048 x 2048 6.4 / 4.7   gate+up 11264 x 2048 19.6 / 13.2   2048 x 5632 10.9 / 8.0
//   16 rows   5.1 / 4.2   4.9 / 4.0   13.0 / 11.1   8.1 / 6.6;  128 rows of 4096 x 14336 39.3 / 27.1
// and against the vendor's product: kvcm_gemm_tiles_preferred, below.
#include <cmath>
#include <utility>

#include "common.h"
#include "gemm_tiles.h"
#include "kvcm_hip.h"
#include "tile_pipe.h"

namespace kvcm {

// act(gate) * up (TileAct), or, limit > 0, the gate with limits
template <class TO>
__device__ __forceinline__ float gated(float gate, float up, float limit, int act) {
  if (limit > 0.f) return act == kSiluStored ? clamped_gate<TO>(gate, up, limit) : clamped_gate<float>(gate, up, limit);
  if (act == kRelu) return fmaxf(gate, 0.f) * up;
  if (act == kSilu) return silu<float>(gate) * up;
  return round_to<TO>(silu<TO>(round_to<TO>(gate))) * round_to<TO>(up);
}

// The waves are WM x WN, each with BM / WM rows and BN / WN columns.  GATED: N is I; a tile's BN rows of W are gate and up rows of
// BN / 2 columns of act: sixteen of each in turn where a wave has an even number of 16-column tiles (its accumulators of
// neighbouring tiles then hold gate and up), else eight and eight (lanes 32 apart then do, and swap halves).
// ss_in (GATED): X = round(g round(x)) of a norm folded into this product (gemm_rows8.hip): the sums are scaled by the rows'
// rsqrt(mean x^2 + eps), from tiles_in sums of squares a row.
// Offset: of an operand's pieces from its tile's beginning, in bytes; uint64_t for rows that are far apart.
template <int BM, int BN, int WM, int WN, int STAGES, bool GATED, class Offset>
__global__ void __launch_bounds__(WM* WN* kWave)
    gemm_tiles_kernel(const uint16_t* __restrict__ X, const uint16_t* __restrict__ W, float* __restrict__ partials, void* __restrict__ out,
                      int out_f32, int M, int N, int K, int ldx, int ldw, int ldo, int S, int tiles_m, int tiles_n,
                      const float* __restrict__ ss_in, int tiles_in, float eps, float limit, int act) {
  using Ring = TileRing<BM, BN, WM, WN, STAGES>;
  constexpr int NW = Ring::NW, TM = Ring::TM, TN = Ring::TN, R = Ring::R;
  constexpr int kHalf = TN % 2 == 0 ? 16 : 8;      // gate rows in front of their up rows
  static_assert(BM / NW <= kWave, "the rows' scales lie one a lane");
  __shared__ __attribute__((aligned(1024))) unsigned char ring[Ring::kBytes];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  int id = neighbours_on_one_xcd();      // row blocks first
  const int tm = id % tiles_m;
  id /= tiles_m;
  const int tn = id % tiles_n, s = id / tiles_n;
  const int m0 = tm * BM, c0 = tn * (GATED ? BN / 2 : BN);
  const int steps_all = K / kStepK;
  const int k_lo = static_cast<int>(static_cast<long long>(steps_all) * s / S);
  const int steps = static_cast<int>(static_cast<long long>(steps_all) * (s + 1) / S) - k_lo;

  const uint64_t xbase = reinterpret_cast<uint64_t>(X + static_cast<size_t>(m0) * ldx) + static_cast<size_t>(k_lo) * 128;
  const uint64_t wbase = reinterpret_cast<uint64_t>(W + static_cast<size_t>(c0) * ldw) + static_cast<size_t>(k_lo) * 128;
  const uint64_t upbase = wbase + static_cast<size_t>(GATED ? N : 0) * ldw * 2;
  // rows past M and columns past N repeat the last one (what they give is not stored)
  Offset offset[R];
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int req = Ring::request_of(q, wave), row = req * 8 + lane / 8;
    int at, ld;
    if (req < BM / 8) {
      at = row < M - m0 ? row : M - 1 - m0;
      ld = ldx;
    } else {
      const int c = row - BM;
      at = GATED ? c / (2 * kHalf) * kHalf + c % kHalf : c;
      if (at > N - 1 - c0) at = N - 1 - c0;
      ld = ldw;
    }
    offset[q] = static_cast<Offset>(at) * static_cast<Offset>(ld) * 2u + static_cast<Offset>(Ring::piece_of(lane)) * 16u;
  }
  // One row block: workgroups walk their slice from different places (and wrap around), or all would ask the same few memory
  // channels for rows a multiple of 4 KB apart at the same time.  Several: those that share
  // columns walk together.
  const int phase = tiles_m == 1 ? tn * 5 % steps : 0;
  auto base = [&](int req) {
    const bool up = GATED && (req - BM / 8) * 8 % (2 * kHalf) >= kHalf;
    return req < BM / 8 ? xbase : up ? upbase : wbase;
  };
  ring_f32x4 acc[TN][TM];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i) acc[j][i] = ring_f32x4{0.f, 0.f, 0.f, 0.f};
  const int wm = wave % WM, wn = wave / WM, frow = lane % 16, fk = lane / 16;
  float rstd = 1.f;      // lane l: of row wave + l NW
  Ring::multiply(ring, offset, base, steps, phase, kStepK, wave, lane, acc, [&] {
    if (GATED && ss_in != nullptr) {      // a wave a row, in a fixed order, while the first stages are on their way
      for (int l = 0; l * NW + wave < BM; ++l) {
        const int m = l * NW + wave;
        if (m0 + m < M) {
          const float* p = ss_in + static_cast<size_t>(m0 + m) * tiles_in;
          float part[4] = {0.f, 0.f, 0.f, 0.f};
          int t = lane;
          for (; t + 3 * kWave < tiles_in; t += 4 * kWave) {
#pragma unroll
            for (int q = 0; q < 4; ++q) part[q] += p[t + q * kWave];
          }
          for (; t < tiles_in; t += kWave) part[0] += p[t];
          const float sum = wave_sum((part[0] + part[1]) + (part[2] + part[3]));
          if (lane == l) rstd = rsqrtf(sum / static_cast<float>(tiles_in * 8) + eps);
        }
      }
    }
  });
  const float* scale = reinterpret_cast<const float*>(ring);
  if (GATED && ss_in != nullptr) {      // (the same for the whole workgroup)
    __syncthreads();
    if (lane * NW + wave < BM) reinterpret_cast<float*>(ring)[lane * NW + wave] = rstd;
    __syncthreads();
  }

  // acc[j][i][r]: row wm * TM * 16 + i * 16 + frow, row of W (in the tile) wn * TN * 16 + j * 16 + fk * 4 + r
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + (wm * TM + i) * 16 + frow;
    if constexpr (GATED) {
      if (ss_in != nullptr) {
        const float f = scale[m - m0];
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[j][i] *= f;
      }
      const size_t row = static_cast<size_t>(m) * ldo;
      if constexpr (kHalf == 16) {
#pragma unroll
        for (int j = 0; j < TN; j += 2) {
          const int c = c0 + (wn * TN + j) * 8 + fk * 4;
          if (m >= M || c >= N) continue;
          const ring_f32x4 g = acc[j][i], u = acc[j + 1][i];
          if (out_f32) {
            *reinterpret_cast<any_f32x4*>(static_cast<float*>(out) + row + c) = any_f32x4{
                gated<float>(g[0], u[0], limit, act), gated<float>(g[1], u[1], limit, act), gated<float>(g[2], u[2], limit, act), gated<float>(g[3], u[3], limit, act)};
          } else {
            *reinterpret_cast<any_u32x2*>(static_cast<uint16_t*>(out) + row + c) =
                any_u32x2{two_bf16(gated<bf16_t>(g[0], u[0], limit, act), gated<bf16_t>(g[1], u[1], limit, act)),
                          two_bf16(gated<bf16_t>(g[2], u[2], limit, act), gated<bf16_t>(g[3], u[3], limit, act))};
          }
        }
      } else {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          // lanes 0..31 hold gate rows, lanes 32..63 the up rows of the same columns: the lower lanes keep the first two of their
          // four columns, the upper ones take the other two
          float g[2], u[2];
#pragma unroll
          for (int r = 0; r < 2; ++r) {
            const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[j][i][r]), __float_as_uint(acc[j][i][r + 2]), false, false);
            g[r] = __uint_as_float(both[0]);
            u[r] = __uint_as_float(both[1]);
          }
          const int c = c0 + (wn * TN + j) * 8 + fk % 2 * 4 + fk / 2 * 2;
          if (m >= M || c >= N) continue;
          if (out_f32)
            *reinterpret_cast<any_f32x2*>(static_cast<float*>(out) + row + c) = any_f32x2{gated<float>(g[0], u[0], limit, act), gated<float>(g[1], u[1], limit, act)};
          else
            *reinterpret_cast<any_u32*>(static_cast<uint16_t*>(out) + row + c) =
                two_bf16(gated<bf16_t>(g[0], u[0], limit, act), gated<bf16_t>(g[1], u[1], limit, act));
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int c = c0 + (wn * TN + j) * 16 + fk * 4;
        if (m >= M || c >= N) continue;
        const ring_f32x4 v = acc[j][i];
        if (S > 1)
          *reinterpret_cast<any_f32x4*>(partials + (static_cast<size_t>(s) * M + m) * N + c) = any_f32x4{v[0], v[1], v[2], v[3]};
        else if (out_f32)
          *reinterpret_cast<any_f32x4*>(static_cast<float*>(out) + static_cast<size_t>(m) * ldo + c) = any_f32x4{v[0], v[1], v[2], v[3]};
        else
          *reinterpret_cast<any_u32x2*>(static_cast<uint16_t*>(out) + static_cast<size_t>(m) * ldo + c) = any_u32x2{two_bf16(v[0], v[1]), two_bf16(v[2], v[3])};
      }
    }
  }
}

template <int... I, class F>
__device__ __forceinline__ void each_of(std::integer_sequence<int, I...>, F f) {
  (f(std::integral_constant<int, I>{}), ...);
}

// The same product in large tiles (tile_pipe.h), 32-bit offsets.  GATED: gate and up rows lie sixteen (an odd number of 16-column tiles a wave: eight) of each
// in turn, as above.
template <int BM, int BN, int WM, int WN, int STAGES, bool GATED>
__global__ void __launch_bounds__(WM* WN* kWave)
    gemm_pipe_kernel(const uint16_t* __restrict__ X, const uint16_t* __restrict__ W, float* __restrict__ partials, void* __restrict__ out,
                     int out_f32, int M, int N, int K, int ldx, int ldw, int ldo, int S, int tiles_m, int tiles_n, float limit, int act) {
  using Pipe = TilePipe<BM, BN, WM, WN, STAGES>;
  constexpr int TM = Pipe::TM, TN = Pipe::TN, R = Pipe::R;
  constexpr bool kEights = GATED && TN % 2 != 0;
  constexpr int kBlocks = GATED ? TN / 2 : TN;      // of 16 columns of the result (kEights: not used)
  __shared__ __attribute__((aligned(1024))) unsigned char ring[Pipe::kBytes];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  int id = neighbours_on_one_xcd(), tm, tn;
  const int s = id / (tiles_m * tiles_n);
  id -= s * tiles_m * tiles_n;
  tile_of<BM>(id, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, c0 = tn * (GATED ? BN / 2 : BN);
  const int steps_all = K / kStepK;
  const int k_lo = static_cast<int>(static_cast<long long>(steps_all) * s / S);
  const int steps = static_cast<int>(static_cast<long long>(steps_all) * (s + 1) / S) - k_lo;
  const uint64_t xbase = reinterpret_cast<uint64_t>(X + static_cast<size_t>(m0) * ldx) + static_cast<size_t>(k_lo) * 128;
  const uint64_t wbase = reinterpret_cast<uint64_t>(W + static_cast<size_t>(c0) * ldw) + static_cast<size_t>(k_lo) * 128;
  const uint64_t upbase = wbase + static_cast<size_t>(GATED ? N : 0) * ldw * 2;
  constexpr int kHalf = kEights ? 8 : 16;
  // rows past M and columns past N repeat the last one (what they give is not stored)
  uint32_t offset[R];
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int req = Pipe::request_of(q, wave), row = req * 8 + lane / 8;
    int at, ld;
    if (req < BM / 8) {
      at = row < M - m0 ? row : M - 1 - m0;
      ld = ldx;
    } else {
      const int r = row - BM, part = r / (TN * 16), block = r / 16 % TN, a = r % 16;
      if constexpr (kEights) at = r / 16 * 8 + a % 8;
      else if constexpr (GATED) at = part * (TN * 8) + paired_row(block / 2, a, kBlocks);
      else at = part * (TN * 16) + paired_row(block, a, kBlocks);
      if (at > N - 1 - c0) at = N - 1 - c0;
      ld = ldw;
    }
    offset[q] = static_cast<uint32_t>(at) * static_cast<uint32_t>(ld) * 2u + static_cast<uint32_t>(Pipe::piece_of(lane)) * 16u;
  }
  // one row block: as above
  const int phase = tiles_m == 1 ? tn * 5 % steps : 0;
  auto base = [&](int req) {
    const bool up = GATED && (req - BM / 8) * 8 % (2 * kHalf) >= kHalf;
    return req < BM / 8 ? xbase : up ? upbase : wbase;
  };
  ring_f32x4 acc[TN][TM];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i) acc[j][i] = ring_f32x4{0.f, 0.f, 0.f, 0.f};
  Pipe::multiply(ring, offset, base, steps, phase, kStepK, wave, lane, acc, [] {});
  const int wm = wave % WM, wn = wave / WM, frow = lane % 16, fk = lane / 16;
  // A row of the result; acc's indexes have to be constants, and what the gated forms compute is too long for the compiler to unroll on
  // request: hence a function of a constant, and the activation chosen outside.
  auto store_row = [&](auto i_, auto gated_by) __attribute__((always_inline)) {
    constexpr int i = decltype(i_)::value;
    const int m = m0 + (wm * TM + i) * 16 + frow;
    if (m >= M) return;
    const size_t row = static_cast<size_t>(m) * ldo;
    if constexpr (kEights) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {      // (as above)
        float g[2], u[2];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[j][i][r]), __float_as_uint(acc[j][i][r + 2]), false, false);
          g[r] = __uint_as_float(both[0]);
          u[r] = __uint_as_float(both[1]);
        }
        const int c = c0 + (wn * TN + j) * 8 + fk % 2 * 4 + fk / 2 * 2;
        if (c >= N) continue;
        if (out_f32) *reinterpret_cast<any_f32x2*>(static_cast<float*>(out) + row + c) = any_f32x2{gated_by(0.f, g[0], u[0]), gated_by(0.f, g[1], u[1])};
        else *reinterpret_cast<any_u32*>(static_cast<uint16_t*>(out) + row + c) = two_bf16(gated_by(bf16_t{}, g[0], u[0]), gated_by(bf16_t{}, g[1], u[1]));
      }
    } else {
      auto four_of = [&](int b, auto type) {      // four columns of the result
        if constexpr (GATED) {
          const ring_f32x4 g = acc[2 * b % TN][i], u = acc[(2 * b + 1) % TN][i];
          return ring_f32x4{gated_by(type, g[0], u[0]), gated_by(type, g[1], u[1]), gated_by(type, g[2], u[2]), gated_by(type, g[3], u[3])};
        } else {
          return acc[b % TN][i];
        }
      };
      if ((!GATED && S > 1) || out_f32) {
#pragma unroll
        for (int b = 0; b < kBlocks; ++b) {
          const int c = c0 + wn * kBlocks * 16 + paired_row(b, fk * 4, kBlocks);
          if (c >= N) continue;
          const ring_f32x4 v = four_of(b, 0.f);
          float* to = !GATED && S > 1 ? partials + (static_cast<size_t>(s) * M + m) * N + c : static_cast<float*>(out) + row + c;
          *reinterpret_cast<any_f32x4*>(to) = any_f32x4{v[0], v[1], v[2], v[3]};
        }
      } else {
#pragma unroll
        for (int b = 0; b < kBlocks; ++b) {
          const bool paired = b / 2 * 2 + 1 < kBlocks;
          if (paired && b % 2 != 0) continue;      // (stored with the block before)
          const int c = c0 + wn * kBlocks * 16 + paired_row(b, fk * 4, kBlocks);
          if (c >= N) continue;
          uint16_t* to = static_cast<uint16_t*>(out) + row + c;
          const ring_f32x4 v = four_of(b, bf16_t{});
          const any_u32x2 four{two_bf16(v[0], v[1]), two_bf16(v[2], v[3])};
          if (paired && c + 4 < N) {
            const ring_f32x4 next = four_of(b + 1, bf16_t{});
            *reinterpret_cast<any_u32x4*>(to) = any_u32x4{four[0], four[1], two_bf16(next[0], next[1]), two_bf16(next[2], next[3])};
          } else {
            *reinterpret_cast<any_u32x2*>(to) = four;
          }
        }
      }
    }
  };
  auto store = [&](auto gated_by) __attribute__((always_inline)) {
    each_of(std::make_integer_sequence<int, TM>{}, [&](auto i) __attribute__((always_inline)) { store_row(i, gated_by); });
  };
  if constexpr (!GATED) {
    store([](auto, float g, float) { return g; });
  } else if (limit > 0.f) {
    store([&](auto type, float g, float u) { return act == kSiluStored ? clamped_gate<decltype(type)>(g, u, limit) : clamped_gate<float>(g, u, limit); });
  } else if (act == kRelu) {
    store([](auto, float g, float u) { return fmaxf(g, 0.f) * u; });
  } else if (act == kSilu) {
    store([](auto, float g, float u) { return silu<float>(g) * u; });
  } else {
    store([](auto type, float g, float u) { return gated<decltype(type)>(g, u, 0.f, kSiluStored); });
  }
}

// The tiles, and what a launch of them takes (TileTime).  Fitted to 120,000 timed launches (kernel times; 1 to 33,000 rows, 64 to
// 32,000 columns, K 256 to 14,336, S as rows_splits has it, gated or not) of these tiles and two more at 5,800 shapes, widths as models have them and random ones; with half of the
// shapes for the fit a pick is 0.6 % slower than the fastest tile below 96 rows and 0.9 % from there on at the other half, 27 % at worst (576 x 3072 x 5120: 96 x 96, 40.6 us,
// 128 x 64 31.9).  From 96 rows on tile_pipe.h's are mostly the faster, but not everywhere: the ring's 128 x 64, 128 x 96 and 128 x 128 stay for short chains and for tiles that just
// fill the chip (us, the best of tile_pipe.h / so: gate and up of 512 x 2816 x 2048 24.6 / 20.2, 128 x 11264 x 2048 in two slices 17.7 / 15.6, 256 x 8192 x 2048 19.2 / 17.1,
// 117 x 7680 x 1600 in four 14.2 / 12.0), its 64 x 32 for few columns (48 x 8192 x 2048 10.3 in 32 x 64, 9.6).
// 16 x 32's constant a round is larger than fitted (0.267): two rounds of it and one of 16 x 64, alike one after the other (9 x 4096 x 14336 in four 21.8 / 22.1; x 8192 14.6 / 13.9), are not
// in a decode step (22.4 / 21.7).
// (columns, after the sizes and waves: the stages, and whether the tile is tile_pipe.h's)
struct Tile {
  int bm, bn;
  bool pipe;
  TileTime time;
};
#define KVCM_TILES(T)                                         \
  T(16, 32, 1, 2, 8, false, 2.786f, 0.121f, 0.654f, 0.800f)   \
  T(16, 48, 1, 3, 8, false, 2.807f, 0.137f, 0.742f, 0.631f)   \
  T(16, 64, 1, 4, 8, false, 2.851f, 0.169f, 0.772f, 0.596f)   \
  T(32, 32, 2, 2, 8, false, 2.822f, 0.137f, 0.779f, 0.448f)   \
  T(32, 64, 2, 2, 6, false, 3.181f, 0.192f, 0.768f, 0.705f)   \
  T(64, 32, 2, 2, 6, false, 3.325f, 0.205f, 0.636f, 0.782f)   \
  T(64, 64, 2, 2, 4, false, 3.307f, 0.257f, 0.813f, 0.702f)   \
  T(64, 96, 2, 3, 6, false, 4.094f, 0.323f, 1.025f, 2.233f)   \
  T(128, 96, 4, 3, 5, false, 5.016f, 0.443f, 1.016f, 2.905f)  \
  T(96, 64, 2, 2, 4, true, 4.215f, 0.262f, 0.807f, 0.743f)    \
  T(96, 96, 2, 2, 4, true, 4.792f, 0.337f, 0.974f, 2.752f)    \
  T(96, 128, 2, 2, 4, true, 5.086f, 0.416f, 0.968f, 2.478f)   \
  T(128, 128, 2, 2, 4, true, 5.719f, 0.475f, 0.956f, 3.012f)  \
  T(192, 128, 2, 2, 3, true, 6.599f, 0.560f, 0.986f, 3.838f)  \
  T(192, 192, 2, 2, 3, true, 7.789f, 0.727f, 1.051f, 4.891f)  \
  T(256, 192, 2, 2, 2, true, 8.017f, 1.076f, 0.992f, 5.221f)  \
  T(256, 256, 2, 2, 2, true, 9.432f, 1.289f, 1.014f, 6.981f)  \
  T(128, 64, 4, 2, 6, false, 4.459f, 0.311f, 1.049f, 2.637f)  \
  T(128, 128, 2, 4, 4, false, 5.580f, 0.519f, 0.993f, 3.535f) \
  T(256, 128, 2, 2, 3, true, 7.905f, 0.649f, 0.998f, 5.019f)

#define KVCM_TILE_ROW(BM, BN, WM, WN, STAGES, PIPE, FIXED, STEP, SHARE, ROUND) {BM, BN, PIPE, {FIXED, STEP, SHARE, ROUND}},
static constexpr Tile kTiles[] = {KVCM_TILES(KVCM_TILE_ROW)};
#undef KVCM_TILE_ROW
constexpr int kTileCount = sizeof(kTiles) / sizeof(kTiles[0]);
constexpr int kFurtherTiles = 3;      // the last ones, which have numbers of their own
constexpr int kCUs = 256;

float tile_time(const TileTime& t, float groups, int steps, float weights, float again) {
  const float each = groups > static_cast<float>(kCUs) ? std::ceil(groups / static_cast<float>(kCUs)) : 1.f;
  const float chain = t.fixed + t.step * static_cast<float>(steps) * (each > 1.f ? each * t.share : 1.f) + t.round * (each - 1.f);
  const float stream = 2.3f + weights * 2e-6f / 5.9f, rows = 2.3f + again * 1.8e-7f;
  const float c2 = chain * chain, s2 = stream * stream, r2 = rows * rows;
  return std::sqrt(std::sqrt(c2 * c2 + s2 * s2 + r2 * r2));
}

// folded: rows whose norm is still to be applied, which the tiles of tile_pipe.h do not take
static int best_tile(int M, int wrows, int K, int S, float* time = nullptr, bool folded = false) {
  int best = 0;
  float best_t = 0.f;
  for (int i = 0; i < kTileCount; ++i) {
    if (folded && kTiles[i].pipe) continue;
    if (kTiles[i].bm > 16 && kTiles[i].bm >= 2 * M) continue;      // more than half of the rows would not exist
    const int cols = (wrows + kTiles[i].bn - 1) / kTiles[i].bn;
    const float groups = static_cast<float>(static_cast<long long>((M + kTiles[i].bm - 1) / kTiles[i].bm) * cols * S), k = static_cast<float>(K);
    const float t = tile_time(kTiles[i].time, groups, (K / kStepK + S - 1) / S, static_cast<float>(wrows) * k, static_cast<float>(M) * k * static_cast<float>(cols));
    if (i == 0 || t < best_t) {
      best = i;
      best_t = t;
    }
  }
  if (time != nullptr) *time = best_t;
  return best;
}

static float stored_time(int M, int N, int S, bool out_f32) {
  return static_cast<float>(M) * static_cast<float>(N) * (S > 1 ? 4.f * S : out_f32 ? 4.f : 2.f) * 0.12e-6f;
}

float gemm_tiles_time(int M, int N, int K, int S, bool is_gated, bool out_f32) {
  float t = 0.f;
  best_tile(M, is_gated ? 2 * N : N, K, S, &t);
  return t + stored_time(M, N, S, out_f32);
}

template <int BM, int BN, int WM, int WN, int STAGES, bool GATED>
static int launch_pipe(const TilesCall& c, hipStream_t st) {
  const int tiles_m = (c.M + BM - 1) / BM, tiles_n = ((GATED ? 2 * c.N : c.N) + BN - 1) / BN;
  const long long grid = static_cast<long long>(tiles_m) * tiles_n * c.S;
  KVCM_REQUIRE(grid < (1ll << 31), "gemm_tiles: too many tiles");
  KVCM_REQUIRE(c.ss_in == nullptr, "gemm_tiles: large tiles take no folded norm");
  gemm_pipe_kernel<BM, BN, WM, WN, STAGES, GATED><<<static_cast<unsigned>(grid), WM * WN * kWave, 0, st>>>(
      c.X, c.W, c.partials, c.out, c.out_f32, c.M, c.N, c.K, c.ldx, c.ldw, c.ldo, c.S, tiles_m, tiles_n, c.limit, c.act);
  return launch_status("gemm_tiles");
}

template <int BM, int BN, int WM, int WN, int STAGES, bool GATED, class Offset = uint32_t>
static int launch_tiles(const TilesCall& c, hipStream_t st) {
  const int tiles_m = (c.M + BM - 1) / BM, tiles_n = ((GATED ? 2 * c.N : c.N) + BN - 1) / BN;
  const long long grid = static_cast<long long>(tiles_m) * tiles_n * c.S;
  KVCM_REQUIRE(grid < (1ll << 31), "gemm_tiles: too many tiles");
  gemm_tiles_kernel<BM, BN, WM, WN, STAGES, GATED, Offset><<<static_cast<unsigned>(grid), WM * WN * kWave, 0, st>>>(
      c.X, c.W, c.partials, c.out, c.out_f32, c.M, c.N, c.K, c.ldx, c.ldw, c.ldo, c.S, tiles_m, tiles_n, c.ss_in, c.tiles_in, c.eps, c.limit,
      c.act);
  return launch_status("gemm_tiles");
}

template <int BM, int BN, int WM, int WN, int STAGES, bool PIPE, bool GATED>
static int launch(const TilesCall& c, hipStream_t st) {
  if constexpr (PIPE) return launch_pipe<BM, BN, WM, WN, STAGES, GATED>(c, st);
  else return launch_tiles<BM, BN, WM, WN, STAGES, GATED>(c, st);
}

int gemm_tiles(const TilesCall& c, bool is_gated, int tile, hipStream_t st) {
  KVCM_REQUIRE(c.M > 0 && c.N > 0 && c.N % 4 == 0 && c.K > 0 && c.K % kStepK == 0 && c.S >= 1 && c.S <= c.K / kStepK,
               "gemm_tiles: unsupported shape M=%d N=%d K=%d in %d slices", c.M, c.N, c.K, c.S);
  KVCM_REQUIRE(!is_gated || (c.N % 8 == 0 && c.S == 1), "gemm_tiles: gated products take widths of multiples of 8 and are unsplit");
  // (rows of 8 MB or that far apart: one tile for all sizes; what such a product takes is its bytes)
  if (c.ldx >= kFarRows || c.ldw >= kFarRows)
    return is_gated ? launch_tiles<64, 64, 2, 2, 4, true, uint64_t>(c, st) : launch_tiles<64, 64, 2, 2, 4, false, uint64_t>(c, st);
  if (tile < 0) tile = best_tile(c.M, is_gated ? 2 * c.N : c.N, c.K, c.S, nullptr, c.ss_in != nullptr);
  int i = 0;
#define KVCM_TILE_LAUNCH(BM, BN, WM, WN, STAGES, PIPE, FIXED, STEP, SHARE, ROUND) \
  if (tile == i++) return is_gated ? launch<BM, BN, WM, WN, STAGES, PIPE, true>(c, st) : launch<BM, BN, WM, WN, STAGES, PIPE, false>(c, st);
  KVCM_TILES(KVCM_TILE_LAUNCH)
#undef KVCM_TILE_LAUNCH
  KVCM_REQUIRE(false, "gemm_tiles: no tile %d", tile);
}

}  // namespace kvcm

using namespace kvcm;

extern "C" {

// How many tiles there are (and how many further ones, numbered on from there), the rows and columns (of W) of one, and the one the rule picks: for
// tests, which run each.
int kvcm_gemm_tiles_count() { return kTileCount - kFurtherTiles; }
int kvcm_gemm_tiles_further() { return kFurtherTiles; }
int kvcm_gemm_tiles_size(int tile, int* rows, int* cols) {
  KVCM_REQUIRE(tile >= 0 && tile < kTileCount, "gemm_tiles_size: no tile %d", tile);
  *rows = kTiles[tile].bm;
  *cols = kTiles[tile].bn;
  return 0;
}
int kvcm_gemm_tiles_pick(int M, int N, int K, int S, int is_gated) {
  KVCM_REQUIRE(M > 0 && N > 0 && K > 0 && S >= 1, "gemm_tiles_pick: bad sizes");
  return best_tile(M, is_gated ? 2 * N : N, K, S);
}
// The product with a given tile (< 0: the one the rule picks).  is_gated: W [2 N, K], out [M, N] = act(gate) * up (act: 0 silu with the
// roundings of a stored product followed by kvcm_swiglu; 1 silu, 2 relu, exact and rounded once), or the gate with limits (limit > 0).
int kvcm_gemm_tiles(const void* X, const void* W, float* partials, void* out, int out_dtype, int M, int N, int K, int ldx, int ldw, int ldo,
                    int S, int is_gated, int act, float limit, int tile, hipStream_t st) {
  KVCM_REQUIRE(ldx % 8 == 0 && ldw % 8 == 0 && reinterpret_cast<uintptr_t>(X) % 16 == 0 && reinterpret_cast<uintptr_t>(W) % 16 == 0,
               "gemm_tiles: operands must be 16-byte aligned with leading dimensions that are multiples of 8");
  KVCM_REQUIRE(ldx >= K && ldw >= K && (S > 1 ? partials != nullptr : out != nullptr && ldo >= N), "gemm_tiles: missing buffer or leading dimension too small");
  KVCM_REQUIRE(out_dtype == kBF16 || out_dtype == kF32, "gemm_tiles: unknown output dtype %d", out_dtype);
  KVCM_REQUIRE(act >= kSiluStored && act <= kRelu, "gemm_tiles: unknown activation %d", act);
  TilesCall c{static_cast<const uint16_t*>(X), static_cast<const uint16_t*>(W), partials, out, out_dtype == kF32, M, N, K, ldx, ldw, ldo, S};
  c.limit = limit;
  c.act = act;
  return gemm_tiles(c, is_gated != 0, tile, st);
}

// What the library takes for M x wrows x K, us: the fastest of three sizes of tile, each with a constant, a step's chain for every round of 256
// workgroups and a step's share of the chip, or tiles of 128 x 128 with K cut into up to 16 slices until they are 256; and the results' storing, by their bytes.
static float library_time(int M, int wrows, int K, bool out_f32) {
  struct LibraryTile {
    int size;
    float fixed, chain, share;
  };
  static constexpr LibraryTile kLibrary[] = {{256, 5.87f, 0.321f, 0.929f}, {128, 7.47f, 0.115f, 0.525f}, {64, 0.68f, 1.28f, 0.182f}};
  const float steps = static_cast<float>(K) / kStepK;
  float best = 0.f, part = 0.f;
  for (const LibraryTile& l : kLibrary) {
    const float tiles = static_cast<float>((M + l.size - 1) / l.size) * static_cast<float>((wrows + l.size - 1) / l.size) / static_cast<float>(kCUs);
    const float t = l.fixed + steps * (l.chain * std::ceil(tiles) + l.share * tiles);
    if (best == 0.f || t < best) best = t;
    if (l.size == 128) part = tiles;
  }
  const float slices = std::fmin(std::fmax(std::floor(1.f / part), 1.f), 16.f), cut = 8.22f + steps * (0.585f / slices + 1.028f * part);
  return std::fmin(best, cut) + static_cast<float>(M) * static_cast<float>(wrows) * (out_f32 ? 1.19e-6f : 0.595e-6f);
}

// Is a product of many rows, in S slices of K that its consumer adds, faster here than by the vendor library (is_gated: than that and
// the launch that applies the activation, 3.4 us and 6 bytes a result at 5 TB/s)?  Beyond 2,048 rows a plain product is the library's, whose tiles of 256 x 256 are 5 to 15 %
// faster once every CU has several (32,768 rows: 2048 x 5632 565 / 505 us, 2560 x 2048 266 / 240), a gated one is not: it saves the second launch and
// the product's trip to memory (32,768 rows of gate and up, 5632 x 2048: 1,118 / 1,276 us; 8,192 rows 308 / 408; 9,608 rows, 14336 x 4096 1,698 / 1,779).  Up to there the
// tile's modelled time, with the slices' reading (4.5 TB/s, and 55 KB a us of one row's through the CU that norms it), against the modelled library's, which was fitted to
// half of 2,329 plain shapes (1,397 of widths as models have them, the others random; 64 to 32,000 columns, K 256 to 14,336, 96 to 2,048 rows).  It is off by 11 and 18 % a shape: which of
// its kernels the library picks hangs on more than the sizes (256 x 128 x 5632 9.1 us, x 5120 17.5).  So the line lies a little on its side, and further where it is known to be better
// than modelled and little is lost by it: 513 to 1,024 rows of fewer than 116 tiles of 128 x 128 (768 x 2048 x 5632 31.9, here 33.2; 513 x 2048 x 2048 12.8, here 10.8: up to 640 rows a factor
// of 0.87, with 0.78 what it picked was a tenth slower there; beyond, 0.78 leaves 700 x 2048 x 2048, 13.1, here 11.1, with the library), and few columns of long K;
// on the tiles' up to 256 rows of more than 16, where it is often far slower than modelled (256 x 5632 x 5632 54, here 37).
// What the rule picks is 2.1 and 5 % slower than the better of the two, gated (1,197 shapes, 96 to 33,000 rows) 1.2 and 0.6 %.  Against the line and the tiles from before there were
// tiles of four waves: 0.96 and 0.93 of the time, gated 0.90 and 0.80, slower by more than 5 % at 53 and 9, gated 19 and 8; with the line that came with those tiles it was 209 and 71,
// gated 64 and 33.  At 1,420 plain shapes that the fit had not seen 0.965 and 0.95, slower by more than 5 % at 83 of 1,220 and 19 of 200; 571 gated 0.92 and 0.85, at 37 and 14.
// 32-bit results, 900 shapes that the fit had not seen: 1.5 % slower than the better of the two, by more than 5 % at 89; with their storing priced as two bytes 3.3 %, at 159
// (2048 x 8256 x 2048 75.7 here, 90.6; 2048 x 8192 x 2048 59.3, 63.3).
// (us, here / library: taken 2048 x 2560 x 2048 25.8 / 29.0, 1040 x 2048 x 2048 17.2 / 23.0, 1024 x 1024 x 512 5.9 / 9.0, 2048 x 2048 x 5632 52.2 / 52.7; 2,048 and 1,024 rows of gate and up,
// 5632 x 2048, 90 / 92 and 49 / 57; not taken 640 x 64 x 14336 30 / 17, 1040 x 8192 x 2048 44 / 36, 2048 x 8192 x 2048 52 / 50, 384 x 2048 x 5632 whole 27 / 25, 2048 x 256 x 5632 21.7 / 20.6.)
int kvcm_gemm_tiles_preferred(int M, int N, int K, int S, int is_gated, int out_dtype) {
  if (M <= 0 || N <= 0 || N % 64 != 0 || K <= 0 || K % kStepK != 0 || S < 1 || S > K / kStepK || (is_gated && S > 1)) return 0;
  if (M > 2048 && !is_gated) return 0;
  const float results = static_cast<float>(M) * static_cast<float>(N);
  const int wrows = is_gated ? 2 * N : N;
  const bool out_f32 = out_dtype == kF32;
  float here = 0.f;
  best_tile(M, wrows, K, S, &here);
  here += stored_time(M, N, S, out_f32) +
          (S > 1 ? results * (4.f * S - 2.f) / 4.5e6f + static_cast<float>(N) * 4.f * S / 55e3f : 0.f);
  const float library = library_time(M, wrows, K, out_f32);
  if (is_gated) return here <= library + 3.4f + results * 6.f / 5e6f;
  const long long tiles = static_cast<long long>((M + 127) / 128) * ((N + 127) / 128);
  const float side = M <= 256 && tiles > 16 ? 1.1f : M > 512 && M <= 1024 && tiles < 116 ? (M <= 640 ? 0.87f : 0.78f) : N <= 320 && K >= 5632 ? 0.84f : 0.98f;
  return here <= side * library;
}

}  // extern "C"
