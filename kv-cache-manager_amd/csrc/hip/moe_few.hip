// The routed feed-forward's two products for steps of a few rows (bfloat16, up to 64 (row, slot) pairs) on the matrix cores,
// expert by expert: an expert's weights are read once for all the rows that chose it, where the row-by-row kernels of moe.hip
// read them once per row.  Eight rows with two of eight experts each read 7 experts instead of 16.
//
// What bounds these launches is how many weight bytes are on their way, so the work is cut as in the products of up to 8 rows
// (gemm_rows8.hip): many workgroups, every lane with all the weight pieces of a trip requested at once, two trips on their way.
// Which rows share an expert is found by every wave from the pairs' experts, one a lane: the lanes that hold the same number
// are a ballot, so nothing is sorted beforehand and no list goes through memory.
//
//   up     A workgroup belongs to one pair and 32 rows of its expert's matrix (gated: 16 gate and 16 up rows, the results 16
//          activations).  It works if its pair is the first with that expert, for every pair with it, sixteen at a time; the
//          others leave at once.  Four waves divide K; their sums meet in LDS in wave order.
//   down   A workgroup owns 8 output columns of every row, so that the sum over a row's slots stays inside it (in slot order, no
//          scratch, no further launch).  Its eight waves take the experts in turn; an instruction serves two halves of K (operand
//          rows and columns 0..7 the first half, 8..15 the second, only the two diagonal blocks mean anything).
//
// A shared feed-forward that runs for every row, and a route by a table, may run in the same two launches (MoeBeside): what they cost otherwise
// is mostly the start and the end of launches that leave CUs idle.
//
// Measured over weights that go round several copies, row by row / here, us: 8 rows, 8 experts of which a row uses 2, width
// 2,048, 1,408 columns an expert: up 31.3 / 19.7 (92 MB, 4.7 TB/s), down 17.3 / 12.6; 15 rows 51.9 / 20.1 and 28.9 / 14.0; 4 rows 18.4 /
// 13.3 and 11.3 / 9.3; width 4,096, 3,584 columns, 8 rows: 135 / 85 and 69 / 48.  Which sizes come here: up_gains, down_gains, below.
#include <cmath>

#include "common.h"
#include "kvcm_hip.h"

namespace kvcm {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

namespace {

constexpr int kUnit = 64;      // k of a unit: 4 lanes x 16, one 128-byte line of a row

union Frag {
  uint4 u;
  bf16x8 v;
};

// the n-th (from 0) set bit of pairs, or the first one where there are fewer
__device__ __forceinline__ int nth_pair(unsigned long long pairs, int n, int most) {
  int p = __ffsll(pairs) - 1;
#pragma unroll 4
  for (int i = 0; i < most && pairs; ++i, pairs &= pairs - 1) p = i == n ? __ffsll(pairs) - 1 : p;
  return p;
}

// GATED: rows of the matrix are 2F, sixteen gate rows, sixteen up rows, ...; else F, and KIND 0 square(relu), 2 gelu
constexpr int kUpWaves = 4, kUpTrip = 2;      // waves that divide K, units of a trip

// What runs beside the experts in their launches: a feed-forward of silu(gate) * up for every row (F columns; w_up [gate rows | up rows], act [T, F],
// w_down [H, F]), and the route by a table per token id (tokens null: none), which is left for the second launch.
struct MoeBeside {
  const uint16_t* w_up; uint16_t* act; int F;
  const int* tokens; const int* table; int vocab, ld_table;
  int* chosen; float* weight; float in_scale;      // in_scale: the factor on what an expert reads where no in_weight is given
};

// BESIDE: the first `beside_rows` rows of the grid are the shared feed-forward's, 16 columns a workgroup.
template <int KIND, bool BESIDE>
__global__ void __launch_bounds__(kUpWaves * kWave, 3)
    moe_few_up_kernel(const uint16_t* __restrict__ h, int ldh, const uint16_t* __restrict__ w_up, const int* __restrict__ chosen,
                      uint16_t* act, int n, int K, int F, int top, int E, const float* __restrict__ in_weight, const MoeBeside by, int beside_rows) {
  constexpr bool GATED = KIND == 1;
  static_assert(GATED || !BESIDE, "a shared feed-forward beside gated experts only");
  __shared__ f32x4 red[kUpWaves][2][kWave];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int r = lane % 16, kq = lane / 16;
  const bool shared = BESIDE && int(blockIdx.y) < beside_rows;
  const int tile = shared ? int(blockIdx.y) * gridDim.x + blockIdx.x : blockIdx.x;      // of 32 rows
  const uint16_t* wrow;
  size_t next;
  unsigned long long pairs;
  if (shared) {      // every row is a pair of its own
    if (tile * 16 >= by.F) return;
    wrow = by.w_up + (size_t(tile) * 16 + r) * K + kq * 16;
    next = size_t(by.F) * K;
    const int T = n / top;
    pairs = T >= 64 ? ~0ull : (1ull << T) - 1;
  } else {
    const int mine = int(blockIdx.y) - (BESIDE ? beside_rows : 0);
    int ch = -1;
    if (lane < n) {
      if (BESIDE && by.tokens) {
        const int tok = by.tokens[lane / top];
        ch = tok >= 0 && tok < by.vocab ? by.table[size_t(tok) * by.ld_table + lane % top] : -1;
      } else {
        ch = chosen[lane];
      }
    }
    if (BESIDE && by.tokens && mine == 0 && tile == 0 && int(threadIdx.x) < n) {
      by.chosen[threadIdx.x] = ch;
      by.weight[threadIdx.x] = 1.0f / float(top);
    }
    const int e = __builtin_amdgcn_readlane(ch, mine);
    if (e < 0 || e >= E) return;
    pairs = __ballot(ch == e);
    if (__ffsll(pairs) - 1 != mine) return;
    wrow = w_up + (size_t(e) * (GATED ? 2 * F : F) + size_t(tile) * 32 + r) * K + kq * 16;
    next = size_t(16) * K;
  }
  const int per_row = shared ? 1 : top;
  const int units = K / kUnit, u_lo = units * wave / kUpWaves, u_hi = units * (wave + 1) / kUpWaves;
  struct Trip {
    Frag w[2][kUpTrip][2], x[kUpTrip][2];
  };
  for (; pairs;) {      // (more than sixteen pairs of one expert: the weights again, from a cache)
    const int count = __popcll(pairs) < 16 ? __popcll(pairs) : 16;
    const uint16_t* xrow = h + size_t(nth_pair(pairs, r, 16) / per_row) * ldh + kq * 16;
    f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
    auto request = [&](int u0, Trip& t) {      // past the slice: its last unit again, not multiplied
#pragma unroll
      for (int d = 0; d < kUpTrip; ++d) {
        const size_t off = size_t(u0 + d < u_hi ? u0 + d : (u_hi > 0 ? u_hi - 1 : 0)) * kUnit;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          t.w[0][d][q].u = *reinterpret_cast<const uint4*>(wrow + off + q * 8);
          t.w[1][d][q].u = *reinterpret_cast<const uint4*>(wrow + next + off + q * 8);
          t.x[d][q].u = *reinterpret_cast<const uint4*>(xrow + off + q * 8);
        }
      }
    };
    auto multiply = [&](int u0, const Trip& t) {
#pragma unroll
      for (int d = 0; d < kUpTrip; ++d) {
        if (u0 + d >= u_hi) break;      // uniform over the wave
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(t.x[d][q].v, t.w[0][d][q].v, acc[0], 0, 0, 0);
          acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(t.x[d][q].v, t.w[1][d][q].v, acc[1], 0, 0, 0);
        }
      }
    };
    if (u_lo < u_hi) {
      Trip ta, tb;
      request(u_lo, ta);
      request(u_lo + kUpTrip, tb);
      for (int u = u_lo; u < u_hi; u += 2 * kUpTrip) {
        multiply(u, ta);
        if (u + 2 * kUpTrip < u_hi) request(u + 2 * kUpTrip, ta);
        multiply(u + kUpTrip, tb);
        if (u + 3 * kUpTrip < u_hi) request(u + 3 * kUpTrip, tb);
      }
    }
    red[wave][0][lane] = acc[0];
    red[wave][1][lane] = acc[1];
    __syncthreads();
    // thread -> (pair m of this group, column c of a tile); results: column lane % 16, rows 4 (lane / 16) + i
    const int m = threadIdx.x / 16, c = threadIdx.x % 16;
    if (m < count) {
      const int pair = nth_pair(pairs, m, 16);
      const float g = shared ? 1.f : in_weight ? in_weight[pair] : BESIDE ? by.in_scale : 1.f;
      float z[2] = {0.f, 0.f};
#pragma unroll
      for (int w = 0; w < kUpWaves; ++w)
#pragma unroll
        for (int t = 0; t < 2; ++t) z[t] += red[w][t][m / 4 * 16 + c][m % 4];
      if (shared) {      // (with the exact functions, as the products of gate and up rows have it)
        if constexpr (BESIDE) by.act[size_t(pair) * by.F + size_t(tile) * 16 + c] = float_to_bf16_bits(silu<float>(z[0]) * z[1]);
      } else if constexpr (GATED) {
        act[size_t(pair) * F + size_t(tile) * 16 + c] = float_to_bf16_bits(silu<bf16_t>(g * z[0]) * (g * z[1]));
      } else {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const float y = g * z[t], p = fmaxf(y, 0.f);
          act[size_t(pair) * F + size_t(tile) * 32 + t * 16 + c] = float_to_bf16_bits(KIND == 2 ? gelu_exact<bf16_t>(y) : p * p);
        }
      }
    }
    for (int i = 0; i < count; ++i) pairs &= pairs - 1;
    if (pairs) __syncthreads();      // the sums are read before the next group's are written
  }
}

constexpr int kDownWaves = 8, kBesideWaves = 4, kMostPairs = 64;

// BESIDE: four more waves take the shared feed-forward's second product, a quarter of its columns each, which is added to the experts' sum in wave
// order.  (As one more turn of the experts' waves it waits for theirs: 19.5 us, as much as two launches.)
template <bool BESIDE>
__global__ void __launch_bounds__((kDownWaves + (BESIDE ? kBesideWaves : 0)) * kWave, BESIDE ? 3 : 2)
    moe_few_down_kernel(const uint16_t* __restrict__ act, const uint16_t* __restrict__ w_down, const int* __restrict__ chosen,
                        const float* __restrict__ weight, const float* __restrict__ add, float* __restrict__ out, int T, int F,
                        int H, int top, int E, const uint16_t* __restrict__ by_act, const uint16_t* __restrict__ by_down, int by_F) {
  __shared__ float z[kMostPairs][8];
  __shared__ float by_z[BESIDE ? kBesideWaves : 1][BESIDE ? kMostPairs : 1][8];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int n = T * top, n0 = blockIdx.x * 8;
  const int em = threadIdx.x / 8, en = threadIdx.x % 8;      // the last step's (row, column)
  const float start = !BESIDE && add && em < T ? add[size_t(em) * H + n0 + en] : 0.f;
  const int ch = lane < n ? chosen[lane] : -1;
  unsigned long long left = __ballot(ch >= 0 && ch < E);
  const int r = lane % 16, kq = lane / 16, half = r / 8, c = r % 8;
  constexpr int kDownTrip = BESIDE ? 3 : 4;      // (twelve waves have fewer registers each)
  struct Trip {
    Frag w[kDownTrip][2], x[kDownTrip][2];
  };
  // `units` of K from u0 on: eight columns' rows of a matrix (wrow: this lane's) with the rows of `pairs` (xs, `width` apart), to zs
  auto turn = [&](const uint16_t* wrow, const uint16_t* xs, int width, int u0, int units, unsigned long long pairs, float(*zs)[8]) {
    const int n_main = units / 2, n_max = units - n_main;      // the second half may have a unit more
    const int u_lo = half * n_main, cnt = half ? n_max : n_main;
    while (pairs) {      // (more than eight pairs of one expert: the weights again, from a cache)
      const uint16_t* xrow = xs + size_t(nth_pair(pairs, c, 8)) * width + kq * 16;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      auto request = [&](int j0, Trip& t) {      // past this half's slice: its last unit again (or the row's first), not multiplied
#pragma unroll
        for (int d = 0; d < kDownTrip; ++d) {
          const int j = j0 + d < cnt ? j0 + d : (cnt > 0 ? cnt - 1 : 0);
          const size_t off = size_t(u0 + (u_lo + j < units ? u_lo + j : 0)) * kUnit;
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            t.w[d][q].u = *reinterpret_cast<const uint4*>(wrow + off + q * 8);
            t.x[d][q].u = *reinterpret_cast<const uint4*>(xrow + off + q * 8);
          }
        }
      };
      auto multiply = [&](int j0, const Trip& t) {
#pragma unroll
        for (int d = 0; d < kDownTrip; ++d) {
          const int j = j0 + d;
          if (j >= n_max) break;      // uniform over the wave
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            Frag x = t.x[d][q], w = t.w[d][q];
            if (j >= n_main && j >= cnt) {      // this half has run out: it adds nothing
              x.u = uint4{0u, 0u, 0u, 0u};
              w.u = uint4{0u, 0u, 0u, 0u};
            }
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x.v, w.v, acc, 0, 0, 0);
          }
        }
      };
      if (n_max > 0) {
        Trip ta, tb;
        request(0, ta);
        request(kDownTrip, tb);
        for (int j = 0; j < n_max; j += 2 * kDownTrip) {
          multiply(j, ta);
          if (j + 2 * kDownTrip < n_max) request(j + 2 * kDownTrip, ta);
          multiply(j + kDownTrip, tb);
          if (j + 3 * kDownTrip < n_max) request(j + 3 * kDownTrip, tb);
        }
      }
      // results: column lane % 16, rows 4 (lane / 16) + i.  Pairs 0..7 of columns 0..7 over the first half are in lanes with column < 8
      // of the first two lane groups, the second half's in lanes with column >= 8 of the last two: 40 lanes apart
      const int count = __popcll(pairs) < 8 ? __popcll(pairs) : 8;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float far = __shfl(acc[q], (lane + 40) % kWave, kWave);
        const int m = 4 * kq + q;
        if (lane < 32 && r < 8 && m < count) zs[nth_pair(pairs, m, 8)][c] = acc[q] + far;
      }
      for (int k = 0; k < count; ++k) pairs &= pairs - 1;
    }
  };
  for (int i = 0; left; ++i) {      // the experts in the order of their first pair, each wave every eighth
    const int e = __builtin_amdgcn_readlane(ch, __ffsll(left) - 1);
    const unsigned long long pairs = __ballot(ch == e);
    left &= ~pairs;
    if (i % kDownWaves == wave) turn(w_down + (size_t(e) * H + n0 + c) * F + kq * 16, act, F, 0, F / kUnit, pairs, z);
  }
  if (BESIDE && wave >= kDownWaves) {
    const int q = wave - kDownWaves, units = by_F / kUnit, u0 = units * q / kBesideWaves, u1 = units * (q + 1) / kBesideWaves;
    turn(by_down + size_t(n0 + c) * by_F + kq * 16, by_act, by_F, u0, u1 - u0, T >= 64 ? ~0ull : (1ull << T) - 1, by_z[q]);
  }
  __syncthreads();
  if (em >= T) return;
  float sum = 0.f;
  for (int s = 0; s < top; ++s) {
    const int pair = em * top + s, e = chosen[pair];
    if (e < 0 || e >= E) continue;
    sum = fmaf(weight ? weight[pair] : 1.f, z[pair][en], sum);
  }
  if constexpr (BESIDE) {
    float shared = by_z[0][em][en];
#pragma unroll
    for (int w = 1; w < kBesideWaves; ++w) shared += by_z[w][em][en];
    out[size_t(em) * H + n0 + en] = shared + sum;
  } else {
    out[size_t(em) * H + n0 + en] = add ? start + sum : sum;
  }
}

}  // namespace

constexpr int kFewRows = 3, kDownExperts = 32;

// Do the kernels take these operands?
static bool up_fits(int dtype, const void* h, int ldh, int T, int K, int F, int top) {
  return dtype == kBF16 && static_cast<long long>(T) * top <= kMostPairs && K % kUnit == 0 && F % 32 == 0 && ldh % 8 == 0 &&
         reinterpret_cast<uintptr_t>(h) % 16 == 0;
}
static bool down_fits(int dtype, const void* act, int T, int F, int H, int top) {
  return dtype == kBF16 && static_cast<long long>(T) * top <= kMostPairs && F % kUnit == 0 && H % 8 == 0 && reinterpret_cast<uintptr_t>(act) % 16 == 0;
}

// How many experts the pairs of T rows name on average, evenly loaded: the row-by-row kernels read T top matrices, these so many.
static float experts_met(int T, int top, int E) {
  return static_cast<float>(E) * (1.f - std::pow(1.f - static_cast<float>(top < E ? top : E) / static_cast<float>(E), static_cast<float>(T)));
}

// Are they the faster?  Lines through 1,745 measured sizes (3 to 15 rows; 2 to 64 experts, of which a row uses 1 to 6; width 512 to 4,096, 256 to
// 14,336 columns an expert; other weights and choices from launch to launch).  Both launches against the row-by-row kernels': 0.87 of the
// time on average and 1.03 at worst where the load is even, 0.77 and 1.09 where all rows name the same experts; 0.95 and 1.73, 0.75 and
// 1.63 if all came here.  Row by row / here, us, evenly loaded:
//   up, rows of an expert's matrices (gate and up together).  From 2,816 on (width 1,024 on) a workgroup for each 32 of them fills the chip
//   for few pairs: 16 experts, one a row, 2,816 x 2,048: 4 rows 11.7 / 12.9, 6 rows 18.6 / 16.1.  From 1,408 on it takes more pairs, or pairs that share
//   experts: 1,408 x 2,048, 8 experts, one a row: 8 rows 11.1 / 11.9, 11 rows 13.7 / 12.7; two a row: 5 rows 13.3 / 12.4.  From 1,024 on (width 768 on) more
//   still: 1,024 x 1,024, 8 experts, two a row: 8 rows 8.6 / 7.7; one a row: 8 rows 5.8 / 6.0, 15 rows 7.8 / 7.5.
//   down: an expert is a turn of a wave, however few its pairs, so that sharing decides: 1,408 columns, width 2,048, 16 experts, one a row: 8
//   rows 10.0 / 10.3, 15 rows 16.1 / 13.7; 8 experts, two a row: 3 rows 8.8 / 9.1, 5 rows 12.4 / 10.6.  Width 1,024 is 128 workgroups: 2,048 columns, 8
//   experts, two a row: 8 rows 13.4 / 13.4, 15 rows 20.4 / 16.1; 4 experts, one a row, 4 rows 5.7 / 7.5.
static bool up_gains(int T, int K, int rows, int top, int E) {
  const float n = static_cast<float>(T * top), met = experts_met(T, top, E);
  if (T < kFewRows || K < 768 || rows < 1024) return false;
  if (K >= 1024 && rows >= 2816) return n >= 5.f || n >= 1.6f * met;
  if (K >= 1024 && rows >= 1408 && (n >= 10.f || (n >= 5.f && n >= 1.6f * met))) return true;
  return n >= 16.f || (n >= 8.f && n >= 2.3f * met);
}
static bool down_gains(int T, int F, int H, int top, int E) {
  const float n = static_cast<float>(T * top), met = experts_met(T, top, E);
  if (T < kFewRows || E > kDownExperts) return false;
  if (H >= 2048 && F >= 704) return n >= 6.f && n >= 1.6f * met;
  return n >= 16.f && n >= 2.6f * met && ((H >= 2048 && F >= 512) || (H >= 1024 && F >= 1024));
}

bool moe_few_up_takes(int dtype, const void* h, int ldh, int T, int K, int F, int top, int E, int kind, bool others) {
  return up_fits(dtype, h, ldh, T, K, F, top) && (!others || up_gains(T, K, kind == 1 ? 2 * F : F, top, E));
}
bool moe_few_down_takes(int dtype, const void* act, int T, int F, int H, int top, int E, bool others) {
  return down_fits(dtype, act, T, F, H, top) && (!others || down_gains(T, F, H, top, E));
}

void launch_moe_few_up(const void* h, int ldh, const void* w_up, const int* chosen, void* act, int T, int K, int F, int top, int E, int kind,
                       const float* in_weight, hipStream_t s) {
  const dim3 grid((kind == 1 ? 2 * F : F) / 32, T * top);
#define KVCM_FEW_UP(KIND)                                                                                                       \
  moe_few_up_kernel<KIND, false><<<grid, kUpWaves * kWave, 0, s>>>(static_cast<const uint16_t*>(h), ldh, static_cast<const uint16_t*>(w_up), chosen, \
                                               static_cast<uint16_t*>(act), T * top, K, F, top, E, in_weight, MoeBeside{}, 0)
  if (kind == 1) KVCM_FEW_UP(1);
  else if (kind == 2) KVCM_FEW_UP(2);
  else KVCM_FEW_UP(0);
#undef KVCM_FEW_UP
}

void launch_moe_few_down(const void* act, const void* w_down, const int* chosen, const float* weight, const float* add, float* out, int T,
                         int F, int H, int top, int E, hipStream_t s) {
  moe_few_down_kernel<false><<<H / 8, kDownWaves * kWave, 0, s>>>(static_cast<const uint16_t*>(act), static_cast<const uint16_t*>(w_down), chosen,
                                                           weight, add, out, T, F, H, top, E, nullptr, nullptr, 0);
}

}  // namespace kvcm

using namespace kvcm;

extern "C" {

// (for the parts, whose other choice from 16 rows on is kvcm_moe_grouped) do both products of T rows come here, whatever their strides?
// At 16 rows an expert has at most sixteen pairs, one pass over its matrices, and the down kernel's workgroups are to be about one a CU: both
// products took 0.87 of the time of all launches of the grouped form on average (60 sizes of width 2,048, up to 32 experts; 1.04 at worst), 0.85 and 1.06 where
// all rows name the same experts.  With more rows an expert may be several passes of one wave: evenly loaded 24 rows with two of 8
// experts each take 36.3 us here and 39.5 grouped (1,408 columns), but 31.0 and 24.1 where all name the same two, 64 rows up to 2.7 times as long.
// Width 4,096, 3,584 columns, 8 experts, two a row, 16 rows: 139 / 134.
int kvcm_moe_few_takes(int T, int K, int F, int H, int top, int E, int kind) {
  if (!up_fits(kBF16, nullptr, 0, T, K, F, top) || !down_fits(kBF16, nullptr, T, F, H, top)) return 0;
  if (T == 16) return H > 1536 && H <= 2048 && F >= 256 && top <= 2 && E <= kDownExperts;
  return T < 16 && up_gains(T, K, kind == 1 ? 2 * F : F, top, E) && down_gains(T, F, H, top, E);
}

// The two products by these kernels whatever is the faster (operands as kvcm_moe_up's and kvcm_moe_down's, bfloat16).
int kvcm_moe_few_up(const void* h, int ldh, const void* w_up, const int* chosen, void* act, int T, int K, int F, int top, int E, int kind,
                    const float* in_weight, hipStream_t s) {
  if (T == 0) return 0;
  KVCM_REQUIRE(T > 0 && K > 0 && F > 0 && top > 0 && E > 0 && ldh >= K && kind >= 0 && kind <= 2, "moe_few_up: bad sizes");
  KVCM_REQUIRE(up_fits(kBF16, h, ldh, T, K, F, top) && reinterpret_cast<uintptr_t>(w_up) % 16 == 0, "moe_few_up: unsupported sizes or alignment");
  launch_moe_few_up(h, ldh, w_up, chosen, act, T, K, F, top, E, kind, in_weight, s);
  return launch_status("moe_few_up");
}
int kvcm_moe_few_down(const void* act, const void* w_down, const int* chosen, const float* weight, const float* add, float* out, int T, int F,
                      int H, int top, int E, hipStream_t s) {
  if (T == 0) return 0;
  KVCM_REQUIRE(T > 0 && H > 0 && F > 0 && top > 0 && E > 0, "moe_few_down: bad sizes");
  KVCM_REQUIRE(down_fits(kBF16, act, T, F, H, top) && reinterpret_cast<uintptr_t>(w_down) % 16 == 0, "moe_few_down: unsupported sizes or alignment");
  launch_moe_few_down(act, w_down, chosen, weight, add, out, T, F, H, top, E, s);
  return launch_status("moe_few_down");
}

// The two products with a shared feed-forward of Fs columns beside gated experts (silu, no biases): silu(gate) * up of w_shared_up [2 Fs, K] (gate rows, up
// rows) to act_shared [T, Fs], and out = act_shared w_shared_down^T + the experts' sum.  tokens (null: chosen and weight are read): the route
// by a table per token id as kvcm_moe_table_route leaves it in chosen and weight.  weigh_input: the weights are factors on what an expert reads.
int kvcm_moe_few_beside_supported(int T, int K, int F, int H, int top, int E, int Fs) {
  return T > 0 && E > 0 && top > 0 && Fs > 0 && Fs % kUnit == 0 && F / 16 > 0 && up_fits(kBF16, nullptr, 0, T, K, F, top) && down_fits(kBF16, nullptr, T, F, H, top);
}
// Are they the faster?  Up to 8 rows: two launches of 0.52 to 1.00 of the time of the four (five) one after the other, also where those are the row-by-row
// kernels (us; width 2,048, 1,408 columns an expert, two of 8, shared 2,816: one row 25.2 / 20.9, 4 rows 43.4 / 32.3, 8 rows 51.8 / 45.0; 704, four of 16, shared 704: 8
// rows 51.1 / 41.4; width 1,024, 704, shared 1,408: 8 rows 28.8 / 21.9; width 4,096, 3,584, shared 7,168: 1 row 80.0 / 74.0, 8 rows 150.4 / 147.3, shared 11,264: 120.1 /
// 120.3).  Up to 16 rows while the shared matrices are small: sixteen of the experts' pairs are one pass, but the products of gate and up rows that the
// shared ones take otherwise read them at a better rate (2,816: 12 rows 47.2 / 43.8, 16 rows 52.9 / 50.1; 5,632: 57.2 / 58.0; 4,096 x 7,168: 182.5 / 189.6).
int kvcm_moe_few_beside_takes(int T, int K, int F, int H, int top, int E, int Fs) {
  const long long shared = 2ll * Fs * K;
  return kvcm_moe_few_beside_supported(T, K, F, H, top, E, Fs) && E <= kDownExperts && ((T <= 8 && shared <= 100000000) || (T <= 16 && shared <= 16000000));
}
int kvcm_moe_few_beside_up(const void* h, int ldh, const void* w_up, int* chosen, float* weight, const int* tokens, const int* table, int vocab, int ld_table,
                           const void* w_shared_up, void* act_shared, int Fs, void* act, int T, int K, int F, int H, int top, int E, int weigh_input, hipStream_t s) {
  if (T == 0) return 0;
  KVCM_REQUIRE(kvcm_moe_few_beside_supported(T, K, F, H, top, E, Fs) && ldh >= K && ldh % 8 == 0, "moe_few_beside_up: unsupported sizes");
  KVCM_REQUIRE(h && w_up && chosen && weight && w_shared_up && act_shared && act && (!tokens || (table && vocab > 0 && ld_table >= top)), "moe_few_beside_up: null operand");
  KVCM_REQUIRE((reinterpret_cast<uintptr_t>(h) | reinterpret_cast<uintptr_t>(w_up) | reinterpret_cast<uintptr_t>(w_shared_up)) % 16 == 0,
               "moe_few_beside_up: operands must be 16-byte aligned");
  const int tiles = 2 * F / 32, beside = (Fs / 16 + tiles - 1) / tiles;
  KVCM_REQUIRE(beside + T * top <= 65535, "moe_few_beside_up: the shared feed-forward is too wide");
  const MoeBeside by{static_cast<const uint16_t*>(w_shared_up), static_cast<uint16_t*>(act_shared), Fs, tokens, table, vocab, ld_table, chosen, weight,
                     tokens && weigh_input ? 1.0f / float(top) : 1.0f};
  moe_few_up_kernel<1, true><<<dim3(tiles, beside + T * top), kUpWaves * kWave, 0, s>>>(
      static_cast<const uint16_t*>(h), ldh, static_cast<const uint16_t*>(w_up), chosen, static_cast<uint16_t*>(act), T * top, K, F, top, E,
      !tokens && weigh_input ? weight : nullptr, by, beside);
  return launch_status("moe_few_beside_up");
}
int kvcm_moe_few_beside_down(const void* act, const void* w_down, const int* chosen, const float* weight, const void* act_shared, const void* w_shared_down, int Fs,
                             float* out, int T, int K, int F, int H, int top, int E, hipStream_t s) {
  if (T == 0) return 0;
  KVCM_REQUIRE(kvcm_moe_few_beside_supported(T, K, F, H, top, E, Fs), "moe_few_beside_down: unsupported sizes");
  KVCM_REQUIRE(act && w_down && chosen && act_shared && w_shared_down && out, "moe_few_beside_down: null operand");
  KVCM_REQUIRE((reinterpret_cast<uintptr_t>(act) | reinterpret_cast<uintptr_t>(w_down) | reinterpret_cast<uintptr_t>(act_shared) | reinterpret_cast<uintptr_t>(w_shared_down)) % 16 == 0,
               "moe_few_beside_down: operands must be 16-byte aligned");
  moe_few_down_kernel<true><<<H / 8, (kDownWaves + kBesideWaves) * kWave, 0, s>>>(static_cast<const uint16_t*>(act), static_cast<const uint16_t*>(w_down), chosen, weight, nullptr, out, T, F, H,
                                                                top, E, static_cast<const uint16_t*>(act_shared), static_cast<const uint16_t*>(w_shared_down), Fs);
  return launch_status("moe_few_beside_down");
}

}  // extern "C"
