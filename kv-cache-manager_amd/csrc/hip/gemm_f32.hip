// Y[M,N] = X[M,K] * W[N,K]^T in true 32-bit, on the matrix cores' 32-bit instruction (v_mfma_f32_16x16x4_f32: 32-bit
// operands, 32-bit fused multiply-adds; no mode of lower precision).
//
// Every output element is the same sequence of operations whatever M, the kernel, the tile or the element's place in it, so a
// row's result does not depend on which other rows share the launch.  K is cut into up to 8 segments whose length depends on K
// alone (segment_units).  A segment is one chain of matrix instructions over its units of 32 k in ascending order, halves of 16
// after one another, instruction m of a half taking k = 4 g + m for g = 0..3 (so that a lane's operands of a half are one
// 16-byte load); the segments' sums are added in ascending order.  Against one chain over all of K this halves the error at K = 2048 (shorter chains).
// (The reference has no 32-bit path; its GEMMs are cuBLAS calls with this same operand layout, src/model/llama.cpp:45-52.)
//
// By sizes:
//   K <= 256    one chain over all of K in ascending order (the instruction takes its four k in ascending order, checked bit
//               for bit); the segments above are for longer sums.  Tiles of 32 x 32 or 64 x 64.
//   up to 8 rows of up to 2,048 columns, one or two rows of many: workgroups of 8 columns (gemm_f32_rows8_kernel).
//   few rows    bound by reading W once.  A workgroup owns 16 columns, its waves one segment each, eight 16-byte loads of W a
//               lane multiplied while the next eight are on their way; segments meet in LDS.  Two rows, K = 2048: N = 11264
//               (92 MB) 22 us, 4.2 TB/s; N = 2048 8 us; K = 5632, N = 2048 20 us.  As 16 x 64 tiles of plain fused
//               multiply-adds with scalar loads these took 304 us in the mean.
//               Up to 32 rows of very many columns: tiles of 32 rows as below.
//   more rows   bound by the matrix cores (157 TFLOP/s).  Tiles of 64 x 64 or 64 x 32, four waves, 32 k a step, three further steps on
//               their way (gemm_f32_ring_kernel).  573 rows, K = 2048: N = 11264 225 us (118 TFLOP/s), N = 2048 54; K = 5632, N =
//               2048 141; staged through registers, one step on its way, 247, 66 and 173.  Rows that are not whole 16-byte pieces
//               are staged so still.
#include "common.h"
#include "gemm_f32_order.h"
#include "kvcm_hip.h"
#include "tile_ring.h"

namespace kvcm {

// ---- up to 8 rows: columns 8 blockIdx.x .. + 7, wave w segments w and w + 4 ------------------------------------------------
// The instruction's 16 x 16 results as two blocks of 8 x 8 on the diagonal: operand rows and columns 0..7 are X's rows and W's columns
// over one segment, 8..15 the same over the other (the two blocks beside the diagonal mean nothing).  Every lane then loads W
// of its own where the kernel below has 16 columns a workgroup, so that N / 8 workgroups of four waves cover the chip where N / 16 of eight
// leave half of it idle.  Per element the same chain.
// GATED: W is N gate rows and N up rows; a workgroup has four columns of silu(gate) * up, as the SwiGLU kernel computes it from the same
// sums, whose launch it saves: 2048 x 5632, us, 1 row 24.0 -> 22.5, 8 rows 28.1 -> 27.3; 1024 x 2816 10.0 -> 8.6, 12.9 -> 10.1.
template <bool FOURS, bool GATED = false>
__global__ void __launch_bounds__(kSegments / 2 * kWave)
    gemm_f32_rows8_kernel(const float* __restrict__ X, const float* __restrict__ W, float* __restrict__ Y, int M, int N, int K,
                          int ldx, int ldw, int ldy) {
  __shared__ float sums[kSegments][8][8];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int r = lane & 15, g = lane >> 4, half = r >> 3, r8 = r & 7;
  const int n0 = blockIdx.x * (GATED ? 4 : 8);
  const int at = n0 + (GATED ? r8 % 4 : r8), n = (at < N ? at : N - 1) + (GATED && r8 >= 4 ? N : 0), m = r8 < M ? r8 : M - 1;
  const int seg = segment_units(K), units = (K + kUnit - 1) / kUnit;
  const int s0 = wave, s1 = wave + kSegments / 2;
  // units of the wave's two segments (the later one is never the longer)
  const int long_units = s0 * seg + seg < units ? seg : units - s0 * seg, short_units = s1 * seg + seg < units ? seg : units - s1 * seg;
  const int lo = (half ? s1 : s0) * seg, mine = half ? short_units : long_units;
  const float *w = W + size_t(n) * ldw, *x = X + size_t(m) * ldx;
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int D = 4;
  f32x4 b[2][D][2], a[2][D][2];
  auto fetch = [&](f32x4 (&bb)[D][2], f32x4 (&aa)[D][2], int u) {
    if (u + D <= short_units && (s1 * seg + u + D) * kUnit <= K) {
#pragma unroll
      for (int d = 0; d < D; ++d)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int k = (lo + u + d) * kUnit + 16 * h + 4 * g;
          bb[d][h] = load4<true, true>(w, k, K);
          aa[d][h] = load4<true, true>(x, k, K);
        }
    } else {
#pragma unroll
      for (int d = 0; d < D; ++d)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int k = u + d < mine ? (lo + u + d) * kUnit + 16 * h + 4 * g : K;      // (beyond the segment: zeros)
          bb[d][h] = load4<FOURS>(w, k, K);
          aa[d][h] = load4<FOURS>(x, k, K);
        }
    }
  };
  auto multiply = [&](const f32x4 (&bb)[D][2], const f32x4 (&aa)[D][2]) {
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(aa[d][h][q], bb[d][h][q], acc, 0, 0, 0);
  };
  if (long_units > 0) fetch(b[0], a[0], 0);
  for (int u = 0; u < long_units; u += 2 * D) {
    if (u + D < long_units) fetch(b[1], a[1], u + D);
    __builtin_amdgcn_sched_barrier(0);
    multiply(b[0], a[0]);
    if (u + D >= long_units) break;
    __builtin_amdgcn_sched_barrier(0);
    if (u + 2 * D < long_units) fetch(b[0], a[0], u + 2 * D);
    __builtin_amdgcn_sched_barrier(0);
    multiply(b[1], a[1]);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (g / 2 == half) {
#pragma unroll
    for (int e = 0; e < 4; ++e) sums[half ? s1 : s0][4 * (g & 1) + e][r8] = acc[e];
  }
  __syncthreads();
  const int segments = (units + seg - 1) / seg;
  auto total = [&](int row, int c) {
    float t = sums[0][row][c];
    for (int i = 1; i < segments; ++i) t += sums[i][row][c];
    return t;
  };
  if constexpr (GATED) {
    const int row = threadIdx.x / 4, c = threadIdx.x % 4;
    if (row < M && n0 + c < N) Y[size_t(row) * ldy + n0 + c] = silu<float>(total(row, c)) * total(row, c + 4);
  } else if (threadIdx.x < 64) {
    const int row = threadIdx.x / 8, c = threadIdx.x % 8;
    const float t = total(row, c);
    if (row < M && n0 + c < N) Y[size_t(row) * ldy + n0 + c] = t;
  }
}

// ---- up to 16 * MT rows: columns 16 blockIdx.x .. + 15, wave w segment w ---------------------------------------------------
template <int MT, bool FOURS>
__global__ void __launch_bounds__(kSegments* kWave)
    gemm_f32_rows_kernel(const float* __restrict__ X, const float* __restrict__ W, float* __restrict__ Y, int M, int N, int K,
                         int ldx, int ldw, int ldy) {
  __shared__ float sums[kSegments][MT][4][kWave];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16, m0 = blockIdx.y * 16 * MT;
  const int n = n0 + r < N ? n0 + r : N - 1;
  const int seg = segment_units(K), units = (K + kUnit - 1) / kUnit;
  const int lo = wave * seg, hi = lo + seg < units ? lo + seg : units;
  const float* w = W + size_t(n) * ldw;
  const float* x[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = m0 + 16 * i + r;
    x[i] = X + size_t(m < M ? m : M - 1) * ldx;
  }
  f32x4 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  // D units at a time, the next D on their way meanwhile (the barriers keep the compiler from moving loads to their uses)
  constexpr int D = MT == 1 ? 4 : MT == 2 ? 2 : 1;
  f32x4 b[2][D][2], a[2][D][2][MT];
  auto fetch = [&](f32x4 (&bb)[D][2], f32x4 (&aa)[D][2][MT], int u) {
    if (u + D <= hi && (u + D) * kUnit <= K) {
#pragma unroll
      for (int d = 0; d < D; ++d)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int k = (u + d) * kUnit + 16 * h + 4 * g;
          bb[d][h] = load4<true, true>(w, k, K);
#pragma unroll
          for (int i = 0; i < MT; ++i) aa[d][h][i] = load4<true, true>(x[i], k, K);
        }
    } else {
#pragma unroll
      for (int d = 0; d < D; ++d)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int k = u + d < hi ? (u + d) * kUnit + 16 * h + 4 * g : K;      // (beyond the segment: zeros)
          if (!FOURS && u + d < hi && (u + d + 1) * kUnit <= K) {               // (single loads in the unit with the row's end only)
            bb[d][h] = load4<true, true>(w, k, K);
#pragma unroll
            for (int i = 0; i < MT; ++i) aa[d][h][i] = load4<true, true>(x[i], k, K);
            continue;
          }
          bb[d][h] = load4<FOURS>(w, k, K);
#pragma unroll
          for (int i = 0; i < MT; ++i) aa[d][h][i] = load4<FOURS>(x[i], k, K);
        }
    }
  };
  auto multiply = [&](const f32x4 (&bb)[D][2], const f32x4 (&aa)[D][2][MT]) {
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
          for (int i = 0; i < MT; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(aa[d][h][i][m], bb[d][h][m], acc[i], 0, 0, 0);
  };
  if (lo < hi) fetch(b[0], a[0], lo);
  for (int u = lo; u < hi; u += 2 * D) {
    if (u + D < hi) fetch(b[1], a[1], u + D);
    __builtin_amdgcn_sched_barrier(0);
    multiply(b[0], a[0]);
    if (u + D >= hi) break;
    __builtin_amdgcn_sched_barrier(0);
    if (u + 2 * D < hi) fetch(b[0], a[0], u + 2 * D);
    __builtin_amdgcn_sched_barrier(0);
    multiply(b[1], a[1]);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) sums[wave][i][e][lane] = acc[i][e];
  __syncthreads();
  const int segments = (units + seg - 1) / seg;
  for (int t = threadIdx.x; t < MT * 4 * kWave; t += kSegments * kWave) {
    const int i = t / (4 * kWave), e = t / kWave % 4, l = t % kWave;
    float total = sums[0][i][e][l];
    for (int s = 1; s < segments; ++s) total += sums[s][i][e][l];
    const int m = m0 + 16 * i + 4 * (l >> 4) + e, c = n0 + (l & 15);
    if (m < M && c < N) Y[size_t(m) * ldy + c] = total;
  }
}

// ---- more rows: tiles of 32 TM x 32 TN, four waves of TM x TN instruction tiles each ----------------------------------------
// LDS rows hold 32 k as eight 16-byte pieces, piece c of row r at place c ^ (r & 7): a wave's read of one piece of 16 rows
// meets no bank twice.
// ASCENDING: one chain over all of K instead, k after k: a piece's four elements then go to four pieces as they are staged, so
// that lane group g's piece holds k = 4 m + g for m = 0..3.
template <int TM, int TN, bool FOURS, bool ASCENDING>
__global__ void __launch_bounds__(256, 2)
    gemm_f32_tiles_kernel(const float* __restrict__ X, const float* __restrict__ W, float* __restrict__ Y, int M, int N, int K,
                          int ldx, int ldw, int ldy) {
  constexpr int BM = 32 * TM, BN = 32 * TN, BK = kUnit;      // (32 rows of 8 pieces: one piece a thread)
  __shared__ f32x4 xs[2][BM * 8], ws[2][BN * 8];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int r = lane & 15, g = lane >> 4;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int wm = (wave >> 1) * 16 * TM, wn = (wave & 1) * 16 * TN;
  const int seg = segment_units(K);
  const int srow = threadIdx.x >> 3, sc = threadIdx.x & 7, kc = 4 * sc;
  const float *xr[TM], *wr[TN];
#pragma unroll
  for (int p = 0; p < TM; ++p) xr[p] = X + size_t(m0 + srow + 32 * p < M ? m0 + srow + 32 * p : M - 1) * ldx;
#pragma unroll
  for (int p = 0; p < TN; ++p) wr[p] = W + size_t(n0 + srow + 32 * p < N ? n0 + srow + 32 * p : N - 1) * ldw;
  const int at = srow * 8 + (sc ^ (srow & 7));      // (rows 32 apart have the same place in a row)
  int spread[4];                                    // ASCENDING: where a piece's elements go
#pragma unroll
  for (int e = 0; e < 4; ++e) spread[e] = 4 * (srow * 8 + (((sc & 4) + e) ^ (srow & 7))) + (sc & 3);
  f32x4 px[TM], pw[TN];
  auto fetch = [&](int k0) {
    if (k0 + BK <= K) {
#pragma unroll
      for (int p = 0; p < TM; ++p) px[p] = load4<true, true>(xr[p], k0 + kc, K);
#pragma unroll
      for (int p = 0; p < TN; ++p) pw[p] = load4<true, true>(wr[p], k0 + kc, K);
    } else {
#pragma unroll
      for (int p = 0; p < TM; ++p) px[p] = load4<FOURS>(xr[p], k0 + kc, K);
#pragma unroll
      for (int p = 0; p < TN; ++p) pw[p] = load4<FOURS>(wr[p], k0 + kc, K);
    }
  };
  auto put = [&](f32x4* rows, int p, f32x4 v) {
    if constexpr (ASCENDING) {
      float* to = reinterpret_cast<float*>(rows);
#pragma unroll
      for (int e = 0; e < 4; ++e) to[spread[e] + 1024 * p] = v[e];
    } else {
      rows[at + 256 * p] = v;
    }
  };
  auto stage = [&](int b) {
#pragma unroll
    for (int p = 0; p < TM; ++p) put(xs[b], p, px[p]);
#pragma unroll
    for (int p = 0; p < TN; ++p) put(ws[b], p, pw[p]);
  };
  f32x4 acc[TM][TN], total[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  fetch(0);
  stage(0);
  __syncthreads();
  int left = seg, b = 0;      // units left in the segment
  for (int k0 = 0; k0 < K; k0 += BK, b ^= 1) {
    if (k0 + BK < K) fetch(k0 + BK);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4 a[TM], w[TN];
      const int c = 4 * h + g;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int row = wm + 16 * i + r;
        a[i] = xs[b][row * 8 + (c ^ (row & 7))];
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int row = wn + 16 * j + r;
        w[j] = ws[b][row * 8 + (c ^ (row & 7))];
      }
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][m], w[j][m], acc[i][j], 0, 0, 0);
    }
    if (!ASCENDING && --left == 0) {      // a segment ends
      left = seg;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          total[i][j] += acc[i][j];
          acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    if (k0 + BK < K) stage(b ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if (ASCENDING) total[i][j] = acc[i][j];
      else if (left != seg) total[i][j] += acc[i][j];      // the last segment, where it is shorter
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + wm + 16 * i + 4 * g + e, n = n0 + wn + 16 * j + r;
        if (m < M && n < N) Y[size_t(m) * ldy + n] = total[i][j][e];
      }
    }
}

// The same tiles with operands by 16-byte requests straight into a ring of stages in LDS (tile_ring.h): where rows are whole 16-byte
// pieces and K whole units.  A step has 1,024 cycles of matrix instructions a wave; staged through registers the stores, the
// wait for them and the barrier came on top, here only the barrier.  Per element the same sequence.
template <int TM, int TN, int STAGES>
__global__ void __launch_bounds__(256, 2)
    gemm_f32_ring_kernel(const float* __restrict__ X, const float* __restrict__ W, float* __restrict__ Y, int M, int N, int K,
                         int ldx, int ldw, int ldy, int tiles_m) {
  constexpr int BM = 32 * TM, BN = 32 * TN, R = (BM + BN) / 32;      // requests of eight rows a wave
  constexpr int kStage = (BM + BN) * 128;
  __shared__ __attribute__((aligned(1024))) unsigned char ring[STAGES * kStage];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int r = lane & 15, g = lane >> 4;
  const int id = neighbours_on_one_xcd();
  const int m0 = id % tiles_m * BM, n0 = id / tiles_m * BN;
  const int wm = (wave >> 1) * 16 * TM, wn = (wave & 1) * 16 * TN;
  const int seg = segment_units(K), steps = K / kUnit;
  const uint64_t xbase = reinterpret_cast<uint64_t>(X + size_t(m0) * ldx), wbase = reinterpret_cast<uint64_t>(W + size_t(n0) * ldw);
  uint32_t offset[R];
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int req = q * 4 + wave, row = req * 8 + lane / 8;
    const int at = req < BM / 8 ? (row < M - m0 ? row : M - 1 - m0) : (row - BM < N - n0 ? row - BM : N - 1 - n0);
    offset[q] = static_cast<uint32_t>(at) * static_cast<uint32_t>(req < BM / 8 ? ldx : ldw) * 4u + static_cast<uint32_t>((lane % 8) ^ (lane / 8)) * 16u;
  }
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(
      reinterpret_cast<uintptr_t>(reinterpret_cast<__attribute__((address_space(3))) void*>(reinterpret_cast<uintptr_t>(ring)))));
  auto request = [&](int t, int stage) {
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int req = q * 4 + wave;
      ring_bring16(offset[q], (req < BM / 8 ? xbase : wbase) + static_cast<uint64_t>(t) * 128, lds0 + stage * kStage + req * 1024);
    }
  };
  f32x4 acc[TM][TN], total[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  int left = seg;      // units left in the segment
  auto step = [&](int stage) {
    const f32x4 *xs = reinterpret_cast<const f32x4*>(ring + stage * kStage), *ws = xs + BM * 8;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4 a[TM], w[TN];
      const int c = (4 * h + g) ^ (r & 7);      // (rows 16 apart have the same place in a row)
#pragma unroll
      for (int i = 0; i < TM; ++i) a[i] = xs[(wm + 16 * i + r) * 8 + c];
#pragma unroll
      for (int j = 0; j < TN; ++j) w[j] = ws[(wn + 16 * j + r) * 8 + c];
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][m], w[j][m], acc[i][j], 0, 0, 0);
    }
    if (--left == 0) {      // a segment ends
      left = seg;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          total[i][j] += acc[i][j];
          acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
  };
#pragma unroll
  for (int t = 0; t < STAGES - 1; ++t)
    if (t < steps) request(t, t);
  int stage = 0, fill = STAGES - 1;
  for (int t = 0; t < steps; ++t) {
    if (t + STAGES - 1 < steps) {
      ring_arrived<(STAGES - 2) * R>();
      request(t + STAGES - 1, fill);      // into the stage that everybody has read by now
    } else {
      ring_arrived<0>();
    }
    step(stage);
    fill = fill + 1 == STAGES ? 0 : fill + 1;
    stage = stage + 1 == STAGES ? 0 : stage + 1;
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if (left != seg) total[i][j] += acc[i][j];      // the last segment, where it is shorter
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + wm + 16 * i + 4 * g + e, n = n0 + wn + 16 * j + r;
        if (m < M && n < N) Y[size_t(m) * ldy + n] = total[i][j][e];
      }
    }
}

// Rows of whole 16-byte pieces, whole units.
inline bool through_ring(const float* X, const float* W, int K, int ldx, int ldw) {
  return K % kUnit == 0 && ldx % 4 == 0 && ldw % 4 == 0 && reinterpret_cast<uintptr_t>(X) % 16 == 0 && reinterpret_cast<uintptr_t>(W) % 16 == 0 &&
         ldx < (1 << 22) && ldw < (1 << 22);
}

template <int TM, int TN, bool FOURS, bool ASCENDING>
void launch_tiles(const float* X, const float* W, float* Y, int M, int N, int K, int ldx, int ldw, int ldy, hipStream_t s) {
  const int tiles_n = (N + 32 * TN - 1) / (32 * TN), tiles_m = (M + 32 * TM - 1) / (32 * TM);
  if constexpr (!ASCENDING) {
    const long long groups = static_cast<long long>(tiles_m) * tiles_n;
    if (through_ring(X, W, K, ldx, ldw) && groups < (1ll << 31)) {
      gemm_f32_ring_kernel<TM, TN, 4><<<static_cast<unsigned>(groups), 256, 0, s>>>(X, W, Y, M, N, K, ldx, ldw, ldy, tiles_m);
      return;
    }
  }
  const dim3 grid(tiles_n, tiles_m);
  gemm_f32_tiles_kernel<TM, TN, FOURS, ASCENDING><<<grid, 256, 0, s>>>(X, W, Y, M, N, K, ldx, ldw, ldy);
}

template <bool FOURS>
void launch_gemm_f32(const float* X, const float* W, float* Y, int M, int N, int K, int ldx, int ldw, int ldy, hipStream_t s) {
  // Measured at K = 2048 (us; rows kernel / tiles of 64 x 32 / of 64 x 64).  The rows kernel takes 22 for up to 256 workgroups
  // and about 0.09 for each beyond; the tiles take 41 / 50 as long as a CU has one or two, and 0.084 / 0.165 each beyond.  So
  // rows while the 64 x 32 tiles are few: N = 2048, 64 rows 22 / 41 / 50, 128 rows 23 / 41 / 50, 200 rows 42 / 41 / 50;
  // N = 11264, 64 rows 64 / 53 / 54; up to 32 rows its blocks are half as long (24 rows, N = 11264: 39 / 52 / 54, N = 32000:
  // 100 / 93 / 87), up to 16 always.  The larger tiles (half the columns' rows from L2) from three a CU on: 573 rows, N = 2048
  // 100 / 68 / 76, N = 11264 497 / 255 / 254, N = 32000 1441 / 705 / 660; 2048 rows, N = 11264: 1764 / 841 / 764
  // (124 TFLOP/s).  Tiles of 128 x 128 and 128 x 64 were never faster (290 and 303 at 573 rows, N = 11264).
  // K up to 256: 32 x 32 tiles until 64 x 64 ones are one a CU.  K = 256, us, as 32 x 32 / 64 x 64 tiles: 64 x 2048 4.8 / 8.2,
  // 300 x 2048 7.7 / 8.6, 128 x 8192 9.4 / 9.0, 1000 x 2048 16.6 / 13.7, 4000 x 2048 56 / 47 (90 TFLOP/s).  With operands straight from
  // L2 into a wave's registers these took 33, 33, 34, 60 and 228 us, as plain fused multiply-adds from LDS 29, 29, 30, 33 and 81.
  const long long few = (long long)((M + 63) / 64) * ((N + 31) / 32), large = (long long)((M + 63) / 64) * ((N + 63) / 64);
  // Through the ring (us, 64 x 32 / 64 x 64, K = 2048): 300 rows, N = 11264 125 / 136, 573 rows 225 / 239, 640 rows 240 / 239, 1000 rows 379 /
  // 372, 2048 rows 808 / 732; 1600 rows, N = 2048 124 / 135, N = 2560 147 / 137: what the fullest CU has to do, a smaller tile 0.53 of
  // a larger one; but not larger tiles that are alone on their CUs (300 rows, N = 2048: 39 / 43).
  const bool larger = through_ring(X, W, K, ldx, ldw) ? large > 256 && 0.53f * static_cast<float>((few + 255) / 256) >= static_cast<float>((large + 255) / 256) : large >= 704;
  if (K <= kShortK) {
    if (large >= 256) launch_tiles<2, 2, FOURS, true>(X, W, Y, M, N, K, ldx, ldw, ldy, s);
    else launch_tiles<1, 1, FOURS, true>(X, W, Y, M, N, K, ldx, ldw, ldy, s);
    return;
  }
  // Up to 32 rows of many columns: tiles of 32 rows, the rows kernel's blocks being short there (a wave has one segment of K).
  // One row / 16 rows, us, rows kernel / 32 x 32 / 32 x 64: K = 512, N = 8192 9.0 / 9.7 / 10.6 and 11.7 / 10.6 / 10.9, N = 20000 21.8 /
  // 13.1 / 14.4 and 27 / 13.5 / 14.7, N = 32000 32 / 15.9 / 14.8 and 41 / 16.5 / 15.4, N = 128000 111 / 49 / 45 and 151 / 52 / 48 (77 and
  // 96 as plain fused multiply-adds); K = 1000, N = 20000 20.7 / 23.0 / 25.6 and 23.6 / 23.7 / 26.1, N = 32000 31 / 28 / 25.6 and 35 /
  // 29 / 26.6; K = 2048, N = 32000 50 / 52 / 46 and 67 / 53 / 48.  A long stream for one row is the rows kernel's: K = 4096, N = 32000,
  // 1 / 8 / 16 / 32 rows, rows kernel (64 x 32 tiles at 32) / 32 x 64: 101 / 116 / 140 / 169 and 120 / 111 / 111 / 114.
  if (M <= 32 && (N + 63) / 64 >= 480 && (M > 4 || K <= 2048)) {
    launch_tiles<1, 2, FOURS, false>(X, W, Y, M, N, K, ldx, ldw, ldy, s);
    return;
  }
  if (M <= 32 && (N + 31) / 32 >= 500 && K <= 768) {
    launch_tiles<1, 1, FOURS, false>(X, W, Y, M, N, K, ldx, ldw, ldy, s);
    return;
  }
  // Up to 8 rows in blocks of 8 columns while those are at most one a CU, one or two rows also from two a CU on; us, 16 columns a workgroup /
  // 8: one row 2048 x 2048 8.3 / 6.2, 2048 x 5632 20.8 / 14.1, 512 x 512 4.7 / 3.8, 11264 x 2048 23.0 / 21.5, 6144 x 4096 28.4 / 22.1, 28672 x 4096 95 / 86;
  // 8 rows 2048 x 2048 9.1 / 7.3, 2048 x 5632 23.5 / 17.5.  In between, and for more rows of many columns, which each block of columns
  // reads again, no: 2560 x 2048 8.2 / 8.4, 8 rows 8192 x 2048 19.2 / 20.9, 28672 x 4096 112 / 120; nor very long K: 4096 x 14336 46.8 / 47.3.
  const int eights = (N + 7) / 8;
  if (M <= 8 && (eights <= 256 || (M <= 2 && eights >= 512 && K <= 8192))) {
    gemm_f32_rows8_kernel<FOURS><<<eights, kSegments / 2 * kWave, 0, s>>>(X, W, Y, M, N, K, ldx, ldw, ldy);
    return;
  }
  if (M <= 16 || few < (M <= 32 ? 600 : 228)) {
    const dim3 grid((N + 15) / 16, M <= 64 ? 1 : (M + 63) / 64);
    if (M <= 16) gemm_f32_rows_kernel<1, FOURS><<<grid, kSegments * kWave, 0, s>>>(X, W, Y, M, N, K, ldx, ldw, ldy);
    else if (M <= 32) gemm_f32_rows_kernel<2, FOURS><<<grid, kSegments * kWave, 0, s>>>(X, W, Y, M, N, K, ldx, ldw, ldy);
    else gemm_f32_rows_kernel<4, FOURS><<<grid, kSegments * kWave, 0, s>>>(X, W, Y, M, N, K, ldx, ldw, ldy);
  } else if (larger) {
    launch_tiles<2, 2, FOURS, false>(X, W, Y, M, N, K, ldx, ldw, ldy, s);
  } else {
    launch_tiles<2, 1, FOURS, false>(X, W, Y, M, N, K, ldx, ldw, ldy, s);
  }
}

}  // namespace kvcm

using namespace kvcm;

extern "C" int kvcm_gemm_f32(const float* X, const float* W, float* Y, int M, int N, int K, int ldx, int ldw,
                             int ldy, hipStream_t s) {
  if (M == 0 || N == 0) return 0;
  KVCM_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_f32: bad sizes M=%d N=%d K=%d", M, N, K);
  KVCM_REQUIRE(ldx >= K && ldw >= K && ldy >= N, "gemm_f32: leading dimensions too small");
  if (K % 4 == 0) launch_gemm_f32<true>(X, W, Y, M, N, K, ldx, ldw, ldy, s);
  else launch_gemm_f32<false>(X, W, Y, M, N, K, ldx, ldw, ldy, s);
  return launch_status("gemm_f32");
}

// Is gate and up in one launch with SwiGLU (kvcm_gemm_f32_swiglu), I columns of K > 256, the faster?  In blocks of 8 columns up to 8 rows
// are no slower than otherwise by more than SwiGLU's launch while the matrix is small (8 rows of 2048 x 8192: 35.8 / 36.0 us; above
// it 8 rows of 4096 x 28672 8 us slower), and not where the other way are tiles of very many columns, or K is very long.
extern "C" int kvcm_gemm_f32_swiglu_preferred(int M, int I, int K) {
  return M >= 1 && M <= 8 && I > 0 && K > kvcm::kShortK && K <= 8192 && K % 4 == 0 && I < 240 * 64 && (M <= 2 || 2ll * I * K <= 60000000);
}

// Y[M, I] = silu(X Wg^T) * (X Wu^T), W = [Wg; Wu]: the bits of kvcm_gemm_f32 and kvcm_swiglu.
extern "C" int kvcm_gemm_f32_swiglu(const float* X, const float* W, float* Y, int M, int I, int K, int ldx, int ldw, int ldy, hipStream_t s) {
  KVCM_REQUIRE(kvcm_gemm_f32_swiglu_preferred(M, I, K), "gemm_f32_swiglu: unsupported shape M=%d I=%d K=%d", M, I, K);
  KVCM_REQUIRE(X && W && Y && ldx >= K && ldw >= K && ldy >= I, "gemm_f32_swiglu: missing operand or leading dimensions too small");
  gemm_f32_rows8_kernel<true, true><<<(I + 3) / 4, kSegments / 2 * kWave, 0, s>>>(X, W, Y, M, I, K, ldx, ldw, ldy);
  return launch_status("gemm_f32_swiglu");
}
