// The generalized delta rule (delta_rule.hip) for long runs, in matrix form (a chunk's rank-one updates as one triangular solve and products, as published for
// products of Householder reflections, Bischof and Van Loan's WY form, and for delta rules over sequences).  In a chunk of C rows that starts from S, with W_i = w_0 .. w_i per
// key channel and the rows
//
//   U_i = u_i W_(i-1)    R_i = r_i W_i    K_j = k_j / W_j    A_j = (a u)_j / W_j
//
// u_i^T S_(i-1) is row i of Z = X S + Y, where L = lower(U A^T) without its diagonal and (I + L) [X | Y] = [U | lower(U K^T) V], and
//
//   o = (R - P X) S + (lower(R K^T) V - P Y)        P = lower(R A^T), with its diagonal
//   S <- diag(W) (I - A^T X) S + diag(W) (K^T V - A^T Y)        W = W_(C-1)
//
// Where keys resemble each other the two sums of N = K^T V - A^T Y, of the outputs and of Y's own equations grow with the rows and nearly cancel, which the walk never
// has: it learns v - what the state already says.  So nothing is summed that way: with a factor t_j a row, the one that brings t_j k_j closest to (a u)_j, B_j = t_j K_j - A_j
// and D_j = v_j - t_j Y_j,
//
//   N = diag(W) (K^T D + B^T Y)      lower(R K^T) D + lower(R B^T) Y      row block b of Y: lower(U K^T) D + lower(U B^T) Y of the blocks before, then the block's own inverse
//
// whose terms are as small as what there is to learn.  lower(U K^T), lower(U B^T) and Y are made in 64 bits (v_mfma_f64_16x16x4_f64), and kept in 32; so are the decays' products.
// Everything but the two products with S is made for all chunks at once (delta_chunk_kernel leaves a chunk's M = diag(W) (I - A^T X), its N, its
// Q = R - P X and what its outputs have without S); what is left of the walk is one product of [M; Q] with S a chunk (delta_pass_kernel), in 32 bits on the
// matrix cores (v_mfma_f32_16x16x4_f32) like all the rest.
//
// The quotients: w is exp(-exp(-1/2) sigmoid(.)), so 0.545 < w <= 1, W of 64 rows is above 1e-17 and a factor W_i / W_j of a term that is used is at
// most one and has the relative error of a few roundings.  What lies above the diagonals may be large and is left out by selection.  A value
// that is not finite cannot be: the matrix cores multiply it by the diagonal blocks' zeros, and rows in front of it would see it.  A chunk whose X or Y holds one is
// walked over again row by row (walk_chunk).
//
// Errors against 64 bits as parts of the walk's: keys and values with a common mean of 0 to 5 times their spread, rates of removal around 0.05 to 0.98:
// outputs 0.54 .. 0.86, states 0.64 .. 0.99; in 32 bits, with N and the outputs as the plain differences above, up to 4.2 times the walk's.
// us, walk / so / with those differences: 32 heads of 64 x 64, 2,048 tokens 291 / 152 / 125, 512 72 / 43 / 37, 192 29 / 33 / 26, 3 of 1,024
// 332 / 249 / 196; 32 heads of 128 x 128, 2,048 tokens 711 / 364 / 322, 4 of 1,024 1,328 / 733 / 657.
//
// A workgroup of the first kernel is eight waves, one a CU: four matrices of C rows by the keys and four of C by C in LDS, a wave with 16 columns of
// X or Y in registers throughout, whose accumulators are the next product's second operand as they lie (key 4 g + e of lane group g is element e; the ones of
// 64 bits, 4 e + g, are turned by four swaps of lanes).
#include "common.h"
#include "kvcm_hip.h"

namespace kvcm {

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
typedef __attribute__((__vector_size__(4 * sizeof(double)))) double f64x4;

struct DeltaChunkArgs {
  const float *r, *k, *v, *w, *au, *u;
  int ldr, ldk, ldv;
  float* o;
  int ldo;
  float* state;
  const int *run_start, *seq_start, *state_slots;
  int heads, dk, dv, col_blocks;
  float* carry;      // per (chunk, head): M, N [DKP][DKP], Q [C][DKP] in tiles of 16 x 16
  int first, window, per_group, by_row;      // chunks first .. first + window - 1 of every run; chunks a workgroup takes one after the other
};

__host__ __device__ constexpr int delta_chunk_rows(int dkp) { return dkp == 64 ? 64 : 32; }
__host__ __device__ constexpr long long delta_chunk_floats(int dkp) { return 2ll * dkp * dkp + delta_chunk_rows(dkp) * dkp; }

// Where chunk p of sequence s lies.  By row, a run's chunks begin at its first row / C + s: a run of n rows has at most n / C chunks and a part of one, so
// they never meet, and T / C + S places hold any step.  Scratch for fewer holds `window` chunks of every sequence, and the step goes in turns.
template <int DKP>
__device__ __forceinline__ float* delta_chunk_place(const DeltaChunkArgs& A, int s, int run0, int p, int head) {
  const size_t place = A.by_row ? size_t(run0 / delta_chunk_rows(DKP)) + s + p : size_t(s) * A.window + (p - A.first);
  return A.carry + (place * A.heads + head) * delta_chunk_floats(DKP);
}

// A sum of products a (16 x 16, a row's four values a lane) times b (16 x 16, as an accumulator lies) in four chains, so that 64 terms are added in
// sixteen steps: in one chain the roundings of the partial sums were most of the error.
struct Chains {
  f32x4 v[4] = {};
  __device__ __forceinline__ void add(float4 a, f32x4 b) {
    v[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b[0], v[0], 0, 0, 0);
    v[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b[1], v[1], 0, 0, 0);
    v[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b[2], v[2], 0, 0, 0);
    v[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b[3], v[3], 0, 0, 0);
  }
  // the transpose of what `add` adds
  __device__ __forceinline__ void add_turned(float4 a, f32x4 b) {
    v[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[0], a.x, v[0], 0, 0, 0);
    v[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[1], a.y, v[1], 0, 0, 0);
    v[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[2], a.z, v[2], 0, 0, 0);
    v[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[3], a.w, v[3], 0, 0, 0);
  }
  __device__ __forceinline__ f32x4 sum() const { return (v[0] + v[1]) + (v[2] + v[3]); }
};

// The same in 64 bits, in two chains (an instruction waits long for the one it adds to): an element of lane group g is row 4 e + g of the sum.
struct Chains64 {
  f64x4 v[2] = {};
  __device__ __forceinline__ void add(float4 a, f32x4 b) {
    v[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b[0], v[0], 0, 0, 0);
    v[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b[1], v[1], 0, 0, 0);
    v[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.z, b[2], v[0], 0, 0, 0);
    v[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.w, b[3], v[1], 0, 0, 0);
  }
  __device__ __forceinline__ f64x4 sum() const { return v[0] + v[1]; }
};
// four registers turned over the four lane groups: element e of group g <- element g of group e
__device__ __forceinline__ void turn(uint32_t (&x)[4]) {
  const auto a = __builtin_amdgcn_permlane32_swap(x[0], x[2], false, false), b = __builtin_amdgcn_permlane32_swap(x[1], x[3], false, false);
  const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false), d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  x[0] = c[0]; x[1] = c[1]; x[2] = d[0]; x[3] = d[1];
}
__device__ __forceinline__ void turn(f32x4& v) {
  uint32_t x[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) x[e] = __float_as_uint(v[e]);
  turn(x);
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = __uint_as_float(x[e]);
}
__device__ __forceinline__ void turn(f64x4& v) {
  uint32_t low[4], high[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint64_t bits = __builtin_bit_cast(uint64_t, static_cast<double>(v[e]));
    low[e] = static_cast<uint32_t>(bits);
    high[e] = static_cast<uint32_t>(bits >> 32);
  }
  turn(low);
  turn(high);
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = __builtin_bit_cast(double, uint64_t(high[e]) << 32 | low[e]);
}

constexpr int kDeltaThreads = 512;

// The same M, N, Q and outputs of a chunk by the recurrence itself, started from the identity (M) and from nothing (N): a thread has a column of either
// and keeps it where the next launch reads it.  (About 2 ms a chunk of 64 rows: for chunks that hold what is not finite.)
template <int DKP>
__device__ __forceinline__ void walk_chunk(const DeltaChunkArgs& A, float* part, int head, size_t r0, int n) {
  constexpr int KT = DKP / 16;
  if (threadIdx.x >= 2 * DKP) return;
  const bool of_v = threadIdx.x >= DKP;
  const int x = threadIdx.x % DKP, dk = A.dk;
  const size_t D = size_t(A.heads) * dk, kc = size_t(head) * dk;
  auto m_at = [&](int key) { return (key / 16 * KT + x / 16) * 256 + (x % 16 / 4 * 16 + key % 16) * 4 + x % 4; };
  float* const Q = part + 2 * DKP * DKP;
  float* const column = of_v ? part + DKP * DKP + x / 16 * 256 + x % 16 * 4 : part + m_at(0);
  auto at = [&](int key) -> float& { return column[of_v ? key / 16 * KT * 256 + key % 16 / 4 * 64 + key % 4 : m_at(key) - m_at(0)]; };
  for (int key = 0; key < DKP; ++key) at(key) = !of_v && key == x ? 1.f : 0.f;
  for (int i = 0; i < n; ++i) {
    const size_t row = r0 + i;
    const float *w = A.w + row * D + kc, *u = A.u + row * D + kc, *au = A.au + row * D + kc, *r = A.r + row * A.ldr + kc, *k = A.k + row * A.ldk + kc;
    const float v = of_v && x < A.dv ? A.v[row * A.ldv + size_t(head) * A.dv + x] : 0.f;
    float z = 0.f, o = 0.f;
#pragma unroll 4
    for (int key = 0; key < dk; ++key) z = fmaf(u[key], at(key), z);
#pragma unroll 4
    for (int key = 0; key < dk; ++key) {
      float m = fmaf(w[key], at(key), -au[key] * z);
      if (of_v) m = fmaf(k[key], v, m);
      at(key) = m;
      o = fmaf(r[key], m, o);
    }
    if (!of_v) Q[m_at(i)] = o;
    else if (x < A.dv) A.o[row * A.ldo + size_t(head) * A.dv + x] = o;
  }
}

template <int DKP>
__global__ void __launch_bounds__(kDeltaThreads) delta_chunk_kernel(DeltaChunkArgs A) {
  constexpr int C = delta_chunk_rows(DKP), RT = C / 16, KT = DKP / 16, KP = DKP + 4, PP = C + 4, NW = kDeltaThreads / kWave;
  constexpr int RG = kDeltaThreads / DKP, RPT = C / RG;      // row groups, rows a thread scales
  constexpr bool kBoth = KT == NW;      // every wave has a column tile of X and one of Y; else half of the waves have either
  static_assert(kBoth || 2 * KT == NW, "the column tiles are dealt out to eight waves");
  __shared__ __attribute__((aligned(16))) float Us[C][KP], Rs[C][KP], Ks[C][KP], Bs[C][KP];
  __shared__ __attribute__((aligned(16))) float Ps[4][C][PP];      // U K^T, U B^T, R K^T, R B^T
  __shared__ __attribute__((aligned(16))) float Ds[RT][16][20];      // the inverses of (I + L)'s diagonal blocks
  __shared__ __attribute__((aligned(16))) double Dd[RT][16][18];      // the same in 64 bits, the columns in the order 0, 4, 8, 12, 1, ..
  __shared__ __attribute__((aligned(16))) float ts[2][C];      // the rows' t, of this chunk and the next
  __shared__ int bad;      // the chunk that is not finite
  __shared__ double tot[RG][DKP];
  __shared__ __attribute__((aligned(16))) float Wc[DKP];
  const int head = blockIdx.x, groups = (A.window + A.per_group - 1) / A.per_group;
  const int s = blockIdx.y / groups, p0 = A.first + blockIdx.y % groups * A.per_group;
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave, col = lane % 16, g = lane / 16;
  const int dk = A.dk, dv = A.dv;
  const int run0 = A.run_start[s], run1 = A.run_start[s + 1], slot = A.state_slots[s];
  int p1 = p0 + A.per_group < A.first + A.window ? p0 + A.per_group : A.first + A.window;
  const int all = (run1 - run0 + C - 1) / C;
  if (p1 > all) p1 = all;
  if (p0 >= p1) return;
  if (slot < 0) {      // a padding sequence: its rows carry nothing
    const int r0 = run0 + p0 * C, r1 = run0 + p1 * C < run1 ? run0 + p1 * C : run1;
    for (int e = tid; e < (r1 - r0) * dv; e += kDeltaThreads) A.o[size_t(r0 + e / dv) * A.ldo + size_t(head) * dv + e % dv] = 0.f;
    return;
  }
  const size_t D = size_t(A.heads) * dk;
  const int c = tid % DKP, q = tid / DKP;
  const bool own = c < dk;
  const size_t kc = size_t(head) * dk + (own ? c : 0);
  const bool has_y = kBoth || wave >= KT;
  const int x0 = (wave % KT) * 16;      // this wave's columns, of X and (or) Y
  const bool vown = x0 + col < dv;
  const size_t vc = size_t(head) * dv + (vown ? x0 + col : 0);
  float wr[RPT], ur[RPT], rr[RPT], kr[RPT], ar[RPT];
  f32x4 vr[RT];
  auto request = [&](int p) {      // (rows beyond the run's end are loaded from its last one and masked afterwards)
    const int r0 = run0 + p * C, n = run1 - r0;
    if (n >= C) {
      const size_t row = r0 + q * RPT;
      const float *wp = A.w + row * D + kc, *up = A.u + row * D + kc, *ap = A.au + row * D + kc, *rp = A.r + row * A.ldr + kc, *kp = A.k + row * A.ldk + kc;
#pragma unroll
      for (int m = 0; m < RPT; ++m) {
        wr[m] = wp[m * D];
        ur[m] = up[m * D];
        ar[m] = ap[m * D];
        rr[m] = rp[size_t(m) * A.ldr];
        kr[m] = kp[size_t(m) * A.ldk];
      }
      const float* vp = A.v + size_t(r0 + g * 4) * A.ldv + vc;
      if (has_y) {
#pragma unroll
        for (int b = 0; b < RT; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i) vr[b][i] = vp[size_t(b * 16 + i) * A.ldv];
      }
      return;
    }
#pragma unroll
    for (int m = 0; m < RPT; ++m) {
      const int i = q * RPT + m;
      const size_t row = r0 + (i < n ? i : n - 1);
      wr[m] = A.w[row * D + kc];
      ur[m] = A.u[row * D + kc];
      ar[m] = A.au[row * D + kc];
      rr[m] = A.r[row * A.ldr + kc];
      kr[m] = A.k[row * A.ldk + kc];
    }
    if (has_y) {
#pragma unroll
      for (int b = 0; b < RT; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int j = b * 16 + g * 4 + i;
          vr[b][i] = A.v[size_t(r0 + (j < n ? j : n - 1)) * A.ldv + vc];
        }
    }
  };
  if (tid == 0) bad = -1;
  request(p0);
  for (int p = p0; p < p1; ++p) {
    const int r0 = run0 + p * C, n = run1 - r0 < C ? run1 - r0 : C;
    float* const tr = ts[(p - p0) % 2];      // (the chunk before may still read its own)
    float* part = delta_chunk_place<DKP>(A, s, run0, p, head);
    // the rows' products of w, and the scaled rows
    double cum[RPT], x = 1.0;
#pragma unroll
    for (int m = 0; m < RPT; ++m) {
      x *= own && q * RPT + m < n ? double(wr[m]) : 1.0;
      cum[m] = x;
    }
    tot[q][c] = x;
    if (c < kWave) {      // (this wave's channels, the first 64, are enough for t)
#pragma unroll
      for (int m = 0; m < RPT; ++m) {
        const float kx = own && q * RPT + m < n ? kr[m] : 0.f;
        const float t = wave_sum(kx * ar[m]) / wave_sum(kx * kx);
        if (lane == 0) tr[q * RPT + m] = fabsf(t) < INFINITY ? t : 0.f;      // (any number would do; a row of zeros has none)
      }
    }
    f32x4 vt[RT];      // v, later D
#pragma unroll
    for (int b = 0; b < RT; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) vt[b][i] = has_y && vown && b * 16 + g * 4 + i < n ? vr[b][i] : 0.f;
    __syncthreads();      // (the chunk before is done with everything in LDS but this)
    double entered = 1.0;
    for (int b = 0; b < q; ++b) entered *= tot[b][c];
    if (q == RG - 1) Wc[c] = static_cast<float>(entered * x);
    double before = entered;
#pragma unroll
    for (int m = 0; m < RPT; ++m) {
      const int i = q * RPT + m;
      const bool in = own && i < n;
      const double W = entered * cum[m];
      double inv = __builtin_amdgcn_rcpf(static_cast<float>(W));
      inv = fma(fma(-W, inv, 1.0), inv, inv);
      Us[i][c] = in ? static_cast<float>(ur[m] * before) : 0.f;
      Rs[i][c] = in ? static_cast<float>(rr[m] * W) : 0.f;
      Ks[i][c] = in ? static_cast<float>(kr[m] * inv) : 0.f;
      Bs[i][c] = in ? static_cast<float>((double(tr[i]) * kr[m] - ar[m]) * inv) : 0.f;
      before = W;
    }
    if (p + 1 < p1) request(p + 1);      // on its way while this chunk is multiplied
    __syncthreads();
    // the products of rows with rows, tile t of those up to the diagonal: with K in 64 bits
    constexpr int LT = RT * (RT + 1) / 2;
    auto rows_product = [&](int m, int t) __attribute__((always_inline)) {
      const int bi = t < 1 ? 0 : t < 3 ? 1 : t < 6 ? 2 : 3, bj = t - bi * (bi + 1) / 2;
      const float* left = m < 2 ? &Us[bi * 16 + col][g * 4] : &Rs[bi * 16 + col][g * 4];
      const float* right = m % 2 == 0 ? &Ks[bj * 16 + col][g * 4] : &Bs[bj * 16 + col][g * 4];
      const int above = m < 2 ? 0 : 1;      // the columns of row r that are used are those below r + above
      if (m % 2 == 0) {
        Chains64 sums;
#pragma unroll
        for (int kk = 0; kk < KT; ++kk) {
          const float4 b = *reinterpret_cast<const float4*>(right + kk * 16);
          sums.add(*reinterpret_cast<const float4*>(left + kk * 16), f32x4{b.x, b.y, b.z, b.w});
        }
        const f64x4 acc = sums.sum();
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = 4 * e + g;
          Ps[m][bi * 16 + row][bj * 16 + col] = bj < bi || col < row + above ? static_cast<float>(acc[e]) : 0.f;
        }
      } else {
        Chains sums[2];
#pragma unroll
        for (int kk = 0; kk < KT; ++kk) {
          const float4 a = *reinterpret_cast<const float4*>(left + kk * 16), b = *reinterpret_cast<const float4*>(right + kk * 16);
          sums[kk % 2].add(a, f32x4{b.x, b.y, b.z, b.w});
        }
        const f32x4 acc = sums[0].sum() + sums[1].sum();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = g * 4 + i;
          Ps[m][bi * 16 + row][bj * 16 + col] = bj < bi || col < row + above ? acc[i] : 0.f;
        }
      }
    };
#pragma unroll 1
    for (int n = 0; n * (NW / 2) + wave / 2 < LT; ++n) rows_product((wave + n) % 2, n * (NW / 2) + wave / 2);
    __syncthreads();
    auto four = [&](int m, int bi, int bj) { return *reinterpret_cast<const float4*>(&Ps[m][bi * 16 + col][bj * 16 + g * 4]); };
    // the same of U A^T or R A^T, and of a key column of A
    auto four_a = [&](int m, int bi, int bj) {
      const float4 x = four(m, bi, bj), y = four(m + 1, bi, bj), t = *reinterpret_cast<const float4*>(&tr[bj * 16 + g * 4]);
      return float4{fmaf(x.x, t.x, -y.x), fmaf(x.y, t.y, -y.y), fmaf(x.z, t.z, -y.z), fmaf(x.w, t.w, -y.w)};
    };
    if (wave < RT) {      // (I + L)^-1 of diagonal block `wave`: X in 32 bits, a column a lane (every sixteen lanes make the same), then X + X (1 - (1 + L) X) in 64
      float (*const inverse)[20] = Ds[wave];
      f64x4 l;      // row `col` of L, columns 4 e + g
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int x = 4 * e + g;
        l[e] = fma(double(Ps[0][wave * 16 + col][wave * 16 + x]), double(tr[wave * 16 + x]), -double(Ps[1][wave * 16 + col][wave * 16 + x]));
      }
      float t[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float y = i == col ? 1.f : 0.f;
#pragma unroll
        for (int j = 0; j < i; ++j) {      // (L's element is in another lane: one scalar for all)
          const float x = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(static_cast<float>(l[j / 4])), j % 4 * 16 + i));
          y = fmaf(-x, t[j], y);
        }
        t[i] = y;
      }
      if (g == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) inverse[i][col] = t[i];
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      // (as it lies in a product's sum, a matrix is the second operand of the next one)
      f64x4 left, right, rest;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int x = 4 * e + g;
        left[e] = inverse[col][x];
        right[e] = inverse[x][col];
        rest[e] = (x == col ? 1. : 0.) - right[e];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) rest = __builtin_amdgcn_mfma_f64_16x16x4f64(-l[e], right[e], rest, 0, 0, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e) right = __builtin_amdgcn_mfma_f64_16x16x4f64(left[e], rest[e], right, 0, 0, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e) Dd[wave][4 * e + g][col % 4 * 4 + col / 4] = right[e];
    } else {      // those with R meanwhile
      constexpr int others = (NW - RT) / 2;
      const int w = wave - RT;
#pragma unroll 1
      for (int n = 0; n * others + w / 2 < LT; ++n) rows_product(2 + (w + n) % 2, n * others + w / 2);
    }
    __syncthreads();
    auto column = [&](const float (&m)[C][KP], int b, int t) {      // four rows of a key column: the first operand of a product with m^T
      const float* at = &m[b * 16 + g * 4][t * 16 + col];
      return float4{at[0], at[KP], at[2 * KP], at[3 * KP]};
    };
    // row tile t of this wave's columns of M, N or Q: 16 x 16 as the next launch's lanes take them
    auto place = [&](float* m, int t) -> float4& { return *reinterpret_cast<float4*>(m + (t * KT + x0 / 16) * 256 + lane * 4); };
    bool odd = false;      // (what is not finite, times nothing, is not nothing)
    if (has_y) {
      f32x4 y[RT];
#pragma unroll
      for (int b = 0; b < RT; ++b) {
        Chains64 own;
        own.add(four(0, b, b), vt[b]);
        f64x4 rhs = own.sum();
        if (b > 0) {      // (terms as small as what there is to learn: 32 bits are enough)
          Chains learnt, left;
#pragma unroll
          for (int a = 0; a < b; ++a) {
            learnt.add(four(0, b, a), vt[a]);
            left.add(four(1, b, a), y[a]);
          }
          f32x4 before = learnt.sum() + left.sum();
          turn(before);
#pragma unroll
          for (int e = 0; e < 4; ++e) rhs[e] += before[e];
        }
        const double* inverse = &Dd[b][col][g * 4];
        f64x4 z = {0., 0., 0., 0.}, w = {0., 0., 0., 0.};
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
          z = __builtin_amdgcn_mfma_f64_16x16x4f64(inverse[e], rhs[e], z, 0, 0, 0);
          w = __builtin_amdgcn_mfma_f64_16x16x4f64(inverse[e + 1], rhs[e + 1], w, 0, 0, 0);
        }
        z += w;
        turn(z);
        const float4 t = *reinterpret_cast<const float4*>(&tr[b * 16 + g * 4]);
        const float te[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          y[b][e] = static_cast<float>(z[e]);
          vt[b][e] = static_cast<float>(fma(-double(te[e]), z[e], double(vt[b][e])));
        }
        const f32x4 none = 0.f * y[b] + 0.f * vt[b];
        odd |= __any((none[0] + none[1]) + (none[2] + none[3]) != 0.f);
      }
      float* N = part + DKP * DKP;
#pragma unroll 1
      for (int t = 0; t < KT; ++t) {
        Chains learnt, left;
#pragma unroll
        for (int b = 0; b < RT; ++b) {
          learnt.add(column(Ks, b, t), vt[b]);
          left.add(column(Bs, b, t), y[b]);
        }
        const f32x4 acc = learnt.sum() + left.sum();
        const float4 through = *reinterpret_cast<const float4*>(&Wc[t * 16 + g * 4]);
        place(N, t) = float4{through.x * acc[0], through.y * acc[1], through.z * acc[2], through.w * acc[3]};
      }
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        Chains learnt, left;
#pragma unroll
        for (int b = 0; b <= t; ++b) {
          learnt.add(four(2, t, b), vt[b]);
          left.add(four(3, t, b), y[b]);
        }
        const f32x4 acc = learnt.sum() + left.sum();
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (vown && t * 16 + g * 4 + i < n) A.o[size_t(r0 + t * 16 + g * 4 + i) * A.ldo + vc] = acc[i];
      }
    }
    if (kBoth || !has_y) {
      f32x4 x[RT];      // -X, block by block
#pragma unroll
      for (int b = 0; b < RT; ++b) {
#pragma unroll
        for (int i = 0; i < 4; ++i) x[b][i] = Us[b * 16 + g * 4 + i][x0 + col];
        if (b > 0) {
          Chains sums;
#pragma unroll
          for (int a = 0; a < b; ++a) sums.add(four_a(0, b, a), x[a]);
          x[b] += sums.sum();
        }
        Chains y;
        y.add(*reinterpret_cast<const float4*>(&Ds[b][col][g * 4]), x[b]);
        x[b] = -y.sum();
        const f32x4 none = 0.f * x[b];
        odd |= __any((none[0] + none[1]) + (none[2] + none[3]) != 0.f);
      }
#pragma unroll 1
      for (int t = 0; t < KT; ++t) {
        Chains sums;
#pragma unroll
        for (int b = 0; b < RT; ++b) {
          const float4 k = column(Ks, b, t), y = column(Bs, b, t), f = *reinterpret_cast<const float4*>(&tr[b * 16 + g * 4]);
          sums.add_turned(float4{fmaf(k.x, f.x, -y.x), fmaf(k.y, f.y, -y.y), fmaf(k.z, f.z, -y.z), fmaf(k.w, f.w, -y.w)}, x[b]);
        }
        const f32x4 acc = sums.sum();
        const int key = t * 16 + col, at = x0 + g * 4;
        const float through = Wc[key];
        place(part, t) = float4{through * (key == at ? 1.f + acc[0] : acc[0]), through * (key == at + 1 ? 1.f + acc[1] : acc[1]),
                                through * (key == at + 2 ? 1.f + acc[2] : acc[2]), through * (key == at + 3 ? 1.f + acc[3] : acc[3])};
      }
      float* Q = part + 2 * DKP * DKP;
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        Chains sums;
#pragma unroll
        for (int b = 0; b <= t; ++b) sums.add_turned(four_a(2, t, b), x[b]);
        const f32x4 acc = sums.sum();
        const float4 own = *reinterpret_cast<const float4*>(&Rs[t * 16 + col][x0 + g * 4]);
        place(Q, t) = float4{own.x + acc[0], own.y + acc[1], own.z + acc[2], own.w + acc[3]};
      }
    }
    if (odd && lane == 0) bad = p;
    __syncthreads();
    if (bad == p) walk_chunk<DKP>(A, delta_chunk_place<DKP>(A, s, run0, p, head), head, run0 + p * C, n);
  }
}

// The states that enter a run's chunks, one after the other, and the outputs' part of them: a workgroup has 16 value columns of a head, a wave a row
// tile of M or of Q.  The state lies in LDS, column by column, in two buffers; the chunks' matrices are on their way kAhead chunks before their use.
template <int DKP>
__global__ void __launch_bounds__((DKP + delta_chunk_rows(DKP)) / 16 * kWave) delta_pass_kernel(DeltaChunkArgs A) {
  constexpr int C = delta_chunk_rows(DKP), KT = DKP / 16, SP = DKP + 4, NT = (DKP + C) / 16 * kWave, kAhead = DKP == 64 ? 4 : 2;
  __shared__ __attribute__((aligned(16))) float Ss[2][16][SP];
  int head, c0;
  head_and_columns(A.heads, A.col_blocks, head, c0);      // (a head's workgroups on one XCD: they read the same M and Q)
  c0 *= 16;
  const int s = blockIdx.y;
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave, col = lane % 16, g = lane / 16;
  const int dk = A.dk, dv = A.dv;
  const int run0 = A.run_start[s], run1 = A.run_start[s + 1], slot = A.state_slots[s];
  if (run1 - run0 <= A.first * C || slot < 0) return;
  const int all = (run1 - run0 + C - 1) / C, end = A.first + A.window < all ? A.first + A.window : all;
  float* home = A.state + (size_t(slot) * A.heads + head) * dk * dv;
  const bool fresh = A.first == 0 && A.seq_start[s] == 0;
  for (int e = tid; e < DKP * 16; e += NT) {
    const int key = e / 16, cc = e % 16;
    Ss[0][cc][key] = !fresh && key < dk && c0 + cc < dv ? home[size_t(key) * dv + c0 + cc] : 0.f;
  }
  const bool keeps = wave < KT;      // a row tile of M, or of Q
  const int tile = keeps ? wave : wave - KT;
  const bool cown = c0 + col < dv;
  const size_t oc = size_t(head) * dv + (cown ? c0 + col : 0);
  float4 m[kAhead][KT];
  f32x4 add[kAhead];
  auto request = [&](int p, int into) {
    const float* part = delta_chunk_place<DKP>(A, s, run0, p, head);
    const float* rows = (keeps ? part : part + 2 * DKP * DKP) + tile * KT * 256 + lane * 4;
#pragma unroll
    for (int kk = 0; kk < KT; ++kk) m[into][kk] = *reinterpret_cast<const float4*>(rows + kk * 256);
    const int r0 = run0 + p * C, n = run1 - r0;
    if (keeps) {
      const float4 x = *reinterpret_cast<const float4*>(part + DKP * DKP + (tile * KT + c0 / 16) * 256 + lane * 4);
      add[into] = f32x4{x.x, x.y, x.z, x.w};
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = tile * 16 + g * 4 + i;
        add[into][i] = A.o[size_t(r0 + (row < n ? row : n - 1)) * A.ldo + oc];
      }
    }
  };
#pragma unroll
  for (int a = 0; a < kAhead; ++a)
    if (A.first + a < end) request(A.first + a, a);
  int at = 0;
  __syncthreads();
  for (int pb = A.first; pb < end; pb += kAhead) {
#pragma unroll
    for (int a = 0; a < kAhead; ++a) {
      const int p = pb + a;
      if (p >= end) break;
      Chains sums[2];
#pragma unroll
      for (int kk = 0; kk < KT; ++kk) {
        const float4 b = *reinterpret_cast<const float4*>(&Ss[at][col][kk * 16 + g * 4]);
        sums[kk % 2].add(m[a][kk], f32x4{b.x, b.y, b.z, b.w});
      }
      const f32x4 acc = add[a] + (sums[0].sum() + sums[1].sum());
      if (p + kAhead < end) request(p + kAhead, a);
      if (keeps) {
        *reinterpret_cast<float4*>(&Ss[at ^ 1][col][tile * 16 + g * 4]) = float4{acc[0], acc[1], acc[2], acc[3]};
      } else {
        const int r0 = run0 + p * C, n = run1 - r0;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (cown && tile * 16 + g * 4 + i < n) A.o[size_t(r0 + tile * 16 + g * 4 + i) * A.ldo + oc] = acc[i];
      }
      at ^= 1;
      __syncthreads();
    }
  }
  for (int e = tid; e < DKP * 16; e += NT) {
    const int key = e / 16, cc = e % 16;
    if (key < dk && c0 + cc < dv) home[size_t(key) * dv + c0 + cc] = Ss[at][cc][key];
  }
}

template <int DKP>
static int launch_delta_chunks(DeltaChunkArgs A, int S, int T, int max_run, long long carry_floats, hipStream_t s) {
  constexpr int C = delta_chunk_rows(DKP);
  const int chunks = (max_run + C - 1) / C;
  const long long place = A.heads * delta_chunk_floats(DKP), rows = T / C + S;      // (the chunks that a step of T rows has at most)
  const long long fit = carry_floats / (S * place);      // of every sequence
  KVCM_REQUIRE(fit >= 1, "delta_chunks: the scratch is too small");
  A.by_row = carry_floats / place >= rows;
  A.window = static_cast<int>(A.by_row || chunks < fit ? chunks : fit);
  // one workgroup a CU: some chunks in a row, whose rows are asked for while the one before is multiplied, once there is more than one a CU
  const long long most = static_cast<long long>(S) * A.window;
  const long long turns = (A.heads * (most < rows ? most : rows) + 255) / 256;
  A.per_group = static_cast<int>(turns < 8 ? turns : 8);
  const int limit = 65535 / S * A.per_group;
  if (A.window > limit) A.window = limit;
  const long long groups = static_cast<long long>(S) * ((A.window + A.per_group - 1) / A.per_group);
  for (A.first = 0; A.first < chunks; A.first += A.window) {
    delta_chunk_kernel<DKP><<<dim3(A.heads, static_cast<unsigned>(groups)), kDeltaThreads, 0, s>>>(A);
    delta_pass_kernel<DKP><<<dim3(A.heads * A.col_blocks, S), (DKP + C) / 16 * kWave, 0, s>>>(A);
  }
  return launch_status("delta_chunks");
}

}  // namespace kvcm

using namespace kvcm;

extern "C" {

// floats of scratch that a step of S sequences and runs of up to max_run rows takes at once (with less, down to a chunk of every sequence, it goes in turns)
long long kvcm_delta_carry_floats(int S, int max_run, int heads, int dk) {
  if (S <= 0 || max_run <= 0 || heads <= 0) return 0;
  const int dkp = dk <= 64 ? 64 : 128, rows = delta_chunk_rows(dkp);
  return static_cast<long long>(S) * ((max_run + rows - 1) / rows) * heads * delta_chunk_floats(dkp);
}

// As kvcm_delta_scan (all operands alike), in matrix form, for key sizes up to 128, values no larger than the keys' tile (64 or 128), and w no smaller
// than exp(-exp(-1/2)), as kvcm_delta_prepare makes it.
int kvcm_delta_chunks(const float* r, int ldr, const float* k, int ldk, const float* v, int ldv, const float* w, const float* au, const float* u,
                      float* o, int ldo, float* state, const int* run_start, const int* seq_start, const int* state_slots, int S, int heads,
                      int dk, int dv, int T, int max_run, float* carry, long long carry_floats, hipStream_t s) {
  if (S == 0) return 0;
  KVCM_REQUIRE(S > 0 && heads > 0 && dk > 0 && dv > 0 && T > 0 && max_run > 0, "delta_chunks: bad sizes S=%d heads=%d dk=%d dv=%d", S, heads, dk, dv);
  KVCM_REQUIRE(dk <= 128 && dv <= (dk <= 64 ? 64 : 128), "delta_chunks: heads of %d x %d are not supported", dk, dv);
  KVCM_REQUIRE(S <= 65535 && heads <= (1 << 20), "delta_chunks: too many sequences or heads for one launch");
  KVCM_REQUIRE(ldr >= heads * dk && ldk >= heads * dk && ldv >= heads * dv && ldo >= heads * dv, "delta_chunks: row strides too small");
  KVCM_REQUIRE(carry && reinterpret_cast<uintptr_t>(carry) % 16 == 0, "delta_chunks: the scratch must be there, 16-byte aligned");
  DeltaChunkArgs A = {r, k, v, w, au, u, ldr, ldk, ldv, o, ldo, state, run_start, seq_start, state_slots, heads, dk, dv, (dv + 15) / 16, carry, 0, 0, 0, 0};
  if (dk <= 64) return launch_delta_chunks<64>(A, S, T, max_run, carry_floats, s);
  return launch_delta_chunks<128>(A, S, T, max_run, carry_floats, s);
}

}  // extern "C"
