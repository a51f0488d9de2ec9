// The matrix memory with exponential gates (mlstm.hip) for long runs, in matrix form.  With every row's factors keep and take (at most
// one each) S_t = keep_t S_(t-1) + take_t k_t v_t^T, n likewise with k alone; D(i, j) = take_j keep_(j+1) .. keep_i and D(i) = keep_0 .. keep_i of a chunk of 64 rows
// that starts from (S, n) give
//
//   S_i^T q_i = D(i) S^T q_i + sum over j <= i of D(i, j) (q_i . k_j) v_j        n_i . q_i = D(i) n . q_i + sum of D(i, j) (q_i . k_j)
//   S <- D(63) S + sum over j of D(63, j) k_j v_j^T                              n <- D(63) n + sum of D(63, j) k_j
//
// four products in 32 bits on the matrix cores (v_mfma_f32_16x16x4_f32).  The D are made as products of what is at most one, never as
// quotients or differences of logarithms, so that they are as exact as the walk's: D(i, j) of rows 16 w and later with a column before them
// is (keep_(16 w) .. keep_i)(take_j keep_(j+1) .. keep_(16 w - 1)), the sixteen columns of the rows' own are walked.
//
// Runs are taken in pieces, all pieces at once: every piece's own part of (S, n) and the product of its keeps; the states that enter the
// pieces, one after another, element by element; every piece again from the state that enters it, now with outputs.
//
// The walk's time is a token's chain of dependent instructions whatever the chip could do.  Here every unit has some 10 us of work for 2,048 tokens of
// 32 heads of 64 x 64 (matrix instructions 11, the vectors' bytes 11, vector instructions 13, LDS 8), and the workgroups, two a CU, are all in the same
// phase: 42 us for the last launch, 14 for the pieces' own parts, 7 between, 15 for the factors.  us, the walk / so: one sequence of 2,048 tokens 300 / 78 (pieces
// of 64, 128, 256 rows: 84, 78, 90), 8 of 509 228 / 128, 32 heads of 128 x 128 550 / 197, 64 heads of 16 x 16, 1,024 tokens 153 / 61.
// Errors against 64 bits as parts of the walk's (1,024 tokens, 64 heads of 64 and 128, keys and queries with and without a common mean): outputs 0.35 .. 1.0,
// states 0.99 .. 1.01 (both have the factors' own roundings; with the factors' products in 32 bits 1.03 .. 1.16), normalizers 0.90 .. 0.98.
// A workgroup is eight waves on 64 value columns of a head: a row tile of 16 belongs to two waves, which halve its columns.  Key sizes beyond 128
// do not fit LDS, and 32-bit storage, where a row's result must not depend on where its run began, keeps the walk.
#include "common.h"
#include "kvcm_hip.h"
#include "mlstm.h"

namespace kvcm {

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

constexpr int kChunk = 64, kChunkCols = 64, kChunkThreads = 512;

struct ChunkArgs {
  const float *q, *k, *v;
  const float4* coef;
  int ldq, ldk, ldv;
  float q_scale;
  float* o;
  int ldo;
  float *s_state, *n_state;
  const int *run_start, *seq_start, *state_slots;
  int heads, dk, dv, col_blocks;
  float* carry;      // per (piece, head): [dk][dv], [dk], the product of the keeps
  int piece, pieces_per_seq;
};

__host__ __device__ __forceinline__ long long chunk_carry(int dk, int dv) { return static_cast<long long>(dk) * dv + dk + 1; }
// where a piece's part of the carry lies (pieces of all sequences are numbered so that no two meet)
__device__ __forceinline__ size_t chunk_place(const ChunkArgs& A, int run0, int s, int p, int head) {
  return (size_t(run0 / A.piece + s + p) * A.heads + head) * chunk_carry(A.dk, A.dv);
}

// four values from place i on of a row of n that begins at base + row; zero where the row is none of the run's or ends (loads from clamped places, masked afterwards)
template <bool WIDE>
__device__ __forceinline__ float4 row_four(const float* base, int row, int i, int n, bool in) {
  if constexpr (WIDE) {      // (n and i are multiples of four)
    const float4 x = *reinterpret_cast<const float4*>(base + static_cast<unsigned>(row + (i < n ? i : 0)));
    return in && i < n ? x : float4{0.f, 0.f, 0.f, 0.f};
  }
  float x[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float y = base[static_cast<unsigned>(row + (i + e < n ? i + e : 0))];
    x[e] = in && i + e < n ? y : 0.f;
  }
  return float4{x[0], x[1], x[2], x[3]};
}

// lane l: the product of x over lanes l + 1 .. 63
template <typename T>
__device__ __forceinline__ T product_above(T x, int lane) {
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const T y = __shfl_down(x, d, kWave);
    x = lane + d < kWave ? x * y : x;
  }
  const T y = __shfl_down(x, 1, kWave);
  return lane == kWave - 1 ? T(1) : y;
}

__device__ __forceinline__ float first_lane(float x) { return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(x))); }

// lane l: the product of x over lanes of its sixteen up to l
__device__ __forceinline__ float product_up_to(float x, int lane) {
#pragma unroll
  for (int d = 1; d < 16; d <<= 1) {
    const float y = __shfl_up(x, d, 16);
    x = lane % 16 >= d ? x * y : x;
  }
  return x;
}

// PARTS: the first of the three launches (no outputs; the piece's own part of the state and its keeps' product go to the carry)
template <int DKP, bool WIDE, bool PARTS>
__global__ void __launch_bounds__(kChunkThreads, DKP == 64 ? 4 : 2) mlstm_chunk_kernel(ChunkArgs A) {
  constexpr int C = kChunk, DVT = kChunkCols, NT = kChunkThreads, KP = DKP + 4, VP = DVT + 4, PP = C + 4;      // pitches: rows four apart lie 16 banks apart
  constexpr int BT = DKP / 64, CT = DVT / 16 / 2, KS = DKP / 16;
  __shared__ __attribute__((aligned(16))) float Ks[C][KP];
  __shared__ __attribute__((aligned(16))) float Vs[C][VP];
  __shared__ __attribute__((aligned(16))) float Ss[PARTS ? 1 : DKP][VP];
  __shared__ __attribute__((aligned(16))) float Ps[PARTS ? 1 : 4][16][PP];
  __shared__ __attribute__((aligned(16))) float ks[C];      // the rows' keep, take and exp(-m)
  __shared__ float ts[C], ls[C];
  __shared__ float out[C];                   // D(63, j)
  __shared__ __attribute__((aligned(16))) float Ns[DKP];
  __shared__ int odd;      // the chunk whose values are not all finite
  __shared__ float sums[PARTS ? 1 : 2][C], nq[PARTS ? 1 : C];
  const int head = blockIdx.x / A.col_blocks, c0 = (blockIdx.x % A.col_blocks) * DVT;
  const int s = blockIdx.y / A.pieces_per_seq, p = blockIdx.y % A.pieces_per_seq;
  const int tid = threadIdx.x, half = tid / 256, lane = tid % kWave, col = lane % 16, g = lane / 16;
  // (a later row tile has more columns in front of it: the two waves of a SIMD, four numbers apart, take an early and a late one)
  const int wave = half == 0 ? tid / kWave : 7 - tid / kWave;
  const int cw = half * CT * 16;      // where this wave's columns of the stretch start
  const int dk = A.dk, dv = A.dv;
  const int run0 = A.run_start[s], run1 = A.run_start[s + 1], slot = A.state_slots[s];
  const int r0 = run0 + p * A.piece, r1 = run1 - r0 > A.piece ? r0 + A.piece : run1;
  if (r1 <= r0) return;
  const bool last = r1 == run1;
  if (PARTS && (last || slot < 0)) return;      // nothing follows the last piece
  const int cols = dv - c0 < DVT ? dv - c0 : DVT;
  if (slot < 0) {
    for (int e = tid; e < (r1 - r0) * cols; e += NT) A.o[size_t(r0 + e / cols) * A.ldo + size_t(head) * dv + c0 + e % cols] = 0.f;
    return;
  }
  float* part = A.carry + chunk_place(A, run0, s, p, head);
  float* home = A.s_state + (size_t(slot) * A.heads + head) * dk * dv;

  // this wave's part of the state: row tiles of 16 keys by column tiles of 16 values; a lane holds rows 4 g + i of column col
  f32x4 S[BT][CT];
#pragma unroll
  for (int b = 0; b < BT; ++b)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = (wave * BT + b) * 16 + g * 4 + i, c = cw + ct * 16 + col;
        if constexpr (PARTS) {
          S[b][ct][i] = 0.f;
        } else {      // (an unconditional load from a clamped place, masked afterwards)
          S[b][ct][i] = part[static_cast<unsigned>((key < dk ? key : 0) * dv + c0 + (c < cols ? c : 0))];
        }
      }
  if constexpr (!PARTS) {
#pragma unroll
    for (int b = 0; b < BT; ++b)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float x = S[b][ct][i];
          asm volatile("" : "+v"(x));      // (or the compiler puts a branch around the load, and each waits for the one before)
          S[b][ct][i] = (wave * BT + b) * 16 + g * 4 + i < dk && cw + ct * 16 + col < cols ? x : 0.f;
        }
  }
  if (tid < DKP) {
    const float x = PARTS ? 0.f : part[size_t(dk) * dv + (tid < dk ? tid : 0)];
    Ns[tid] = tid < dk ? x : 0.f;
  }
  double kept = 1.;

  constexpr int KQ = C * DKP / 4 / NT, VQ = C * DVT / 4 / NT;
  float4 kreg[KQ], vreg[VQ], qreg[PARTS ? 1 : KS], creg;
  // rows t0 .. t0 + 63 of the piece; what lies outside is zero and keeps the state (32-bit places from the chunk's first row on)
  auto request = [&](int t0) {
    const int rows = r1 - t0;
    const float* kb = A.k + size_t(t0) * A.ldk + size_t(head) * dk;
    const float* vb = A.v + size_t(t0) * A.ldv + size_t(head) * dv + c0;
#pragma unroll
    for (int n = 0; n < KQ; ++n) {
      const int e = tid + n * NT, row = e / (DKP / 4);
      kreg[n] = row_four<WIDE>(kb, (row < rows ? row : rows - 1) * A.ldk, (e % (DKP / 4)) * 4, dk, row < rows);
    }
#pragma unroll
    for (int n = 0; n < VQ; ++n) {
      const int e = tid + n * NT, row = e / (DVT / 4);
      vreg[n] = row_four<WIDE>(vb, (row < rows ? row : rows - 1) * A.ldv, (e % (DVT / 4)) * 4, cols, row < rows);
    }
    if constexpr (!PARTS) {
      const float* qb = A.q + size_t(t0) * A.ldq + size_t(head) * dk;
      const int row = wave * 16 + col;
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) qreg[kk] = row_four<WIDE>(qb, (row < rows ? row : rows - 1) * A.ldq, kk * 16 + g * 4, dk, row < rows);
    }
    const int row = tid % C;
    const float4 c = (A.coef + size_t(t0) * A.heads + head)[static_cast<unsigned>((row < rows ? row : rows - 1) * A.heads)];
    creg = row < rows ? c : float4{1.f, 0.f, 1.f, 0.f};
  };

  if (tid == 0) odd = -1;
  request(r0);
  for (int t0 = r0; t0 < r1; t0 += C) {
    const int n = r1 - t0 < C ? r1 - t0 : C;
    __syncthreads();      // the chunk before is done with everything in LDS
#pragma unroll
    for (int m = 0; m < KQ; ++m) {
      const int e = tid + m * NT;
      *reinterpret_cast<float4*>(&Ks[e / (DKP / 4)][(e % (DKP / 4)) * 4]) = kreg[m];
    }
#pragma unroll
    for (int m = 0; m < VQ; ++m) {
      const int e = tid + m * NT;
      *reinterpret_cast<float4*>(&Vs[e / (DVT / 4)][(e % (DVT / 4)) * 4]) = vreg[m];
      if constexpr (!PARTS) {      // (what is not finite, times nothing, is not nothing)
        const float none = 0.f * ((vreg[m].x + vreg[m].y) + (vreg[m].z + vreg[m].w));
        if (none != 0.f) odd = t0;
      }
    }
    if (tid < C) {
      ks[tid] = creg.x;
      ts[tid] = creg.y;
      ls[tid] = creg.z;
    }
    // (every wave has the factors of all rows, one a lane)
    const double above = product_above(double(creg.x), lane);      // (an error here is every element's of the state: 64 bits)
    if (tid < C) out[tid] = static_cast<float>(creg.y * above);
    const float through = first_lane(static_cast<float>(creg.x * above));      // D(63)
    float4 qf[PARTS ? 1 : KS];
    // keep_0 .. keep_(16 wave - 1); lane j: take_j keep_(j+1) .. keep_(16 wave - 1); lane l: keep_(16 wave) .. keep_(16 wave + l % 16)
    float entered = 1.f, before = 1.f, within = 1.f;
    if constexpr (!PARTS) {
      const float mine = lane < wave * 16 ? creg.x : 1.f, above16 = product_above(mine, lane);
      entered = first_lane(mine * above16);
      before = creg.y * above16;
      within = product_up_to(__shfl(creg.x, wave * 16 + col, kWave), lane);
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) {
        qf[kk] = qreg[kk];
        qf[kk].x *= A.q_scale; qf[kk].y *= A.q_scale; qf[kk].z *= A.q_scale; qf[kk].w *= A.q_scale;
      }
#pragma unroll
      for (int b = 0; b < BT; ++b)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int i = 0; i < 4; ++i) Ss[(wave * BT + b) * 16 + g * 4 + i][cw + ct * 16 + col] = S[b][ct][i];
    }
    __syncthreads();
    if constexpr (PARTS) {
      if (t0 + C < r1) request(t0 + C);      // on its way while this chunk is multiplied
    } else {
      const bool busy = wave * 16 < n;
      float f[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) f[i] = __shfl(within, g * 4 + i, 16);
      f32x4 acc[CT];
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) acc[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (busy) {
        // Q K^T of this wave's rows with the rows up to its own, times D, to LDS as the next product's first operand
        float rowsum[4] = {};
#pragma unroll 1
        for (int jt = half; jt <= wave; jt += 2) {      // (the row tile's other wave makes the others)
          f32x4 P = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int kk = 0; kk < KS; ++kk) {
            const float4 kf = *reinterpret_cast<const float4*>(&Ks[jt * 16 + col][kk * 16 + g * 4]);
            P = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[kk].x, kf.x, P, 0, 0, 0);
            P = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[kk].y, kf.y, P, 0, 0, 0);
            P = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[kk].z, kf.z, P, 0, 0, 0);
            P = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[kk].w, kf.w, P, 0, 0, 0);
          }
          float D[4];
          if (jt < wave) {
            const float tail = __shfl(before, jt * 16 + col, kWave);
#pragma unroll
            for (int i = 0; i < 4; ++i) D[i] = f[i] * tail;
          } else {      // the columns of these rows: a walk down every column, four rows of which are this lane's
            const float take = ts[wave * 16 + col];
            float keeps[16], d = 0.f;
#pragma unroll
            for (int r = 0; r < 16; r += 4) {
              const float4 x = *reinterpret_cast<const float4*>(&ks[wave * 16 + r]);
              keeps[r] = x.x; keeps[r + 1] = x.y; keeps[r + 2] = x.z; keeps[r + 3] = x.w;
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const float on = d * keeps[r];
              d = r == col ? take : on;
              D[r % 4] = r / 4 == g || r < 4 ? d : D[r % 4];
            }
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float x = jt < wave || col <= g * 4 + i ? P[i] * D[i] : 0.f;
            Ps[wave][g * 4 + i][jt * 16 + col] = x;
            rowsum[i] += x;
          }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          rowsum[i] = group_sum<16>(rowsum[i]);
          if (col == 0) sums[half][wave * 16 + g * 4 + i] = rowsum[i];
        }
        if (half == 0) {      // n . q of row 16 wave + col, a quarter of the keys a lane
          float d = 0.f;
#pragma unroll
          for (int kk = 0; kk < KS; ++kk) {
            const float4 nf = *reinterpret_cast<const float4*>(&Ns[kk * 16 + g * 4]);
            d = fmaf(qf[kk].x, nf.x, d); d = fmaf(qf[kk].y, nf.y, d); d = fmaf(qf[kk].z, nf.z, d); d = fmaf(qf[kk].w, nf.w, d);
          }
          d += __shfl_xor(d, 16, kWave);
          d += __shfl_xor(d, 32, kWave);
          if (g == 0) nq[wave * 16 + col] = d;
        }
#pragma unroll
        for (int kk = 0; kk < KS; ++kk) {
          const float qe[4] = {qf[kk].x, qf[kk].y, qf[kk].z, qf[kk].w};
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
              acc[ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(qe[e], Ss[kk * 16 + g * 4 + e][cw + ct * 16 + col], acc[ct], 0, 0, 0);
        }
      }
      __syncthreads();
      if (t0 + C < r1) request(t0 + C);      // (not before q is done with: one set of its registers)
      if (busy) {
        float* ob = A.o + size_t(t0) * A.ldo + size_t(head) * dv + c0;
        float by[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = wave * 16 + g * 4 + i;
          const float d = entered * f[i];
          const float under = fmaf(d, nq[row], sums[0][row] + sums[1][row]);
          by[i] = fmaxf(fabsf(under), ls[row]) + 1e-6f;
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) acc[ct][i] *= d;
        }
        const int whole = __builtin_amdgcn_readfirstlane(odd == t0 ? wave : wave + 1);      // tiles for the matrix cores, which multiply by zeros too
#pragma unroll 1
        for (int jt = 0; jt < whole; ++jt) {
          const float4 pf = *reinterpret_cast<const float4*>(&Ps[wave][col][jt * 16 + g * 4]);
          const float pe[4] = {pf.x, pf.y, pf.z, pf.w};
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
              acc[ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(pe[e], Vs[jt * 16 + g * 4 + e][cw + ct * 16 + col], acc[ct], 0, 0, 0);
        }
        if (whole == wave) {      // rows in front of what is not finite must not see it: the last tile's sums without its zeros
#pragma unroll 1
          for (int j = 0; j < 16; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
              for (int ct = 0; ct < CT; ++ct) {
                const float x = Ps[wave][g * 4 + i][wave * 16 + j] * Vs[wave * 16 + j][cw + ct * 16 + col];
                acc[ct][i] += j <= g * 4 + i ? x : 0.f;
              }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = wave * 16 + g * 4 + i;
          if (row >= n) continue;
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
            if (cw + ct * 16 + col < cols) ob[static_cast<unsigned>(row * A.ldo + cw + ct * 16 + col)] = acc[ct][i] / by[i];
        }
      }
      if (t0 + C >= r1 && !last) break;      // the state that leaves this piece is another piece's business
    }
    kept *= through;
#pragma unroll
    for (int b = 0; b < BT; ++b)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int i = 0; i < 4; ++i) S[b][ct][i] *= through;
    const int tiles = (n + 15) / 16;
    float nsum[BT] = {};
#pragma unroll 1
    for (int jt = 0; jt < tiles; ++jt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = jt * 16 + g * 4 + e;
        const float w = out[j];
        float kf[BT];
#pragma unroll
        for (int b = 0; b < BT; ++b) {
          kf[b] = Ks[j][(wave * BT + b) * 16 + col] * w;
          nsum[b] += kf[b];
        }
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          const float vf = Vs[j][cw + ct * 16 + col];
#pragma unroll
          for (int b = 0; b < BT; ++b) S[b][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[b], vf, S[b][ct], 0, 0, 0);
        }
      }
    if (half == 0) {      // (a key's sixteen belong to one wave; n . q was made in front of the last barrier)
#pragma unroll
      for (int b = 0; b < BT; ++b) {
        float d = nsum[b];
        d += __shfl_xor(d, 16, kWave);
        d += __shfl_xor(d, 32, kWave);
        if (g == 0) Ns[(wave * BT + b) * 16 + col] = fmaf(through, Ns[(wave * BT + b) * 16 + col], d);
      }
    }
  }
  if (PARTS || last) {
    float* dst = PARTS ? part : home;
#pragma unroll
    for (int b = 0; b < BT; ++b)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = (wave * BT + b) * 16 + g * 4 + i, c = cw + ct * 16 + col;
          if (key < dk && c < cols) dst[static_cast<unsigned>(key * dv + c0 + c)] = S[b][ct][i];
        }
    if (c0 == 0) {      // n, and the keeps' product, once
      float* ndst = PARTS ? part + size_t(dk) * dv : A.n_state + (size_t(slot) * A.heads + head) * dk;
      if (half == 0 && g == 0) {
#pragma unroll
        for (int b = 0; b < BT; ++b) {
          const int key = (wave * BT + b) * 16 + col;
          if (key < dk) ndst[key] = Ns[key];      // (this lane wrote it)
        }
      }
      if (PARTS && tid == 0) part[size_t(dk) * dv + dk] = static_cast<float>(kept);
    }
  }
}

// the states that enter a run's pieces, from its slot (or zero): carry[piece] <- (S, n), then (S, n) <- the piece's keeps times (S, n) +
// what the piece had left there.  grid (element blocks, heads, sequences); an element's chain is one thread's.
__global__ void __launch_bounds__(256) mlstm_pass_kernel(ChunkArgs A) {
  const int e = blockIdx.x * 256 + threadIdx.x, head = blockIdx.y, s = blockIdx.z;
  const int run0 = A.run_start[s], len = A.run_start[s + 1] - run0, slot = A.state_slots[s], whole = A.dk * A.dv, size = whole + A.dk;
  if (len <= 0 || slot < 0 || e >= size) return;
  const int n = (len + A.piece - 1) / A.piece;
  const size_t at_head = size_t(slot) * A.heads + head;
  float cur = A.seq_start[s] == 0 ? 0.f : e < whole ? A.s_state[at_head * whole + e] : A.n_state[at_head * A.dk + e - whole];
  float* base = A.carry + chunk_place(A, run0, s, 0, head);
  const size_t stride = size_t(A.heads) * chunk_carry(A.dk, A.dv);
  constexpr int AHEAD = 8;      // parts requested together
  for (int p0 = 0; p0 < n; p0 += AHEAD) {
    float b[AHEAD], keep[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {      // (the last piece left none)
      const float* at = base + (p0 + i + 1 < n ? p0 + i : 0) * stride;
      b[i] = at[e];
      keep[i] = at[size];
    }
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      if (p0 + i >= n) break;
      base[(p0 + i) * stride + e] = cur;
      cur = p0 + i + 1 < n ? fmaf(keep[i], cur, b[i]) : cur;
    }
  }
}

template <int DKP>
static void launch_chunks(const ChunkArgs& A, int S, bool wide, hipStream_t s) {
  const dim3 grid(A.heads * A.col_blocks, S * A.pieces_per_seq);
  if (wide) mlstm_chunk_kernel<DKP, true, true><<<grid, kChunkThreads, 0, s>>>(A);
  else mlstm_chunk_kernel<DKP, false, true><<<grid, kChunkThreads, 0, s>>>(A);
  mlstm_pass_kernel<<<dim3((A.dk * (A.dv + 1) + 255) / 256, A.heads, S), 256, 0, s>>>(A);
  if (wide) mlstm_chunk_kernel<DKP, true, false><<<grid, kChunkThreads, 0, s>>>(A);
  else mlstm_chunk_kernel<DKP, false, false><<<grid, kChunkThreads, 0, s>>>(A);
}

}  // namespace kvcm

using namespace kvcm;

extern "C" {

// floats of scratch for a step of `rows` rows and S sequences in pieces
long long kvcm_mlstm_carry_floats(int rows, int S, int heads, int dk, int dv, int piece) {
  if (piece <= 0 || rows < 0 || S < 0) return 0;
  return (static_cast<long long>(rows) / piece + S + 1) * heads * chunk_carry(dk, dv);
}

// As kvcm_mlstm_scan (all operands alike), in matrix form, for key sizes up to 128: a row's sums are taken in chunks of 64 rows from where its run
// began.  piece (a multiple of 64): rows of a piece, with `carry` as scratch.
int kvcm_mlstm_chunks(const float* q, int ldq, const float* k, int ldk, const float* v, int ldv, const float* ig, int ldi, const float* fg,
                      int ldf, const float* i_bias, const float* f_bias, float cap, float q_scale, float* coef, float* o, int ldo, float* s_state,
                      float* n_state, float* m_state, const int* run_start, const int* seq_start, const int* state_slots, int S, int heads,
                      int dk, int dv, int T, int max_run, int piece, float* carry, long long carry_floats, hipStream_t s) {
  if (S == 0) return 0;
  KVCM_REQUIRE(S > 0 && heads > 0 && dk > 0 && dv > 0 && T > 0 && max_run > 0, "mlstm_chunks: bad sizes S=%d heads=%d dk=%d dv=%d", S, heads, dk, dv);
  KVCM_REQUIRE(dk <= 128, "mlstm_chunks: a key size of %d is not supported (up to 128)", dk);
  KVCM_REQUIRE(dv <= (1 << 22) && ldq < (1 << 24) && ldk < (1 << 24) && ldv < (1 << 24) && ldo < (1 << 24) && heads < (1 << 22), "mlstm_chunks: rows too far apart");
  KVCM_REQUIRE(cap > 0.f, "mlstm_chunks: the gates' cap must be positive (%g)", cap);
  KVCM_REQUIRE(ldq >= heads * dk && ldk >= heads * dk && ldv >= heads * dv && ldo >= heads * dv && ldi >= heads && ldf >= heads,
               "mlstm_chunks: row strides too small");
  KVCM_REQUIRE(coef && reinterpret_cast<uintptr_t>(coef) % 16 == 0, "mlstm_chunks: the scratch must be there, 16-byte aligned");
  KVCM_REQUIRE(piece > 0 && piece % kChunk == 0, "mlstm_chunks: pieces of %d rows are not supported (a multiple of %d)", piece, kChunk);
  KVCM_REQUIRE(carry && carry_floats >= kvcm_mlstm_carry_floats(T, S, heads, dk, dv, piece), "mlstm_chunks: the scratch for the pieces is too small");
  float4* cf = reinterpret_cast<float4*>(coef);
  ChunkArgs A = {q, k, v, cf, ldq, ldk, ldv, q_scale, o, ldo, s_state, n_state, run_start, seq_start, state_slots, heads, dk, dv,
                 (dv + kChunkCols - 1) / kChunkCols, carry, piece, (max_run + piece - 1) / piece};
  KVCM_REQUIRE(static_cast<long long>(S) * A.pieces_per_seq <= 65535 && heads <= 65535 && static_cast<long long>(heads) * A.col_blocks < (1ll << 31),
               "mlstm_chunks: too many sequences and pieces for one launch");
  mlstm_factors(ig, ldi, fg, ldf, i_bias, f_bias, cap, cf, m_state, run_start, seq_start, state_slots, S, heads, T, max_run, 0, static_cast<long long>(S) * heads <= 512, s);
  auto aligned = [](const void* x) { return reinterpret_cast<uintptr_t>(x) % 16 == 0; };
  const bool wide = dk % 4 == 0 && dv % 4 == 0 && ldq % 4 == 0 && ldk % 4 == 0 && ldv % 4 == 0 && aligned(q) && aligned(k) && aligned(v);
  if (dk <= 64) launch_chunks<64>(A, S, wide, s);
  else launch_chunks<128>(A, S, wide, s);
  return launch_status("mlstm_chunks");
}

}  // extern "C"
