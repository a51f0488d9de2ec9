// A matrix memory with exponential gates (the mLSTM cell): per head a state S [dk, dv], a normalizer n [dk] and
// a running maximum m of the gates' logarithms, which keeps every exponential at or below one:
//
//   li = cap * tanh((i_lin + i_bias) / cap)                      log of the input gate
//   lf = logsigmoid(cap * tanh((f_lin + f_bias) / cap))          log of the forget gate
//   m' = max(lf + m, li)
//   S' = exp(lf + m - m') S + exp(li - m') k v^T        n' = exp(lf + m - m') n + exp(li - m') k
//   o  = S'^T q / (max(|n' . q|, exp(-m')) + 1e-6)               q comes scaled by q_scale
//
// S, n and m start at zero (m at 0, not at minus infinity), are 32-bit and live in the request's state slot.
// A run is walked token by token, in prompts and in decoding.  Only m_t = max(lf_t + m_(t-1), li_t) has to go first: a launch
// with one wave per (sequence, head) scans it 64 tokens at a time (the step (lf, li): m -> max(m + lf, li) composes; in 32-bit
// storage, where a row's result depends on that row alone, it takes them one by one) and leaves every row's three factors (for runs of 16 rows or more the two logarithms of all rows are made before that, in parallel).
// The main walk needs no transcendental function.  A value column j of S needs nothing of another column, so columns are spread
// over lanes and waves, the key dimension of a column over G lanes; every wave carries n along beside its columns (n is a
// column of S whose value is always one) and sums n . q like any column's output.  What bounds the walk is a token's chain of
// dependent instructions, so a wave has few columns and a workgroup is one wave: nothing is shared and nobody waits.  The
// per-token vectors go from L2 into the lanes that use them, a few tokens ahead.  All waves of a head read the old n from the
// slot; the first one leaves the new n in scratch, and a small launch moves it to the slot afterwards, so that no wave reads a
// state that another one of the same launch writes.
#include "common.h"
#include "kvcm_hip.h"
#include "mlstm.h"

namespace kvcm {

__device__ __forceinline__ float soft_cap(float z, float cap) { return cap * tanhf(z / cap); }
__device__ __forceinline__ float log_sigmoid(float z) { return z >= 0.f ? -log1pf(expf(-z)) : z - log1pf(expf(z)); }

// For steps with long runs the gates' logarithms of all rows are made first, in parallel: coef[row, head] = (li, lf, ., .).
__global__ void __launch_bounds__(256)
    mlstm_gate_logs_kernel(const float* __restrict__ ig, int ldi, const float* __restrict__ fg, int ldf,
                           const float* __restrict__ i_bias, const float* __restrict__ f_bias, float cap,
                           float4* __restrict__ coef, long long n, int heads) {
  const long long idx = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
  if (idx >= n) return;
  const long long row = idx / heads;
  const int head = static_cast<int>(idx % heads);
  coef[idx] = float4{soft_cap(ig[row * ldi + head] + i_bias[head], cap), log_sigmoid(soft_cap(fg[row * ldf + head] + f_bias[head], cap)),
                     0.f, 0.f};
}

__device__ __forceinline__ float lane_of(float v, int lane) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), lane)); }

// one wave per (sequence, head): coef[row, head] = (exp(lf + m before - m), exp(li - m), exp(-m), .) for every row of the run;
// the slot's m is read at the start (a run that starts at position 0 starts from 0) and written at the end.  IN_ORDER: token by
// token, so that a row's factors do not depend on where its run began; 2,048 tokens: 56 us, as a scan 27 us.
template <bool IN_ORDER>
__global__ void __launch_bounds__(kWave)
    mlstm_max_kernel(const float* __restrict__ ig, int ldi, const float* __restrict__ fg, int ldf,
                     const float* __restrict__ i_bias, const float* __restrict__ f_bias, float cap, float4* __restrict__ coef,
                     float* __restrict__ m_state, const int* __restrict__ run_start, const int* __restrict__ seq_start,
                     const int* __restrict__ state_slots, int heads, int logs_ready) {
  const int s = blockIdx.x / heads, head = blockIdx.x % heads, lane = threadIdx.x;
  const int r0 = run_start[s], r1 = run_start[s + 1];
  const int slot = state_slots[s];
  if (r1 <= r0) return;
  if (slot < 0) {
    for (int row = r0 + lane; row < r1; row += kWave) coef[size_t(row) * heads + head] = float4{0.f, 0.f, 0.f, 0.f};
    return;
  }
  float* mst = m_state + size_t(slot) * heads + head;
  float m = seq_start[s] == 0 ? 0.f : *mst;
  const float ib = i_bias[head], fb = f_bias[head];
  auto request = [&](int t0) {
    const int row = t0 + lane < r1 ? t0 + lane : r1 - 1;
    float4 c;
    if (logs_ready) {
      c = coef[size_t(row) * heads + head];
    } else {
      c.x = soft_cap(ig[size_t(row) * ldi + head] + ib, cap);
      c.y = log_sigmoid(soft_cap(fg[size_t(row) * ldf + head] + fb, cap));
    }
    return c;
  };
  float4 next = request(r0);
  for (int t0 = r0; t0 < r1; t0 += kWave) {
    const bool in = t0 + lane < r1;
    const float li = in ? next.x : -INFINITY, lf = in ? next.y : 0.f;      // (beyond the run: m stays)
    if (t0 + kWave < r1) next = request(t0 + kWave);
    float before, after;
    if constexpr (IN_ORDER) {
      const int n = r1 - t0 < kWave ? r1 - t0 : kWave;
      const float entered = m;
      after = m;
      auto token = [&](int t) {
        m = fmaxf(lane_of(lf, t) + m, lane_of(li, t));
        after = lane == t ? m : after;
      };
      if (n == kWave) {
#pragma unroll
        for (int t = 0; t < kWave; ++t) token(t);
      } else {
        for (int t = 0; t < n; ++t) token(t);
      }
      before = __shfl_up(after, 1, kWave);
      before = lane == 0 ? entered : before;
    } else {
      float a = lf, b = li;      // the steps up to this token together: m -> max(m + a, b)
#pragma unroll
      for (int d = 1; d < kWave; d <<= 1) {
        const float pa = __shfl_up(a, d, kWave), pb = __shfl_up(b, d, kWave);
        if (lane >= d) {
          b = fmaxf(pb + a, b);
          a += pa;
        }
      }
      after = fmaxf(m + a, b);
      before = __shfl_up(after, 1, kWave);
      before = lane == 0 ? m : before;
      m = __shfl(after, kWave - 1, kWave);
    }
    if (in) coef[size_t(t0 + lane) * heads + head] = float4{expf(lf + before - after), expf(li - after), expf(-after), 0.f};
  }
  if (lane == 0) *mst = m;
}

// The same for long runs, whose scan is a chain of tiles of 64 rows (0.85 us each): kMaxWaves waves take a stretch of the run each, put its steps
// together first (m -> max(m + a, b), as the scan's), and scan it from the maximum that enters it.  2,048 rows of 32 heads: 27 us with one
// wave, 9 us so.  Not for many runs (32 of 256 rows and 64 heads: 20 us with one wave, 26 so), and not in front of a walk of several: its workgroups of one
// wave come to lie otherwise after it (32 heads of 128 x 128, 1,024 rows beside 7 single tokens, the walk after one wave 279 us, after this 322).
constexpr int kMaxWaves = 8;
__global__ void __launch_bounds__(kMaxWaves* kWave)
    mlstm_max_stretches_kernel(float4* __restrict__ coef, float* __restrict__ m_state, const int* __restrict__ run_start,
                               const int* __restrict__ seq_start, const int* __restrict__ state_slots, int heads) {
  __shared__ float whole_a[kMaxWaves], whole_b[kMaxWaves];
  const int s = blockIdx.x / heads, head = blockIdx.x % heads, lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int r0 = run_start[s], r1 = run_start[s + 1];
  const int slot = state_slots[s];
  if (r1 <= r0) return;
  if (slot < 0) {
    for (int row = r0 + static_cast<int>(threadIdx.x); row < r1; row += kMaxWaves * kWave) coef[size_t(row) * heads + head] = float4{0.f, 0.f, 0.f, 0.f};
    return;
  }
  float* mst = m_state + size_t(slot) * heads + head;
  float m = seq_start[s] == 0 ? 0.f : *mst;
  const int tiles = (r1 - r0 + kWave - 1) / kWave, per = (tiles + kMaxWaves - 1) / kMaxWaves;
  const int first = wave * per, last = first + per < tiles ? first + per : tiles;
  auto request = [&](int tile) {
    const int row = r0 + tile * kWave + lane;
    return coef[size_t(row < r1 ? row : r1 - 1) * heads + head];
  };
  // a, b: the steps up to this lane's token together (beyond the run: m stays)
  auto scanned = [&](int tile, const float4& c, float& a, float& b) {
    const bool in = r0 + tile * kWave + lane < r1;
    b = in ? c.x : -INFINITY;
    a = in ? c.y : 0.f;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const float pa = __shfl_up(a, d, kWave), pb = __shfl_up(b, d, kWave);
      if (lane >= d) {
        b = fmaxf(pb + a, b);
        a += pa;
      }
    }
  };
  float all_a = 0.f, all_b = -INFINITY;
  if (first < last && wave + 1 < kMaxWaves) {
    float4 next = request(first);
    for (int t = first; t < last; ++t) {
      const float4 c = next;
      if (t + 1 < last) next = request(t + 1);
      float a, b;
      scanned(t, c, a, b);
      a = lane_of(a, kWave - 1);
      b = lane_of(b, kWave - 1);
      all_b = fmaxf(all_b + a, b);
      all_a += a;
    }
  }
  if (lane == 0) {
    whole_a[wave] = all_a;
    whole_b[wave] = all_b;
  }
  __syncthreads();      // (everybody has read the slot's m)
  for (int w = 0; w < wave; ++w) m = fmaxf(m + whole_a[w], whole_b[w]);
  if (first >= last) return;
  float4 next = request(first);
  for (int t = first; t < last; ++t) {
    const float4 c = next;
    if (t + 1 < last) next = request(t + 1);
    const int row = r0 + t * kWave + lane;
    float a, b;
    scanned(t, c, a, b);
    const float after = fmaxf(m + a, b);
    float before = __shfl_up(after, 1, kWave);
    before = lane == 0 ? m : before;
    m = __shfl(after, kWave - 1, kWave);
    if (row < r1) coef[size_t(row) * heads + head] = float4{expf(c.y + before - after), expf(c.x - after), expf(-after), 0.f};
  }
  if (last == tiles && lane == 0) *mst = m;
}

// A wave owns 64 / G * NC value columns of one head of one sequence (NC a lane); U tokens' vectors are in registers or on their way.  Runs of a
// few tokens are bound by the state's own bytes: they take workgroups of 32 columns (whole lines of the state's rows).
// One sequence of 2,048 tokens, 32 heads of 64 x 64: 819 us with workgroups of 256 threads that staged the vectors through LDS
// (64 workgroups on 256 CUs), 292 us here; the maxima 214 us as one lane's chain, 27 us as a scan.
template <int DKP, int G, int NC, int U, int NT, int HOW>
__global__ void __launch_bounds__(NT)
    mlstm_scan_kernel(const float* __restrict__ q, int ldq, const float* __restrict__ k, int ldk, const float* __restrict__ v,
                      int ldv, const float4* __restrict__ coef, float q_scale, float* __restrict__ o, int ldo,
                      float* __restrict__ s_state, const float* __restrict__ n_state, float* __restrict__ n_new,
                      const int* __restrict__ run_start, const int* __restrict__ seq_start,
                      const int* __restrict__ state_slots, int heads, int dk, int dv, int col_blocks) {
  constexpr int IPT = DKP / G, LC = NT / G, CB = LC * NC, Q = IPT / 4;      // LC columns apart: a lane's NC columns
  int head, cb;
  head_and_columns(heads, col_blocks, head, cb);
  const int s = blockIdx.y;
  const int g = threadIdx.x % G, j0 = cb * CB + threadIdx.x / G;
  const int r0 = run_start[s], r1 = run_start[s + 1];
  const int slot = state_slots[s];
  if (r1 <= r0) return;
  bool owns[NC];
  int j[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    owns[c] = j0 + c * LC < dv;
    j[c] = owns[c] ? j0 + c * LC : 0;
  }
  if (slot < 0) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
      if (owns[c] && g == 0)
        for (int row = r0; row < r1; ++row) o[size_t(row) * ldo + size_t(head) * dv + j[c]] = 0.f;
    return;
  }
  float* st = s_state + ((size_t(slot) * heads + head) * dk) * dv;      // [slot][head][i][j]
  const float* nst = n_state + (size_t(slot) * heads + head) * dk;
  const bool fresh = seq_start[s] == 0;
  float S[NC][IPT], N[IPT];
#pragma unroll
  for (int il = 0; il < IPT; ++il) {
    const int from = g * IPT + il / 4 * 4, i = entry_place<HOW>(from, il % 4, dk);
    const bool own = entry_own<HOW>(from, il % 4, dk) && !fresh;      // (what is not takes part from zero and is left out of sums and stores)
#pragma unroll
    for (int c = 0; c < NC; ++c) S[c][il] = (own && owns[c]) ? st[size_t(i) * dv + j[c]] : 0.f;
    N[il] = own ? nst[i] : 0.f;
  }
  static_assert(U <= G, "lane n of a column keeps token n's sums until the U tokens are stored together");
  const size_t col = size_t(head) * dk;
  const float *qp = q + size_t(r0) * ldq + col, *kp = k + size_t(r0) * ldk + col, *vp = v + size_t(r0) * ldv + size_t(head) * dv;
  const float4* cp = coef + size_t(r0) * heads + head;
  float* op = o + size_t(r0 + g) * ldo + size_t(head) * dv;
  float4 qv[U][Q], kv[U][Q], cf[U];
  float vv[U][NC];
  auto request = [&](int n) {      // the next row
#pragma unroll
    for (int p = 0; p < Q; ++p) {
      const int i = g * IPT + 4 * p;
      kv[n][p] = load_four<HOW>(kp, i, dk);
      qv[n][p] = load_own<HOW>(qp, i, dk);      // (what is not own is left out of the sums)
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) vv[n][c] = vp[j[c]];
    cf[n] = *cp;
    kp += ldk; qp += ldq; vp += ldv; cp += heads;
  };
  float over[NC] = {}, under = 0.f, least = 0.f;
  auto walk = [&](int n) {
    const float keep = cf[n].x, take = cf[n].y;
    float vj[NC], acc[NC] = {}, nq = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c) vj[c] = take * vv[n][c];
#pragma unroll
    for (int p = 0; p < Q; ++p) {
      const float ke[4] = {kv[n][p].x, kv[n][p].y, kv[n][p].z, kv[n][p].w}, qe[4] = {qv[n][p].x, qv[n][p].y, qv[n][p].z, qv[n][p].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int il = 4 * p + e;
        const float qd = qe[e] * q_scale;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          S[c][il] = fmaf(keep, S[c][il], ke[e] * vj[c]);
          acc[c] = fmaf(S[c][il], qd, acc[c]);
        }
        N[il] = fmaf(keep, N[il], take * ke[e]);
        nq = fmaf(N[il], qd, nq);
      }
    }
    nq = group_sum<G>(nq);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      acc[c] = group_sum<G>(acc[c]);
      over[c] = g == n ? acc[c] : over[c];
    }
    under = g == n ? nq : under;
    least = g == n ? cf[n].z : least;
  };
  auto store = [&]() {
    const float by = fmaxf(fabsf(under), least) + 1e-6f;
#pragma unroll
    for (int c = 0; c < NC; ++c)
      if (owns[c]) op[j[c]] = over[c] / by;
  };
#pragma unroll
  for (int n = 0; n < U; ++n)
    if (r0 + n < r1) request(n);
  int t0 = r0;
  for (; t0 + 2 * U <= r1; t0 += U, op += size_t(U) * ldo) {
#pragma unroll
    for (int n = 0; n < U; ++n) {
      walk(n);
      request(n);
      __builtin_amdgcn_sched_barrier(0x7);      // (loads stay here, U tokens ahead of their use; arithmetic may move)
    }
    if (g < U) store();
  }
  for (; t0 < r1; t0 += U, op += size_t(U) * ldo) {
#pragma unroll
    for (int n = 0; n < U; ++n)
      if (t0 + n < r1) {
        walk(n);
        if (t0 + n + U < r1) request(n);
      }
    if (g < U && t0 + g < r1) store();
  }
#pragma unroll
  for (int il = 0; il < IPT; ++il) {
    const int from = g * IPT + il / 4 * 4, i = entry_place<HOW>(from, il % 4, dk);
    if (!entry_own<HOW>(from, il % 4, dk)) continue;
#pragma unroll
    for (int c = 0; c < NC; ++c)
      if (owns[c]) st[size_t(i) * dv + j[c]] = S[c][il];
    if (cb == 0 && threadIdx.x < G) n_new[(size_t(s) * heads + head) * dk + i] = N[il];
  }
}

// n_state[slot of sequence s] = n_new[s] for the sequences that ran
__global__ void __launch_bounds__(256)
    mlstm_keep_n_kernel(const float* __restrict__ n_new, float* __restrict__ n_state, const int* __restrict__ run_start,
                        const int* __restrict__ state_slots, int S, int per_seq) {
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= S * per_seq) return;
  const int s = idx / per_seq, slot = state_slots[s];
  if (slot < 0 || run_start[s + 1] <= run_start[s]) return;
  n_state[size_t(slot) * per_seq + idx % per_seq] = n_new[idx];
}

void mlstm_factors(const float* ig, int ldi, const float* fg, int ldf, const float* i_bias, const float* f_bias, float cap, float4* coef,
                   float* m_state, const int* run_start, const int* seq_start, const int* state_slots, int S, int heads, int T, int max_run,
                   int one_order, bool stretches, hipStream_t s) {
  const int logs_first = max_run >= 16 ? 1 : 0;      // long runs: the gates' logarithms of all T rows first, in parallel
  if (logs_first) {
    const long long n = static_cast<long long>(T) * heads;
    mlstm_gate_logs_kernel<<<static_cast<unsigned>((n + 255) / 256), 256, 0, s>>>(ig, ldi, fg, ldf, i_bias, f_bias, cap, coef, n, heads);
    if (stretches && !one_order && max_run > 2 * kWave) {
      mlstm_max_stretches_kernel<<<S * heads, kMaxWaves * kWave, 0, s>>>(coef, m_state, run_start, seq_start, state_slots, heads);
      return;
    }
  }
  auto* maxima = one_order ? mlstm_max_kernel<true> : mlstm_max_kernel<false>;
  maxima<<<S * heads, kWave, 0, s>>>(ig, ldi, fg, ldf, i_bias, f_bias, cap, coef, m_state, run_start, seq_start, state_slots, heads, logs_first);
}

}  // namespace kvcm

using namespace kvcm;

extern "C" {

// q, k [T, heads*dk], v [T, heads*dv], ig, fg [T, heads] (the gates' projections without their biases), at their own
// strides; i_bias, f_bias [heads]; coef: scratch of 4 T heads floats (T: the step's rows, max_run: its longest run); n_new:
// scratch of S heads dk floats; o [T, >= heads*dv]; s_state [slots, heads, dk, dv], n_state [slots, heads, dk],
// m_state [slots, heads]; all 32-bit.
int kvcm_mlstm_scan(const float* q, int ldq, const float* k, int ldk, const float* v, int ldv, const float* ig, int ldi,
                    const float* fg, int ldf, const float* i_bias, const float* f_bias, float cap, float q_scale, float* coef,
                    float* n_new, float* o, int ldo, float* s_state, float* n_state, float* m_state, const int* run_start,
                    const int* seq_start, const int* state_slots, int S, int heads, int dk, int dv, int T, int max_run, int one_order,
                    hipStream_t s) {
  if (S == 0) return 0;
  KVCM_REQUIRE(S > 0 && heads > 0 && dk > 0 && dv > 0, "mlstm_scan: bad sizes S=%d heads=%d dk=%d dv=%d", S, heads, dk, dv);
  KVCM_REQUIRE(dk <= 256, "mlstm_scan: a key size of %d is not supported (up to 256)", dk);
  KVCM_REQUIRE(cap > 0.f, "mlstm_scan: the gates' cap must be positive (%g)", cap);
  KVCM_REQUIRE(static_cast<long long>(heads) * ((dv + 3) / 4) < (1ll << 31), "mlstm_scan: too many heads");
  KVCM_REQUIRE(S <= 65535 && static_cast<long long>(S) * heads * dk < (1ll << 31), "mlstm_scan: too many sequences for one launch (%d)", S);
  KVCM_REQUIRE(ldq >= heads * dk && ldk >= heads * dk && ldv >= heads * dv && ldo >= heads * dv && ldi >= heads && ldf >= heads,
               "mlstm_scan: row strides too small");
  KVCM_REQUIRE(coef && n_new && reinterpret_cast<uintptr_t>(coef) % 16 == 0, "mlstm_scan: the scratch must be there, 16-byte aligned");
  float4* cf = reinterpret_cast<float4*>(coef);
  KVCM_REQUIRE(max_run < 16 || T > 0, "mlstm_scan: the row count is needed for runs of %d", max_run);
  mlstm_factors(ig, ldi, fg, ldf, i_bias, f_bias, cap, cf, m_state, run_start, seq_start, state_slots, S, heads, T, max_run, one_order, S == 1, s);
#define KVCM_MLSTM_AS(DKP, G, NC, U, NT, HOW)                                                                                    \
  {                                                                                                                          \
    const int col_blocks = (dv + NT / G * NC - 1) / (NT / G * NC);                                                                     \
    mlstm_scan_kernel<DKP, G, NC, U, NT, HOW><<<dim3(heads * col_blocks, S), NT, 0, s>>>(q, ldq, k, ldk, v, ldv, cf, q_scale, o,  \
                                                                                     ldo, s_state, n_state, n_new, run_start, \
                                                                                     seq_start, state_slots, heads, dk, dv,  \
                                                                                     col_blocks);                            \
  }
#define KVCM_MLSTM(DKP, G, NC, U, NT)                                  \
  {                                                                \
    if (dk == DKP) KVCM_MLSTM_AS(DKP, G, NC, U, NT, kRowFull)          \
    else if (dk % 4 == 0) KVCM_MLSTM_AS(DKP, G, NC, U, NT, kRowWide)   \
    else KVCM_MLSTM_AS(DKP, G, NC, U, NT, kRowPart)                    \
  }
  // A column over 16 lanes is the shorter chain, over 8 the fewer instructions: once waves of eight columns fill the SIMDs, those.
  // 2,048 tokens of one sequence / 8 sequences of 509, 32 heads of 64 x 64, us: 292 (16 lanes) / 247 and 217 (16 lanes; 8 lanes of two columns).
  // The other sizes, us with the maxima, workgroups that share a token's vectors through LDS / so, 64 heads of 16 x 16, 64 of 32 x 32, 8 of
  // 48 x 48, 32 of 128 x 128, 8 of 256 x 256: one sequence of 1,024 tokens 416 / 163, 423 / 162, 499 / 146, 587 / 287, 1,367 / 508; 8 of 129
  // 70 / 38, 73 / 51, 75 / 33, 307 / 189, 526 / 276; 8 single tokens 10.1 / 9.5, 10.5 / 10.2, 10.7 / 10.0, 37 / 32, 36 / 33.
  // The lanes of a column are the order of its sums: with one_order they follow from the key size alone (8 from 33 to
  // 64: 394 us for the one sequence).
  const bool few = static_cast<long long>(S) * heads * ((dv + 7) / 8) < 1024;
  if (max_run >= 16) {
    if (dk < 4) KVCM_MLSTM_AS(16, 4, 1, 4, kWave, kRowSingle)
    else if (dk <= 16) KVCM_MLSTM(16, 4, 1, 4, kWave)
    else if (dk <= 32) KVCM_MLSTM(32, 8, 1, 4, kWave)
    else if (dk <= 64 && few && !one_order) KVCM_MLSTM(64, 16, 1, 8, kWave)
    else if (dk <= 64 && few) KVCM_MLSTM(64, 8, 1, 8, kWave)
    else if (dk <= 64) KVCM_MLSTM(64, 8, 2, 4, kWave)
    else if (dk <= 128) KVCM_MLSTM(128, 16, 1, 6, kWave)
    else KVCM_MLSTM(256, 16, 1, 4, kWave)
  } else {
    if (dk < 4) KVCM_MLSTM_AS(16, 4, 1, 1, 128, kRowSingle)
    else if (dk <= 16) KVCM_MLSTM(16, 4, 1, 1, 128)
    else if (dk <= 32) KVCM_MLSTM(32, 8, 1, 1, 256)
    else if (dk <= 64) KVCM_MLSTM(64, 8, 1, 1, 256)
    else if (dk <= 128) KVCM_MLSTM(128, 16, 1, 1, 256)
    else KVCM_MLSTM(256, 16, 1, 1, 256)
  }
#undef KVCM_MLSTM_AS
#undef KVCM_MLSTM
  const int per_seq = heads * dk;
  mlstm_keep_n_kernel<<<(S * per_seq + 255) / 256, 256, 0, s>>>(n_new, n_state, run_start, state_slots, S, per_seq);
  return launch_status("mlstm_scan");
}

}  // extern "C"
