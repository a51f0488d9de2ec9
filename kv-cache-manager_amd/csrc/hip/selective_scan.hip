// Selective scan (a diagonal linear recurrence whose step, input and output maps depend on the token),
// over rows that are packed runs of several sequences, the state of each sequence kept in its slot.
//
//   dt = softplus(dt_lin + dt_bias)                         one step size per channel c
//   S[c, n] <- exp(dt * A[c, n]) * S[c, n] + dt * x_c * B_n,  A = -exp(A_log)
//   y_c = sum_n S[c, n] * C_n + D_c * x_c;   out_c = y_c * silu(z_c)
//
// Everything of the recurrence is 32-bit: the state, the step size with its softplus, the decay's
// exponential, the sums.  Runs are walked with the states of a channel spread over LPC lanes (a power of two, up to a
// whole wave; NPL states a lane beyond that), so that a wave of 64 lanes walks 64 / LPC channels: the run's
// tokens are taken in order, one exponential and two multiply-adds a lane and token, and the sum over a
// channel's states crosses its lanes in a fixed tree.  With 8 or 16 states, steps of single tokens and the pieces of
// long runs have a channel's states in one lane instead; in 32-bit storage they are added in the same tree.
// What a token brings (its step size, input, gate, B and C) does not depend on the state: it is requested a few
// tokens ahead, so that the walk waits for arithmetic and not for memory.  A run that starts at position 0 starts from
// zero without reading its slot; the state after the run's last token goes back to the slot.  Tokens are taken one by
// one in prompts and in decoding, so in 32-bit storage a position's result does not depend on how the prompt was cut,
// but for runs walked in pieces, where a piece's entering state comes by one multiply-add instead of one per token.
#include <type_traits>

#include "common.h"
#include "kvcm_hip.h"

namespace kvcm {

// exp of a decay's exponent for a walk whose inputs and outputs are stored as T: exact for float; for bfloat16 the
// hardware's exp2 (about one unit in the last place of a 32-bit value, a tenth of the instructions), which is far
// inside what the storage type keeps of x and of the result.
template <class T> __device__ __forceinline__ float decay_exp(float v);
template <> __device__ __forceinline__ float decay_exp<float>(float v) { return expf(v); }
template <> __device__ __forceinline__ float decay_exp<bf16_t>(float v) { return __builtin_amdgcn_exp2f(1.44269504088896341f * v); }

// log(1 + exp(v)) = max(v, 0) + log1p(exp(-|v|)): exp2 of -|v| log2(e) times what that product's rounding lost, and the logarithm of the
// rounded 1 + e with what its rounding lost.  A dozen instructions with three of a quarter's rate, where log1pf(expf(v)) is some
// hundred (21 of a pass's 62 us at 2,048 x 4,096).  Largest error against 64 bits, log1pf(expf(v)) / so: 1.4e-6 / 2.6e-7 over
// [-30, -15), 8.5e-7 / 2.3e-7 to -5, 3.4e-7 / 2.2e-7 to -1, 2.1e-7 / 1.7e-7 to 0, 1.5e-7 / 1.1e-7 beyond.
__device__ __forceinline__ float softplus(float v) {
  const float m = fabsf(v), a = m > 200.f ? 200.f : m;      // (what is no number stays none)
  const float p = a * 1.44269504088896341f;
  const float lost = fmaf(a, 1.925962991e-8f, fmaf(a, 1.44269504088896341f, -p));
  const float e0 = __builtin_amdgcn_exp2f(-p), e = fmaf(e0 * lost, -0.69314718055994531f, e0);
  const float w = 1.f + e, c = e - (w - 1.f);
  return fmaxf(v, 0.f) + fmaf(__builtin_amdgcn_logf(w), 0.69314718055994531f, c * __builtin_amdgcn_rcpf(w));      // (logf: to base 2)
}

constexpr int kScanAhead = 4;      // tokens whose inputs are on their way while the ones before are computed

template <class T, int LPC, int NPL>
__global__ void __launch_bounds__(kWave)
    selective_scan_kernel(const T* __restrict__ x, int ldx, const float* __restrict__ dt_lin, int lddt,
                          const float* __restrict__ dt_bias, const float* __restrict__ bc, int ldbc, int off_b, int off_c,
                          const float* __restrict__ a_log, const float* __restrict__ dskip, const float* __restrict__ z,
                          int ldz, T* __restrict__ out, int ldo, float* __restrict__ state,
                          const int* __restrict__ run_start, const int* __restrict__ seq_start,
                          const int* __restrict__ state_slots, int C, int N, int prepared, int phase, int chunk_len,
                          float* __restrict__ carry, float* __restrict__ dsum) {
  constexpr int U = kScanAhead;
  const int s = blockIdx.y;
  const int sub = threadIdx.x % LPC;
  const int c_real = blockIdx.x * (kWave / LPC) + threadIdx.x / LPC;
  const bool owns = c_real < C;
  const int c = owns ? c_real : C - 1;      // lanes beyond the last channel walk along (the sums cross lanes) and store nothing
  int r0 = run_start[s], r1 = run_start[s + 1];
  const int slot = state_slots[s];
  // phases 1 and 2 walk one piece of chunk_len rows of the run each (blockIdx.z): 1 from zero, leaving the piece's
  // end state and the sum of its step sizes; 2 from the state that enters the piece, writing the outputs
  size_t piece = 0;
  if (phase != 0) {
    piece = size_t(r0 / chunk_len + s) + blockIdx.z;
    r0 += blockIdx.z * chunk_len;
    r1 = r1 < r0 + chunk_len ? r1 : r0 + chunk_len;
  }
  if (r1 <= r0) return;
  if (slot < 0) {      // a padding sequence: its rows carry nothing
    if (owns && sub == 0 && phase != 1)
      for (int r = r0; r < r1; ++r) store_f(out + size_t(r) * ldo + c, 0.f);
    return;
  }
  float* st = phase == 0 ? state + (size_t(slot) * C + c) * N : carry + (piece * C + c) * N;
  const bool fresh = phase == 1 || (phase == 0 && seq_start[s] == 0);
  float S[NPL], A[NPL];
  int nidx[NPL];
  bool has[NPL];
#pragma unroll
  for (int k = 0; k < NPL; ++k) {
    const int n = sub + k * LPC;
    has[k] = n < N;
    nidx[k] = has[k] ? n : N - 1;
    A[k] = has[k] ? -expf(a_log[size_t(c) * N + nidx[k]]) : 0.f;
    S[k] = (has[k] && !fresh) ? st[nidx[k]] : 0.f;
  }
  const float db = dt_bias ? dt_bias[c] : 0.f, dk = dskip[c];

  float dt_total = 0.f;
  float dtv[2][U], xv[2][U], zv[2][U], bv[2][U][NPL], cv[2][U][NPL];
  auto request = [&](int first, int into) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int r = first + u < r1 ? first + u : r1 - 1;
      dtv[into][u] = dt_lin[size_t(r) * lddt + c];
      xv[into][u] = load_f(x + size_t(r) * ldx + c);
#pragma unroll
      for (int k = 0; k < NPL; ++k) bv[into][u][k] = bc[size_t(r) * ldbc + off_b + nidx[k]];
      if (phase != 1) {      // (the same for every lane) the pass that only wants the state needs neither the gate nor C
        zv[into][u] = z[size_t(r) * ldz + c];
#pragma unroll
        for (int k = 0; k < NPL; ++k) cv[into][u][k] = bc[size_t(r) * ldbc + off_c + nidx[k]];
      }
    }
  };
  auto walk = [&](int first, int from) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int r = first + u;
      if (r < r1) {
        const float v = dtv[from][u] + db;
        const float dt = prepared ? dtv[from][u] : softplus(v);
        const float dx = dt * xv[from][u];
        dt_total += dt;
        float y = 0.f;
#pragma unroll
        for (int k = 0; k < NPL; ++k) {
          const float sn = fmaf(decay_exp<T>(dt * A[k]), S[k], dx * bv[from][u][k]);
          S[k] = has[k] ? sn : 0.f;
        }
        if (phase == 1) continue;      // only the state is wanted
#pragma unroll
        for (int k = 0; k < NPL; ++k) y = fmaf(S[k], cv[from][u][k], y);
        y = group_sum<LPC>(y);
        if (owns && sub == 0) {
          y = fmaf(dk, xv[from][u], y);
          const float zz = zv[from][u];
          store_f(out + size_t(r) * ldo + c, y * (prepared ? zz : zz / (1.0f + expf(-zz))));
        }
      }
    }
  };
  request(r0, 0);
  for (int r = r0; r < r1; r += 2 * U) {
    if (r + U < r1) request(r + U, 1);
    walk(r, 0);
    if (r + U < r1) {
      if (r + 2 * U < r1) request(r + 2 * U, 0);
      walk(r + U, 1);
    }
  }
  if (owns && phase != 2) {
#pragma unroll
    for (int k = 0; k < NPL; ++k)
      if (has[k]) st[nidx[k]] = S[k];
    if (phase == 1 && sub == 0) dsum[piece * C + c] = dt_total;
  }
}

// Pieces of long runs with 8 or 16 states a channel: a lane owns a channel with all its states, so that a token costs a lane one
// exponential and three multiply-adds a state and no sum crosses lanes (with the states over lanes every lane also fetched the
// channel's step size, input and gate, and a wave's sums took a sixth of its instructions).  B and C, the same for all channels,
// are staged through LDS 64 tokens at a time and read by all lanes at once.  Bound by a wave's own chain while there are few waves, then by
// the exponentials, a quarter of the rate of other instructions.  4,096 channels, 16 states, both passes and what is between: 512 / 1,024 / 2,048
// tokens 98 / 170 / 136 us in pieces of 128 tokens behind a launch that made step sizes and gates; 48 / 71 / 112 us in pieces of 32 to 64
// without it, and the last, with the step size's formula above, 94 us (41, 8 and 45).
template <class T> __device__ __forceinline__ float scaled_rate(float a) { return a; }
template <> __device__ __forceinline__ float scaled_rate<bf16_t>(float a) { return 1.44269504088896341f * a; }      // for exp2
template <class T> __device__ __forceinline__ float scaled_exp(float v) { return expf(v); }
template <> __device__ __forceinline__ float scaled_exp<bf16_t>(float v) { return __builtin_amdgcn_exp2f(v); }

constexpr int kScanTile = 64;      // tokens whose B and C lie in LDS

// Sum over a channel's states in the order of group_sum, where the states lie over lanes: neighbours, pairs, fours, eights.
template <int N>
__device__ __forceinline__ float states_sum(float (&v)[N]) {
#pragma unroll
  for (int d = 1; d < N; d *= 2)
#pragma unroll
    for (int n = 0; n < N; n += 2 * d) v[n] += v[n + d];
  return v[0];
}

// Runs of one token (decoding), a lane a channel with all its states: with the states over lanes a wave's four channels each
// fetched their step size, input and gate sixteen times and asked for four tokens; 8 rows, 4,096 channels, 16 states: 14.5 us a
// launch, 4.5 us so (2 MB of states read and written).
template <class T, int N>
__global__ void __launch_bounds__(kWave)
    scan_single_kernel(const T* __restrict__ x, int ldx, const float* __restrict__ dt_lin, int lddt, const float* __restrict__ dt_bias,
                       const float* __restrict__ bc, int ldbc, int off_b, int off_c, const float* __restrict__ a_log,
                       const float* __restrict__ dskip, const float* __restrict__ z, int ldz, T* __restrict__ out, int ldo,
                       float* __restrict__ state, const int* __restrict__ run_start, const int* __restrict__ seq_start,
                       const int* __restrict__ state_slots, int C, int prepared) {
  const int s = blockIdx.y, c = blockIdx.x * kWave + threadIdx.x;
  const int r = run_start[s], slot = state_slots[s];
  if (run_start[s + 1] <= r || c >= C) return;
  if (slot < 0) {      // a padding sequence: its row carries nothing
    store_f(out + size_t(r) * ldo + c, 0.f);
    return;
  }
  float* at = state + (size_t(slot) * C + c) * N;
  const float keep = seq_start[s] == 0 ? 0.f : 1.f;
  float4 sv[N / 4], av[N / 4];
#pragma unroll
  for (int n = 0; n < N / 4; ++n) {
    sv[n] = *reinterpret_cast<const float4*>(at + 4 * n);
    av[n] = *reinterpret_cast<const float4*>(a_log + size_t(c) * N + 4 * n);
  }
  const float lin = dt_lin[size_t(r) * lddt + c], xx = load_f(x + size_t(r) * ldx + c), zz = z[size_t(r) * ldz + c];
  const float v = lin + (dt_bias ? dt_bias[c] : 0.f), skip = dskip[c];
  const float *b = bc + size_t(r) * ldbc + off_b, *cc = bc + size_t(r) * ldbc + off_c;
  const float dt = prepared ? lin : softplus(v), dx = dt * xx;
  float ys[N];
#pragma unroll
  for (int n = 0; n < N / 4; ++n) {
    float se[4] = {sv[n].x, sv[n].y, sv[n].z, sv[n].w};
    const float ae[4] = {av[n].x, av[n].y, av[n].z, av[n].w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float was = keep != 0.f ? se[e] : 0.f;      // (a first token starts from zero, whatever the slot holds)
      se[e] = fmaf(decay_exp<T>(dt * -expf(ae[e])), was, dx * b[4 * n + e]);
      ys[4 * n + e] = fmaf(se[e], cc[4 * n + e], 0.f);      // (rounded before it is added, like a lane's own)
    }
    *reinterpret_cast<float4*>(at + 4 * n) = float4{se[0], se[1], se[2], se[3]};
  }
  store_f(out + size_t(r) * ldo + c, fmaf(skip, xx, states_sum(ys)) * (prepared ? zz : zz / (1.0f + expf(-zz))));
}

// The first pass makes the step sizes as it walks and leaves them in place for the second, which makes the gates (a launch of
// their own read and wrote both, 134 MB of 32-bit rows and 37 us at 2,048 x 4,096), unless they are prepared already.
template <class T, int N, bool OUT>
__global__ void __launch_bounds__(256)
    scan_channels_kernel(const T* __restrict__ x, int ldx, float* __restrict__ dt, int lddt, const float* __restrict__ dt_bias,
                         const float* __restrict__ bc, int ldbc, int off_b, int off_c, const float* __restrict__ a_log,
                         const float* __restrict__ dskip, const float* __restrict__ z, int ldz, T* __restrict__ out, int ldo,
                         const int* __restrict__ run_start, const int* __restrict__ state_slots, int C, int prepared, int chunk_len,
                         float* __restrict__ carry, float* __restrict__ dsum) {
  constexpr int U = 4, W = OUT ? 2 * N : N;
  constexpr bool kOneOrder = std::is_same<T, float>::value;      // (32-bit results do not depend on how the states are dealt out)
  __shared__ __attribute__((aligned(16))) float tile[kScanTile][W];
  const int s = blockIdx.y, c_real = blockIdx.x * 256 + threadIdx.x;
  const bool owns = c_real < C;
  const int c = owns ? c_real : C - 1;
  int r0 = run_start[s], r1 = run_start[s + 1];
  const size_t piece = size_t(r0 / chunk_len + s) + blockIdx.z;
  r0 += blockIdx.z * chunk_len;
  r1 = r1 < r0 + chunk_len ? r1 : r0 + chunk_len;
  if (r1 <= r0) return;
  if (state_slots[s] < 0) {      // a padding sequence: its rows carry nothing
    if (owns && OUT)
      for (int r = r0; r < r1; ++r) store_f(out + size_t(r) * ldo + c, 0.f);
    return;
  }
  float* at = carry + (piece * C + c) * N;
  float S[N], A[N];
#pragma unroll
  for (int n = 0; n < N; ++n) {
    A[n] = scaled_rate<T>(-expf(a_log[size_t(c) * N + n]));
    S[n] = OUT ? at[n] : 0.f;
  }
  const float skip = OUT ? dskip[c] : 0.f, db = !OUT && dt_bias ? dt_bias[c] : 0.f;
  float dt_total = 0.f;
  float dtv[2][U], xv[2][U], zv[2][U];
  auto request = [&](int first, int into) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int r = first + u < r1 ? first + u : r1 - 1;
      dtv[into][u] = dt[size_t(r) * lddt + c];
      xv[into][u] = load_f(x + size_t(r) * ldx + c);
      if (OUT) zv[into][u] = z[size_t(r) * ldz + c];
    }
  };
  auto walk = [&](int first, int from, int t0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int r = first + u;
      if (r >= r1) break;
      float step = dtv[from][u];
      if (!OUT && !prepared) {
        step = softplus(step + db);
        if (owns) dt[size_t(r) * lddt + c] = step;
      }
      const float dx = step * xv[from][u];
      const float* bt = tile[r - t0];
      dt_total += step;
      float y = 0.f, ys[N];
#pragma unroll
      for (int n = 0; n < N; ++n) {
        S[n] = fmaf(scaled_exp<T>(step * A[n]), S[n], dx * bt[n]);
        if (OUT && kOneOrder) ys[n] = fmaf(S[n], bt[N + n], 0.f);
        else if (OUT) y = fmaf(S[n], bt[N + n], y);
      }
      if (OUT && kOneOrder) y = states_sum(ys);
      if (OUT && owns) {
        const float zz = zv[from][u];
        store_f(out + size_t(r) * ldo + c, fmaf(skip, xv[from][u], y) * (prepared ? zz : zz / (1.0f + expf(-zz))));
      }
    }
  };
  request(r0, 0);
  for (int t0 = r0; t0 < r1; t0 += kScanTile) {
    if (t0 > r0) __syncthreads();
    const int end = r1 < t0 + kScanTile ? r1 : t0 + kScanTile;
    for (int e = threadIdx.x; e < (end - t0) * W; e += 256) {
      const int t = e / W, n = e % W;
      tile[t][n] = bc[size_t(t0 + t) * ldbc + (n < N ? off_b + n : off_c + n - N)];
    }
    __syncthreads();
    for (int r = t0; r < end; r += 2 * U) {      // (a tile is a multiple of 2 U tokens)
      request(r + U, 1);
      walk(r, 0, t0);
      request(r + 2 * U, 0);
      walk(r + U, 1, t0);
    }
  }
  if (!OUT && owns) {
#pragma unroll
    for (int n = 0; n < N; ++n) at[n] = S[n];
    dsum[piece * C + c] = dt_total;
  }
}

// Between the two phases: per (sequence, channel, state) the pieces' end states become the states that enter them,
// S_in[0] = the slot's (zero for a sequence's first portion), S_in[j+1] = exp(A * sum of the piece's step sizes) *
// S_in[j] + end[j]; the last one goes to the slot.
__global__ void __launch_bounds__(256)
    scan_carry_kernel(float* __restrict__ carry, const float* __restrict__ dsum, const float* __restrict__ a_log,
                      float* __restrict__ state, const int* __restrict__ run_start, const int* __restrict__ seq_start,
                      const int* __restrict__ state_slots, int C, int N, int chunk_len) {
  const int s = blockIdx.y;
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= C * N) return;
  const int r0 = run_start[s], len = run_start[s + 1] - r0, slot = state_slots[s];
  if (len <= 0 || slot < 0) return;
  const int c = e / N;
  const float A = -expf(a_log[e]);
  float* st = state + size_t(slot) * C * N + e;
  float S = seq_start[s] == 0 ? 0.f : *st;
  const size_t first = size_t(r0 / chunk_len + s);
  const int pieces = (len + chunk_len - 1) / chunk_len;
  constexpr int kAhead = 16;      // pieces requested together
  for (int j0 = 0; j0 < pieces; j0 += kAhead) {
    float end[kAhead], steps[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const size_t at = first + (j0 + i < pieces ? j0 + i : pieces - 1);
      end[i] = carry[at * C * N + e];
      steps[i] = dsum[at * C + c];
    }
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      if (j0 + i >= pieces) break;
      carry[(first + j0 + i) * C * N + e] = S;
      S = fmaf(expf(A * steps[i]), S, end[i]);
    }
  }
  *st = S;
}

// For long runs: the step sizes and the gates of all rows at once, in place (dt <- softplus(dt + bias), z <- silu(z)),
// so that the walk along a run, whose lanes would each repeat them, finds them made.
__global__ void __launch_bounds__(256)
    scan_prepare_kernel(float* __restrict__ dt, int lddt, const float* __restrict__ dt_bias, float* __restrict__ z, int ldz, int C) {
  const int r = blockIdx.y, c = blockIdx.x * 256 + threadIdx.x;
  if (c >= C) return;
  const float v = dt[size_t(r) * lddt + c] + (dt_bias ? dt_bias[c] : 0.f);
  dt[size_t(r) * lddt + c] = softplus(v);
  const float zz = z[size_t(r) * ldz + c];
  z[size_t(r) * ldz + c] = zz / (1.0f + expf(-zz));
}

// Pieces: a lane a channel or states over lanes.  bfloat16, both passes with what is between, pieces of 32 rows, us, states over lanes / a
// lane a channel, 16 states (before the step size's formula above): 256 rows of 1,024 channels 32 / 40, of 2,048 38 / 41, of 4,096 60 / 42; 512 of 1,024 42 / 43, of 2,048 64 / 44;
// 1,024 of 4,096 183 / 71.  32-bit exponentials take longer, and a wave all of them (pieces of 128): 1 x 2,048 of 1,024 110 / 198, of 2,048
// 182 / 207, of 4,096 330 / 227, 8 x 512 of 1,024 173 / 203, of 2,048 311 / 220.
bool scan_by_channels(bool f32, int T, int C, int N, int chunk_len) {      // (from about one wave, 64 channels of a piece, a CU on)
  return (N == 8 || N == 16) && static_cast<long long>(T) * C >= (f32 ? 640ll : 256ll) * kWave * chunk_len;
}

int prepare_scan(float* dt, int lddt, const float* dt_bias, float* z, int ldz, int T, int C, hipStream_t s) {
  KVCM_REQUIRE(T <= 65535, "scan_prepare: too many rows for one launch (%d)", T);
  scan_prepare_kernel<<<dim3((C + 255) / 256, T), 256, 0, s>>>(dt, lddt, dt_bias, z, ldz, C);
  return launch_status("scan_prepare");
}

template <class X>
int launch_scan(const void* x, int ldx, float* dt_lin, int lddt, const float* dt_bias, const float* bc, int ldbc,
                int off_b, int off_c, const float* a_log, const float* dskip, const float* z, int ldz, void* out, int ldo,
                float* state, const int* run_start, const int* seq_start, const int* state_slots, int S, int C, int N,
                int prepared, int phase, int chunk_len, int pieces, int max_run, int T, float* carry, float* dsum, hipStream_t s) {
  auto aligned = [](const float* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  // (sixteen states with 32-bit exponentials, one after the other in a lane, pay from 8,192 channels on: us, states over lanes / a lane
  // a channel, 8 rows of 64 channels 4.1 / 4.4, 1 of 4,096 4.2 / 4.5, 1 of 8,192 4.7 / 4.5, 8 of 4,096 7.9 / 5.0)
  const bool lanes = std::is_same<X, float>::value && N == 16 && static_cast<long long>(S) * C < 8192;
  if (phase == 0 && max_run == 1 && !lanes && (N == 8 || N == 16) && aligned(state) && aligned(a_log)) {
    const dim3 grid((C + kWave - 1) / kWave, S);
#define KVCM_SCAN_SINGLE(N)                                                                                                    \
  scan_single_kernel<X, N><<<grid, kWave, 0, s>>>(static_cast<const X*>(x), ldx, dt_lin, lddt, dt_bias, bc, ldbc, off_b, off_c, \
                                                  a_log, dskip, z, ldz, static_cast<X*>(out), ldo, state, run_start, seq_start, \
                                                  state_slots, C, prepared)
    if (N == 8) KVCM_SCAN_SINGLE(8);
    else KVCM_SCAN_SINGLE(16);
#undef KVCM_SCAN_SINGLE
    return launch_status("selective_scan");
  }
  if (phase != 0 && scan_by_channels(std::is_same<X, float>::value, T, C, N, chunk_len)) {
    const dim3 grid((C + 255) / 256, S, pieces);
#define KVCM_SCAN_CHANNELS(N, OUT)                                                                                            \
  scan_channels_kernel<X, N, OUT><<<grid, 256, 0, s>>>(static_cast<const X*>(x), ldx, dt_lin, lddt, dt_bias, bc, ldbc, off_b,   \
                                                       off_c, a_log, dskip, z, ldz, static_cast<X*>(out), ldo, run_start,       \
                                                       state_slots, C, prepared, chunk_len, carry, dsum)
    if (N == 8 && phase == 1) KVCM_SCAN_CHANNELS(8, false);
    else if (N == 8) KVCM_SCAN_CHANNELS(8, true);
    else if (phase == 1) KVCM_SCAN_CHANNELS(16, false);
    else KVCM_SCAN_CHANNELS(16, true);
#undef KVCM_SCAN_CHANNELS
    return launch_status("selective_scan");
  }
#define KVCM_SCAN(LPC, NPL)                                                                                             \
  selective_scan_kernel<X, LPC, NPL><<<dim3((C + kWave / LPC - 1) / (kWave / LPC), S, pieces), kWave, 0, s>>>(           \
      static_cast<const X*>(x), ldx, dt_lin, lddt, dt_bias, bc, ldbc, off_b, off_c, a_log, dskip, z, ldz,               \
      static_cast<X*>(out), ldo, state, run_start, seq_start, state_slots, C, N, prepared, phase, chunk_len, carry, dsum)
  if (N <= 1) KVCM_SCAN(1, 1);
  else if (N <= 2) KVCM_SCAN(2, 1);
  else if (N <= 4) KVCM_SCAN(4, 1);
  else if (N <= 8) KVCM_SCAN(8, 1);
  else if (N <= 16) KVCM_SCAN(16, 1);
  else if (N <= 32) KVCM_SCAN(32, 1);
  else if (N <= 64) KVCM_SCAN(64, 1);
  else if (N <= 128) KVCM_SCAN(64, 2);
  else KVCM_SCAN(64, 4);
#undef KVCM_SCAN
  return launch_status("selective_scan");
}

}  // namespace kvcm

using namespace kvcm;

// x [T, C] (after its convolution and activation) and out [T, C] in the storage type; dt_lin [T, C], bc [T, ldbc]
// (B at off_b, C at off_c, N each), z [T, ldz], a_log [C, N], dt_bias, dskip [C], state [slots, C, N]: 32-bit.
// prepared: dt_lin holds the step sizes and z the gates already (kvcm_scan_prepare).
// chunk_len > 0: runs (of up to max_run rows, T rows in all) are walked in pieces of chunk_len rows, all pieces at once, with
// carry (at least (T / chunk_len + S + 1) * C * (N + 1) floats) between the phases; what is not prepared is then made here, dt_lin (and
// z, where the states lie over lanes) hold it afterwards; 0: every run in one walk.
extern "C" int kvcm_selective_scan(const void* x, int dtype, int ldx, float* dt_lin, int lddt, const float* dt_bias,
                                   const float* bc, int ldbc, int off_b, int off_c, const float* a_log, const float* dskip,
                                   float* z, int ldz, void* out, int ldo, float* state, const int* run_start,
                                   const int* seq_start, const int* state_slots, int S, int C, int N, int prepared,
                                   int chunk_len, int max_run, float* carry, long long carry_floats, int T, hipStream_t s) {
  if (S == 0) return 0;
  KVCM_REQUIRE(S > 0 && C > 0 && N > 0, "selective_scan: bad sizes S=%d C=%d N=%d", S, C, N);
  KVCM_REQUIRE(N <= 256, "selective_scan: a state of %d per channel is not supported (up to 256)", N);
  KVCM_REQUIRE(S <= 65535, "selective_scan: too many sequences for one launch (%d)", S);
  KVCM_REQUIRE(ldx >= C && lddt >= C && ldz >= C && ldo >= C && off_b >= 0 && off_c >= 0 && ldbc >= off_b + N &&
                   ldbc >= off_c + N, "selective_scan: row strides too small");
  KVCM_REQUIRE(dtype == kF32 || dtype == kBF16, "selective_scan: unknown dtype %d", dtype);
  auto launch = [&](int phase, int pieces, float* cr, float* ds) {
    if (dtype == kF32)
      return launch_scan<float>(x, ldx, dt_lin, lddt, dt_bias, bc, ldbc, off_b, off_c, a_log, dskip, z, ldz, out, ldo, state,
                                run_start, seq_start, state_slots, S, C, N, prepared, phase, chunk_len, pieces, max_run, T, cr, ds, s);
    return launch_scan<bf16_t>(x, ldx, dt_lin, lddt, dt_bias, bc, ldbc, off_b, off_c, a_log, dskip, z, ldz, out, ldo, state,
                               run_start, seq_start, state_slots, S, C, N, prepared, phase, chunk_len, pieces, max_run, T, cr, ds, s);
  };
  if (chunk_len <= 0) return launch(0, 1, nullptr, nullptr);
  // long runs in pieces of chunk_len rows: every piece from zero, the states that enter the pieces, every piece again
  const int pieces = (max_run + chunk_len - 1) / chunk_len;
  const long long slots = static_cast<long long>(T) / chunk_len + S + 1;      // piece j of sequence s: run_start / chunk_len + s + j
  KVCM_REQUIRE(pieces >= 1 && pieces <= 65535 && carry != nullptr && carry_floats >= slots * C * (N + 1),
               "selective_scan: the scratch for %lld pieces is too small", slots);
  float* dsum = carry + slots * C * N;
  if (!prepared && !scan_by_channels(dtype == kF32, T, C, N, chunk_len)) {
    if (int rc = prepare_scan(dt_lin, lddt, dt_bias, z, ldz, T, C, s)) return rc;
    prepared = 1;
  }
  if (int rc = launch(1, pieces, carry, dsum)) return rc;
  scan_carry_kernel<<<dim3((C * N + 255) / 256, S), 256, 0, s>>>(carry, dsum, a_log, state, run_start, seq_start, state_slots, C, N,
                                                                 chunk_len);
  if (int rc = launch_status("scan_carry")) return rc;
  return launch(2, pieces, carry, dsum);
}

// dt [T, C] <- softplus(dt + dt_bias), z [T, C] <- silu(z), in place; kvcm_selective_scan then runs with prepared = 1.
extern "C" int kvcm_scan_prepare(float* dt, int lddt, const float* dt_bias, float* z, int ldz, int T, int C, hipStream_t s) {
  if (T == 0) return 0;
  KVCM_REQUIRE(T > 0 && C > 0 && lddt >= C && ldz >= C, "scan_prepare: bad sizes T=%d C=%d", T, C);
  return prepare_scan(dt, lddt, dt_bias, z, ldz, T, C, s);
}
