// The generalized delta rule: a matrix state per head that decays per key channel, forgets along the
// current unit key and learns the current key-value pair,
//
//   u = k / sqrt(|k|^2 + 1e-6)
//   S <- diag(w) S - (a * u) (u^T S) + k v^T        (both terms read the old S)
//   o = S^T r
//
// with w = exp(-exp(-1/2) * sigmoid(w_lin + w0)) and a = sigmoid(a_lin + a_bias) per head and key channel.
// State, decay, removal rate, unit key and all sums are 32-bit.
//
// Two launches.  The first turns the projections of every row into (w, a * u, u), in parallel over rows
// (the second step of the decay's projection included).
// The second walks each sequence's run token by token: a value column j of S needs u^T S[:, j], updates itself
// and sums o_j, and needs no other column, so columns are spread over lanes and waves.  What bounds the walk is a token's
// chain of dependent instructions, so a wave has few columns, its key dimension over up to 16 lanes, and a workgroup is one
// wave: nothing is shared and nobody waits.  The per-token vectors (r, k, w, a*u, u, v) go from L2 into the lanes that use
// them, a few tokens ahead.  A run that starts at position 0 starts from zero without reading its slot.  Tokens are taken one
// by one in prompts and in decoding; delta_chunks.hip takes long runs in matrix form.
#include "common.h"
#include "kvcm_hip.h"

namespace kvcm {

// A wave makes R rows of a head, a workgroup those of up to four heads (of five, three and two).  The decay's logit
// is a two-step projection whose second step runs here in 32-bit: w_lin[c] = sum_j w2[c, j] * tanh(low[j]), low = the first step's output (rank values
// a row), tanh once for the workgroup's heads; w2 comes transposed, [rank, heads*d], sixteen of a channel's values on their way together: one at a time a
// step of few rows was a chain of `rank` trips to L2.  us, a wave of its own for every row and head, its values one at a time /
// so (the bits are the same either way), heads, size, rank, rows: 32, 64, 64, 8 rows 4.8 / 3.8, 2,048 rows 66 / 42; 32, 128, 64 7.0 / 5.2 and 112 / 73; 32, 64, 8
// 3.3 / 3.2 and 34 / 30; 5, 64, 64, 2,048 rows 13.0 / 10.4; 1, 64, 64, 2,048 rows 5.3 / 4.9.  Up to 0.8 us slower at a few thousand rows and heads with short ranks (9, 48, 20, 512
// rows 5.2 / 6.0; 3, 64, 15, 2,048 rows 6.0 / 6.9).
constexpr int kDeltaMaxRank = 256;
template <int R>
__global__ void __launch_bounds__(256)
    delta_prepare_kernel(const float* __restrict__ k, int ldk, const float* __restrict__ a_lin, int lda,
                         const float* __restrict__ a_bias, const float* __restrict__ low, int ldlow,
                         const float* __restrict__ w2t, int rank, const float* __restrict__ w0,
                         float* __restrict__ w_out, float* __restrict__ au_out, float* __restrict__ u_out, int heads, int d, int T,
                         unsigned row_blocks) {
  __shared__ __attribute__((aligned(16))) float th[kDeltaMaxRank][R];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave, waves = blockDim.x / kWave;
  const int row0 = static_cast<int>(blockIdx.x % row_blocks) * R, head = static_cast<int>(blockIdx.x / row_blocks) * waves + wave;
  auto row_of = [&](int n) { return size_t(row0 + n < T ? row0 + n : T - 1); };      // (rows beyond the last are left out of the stores)
  if constexpr (R == 1) {
    for (int j = threadIdx.x; j < rank; j += blockDim.x) th[j][0] = tanhf(low[row_of(0) * ldlow + j]);
  } else {
    for (int n = wave; n < R; n += waves)
      for (int j = lane; j < rank; j += kWave) th[j][n] = tanhf(low[row_of(n) * ldlow + j]);
  }
  __syncthreads();
  if (head >= heads) return;
  const size_t col = size_t(head) * d, D = size_t(heads) * d;
  float inv[R];
#pragma unroll
  for (int n = 0; n < R; ++n) {
    const float* kr = k + row_of(n) * ldk + col;
    float ss = 0.f;
    for (int i = lane; i < d; i += kWave) ss = fmaf(kr[i], kr[i], ss);
    inv[n] = 1.0f / sqrtf(wave_sum(ss) + 1e-6f);
  }
  const float rate = 0.60653065971263342f;      // exp(-1/2)
  for (int i = lane; i < d; i += kWave) {
    const float* w2 = w2t + col + i;      // neighbours read neighbours
    float wl[R] = {}, kx[R], ax[R];
#pragma unroll
    for (int n = 0; n < R; ++n) {
      kx[n] = k[row_of(n) * ldk + col + i];
      ax[n] = a_lin[row_of(n) * lda + col + i];
    }
    int j = 0;
    auto add = [&](auto ahead, int values) __attribute__((always_inline)) {      // `values` of a channel's from j on, all on their way together
      constexpr int N = decltype(ahead)::value;
      float x[N];
#pragma unroll
      for (int m = 0; m < N; ++m) x[m] = w2[size_t(j + (m < values ? m : values - 1)) * D];
#pragma unroll
      for (int m = 0; m < N; ++m)
        if (m < values) {
#pragma unroll
          for (int n = 0; n < R; ++n) wl[n] = fmaf(x[m], th[j + m][n], wl[n]);
        }
      j += values;
    };
    while (j + 16 <= rank) add(std::integral_constant<int, 16>{}, 16);
    if (j + 8 <= rank) add(std::integral_constant<int, 8>{}, 8);
    if (j + 4 <= rank) add(std::integral_constant<int, 4>{}, 4);
    if (j < rank) add(std::integral_constant<int, 3>{}, rank - j);
    const float ab = a_bias[col + i], wb = w0[col + i];
#pragma unroll
    for (int n = 0; n < R; ++n) {
      const float u = kx[n] * inv[n];
      const float a = 1.0f / (1.0f + expf(-(ax[n] + ab)));
      const float g = 1.0f / (1.0f + expf(-(wl[n] + wb)));
      if (row0 + n >= T) break;
      const size_t at = size_t(row0 + n) * D + col + i;
      w_out[at] = expf(-rate * g);
      au_out[at] = a * u;
      u_out[at] = u;
    }
  }
}

// The state of one head is dk x dv.  A wave owns 64 / G * NC value columns of one head of one sequence; the key dimension of a
// column is spread over G lanes (IPT = DKP / G entries each, DKP: dk padded with zeros), so a token costs a lane IPT
// multiply-adds for u^T S, a sum across its G lanes, 3 IPT multiply-adds for the update, IPT for o and another sum across the
// lanes; a lane has NC such columns.  U tokens' vectors are in registers or on their way.  Runs of a few tokens are bound by the state's own bytes instead:
// they take workgroups of 32 columns (whole lines of the state's rows; 8 sequences of one token: 13 us as waves of 4 columns).
// One sequence of 2,048 tokens, 32 heads of 64 x 64: 999 us with workgroups of 256 threads that staged the vectors through LDS
// (64 workgroups on 256 CUs, ten reads of LDS and a quarter of a barrier a token), 294 us here.
template <int DKP, int G, int NC, int U, int NT, int HOW>
__global__ void __launch_bounds__(NT)
    delta_scan_kernel(const float* __restrict__ r, int ldr, const float* __restrict__ k, int ldk,
                      const float* __restrict__ v, int ldv, const float* __restrict__ w, const float* __restrict__ au,
                      const float* __restrict__ u, float* __restrict__ o, int ldo, float* __restrict__ state,
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
  const size_t D = size_t(heads) * dk;
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
  float* st = state + ((size_t(slot) * heads + head) * dk) * dv;      // [slot][head][i][j]
  const bool fresh = seq_start[s] == 0;
  float S[NC][IPT];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int il = 0; il < IPT; ++il) {      // (what is not own takes part from zero and is left out of sums and stores)
      const int i = g * IPT + il / 4 * 4;
      S[c][il] = (entry_own<HOW>(i, il % 4, dk) && owns[c] && !fresh) ? st[size_t(entry_place<HOW>(i, il % 4, dk)) * dv + j[c]] : 0.f;
    }
  static_assert(U <= G, "lane n of a column keeps token n's output until the U tokens are stored together");
  const size_t col = size_t(head) * dk;
  const float *rp = r + size_t(r0) * ldr + col, *kp = k + size_t(r0) * ldk + col, *vp = v + size_t(r0) * ldv + size_t(head) * dv;
  const float *wp = w + size_t(r0) * D + col, *ap = au + size_t(r0) * D + col, *up = u + size_t(r0) * D + col;
  float* op = o + size_t(r0 + g) * ldo + size_t(head) * dv;
  float4 rv[U][Q], kv[U][Q], wv[U][Q], av[U][Q], uv[U][Q];
  float vv[U][NC];
  auto request = [&](int n) {      // the next row
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int i = g * IPT + 4 * q;
      uv[n][q] = load_own<HOW>(up, i, dk);      // (what is not own is left out of both sums)
      wv[n][q] = load_four<HOW>(wp, i, dk);
      av[n][q] = load_four<HOW>(ap, i, dk);
      kv[n][q] = load_four<HOW>(kp, i, dk);
      rv[n][q] = load_own<HOW>(rp, i, dk);
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) vv[n][c] = vp[j[c]];
    up += D; wp += D; ap += D; kp += ldk; rp += ldr; vp += ldv;
  };
  float out[NC] = {};
  auto walk = [&](int n) {
    float sa[NC] = {}, acc[NC] = {};
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const float ue[4] = {uv[n][q].x, uv[n][q].y, uv[n][q].z, uv[n][q].w};
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int c = 0; c < NC; ++c) sa[c] = fmaf(ue[e], S[c][4 * q + e], sa[c]);
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) sa[c] = group_sum<G>(sa[c]);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const float we[4] = {wv[n][q].x, wv[n][q].y, wv[n][q].z, wv[n][q].w}, ae[4] = {av[n][q].x, av[n][q].y, av[n][q].z, av[n][q].w};
      const float ke[4] = {kv[n][q].x, kv[n][q].y, kv[n][q].z, kv[n][q].w}, re[4] = {rv[n][q].x, rv[n][q].y, rv[n][q].z, rv[n][q].w};
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          float sn = we[e] * S[c][4 * q + e];
          sn = fmaf(-ae[e], sa[c], sn);
          sn = fmaf(ke[e], vv[n][c], sn);
          S[c][4 * q + e] = sn;
          acc[c] = fmaf(sn, re[e], acc[c]);
        }
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      acc[c] = group_sum<G>(acc[c]);
      out[c] = g == n ? acc[c] : out[c];
    }
  };
  auto store = [&]() {
#pragma unroll
    for (int c = 0; c < NC; ++c)
      if (owns[c]) op[j[c]] = out[c];
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
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int il = 0; il < IPT; ++il) {
      const int i = g * IPT + il / 4 * 4;
      if (entry_own<HOW>(i, il % 4, dk) && owns[c]) st[size_t(entry_place<HOW>(i, il % 4, dk)) * dv + j[c]] = S[c][il];
    }
}

}  // namespace kvcm

using namespace kvcm;

extern "C" {

// k, a_lin: 32-bit rows with heads*d columns each (at their own strides); low: 32-bit rows of `rank` columns;
// w2t [rank, heads*d] (the second step's matrix, transposed), a_bias, w0 [heads*d]; w_out, au_out, u_out [T, heads*d]: all 32-bit.
int kvcm_delta_prepare(const float* k, int ldk, const float* a_lin, int lda, const float* a_bias, const float* low, int ldlow,
                       const float* w2t, int rank, const float* w0, float* w_out, float* au_out, float* u_out, int T, int heads,
                       int d, hipStream_t s) {
  if (T == 0) return 0;
  KVCM_REQUIRE(T > 0 && heads > 0 && d > 0, "delta_prepare: bad sizes T=%d heads=%d d=%d", T, heads, d);
  KVCM_REQUIRE(rank > 0 && rank <= kDeltaMaxRank, "delta_prepare: a rank of %d is not supported (1 to %d)", rank, kDeltaMaxRank);
  KVCM_REQUIRE(ldk >= heads * d && lda >= heads * d && ldlow >= rank, "delta_prepare: row strides too small");
  const int groups = (heads + 3) / 4, threads = (heads + groups - 1) / groups * kWave;
  // Rows of a wave: as many as leave eight waves a CU, or six of four rows (us, one row / four / eight: 5 heads of 64, rank 64, 2,048 rows 15.7 / 10.4 / 13.9, 2 heads 6.5 / 8.4 / 12.2,
  // 32 heads of rank 8 55 / - / 30).
  const long long items = static_cast<long long>(T) * heads;
  const int rows = items >= 8 * 2048 ? 8 : items >= 4 * 1536 ? 4 : 1;
  const unsigned row_blocks = static_cast<unsigned>((static_cast<long long>(T) + rows - 1) / rows);
  const long long blocks = static_cast<long long>(row_blocks) * groups;
  KVCM_REQUIRE(blocks < (1ll << 31), "delta_prepare: too many rows");
  auto* kernel = rows == 8 ? delta_prepare_kernel<8> : rows == 4 ? delta_prepare_kernel<4> : delta_prepare_kernel<1>;
  kernel<<<static_cast<unsigned>(blocks), threads, 0, s>>>(k, ldk, a_lin, lda, a_bias, low, ldlow, w2t, rank, w0, w_out, au_out, u_out, heads, d, T,
                                                           row_blocks);
  return launch_status("delta_prepare");
}

// r, k [T, heads*dk], v [T, heads*dv] at their own strides; w, au, u [T, heads*dk] dense; o [T, >= heads*dv];
// state [slots, heads, dk, dv]; all 32-bit.  max_run: tokens of the longest run (what the lanes are dealt out by);
// one_order: not 0: a row's sums are taken in an order that depends on the key size alone.
int kvcm_delta_scan(const float* r, int ldr, const float* k, int ldk, const float* v, int ldv, const float* w, const float* au,
                    const float* u, float* o, int ldo, float* state, const int* run_start, const int* seq_start,
                    const int* state_slots, int S, int heads, int dk, int dv, int max_run, int one_order, hipStream_t s) {
  if (S == 0) return 0;
  KVCM_REQUIRE(S > 0 && heads > 0 && dk > 0 && dv > 0, "delta_scan: bad sizes S=%d heads=%d dk=%d dv=%d", S, heads, dk, dv);
  KVCM_REQUIRE(dk <= 256, "delta_scan: a key size of %d is not supported (up to 256)", dk);
  KVCM_REQUIRE(static_cast<long long>(heads) * ((dv + 3) / 4) < (1ll << 31), "delta_scan: too many heads");
  KVCM_REQUIRE(S <= 65535, "delta_scan: too many sequences for one launch (%d)", S);
  KVCM_REQUIRE(ldr >= heads * dk && ldk >= heads * dk && ldv >= heads * dv && ldo >= heads * dv, "delta_scan: row strides too small");
#define KVCM_DELTA_AS(DKP, G, NC, U, NT, HOW)                                                                                      \
  {                                                                                                                           \
    const int col_blocks = (dv + NT / G * NC - 1) / (NT / G * NC);                                                                      \
    delta_scan_kernel<DKP, G, NC, U, NT, HOW><<<dim3(heads * col_blocks, S), NT, 0, s>>>(r, ldr, k, ldk, v, ldv, w, au, u, o, ldo, \
                                                                                     state, run_start, seq_start,             \
                                                                                     state_slots, heads, dk, dv, col_blocks); \
  }
#define KVCM_DELTA(DKP, G, NC, U, NT)                                  \
  {                                                                \
    if (dk == DKP) KVCM_DELTA_AS(DKP, G, NC, U, NT, kRowFull)          \
    else if (dk % 4 == 0) KVCM_DELTA_AS(DKP, G, NC, U, NT, kRowWide)   \
    else KVCM_DELTA_AS(DKP, G, NC, U, NT, kRowPart)                    \
  }
  // A column over 16 lanes is the shorter chain, over 8 the fewer instructions: once waves of eight columns fill the SIMDs, those.
  // 2,048 tokens of one sequence / 8 sequences of 509, 32 heads of 64 x 64, us: 294 (16 lanes) / 374 and 261 (16 lanes; 8 lanes of two columns).
  // The other sizes, us, workgroups that share a token's vectors through LDS / so, 64 heads of 16 x 16, 64 of 32 x 32, 8 of 48 x 48, 32 of
  // 128 x 128: one sequence of 1,024 tokens 420 / 151, 454 / 155, 493 / 121, 1,045 / 343; 8 of 129 64 / 28, 70 / 52, 70 / 26, 563 / 311;
  // 8 single tokens 6.5 / 3.8, 6.7 / 4.4, 7.6 / 4.2, 43 / 16.
  // The lanes of a column are the order of its sums.  With one_order (32-bit storage, where a row's result depends on that row
  // alone) they follow from the key size, whatever the runs: 8 lanes from 33 to 64, 405 / 211 us; 16 beyond, also for single
  // tokens (8 rows, 32 heads of 128 x 128: 20 us, with 8 lanes and workgroups of 32 columns 14 us).
  // Beyond 128 a wave of four columns is bound by fetching the vectors, which each column needs whole: 8 x 509 tokens, 8 heads of
  // 256 x 256 2,335 us, 1,330 us with two columns a lane (1,850 as workgroups of 16 columns that shared them through LDS).
  const bool few = static_cast<long long>(S) * heads * ((dv + 7) / 8) < 1024;
  if (max_run >= 16) {
    if (dk < 4) KVCM_DELTA_AS(16, 4, 1, 4, kWave, kRowSingle)
    else if (dk <= 16) KVCM_DELTA(16, 4, 1, 4, kWave)
    else if (dk <= 32) KVCM_DELTA(32, 8, 1, 4, kWave)
    else if (dk <= 64 && few && !one_order) KVCM_DELTA(64, 16, 1, 8, kWave)
    else if (dk <= 64 && few) KVCM_DELTA(64, 8, 1, 4, kWave)
    else if (dk <= 64) KVCM_DELTA(64, 8, 2, 4, kWave)
    else if (dk <= 128) KVCM_DELTA(128, 16, 1, 4, kWave)
    else if (few) KVCM_DELTA(256, 16, 1, 1, kWave)
    else KVCM_DELTA(256, 16, 2, 1, kWave)
  } else {
    if (dk < 4) KVCM_DELTA_AS(16, 4, 1, 1, 128, kRowSingle)
    else if (dk <= 16) KVCM_DELTA(16, 4, 1, 1, 128)
    else if (dk <= 32) KVCM_DELTA(32, 8, 1, 1, 256)
    else if (dk <= 64) KVCM_DELTA(64, 8, 1, 1, 256)
    else if (dk <= 128 && one_order) KVCM_DELTA(128, 16, 1, 1, 256)
    else if (dk <= 128) KVCM_DELTA(128, 8, 1, 1, 256)
    else KVCM_DELTA(256, 16, 1, 1, 256)
  }
#undef KVCM_DELTA_AS
#undef KVCM_DELTA
  return launch_status("delta_scan");
}

}  // extern "C"
