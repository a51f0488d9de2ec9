// Attention over a sliding window of tokens and, beside them, one pooled key and value for every
// block of P tokens that lies wholly before the window; rotary positions by interleaved pairs on the
// first dims of a head; keys and values of different sizes.
//
//   row at position i sees   tokens j with 0 <= i - j < window
//                            blocks b with b*P + P - 1 <= i - window   (mean key, mean value of its P tokens)
//                            tokens j < keep_first (the sequence's first tokens stay visible beyond the window)
//                            with a chunk size instead of a window: tokens j <= i with j / chunk == i / chunk
//   and all of them share one softmax; score = (q . k) * scale_h with a factor per query head, and with a cap c > 0
//   score <- c tanh(score / c); then, with a slope per query head, score <- score - slope_h * (i - j) for token j (a bias
//   that grows with the distance; not offered together with pooled blocks, which have no one distance).  The output may be
//   multiplied with sigmoid(gate) before it is stored, element by element (32-bit gate logits of the output's shape) or head by
//   head (one logit each), and by a constant factor.  With a sink, one summand more joins the softmax's denominator: a key
//   without a value whose score is 0, or a number per query head that neither scale nor cap touches.
//
// Pages: keys [pages, kv_heads, B, d], values transposed [pages, kv_heads, dv, B] (as the other
// attentions of this library keep them).  Pooled entries are 32-bit and live with the page that holds
// their block's last token: [pages, kv_heads, E, d] and [pages, kv_heads, E, dv] with E = ceil(B / P)
// entries a page; block b, whose last token e = b*P + P - 1 lies in the sequence's page number e / B,
// is entry b - floor((e / B) * B / P) there.  An entry is made by the step that stores its block's last
// token, from the P keys and values as the pages hold them, added in ascending position: it does not
// depend on how the prompt was cut.  Giving a page back gives its entries back.
//
// Waves per row and query head, or group of query heads; blocks are walked 64 at a time from block 0, tokens 64 at a time in
// chunks that start at absolute multiples of 64, with a running maximum: a row's result is a fixed
// sequence of operations on its own keys, whatever else the launch holds and whichever pages it reads.
#include <algorithm>
#include <cfloat>
#include <type_traits>

#include "common.h"
#include "kvcm_hip.h"

namespace kvcm {

constexpr int kWpWaves = 4;
constexpr int kWpMaxValueDim = 512;

// ------------------------------------------------------------------------- angles of a step
// cos_sin[t, i] = (cos, sin) of position * base^(-2i/dims).  The angle is formed in double precision
// (a 32-bit product of a position in the thousands loses the low bits of the angle).
__global__ void rotary_pairs_table_kernel(const int* __restrict__ positions, float2* __restrict__ cos_sin, int T, int half,
                                          double log_base, int dims) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= T * half) return;
  const int t = idx / half, i = idx % half;
  const double freq = exp(-log_base * (2.0 * i) / double(dims));
  const double a = double(positions[t]) * freq;
  cos_sin[idx] = float2{static_cast<float>(cos(a)), static_cast<float>(sin(a))};
}

// cos_sin[t, i] = factor * (cos, sin) of position * freqs[i], for rotations whose frequencies are not a plain power
// law (rescaled for longer contexts pair by pair): the caller brings them as a table, in double precision.
__global__ void rotary_freq_table_kernel(const int* __restrict__ positions, const double* __restrict__ freqs,
                                         float2* __restrict__ cos_sin, int T, int half, double factor) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= T * half) return;
  const double a = double(positions[idx / half]) * freqs[idx % half];
  cos_sin[idx] = float2{static_cast<float>(factor * cos(a)), static_cast<float>(factor * sin(a))};
}

// ------------------------------------------------------- rotation and the page write of a step
// src [T, nh*d + nkv*d + nkv*dv] 32-bit (q | k | v); or q alone there and (k | v) in rows of their own, kv_src
// [T, nkv*d + nkv*dv] (a query that is made by a later product than the keys).  q (rotated) -> q_out [T, nh*d]; k
// (rotated) and v -> their page slot; a row without a slot reads no k and no v.  halves 0: the pair (2i, 2i+1),
// i < rot/2, is turned; halves 1: the pair (i, i + rot/2); the rest passes.
template <class T>
__global__ void __launch_bounds__(256)
    rotate_store_kernel(const float* __restrict__ src, int ld, const float* __restrict__ kv_src, int ldkv,
                        const float2* __restrict__ cos_sin, int rot, int halves,
                        const int* __restrict__ slots, T* __restrict__ q_out, int ldq, T* __restrict__ kcache,
                        T* __restrict__ vcache, int nh, int nkv, int d, int dv, int B) {
  const int row = blockIdx.x;
  const float* rq = src + size_t(row) * ld;
  const float* rk = kv_src ? kv_src + size_t(row) * ldkv : rq + size_t(nh) * d;      // (k | v) of the row
  const float2* cs = cos_sin + size_t(row) * (rot / 2);
  const int slot = slots ? slots[row] : -1;
  const int heads = slot >= 0 ? nh + nkv : nh;
  // grid (rows, 1): one workgroup does a whole row; grid (rows, nh + nkv + 1), for steps of few rows: workgroup y does
  // head y of q | k and the last one the values (the same operations on every element either way)
  int e0 = 0, e1 = heads * d;
  bool values = true;
  if (gridDim.y > 1) {
    const int part = blockIdx.y;
    values = part == nh + nkv;
    e0 = values || part >= heads ? 0 : part * d;
    e1 = values || part >= heads ? 0 : e0 + d;
  }
  for (int e = e0 + threadIdx.x; e < e1; e += blockDim.x) {
    const int head = e / d, i = e % d;
    const float* r = head < nh ? rq + size_t(head) * d : rk + size_t(head - nh) * d;      // this head's entries
    float x = r[i];
    if (i < rot) {      // rot is even: the partner lies inside the rotated part too
      const int hr = rot / 2;
      const bool second = halves ? i >= hr : (i & 1);
      const float y = r[halves ? (second ? i - hr : i + hr) : (i ^ 1)];
      const float2 a = cs[halves ? (second ? i - hr : i) : i / 2];
      x = second ? __fmaf_rn(x, a.x, __fmul_rn(y, a.y)) : __fmaf_rn(x, a.x, -__fmul_rn(y, a.y));
    }
    if (head < nh) store_f(q_out + size_t(row) * ldq + e, x);
    else if (slot >= 0) store_f(kcache + ((size_t(slot / B) * nkv + (head - nh)) * B + slot % B) * d + i, x);
  }
  if (slot < 0 || !values) return;
  const float* v = rk + size_t(nkv) * d;
  for (int e = threadIdx.x; e < nkv * dv; e += blockDim.x) {
    const int head = e / dv, i = e % dv;
    store_f(vcache + ((size_t(slot / B) * nkv + head) * dv + i) * B + slot % B, v[e]);
  }
}

// rotate_store with what some attentions do to the projection before the rotation.  q and k are each divided by the
// root mean square over their WHOLE stretch of the row (all heads at once, eps inside the root) and multiplied by a weight
// of that size (wq, wk; null: that stretch passes as it is).  v may be blended with the values another layer made for the
// same row, v <- (1 - mix) v + mix * v_other (v_other null: none); v_keep (null: none) receives the row's values as the
// projection made them, for later layers to blend with.  What is stored in the pages is the blended v.
// Grid (rows, parts).  parts 1: one workgroup does a whole row.  parts nh + nkv + 1, for steps of few rows: workgroup y
// does head y of q | k (it sums the squares of that head's whole stretch itself, in the same order, so the bits are those
// of the one-workgroup form) and the last one the values.
constexpr int kNormRotateFewRows = 16;

template <class T>
__global__ void __launch_bounds__(256)
    norm_rotate_store_kernel(const float* __restrict__ src, int ld, const float* __restrict__ wq, const float* __restrict__ wk,
                             float eps, const float* __restrict__ v_other, int ldvo, float mix, float* __restrict__ v_keep,
                             int ldvk, const float2* __restrict__ cos_sin, int rot, int halves, const int* __restrict__ slots,
                             T* __restrict__ q_out, int ldq, T* __restrict__ kcache, T* __restrict__ vcache, int nh, int nkv,
                             int d, int dv, int B) {
  __shared__ float scratch[256 / kWave + 1];
  const int row = blockIdx.x;
  const float* r = src + size_t(row) * ld;
  const int nq = nh * d, nk = nkv * d;
  int e0 = 0, e1 = nq + nk;
  bool values = true;
  if (gridDim.y > 1) {
    const int part = blockIdx.y;
    values = part == nh + nkv;
    e0 = values ? 0 : part * d;
    e1 = values ? 0 : e0 + d;
  }
  const float2* cs = cos_sin + size_t(row) * (rot / 2);
  const int slot = slots ? slots[row] : -1;
  // an entry of q or k, the one it is turned with, their weights and the angle: a thread's first on their way before the sums (us, asked for behind
  // them / so: 32 heads of 64 over 4, 8 rows 4.4 / 3.7, 64 rows 9.5 / 7.6, 2,048 rows 21.8 / 19.5; 32 of 128 over 8 5.3 / 4.1, 17.8 / 13.5, 54.5 / 48.8)
  struct Entry {
    float x, y, wx, wy;
    float2 turn;
  };
  const int hr = rot / 2;
  auto gather = [&](int e, Entry& en) {
    const int i = e % d;
    const bool second = halves ? i >= hr : (i & 1), turned = i < rot;
    const int to = !turned ? e : halves ? (second ? e - hr : e + hr) : e - i + (i ^ 1);
    const float* w = e < nq ? wq : wk;
    const int base = e < nq ? 0 : nq;
    en.x = r[e];
    en.y = r[to];
    en.wx = w ? w[e - base] : 1.f;
    en.wy = w ? w[to - base] : 1.f;
    if (turned) en.turn = cs[halves ? (second ? i - hr : i) : i / 2];
  };
  Entry first;
  if (e0 + int(threadIdx.x) < e1) gather(e0 + threadIdx.x, first);
  float inv_q = 1.f, inv_k = 1.f;
  if (wq && e0 < nq && e1 > e0) {
    float ss = 0.f;
#pragma unroll 8
    for (int e = threadIdx.x; e < nq; e += 256) ss = fmaf(r[e], r[e], ss);
    inv_q = 1.0f / sqrtf(block_sum<256>(ss, scratch) / float(nq) + eps);
  }
  if (wk && e1 > nq) {
    float ss = 0.f;
    for (int e = threadIdx.x; e < nk; e += 256) ss = fmaf(r[nq + e], r[nq + e], ss);
    inv_k = 1.0f / sqrtf(block_sum<256>(ss, scratch) / float(nk) + eps);
  }
  auto finish = [&](int e, const Entry& en) {
    const int head = e / d, i = e % d;
    const bool normed = e < nq ? wq : wk;
    const float inv = e < nq ? inv_q : inv_k;
    float x = normed ? en.x * inv * en.wx : en.x;
    if (i < rot) {
      const float y = normed ? en.y * inv * en.wy : en.y;
      const bool second = halves ? i >= hr : (i & 1);
      x = second ? __fmaf_rn(x, en.turn.x, __fmul_rn(y, en.turn.y)) : __fmaf_rn(x, en.turn.x, -__fmul_rn(y, en.turn.y));
    }
    if (head < nh) store_f(q_out + size_t(row) * ldq + e, x);
    else if (slot >= 0) store_f(kcache + ((size_t(slot / B) * nkv + (head - nh)) * B + slot % B) * d + i, x);
  };
  if (e0 + int(threadIdx.x) < e1) finish(e0 + threadIdx.x, first);
  for (int e = e0 + threadIdx.x + 256; e < e1; e += 256) {
    Entry en;
    gather(e, en);
    finish(e, en);
  }
  if (!values) return;
  const float* v = r + nq + nk;
  for (int e = threadIdx.x; e < nkv * dv; e += 256) {
    float x = v[e];
    if (v_keep) v_keep[size_t(row) * ldvk + e] = x;
    if (v_other) x = __fmaf_rn(mix, v_other[size_t(row) * ldvo + e], __fmul_rn(1.0f - mix, x));
    if (slot >= 0) store_f(vcache + ((size_t(slot / B) * nkv + e / dv) * dv + e % dv) * B + slot % B, x);
  }
}

// ------------------------------------------------------------------- pooled entries of a step
// A row whose position is the last of a block of P makes that block's entry from the pages.  A wave looks at R rows (one of
// them, in a run, ends a block where R <= P) and makes keys or values (blockIdx.z) of one kv head, AHEAD tokens' pages, then their
// values, requested before the first is added, in order.  A workgroup per row that waited for every token's value in turn took
// 86 us for a prompt of 2,048 tokens in blocks of 64, four heads of 64; 13 us so.
// A wave makes the mean key (or value) of the block that ends at position p, whose token lies in `slot`.
template <class T, int AHEAD>
__device__ __forceinline__ void pool_entry(const T* kcache, const T* vcache, float* pk, float* pv, const int* table, bool keys, int p, int slot, int kvh,
                                           int lane, int nkv, int d, int dv, int B, int P, int E) {
  const int first = p - P + 1, entry = p / P - (p / B * B) / P;
  const size_t at = (size_t(slot / B) * nkv + kvh) * E + entry;
  const float inv = 1.0f / float(P);
  for (int i = lane; i < (keys ? d : dv); i += kWave) {
    float acc = 0.f;
    for (int t0 = first; t0 <= p; t0 += AHEAD) {
      float x[AHEAD];
#pragma unroll
      for (int a = 0; a < AHEAD; ++a) {
        const int t = t0 + a <= p ? t0 + a : p;
        const size_t page = size_t(table[t / B]) * nkv + kvh;
        x[a] = load_f(keys ? kcache + (page * B + t % B) * d + i : vcache + (page * dv + i) * B + t % B);
      }
#pragma unroll
      for (int a = 0; a < AHEAD; ++a) acc = t0 + a <= p ? acc + x[a] : acc;
    }
    (keys ? pk[at * d + i] : pv[at * dv + i]) = acc * inv;
  }
}

template <class T, int AHEAD>
__global__ void __launch_bounds__(kWave)
    pool_update_kernel(const T* __restrict__ kcache, const T* __restrict__ vcache, float* __restrict__ pk,
                       float* __restrict__ pv, const int* __restrict__ tables, int table_stride,
                       const int* __restrict__ row_seq, const int* __restrict__ positions, const int* __restrict__ slots,
                       int rows, int R, int nkv, int d, int dv, int B, int P, int E) {
  const int kvh = blockIdx.y, lane = threadIdx.x, row0 = blockIdx.x * R;
  const bool keys = blockIdx.z == 0;
  const int mine = row0 + lane < rows ? row0 + lane : rows - 1;
  const bool ends = lane < R && row0 + lane < rows && slots[mine] >= 0 && (positions[mine] + 1) % P == 0;
  for (unsigned long long left = __ballot(ends); left != 0; left &= left - 1) {
    const int row = row0 + __builtin_ctzll(left);
    const int p = positions[row], slot = slots[row];
    const int* table = tables + size_t(row_seq[row]) * table_stride;
    pool_entry<T, AHEAD>(kcache, vcache, pk, pv, table, keys, p, slot, kvh, lane, nkv, d, dv, B, P, E);
  }
}

// -------------------------------------------------------------------------------- attention
// dot of a 32-bit vector (LDS) with a stored row, 16 bytes of the row at a time where its length allows
template <class T> struct RowPiece;
template <> struct RowPiece<float> { static constexpr int N = 4; };
template <> struct RowPiece<bf16_t> { static constexpr int N = 8; };

__device__ __forceinline__ void unpack_piece(const float* p, float* f) {
  const float4 v = *reinterpret_cast<const float4*>(p);
  f[0] = v.x; f[1] = v.y; f[2] = v.z; f[3] = v.w;
}
__device__ __forceinline__ void unpack_piece(const bf16_t* p, float* f) {
  const uint4 v = *reinterpret_cast<const uint4*>(p);
  f[0] = bf16_bits_to_float(v.x & 0xffffu); f[1] = bf16_bits_to_float(v.x >> 16);
  f[2] = bf16_bits_to_float(v.y & 0xffffu); f[3] = bf16_bits_to_float(v.y >> 16);
  f[4] = bf16_bits_to_float(v.z & 0xffffu); f[5] = bf16_bits_to_float(v.z >> 16);
  f[6] = bf16_bits_to_float(v.w & 0xffffu); f[7] = bf16_bits_to_float(v.w >> 16);
}

// (four pieces of the row are requested before the first is multiplied: a load per trip of the loop would wait for
// each one in turn)
template <class T>
__device__ __forceinline__ float dot_row(const float* qs, const T* kp, int d, bool wide) {
  constexpr int N = RowPiece<T>::N;
  float s = 0.f;
  if (wide) {
    int i = 0;
    for (; i + 4 * N <= d; i += 4 * N) {
      float f[4][N];
#pragma unroll
      for (int g = 0; g < 4; ++g) unpack_piece(kp + i + g * N, f[g]);
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int e = 0; e < N; ++e) s = fmaf(qs[i + g * N + e], f[g][e], s);
    }
    for (; i < d; i += N) {
      float f[N];
      unpack_piece(kp + i, f);
#pragma unroll
      for (int e = 0; e < N; ++e) s = fmaf(qs[i + e], f[e], s);
    }
  } else {
    for (int i = 0; i < d; ++i) s = fmaf(qs[i], load_f(kp + i), s);
  }
  return s;
}

// One workgroup of four waves per (row, query head).  The row's chunks (pooled blocks 64 at a time from block 0,
// then tokens in chunks that start at absolute multiples of 64) are dealt to the waves in turn by their number;
// each wave keeps a running maximum over its chunks and the four results are merged at the end in wave order.
// Inside a chunk a lane takes one key for the scores; for the values a lane takes value columns and reads the
// tokens of its column 16 bytes at a time (values are stored transposed: a column's tokens lie side by side).
template <class T>
__global__ void __launch_bounds__(kWpWaves* kWave)
    attention_window_pool_kernel(const T* __restrict__ q, int ldq, T* __restrict__ out, int ldo,
                                 const T* __restrict__ kcache, const T* __restrict__ vcache,
                                 const float* __restrict__ pk, const float* __restrict__ pv,
                                 const int* __restrict__ tables, int table_stride, const int* __restrict__ row_seq,
                                 const int* __restrict__ ctx_lens, const float* __restrict__ head_scale,
                                 const float* __restrict__ dist_slope, const float* __restrict__ gate, int ldg,
                                 int nh, int nkv, int d, int dv, int B, float scale, int window, int P, int E, int keep_first,
                                 float softcap, int chunk, int sink, const float* __restrict__ sink_logit, int gate_heads, float out_scale) {
  extern __shared__ float lds[];      // [d] q * scale * head_scale[h]; [waves][64] probabilities; [waves][dv + 2] results
  constexpr int N = RowPiece<T>::N, COLS = kWpMaxValueDim / kWave;
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int row = blockIdx.x / nh, head = blockIdx.x % nh;
  float* qs = lds;
  float* ps = lds + d + wave * kWave;
  float* merge = lds + d + kWpWaves * kWave;
  {
    const float f = head_scale ? scale * head_scale[head] : scale;
    for (int i = threadIdx.x; i < d; i += kWpWaves * kWave) qs[i] = load_f(q + size_t(row) * ldq + size_t(head) * d + i) * f;
  }
  __syncthreads();
  const int kvh = head / (nh / nkv);
  const int ctx = ctx_lens[row];
  T* orow = out + size_t(row) * ldo + size_t(head) * dv;
  if (ctx <= 0) {
    for (int i = threadIdx.x; i < dv; i += kWpWaves * kWave) store_f(orow + i, 0.f);
    return;
  }
  const int* table = tables + size_t(row_seq[row]) * table_stride;
  const int first = chunk > 0 ? (ctx - 1) / chunk * chunk : (window > 0 && ctx > window) ? ctx - window : 0;
  const int blocks = (P > 0 && window > 0 && ctx - window >= P) ? (ctx - window) / P : 0;      // those that end at or before ctx - 1 - window
  const int block_chunks = (blocks + kWave - 1) / kWave;
  // tokens at the sequence's start that stay visible beyond the window: those of them that lie before the window's
  // first token get chunks of their own, from token 0, walked after the blocks and before the window
  const int kept = keep_first < first ? keep_first : first;
  const int head_chunks = block_chunks + (kept + kWave - 1) / kWave;
  const int first_chunk = first / kWave, chunks = head_chunks + ((ctx - 1) / kWave - first_chunk + 1);
  const float inv_cap = softcap > 0.f ? 1.0f / softcap : 0.f;
  const float slope = dist_slope ? dist_slope[head] : 0.f;
  const bool wide_k = (d % N == 0) && (reinterpret_cast<uintptr_t>(kcache) % 16 == 0);
  const bool wide_pk = (d % 4 == 0);
  const bool wide_v = (B % N == 0) && (reinterpret_cast<uintptr_t>(vcache) % 16 == 0);
  const size_t khead = size_t(B) * d, kpage = khead * nkv;
  const size_t vhead = size_t(B) * dv, vpage = vhead * nkv;

  float m = -INFINITY, l = 0.f;
  float o[COLS];
#pragma unroll
  for (int i = 0; i < COLS; ++i) o[i] = 0.f;

  for (int c = wave; c < chunks; c += kWpWaves) {
    const bool pooled = c < block_chunks, early = !pooled && c < head_chunks;
    const int c0 = pooled ? c * kWave : early ? (c - block_chunks) * kWave : (first_chunk + (c - head_chunks)) * kWave;
    // the stretch of tokens this chunk may see: the kept first tokens before the window, or the window
    const int lo = early ? 0 : first, hi = early ? kept : ctx;
    const int t = c0 + lane;
    float s = -INFINITY;
    int page = 0, entry = 0;
    bool valid;
    if (pooled) {
      valid = t < blocks;
      if (valid) {
        const int e = t * P + P - 1, pgi = e / B;
        page = table[pgi];
        entry = t - (pgi * B) / P;
        s = dot_row<float>(qs, pk + ((size_t(page) * nkv + kvh) * E + entry) * d, d, wide_pk);
      }
    } else {
      valid = t >= lo && t < hi;
      if (valid) s = dot_row<T>(qs, kcache + size_t(table[t / B]) * kpage + kvh * khead + size_t(t % B) * d, d, wide_k);
    }
    if (softcap > 0.f && valid) s = softcap * tanhf(s * inv_cap);
    if (dist_slope && valid) s = fmaf(-slope, float(ctx - 1 - t), s);
    const float m_new = fmaxf(m, wave_max(s));
    const float alpha = expf(m - m_new);
    const float p = valid ? expf(s - m_new) : 0.f;
    l = l * alpha + wave_sum(p);
#pragma unroll
    for (int i = 0; i < COLS; ++i) o[i] *= alpha;
    m = m_new;
    __builtin_amdgcn_wave_barrier();
    ps[lane] = p;
    __builtin_amdgcn_wave_barrier();
    if (pooled) {
      const int n = blocks - c0 < kWave ? blocks - c0 : kWave;
      for (int j = 0; j < n; ++j) {
        const int page_j = __shfl(page, j, kWave), entry_j = __shfl(entry, j, kWave);
        const float* vp = pv + ((size_t(page_j) * nkv + kvh) * E + entry_j) * dv;
        const float pj = ps[j];
#pragma unroll
        for (int i = 0; i < COLS; ++i) {
          const int cc = lane + i * kWave;
          if (cc < dv) o[i] = fmaf(pj, vp[cc], o[i]);
        }
      }
    } else {
      const int j_lo = lo > c0 ? lo - c0 : 0;
      const int j_hi = hi - c0 < kWave ? hi - c0 : kWave;
      if (wide_v) {
        // all of the chunk's pieces (N tokens of one page each) are requested at once, from places clamped into the
        // context; probabilities of tokens before the window are zero, values beyond the context are cut
        // (pages that the window has passed may have been given back: nothing before the window's first piece is read)
        const int last_piece = ((hi - 1) / N) * N, first_piece = (lo / N) * N;
#pragma unroll
        for (int i = 0; i < COLS; ++i) {
          if (i * kWave >= dv) break;      // the same for every lane: 64 columns at a time, each with its own trip of loads
          const int cc = lane + i * kWave;
          const int col = cc < dv ? cc : dv - 1;
          float f[kWave / N][N];
#pragma unroll
          for (int g = 0; g < kWave / N; ++g) {
            const int tg = c0 + g * N < first_piece ? first_piece : c0 + g * N;
            const int tj = tg < last_piece ? tg : last_piece;
            unpack_piece(vcache + size_t(table[tj / B]) * vpage + kvh * vhead + size_t(col) * B + tj % B, f[g]);
          }
          float acc = o[i];
#pragma unroll
          for (int g = 0; g < kWave / N; ++g)
#pragma unroll
            for (int e = 0; e < N; ++e) {
              const int j = g * N + e;
              acc = fmaf(ps[j], (j >= j_lo && j < j_hi) ? f[g][e] : 0.f, acc);
            }
          if (cc < dv) o[i] = acc;
        }
      } else {
        for (int j = j_lo; j < j_hi; ++j) {
          const int tj = c0 + j;
          const T* vp = vcache + size_t(table[tj / B]) * vpage + kvh * vhead + tj % B;
          const float pj = ps[j];
#pragma unroll
          for (int i = 0; i < COLS; ++i) {
            const int cc = lane + i * kWave;
            if (cc < dv) o[i] = fmaf(pj, load_f(vp + size_t(cc) * B), o[i]);
          }
        }
      }
    }
  }
  // merge the waves' results in wave order
  float* mine = merge + wave * (dv + 2);
#pragma unroll
  for (int i = 0; i < COLS; ++i) {
    const int cc = lane + i * kWave;
    if (cc < dv) mine[cc] = o[i];
  }
  if (lane == 0) {
    mine[dv] = m;
    mine[dv + 1] = l;
  }
  __syncthreads();
  const float sl = sink_logit ? sink_logit[head] : 0.f;
  float mm = sink ? sl : -INFINITY;
#pragma unroll
  for (int w = 0; w < kWpWaves; ++w) mm = fmaxf(mm, merge[w * (dv + 2) + dv]);
  float wgt[kWpWaves], ll = sink ? expf(sl - mm) : 0.f;
#pragma unroll
  for (int w = 0; w < kWpWaves; ++w) {
    const float mw = merge[w * (dv + 2) + dv];
    wgt[w] = mw == -INFINITY ? 0.f : expf(mw - mm);
    ll = fmaf(merge[w * (dv + 2) + dv + 1], wgt[w], ll);
  }
  const float* gr = gate ? gate + size_t(row) * ldg + (gate_heads ? head : head * dv) : nullptr;
  for (int cc = threadIdx.x; cc < dv; cc += kWpWaves * kWave) {
    float acc = 0.f;
#pragma unroll
    for (int w = 0; w < kWpWaves; ++w) acc = fmaf(merge[w * (dv + 2) + cc], wgt[w], acc);
    float res = acc / ll * out_scale;
    if (gate) res *= 1.0f / (1.0f + expf(-gr[gate_heads ? 0 : cc]));      // a gate per element of the output, or one per head
    store_f(orow + cc, res);
  }
}

// ------------------------------------------------------------- attention of a row's query heads together
// The same attention for heads of bfloat16 whose sizes are multiples of 8: a workgroup takes a row and up to sixteen query
// heads of one kv head, a wave walks chunks as above, on the matrix cores: S^T = K Q^T (64 keys x 16 heads, fragments straight
// from the pages; a tile's 16 keys are dealt out so that a lane's eight of 32 are consecutive), softmax in 32-bit on the
// accumulators, O^T += V^T P^T with each 32-bit probability as the exact sum of three bfloat16 pieces.  Pooled entries, which are
// 32-bit, are multiplied in 32-bit by v_mfma_f32_16x16x4.
// Bound by the waits for the table, then for keys and values (asked for at once), and by the merge.  The workgroup per row and
// query head above, whose dots and sums over values are a thousand vector instructions for each chunk and head and which reads
// the keys once per head, took 19.0 us a step of 8 rows of 32 heads over 4 kv heads of 64 in a window of 512 (sixteen waves in
// place of four: 14.5 us), this 12.2 us; 1,100 such rows at once 814 us then, 137 us now; heads of 128 over 8 kv heads in a
// window of 1,024 with pooled blocks 29.7 us then, 24.8 us now.
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
typedef float any_four __attribute__((ext_vector_type(4), aligned(4)));      // (pooled entries may lie at any float)

// the upper halves of two floats
__device__ __forceinline__ uint32_t upper_halves(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
// what a probability's upper half leaves of it, or, where that is nothing of a probability above zero, the least bfloat16
// (nothing beside the rest of it, but times an infinite value it is not the NaN that zero would make)
__device__ __forceinline__ float below_upper(float x) {
  return fmaxf(x - __uint_as_float(__float_as_uint(x) & 0xFFFF0000u), fminf(x, 1.17549435e-38f));
}

// What steps in which every sequence runs one row do between the projection and the attention: the workgroup of a row and a kv head, which
// alone needs and stores them, takes its channels from the projection's row [q | k | v] and gives them, with the operations of the kernels
// above and of short_conv.hip in their order: the convolution (its state moved on), the rotation, the page's new key and value, and at last the
// pooled entry where one is due.  Bound by the trips to memory one after the other; the first keys and values and what the front
// needs are on their way together.  Four launches as one, 8 rows of 32 heads over 4 kv heads of 64, window 512, blocks of 64, 4 taps: in a row
// of such launches 540 tokens 16.7 -> 15.6 us, 60 tokens 14.0 -> 11.4; between a decoder's other launches 22.8 -> 16.9.  Heads of 128, whose first
// keys and values the registers do not hold beside it, lose (8 rows, 30.1 -> 31.2), and so do norms over all heads in its place (13.4 -> 13.8).
// With the front the kernel has 168 registers, 14 of which are spilled (60 bytes a lane), without it 138 and none: a workgroup fills its CU, which is
// why more workgroups than CUs run the launches one by one (kvcm_attention_window_pool_rows_takes).
struct WpFront {
  const float* src; int ld;
  const float* conv_w; const float* conv_bias; float* conv_state; const int* state_slots; int taps;
  const float2* cos_sin; int rot, halves;
  const int* slots;
};

// what an entry of the front needs from memory besides its convolution's state
constexpr int kFrontTaps = 8;
struct FrontEntry {
  float x, bias, w[kFrontTaps];
  float2 turn;
};

// DP: key size padded to a multiple of 32; DVT: tiles of 16 value columns.  FRONT: q comes from `fr` (a workgroup per row and kv head: at most
// 16 query heads each); no cap, kept tokens, chunk, sink, slope or gate.
template <int DP, int DVT, int WAVES, bool FRONT>
__global__ void __launch_bounds__(WAVES* kWave)
    attention_window_pool_heads_kernel(const uint16_t* __restrict__ q, int ldq, uint16_t* __restrict__ out, int ldo,
                                       const uint16_t* kcache, const uint16_t* vcache,
                                       const float* pk, const float* pv,
                                       const int* __restrict__ tables, int table_stride, const int* __restrict__ row_seq,
                                       const int* __restrict__ ctx_lens, const float* __restrict__ head_scale,
                                       const float* __restrict__ dist_slope, const float* __restrict__ gate, int ldg,
                                       int nh, int nkv, int d, int dv, int B, float scale, int window, int P, int E, int keep_first,
                                       float softcap, int chunk, int sink, const float* __restrict__ sink_logit, int gate_heads, float out_scale,
                                       const WpFront fr) {
  if constexpr (FRONT) softcap = 0.f, keep_first = chunk = sink = 0, out_scale = 1.0f;
  constexpr int KS = DP / 32, DVP = DVT * 16, PITCH = DVP + 4;
  constexpr bool kAhead = FRONT;      // the first chunk's keys and values asked for before the front
  __shared__ __attribute__((aligned(16))) float parts[WAVES][16][PITCH];      // a wave's sums, head by head
  __shared__ float maxima[WAVES][16], sums[WAVES][16], weights[WAVES][16];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
  const int col = lane % 16, quad = lane / 16;
  const int group = nh / nkv, head_tiles = (group + 15) / 16;
  const int row = blockIdx.x, kvh = blockIdx.y / head_tiles, in_group = blockIdx.y % head_tiles * 16;
  const int head0 = kvh * group + in_group, heads = group - in_group < 16 ? group - in_group : 16;
  const int my_head = head0 + (col < heads ? col : 0);
  const int ctx = ctx_lens[row], seq = row_seq[row];
  uint16_t* orow = out + size_t(row) * ldo + size_t(head0) * dv;
  // the front's entries: q of the heads, k, v.  The first of a thread is on its way before the context, the pages and the state's place are known.
  const int nq = nh * d, nk = nkv * d, mine = heads * d, entries = mine + d + dv;
  const float* r = FRONT ? fr.src + size_t(row) * fr.ld : nullptr;
  const int new_slot = FRONT ? fr.slots[row] : -1;
  const auto channel = [&](int e) { return e < mine ? head0 * d + e : e < mine + d ? nq + kvh * d + (e - mine) : nq + nk + kvh * dv + (e - mine - d); };
  const auto turned_with = [&](int i) { return !fr.halves ? i ^ 1 : i >= fr.rot / 2 ? i - fr.rot / 2 : i + fr.rot / 2; };
  const auto gather = [&](int e, FrontEntry& en) {
    const int ch = channel(e);
    en.x = r[ch];
    en.bias = fr.conv_bias ? fr.conv_bias[ch] : 0.f;
#pragma unroll
    for (int j = 0; j < kFrontTaps; ++j) en.w[j] = fr.conv_w[size_t(ch) * fr.taps + (j < fr.taps ? j : 0)];
    if (e < mine + d) {
      const int i = e % d, j = i < fr.rot ? turned_with(i) : i;
      if (i < fr.rot) en.turn = fr.cos_sin[size_t(row) * (fr.rot / 2) + (fr.halves ? (i < j ? i : j) : i / 2)];
    }
  };
  FrontEntry early_entry;
  if constexpr (FRONT) {
    if (tid < entries) gather(tid, early_entry);
  }
  if (ctx <= 0) {
    for (int i = tid; i < heads * dv; i += WAVES * kWave) orow[i] = 0;
    return;
  }
  const int* table = tables + size_t(seq) * table_stride;
  const float f = head_scale ? scale * head_scale[my_head] : scale;
  const float slope = !FRONT && dist_slope ? dist_slope[my_head] : 0.f;
  const float inv_cap = softcap > 0.f ? 1.0f / softcap : 0.f;

  const int first = chunk > 0 ? (ctx - 1) / chunk * chunk : (window > 0 && ctx > window) ? ctx - window : 0;
  const int blocks = (P > 0 && window > 0 && ctx - window >= P) ? (ctx - window) / P : 0;
  const int block_chunks = (blocks + kWave - 1) / kWave;
  const int kept = keep_first < first ? keep_first : first;
  const int head_chunks = block_chunks + (kept + kWave - 1) / kWave;
  const int first_chunk = first / kWave, chunks = head_chunks + ((ctx - 1) / kWave - first_chunk + 1);

  // the chunk's tokens (place j of a lane below): the kept first tokens before the window, or the window; [lo, hi) is what it sees
  const auto stretch = [&](int c, int& c0, int& lo, int& hi) {
    const bool early = c < head_chunks;
    c0 = early ? (c - block_chunks) * kWave : (first_chunk + (c - head_chunks)) * kWave;
    lo = early ? 0 : first;
    hi = early ? kept : ctx;
  };
  uint4 kreg[2][2][KS], vreg[2][DVT];
  // A lane looks up the page of the token at its place, clamped into the stretch (pages that the window has passed may have been given back).
  const auto ask = [&](int c) {
    int c0, lo, hi;
    stretch(c, c0, lo, hi);
    const int at = c0 + lane < lo ? lo : c0 + lane < hi ? c0 + lane : hi - 1;
    const int page_no = at / B, slot = at - page_no * B, page = table[page_no];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int from = 32 * g + 8 * (col / 4) + 4 * t + col % 4;
        const uint16_t* src = kcache + ((size_t(__shfl(page, from, kWave)) * nkv + kvh) * B + __shfl(slot, from, kWave)) * d;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const int k = ks * 32 + quad * 8;
          kreg[g][t][ks] = *reinterpret_cast<const uint4*>(src + (k < d ? k : 0));
        }
      }
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int from = 32 * g + 8 * quad;
      const uint16_t* src = vcache + (size_t(__shfl(page, from, kWave)) * nkv + kvh) * dv * B + __shfl(slot, from, kWave) / 8 * 8;
#pragma unroll
      for (int vt = 0; vt < DVT; ++vt) {
        const int dim = vt * 16 + col;
        vreg[g][vt] = *reinterpret_cast<const uint4*>(src + size_t(dim < dv ? dim : dv - 1) * B);
      }
    }
    __builtin_amdgcn_sched_barrier(0);      // (all of them on their way before the first is waited for)
  };

  // the front's values, where the waves' sums come later: 32-bit, then as stored (q of the heads, k, v)
  constexpr int kMostFront = 16 * DP + DP + DVP;
  float* const xs = &parts[0][0][0];
  uint16_t* const stored = reinterpret_cast<uint16_t*>(xs + kMostFront);
  static_assert(sizeof(parts) >= size_t(kMostFront) * (sizeof(float) + sizeof(uint16_t)), "the front's values lie where the sums come");
  int c = wave;
  if constexpr (FRONT) {
    const int C = nq + nk + nkv * dv, state_slot = fr.state_slots ? fr.state_slots[seq] : -1;
    if (kAhead && c >= block_chunks && c < chunks) ask(c);
    const auto convolved = [&](int e, const FrontEntry& en) {
      float* st = state_slot >= 0 ? fr.conv_state + size_t(state_slot) * (fr.taps - 1) * C + channel(e) : nullptr;
      float seen[kFrontTaps];
#pragma unroll
      for (int j = 0; j < kFrontTaps; ++j) {
        seen[j] = 0.f;
        if (j < fr.taps - 1 && st && ctx - fr.taps + j >= 0) seen[j] = st[size_t(j) * C];
      }
      float y = 0.f;
#pragma unroll
      for (int j = 0; j < kFrontTaps; ++j)
        if (j < fr.taps) {
          if (j == fr.taps - 1) seen[j] = en.x + en.bias;
          y = fmaf(en.w[j], seen[j], y);
        }
      if (st) {
#pragma unroll
        for (int j = 1; j < kFrontTaps; ++j)
          if (j < fr.taps) st[size_t(j - 1) * C] = seen[j];
      }
      return y;
    };
    if (tid < entries) xs[tid] = convolved(tid, early_entry);
    for (int e = tid + WAVES * kWave; e < entries; e += WAVES * kWave) {
      FrontEntry en;
      gather(e, en);
      xs[e] = convolved(e, en);
    }
    __syncthreads();
    const size_t new_page = size_t(new_slot < 0 ? 0 : new_slot / B) * nkv + kvh;
    uint16_t* kp = const_cast<uint16_t*>(kcache) + (new_page * B + (new_slot < 0 ? 0 : new_slot % B)) * d;
    uint16_t* vp = const_cast<uint16_t*>(vcache) + new_page * dv * B + (new_slot < 0 ? 0 : new_slot % B);
    const auto finish = [&](int e, const FrontEntry& en) {
      float x = xs[e];
      if (e < mine + d) {
        const int i = e % d;
        if (i < fr.rot) {
          const int j = turned_with(i);
          const float y = xs[e - i + j];
          x = i > j ? __fmaf_rn(x, en.turn.x, __fmul_rn(y, en.turn.y)) : __fmaf_rn(x, en.turn.x, -__fmul_rn(y, en.turn.y));
        }
      }
      const uint16_t bits = float_to_bf16_bits(x);
      stored[e] = bits;
      if (new_slot >= 0 && e >= mine) {
        if (e < mine + d) kp[e - mine] = bits;
        else vp[size_t(e - mine - d) * B] = bits;
      }
    };
    if (tid < entries) finish(tid, early_entry);
    for (int e = tid + WAVES * kWave; e < entries; e += WAVES * kWave) {
      FrontEntry en;
      gather(e, en);
      finish(e, en);
    }
    __syncthreads();
  }
  const uint16_t* my_q = q + size_t(row) * ldq + size_t(my_head) * d;
  bf16x8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int k = ks * 32 + quad * 8;
    uint4 v;
    if constexpr (FRONT) v = *reinterpret_cast<const uint4*>(stored + (my_head - head0) * d + (k < d ? k : 0));
    else v = *reinterpret_cast<const uint4*>(my_q + (k < d ? k : 0));
    qf[ks] = __builtin_bit_cast(bf16x8, k < d ? v : uint4{0u, 0u, 0u, 0u});
  }

  float m = -INFINITY, l = 0.f;      // the head's largest score; this lane's part of its sum
  f32x4 o[DVT];                      // O^T: column = head, rows = dims 16 vt + 4 quad + i
#pragma unroll
  for (int vt = 0; vt < DVT; ++vt) o[vt] = f32x4{0.f, 0.f, 0.f, 0.f};

  // scores -> probabilities (key_of(j): the token or block of this lane's score j); the running maximum moves on
  auto softmax = [&](float (&sv)[16], auto&& key_of, int lo, int hi, bool tokens) {
    float mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int key = key_of(j);
      sv[j] *= f;
      if (softcap > 0.f) sv[j] = softcap * tanhf(sv[j] * inv_cap);
      if (!FRONT && dist_slope && tokens) sv[j] = fmaf(-slope, float(ctx - 1 - key), sv[j]);
      sv[j] = key >= lo && key < hi ? sv[j] : -INFINITY;
      mx = fmaxf(mx, sv[j]);
    }
    const float m_new = fmaxf(m, rows_max(mx));
    const float alpha = expf(m - m_new);
    m = m_new;
    l *= alpha;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int key = key_of(j);
      sv[j] = key >= lo && key < hi ? expf(sv[j] - m_new) : 0.f;
      l += sv[j];
    }
#pragma unroll
    for (int vt = 0; vt < DVT; ++vt)
#pragma unroll
      for (int i = 0; i < 4; ++i) o[vt][i] *= alpha;
  };

  if (c < block_chunks) {      // (the chunk asked for ahead is not kept through this: it is another wave's)
    do {      // pooled: score 4 t + i is block c0 + 16 t + 4 quad + i
      const int c0 = c * kWave;
      const int b = c0 + lane < blocks ? c0 + lane : blocks - 1, page_no = (b * P + P - 1) / B;
      const int page = table[page_no], entry = b - page_no * B / P;
      auto entry_of = [&](int at) { return (size_t(__shfl(page, at, kWave)) * nkv + kvh) * E + __shfl(entry, at, kWave); };
      float sv[16];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        f32x4 sc = {0.f, 0.f, 0.f, 0.f};
        if (c0 + 16 * t < blocks) {      // (the same for all lanes)
          const float* src = pk + entry_of(16 * t + col) * d;
          any_four x[DP / 16];
          uint2 y[DP / 16];
#pragma unroll
          for (int n = 0; n < DP / 16; ++n) {
            const int k = 16 * n + 4 * quad;
            x[n] = *reinterpret_cast<const any_four*>(src + (k < d ? k : 0));
            if constexpr (FRONT) y[n] = *reinterpret_cast<const uint2*>(stored + (my_head - head0) * d + (k < d ? k : 0));
            else y[n] = *reinterpret_cast<const uint2*>(my_q + (k < d ? k : 0));
          }
#pragma unroll
          for (int n = 0; n < DP / 16; ++n) {
            const bool in = 16 * n + 4 * quad < d;
            const float z[4] = {bf16_bits_to_float(y[n].x & 0xffffu), bf16_bits_to_float(y[n].x >> 16), bf16_bits_to_float(y[n].y & 0xffffu),
                                bf16_bits_to_float(y[n].y >> 16)};
#pragma unroll
            for (int i = 0; i < 4; ++i) sc = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? x[n][i] : 0.f, in ? z[i] : 0.f, sc, 0, 0, 0);
          }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) sv[4 * t + i] = sc[i];
      }
      softmax(sv, [&](int j) { return c0 + 16 * (j / 4) + 4 * quad + j % 4; }, 0, blocks, false);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (c0 + 16 * t >= blocks) break;
#pragma unroll
        for (int i0 = 0; i0 < 4; i0 += 2) {
          float x[2][DVT];
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const float* src = pv + entry_of(16 * t + 4 * quad + i0 + i) * dv;
#pragma unroll
            for (int vt = 0; vt < DVT; ++vt) x[i][vt] = src[vt * 16 + col < dv ? vt * 16 + col : dv - 1];
          }
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const bool in = c0 + 16 * t + 4 * quad + i0 + i < blocks;      // (an infinite entry times zero is not zero)
#pragma unroll
            for (int vt = 0; vt < DVT; ++vt) o[vt] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? x[i][vt] : 0.f, sv[4 * t + i0 + i], o[vt], 0, 0, 0);
          }
        }
      }
      c += WAVES;
    } while (c < block_chunks);
    if (kAhead && c < chunks) ask(c);
  }
  while (c < chunks) {
    // tokens: score 8 g + 4 t + i is token c0 + 32 g + 8 quad + 4 t + i
    int c0, lo, hi;
    stretch(c, c0, lo, hi);
    if (!kAhead) ask(c);
    if (FRONT && new_slot >= 0 && c == chunks - 1) {      // the newest token: its key and value as they were just made
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          if (c0 + 32 * g + 8 * (col / 4) + 4 * t + col % 4 == ctx - 1) {
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
              const int k = ks * 32 + quad * 8;
              kreg[g][t][ks] = *reinterpret_cast<const uint4*>(stored + heads * d + (k < d ? k : 0));
            }
          }
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const int j = ctx - 1 - (c0 + 32 * g + 8 * quad);
        if (j >= 0 && j < 8) {
#pragma unroll
          for (int vt = 0; vt < DVT; ++vt) {
            const int dim = vt * 16 + col;
            const uint32_t bits = stored[heads * d + d + (dim < dv ? dim : dv - 1)];
            const auto with = [&](uint32_t w, int n) {      // word n of the piece: tokens 2 n and 2 n + 1
              return j == 2 * n ? (w & 0xFFFF0000u) | bits : j == 2 * n + 1 ? (w & 0xFFFFu) | bits << 16 : w;
            };
            vreg[g][vt] = uint4{with(vreg[g][vt].x, 0), with(vreg[g][vt].y, 1), with(vreg[g][vt].z, 2), with(vreg[g][vt].w, 3)};
          }
        }
      }
    }
    if (d < DP) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int j = 0; j < 4; ++j) kreg[j / 2][j % 2][ks] = keep_first_bf16(kreg[j / 2][j % 2][ks], d - ks * 32 - quad * 8);
    }
    float sv[16];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        f32x4 sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kreg[g][t][ks]), qf[ks], sc, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) sv[8 * g + 4 * t + i] = sc[i];
      }
    softmax(sv, [&](int j) { return c0 + 32 * (j / 8) + 8 * quad + j % 8; }, lo, hi, true);
    if (c0 < lo || c0 + kWave > hi) {      // values outside the stretch: whatever was there, but zero times it need not be zero
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const int tok = c0 + 32 * g + 8 * quad;
        const uint4 ends = keep_first_bf16(uint4{~0u, ~0u, ~0u, ~0u}, hi - tok), begins = keep_first_bf16(uint4{~0u, ~0u, ~0u, ~0u}, lo - tok);
#pragma unroll
        for (int vt = 0; vt < DVT; ++vt) {
          vreg[g][vt].x &= ends.x & ~begins.x;
          vreg[g][vt].y &= ends.y & ~begins.y;
          vreg[g][vt].z &= ends.z & ~begins.z;
          vreg[g][vt].w &= ends.w & ~begins.w;
        }
      }
    }
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int piece = 0; piece < 3; ++piece) {
        const float* p = sv + 8 * g;
        const bf16x8 pf = __builtin_bit_cast(bf16x8, uint4{upper_halves(p[0], p[1]), upper_halves(p[2], p[3]), upper_halves(p[4], p[5]), upper_halves(p[6], p[7])});
#pragma unroll
        for (int vt = 0; vt < DVT; ++vt) o[vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, vreg[g][vt]), pf, o[vt], 0, 0, 0);
#pragma unroll
        for (int j = 8 * g; j < 8 * g + 8; ++j) sv[j] = below_upper(sv[j]);
      }
    c += WAVES;
    if (kAhead && c < chunks) ask(c);
  }
  l = rows_sum(l);
  if constexpr (FRONT) __syncthreads();      // (the sums come where the front's values were)
#pragma unroll
  for (int vt = 0; vt < DVT; ++vt) *reinterpret_cast<f32x4*>(&parts[wave][col][vt * 16 + 4 * quad]) = o[vt];
  if (quad == 0) {
    maxima[wave][col] = m;
    sums[wave][col] = l;
  }
  __syncthreads();
  if (tid < WAVES * 16) {      // a wave's weight in a head's result
    const int w = tid / 16, h = tid % 16;
    const float sl = sink && sink_logit && h < heads ? sink_logit[head0 + h] : 0.f;
    float mm = sink ? sl : -INFINITY;
#pragma unroll
    for (int v = 0; v < WAVES; ++v) mm = fmaxf(mm, maxima[v][h]);
    const float mw = maxima[w][h];
    weights[w][h] = mw == -INFINITY ? 0.f : expf(mw - mm);
    if (w == 0) {      // (in this wave's place: nobody else reads these)
      float ll = sink ? expf(sl - mm) : 0.f;
#pragma unroll
      for (int v = 0; v < WAVES; ++v) ll = fmaf(sums[v][h], maxima[v][h] == -INFINITY ? 0.f : expf(maxima[v][h] - mm), ll);
      sums[0][h] = ll;
    }
  }
  __syncthreads();
  for (int i = tid; i < heads * dv; i += WAVES * kWave) {
    const int h = i / dv, e = i - h * dv;
    float acc = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) acc = fmaf(parts[w][h][e], weights[w][h], acc);
    float res = acc / sums[0][h] * out_scale;
    if (!FRONT && gate) res *= 1.0f / (1.0f + expf(-gate[size_t(row) * ldg + (gate_heads ? head0 + h : (head0 + h) * dv + e)]));
    orow[i] = float_to_bf16_bits(res);
  }
  if constexpr (FRONT) {      // the block that this token ends lies in the window: its entry is for later steps
    if (P > 0 && new_slot >= 0 && ctx % P == 0 && wave < 2)
      pool_entry<bf16_t, 8>(reinterpret_cast<const bf16_t*>(kcache), reinterpret_cast<const bf16_t*>(vcache), const_cast<float*>(pk), const_cast<float*>(pv), table,
                             wave == 0, ctx - 1, new_slot, kvh, lane, nkv, d, dv, B, P, E);
  }
}

}  // namespace kvcm

using namespace kvcm;

extern "C" {

int kvcm_rotary_pairs_table(const int* positions, float* cos_sin, int T, int dims, float base, hipStream_t s) {
  if (T == 0 || dims == 0) return 0;
  KVCM_REQUIRE(T > 0 && dims > 0 && dims % 2 == 0 && base > 0.f, "rotary_pairs_table: bad sizes T=%d dims=%d base=%g", T,
               dims, double(base));
  const int n = T * (dims / 2);
  rotary_pairs_table_kernel<<<(n + 255) / 256, 256, 0, s>>>(positions, reinterpret_cast<float2*>(cos_sin), T, dims / 2,
                                                            log(double(base)), dims);
  return launch_status("rotary_pairs_table");
}

int kvcm_rotary_freq_table(const int* positions, const double* freqs, float* cos_sin, int T, int dims, float factor,
                           hipStream_t s) {
  if (T == 0) return 0;
  KVCM_REQUIRE(T > 0 && dims > 0 && dims % 2 == 0 && positions && freqs && cos_sin, "rotary_freq_table: bad sizes T=%d dims=%d", T, dims);
  const int n = T * (dims / 2);
  rotary_freq_table_kernel<<<(n + 255) / 256, 256, 0, s>>>(positions, freqs, reinterpret_cast<float2*>(cos_sin), T, dims / 2,
                                                           double(factor));
  return launch_status("rotary_freq_table");
}

int kvcm_rotate_store(const float* src, int ld, const float* kv_src, int ldkv, const float* cos_sin, int rot, int halves,
                      const int* slots, void* q_out, int dtype, int ldq, void* kcache, void* vcache, int T, int nh, int nkv, int d,
                      int dv, int B, hipStream_t s) {
  if (T == 0) return 0;
  KVCM_REQUIRE(T > 0 && nh > 0 && nkv > 0 && d > 0 && dv > 0 && B > 0, "rotate_store: bad sizes");
  KVCM_REQUIRE(rot % 2 == 0 && rot >= 0 && rot <= d, "rotate_store: %d rotated of %d dims is not supported "
               "(an even number, at most the head's size)", rot, d);
  KVCM_REQUIRE(rot == 0 || cos_sin != nullptr, "rotate_store: a rotation needs its table");
  if (kv_src) KVCM_REQUIRE(ld >= nh * d && ldkv >= nkv * (d + dv) && ldq >= nh * d, "rotate_store: row strides too small");
  else KVCM_REQUIRE(ld >= (slots ? (nh + nkv) * d + nkv * dv : nh * d) && ldq >= nh * d, "rotate_store: row strides too small");
  KVCM_REQUIRE(!slots || (kcache && vcache), "rotate_store: slots without pages");
  const float2* cs = reinterpret_cast<const float2*>(cos_sin);
  const dim3 T_by_parts(T, T <= kNormRotateFewRows ? nh + nkv + 1 : 1);
  if (dtype == kF32)
    rotate_store_kernel<float><<<T_by_parts, 256, 0, s>>>(src, ld, kv_src, ldkv, cs, rot, halves, slots, static_cast<float*>(q_out), ldq,
                                                  static_cast<float*>(kcache), static_cast<float*>(vcache), nh, nkv, d, dv, B);
  else if (dtype == kBF16)
    rotate_store_kernel<bf16_t><<<T_by_parts, 256, 0, s>>>(src, ld, kv_src, ldkv, cs, rot, halves, slots, static_cast<bf16_t*>(q_out), ldq,
                                                   static_cast<bf16_t*>(kcache), static_cast<bf16_t*>(vcache), nh, nkv, d, dv, B);
  else KVCM_REQUIRE(false, "rotate_store: unknown dtype %d", dtype);
  return launch_status("rotate_store");
}

int kvcm_norm_rotate_store(const float* src, int ld, const float* wq, const float* wk, float eps, const float* v_other, int ldvo,
                           float mix, float* v_keep, int ldvk, const float* cos_sin, int rot, int halves, const int* slots,
                           void* q_out, int dtype, int ldq, void* kcache, void* vcache, int T, int nh, int nkv, int d, int dv, int B,
                           hipStream_t s) {
  if (T == 0) return 0;
  KVCM_REQUIRE(T > 0 && nh > 0 && nkv > 0 && d > 0 && dv > 0 && B > 0, "norm_rotate_store: bad sizes");
  KVCM_REQUIRE(rot % 2 == 0 && rot >= 0 && rot <= d, "norm_rotate_store: %d rotated of %d dims is not supported "
               "(an even number, at most the head's size)", rot, d);
  KVCM_REQUIRE(rot == 0 || cos_sin != nullptr, "norm_rotate_store: a rotation needs its table");
  KVCM_REQUIRE(ld >= (nh + nkv) * d + nkv * dv && ldq >= nh * d, "norm_rotate_store: row strides too small");
  KVCM_REQUIRE((!v_other || ldvo >= nkv * dv) && (!v_keep || ldvk >= nkv * dv), "norm_rotate_store: rows of values too short");
  KVCM_REQUIRE(!slots || (kcache && vcache), "norm_rotate_store: slots without pages");
  const float2* cs = reinterpret_cast<const float2*>(cos_sin);
  // few rows: a workgroup per head, so that a single row is not the work of one compute unit (the same bits either way)
  const dim3 grid(T, T <= kNormRotateFewRows ? nh + nkv + 1 : 1);
  if (dtype == kF32)
    norm_rotate_store_kernel<float><<<grid, 256, 0, s>>>(src, ld, wq, wk, eps, v_other, ldvo, mix, v_keep, ldvk, cs, rot, halves, slots,
                                                       static_cast<float*>(q_out), ldq, static_cast<float*>(kcache),
                                                       static_cast<float*>(vcache), nh, nkv, d, dv, B);
  else if (dtype == kBF16)
    norm_rotate_store_kernel<bf16_t><<<grid, 256, 0, s>>>(src, ld, wq, wk, eps, v_other, ldvo, mix, v_keep, ldvk, cs, rot, halves, slots,
                                                        static_cast<bf16_t*>(q_out), ldq, static_cast<bf16_t*>(kcache),
                                                        static_cast<bf16_t*>(vcache), nh, nkv, d, dv, B);
  else KVCM_REQUIRE(false, "norm_rotate_store: unknown dtype %d", dtype);
  return launch_status("norm_rotate_store");
}

int kvcm_pool_update(const void* kcache, const void* vcache, int dtype, float* pk, float* pv, const int* tables,
                     int table_stride, const int* row_seq, const int* positions, const int* slots, int T, int nkv, int d,
                     int dv, int B, int P, int E, hipStream_t s) {
  if (T == 0 || P <= 0) return 0;
  KVCM_REQUIRE(T > 0 && nkv > 0 && d > 0 && dv > 0 && B > 0, "pool_update: bad sizes");
  KVCM_REQUIRE(E == (B + P - 1) / P, "pool_update: %d entries a page do not fit pages of %d and blocks of %d", E, B, P);
  KVCM_REQUIRE(nkv <= 65535, "pool_update: too many kv heads");
  // Rows a wave.  In a run at most one of them ends a block where R <= P, and few waves look at many rows; but requests that
  // decode in step may all end one, and a wave makes its entries one after the other.  Growing with the rows, both stay below
  // what a workgroup per row takes.  Blocks of 64, 4 kv heads of 64, us, this / a row each / 64 rows each: a prompt of 2,048
  // 11.5 / 64 / 11.5, 8 of 2,048 17 / 475 / 17; 128 rows that all end a block 11.6 / 11.6 / 660, 512 such rows 40 / 34 / 615.
  const int R = T < 256 ? 1 : std::min({T / 128, P, kWave});
  const dim3 grid((T + R - 1) / R, nkv, 2);      // keys, values
  // (short blocks do not ask for many more tokens than they have: blocks of 8, 64 rows that end one, 7.0 us as 32 ahead, 3.7 as 8)
  auto launch = [&](auto* kc, auto* vc) {
    using T_ = std::remove_const_t<std::remove_pointer_t<decltype(kc)>>;
    auto* kernel = P <= 8 ? pool_update_kernel<T_, 8> : P <= 16 ? pool_update_kernel<T_, 16> : pool_update_kernel<T_, 32>;
    kernel<<<grid, kWave, 0, s>>>(kc, vc, pk, pv, tables, table_stride, row_seq, positions, slots, T, R, nkv, d, dv, B, P, E);
  };
  if (dtype == kF32) launch(static_cast<const float*>(kcache), static_cast<const float*>(vcache));
  else if (dtype == kBF16) launch(static_cast<const bf16_t*>(kcache), static_cast<const bf16_t*>(vcache));
  else KVCM_REQUIRE(false, "pool_update: unknown dtype %d", dtype);
  return launch_status("pool_update");
}

int kvcm_attention_window_pool(const void* q, int dtype, int ldq, void* out, int ldo, const void* kcache, const void* vcache,
                               const float* pk, const float* pv, const int* tables, int table_stride, const int* row_seq,
                               const int* ctx_lens, const float* head_scale, const float* dist_slope, const float* gate, int ldg,
                               int T, int nh, int nkv, int d, int dv, int B, float scale, int window, int P, int E, int keep_first,
                               float softcap, int chunk, int sink, const float* __restrict__ sink_logit, int gate_heads, float out_scale, hipStream_t s) {
  if (T == 0) return 0;
  KVCM_REQUIRE(T > 0 && nh > 0 && nkv > 0 && B > 0 && d > 0, "attention_window_pool: bad sizes T=%d heads=%d kv_heads=%d", T, nh, nkv);
  KVCM_REQUIRE(nh % nkv == 0, "attention_window_pool: %d query heads are not a multiple of %d kv heads", nh, nkv);
  KVCM_REQUIRE(dv > 0 && dv <= kWpMaxValueDim, "attention_window_pool: value size %d is not supported (up to %d)", dv, kWpMaxValueDim);
  KVCM_REQUIRE(d <= 1024, "attention_window_pool: key size %d is not supported (up to 1024)", d);
  KVCM_REQUIRE(ldq >= nh * d && ldo >= nh * dv, "attention_window_pool: row strides too small");
  KVCM_REQUIRE(window >= 0 && P >= 0, "attention_window_pool: negative window or block");
  KVCM_REQUIRE(P == 0 || (pk && pv && E == (B + P - 1) / P), "attention_window_pool: pooled blocks need their entries");
  KVCM_REQUIRE(keep_first >= 0 && softcap >= 0.f, "attention_window_pool: negative count of kept tokens or score cap");
  KVCM_REQUIRE(!dist_slope || P == 0, "attention_window_pool: a distance bias beside pooled blocks is not supported");
  KVCM_REQUIRE(!gate || ldg >= (gate_heads ? nh : nh * dv), "attention_window_pool: the gate's rows are too short");
  KVCM_REQUIRE(chunk >= 0 && (chunk == 0 || (window == 0 && P == 0 && keep_first == 0)),
               "attention_window_pool: a chunk beside a window, pooled blocks or kept first tokens is not supported");
  const long long blocks = static_cast<long long>(T) * nh;
  KVCM_REQUIRE(blocks < (1ll << 31), "attention_window_pool: too many rows");
  // heads together where 16-byte loads fit rows and pages and a wave's sums and fragments fit its registers (at 256 values they
  // do not), from two query heads a kv head on; us, a workgroup per row and head / heads together, window 512, heads of 64:
  //   8 per kv head, 8 / 64 / 1,000 rows of 600 tokens: 17 / 10, 74 / 12, 894 / 136; of 64 tokens 7.8 / 6.9, 29 / 7, 376 / 80
  //   2 per kv head (16 in all): 15.6 / 10.0, 40 / 23, 452 / 260; 7.7 / 6.7, 14.5 / 11.7, 192 / 151
  //   1 per kv head (32): 17.2 / 11.8, 80 / 80, 894 / 1,005; 7.8 / 6.9, 28.5 / 41, 376 / 581: one column of sixteen does the work
  // The rule looks at sizes and places alone, never at the rows: a row's bits do not depend on what else the launch holds.
  if (dtype == kBF16 && nh / nkv >= 2 && d % 8 == 0 && d <= 128 && dv % 8 == 0 && dv <= 128 && B % 8 == 0 && ldq % 8 == 0 &&
      (reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(kcache) | reinterpret_cast<uintptr_t>(vcache)) % 16 == 0 &&
      nkv * ((nh / nkv + 15) / 16) <= 65535) {
    const dim3 grid(T, nkv * ((nh / nkv + 15) / 16));
#define KVCM_WINDOW_POOL_HEADS(DP, DVT, WAVES)                                                                                 \
  attention_window_pool_heads_kernel<DP, DVT, WAVES, false><<<grid, (WAVES) * kWave, 0, s>>>(                                         \
      static_cast<const uint16_t*>(q), ldq, static_cast<uint16_t*>(out), ldo, static_cast<const uint16_t*>(kcache),            \
      static_cast<const uint16_t*>(vcache), pk, pv, tables, table_stride, row_seq, ctx_lens, head_scale, dist_slope, gate, ldg, \
      nh, nkv, d, dv, B, scale, window, P, E, keep_first, softcap, chunk, sink, sink_logit, gate_heads, out_scale, WpFront{})
    if (d <= 64 && dv <= 64) KVCM_WINDOW_POOL_HEADS(64, 4, 12);
    else KVCM_WINDOW_POOL_HEADS(128, 8, 7);      // (what 64 KB of local memory hold)
#undef KVCM_WINDOW_POOL_HEADS
    return launch_status("attention_window_pool");
  }
  const size_t lds = sizeof(float) * (d + kWpWaves * kWave + kWpWaves * (dv + 2));
  if (dtype == kF32)
    attention_window_pool_kernel<float><<<static_cast<unsigned>(blocks), kWpWaves * kWave, lds, s>>>(
        static_cast<const float*>(q), ldq, static_cast<float*>(out), ldo, static_cast<const float*>(kcache),
        static_cast<const float*>(vcache), pk, pv, tables, table_stride, row_seq, ctx_lens, head_scale, dist_slope, gate,
        ldg, nh, nkv, d, dv, B, scale, window, P, E, keep_first, softcap, chunk, sink, sink_logit, gate_heads, out_scale);
  else if (dtype == kBF16)
    attention_window_pool_kernel<bf16_t><<<static_cast<unsigned>(blocks), kWpWaves * kWave, lds, s>>>(
        static_cast<const bf16_t*>(q), ldq, static_cast<bf16_t*>(out), ldo, static_cast<const bf16_t*>(kcache),
        static_cast<const bf16_t*>(vcache), pk, pv, tables, table_stride, row_seq, ctx_lens, head_scale, dist_slope, gate,
        ldg, nh, nkv, d, dv, B, scale, window, P, E, keep_first, softcap, chunk, sink, sink_logit, gate_heads, out_scale);
  else KVCM_REQUIRE(false, "attention_window_pool: unknown dtype %d", dtype);
  return launch_status("attention_window_pool");
}

// 1 when kvcm_attention_window_pool_rows takes the head shape and pages.
int kvcm_attention_window_pool_rows_supported(int nh, int nkv, int d, int dv, int B) {
  return nkv > 0 && nh % nkv == 0 && nh / nkv >= 2 && nh / nkv <= 16 && d > 0 && dv > 0 && d % 8 == 0 && d <= 64 && dv % 8 == 0 && dv <= 64 && B > 0 &&
         B % 8 == 0 && nkv <= 65535;
}

// ... and T rows of them faster than the four launches do: while every workgroup has a CU to itself.  Its registers leave no room for a second one beside
// it, and where a second turn follows, a workgroup that ends with a pooled entry (a wave that walks the block's tokens) holds everything up.  us, four
// launches / one, blocks of 64, window 512: 32 heads over 4 of 64, 16 / 32 / 64 rows of 540 tokens 18.3 / 16.6, 23.1 / 17.0, 26.0 / 19.6, some of them
// at the end of a block (60 to 75 tokens) 23.7 / 20.2, 27.8 / 20.4, 29.8 / 21.1; 80, 128, 256, 512 rows 34.1 / 32.6, 37.4 / 36.8, 72.3 / 82.4, 125.3 / 153.5 and 34.8 / 39.3, 38.9 /
// 39.9, 56.1 / 76.8, 84.2 / 149.4; 16 heads over 8, 32 rows 24.6 / 17.7, 48 rows 32.0 / 29.9 and 33.4 / 37.4, 128 rows 61.0 / 70.0.
int kvcm_attention_window_pool_rows_takes(int T, int nh, int nkv, int d, int dv, int B) {
  constexpr int kCUs = 256;
  return kvcm_attention_window_pool_rows_supported(nh, nkv, d, dv, B) && T > 0 && T <= kCUs / nkv;
}

// bfloat16 rows of T different sequences, one each, from the projection's 32-bit rows [q | k | v] to the attention's: convolution (conv_w [C][taps],
// bias before it, conv_state [slots][taps - 1][C] moved on), rotation (as kvcm_rotate_store), keys and values to slots [T] (negative: not
// stored), the attention, and the pooled entries that end with these rows.  The rows' positions are ctx_lens - 1.  The results are those of the
// launches one by one, bit for bit.
int kvcm_attention_window_pool_rows(const float* src, int ld, const float* conv_w, const float* conv_bias, float* conv_state, const int* state_slots,
                                    int taps, const float* cos_sin, int rot, int halves, const int* slots, void* out, int ldo, void* kcache, void* vcache,
                                    float* pk, float* pv, const int* tables, int table_stride, const int* row_seq, const int* ctx_lens,
                                    const float* head_scale, int T, int nh, int nkv, int d, int dv, int B, float scale, int window, int P, hipStream_t s) {
  if (T == 0) return 0;
  KVCM_REQUIRE(T > 0 && kvcm_attention_window_pool_rows_supported(nh, nkv, d, dv, B),
               "attention_window_pool_rows: unsupported shape T=%d heads=%d kv_heads=%d d=%d dv=%d page=%d", T, nh, nkv, d, dv, B);
  const int C = (nh + nkv) * d + nkv * dv;
  KVCM_REQUIRE(src && conv_w && out && kcache && vcache && slots && tables && row_seq && ctx_lens, "attention_window_pool_rows: null operand");
  KVCM_REQUIRE(ld >= C && ldo >= nh * dv, "attention_window_pool_rows: row strides too small");
  KVCM_REQUIRE(taps >= 1 && taps <= kFrontTaps && (taps == 1 || (conv_state && state_slots)),
               "attention_window_pool_rows: %d taps are not supported (1 to %d are), or the state is missing", taps, kFrontTaps);
  KVCM_REQUIRE(rot % 2 == 0 && rot >= 0 && rot <= d && (rot == 0 || cos_sin), "attention_window_pool_rows: bad rotation of %d dims", rot);
  KVCM_REQUIRE(window >= 0 && P >= 0 && (P == 0 || (pk && pv)), "attention_window_pool_rows: bad window or blocks");
  KVCM_REQUIRE((reinterpret_cast<uintptr_t>(kcache) | reinterpret_cast<uintptr_t>(vcache)) % 16 == 0 && reinterpret_cast<uintptr_t>(cos_sin) % 8 == 0,
               "attention_window_pool_rows: pages must be 16-byte aligned");
  const int E = P > 0 ? (B + P - 1) / P : 0;
  const WpFront fr{src, ld, conv_w, conv_bias, taps > 1 ? conv_state : nullptr, taps > 1 ? state_slots : nullptr, taps,
                   reinterpret_cast<const float2*>(cos_sin), rot, halves, slots};
  attention_window_pool_heads_kernel<64, 4, 12, true><<<dim3(T, nkv), 12 * kWave, 0, s>>>(
      nullptr, 0, static_cast<uint16_t*>(out), ldo, static_cast<const uint16_t*>(kcache), static_cast<const uint16_t*>(vcache), pk, pv, tables,
      table_stride, row_seq, ctx_lens, head_scale, nullptr, nullptr, 0, nh, nkv, d, dv, B, scale, window, P, E, 0, 0.f, 0, 0, nullptr, 0, 1.0f, fr);
  return launch_status("attention_window_pool_rows");
}

}  // extern "C"
