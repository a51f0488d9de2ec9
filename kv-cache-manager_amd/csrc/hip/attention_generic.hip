// Attention of query rows over the paged cache, one wave per (row, query head).
//
// The same arithmetic as the reference kernel (src/cuda/paged_attention.cu:50-183): q is scaled
// in 32-bit before the dot product, a row with context length c sees keys 0 .. c-1 of its own
// sequence through the block table (causality is nothing but c = position + 1), query head h
// reads KV head h / (heads / kv_heads), softmax and the P*V sums are 32-bit and the result is
// divided by the sum once.  Differences: keys are taken 64 at a time with a running maximum
// (no score buffer that grows with the context), any head_dim that is a multiple of 8 up to 256
// and any group size work, storage is float or bfloat16, and an optional window hides keys with
// position <= row position - window.
//
// A row's result is a fixed sequence of operations on its own keys: chunks start at absolute
// multiples of 64, lanes map to keys and dims the same way every time.  It therefore does not
// depend on which other rows are in the launch, nor on which physical pages hold the keys.
//
// 32-bit storage with head sizes 16, 32, 64 and 128, up to 16 query heads per kv head and pages of a multiple of 4 tokens
// takes attention_f32_kernel below: the same products on the matrix cores' 32-bit instruction.
#include <algorithm>
#include <cfloat>
#include <type_traits>

#include "common.h"

namespace kvcm {

constexpr int kAttnWaves = 4;
constexpr int kMaxHeadDim = 256;

template <class T> struct Vec;
template <> struct Vec<float> { static constexpr int N = 4; };
template <> struct Vec<bf16_t> { static constexpr int N = 8; };

template <class T>
__device__ __forceinline__ float dot_piece(const float* q, const T* k);
template <>
__device__ __forceinline__ float dot_piece<float>(const float* q, const float* k) {
  const float4 v = *reinterpret_cast<const float4*>(k);
  float s = q[0] * v.x;
  s = fmaf(q[1], v.y, s);
  s = fmaf(q[2], v.z, s);
  return fmaf(q[3], v.w, s);
}
template <>
__device__ __forceinline__ float dot_piece<bf16_t>(const float* q, const bf16_t* k) {
  const uint4 v = *reinterpret_cast<const uint4*>(k);
  float s = q[0] * bf16_bits_to_float(v.x & 0xffffu);
  s = fmaf(q[1], bf16_bits_to_float(v.x >> 16), s);
  s = fmaf(q[2], bf16_bits_to_float(v.y & 0xffffu), s);
  s = fmaf(q[3], bf16_bits_to_float(v.y >> 16), s);
  s = fmaf(q[4], bf16_bits_to_float(v.z & 0xffffu), s);
  s = fmaf(q[5], bf16_bits_to_float(v.z >> 16), s);
  s = fmaf(q[6], bf16_bits_to_float(v.w & 0xffffu), s);
  return fmaf(q[7], bf16_bits_to_float(v.w >> 16), s);
}

template <class T>
__global__ void __launch_bounds__(kAttnWaves* kWave)
    attention_generic_kernel(const T* __restrict__ q, int q_stride, T* __restrict__ out, int out_stride,
                             const T* __restrict__ kcache, const T* __restrict__ vcache,
                             const int* __restrict__ tables, int table_stride, const int* __restrict__ row_seq,
                             const int* __restrict__ ctx_lens, long long items, int nh, int nkv, int hd, int B,
                             float scale, int window) {
  extern __shared__ float q_lds[];  // [waves][hd], q * scale
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const long long item = static_cast<long long>(blockIdx.x) * kAttnWaves + wave;
  const bool active = item < items;
  const int row = active ? static_cast<int>(item / nh) : 0;
  const int head = active ? static_cast<int>(item % nh) : 0;
  float* qs = q_lds + wave * hd;
  if (active)
    for (int d = lane; d < hd; d += kWave) qs[d] = load_f(q + size_t(row) * q_stride + size_t(head) * hd + d) * scale;
  __syncthreads();
  if (!active) return;

  const int kvh = head / (nh / nkv);
  const int ctx = ctx_lens[row];
  T* orow = out + size_t(row) * out_stride + size_t(head) * hd;
  if (ctx <= 0) {
    for (int d = lane; d < hd; d += kWave) store_f(orow + d, 0.f);
    return;
  }
  const int first = (window > 0 && ctx > window) ? ctx - window : 0;
  const int* table = tables + size_t(row_seq[row]) * table_stride;
  const size_t head_stride = size_t(B) * hd, page_stride = head_stride * nkv;

  float m = -INFINITY, l = 0.f;
  float o[kMaxHeadDim / kWave] = {0.f, 0.f, 0.f, 0.f};
  for (int c0 = (first / kWave) * kWave; c0 < ctx; c0 += kWave) {
    const int t = c0 + lane;
    const bool valid = t >= first && t < ctx;
    float s = -INFINITY;
    if (valid) {
      const T* kp = kcache + size_t(table[t / B]) * page_stride + kvh * head_stride + size_t(t % B) * hd;
      s = 0.f;
      for (int d = 0; d < hd; d += Vec<T>::N) s += dot_piece<T>(qs + d, kp + d);
    }
    const float m_new = fmaxf(m, wave_max(s));
    const float alpha = expf(m - m_new);
    const float p = valid ? expf(s - m_new) : 0.f;
    l = l * alpha + wave_sum(p);
#pragma unroll
    for (int i = 0; i < kMaxHeadDim / kWave; ++i) o[i] *= alpha;
    const int j_lo = first > c0 ? first - c0 : 0;
    const int j_hi = ctx - c0 < kWave ? ctx - c0 : kWave;
    for (int j = j_lo; j < j_hi; ++j) {
      const float pj = __shfl(p, j, kWave);
      const int tj = c0 + j;
      const T* vp = vcache + size_t(table[tj / B]) * page_stride + kvh * head_stride + tj % B;  // [dim][slot]
#pragma unroll
      for (int i = 0; i < kMaxHeadDim / kWave; ++i) {
        const int d = lane + i * kWave;
        if (d < hd) o[i] = fmaf(pj, load_f(vp + size_t(d) * B), o[i]);
      }
    }
    m = m_new;
  }
#pragma unroll
  for (int i = 0; i < kMaxHeadDim / kWave; ++i) {
    const int d = lane + i * kWave;
    if (d < hd) store_f(orow + d, o[i] / l);
  }
}

// ---- 32-bit storage on the matrix cores (v_mfma_f32_16x16x4_f32) -----------------------------------------------------------
// A workgroup owns 16 items, an item being one query head of one row: the heads of a kv head's group, of one row or of 16 /
// group consecutive rows, so that the keys and values of the group are read once.  Its waves take the chunks of 64 keys in turn
// (chunk c is of share c % WAVES, a wave's own for each sequence) and meet in LDS at the end, in the order of the shares.  Products are transposed as in the bfloat16
// kernels, S^T = K Q^T and O^T += V^T P^T: a lane's scores are four consecutive keys of one item, which is where the second
// product wants their probabilities, and both caches are read in 16-byte pieces.
// A chunk in which an item sees nothing changes nothing of it, so its result does not depend on the items beside it.
// One wave per (row, head) that reads values one token at a time (the kernel above) was bound by that chain of loads: two prompts
// of 301 and 272 tokens and 15 decode steps behind them, 32 heads of 64: 123.6 us a launch in the mean -> 13.8 us.
using f32x4 = __attribute__((__vector_size__(4 * sizeof(float)))) float;

template <int NT>      // head size / 16
constexpr int f32_waves() { return NT <= 4 ? 8 : 4; }      // (a wave's share of the output lies in LDS: 1 KB a tile, 32 KB in all)

// STORES: q are rows of the projection [q | k | v], every row of a sequence of its own; its key and value go to their slot first, q and k
// rotated by cos_sin [T][hd / 2] (null: not), with the operations of the rotation's own kernel: a launch and 4 to 5 us a layer less.
template <int NT, bool STORES>
__global__ void __launch_bounds__(f32_waves<NT>() * kWave)
    attention_f32_kernel(const float* __restrict__ q, int q_stride, float* __restrict__ out, int out_stride,
                         const float* kcache, const float* vcache, const int* __restrict__ tables,
                         int table_stride, const int* __restrict__ row_seq, const int* __restrict__ ctx_lens, int T, int nh, int nkv,
                         int rows_per_tile, int B, float scale, int window, const float2* __restrict__ cos_sin, const int* __restrict__ slots) {
  constexpr int WAVES = f32_waves<NT>(), hd = 16 * NT;
  __shared__ f32x4 part_o[WAVES][16][NT * 4];
  __shared__ float part_m[WAVES][16], part_l[WAVES][16];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int it = lane & 15, g = lane >> 4;
  const int group = nh / nkv, kvh = blockIdx.x % nkv, r0 = blockIdx.x / nkv * rows_per_tile;
  const int rows = T - r0 < rows_per_tile ? T - r0 : rows_per_tile;
  const int own = it / group;                                   // the item's row within the tile
  const bool real = it < rows * group;
  const int row = r0 + (real ? own : 0), head = kvh * group + (real ? it % group : 0);
  const int ctx = real ? ctx_lens[row] : 0;
  const int first = (window > 0 && ctx > window) ? ctx - window : 0;
  // the tile's rows, a lane each: no load waits for another as they are looked through
  const int seqs = row_seq[r0 + (lane < rows ? lane : 0)], ctxs = ctx_lens[r0 + (lane < rows ? lane : 0)];
  f32x4 qf[NT];
#pragma unroll
  for (int u = 0; u < NT; ++u) qf[u] = *reinterpret_cast<const f32x4*>(q + size_t(row) * q_stride + size_t(head) * hd + 16 * u + 4 * g);
  if constexpr (STORES) {
    constexpr int half = hd / 2;
    if (cos_sin) {
      const float2* angle = cos_sin + size_t(row) * half;
      if constexpr (NT == 1) {      // dims 4 g + e: the partner's lane is 32 away
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float2 t = angle[4 * (g & 1) + e];
          const float there = __shfl_xor(qf[0][e], 32, kWave);
          float a = g < 2 ? qf[0][e] : there, b = g < 2 ? there : qf[0][e];
          rotate_pair(a, b, t.x, t.y);
          qf[0][e] = g < 2 ? a : b;
        }
      } else {
#pragma unroll
        for (int u = 0; u < NT / 2; ++u)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float2 t = angle[16 * u + 4 * g + e];
            float a = qf[u][e], b = qf[u + NT / 2][e];
            rotate_pair(a, b, t.x, t.y);
            qf[u][e] = a;
            qf[u + NT / 2][e] = b;
          }
      }
    }
    for (int i = threadIdx.x; i < rows * hd; i += WAVES * kWave) {      // pairs of k, then pairs of v, of every row
      const int t = r0 + i / hd, j = i % half, slot = slots[t];
      const bool is_v = i % hd >= half;
      if (slot < 0) continue;
      const float* src = q + size_t(t) * q_stride + size_t(nh + (is_v ? nkv : 0) + kvh) * hd + j;
      float a = src[0], b = src[half];
      const size_t page = slot / B;
      const int off = slot % B;
      if (is_v) {
        float* to = const_cast<float*>(vcache) + (page * nkv + kvh) * size_t(hd) * B + off;
        to[size_t(j) * B] = a;
        to[size_t(j + half) * B] = b;
      } else {
        if (cos_sin) {
          const float2 c = cos_sin[size_t(t) * half + j];
          rotate_pair(a, b, c.x, c.y);
        }
        float* to = const_cast<float*>(kcache) + ((page * nkv + kvh) * B + off) * hd + j;
        to[0] = a;
        to[half] = b;
      }
    }
    __syncthreads();      // stored before any wave of this workgroup, which alone reads them, loads them
  }
#pragma unroll
  for (int u = 0; u < NT; ++u) qf[u] = qf[u] * scale;

  const size_t head_stride = size_t(B) * hd, page_stride = head_stride * nkv;
  float m = -INFINITY, l = 0.f;
  f32x4 o[NT];
#pragma unroll
  for (int d = 0; d < NT; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};

  // consecutive rows of one sequence walk its keys together; a wave takes another share of the chunks with each sequence, so that
  // sequences of few chunks are walked by as many waves
  int share = wave, own_share = wave;                           // of the sequence at hand; of the item's
  for (int j = 0; j < rows; share = share + 1 == WAVES ? 0 : share + 1) {
    const int seq = __builtin_amdgcn_readlane(seqs, j);
    int end = j, most = 0, least = 0x7fffffff;                  // rows j .. end - 1 see tokens in [least, most)
    for (; end < rows && __builtin_amdgcn_readlane(seqs, end) == seq; ++end) {
      const int c = __builtin_amdgcn_readlane(ctxs, end);
      if (c <= 0) continue;
      const int f = (window > 0 && c > window) ? c - window : 0;
      most = c > most ? c : most;
      least = f < least ? f : least;
    }
    const bool mine = real && own >= j && own < end;
    own_share = mine ? share : own_share;
    const int* table = tables + size_t(seq) * table_stride;
    int chunk = most > 0 ? least / kWave : 0;
    chunk += (share - chunk % WAVES + WAVES) % WAVES;
    auto walk = [&](int c0, auto groups) {                      // the first G sixteens of a chunk's keys
      constexpr int G = decltype(groups)::value;
      f32x4 kf[G][NT], vf[G][NT];
      const float *kp[G], *vp[G];
#pragma unroll
      for (int i = 0; i < G; ++i) {                             // tokens outside [least, most) read an inner token's place
        int t = c0 + 16 * i + it;
        t = t < most ? (t > least ? t : least) : most - 1;
        kp[i] = kcache + size_t(table[t / B]) * page_stride + kvh * head_stride + size_t(t % B) * hd + 4 * g;
        int t4 = c0 + 16 * i + 4 * g;
        t4 = t4 < most ? (t4 > least ? t4 : least) : most - 1;
        t4 &= ~3;
        vp[i] = vcache + size_t(table[t4 / B]) * page_stride + kvh * head_stride + size_t(it) * B + t4 % B;
      }
#pragma unroll
      for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int i = 0; i < G; ++i) kf[i][u] = *reinterpret_cast<const f32x4*>(kp[i] + 16 * u);
#pragma unroll
      for (int d = 0; d < NT; ++d)
#pragma unroll
        for (int i = 0; i < G; ++i) vf[i][d] = *reinterpret_cast<const f32x4*>(vp[i] + size_t(16 * d) * B);
      f32x4 s[G];
#pragma unroll
      for (int i = 0; i < G; ++i) s[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < G; ++i) s[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i][u][e], qf[u][e], s[i], 0, 0, 0);
      float top = -INFINITY;
#pragma unroll
      for (int i = 0; i < G; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int t = c0 + 16 * i + 4 * g + e;
          const bool sees = mine && t >= first && t < ctx;
          s[i][e] = sees ? s[i][e] : -INFINITY;
          top = fmaxf(top, s[i][e]);
        }
      top = rows_max(top);
      const float m_new = fmaxf(m, top);
      const bool some = m_new > -INFINITY;                      // the item has seen a key with a finite score
      const float alpha = some ? expf(m - m_new) : 1.f;
      float sum = 0.f, bad = 0.f;
#pragma unroll
      for (int i = 0; i < G; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int t = c0 + 16 * i + 4 * g + e;
          const bool sees = mine && t >= first && t < ctx;
          s[i][e] = sees ? expf(s[i][e] - m_new) : 0.f;
          sum += s[i][e];
          // values outside [least, most) are a page's previous owner's: zero times a stale Inf or NaN would not be zero
          const bool kept = t >= least && t < most;
#pragma unroll
          for (int d = 0; d < NT; ++d) {
            vf[i][d][e] = kept ? vf[i][d][e] : 0.f;
            bad = fmaf(vf[i][d][e], 0.f, bad);                  // NaN when some value is not finite
          }
        }
      l = l * alpha + sum;
      m = m_new;
#pragma unroll
      for (int d = 0; d < NT; ++d) o[d] *= alpha;
      if (rows == 1 || __ballot(bad != bad) == 0) {      // (zero times these values is zero, or nobody else is here)
#pragma unroll
        for (int i = 0; i < G; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int d = 0; d < NT; ++d) o[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[i][d][e], s[i][e], o[d], 0, 0, 0);
      } else {
        // a value that is not finite counts for the rows that see it only: row by row, the others' values zero
        for (int r = j; r < end; ++r) {
          const int c = __builtin_amdgcn_readlane(ctxs, r), f = (window > 0 && c > window) ? c - window : 0;
          f32x4 one[NT];
#pragma unroll
          for (int d = 0; d < NT; ++d) one[d] = o[d];
#pragma unroll
          for (int i = 0; i < G; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int t = c0 + 16 * i + 4 * g + e;
#pragma unroll
              for (int d = 0; d < NT; ++d)
                one[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(t >= f && t < c ? vf[i][d][e] : 0.f, s[i][e], one[d], 0, 0, 0);
            }
#pragma unroll
          for (int d = 0; d < NT; ++d) o[d] = own == r ? one[d] : o[d];
        }
      }
    };
    int c0 = chunk * kWave;
    for (; c0 + 16 < most; c0 += WAVES * kWave) walk(c0, std::integral_constant<int, 4>());
    if (c0 < most) walk(c0, std::integral_constant<int, 1>());      // (absent keys add zeros: left out where they are most of the last chunk)
    j = end;
  }
  l = rows_sum(l);
  if (g == 0) {
    part_m[own_share][it] = m;
    part_l[own_share][it] = l;
  }
#pragma unroll
  for (int d = 0; d < NT; ++d) part_o[own_share][it][4 * d + g] = o[d];
  __syncthreads();
  for (int t = threadIdx.x; t < rows * group * NT * 4; t += WAVES * kWave) {
    const int i = t / (NT * 4), d = t % (NT * 4), r = r0 + i / group;
    float* to = out + size_t(r) * out_stride + size_t(kvh * group + i % group) * hd + 4 * d;
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    if (ctx_lens[r] > 0) {
      float high = part_m[0][i], total = 0.f;
#pragma unroll
      for (int w = 1; w < WAVES; ++w) high = fmaxf(high, part_m[w][i]);
#pragma unroll
      for (int w = 0; w < WAVES; ++w) {
        const float f = part_m[w][i] > -INFINITY ? expf(part_m[w][i] - high) : 0.f;      // (a wave that saw nothing: zero)
        if (part_m[w][i] > -INFINITY || part_l[w][i] != 0.f) {
          total += f * part_l[w][i];
          sum += f * part_o[w][i][d];
        }
      }
      sum = sum / total;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) to[e] = sum[e];
  }
}

// Shapes of the kernel above: a rule on the model's sizes alone, so that all rows of a model take the same one.
bool attention_f32_takes(int nh, int nkv, int hd, int B) {
  return (hd == 16 || hd == 32 || hd == 64 || hd == 128) && nh / nkv <= 16 && B % 4 == 0;
}

template <int NT>
void launch_attention_f32(const float* q, int q_stride, float* out, int out_stride, const float* kcache, const float* vcache,
                          const int* tables, int table_stride, const int* row_seq, const int* ctx_lens, int T, int nh, int nkv,
                          int B, float scale, int window, const float2* cos_sin, const int* slots, hipStream_t s) {
  // As many rows a workgroup as leave each CU one (the smallest heads' registers allow two), where the 16 items hold them.
  // Single rows of as many sequences, us, the kernel above / a full tile walked by the same wave for each sequence, all keys of a
  // chunk multiplied / this: 32 heads over 32 kv heads of 64, 64 rows of 16 tokens 12.6 / 71.8 / 8.9, of 600 413 / 238 / 123; 256
  // rows of 16 34 / 154 / 28; 8 over 8 of 128, 256 rows of 16 19 / 134 / 14; 32 over 4 of 64, 8 rows of 16 9.3 / 8.0 / 5.8.
  const long long units = static_cast<long long>(T) * nkv;
  const int per = static_cast<int>(units <= (NT == 1 ? 512 : 256) ? 1 : std::min<long long>((units + 255) / 256, 16 / (nh / nkv)));
  const unsigned blocks = static_cast<unsigned>((T + per - 1) / per) * nkv;
  auto* kernel = slots ? attention_f32_kernel<NT, true> : attention_f32_kernel<NT, false>;
  kernel<<<blocks, f32_waves<NT>() * kWave, 0, s>>>(q, q_stride, out, out_stride, kcache, vcache, tables, table_stride, row_seq, ctx_lens, T, nh, nkv,
                                                    per, B, scale, window, cos_sin, slots);
}

}  // namespace kvcm

using namespace kvcm;

// out = {vector registers per lane, bytes of LDS per workgroup, workgroups that fit on one CU,
// threads per workgroup} of the bfloat16 kernel at this head size.
extern "C" int kvcm_attention_generic_info(int hd, int* out) {
  hipFuncAttributes a;
  const size_t lds = sizeof(float) * kAttnWaves * hd;
  int per_cu = 0;
  KVCM_REQUIRE(hipFuncGetAttributes(&a, reinterpret_cast<const void*>(&attention_generic_kernel<bf16_t>)) == hipSuccess &&
                   hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, attention_generic_kernel<bf16_t>,
                                                                kAttnWaves * kWave, lds) == hipSuccess,
               "attention_generic_info: the runtime gave no attributes");
  out[0] = a.numRegs; out[1] = static_cast<int>(a.sharedSizeBytes + lds); out[2] = per_cu; out[3] = kAttnWaves * kWave;
  return 0;
}

extern "C" int kvcm_attention_generic(const void* q, int dtype, int q_stride, void* out, int out_stride,
                                      const void* kcache, const void* vcache, const int* tables, int table_stride,
                                      const int* row_seq, const int* ctx_lens, int T, int nh, int nkv, int hd,
                                      int B, float scale, int window, hipStream_t s) {
  if (T == 0) return 0;
  KVCM_REQUIRE(T > 0 && nh > 0 && nkv > 0 && B > 0, "attention: bad sizes T=%d heads=%d kv_heads=%d B=%d", T, nh, nkv, B);
  KVCM_REQUIRE(nh % nkv == 0, "attention: %d query heads are not a multiple of %d kv heads", nh, nkv);
  KVCM_REQUIRE(hd % 8 == 0 && hd > 0 && hd <= kMaxHeadDim,
               "attention: head_dim %d is not supported (multiples of 8 up to %d are)", hd, kMaxHeadDim);
  KVCM_REQUIRE(q_stride >= nh * hd && out_stride >= nh * hd, "attention: row strides too small");
  KVCM_REQUIRE(window >= 0, "attention: negative window");
  const long long items = static_cast<long long>(T) * nh;
  const long long blocks = (items + kAttnWaves - 1) / kAttnWaves;
  KVCM_REQUIRE(blocks < (1ll << 31), "attention: too many rows");
  const size_t lds = sizeof(float) * kAttnWaves * hd;
  auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  if (dtype == kF32 && attention_f32_takes(nh, nkv, hd, B) && q_stride % 4 == 0 && aligned(q) && aligned(kcache) && aligned(vcache)) {
    KVCM_REQUIRE(static_cast<long long>(T) * nkv < (1ll << 31), "attention: too many rows");
    auto* launch = hd == 16 ? launch_attention_f32<1> : hd == 32 ? launch_attention_f32<2> : hd == 64 ? launch_attention_f32<4>
                                                                                              : launch_attention_f32<8>;
    launch(static_cast<const float*>(q), q_stride, static_cast<float*>(out), out_stride, static_cast<const float*>(kcache),
           static_cast<const float*>(vcache), tables, table_stride, row_seq, ctx_lens, T, nh, nkv, B, scale, window, nullptr, nullptr, s);
    return launch_status("attention_f32");
  }
  if (dtype == kF32)
    attention_generic_kernel<float><<<dim3(static_cast<unsigned>(blocks)), kAttnWaves * kWave, lds, s>>>(
        static_cast<const float*>(q), q_stride, static_cast<float*>(out), out_stride,
        static_cast<const float*>(kcache), static_cast<const float*>(vcache), tables, table_stride, row_seq,
        ctx_lens, items, nh, nkv, hd, B, scale, window);
  else if (dtype == kBF16)
    attention_generic_kernel<bf16_t><<<dim3(static_cast<unsigned>(blocks)), kAttnWaves * kWave, lds, s>>>(
        static_cast<const bf16_t*>(q), q_stride, static_cast<bf16_t*>(out), out_stride,
        static_cast<const bf16_t*>(kcache), static_cast<const bf16_t*>(vcache), tables, table_stride, row_seq,
        ctx_lens, items, nh, nkv, hd, B, scale, window);
  else KVCM_REQUIRE(false, "attention: unknown dtype %d", dtype);
  return launch_status("attention_generic");
}

// 1 when kvcm_attention_f32_decode takes the shape, else 0.
extern "C" int kvcm_attention_f32_decode_supported(int nh, int nkv, int hd, int B) {
  return nkv > 0 && nh > 0 && nh % nkv == 0 && B > 0 && attention_f32_takes(nh, nkv, hd, B);
}

// 32-bit rows of T different sequences, from the projection's rows [q | k | v] to the attention's: q and k rotated by cos_sin [T][hd / 2]
// (null: not), keys and values stored to slots [T] (negative: not stored).  The bits of kvcm_rope_cache and kvcm_attention_generic; the
// rows themselves stay as they are.
extern "C" int kvcm_attention_f32_decode(const float* qkv, int qkv_stride, float* out, int out_stride, const float* cos_sin, const int* slots,
                                         float* kcache, float* vcache, const int* tables, int table_stride, const int* row_seq, const int* ctx_lens,
                                         int T, int nh, int nkv, int hd, int B, float scale, int window, hipStream_t s) {
  if (T == 0) return 0;
  KVCM_REQUIRE(kvcm_attention_f32_decode_supported(nh, nkv, hd, B), "attention_f32_decode: unsupported shape heads=%d kv_heads=%d head_dim=%d page=%d", nh, nkv, hd, B);
  KVCM_REQUIRE(T > 0 && static_cast<long long>(T) * nkv < (1ll << 31), "attention_f32_decode: bad row count %d", T);
  KVCM_REQUIRE(qkv && out && slots && kcache && vcache && tables && row_seq && ctx_lens, "attention_f32_decode: null operand");
  KVCM_REQUIRE(qkv_stride >= (nh + 2 * nkv) * hd && out_stride >= nh * hd && window >= 0, "attention_f32_decode: row strides too small or a negative window");
  const auto piece = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  KVCM_REQUIRE(piece(qkv) && qkv_stride % 4 == 0 && piece(kcache) && piece(vcache) && reinterpret_cast<uintptr_t>(cos_sin) % 8 == 0,
               "attention_f32_decode: operands must be 16-byte aligned");
  auto* launch = hd == 16 ? launch_attention_f32<1> : hd == 32 ? launch_attention_f32<2> : hd == 64 ? launch_attention_f32<4> : launch_attention_f32<8>;
  launch(qkv, qkv_stride, out, out_stride, kcache, vcache, tables, table_stride, row_seq, ctx_lens, T, nh, nkv, B, scale, window,
         reinterpret_cast<const float2*>(cos_sin), slots, s);
  return launch_status("attention_f32_decode");
}
