// The attention over a window and pooled blocks (attention_window_pool.hip) for runs of consecutive
// positions, on the matrix cores: a workgroup of four waves takes 64 consecutive rows of one run and one
// query head, walks the keys those rows can see 64 at a time (first the pooled blocks from block 0, then the
// tokens in chunks that start at absolute multiples of 64), stages each chunk's keys and values once in LDS
// as bfloat16 and multiplies with v_mfma_f32_16x16x32_bf16, transposed: S^T = K Q^T (a wave: 64 keys x 16 rows), the
// mask and a running-maximum softmax in 32-bit on the accumulators, whose lane holds sixteen keys of one row, P rounded to
// bfloat16, which is the second operand of O^T += V^T P^T as it lies there (a tile's 16 keys are dealt out so that a lane's
// eight of 32 are consecutive).  Which keys a row sees is decided per score
// (window, causality, blocks wholly before the window) in the chunks at the ends of what the tile sees, so a chunk that some
// rows of the tile do not see costs them nothing but zeros; a row's chunks and their order depend on its own position only.
// Bound by its vector instructions: with P handed over through LDS, a row's statistics over 16 lanes, the mask at every score
// and divisions by the page size this took 86 us for 2,048 rows of 32 heads of 64 in a window of 512 with pooled blocks,
// 54 us as it is, with the same error against 64 bits (without pooled blocks 71 and 46 us, with capped scores 81 and 58 us).  The bound of four workgroups on a CU (128
// registers) leaves heads of 64 with 76 bytes of scratch a lane.  The first
// keep_first tokens of a sequence may stay visible beyond the window (chunks of their own, from token 0), and the
// scores may be capped, score <- c tanh(score / c), and a bias that grows with the distance may be taken off them,
// score <- score - slope_h * (i - j) with a slope per query head (tokens only: not beside pooled blocks); the output may be
// multiplied with sigmoid(gate) before it is stored, element by element or head by head, and by a constant factor.  With a
// chunk size in the window's place a row sees its own chunk of positions only; with a sink, a key without a value (score 0, or
// a number per query head) joins the softmax's denominator.
// bfloat16 storage only; sizes d and dv in multiples of 8, pages whose size is a multiple of 8 and divides 64.
#include <cfloat>

#include "common.h"
#include "kvcm_hip.h"

namespace kvcm {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
typedef float pooled_four __attribute__((ext_vector_type(4), aligned(4)));      // (pooled entries may lie at any float)

constexpr int kTileRows = 64, kChunk = 64, kVtPitch = kChunk + 8;
constexpr float kMasked = -1.0e30f;

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  return uint32_t(float_to_bf16_bits(a)) | (uint32_t(float_to_bf16_bits(b)) << 16);
}

// tanh of a score: an odd polynomial up to 5/8 (x + x^3 p(x^2), p fitted to 4e-9 of the result), (1 - e) / (1 + e) with
// e = 2^(-2 |x| log2 e) by the hardware's exp2 and reciprocal beyond.  As exact as tanhf, which is some thirty instructions of a
// score's fifty: over [-12, 12] at most 1.6e-7 of the result off (tanhf 1.7e-7), 2.7e-8 on average up to 5/8 and 4e-8 beyond (the same).
__device__ __forceinline__ float score_tanh(float x) {
  const float y = x * x;
  const float p = fmaf(y, fmaf(y, fmaf(y, fmaf(y, -0.005704974f, 0.020639075f), -0.05373971f), 0.13331442f), -0.3333328f);
  const float near = fmaf(x * y, p, x);
  const float e = __builtin_amdgcn_exp2f(-2.88539008177792681f * fabsf(x));
  const float far = copysignf(fmaf(-2.0f * e, __builtin_amdgcn_rcpf(1.0f + e), 1.0f), x);
  return y < 0.390625f ? near : far;
}

// DP: key size padded to a multiple of 32; DVT: tiles of 16 value columns
// (bounds that keep the accumulators in ordinary registers and, at sizes up to 64, four workgroups on a CU)
template <int DP, int DVT>
__global__ void __launch_bounds__(256, DP <= 64 && DVT <= 4 ? 4 : DVT <= 8 ? 2 : 1)
    attention_window_pool_tiles_kernel(const uint16_t* __restrict__ q, int ldq, uint16_t* __restrict__ out, int ldo,
                                       const uint16_t* __restrict__ kcache, const uint16_t* __restrict__ vcache,
                                       const float* __restrict__ pk, const float* __restrict__ pv,
                                       const int* __restrict__ tables, int table_stride, const int* __restrict__ run_start,
                                       const int* __restrict__ seq_start, const float* __restrict__ head_scale,
                                       const float* __restrict__ dist_slope, const float* __restrict__ gate, int ldg, int tiles_per_seq,
                                       int nh, int nkv, int d, int dv, int B, float scale, int window, int P, int E,
                                       int keep_first, float softcap, int chunk, int sink, const float* __restrict__ sink_logit, int gate_heads, float out_scale) {
  constexpr int KP = DP + 8, KS = DP / 32, DVP = DVT * 16;
  __shared__ __attribute__((aligned(16))) uint16_t Ks[kChunk][KP];
  __shared__ __attribute__((aligned(16))) uint16_t Vt[DVP][kVtPitch];
  const int s = blockIdx.x / tiles_per_seq, tile = blockIdx.x % tiles_per_seq, head = blockIdx.y;
  const int run0 = run_start[s], run_len = run_start[s + 1] - run0;
  if (tile * kTileRows >= run_len) return;
  const int r0 = run0 + tile * kTileRows;
  const int nrows = run_len - tile * kTileRows < kTileRows ? run_len - tile * kTileRows : kTileRows;
  const int p0 = seq_start[s] + tile * kTileRows, p_last = p0 + nrows - 1;
  const int kvh = head / (nh / nkv);
  const int* table = tables + size_t(s) * table_stride;
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
  const int col = lane % 16, quad = lane / 16;
  // scores are kept in units of log 2 (the factor rides along with the scale), so that the exponentials are the
  // hardware's exp2: a bfloat16 probability keeps 8 bits of it
  // (with a cap c on the scores, score <- c tanh(score / c): f then brings the product to score / c and the capped
  // value is scaled to units of log 2 afterwards)
  constexpr float kLog2e = 1.44269504088896341f;
  const float f = (head_scale ? scale * head_scale[head] : scale) * (softcap > 0.f ? 1.0f / softcap : kLog2e);
  const float cap2 = softcap * kLog2e;
  const float slope2 = dist_slope ? dist_slope[head] * kLog2e : 0.f;      // the bias in units of log 2, like the scores

  // this wave's 16 query rows as second operands (row = lane % 16, k = 8 * (lane / 16) .. + 8 of every 32)
  bf16x8 qf[KS];
  const int my_row = wave * 16 + col;      // the row whose scores and output this lane holds
  {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int k = ks * 32 + quad * 8;
      uint4 v = {0u, 0u, 0u, 0u};
      if (my_row < nrows && k < d) v = *reinterpret_cast<const uint4*>(q + size_t(r0 + my_row) * ldq + size_t(head) * d + k);
      qf[ks] = __builtin_bit_cast(bf16x8, v);
    }
  }
  const int pos = my_row < nrows ? p0 + my_row : -1;
  const int seen_blocks = (P > 0 && window > 0 && pos + 1 > window) ? (pos + 1 - window) / P : 0;
  const int lo_pos = chunk > 0 ? pos / chunk * chunk : window > 0 ? pos - window + 1 : 0;      // the first token of the row's window or chunk
  float m = kMasked;
  f32x4 o[DVT], lsum = {0.f, 0.f, 0.f, 0.f};      // O^T: column = row, rows = dims 16 vt + 4 quad + i; the sums of P by a product with ones
#pragma unroll
  for (int vt = 0; vt < DVT; ++vt) o[vt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint32_t one2 = 0x3F803F80u;
  const bf16x8 ones = __builtin_bit_cast(bf16x8, uint4{one2, one2, one2, one2});

  const int blocks = (P > 0 && window > 0 && p_last + 1 > window) ? (p_last + 1 - window) / P : 0;      // of the tile's last row
  const int t_lo = chunk > 0 ? p0 / chunk * chunk : (window > 0 && p0 + 1 > window) ? p0 + 1 - window : 0;
  const int block_chunks = (blocks + kChunk - 1) / kChunk;
  // the sequence's first tokens that stay visible beyond the window: those before the tile's first seen token get chunks
  // of their own, from token 0, between the blocks and the window (every row of the tile sees all of them)
  const int kept = keep_first < t_lo ? keep_first : t_lo;
  const int head_chunks = block_chunks + (kept + kChunk - 1) / kChunk;
  // tokens from here to p0 are seen by every row of the tile
  const int all_from = chunk > 0 ? p_last / chunk * chunk : window > 0 ? p_last - window + 1 : 0;
  const int page_bits = 31 - __builtin_clz(B);      // (a page size that is a multiple of 8 and divides 64 is a power of two)
  const int first_token_chunk = t_lo / kChunk, last_token_chunk = p_last / kChunk;
  const int chunks = head_chunks + (last_token_chunk - first_token_chunk + 1);
  auto chunk_start = [&](int c) {
    return c < block_chunks ? c * kChunk : c < head_chunks ? (c - block_chunks) * kChunk : (first_token_chunk + (c - head_chunks)) * kChunk;
  };

  // A chunk of tokens on its way from the pages to LDS, held in registers meanwhile: the next chunk is requested
  // before the current one is multiplied.  Loads are unconditional, from places clamped into the sequence, and
  // masked afterwards (a branch around a load would make each wait for the one before).
  constexpr int KQ = (kChunk * (DP / 8) + 255) / 256, VQ = (DVP * (kChunk / 8) + 255) / 256;
  uint4 kreg[KQ], vreg[VQ];
  // a chunk of tokens c0 .. c0 + 63 of which the stretch [lo, hi] may be read (the window up to the newest token, or the
  // kept first tokens)
  auto request_tokens = [&](int c0, int lo, int hi) {
#pragma unroll
    for (int qq = 0; qq < KQ; ++qq) {
      const int e = tid + qq * 256;
      const int key = (e / (DP / 8)) % kChunk, k = (e % (DP / 8)) * 8, t = c0 + key;
      // (pages that the window has passed may have been given back: nothing outside the stretch is read)
      const int tl = t < lo ? lo : t;
      const int tc = tl <= hi ? tl : hi, kc = k < d ? k : d - 8;
      const uint4 v = *reinterpret_cast<const uint4*>(kcache + (((size_t(table[tc >> page_bits]) * nkv + kvh) << page_bits) + (tc & (B - 1))) * d + kc);
      kreg[qq] = (t <= hi && k < d) ? v : uint4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int qq = 0; qq < VQ; ++qq) {
      const int e = tid + qq * 256;
      const int cc = (e / (kChunk / 8)) % DVP, piece = e % (kChunk / 8), t = c0 + piece * 8;
      const int tl = t < (lo / 8) * 8 ? (lo / 8) * 8 : t;
      const int tc = tl <= hi ? tl : (hi / 8) * 8, ccl = cc < dv ? cc : dv - 1;
      uint4 v = *reinterpret_cast<const uint4*>(vcache + (((size_t(table[tc >> page_bits]) * nkv + kvh) * dv + ccl) << page_bits) + (tc & (B - 1)));
      v = keep_first_bf16(v, hi + 1 - tc < 8 ? hi + 1 - tc : 8);      // beyond the stretch: whatever was there (counted from the piece that was read)
      vreg[qq] = cc < dv ? v : uint4{0u, 0u, 0u, 0u};
    }
  };
  auto request_chunk = [&](int c) {      // c >= block_chunks
    if (c < head_chunks) request_tokens(chunk_start(c), 0, kept - 1);
    else request_tokens(chunk_start(c), t_lo, p_last);
  };
  auto stage_tokens = [&]() {
#pragma unroll
    for (int qq = 0; qq < KQ; ++qq) {
      const int e = tid + qq * 256;
      if (e < kChunk * (DP / 8)) *reinterpret_cast<uint4*>(&Ks[e / (DP / 8)][(e % (DP / 8)) * 8]) = kreg[qq];
    }
#pragma unroll
    for (int qq = 0; qq < VQ; ++qq) {
      const int e = tid + qq * 256;
      if (e < DVP * (kChunk / 8)) *reinterpret_cast<uint4*>(&Vt[e / (kChunk / 8)][(e % (kChunk / 8)) * 8]) = vreg[qq];
    }
  };

  // where block b's entry (the last one's beyond the blocks) lies: in the page of its last token
  constexpr int PVQ = (kChunk * (DVP / 4) + 255) / 256;
  auto pooled_entry = [&](int b) {
    b = b < blocks ? b : blocks - 1;
    const int pgi = (b * P + P - 1) >> page_bits;
    return (size_t(table[pgi]) * nkv + kvh) * E + (b - (pgi << page_bits) / P);
  };

  for (int c = 0; c < chunks; ++c) {
    const bool pooled = c < block_chunks, early = !pooled && c < head_chunks;
    const int c0 = chunk_start(c);
    if (!pooled && c == block_chunks) request_chunk(c);      // the first chunk of tokens: nobody asked for it yet
    __syncthreads();      // the chunk before is done with Ks and Vt
    if (pooled) {      // (loads from places clamped to the last block, masked afterwards)
      {
        pooled_four x[KQ][2];
#pragma unroll
        for (int qq = 0; qq < KQ; ++qq) {
          const int e = tid + qq * 256, k = (e % (DP / 8)) * 8;
          const float* src = pk + pooled_entry(c0 + (e / (DP / 8)) % kChunk) * d + (k < d ? k : d - 8);
          x[qq][0] = *reinterpret_cast<const pooled_four*>(src);
          x[qq][1] = *reinterpret_cast<const pooled_four*>(src + 4);
        }
#pragma unroll
        for (int qq = 0; qq < KQ; ++qq) {
          const int e = tid + qq * 256, key = e / (DP / 8), k = (e % (DP / 8)) * 8;
          uint4 v = {pack_bf16(x[qq][0].x, x[qq][0].y), pack_bf16(x[qq][0].z, x[qq][0].w), pack_bf16(x[qq][1].x, x[qq][1].y),
                     pack_bf16(x[qq][1].z, x[qq][1].w)};
          if (c0 + key >= blocks || k >= d) v = uint4{0u, 0u, 0u, 0u};
          if (e < kChunk * (DP / 8)) *reinterpret_cast<uint4*>(&Ks[key][k]) = v;
        }
      }
      __builtin_amdgcn_sched_barrier(0);      // (keys, then values: both at once do not fit the registers)
      {
        pooled_four x[PVQ];
#pragma unroll
        for (int qq = 0; qq < PVQ; ++qq) {
          const int e = tid + qq * 256, cc = (e % (DVP / 4)) * 4;
          x[qq] = *reinterpret_cast<const pooled_four*>(pv + pooled_entry(c0 + (e / (DVP / 4)) % kChunk) * dv + (cc < dv ? cc : dv - 4));
        }
#pragma unroll
        for (int qq = 0; qq < PVQ; ++qq) {
          const int e = tid + qq * 256, key = e / (DVP / 4), cc = (e % (DVP / 4)) * 4;
          const float v[4] = {x[qq].x, x[qq].y, x[qq].z, x[qq].w};
          const bool in = c0 + key < blocks && cc < dv;
          if (e < kChunk * (DVP / 4))
#pragma unroll
            for (int i = 0; i < 4; ++i) Vt[cc + i][key] = in ? float_to_bf16_bits(v[i]) : uint16_t(0);
        }
      }
    } else {
      stage_tokens();
    }
    __syncthreads();
    if (!pooled && c + 1 < chunks) request_chunk(c + 1);      // on its way while this chunk is multiplied

    // scores of 64 keys x 16 rows, two groups of 32 keys as two tiles each: row r of tile t is key 8 (r / 4) + 4 t + r % 4 of
    // the group, so that this lane's sc[g][t][i] is key 8 quad + 4 t + i of it
    f32x4 sc[2][2];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        sc[g][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int key = g * 32 + 8 * (col / 4) + 4 * t + col % 4;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const bf16x8 kf = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(&Ks[key][ks * 32 + quad * 8]));
          sc[g][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[ks], sc[g][t], 0, 0, 0);
        }
      }
    const int key0 = c0 + 8 * quad;
    const bool all_see = !pooled && !early && c0 >= all_from && c0 + kChunk - 1 <= p0;      // (the same for the whole tile)
    float sv[16];      // of key0 + 32 (j / 8) + j % 8
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      sv[j] = sc[j / 8][j / 4 % 2][j % 4] * f;
      if (softcap > 0.f) sv[j] = cap2 * score_tanh(sv[j]);
      if (dist_slope) sv[j] = fmaf(-slope2, float(pos - (key0 + j / 8 * 32 + j % 8)), sv[j]);
    }
    uint32_t seen = 0xFFFFu;      // bit j
    if (!all_see) {
      seen = 0u;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int key = key0 + j / 8 * 32 + j % 8;
        const bool vis = pooled ? key < seen_blocks
                         : early ? (key < kept && pos >= 0)
                                 : (key >= t_lo && key <= pos && (key >= lo_pos || key < keep_first));
        seen |= vis ? 1u << j : 0u;
        sv[j] = vis ? sv[j] : kMasked;
      }
    }
    float mx = kMasked;
#pragma unroll
    for (int j = 0; j < 16; ++j) mx = fmaxf(mx, sv[j]);
    const float m_new = fmaxf(m, rows_max(mx));
    const float alpha = __builtin_amdgcn_exp2f(m - m_new);
    m = m_new;
#pragma unroll
    for (int j = 0; j < 16; ++j) sv[j] = __builtin_amdgcn_exp2f(sv[j] - m_new);
    if (!all_see) {
#pragma unroll
      for (int j = 0; j < 16; ++j) sv[j] = seen >> j & 1u ? sv[j] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) lsum[i] *= alpha;
#pragma unroll
    for (int vt = 0; vt < DVT; ++vt)
#pragma unroll
      for (int i = 0; i < 4; ++i) o[vt][i] *= alpha;
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const bf16x8 pf = __builtin_bit_cast(bf16x8, uint4{pack_bf16(sv[8 * g], sv[8 * g + 1]), pack_bf16(sv[8 * g + 2], sv[8 * g + 3]),
                                                         pack_bf16(sv[8 * g + 4], sv[8 * g + 5]), pack_bf16(sv[8 * g + 6], sv[8 * g + 7])});
      lsum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pf, lsum, 0, 0, 0);      // (of what is multiplied, so that the weights add up to one)
#pragma unroll
      for (int vt = 0; vt < DVT; ++vt) {
        const bf16x8 vf = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(&Vt[vt * 16 + col][g * 32 + quad * 8]));
        o[vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf, o[vt], 0, 0, 0);
      }
    }
  }
  const float sl2 = sink_logit ? sink_logit[head] * kLog2e : 0.f;
  float l = lsum[0], factor = out_scale;
  if (sink) {      // the head's sink (a score of 0 without a number of its own) joins the denominator, in units of log 2 too
    const float m_all = fmaxf(m, sl2);
    const float keep = __builtin_amdgcn_exp2f(m - m_all);
    l = l * keep + __builtin_amdgcn_exp2f(sl2 - m_all);
    factor *= keep;
  }
  if (my_row >= nrows) return;
  float inv = factor / l;
  if (gate && gate_heads) inv *= 1.0f / (1.0f + expf(-gate[size_t(r0 + my_row) * ldg + head]));      // one gate per head
  uint16_t* orow = out + size_t(r0 + my_row) * ldo + size_t(head) * dv;
  const float* grow = gate && !gate_heads ? gate + size_t(r0 + my_row) * ldg + size_t(head) * dv : nullptr;      // a gate per element
  const bool wide = ldo % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 8 == 0;
#pragma unroll
  for (int vt = 0; vt < DVT; ++vt) {
    const int c4 = vt * 16 + 4 * quad;      // (dv is a multiple of 8: the four lie inside or outside)
    if (c4 >= dv) continue;
    float res[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      res[i] = o[vt][i] * inv;
      if (grow) res[i] *= 1.0f / (1.0f + expf(-grow[c4 + i]));
    }
    if (wide) {
      *reinterpret_cast<uint2*>(orow + c4) = uint2{pack_bf16(res[0], res[1]), pack_bf16(res[2], res[3])};
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) orow[c4 + i] = float_to_bf16_bits(res[i]);
    }
  }
}

template <int DP>
int launch_tiles(int dvt, dim3 grid, hipStream_t s, const uint16_t* q, int ldq, uint16_t* out, int ldo, const uint16_t* kc,
                 const uint16_t* vc, const float* pk, const float* pv, const int* tables, int table_stride, const int* run_start,
                 const int* seq_start, const float* head_scale, const float* dist_slope, const float* gate, int ldg, int tiles_per_seq,
                 int nh, int nkv, int d, int dv, int B, float scale, int window, int P, int E, int keep_first, float softcap,
                 int chunk, int sink, const float* __restrict__ sink_logit, int gate_heads, float out_scale) {
#define KVCM_TILES(DVT)                                                                                                     \
  attention_window_pool_tiles_kernel<DP, DVT><<<grid, 256, 0, s>>>(q, ldq, out, ldo, kc, vc, pk, pv, tables, table_stride,   \
                                                                   run_start, seq_start, head_scale, dist_slope, gate, ldg, tiles_per_seq, \
                                                                   nh, nkv, d, dv, B, scale, window, P, E, keep_first, softcap, chunk, sink, sink_logit, gate_heads, out_scale)
  if (dvt <= 2) KVCM_TILES(2);
  else if (dvt <= 4) KVCM_TILES(4);
  else if (dvt <= 8) KVCM_TILES(8);
  else KVCM_TILES(16);
#undef KVCM_TILES
  return launch_status("attention_window_pool_tiles");
}

}  // namespace kvcm

using namespace kvcm;

extern "C" {

int kvcm_attention_window_pool_tiles_supported(int d, int dv, int B) {
  return d > 0 && d % 8 == 0 && d <= 128 && dv > 0 && dv % 8 == 0 && dv <= 256 && B % 8 == 0 && B > 0 && kChunk % B == 0;
}

// q, out, pages: bfloat16; pooled entries: 32-bit.  S sequences with runs of up to max_run rows.
int kvcm_attention_window_pool_tiles(const void* q, int ldq, void* out, int ldo, const void* kcache, const void* vcache,
                                     const float* pk, const float* pv, const int* tables, int table_stride,
                                     const int* run_start, const int* seq_start, const float* head_scale, const float* dist_slope,
                                     const float* gate, int ldg, int S, int max_run, int nh, int nkv, int d, int dv, int B, float scale, int window, int P,
                                     int E, int keep_first, float softcap, int chunk, int sink, const float* __restrict__ sink_logit, int gate_heads, float out_scale, hipStream_t s) {
  if (S == 0 || max_run == 0) return 0;
  KVCM_REQUIRE(S > 0 && max_run > 0 && nh > 0 && nkv > 0 && nh % nkv == 0, "attention_window_pool_tiles: bad sizes");
  KVCM_REQUIRE(kvcm_attention_window_pool_tiles_supported(d, dv, B),
               "attention_window_pool_tiles: key size %d, value size %d, pages of %d are not supported", d, dv, B);
  KVCM_REQUIRE(ldq >= nh * d && ldo >= nh * dv && ldq % 8 == 0 && reinterpret_cast<uintptr_t>(q) % 16 == 0,
               "attention_window_pool_tiles: q rows must be 16-byte aligned and long enough");
  KVCM_REQUIRE(window >= 0 && P >= 0 && (P == 0 || (pk && pv && E == (B + P - 1) / P)),
               "attention_window_pool_tiles: pooled blocks need their entries");
  KVCM_REQUIRE(P == 0 || d % 8 == 0, "attention_window_pool_tiles: pooled keys are read eight at a time");
  KVCM_REQUIRE(keep_first >= 0 && softcap >= 0.f, "attention_window_pool_tiles: negative count of kept tokens or score cap");
  KVCM_REQUIRE(!dist_slope || P == 0, "attention_window_pool_tiles: a distance bias beside pooled blocks is not supported");
  KVCM_REQUIRE(!gate || ldg >= (gate_heads ? nh : nh * dv), "attention_window_pool_tiles: the gate's rows are too short");
  KVCM_REQUIRE(chunk >= 0 && (chunk == 0 || (window == 0 && P == 0 && keep_first == 0)),
               "attention_window_pool_tiles: a chunk beside a window, pooled blocks or kept first tokens is not supported");
  const int tiles_per_seq = (max_run + kTileRows - 1) / kTileRows;
  KVCM_REQUIRE(static_cast<long long>(S) * tiles_per_seq < (1ll << 31) && nh <= 65535, "attention_window_pool_tiles: too many rows");
  const dim3 grid(S * tiles_per_seq, nh);
  const int dvt = (dv + 15) / 16;
  const uint16_t* qq = static_cast<const uint16_t*>(q);
  uint16_t* oo = static_cast<uint16_t*>(out);
  const uint16_t* kc = static_cast<const uint16_t*>(kcache);
  const uint16_t* vc = static_cast<const uint16_t*>(vcache);
  if (d <= 32)
    return launch_tiles<32>(dvt, grid, s, qq, ldq, oo, ldo, kc, vc, pk, pv, tables, table_stride, run_start, seq_start, head_scale,
                            dist_slope, gate, ldg, tiles_per_seq, nh, nkv, d, dv, B, scale, window, P, E, keep_first, softcap, chunk, sink, sink_logit, gate_heads, out_scale);
  if (d <= 64)
    return launch_tiles<64>(dvt, grid, s, qq, ldq, oo, ldo, kc, vc, pk, pv, tables, table_stride, run_start, seq_start, head_scale,
                            dist_slope, gate, ldg, tiles_per_seq, nh, nkv, d, dv, B, scale, window, P, E, keep_first, softcap, chunk, sink, sink_logit, gate_heads, out_scale);
  return launch_tiles<128>(dvt, grid, s, qq, ldq, oo, ldo, kc, vc, pk, pv, tables, table_stride, run_start, seq_start, head_scale,
                           dist_slope, gate, ldg, tiles_per_seq, nh, nkv, d, dv, B, scale, window, P, E, keep_first, softcap, chunk, sink, sink_logit, gate_heads, out_scale);
}

}  // extern "C"
