// The attention half of a decoding layer in one launch, for at most 8 rows of different sequences (bfloat16): the QKV product with the
// scale of the norm before it, rotation, page write, attention over the paged context, the output product, its addition to the
// residual stream and the next norm's preparation (gemm_rows8.hip explains the two halves of the folded norm).  The reference runs
// these as eight kernels (src/model/llama.cpp:104-118).
//
// What bounds such a step is not bytes but the chain of launches: QKV 5.3, attention 10.2 and output product 4.8 us a layer at
// TinyLlama sizes and one row, of which the weights account for 3 us.  A launch costs 2.6 us from the last store to the next
// launch's first instructions, its first operands another 1.5 to 3 us, and the attention, which must wait for both, ran on 4 of 256
// CUs.  Here all three are workgroups of one launch.  They ask for their weights, keys and values while the ones before them
// work, and hand results on through memory, past the caches, in words that are their own flags: a buffer is full of kEmpty before
// the launch, a word that is something else is there.  No counter, no fence, no order between words is needed, and a hand-over
// costs 0.8 to 1 us.  Measured (us a layer: three launches / this one, eight layers of distinct weights in a graph, contexts of 600 and
// 1,900 tokens): TinyLlama sizes 1 row 18.5 / 11.7 and 18.9 / 12.0, 8 rows 20.1 / 13.7 and 21.6 / 16.8; width 4096, 8 KV heads of 128, 1
// row 33.9 / 29.0 and 34.3 / 29.0, 8 rows 42.1 / 33.1 and 49.5 / 41.8; 32 KV heads of 128, 1 row of 600 45.3 / 41.2.
//
// Nobody waits for a workgroup of a higher number: [QKV tiles | attention, a row's and KV head's parts in ascending order | output tiles],
// and workgroups are started in the order of their numbers on each XCD, so a launch that has the chip to itself always gets on.  Two at a time (engines with a
// stream each, or two processes) may not: a waiting workgroup keeps its place, and what waits in one launch can fill an XCD on which the other
// still has products to start, while the other does the same elsewhere.  So every wait has an end, after which the workgroup makes what it
// waits for itself: an attention workgroup the QKV tiles of its heads, an output tile all QKV tiles and all of the attention, in order, and
// then its own part again.  It is the same code on the same operands, which the launch leaves as they are, so whoever else makes a word
// too, and however late, stores the same bits; nothing depends on who runs beside whom.  This costs 0.3 to 0.4 us a layer (in the code's
// shape, no wait more).  Several streams of such layers at once, us a layer of each, three launches / this one: TinyLlama sizes, 8 rows of 600, two
// streams 26.0 / 20.0, three 29.5 / 25.5, four 33.4 / 33.4 to 44; width 4096, 8 KV heads, 8 rows of 1,900, whose 256 output tiles are all the places
// there are, 80.5 / 68, 120 / 128 to 375, 155 / 133 to 324: three or more engines of that size share a GPU better without (giving up takes an
// output tile some 2 ms, as it makes everything).
//
// Attention: a wave takes windows of 64 tokens (both products on the matrix cores, transposed, as in attention_decode_fused.hip), one
// each: `parts` workgroups of eight waves share a row's KV head, window 8 w + part belonging to wave w.  The last part adds the
// others' results to its own, and the newest token, whose key and value never leave the chip on their way (a score of its
// own, computed in 32 bits from the same bfloat16 values).  As one workgroup of two trips a wave the attention took 3.3 us after q had
// arrived, half of it in the vector instructions of one CU; two parts take 1.9 us, three or four 0.1 to 0.3 us more a layer.
//
// The output product's tiles wait for one word of the QKV product before they ask for their weights, so that QKV's come first
// (13.0 -> 11.8 us at one row); with more than two rows one wave looks whether every row and KV head has left something, then
// all read through the L2, and past the caches again what was too early (8 rows: 15.4 -> 15.1 us; 128 workgroups read 4 MB).
#include "common.h"
#include "kvcm_hip.h"

namespace kvcm {
namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2v;
typedef __attribute__((__vector_size__(2 * sizeof(float)))) float f32x2v;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
union Frag {
  uint4 u;
  uint64_t d[2];
  uint32_t w[4];
  bf16x8 v;
};
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  union { bf16x2v v; uint32_t u; } r;
  r.v = __builtin_convertvector(f32x2v{a, b}, bf16x2v);
  return r.u;
}
__device__ __forceinline__ float low_bf16(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float high_bf16(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

constexpr int kWaves = 8, kThreads = kWaves * kWave;
// products: units of 64 k, two groups of 8 columns a workgroup, four units of W and X on their way, 16 slices of K (a matrix
// instruction serves two: gemm_rows8.hip)
constexpr int kUnit = 64, kCols = 8, kGroups = 2, kTrip = 4, kSlots = 2 * kWaves;
constexpr int kWindow = 64;                 // tokens of a wave
constexpr int kMaxParts = 4;
constexpr float kNone = -1.0e30f;           // "no score": finite, so that differences stay finite
constexpr float kLate = 3.40282347e38f;     // a wave's largest score where q, the key or the value did not come
constexpr uint32_t kEmpty = 0xFFFFFFFFu;    // no 32-bit float rounded to bfloat16 has these bits; other words that would have them are stored as another NaN
// Looks at what is not there before a workgroup makes it itself.  A look takes some 0.8 us: an attention workgroup waits 50 us (its 12 to 40
// tiles then take it about 100), an output tile, which would have all of the launch to make, a millisecond at each of its waits.
constexpr int kNearPolls = 64, kFarPolls = 1024;
constexpr int kOwnPolls = 1 << 18;          // ... at what the workgroup has stored itself: there at the first or second look

struct FrontArgs {
  const uint16_t *X, *Wqkv, *Wo;
  const float* ss_in;
  float* resid; const void* g; uint16_t* xg; float* ss_out;
  const float2* cos_sin; const int *slots, *tables, *row_seq, *ctx_lens;
  uint16_t *kcache, *vcache;
  uint32_t *now, *next;      // handed over in this launch: q, k, v [M][width] as floats, attention [M][nh hd / 2] as pairs, parts; emptied for the next
  int ldx, ldqkv, ldo, tiles_in, M, H, g_f32, table_stride, nh, nkv, B, seqs, parts, n_qkv, n_att, near_polls, far_polls;
  uint32_t per_page;
  float inv_width, eps, scale;
};
__device__ __forceinline__ uint32_t take(const uint32_t* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ uint64_t take_two(const void* p) {
  return __hip_atomic_load(static_cast<const uint64_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void leave(uint32_t* p, uint32_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ uint32_t filled(float v) {
  const uint32_t w = __float_as_uint(v);
  return w == kEmpty ? 0x7FC00000u : w;
}
// 2^(s - top), nothing for what is masked.  (The hardware's exp2: exact to an ulp, but a share below 2^-126 is zero where exp2f's is 2^-149 at the least.  Values
// are at most 2^128, so what is lost matters where one's value is 2^117 times the result's; exp2f costs 0.3 us a layer at width 2,048, 2 at 4,096.)
__device__ __forceinline__ float share(float s, float top) { return s > 0.5f * kNone ? __builtin_amdgcn_exp2f(s - top) : 0.f; }
__device__ __forceinline__ bool empty_half(uint64_t v) { return uint32_t(v) == kEmpty || uint32_t(v >> 32) == kEmpty; }

// A lane's slice of K, in units; `main` and `most`: what both slices of its wave, and the longer of them, have.
struct Slice {
  int lo, cnt, main, most, units;
  __device__ Slice(int units_, int slot) : units(units_) {
    lo = units * slot / kSlots;
    cnt = units * (slot + 1) / kSlots - lo;
    const int o = units * (slot ^ 1) / kSlots, oc = units * ((slot ^ 1) + 1) / kSlots - o;
    main = __builtin_amdgcn_readfirstlane(cnt < oc ? cnt : oc);
    most = __builtin_amdgcn_readfirstlane(cnt > oc ? cnt : oc);
  }
  __device__ size_t unit(int j) const {
    j = j < cnt ? j : (cnt > 0 ? cnt - 1 : 0);
    return size_t(lo + j < units ? lo + j : 0) * kUnit;
  }
};
struct WTrip { Frag w[kTrip][kGroups][2]; };
struct XTrip { Frag x[kTrip][2]; };
// What fragments hold before they are loaded is nothing (else the registers of one part of the work are kept for the next: 210 in place of 163)
template <class T>
__device__ __forceinline__ void nothing(T& t) {
  Frag* f = reinterpret_cast<Frag*>(&t);
#pragma unroll
  for (unsigned i = 0; i < sizeof(T) / sizeof(Frag); ++i) asm volatile("" : "=v"(f[i].u.x), "=v"(f[i].u.y), "=v"(f[i].u.z), "=v"(f[i].u.w));
}

template <int HD, int GROUP>
union Lds {
  struct { f32x4 red[kWaves][kGroups][kWave]; float rstd[8]; int late[kWaves]; } p;
  struct {
    uint16_t q[GROUP][HD], k_new[HD], v_new[HD];
    float red[kWaves][GROUP][HD + 4];
    float top[kWaves][16], sum[kWaves][16];
  } a;
};

// A tile of 16 columns of the QKV product (first) or of the output product.  True: what it waits for did not come, and it has
// stored nothing.  `made`: the workgroup has made all of that itself.
template <int HD, int GROUP>
__device__ __forceinline__ bool products(const FrontArgs& a, Lds<HD, GROUP>& L, int tid, bool first, int tile, bool made) {
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
  const int M = a.M, H = a.H, qw = a.nh * HD, width = qw + 2 * a.nkv * HD;
  const int n0 = tile * (kCols * kGroups);
  const int r = lane % 16, kq = lane / 16, half = r / 8, c = r % 8;
  const Slice s((first ? H : qw) / kUnit, 2 * wave + half);
  const uint16_t* W = first ? a.Wqkv : a.Wo;
  const int ldw = first ? a.ldqkv : a.ldo;
  const uint16_t* wrow[kGroups];
#pragma unroll
  for (int g = 0; g < kGroups; ++g) wrow[g] = W + size_t(n0 + g * kCols + c) * ldw + kq * 16;
  f32x4 acc[kGroups];
#pragma unroll
  for (int g = 0; g < kGroups; ++g) acc[g] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto fetch_w = [&](int j0, WTrip& t) {
#pragma unroll
    for (int d = 0; d < kTrip; ++d) {
      if (j0 + d >= s.most) break;
      const size_t off = s.unit(j0 + d);
#pragma unroll
      for (int g = 0; g < kGroups; ++g) {
        t.w[d][g][0].u = *reinterpret_cast<const uint4*>(wrow[g] + off);
        t.w[d][g][1].u = *reinterpret_cast<const uint4*>(wrow[g] + off + 8);
      }
    }
  };
  auto multiply = [&](int j0, const WTrip& t, const XTrip& x) {
#pragma unroll
    for (int d = 0; d < kTrip; ++d) {
      const int j = j0 + d;
      if (j >= s.most) break;
      Frag x0 = x.x[d][0], x1 = x.x[d][1];
      if (j >= s.main && j >= s.cnt) {
        x0.u = uint4{0u, 0u, 0u, 0u};
        x1.u = uint4{0u, 0u, 0u, 0u};
      }
#pragma unroll
      for (int g = 0; g < kGroups; ++g) {
        acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x0.v, t.w[d][g][0].v, acc[g], 0, 0, 0);
        acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x1.v, t.w[d][g][1].v, acc[g], 0, 0, 0);
      }
    }
  };
  // the first 128 threads' element of the result
  const int eg = tid / kWave, em = lane / 8, en = lane % 8;
  const int col = n0 + (eg < kGroups ? eg : 0) * kCols + en;
  const bool live = eg < kGroups && em < M;
  float resid_in = 0.f, g_in = 0.f;
  if (first) {
    const uint16_t* xrow = a.X + size_t(c < M ? c : 0) * a.ldx + kq * 16;
    auto fetch_x = [&](int j0, XTrip& t) {
#pragma unroll
      for (int d = 0; d < kTrip; ++d) {
        if (j0 + d >= s.most) break;
        const size_t off = s.unit(j0 + d);
        t.x[d][0].u = *reinterpret_cast<const uint4*>(xrow + off);
        t.x[d][1].u = *reinterpret_cast<const uint4*>(xrow + off + 8);
      }
    };
    float ssv[4], more = 0.f;
    if (a.ss_in) {
      const float* p = a.ss_in + size_t(wave < M ? wave : 0) * a.tiles_in;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int t = lane + q * kWave;
        ssv[q] = p[t < a.tiles_in ? t : 0];
      }
      if (a.tiles_in > 4 * kWave)
        for (int t = lane + 4 * kWave; t < a.tiles_in; t += kWave) more += p[t];
    }
    WTrip wa;
    XTrip xa;
    nothing(wa);
    nothing(xa);
    fetch_w(0, wa);
    fetch_x(0, xa);
    if (live) leave(a.next + size_t(em) * width + col, kEmpty);
    if (a.ss_in) {
      float part = more;
#pragma unroll
      for (int q = 0; q < 4; ++q) part += lane + q * kWave < a.tiles_in ? ssv[q] : 0.f;
      const float t = wave_sum(part);
      if (lane == 0) L.p.rstd[wave] = rsqrtf(t * a.inv_width + a.eps);
    }
    multiply(0, wa, xa);
    for (int j0 = kTrip; j0 < s.most; j0 += kTrip) {
      fetch_w(j0, wa);
      fetch_x(j0, xa);
      multiply(j0, wa, xa);
    }
  } else {
    if (eg < kGroups) {
      resid_in = a.resid[size_t(em < M ? em : 0) * H + col];
      g_in = a.g_f32 ? static_cast<const float*>(a.g)[col] : load_f(static_cast<const bf16_t*>(a.g) + col);
    }
    int polls = made ? kOwnPolls : a.far_polls;
    bool late = false;
    if (wave == 0) {      // QKV's weights first
      const uint32_t* word = a.now + size_t(tile) * a.n_qkv / (H / (kCols * kGroups)) * (kCols * kGroups);
      for (int poll = 0; poll < polls && take(word) == kEmpty; ++poll) __builtin_amdgcn_s_sleep(4);
    }
    __syncthreads();
    WTrip wa;
    nothing(wa);
    fetch_w(0, wa);
    const uint32_t* xrow = a.now + size_t(M) * width + (size_t(c < M ? c : 0) * qw + kq * 16) / 2;
    const bool cached = M > 2;
    if (cached) {
      if (wave == 0) {
        for (int poll = 0; poll < polls; ++poll) {
          bool none = false;
          for (int i = lane; i < M * a.nkv; i += kWave) none |= take(a.now + size_t(M) * width + size_t(i) * (GROUP * HD / 2)) == kEmpty;
          if (!__any(none)) break;
          __builtin_amdgcn_s_sleep(1);
        }
      }
      __syncthreads();
    }
    auto await = [&](int j0, XTrip& t) {
      bool none = false;
      if (cached) {
#pragma unroll
        for (int d = 0; d < kTrip; ++d) {
          if (j0 + d >= s.most) break;
          const uint32_t* src = xrow + s.unit(j0 + d) / 2;
          t.x[d][0].u = *reinterpret_cast<const uint4*>(src);
          t.x[d][1].u = *reinterpret_cast<const uint4*>(src + 4);
        }
#pragma unroll
        for (int d = 0; d < kTrip; ++d) {
          if (j0 + d >= s.most) break;
#pragma unroll
          for (int e = 0; e < 4; ++e) none |= empty_half(t.x[d][e / 2].d[e % 2]);
        }
        if (!__any(none)) return;
      }
      auto look = [&] {
        none = false;
#pragma unroll
        for (int d = 0; d < kTrip; ++d) {
          if (j0 + d >= s.most) break;
          const uint32_t* src = xrow + s.unit(j0 + d) / 2;
#pragma unroll
          for (int e = 0; e < 4; ++e) t.x[d][e / 2].d[e % 2] = take_two(src + 2 * e);
        }
#pragma unroll
        for (int d = 0; d < kTrip; ++d) {
          if (j0 + d >= s.most) break;
#pragma unroll
          for (int e = 0; e < 4; ++e) none |= empty_half(t.x[d][e / 2].d[e % 2]);
        }
        return __any(none);
      };
      bool empty = look();
      for (int poll = 0; empty && poll < polls; ++poll) {
        __builtin_amdgcn_s_sleep(1);
        empty = look();
      }
      if (empty) late = true, polls = 0;
    };
    XTrip xa;
    nothing(xa);
    await(0, xa);
    multiply(0, wa, xa);
    for (int j0 = kTrip; j0 < s.most; j0 += kTrip) {
      fetch_w(j0, wa);
      await(j0, xa);
      multiply(j0, wa, xa);
    }
    if (lane == 0) L.p.late[wave] = late;
    if (late) {      // (all of the results are then NaN, in both waves that add them up: they look at the flags only where they meet one)
#pragma unroll
      for (int g = 0; g < kGroups; ++g) acc[g] = f32x4{NAN, NAN, NAN, NAN};
    }
  }
#pragma unroll
  for (int g = 0; g < kGroups; ++g) L.p.red[wave][g][lane] = acc[g];
  __syncthreads();
  float v = 0.f;
  if (eg < kGroups) {
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      v += L.p.red[w][eg][(em / 4) * 16 + en][em % 4];
      v += L.p.red[w][eg][(2 + em / 4) * 16 + en + 8][em % 4];
    }
  }
  if (!first && !made && (eg >= kGroups || __any(v != v))) {
    int late = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) late |= L.p.late[w];
    if (__builtin_amdgcn_readfirstlane(late)) return true;
  }
  if (eg >= kGroups) return false;
  if (first) {
    if (a.ss_in) v *= L.p.rstd[em];
    if (live) leave(a.now + size_t(em) * width + col, __float_as_uint(round_to<bf16_t>(v)));
  } else {
    float xn = 0.f;
    if (live) {
      xn = resid_in + round_to<bf16_t>(v);
      a.resid[size_t(em) * H + col] = xn;
      a.xg[size_t(em) * H + col] = float_to_bf16_bits(g_in * round_to<bf16_t>(xn));
    }
    const float sq = group_sum<8>(xn * xn);
    if (live && en == 0) a.ss_out[size_t(em) * (H / kCols) + tile * kGroups + eg] = sq;
  }
  return false;
}

// Part `id` of (row, KV head, part): the row's query heads of that KV head over the part's windows.  True: q, the key or the value did not
// come, and no word is stored.  `made`: the workgroup has made them itself.
template <int HD, int GROUP>
__device__ __forceinline__ bool attend(const FrontArgs& a, Lds<HD, GROUP>& L, int tid, int id, bool made) {
  constexpr int KSTEPS = HD / 32, DT = HD / 16, HALF = HD / 2;
  constexpr int kPartWords = GROUP * (HD + 2);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
  const int part = id % a.parts, kvh = id / a.parts % a.nkv, row = id / a.parts / a.nkv;
  const bool merges = part == a.parts - 1;
  const int qw = a.nh * HD, width = qw + 2 * a.nkv * HD, B = a.B;
  const size_t head_elems = size_t(B) * HD, page_elems = head_elems * a.nkv;
  auto page_of = [&](int t) { return int(__umulhi(uint32_t(t), a.per_page)); };
  const int t_first = (wave * a.parts + part) * kWindow;
  const int entry = min(page_of(t_first + lane), a.table_stride - 1);
  int page = a.tables[size_t(row < a.seqs ? row : 0) * a.table_stride + entry];
  const int ctx_all = a.ctx_lens[row], slot = a.slots[row], seq = a.row_seq[row];
  const int ih = tid / HALF, ij = tid % HALF;
  static_assert((GROUP + 2) * HALF <= 2 * kThreads, "two pairs a thread");
  float2 rot = float2{1.0f, 0.0f};
  if (a.cos_sin) rot = a.cos_sin[size_t(row) * HALF + ij];
  const size_t a_at = size_t(a.M) * width, p_at = a_at + size_t(a.M) * qw / 2 + size_t(row * a.nkv + kvh) * (a.parts - 1) * kPartWords;
  const size_t out = a_at + (size_t(row) * qw + size_t(kvh) * GROUP * HD) / 2;
  if (merges) {
    for (int i = tid; i < GROUP * HALF; i += kThreads) leave(a.next + out + i, kEmpty);
  } else {
    for (int i = tid; i < kPartWords; i += kThreads) leave(a.next + p_at + size_t(part) * kPartWords + i, kEmpty);
  }
  if (ctx_all <= 0) {
    if (merges)
      for (int i = tid; i < GROUP * HALF; i += kThreads) leave(a.now + out + i, 0u);
    return false;
  }
  const int ctx = slot >= 0 ? ctx_all - 1 : ctx_all;      // tokens whose keys are in their pages
  if (!merges && part * kWindow >= ctx) return false;
  // (a row's sequence is nearly always the row itself: its page numbers are asked for before that is known)
  if (seq != row) page = a.tables[size_t(seq) * a.table_stride + entry];
  asm volatile("" : "+v"(page));      // here, once (a wave without tokens would wait for it, and all behind it, where its register is next used)
  const int n16 = lane % 16, kq = lane / 16;
  Frag kf[2][2][KSTEPS], vf[2][DT];
  nothing(kf);
  nothing(vf);
  const bool works = t_first < ctx;
  if (works) {
    const int t0 = t_first + lane, over = t0 - (ctx - 1);
    const int t = over > 0 ? ctx - 1 : t0, tv = over > 0 ? (ctx - 1) & ~7 : t0;
    const int pg = __shfl(page, over > 0 ? lane - over : lane, kWave);
    const uint32_t wk = uint32_t((size_t(pg) * page_elems + kvh * head_elems + size_t(t - page_of(t) * B) * HD) / 8);
    const uint32_t wv = uint32_t((size_t(pg) * page_elems + kvh * head_elems + (tv - page_of(tv) * B)) / 8);
#pragma unroll
    for (int g = 0; g < 2; ++g) {
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) {
        const int tok = g * 32 + 8 * (n16 / 4) + 4 * t2 + n16 % 4;
        const uint16_t* kp = a.kcache + (size_t(__shfl(wk, tok, kWave)) << 3) + kq * 8;
#pragma unroll
        for (int c = 0; c < KSTEPS; ++c) kf[g][t2][c].u = *reinterpret_cast<const uint4*>(kp + c * 32);
      }
      const uint16_t* vp = a.vcache + (size_t(__shfl(wv, g * 32 + 8 * kq, kWave)) << 3) + size_t(n16) * B;
#pragma unroll
      for (int d = 0; d < DT; ++d) vf[g][d].u = *reinterpret_cast<const uint4*>(vp + size_t(d) * 16 * B);
    }
  }
  const uint32_t* qrow = a.now + size_t(row) * width;
  const int polls = made ? kOwnPolls : a.near_polls;
  bool late = false;
  auto await_pair = [&](int col, float& va, float& vb) {
    // (the first look apart: in front of a loop the compiler waits for all that is on its way, here the keys and values)
    uint32_t wa = take(qrow + col), wb = take(qrow + col + HALF);
    for (int poll = 0; __any(wa == kEmpty || wb == kEmpty); ++poll) {
      if (poll >= polls) {
        late = true;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
      wa = take(qrow + col);
      wb = take(qrow + col + HALF);
    }
    va = __uint_as_float(wa);
    vb = __uint_as_float(wb);
  };
  // q: a pair (j, j + HD / 2) of a head a thread
  if (tid < GROUP * HALF) {
    float va, vb;
    await_pair((kvh * GROUP + ih) * HD + ij, va, vb);
    if (a.cos_sin) rotate_pair(va, vb, rot.x, rot.y);
    L.a.q[ih][ij] = float_to_bf16_bits(va);
    L.a.q[ih][ij + HALF] = float_to_bf16_bits(vb);
  }
  // the last threads (other waves where there are enough): the new key and value
  if (merges && slot >= 0 && tid >= kThreads - 2 * HALF) {
    const bool is_v = tid >= kThreads - HALF;
    float va, vb;
    await_pair((a.nh + (is_v ? a.nkv : 0) + kvh) * HD + ij, va, vb);
    if (!is_v && a.cos_sin) rotate_pair(va, vb, rot.x, rot.y);
    const uint16_t ab = float_to_bf16_bits(va), bb = float_to_bf16_bits(vb);
    const size_t pg = slot / B;
    const int off = slot % B;
    uint16_t* kr = a.kcache + ((pg * a.nkv + kvh) * B + off) * HD;
    uint16_t* vr = a.vcache + (pg * a.nkv + kvh) * size_t(HD) * B + off;
    uint16_t* fresh = is_v ? L.a.v_new : L.a.k_new;
    fresh[ij] = ab;
    fresh[ij + HALF] = bb;
    if (!late && !is_v) {
      kr[ij] = ab;
      kr[ij + HALF] = bb;
    } else if (!late) {
      vr[size_t(ij) * B] = ab;
      vr[size_t(ij + HALF) * B] = bb;
    }
  }
  __syncthreads();
  const float scale2 = a.scale * 1.4426950408889634f;
  float m_run = kNone, l_run = 0.f;
  f32x4 o[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (works) {
    Frag qf[KSTEPS];
#pragma unroll
    for (int c = 0; c < KSTEPS; ++c) {
      qf[c].u = *reinterpret_cast<const uint4*>(&L.a.q[n16 < GROUP ? n16 : 0][c * 32 + kq * 8]);
      if (n16 >= GROUP) qf[c].u = uint4{0u, 0u, 0u, 0u};
    }
    const int base = t_first + 8 * kq;
    float s[2][8];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < KSTEPS; ++k) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[g][t][k].v, qf[k].v, acc, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) s[g][4 * t + i] = acc[i] * scale2;
      }
    if (t_first + kWindow > ctx) {
#pragma unroll
      for (int g = 0; g < 2; ++g) {
#pragma unroll
        for (int j = 0; j < 8; ++j) s[g][j] = base + g * 32 + j < ctx ? s[g][j] : kNone;
#pragma unroll
        for (int d = 0; d < DT; ++d) vf[g][d].u = keep_first_bf16(vf[g][d].u, ctx - (base + g * 32));
      }
    }
    float mx = kNone;
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int j = 0; j < 8; ++j) mx = fmaxf(mx, s[g][j]);
    m_run = rows_max(mx);
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      Frag hi, lo;
#pragma unroll
      for (int j = 0; j < 8; j += 2) {
        const float p0 = share(s[g][j], m_run), p1 = share(s[g][j + 1], m_run);
        l_run += p0 + p1;
        hi.w[j / 2] = pack2(p0, p1);
        lo.w[j / 2] = pack2(p0 - low_bf16(hi.w[j / 2]), p1 - high_bf16(hi.w[j / 2]));
      }
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        o[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[g][d].v, hi.v, o[d], 0, 0, 0);
        o[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[g][d].v, lo.v, o[d], 0, 0, 0);
      }
    }
    l_run = rows_sum(l_run);
  }
  if (__any(late)) m_run = kLate;
  if (kq == 0) { L.a.top[wave][n16] = m_run; L.a.sum[wave][n16] = l_run; }
  if (n16 < GROUP) {
#pragma unroll
    for (int d = 0; d < DT; ++d) *reinterpret_cast<f32x4*>(&L.a.red[wave][n16][d * 16 + 4 * kq]) = o[d];
  }
  __syncthreads();
  // a pair of dims of a head a thread: this workgroup's waves, the other parts, the newest token
  const int g = tid / HALF, d = 2 * (tid % HALF);
  static_assert(kThreads / HALF <= 16, "every thread has a column of top");
  float m = L.a.top[0][g];
  bool in_vain = m == kLate;
#pragma unroll
  for (int w = 1; w < kWaves; ++w) {
    in_vain |= L.a.top[w][g] == kLate;
    m = fmaxf(m, L.a.top[w][g]);
  }
  if (__any(in_vain) && !made) return true;
  if (g >= GROUP) return false;
  float n0 = 0.f, n1 = 0.f, den = 0.f;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const float e = __builtin_amdgcn_exp2f(L.a.top[w][g] - m);
    const float2 x = *reinterpret_cast<const float2*>(&L.a.red[w][g][d]);
    n0 = fmaf(e, x.x, n0);
    n1 = fmaf(e, x.y, n1);
    den = fmaf(e, L.a.sum[w][g], den);
  }
  if (!merges) {
    uint32_t* dst = a.now + p_at + size_t(part) * kPartWords + g * (HD + 2);
    leave(dst + d, filled(n0));
    leave(dst + d + 1, filled(n1));
    if (d == 0) {
      leave(dst + HD, filled(m));
      leave(dst + HD + 1, filled(den));
    }
    return false;
  }
  const int others = min(a.parts - 1, (ctx + kWindow - 1) / kWindow);
  if (others > 0) {
    uint64_t v[kMaxParts - 1], ml[kMaxParts - 1];
    const int looks = made ? kOwnPolls : a.far_polls;
    auto look = [&] {
#pragma unroll
      for (int p = 0; p < kMaxParts - 1; ++p) {
        const uint32_t* src = a.now + p_at + size_t(p < others ? p : 0) * kPartWords + g * (HD + 2);
        v[p] = take_two(src + d);
        ml[p] = take_two(src + HD);
      }
      bool none = false;
#pragma unroll
      for (int p = 0; p < kMaxParts - 1; ++p) none |= empty_half(v[p]) || empty_half(ml[p]);
      return __any(none);
    };
    bool empty = look();
    for (int poll = 0; empty && poll < looks; ++poll) {
      __builtin_amdgcn_s_sleep(1);
      empty = look();
    }
    if (empty) return false;      // (left to the output tiles: these words stay empty)
#pragma unroll
    for (int p = 0; p < kMaxParts - 1; ++p)
      if (p < others) {
        const float pm = __uint_as_float(uint32_t(ml[p])), mn = fmaxf(m, pm);
        const float ea = __builtin_amdgcn_exp2f(m - mn), eb = __builtin_amdgcn_exp2f(pm - mn);
        n0 = n0 * ea + eb * __uint_as_float(uint32_t(v[p]));
        n1 = n1 * ea + eb * __uint_as_float(uint32_t(v[p] >> 32));
        den = den * ea + eb * __uint_as_float(uint32_t(ml[p] >> 32));
        m = mn;
      }
  }
  if (slot >= 0) {
    const uint32_t qq = *reinterpret_cast<const uint32_t*>(&L.a.q[g][d]), kk = *reinterpret_cast<const uint32_t*>(&L.a.k_new[d]);
    const uint32_t vv = *reinterpret_cast<const uint32_t*>(&L.a.v_new[d]);
    const float s = group_sum<HALF>(low_bf16(qq) * low_bf16(kk) + high_bf16(qq) * high_bf16(kk)) * scale2;
    const float mn = fmaxf(m, s), ea = __builtin_amdgcn_exp2f(m - mn), eb = share(s, mn);
    n0 = n0 * ea + eb * low_bf16(vv);
    n1 = n1 * ea + eb * high_bf16(vv);
    den = den * ea + eb;
  }
  uint32_t word = pack2(n0 / den, n1 / den);
  leave(a.now + out + tid, word == kEmpty ? 0x7FFF7FFFu : word);
  return false;
}

// Tells the compiler that pointers lead to device memory (it knows so of a kernel's own arguments only).
template <class... P>
__device__ __forceinline__ void in_memory(P*&... p) {
  ((p = (P*)(__attribute__((address_space(1))) P*)p), ...);
}

template <int HD, int GROUP>
__global__ void __launch_bounds__(kThreads, 2) decode_front_kernel(const FrontArgs) {
  __shared__ Lds<HD, GROUP> L;
  typedef __attribute__((address_space(4))) const FrontArgs KernelArgs;
  const int own = blockIdx.x;
  int id = own, next = -1;      // -1: nothing of what it waits for
  for (;;) {
    // The arguments and the thread's number anew for each part (nothing made of them is kept through the loop, which is for workgroups
    // that waited in vain: 256 registers and spills otherwise).  All arguments at once: asked for where they are used they are three
    // trips one behind the other (0.2 to 0.4 us)
    auto* given = (KernelArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    unsigned thread = threadIdx.x;
    asm volatile("" : "+s"(given), "+v"(thread));
    const int tid = thread % kThreads;
    FrontArgs a = *(const FrontArgs*)given;
    in_memory(a.X, a.Wqkv, a.Wo, a.ss_in, a.resid, a.g, a.xg, a.ss_out, a.cos_sin, a.slots, a.tables, a.row_seq, a.ctx_lens, a.kcache, a.vcache, a.now, a.next);
    asm volatile("" ::"s"(a.X), "s"(a.Wqkv), "s"(a.Wo), "s"(a.ss_in), "s"(a.resid), "s"(a.g), "s"(a.xg), "s"(a.ss_out), "s"(a.cos_sin), "s"(a.slots));
    asm volatile("" ::"s"(a.tables), "s"(a.row_seq), "s"(a.ctx_lens), "s"(a.kcache), "s"(a.vcache), "s"(a.now), "s"(a.next), "s"(a.ldx), "s"(a.ldqkv), "s"(a.ldo), "s"(a.tiles_in), "s"(a.M), "s"(a.H));
    asm volatile("" ::"s"(a.table_stride), "s"(a.nh), "s"(a.nkv), "s"(a.B), "s"(a.seqs), "s"(a.parts), "s"(a.n_qkv), "s"(a.n_att), "s"(a.per_page), "s"(a.inv_width), "s"(a.eps), "s"(a.scale), "s"(a.g_f32));
    const int n_in = a.n_qkv + a.n_att;
    bool late;
    if (id >= a.n_qkv && id < n_in) late = attend<HD, GROUP>(a, L, tid, id - a.n_qkv, next >= 0);
    else late = products<HD, GROUP>(a, L, tid, id < a.n_qkv, id < a.n_qkv ? id : id - n_in, next >= 0);
    if (id == own) {
      if (!__builtin_amdgcn_readfirstlane(late)) return;
      next = 0;
    }
    __syncthreads();      // (the next part writes the LDS that this one reads)
    // an attention workgroup: the tiles of its q heads, key and value; an output tile: all QKV tiles and the attention; then its own part again
    const bool attends = own < n_in;
    constexpr int kHeadTiles = HD / (kCols * kGroups);
    if (next >= (attends ? (GROUP + 2) * kHeadTiles : n_in)) {
      id = own;
    } else if (!attends) {
      id = next;
    } else {
      const int kvh = (own - a.n_qkv) / a.parts % a.nkv, h = next / kHeadTiles;
      id = (h < GROUP ? kvh * GROUP + h : a.nh + (h - GROUP) * a.nkv + kvh) * kHeadTiles + next % kHeadTiles;
    }
    ++next;
  }
}

}  // namespace
}  // namespace kvcm


using namespace kvcm;

namespace {

template <int HD>
int launch_front(int group, int grid, hipStream_t st, const FrontArgs& a) {
#define KVCM_FRONT(G) \
  case G: decode_front_kernel<HD, G><<<grid, kThreads, 0, st>>>(a); return 0
  switch (group) {
    KVCM_FRONT(1); KVCM_FRONT(2); KVCM_FRONT(3); KVCM_FRONT(4); KVCM_FRONT(5); KVCM_FRONT(6); KVCM_FRONT(7); KVCM_FRONT(8);
    default: return -1;
  }
#undef KVCM_FRONT
}

__global__ void __launch_bounds__(256) empty_words_kernel(uint4* __restrict__ p, long long n) {
  for (long long i = blockIdx.x * 256ll + threadIdx.x; i < n; i += gridDim.x * 256ll) p[i] = uint4{kEmpty, kEmpty, kEmpty, kEmpty};
}

}  // namespace

extern "C" {

// Does the launch take rows of these sizes?  H: width of the residual stream.
int kvcm_decode_front_supported(int M, int H, int nh, int nkv, int hd, int B) {
  if (M < 1 || M > 8 || nkv <= 0 || nh <= 0 || nh % nkv || nh / nkv > 8 || (hd != 64 && hd != 128)) return 0;
  return H >= kUnit && H % kUnit == 0 && B >= 8 && B % 8 == 0 && B <= 65536;
}

// Workgroups that share a row's KV head for contexts of up to max_context tokens (0: too long for one launch).
int kvcm_decode_front_parts(int max_context) {
  const int fit = (max_context + kWaves * kWindow - 1) / (kWaves * kWindow);
  return max_context <= 0 || fit > kMaxParts ? 0 : fit;
}

// The parts for rows that the launch takes, and faster than three launches do; else 0.  It is not for heads of 64 with more than 192 (row, KV head)
// pairs in more than one part each, where its attention, a workgroup a CU, is the longer (us, three launches / this one; 32 KV heads, contexts of 100, 600, 1,000, 1,200 and
// 1,900 tokens: 6 rows 20.5 / 21.8, 24.4 / 23.5, 29.8 / 26.8, 38.5 / 33.9, 46.4 / 37.5; 8 rows 21.1 / 23.5, 26.9 / 27.3, 32.4 / 32.6, 34.4 / 39.8, 42.7 / 44.7; heads of
// 128, 8 rows 51.6 / 48.5, 61.8 / 57.9, 70.0 / 66.4, 74.4 / 73.6, 90.5 / 88.4).
int kvcm_decode_front_takes(int M, int H, int nh, int nkv, int hd, int B, int max_context) {
  if (!kvcm_decode_front_supported(M, H, nh, nkv, hd, B)) return 0;
  const int parts = kvcm_decode_front_parts(max_context);
  return hd == 64 && M * nkv > 192 && parts > 1 ? 0 : parts;
}

// 32-bit words of one of the two hand-over buffers (a multiple of four).
long long kvcm_decode_front_words(int M, int nh, int nkv, int hd, int parts) {
  const long long n = static_cast<long long>(M) * ((nh + 2 * nkv) * hd + nh * hd / 2 + nh * (parts - 1) * (hd + 2));
  return (n + 3) / 4 * 4;
}

// Empties a hand-over buffer: in front of a step's first kvcm_decode_front (each of those empties its `next`).
int kvcm_decode_front_empty(uint32_t* words, long long n, hipStream_t st) {
  KVCM_REQUIRE(words != nullptr && n >= 0 && n % 4 == 0 && reinterpret_cast<uintptr_t>(words) % 16 == 0, "decode_front_empty: not whole 16-byte pieces");
  if (n == 0) return 0;
  const long long blocks = (n / 4 + 255) / 256;
  empty_words_kernel<<<static_cast<int>(blocks < 512 ? blocks : 512), 256, 0, st>>>(reinterpret_cast<uint4*>(words), n / 4);
  return launch_status("decode_front_empty");
}

// resid[M, H] += round(attention(X Wqkv^T) Wo^T), xg = round(g round(resid)), ss_out[M][H / 8] its sums of squares per 8 columns.
// X: normed rows, or with ss_in [M][tiles_in] what a producer of the folded norm left (kvcm_gemm8).  cos_sin, slots, tables, row_seq,
// ctx_lens as kvcm_attention_decode_fused takes them, tables of `seqs` sequences; no context exceeds 512 * parts tokens.  now: empty
// (kvcm_decode_front_empty, or the launch before had it as next); both of `words` words.  kvcm_decode_front_waiting: polls: looks at what is not there before a workgroup
// makes it itself (negative: as measured).
int kvcm_decode_front_waiting(const void* X, int ldx, const void* Wqkv, int ldqkv, const float* ss_in, int tiles_in, float eps, const void* Wo, int ldo,
                      int M, int H, const float* cos_sin, const int* slots, void* kcache, void* vcache, const int* tables, int table_stride,
                      int seqs, const int* row_seq, const int* ctx_lens, int nh, int nkv, int hd, int B, float scale, float* resid, const void* g,
                      int g_dtype, void* xg, float* ss_out, uint32_t* now, uint32_t* next, long long words, int parts, int polls, hipStream_t st) {
  KVCM_REQUIRE(kvcm_decode_front_supported(M, H, nh, nkv, hd, B), "decode_front: unsupported shape M=%d H=%d heads=%d kv_heads=%d head_dim=%d page=%d", M, H, nh,
               nkv, hd, B);
  KVCM_REQUIRE(parts >= 1 && parts <= kMaxParts, "decode_front: %d parts", parts);
  KVCM_REQUIRE(words >= kvcm_decode_front_words(M, nh, nkv, hd, parts), "decode_front: hand-over buffers too small");
  KVCM_REQUIRE(X && Wqkv && Wo && slots && kcache && vcache && tables && row_seq && ctx_lens && resid && g && xg && ss_out && now && next && now != next,
               "decode_front: null operand");
  KVCM_REQUIRE(g_dtype == kBF16 || g_dtype == kF32, "decode_front: unknown weight dtype %d", g_dtype);
  KVCM_REQUIRE(ss_in == nullptr || tiles_in > 0, "decode_front: sums of squares without their count");
  KVCM_REQUIRE(X != xg && ss_in != ss_out, "decode_front: the rows it reads are still wanted while it writes");
  KVCM_REQUIRE(table_stride >= 1 && seqs >= 1, "decode_front: empty page tables");
  const int qw = nh * hd, width = qw + 2 * nkv * hd;
  const auto piece = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  KVCM_REQUIRE(ldx % 8 == 0 && ldqkv % 8 == 0 && ldo % 8 == 0 && ldx >= H && ldqkv >= H && ldo >= qw && piece(X) && piece(Wqkv) && piece(Wo) && piece(kcache) &&
                   piece(vcache) && piece(now) && piece(next) && reinterpret_cast<uintptr_t>(cos_sin) % 8 == 0,
               "decode_front: operands must be 16-byte aligned with leading dimensions that are multiples of 8 and long enough");
  FrontArgs a{};
  a.X = static_cast<const uint16_t*>(X); a.Wqkv = static_cast<const uint16_t*>(Wqkv); a.Wo = static_cast<const uint16_t*>(Wo);
  a.ldx = ldx; a.ldqkv = ldqkv; a.ldo = ldo; a.M = M; a.H = H;
  a.ss_in = ss_in; a.tiles_in = tiles_in; a.inv_width = tiles_in > 0 ? 1.0f / float(tiles_in * kCols) : 0.f; a.eps = eps;
  a.cos_sin = reinterpret_cast<const float2*>(cos_sin); a.slots = slots; a.tables = tables; a.row_seq = row_seq; a.ctx_lens = ctx_lens;
  a.kcache = static_cast<uint16_t*>(kcache); a.vcache = static_cast<uint16_t*>(vcache); a.table_stride = table_stride; a.seqs = seqs;
  a.nh = nh; a.nkv = nkv; a.B = B; a.scale = scale; a.per_page = static_cast<uint32_t>(((1ull << 32) + B - 1) / B);
  a.resid = resid; a.g = g; a.g_f32 = g_dtype == kF32; a.xg = static_cast<uint16_t*>(xg); a.ss_out = ss_out;
  a.now = now; a.next = next; a.parts = parts; a.near_polls = polls < 0 ? kNearPolls : polls; a.far_polls = polls < 0 ? kFarPolls : polls;
  a.n_qkv = width / (kCols * kGroups); a.n_att = M * nkv * parts;
  const int grid = a.n_qkv + a.n_att + H / (kCols * kGroups);
  const int rc = hd == 64 ? launch_front<64>(nh / nkv, grid, st, a) : launch_front<128>(nh / nkv, grid, st, a);
  KVCM_REQUIRE(rc == 0, "decode_front: no kernel for group size %d", nh / nkv);
  return launch_status("decode_front");
}
int kvcm_decode_front(const void* X, int ldx, const void* Wqkv, int ldqkv, const float* ss_in, int tiles_in, float eps, const void* Wo, int ldo,
                      int M, int H, const float* cos_sin, const int* slots, void* kcache, void* vcache, const int* tables, int table_stride,
                      int seqs, const int* row_seq, const int* ctx_lens, int nh, int nkv, int hd, int B, float scale, float* resid, const void* g,
                      int g_dtype, void* xg, float* ss_out, uint32_t* now, uint32_t* next, long long words, int parts, hipStream_t st) {
  return kvcm_decode_front_waiting(X, ldx, Wqkv, ldqkv, ss_in, tiles_in, eps, Wo, ldo, M, H, cos_sin, slots, kcache, vcache, tables, table_stride, seqs, row_seq,
                                   ctx_lens, nh, nkv, hd, B, scale, resid, g, g_dtype, xg, ss_out, now, next, words, parts, -1, st);
}

}  // extern "C"
