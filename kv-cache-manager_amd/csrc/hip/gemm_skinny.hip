// Decode-shaped products: Y[M,N] = X[M,K] * W[N,K]^T with few rows and a weight matrix that has to be
// streamed from HBM once.  The reference leaves these to cuBLAS (src/model/llama.cpp:45-52); here the
// point is to keep enough weight bytes in flight on 256 CUs.  Widths that are multiples of 64 run in tiles whose
// waves share both operands through LDS (gemm_tiles.hip), up to 512 rows; the kernel here serves the other multiples of
// 16, up to 64 rows, each column tile reading the rows from L2 itself.
//
// One workgroup (4 waves) owns 16 output columns and one slice of K ("split"); its waves divide
// the slice among themselves, each streaming its rows of W straight from global memory into
// MFMA operand registers (every lane 32 contiguous bytes, four lanes one 128-byte line) and
// multiplying with the matching pieces of X (v_mfma_f32_16x16x32_bf16).  The four waves' sums
// are added through LDS in a fixed order.  With one split the result is stored; with S splits the
// 32-bit partial sums go to scratch [S][M][N] and the consumer adds them in split order:
// reduce_store below, or the fused consumers (residual add + RMS norm, SwiGLU, rotary + cache
// write) in elementwise.hip.  No atomics: the result is the same on every run.
//
// SWIGLU variant: W is a fused [gate (I rows) | up (I rows)] matrix; a workgroup takes 8 gate rows
// and the 8 up rows of the same columns, and stores act = round(round(silu(g)) * u) [M, I]
// directly (g, u rounded to the storage type first, exactly what the separate SwiGLU kernel
// computes from the stored product).  Unsplit only.
#include <mutex>

#include "common.h"
#include "gemm_tiles.h"
#include "kvcm_hip.h"

namespace kvcm {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

constexpr int kUnit = 64;  // k elements per unit: 4 lanes x 16 elements = one 128-byte line per row

union Frag {
  uint4 u;
  bf16x8 v;
};

template <int MT, class TO, bool SWIGLU>
__global__ void __launch_bounds__(256)
    gemm_skinny_kernel(const uint16_t* __restrict__ X, const uint16_t* __restrict__ W, float* __restrict__ partials,
                       TO* __restrict__ out, int M, int N, int K, int ldx, int ldw, int ldo, int S, float limit) {
  __shared__ f32x4 red[4][MT][kWave];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int r = lane % 16, kq = lane / 16;
  const int n0 = blockIdx.x * (SWIGLU ? 8 : 16);   // SWIGLU: N is I, the width of the result
  const int s = blockIdx.y;
  const int units = K / kUnit;
  const int u_lo = int((long long)units * s / S), u_hi = int((long long)units * (s + 1) / S);
  const int span = u_hi - u_lo;
  const int w_lo = u_lo + span * wave / 4, w_hi = u_lo + span * (wave + 1) / 4;

  const uint16_t* wrow = W + size_t(SWIGLU ? (r < 8 ? n0 + r : N + n0 + r - 8) : n0 + r) * ldw + kq * 16;
  const uint16_t* xrow[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = t * 16 + r;
    xrow[t] = X + size_t(m < M ? m : 0) * ldx + kq * 16;
  }
  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};

  int u = w_lo;
  if constexpr (MT == 1) {
    for (; u + 8 <= w_hi; u += 8) {  // long slices: eight units per trip
      Frag b[16], a[16];
      const uint16_t* p = wrow + size_t(u) * kUnit;
      const uint16_t* q = xrow[0] + size_t(u) * kUnit;
#pragma unroll
      for (int i = 0; i < 16; ++i) b[i].u = *reinterpret_cast<const uint4*>(p + (i / 2) * kUnit + (i % 2) * 8);
#pragma unroll
      for (int i = 0; i < 16; ++i) a[i].u = *reinterpret_cast<const uint4*>(q + (i / 2) * kUnit + (i % 2) * 8);
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i].v, b[i].v, acc[0], 0, 0, 0);
    }
    for (; u + 4 <= w_hi; u += 4) {  // few rows leave registers for four units per trip: eight weight loads in flight per lane
      Frag b[8], a[8];
      const uint16_t* p = wrow + size_t(u) * kUnit;
      const uint16_t* q = xrow[0] + size_t(u) * kUnit;
#pragma unroll
      for (int i = 0; i < 8; ++i) b[i].u = *reinterpret_cast<const uint4*>(p + (i / 2) * kUnit + (i % 2) * 8);
#pragma unroll
      for (int i = 0; i < 8; ++i) a[i].u = *reinterpret_cast<const uint4*>(q + (i / 2) * kUnit + (i % 2) * 8);
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i].v, b[i].v, acc[0], 0, 0, 0);
    }
  }
  for (; u + 2 <= w_hi; u += 2) {  // two units per trip: four weight loads in flight per lane
    Frag b[4];
    const uint16_t* p = wrow + size_t(u) * kUnit;
    b[0].u = *reinterpret_cast<const uint4*>(p);
    b[1].u = *reinterpret_cast<const uint4*>(p + 8);
    b[2].u = *reinterpret_cast<const uint4*>(p + kUnit);
    b[3].u = *reinterpret_cast<const uint4*>(p + kUnit + 8);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      // rows beyond M read row 0 (always there) and are dropped at the store: no branch
      // around a load, which would make the compiler wait for it on the spot
      Frag a[4];
      const uint16_t* q = xrow[t] + size_t(u) * kUnit;
      a[0].u = *reinterpret_cast<const uint4*>(q);
      a[1].u = *reinterpret_cast<const uint4*>(q + 8);
      a[2].u = *reinterpret_cast<const uint4*>(q + kUnit);
      a[3].u = *reinterpret_cast<const uint4*>(q + kUnit + 8);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i].v, b[i].v, acc[t], 0, 0, 0);
    }
  }
  for (; u < w_hi; ++u) {
    Frag b[2];
    const uint16_t* p = wrow + size_t(u) * kUnit;
    b[0].u = *reinterpret_cast<const uint4*>(p);
    b[1].u = *reinterpret_cast<const uint4*>(p + 8);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      Frag a[2];
      const uint16_t* q = xrow[t] + size_t(u) * kUnit;
      a[0].u = *reinterpret_cast<const uint4*>(q);
      a[1].u = *reinterpret_cast<const uint4*>(q + 8);
#pragma unroll
      for (int i = 0; i < 2; ++i) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i].v, b[i].v, acc[t], 0, 0, 0);
    }
  }

#pragma unroll
  for (int t = 0; t < MT; ++t) red[wave][t][lane] = acc[t];
  __syncthreads();
  if constexpr (SWIGLU) {
    for (int item = threadIdx.x; item < MT * kWave; item += 256) {
      const int t = item / kWave, l = item % kWave;
      if (l % 16 >= 8) continue;
      f32x4 g = red[0][t][l], up = red[0][t][l + 8];
#pragma unroll
      for (int w = 1; w < 4; ++w) {
        const f32x4 a = red[w][t][l], b = red[w][t][l + 8];
        g[0] += a[0]; g[1] += a[1]; g[2] += a[2]; g[3] += a[3];
        up[0] += b[0]; up[1] += b[1]; up[2] += b[2]; up[3] += b[3];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = t * 16 + (l / 16) * 4 + i;
        if (m >= M) continue;
        TO* dst = out + size_t(m) * ldo + n0 + l % 16;
        if (limit > 0.f) {
          store_f(dst, clamped_gate<TO>(g[i], up[i], limit));
          continue;
        }
        const float x = round_to<TO>(g[i]);
        const float act = silu<TO>(x);
        store_f(dst, round_to<TO>(act) * round_to<TO>(up[i]));
      }
    }
    return;
  }
  for (int item = threadIdx.x; item < MT * kWave; item += 256) {
    const int t = item / kWave, l = item % kWave;
    f32x4 v = red[0][t][l];
#pragma unroll
    for (int w = 1; w < 4; ++w) {
      const f32x4 o = red[w][t][l];
      v[0] += o[0]; v[1] += o[1]; v[2] += o[2]; v[3] += o[3];
    }
    const int n = n0 + l % 16;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = t * 16 + (l / 16) * 4 + i;
      if (m >= M) continue;
      if (S > 1) partials[(size_t(s) * M + m) * N + n] = v[i];
      else store_f(out + size_t(m) * ldo + n, v[i]);
    }
  }
}

// out[m][n] = sum over splits, in split order.
template <class TO>
__global__ void reduce_store_kernel(const float* __restrict__ partials, TO* __restrict__ out, int M, int N, int ldo, int S) {
  const size_t i = blockIdx.x * size_t(blockDim.x) + threadIdx.x;
  if (i >= size_t(M) * N) return;
  float v = 0.f;
  for (int s = 0; s < S; ++s) v += partials[size_t(s) * M * N + i];
  store_f(out + (i / N) * ldo + i % N, v);
}

}  // namespace kvcm

using namespace kvcm;

// Whole groups of 64 columns: the tiles.
constexpr int kMaxTileRows = 512, kRowBlock = 128;
static bool in_tiles(int M, int N) { return M > 0 && M <= kMaxTileRows && N % 64 == 0; }
static int row_blocks(int M) { return (M + kRowBlock - 1) / kRowBlock; }
// The SwiGLU form (I: the activation's width) is unsplit: with too few workgroups a split product and a
// launch for SwiGLU fill the chip better.
static bool swiglu_in_tiles(int M, int I) {
  return M > 0 && M <= kMaxTileRows && I % 32 == 0 && static_cast<long long>(I / 32) * row_blocks(M) >= 160;
}

// Splits of K of a plain product in tiles: eight where there are few columns, or where K is long
// against the rows (the partial sums, S*M*N floats that the next kernel reads, are small against the
// weights then), else four; as long as every slice has 256 k (more than 64 rows: 128), two to four steps of the ring,
// and the partial sums stay below the weights' bytes; none where the columns are enough for the chip, and halved where the slices
// would be more than eight 16-column tiles a CU.  Measured at 17 to 128 rows over the projections of TinyLlama and Llama-3-8B sizes,
// alone and in whole decode steps, with the kernel that streamed W into registers, and kept for its successor: the tile is chosen for
// these slices (gemm_tiles.hip).  (With the tiles free to choose among 1, 2, 4 and 8 as well, launches and the reading of the
// partial sums together would be 4 % shorter at 8 to 512 rows.)  Up to 16 rows the norm that follows is a workgroup a row, each reading
// all slices of its row: four of 128 column tiles too (Kasuvik and Fisesun, eight requests, 34.61 -> 34.09 and 30.69 -> 30.30 ms a pass;
// at 64 rows of TinyLlama sizes four were slower, 150.8 -> 152.0).
constexpr int kRowsCUs = 256;
static int rows_splits(int M, int N, int K) {
  const long long tiles = static_cast<long long>(N / 16) * row_blocks(M);
  const int units = K / kUnit;
  if (tiles >= 4 * kRowsCUs) return 1;
  int S = tiles <= (M <= 16 ? 64 : 128) || (M > 48 && K >= 112 * M) ? 8 : 4;
  const int least = M <= 64 ? 4 : 2;   // units of a slice
  const int cap = units / least < K / (2 * M) ? units / least : K / (2 * M);
  while (S > 1 && S > cap) S >>= 1;
  while (S > 1 && tiles * S > 8 * kRowsCUs) S >>= 1;
  return S;
}

extern "C" {

// How many splits of K a launch of this shape uses (0: the shape is not supported by this kernel).
int kvcm_gemm_skinny_splits(int M, int N, int K) {
  if (M <= 0 || N % 16 != 0 || K % kUnit != 0 || N <= 0 || K <= 0) return 0;
  if (in_tiles(M, N)) return rows_splits(M, N, K);
  if (M > 64) return 0;
  const int tiles = N / 16, units = K / kUnit;
  int S = (640 + tiles - 1) / tiles;           // aim at >= 640 workgroups (2.5 per CU) ...
  if (S >= 5) S = 8;                           // ... five to seven slices lose to eight in whole decode steps (measured)
  while (S > 1 && S > units / 2) --S;          // at least two units per slice
  return S;
}

// The same where nobody takes the partial sums: a second launch adds them then, and one slice may be the faster whole (a launch that
// adds them takes 3.2 us and its bytes at 5 TB/s).
int kvcm_gemm_skinny_whole_splits(int M, int N, int K) {
  const int S = kvcm_gemm_skinny_splits(M, N, K);
  if (S <= 1 || !in_tiles(M, N)) return S;
  const float add = 3.2f + static_cast<float>(M) * static_cast<float>(N) * (4.f * S + 4.f) / 5e6f;
  return gemm_tiles_time(M, N, K, 1, false, false) <= gemm_tiles_time(M, N, K, S, false, false) + add ? 1 : S;
}

// S == 1: the result is stored to `out` (bfloat16 or float32).  S > 1: partial sums are written to
// `partials` [S][M][N]; `out` is not touched (pass S from kvcm_gemm_skinny_splits).
int kvcm_gemm_skinny(const void* X, const void* W, float* partials, void* out, int out_dtype, int M, int N, int K,
                     int ldx, int ldw, int ldo, int S, hipStream_t st) {
  KVCM_REQUIRE(kvcm_gemm_skinny_splits(M, N, K) > 0, "gemm_skinny: unsupported shape M=%d N=%d K=%d", M, N, K);
  KVCM_REQUIRE(S >= 1 && S <= K / kUnit, "gemm_skinny: bad split count %d", S);
  KVCM_REQUIRE(ldx % 8 == 0 && ldw % 8 == 0 && reinterpret_cast<uintptr_t>(X) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(W) % 16 == 0,
               "gemm_skinny: operands must be 16-byte aligned with leading dimensions that are multiples of 8");
  KVCM_REQUIRE(ldx >= K && ldw >= K, "gemm_skinny: leading dimensions too small");
  KVCM_REQUIRE(S == 1 ? (out != nullptr && ldo >= N) : partials != nullptr, "gemm_skinny: missing output buffer");
  KVCM_REQUIRE(out_dtype == kBF16 || out_dtype == kF32, "gemm_skinny: unknown output dtype %d", out_dtype);
  const uint16_t* x = static_cast<const uint16_t*>(X);
  const uint16_t* w = static_cast<const uint16_t*>(W);
  const int mt = (M + 15) / 16;
  if (in_tiles(M, N)) return gemm_tiles(TilesCall{x, w, partials, out, out_dtype == kF32, M, N, K, ldx, ldw, ldo, S}, false, -1, st);
  const dim3 grid(N / 16, S);
#define KVCM_SKINNY(MT, TO) \
  gemm_skinny_kernel<MT, TO, false><<<grid, 256, 0, st>>>(x, w, partials, static_cast<TO*>(out), M, N, K, ldx, ldw, ldo, S, 0.f)
  if (out_dtype == kBF16) {
    if (mt == 1) KVCM_SKINNY(1, bf16_t); else if (mt == 2) KVCM_SKINNY(2, bf16_t); else if (mt == 3) KVCM_SKINNY(3, bf16_t); else KVCM_SKINNY(4, bf16_t);
  } else {
    if (mt == 1) KVCM_SKINNY(1, float); else if (mt == 2) KVCM_SKINNY(2, float); else if (mt == 3) KVCM_SKINNY(3, float); else KVCM_SKINNY(4, float);
  }
#undef KVCM_SKINNY
  return launch_status("gemm_skinny");
}

// May act = swiglu(X * [gate | up]^T) be computed in one launch?  I is the width of the result.
int kvcm_gemm_skinny_swiglu_supported(int M, int I, int K) {
  if (!(M > 0 && I > 0 && I % 8 == 0 && K > 0 && K % kUnit == 0)) return 0;
  if (swiglu_in_tiles(M, I)) return 1;
  // with too few workgroups a split product fills the chip better than an unsplit one; the kernel whose
  // every tile reads the rows from L2 serves a few rows, or widths that are no multiple of 32
  if (I % 32 == 0 && M > 16) return 0;
  return M <= 64 && I / 8 >= 320;
}

// W [2 I, K] (gate rows, then up rows); out [M, I].  limit > 0: the gate with limits (clamped_gate) instead of silu(gate) * up.
int kvcm_gemm_skinny_swiglu(const void* X, const void* W, void* out, int out_dtype, int M, int I, int K, int ldx,
                            int ldw, int ldo, float limit, hipStream_t st) {
  KVCM_REQUIRE(kvcm_gemm_skinny_swiglu_supported(M, I, K), "gemm_skinny_swiglu: unsupported shape M=%d I=%d K=%d", M, I, K);
  KVCM_REQUIRE(ldx % 8 == 0 && ldw % 8 == 0 && reinterpret_cast<uintptr_t>(X) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(W) % 16 == 0,
               "gemm_skinny_swiglu: operands must be 16-byte aligned with leading dimensions that are multiples of 8");
  KVCM_REQUIRE(ldx >= K && ldw >= K && out != nullptr && ldo >= I, "gemm_skinny_swiglu: leading dimensions too small");
  KVCM_REQUIRE(out_dtype == kBF16 || out_dtype == kF32, "gemm_skinny_swiglu: unknown output dtype %d", out_dtype);
  const uint16_t* x = static_cast<const uint16_t*>(X);
  const uint16_t* w = static_cast<const uint16_t*>(W);
  const int mt = (M + 15) / 16;
  if (swiglu_in_tiles(M, I)) {
    TilesCall c{x, w, nullptr, out, out_dtype == kF32, M, I, K, ldx, ldw, ldo, 1};
    c.limit = limit;
    return gemm_tiles(c, true, -1, st);
  }
  const dim3 grid(I / 8, 1);
#define KVCM_SKINNY(MT, TO) \
  gemm_skinny_kernel<MT, TO, true><<<grid, 256, 0, st>>>(x, w, nullptr, static_cast<TO*>(out), M, I, K, ldx, ldw, ldo, 1, limit)
  if (out_dtype == kBF16) {
    if (mt == 1) KVCM_SKINNY(1, bf16_t); else if (mt == 2) KVCM_SKINNY(2, bf16_t); else if (mt == 3) KVCM_SKINNY(3, bf16_t); else KVCM_SKINNY(4, bf16_t);
  } else {
    if (mt == 1) KVCM_SKINNY(1, float); else if (mt == 2) KVCM_SKINNY(2, float); else if (mt == 3) KVCM_SKINNY(3, float); else KVCM_SKINNY(4, float);
  }
#undef KVCM_SKINNY
  return launch_status("gemm_skinny_swiglu");
}

// The same with a folded RMS norm in front (gemm_rows8.hip): X is xg = round(g round(x)) of the norm's producer,
// ss_in its [M][tiles_in] sums of x^2 per 8-column tile, eps the norm's; the sums are scaled by
// rsqrt(mean x^2 + eps) before they are rounded.  For the widths at which the tiles' few long-lived
// workgroups stream the gate/up matrix faster than the 8-row kernel's many short ones (from 1,024 tiles of 8 columns on:
// Llama-3-8B sizes, one row: 50.8 against 43.9 us).
int kvcm_gemm_skinny_swiglu_normed_preferred(int M, int I, int K) {
  return K > 0 && K % kUnit == 0 && swiglu_in_tiles(M, I) && I / 8 >= 4 * kRowsCUs;
}
int kvcm_gemm_skinny_swiglu_normed(const void* X, const void* W, const float* ss_in, int tiles_in, float eps, void* out,
                                   int M, int I, int K, int ldx, int ldw, int ldo, hipStream_t st) {
  KVCM_REQUIRE(K > 0 && K % kUnit == 0 && swiglu_in_tiles(M, I), "gemm_skinny_swiglu_normed: unsupported shape M=%d I=%d K=%d", M, I, K);
  KVCM_REQUIRE(ss_in != nullptr && tiles_in > 0 && tiles_in * 8 == K, "gemm_skinny_swiglu_normed: %d tiles of sums for a width of %d", tiles_in, K);
  KVCM_REQUIRE(ldx % 8 == 0 && ldw % 8 == 0 && reinterpret_cast<uintptr_t>(X) % 16 == 0 && reinterpret_cast<uintptr_t>(W) % 16 == 0,
               "gemm_skinny_swiglu_normed: operands must be 16-byte aligned with leading dimensions that are multiples of 8");
  KVCM_REQUIRE(ldx >= K && ldw >= K && out != nullptr && ldo >= I, "gemm_skinny_swiglu_normed: leading dimensions too small");
  TilesCall c{static_cast<const uint16_t*>(X), static_cast<const uint16_t*>(W), nullptr, out, 0, M, I, K, ldx, ldw, ldo, 1};
  c.ss_in = ss_in;
  c.tiles_in = tiles_in;
  c.eps = eps;
  return gemm_tiles(c, true, -1, st);
}

int kvcm_reduce_store(const float* partials, void* out, int out_dtype, int M, int N, int ldo, int S, hipStream_t st) {
  if (M == 0 || N == 0) return 0;
  KVCM_REQUIRE(M > 0 && N > 0 && S >= 1 && ldo >= N, "reduce_store: bad sizes");
  const size_t n = size_t(M) * N;
  const unsigned blocks = static_cast<unsigned>((n + 255) / 256);
  if (out_dtype == kBF16) reduce_store_kernel<bf16_t><<<blocks, 256, 0, st>>>(partials, static_cast<bf16_t*>(out), M, N, ldo, S);
  else if (out_dtype == kF32) reduce_store_kernel<float><<<blocks, 256, 0, st>>>(partials, static_cast<float*>(out), M, N, ldo, S);
  else KVCM_REQUIRE(false, "reduce_store: unknown output dtype %d", out_dtype);
  return launch_status("reduce_store");
}

// ---- the product for callers that cannot allocate -------------------------------------------
// Partial sums of a split product, for kvcm_gemm_skinny_noalloc: part of the library's device
// image, one copy per GPU at that GPU's own address.  Host code never passes the array's name to a
// kernel (on the host it is a stand-in, not a device address): it passes the address that
// hipGetSymbolAddress gave for the current device.
constexpr long long kNoAllocFloats = 2ll << 20;
static __device__ __align__(256) float scratch[kNoAllocFloats];

constexpr int kMaxDevices = 64;
static float* g_noalloc_ptr[kMaxDevices];
static std::mutex g_noalloc_lock;

// The current device's copy of the array; looked up once per device, with that device current.
static int noalloc_scratch(float** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    set_error("gemm_skinny_noalloc: hipGetDevice: %s", hipGetErrorString(e));
    return -2;
  }
  KVCM_REQUIRE(dev >= 0 && dev < kMaxDevices, "gemm_skinny_noalloc: device %d beyond the %d this library keeps track of", dev, kMaxDevices);
  std::lock_guard<std::mutex> hold(g_noalloc_lock);
  if (g_noalloc_ptr[dev] == nullptr) {
    float* p = nullptr;
    e = hipGetSymbolAddress(reinterpret_cast<void**>(&p), HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) {
      set_error("gemm_skinny_noalloc: hipGetSymbolAddress on device %d: %s", dev, hipGetErrorString(e));
      return -2;
    }
    g_noalloc_ptr[dev] = p;
  }
  *out = g_noalloc_ptr[dev];
  return 0;
}

long long kvcm_gemm_skinny_noalloc_capacity() { return kNoAllocFloats; }

int kvcm_gemm_skinny_noalloc(const void* X, const void* W, void* out, int out_dtype, int M, int N, int K, int ldx,
                             int ldw, int ldo, hipStream_t st) {
  const int S = kvcm_gemm_skinny_splits(M, N, K);
  KVCM_REQUIRE(S > 0, "gemm_skinny_noalloc: unsupported shape M=%d N=%d K=%d", M, N, K);
  KVCM_REQUIRE(out != nullptr && ldo >= N, "gemm_skinny_noalloc: missing output buffer or leading dimension below N");
  if (S == 1) return kvcm_gemm_skinny(X, W, nullptr, out, out_dtype, M, N, K, ldx, ldw, ldo, 1, st);
  const long long need = (long long)S * M * N;
  KVCM_REQUIRE(need <= kNoAllocFloats,
               "gemm_skinny_noalloc: M=%d N=%d K=%d needs %lld floats of partial sums (%d slices), the built-in array holds %lld",
               M, N, K, need, S, kNoAllocFloats);
  if (kvcm_gemm_skinny_whole_splits(M, N, K) == 1) return kvcm_gemm_skinny(X, W, nullptr, out, out_dtype, M, N, K, ldx, ldw, ldo, 1, st);
  float* partials = nullptr;
  if (int rc = noalloc_scratch(&partials)) return rc;
  if (int rc = kvcm_gemm_skinny(X, W, partials, out, out_dtype, M, N, K, ldx, ldw, ldo, S, st)) return rc;
  return kvcm_reduce_store(partials, out, out_dtype, M, N, ldo, S, st);
}

}  // extern "C"
