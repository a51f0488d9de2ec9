// 32-bit products of rows of up to 256 entries with what surrounds them in a decoder layer: the RMS norm of the rows they multiply in
// front, SwiGLU or the addition to the residual stream behind.  The reference runs these as kernels of their own
// (src/cuda/kernels.cu:34-49,72-88); at these widths a launch costs 2 to 4.5 us whatever it computes, and a layer had ten of them: with
// these products and attention_f32_decode it has five.  A test run of three short requests on two layers of width 64: 0.845 -> 0.738 ms.
// (Wider rows keep the norm's launch: as a prologue of every workgroup of 8 columns, 2,048 entries, one row, it made QKV's 2560
// columns 12.2 us where norm and product are 11.5, gate and up 29.9 of 26.7 with SwiGLU's launch.)
//
// Every element is the same sequence of operations as in gemm_f32.hip, in the norm and SwiGLU kernels of elementwise.hip (the sum
// of squares as a workgroup of 256 threads adds it), so the bits are those of the separate launches whatever the rows beside.
//
// A workgroup has 16 rows x 64 columns, one ascending chain of k an element (gemm_f32.hip), all of W on its way before the norm begins.
// A lane's 16 bytes of a row of W hold four consecutive k where the chain wants every fourth: four lanes 16 apart exchange them
// by row and half swaps.
#include "common.h"
#include "gemm_f32_order.h"
#include "kvcm_hip.h"

namespace kvcm {
namespace {

constexpr int kFewThreads = 256, kFewWaves = kFewThreads / kWave;
enum Behind : int { kPlain = 0, kAdd = 1, kSwiglu = 2 };

struct FewArgs {
  const float *X, *g, *W;      // g: the norm's weight (null: X is multiplied as it is)
  float* Y;
  int M, N, K, ldx, ldw, ldy;      // kSwiglu: N columns of the result, W its gate rows and its up rows
  float eps;
};

// Row of W behind column c of a block that starts at n0 and has `half` gate and `half` up columns.
__device__ __forceinline__ int gated_row(int n0, int c, int half, int N) {
  const int n = n0 + c % half;
  return (n < N ? n : N - 1) + (c < half ? 0 : N);
}

// Lane group g (16 lanes) holds k = 4 g + e in v[e]; afterwards v[i] holds k = 4 i + g: the two bits of e and of g change places.
__device__ __forceinline__ void every_fourth(f32x4& v) {
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[e]), __float_as_uint(v[e + 2]), false, false);
    v[e] = __uint_as_float(s[0]);
    v[e + 2] = __uint_as_float(s[1]);
  }
#pragma unroll
  for (int e = 0; e < 4; e += 2) {
    const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[e]), __float_as_uint(v[e + 1]), false, false);
    v[e] = __uint_as_float(s[0]);
    v[e + 1] = __uint_as_float(s[1]);
  }
}

template <bool NORMED, int BEHIND, int PIECES>
__global__ void __launch_bounds__(kFewThreads) gemm_f32_short_kernel(const FewArgs a) {
  constexpr int kPitch = 16 * PIECES + 4;
  __shared__ __attribute__((aligned(16))) float rows[16][kPitch];
  __shared__ f32x4 ups[2][kWave];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int r = lane & 15, g = lane >> 4;
  const int M = a.M, N = a.N, K = a.K, m0 = blockIdx.y * 16, n0 = blockIdx.x * (BEHIND == kSwiglu ? 32 : 64);
  const int n = n0 + wave * 16 + r;
  const int wrow = BEHIND == kSwiglu ? gated_row(n0, wave * 16 + r, 32, N) : (n < N ? n : N - 1);
  const float* w = a.W + size_t(wrow) * a.ldw;
  f32x4 b[PIECES];
#pragma unroll
  for (int p = 0; p < PIECES; ++p) b[p] = load4<true>(w, 16 * p + 4 * g, K);
  // rows wave, wave + 4, ..: a lane's four entries (the first wave's of the norm's own kernel; its other threads have none)
  const int at = 4 * lane;
  const bool own = at < K;
  float4 gw = float4{0.f, 0.f, 0.f, 0.f};
  if constexpr (NORMED) gw = *reinterpret_cast<const float4*>(a.g + (own ? at : 0));
  float4 v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + wave + kFewWaves * i;
    const float* x = a.X + size_t(m < M ? m : M - 1) * a.ldx + (own ? at : 0);
    if constexpr (NORMED) v[i] = *reinterpret_cast<const float4*>(x);
    else { const f32x4 t = load4<true, true>(x, 0, K); v[i] = float4{t[0], t[1], t[2], t[3]}; }
    if (!own) v[i] = float4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (NORMED) {
      const float inv = 1.0f / sqrtf(wave_sum(add_squares(0.f, true, v[i].x, v[i].y, v[i].z, v[i].w)) / float(K) + a.eps);
      v[i] = float4{gw.x * (v[i].x * inv), gw.y * (v[i].y * inv), gw.z * (v[i].z * inv), gw.w * (v[i].w * inv)};
      if (!own) v[i] = float4{0.f, 0.f, 0.f, 0.f};
    }
    if (at < 16 * PIECES) *reinterpret_cast<float4*>(&rows[wave + kFewWaves * i][at]) = v[i];
  }
  __syncthreads();
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  const int pieces = (K + kUnit - 1) / kUnit * 2;      // whole units, as the tiles
#pragma unroll
  for (int p = 0; p < PIECES; ++p) {
    if (p < pieces) {
      every_fourth(b[p]);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(rows[r][16 * p + 4 * i + g], b[p][i], acc, 0, 0, 0);
    }
  }
  if constexpr (BEHIND == kSwiglu) {
    if (wave >= 2) ups[wave - 2][lane] = acc;
    __syncthreads();
    if (wave >= 2) return;
    const f32x4 up = ups[wave][lane];
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] = silu<float>(acc[e]) * up[e];
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int m = m0 + 4 * g + e;
    if (m < M && n < N) {
      float* y = a.Y + size_t(m) * a.ldy + n;
      *y = BEHIND == kAdd ? *y + acc[e] : acc[e];
    }
  }
}

template <bool NORMED, int BEHIND>
void launch_few(const FewArgs& a, hipStream_t st) {
  const int cols = BEHIND == kSwiglu ? 32 : 64;
  const dim3 grid((a.N + cols - 1) / cols, (a.M + 15) / 16);
  if (a.K <= 64) gemm_f32_short_kernel<NORMED, BEHIND, 4><<<grid, kFewThreads, 0, st>>>(a);
  else if (a.K <= 128) gemm_f32_short_kernel<NORMED, BEHIND, 8><<<grid, kFewThreads, 0, st>>>(a);
  else gemm_f32_short_kernel<NORMED, BEHIND, 16><<<grid, kFewThreads, 0, st>>>(a);
}

}  // namespace
}  // namespace kvcm

using namespace kvcm;

extern "C" {

// Does kvcm_gemm_f32_few take rows of K entries?
int kvcm_gemm_f32_few_supported(int M, int K) { return M >= 1 && M <= 64 && K >= 4 && K <= kShortK && K % 4 == 0; }

// Y = X' W^T (behind 0), Y += X' W^T (1), Y = silu(X' Wg^T) * (X' Wu^T) with W = [Wg; Wu] (2), where X' are the rows of X, or with g their
// RMS norms g * (x * rsqrt(mean x^2 + eps)).  The bits of kvcm_rmsnorm, kvcm_gemm_f32, kvcm_swiglu and kvcm_add_residual.
int kvcm_gemm_f32_few(const float* X, const float* g, float eps, const float* W, float* Y, int M, int N, int K, int ldx, int ldw, int ldy,
                      int behind, hipStream_t st) {
  KVCM_REQUIRE(kvcm_gemm_f32_few_supported(M, K) && N > 0, "gemm_f32_few: unsupported shape M=%d N=%d K=%d", M, N, K);
  KVCM_REQUIRE(X && W && Y && ldx >= K && ldw >= K && ldy >= N, "gemm_f32_few: missing operand or leading dimensions too small");
  KVCM_REQUIRE(behind >= kPlain && behind <= kSwiglu, "gemm_f32_few: unknown epilogue %d", behind);
  KVCM_REQUIRE(!g || (ldx % 4 == 0 && reinterpret_cast<uintptr_t>(X) % 16 == 0 && reinterpret_cast<uintptr_t>(g) % 16 == 0),
               "gemm_f32_few: normed rows must be 16-byte aligned");
  const FewArgs a{X, g, W, Y, M, N, K, ldx, ldw, ldy, eps};
  if (g) {
    if (behind == kPlain) launch_few<true, kPlain>(a, st);
    else if (behind == kAdd) launch_few<true, kAdd>(a, st);
    else launch_few<true, kSwiglu>(a, st);
  } else {
    if (behind == kPlain) launch_few<false, kPlain>(a, st);
    else if (behind == kAdd) launch_few<false, kAdd>(a, st);
    else launch_few<false, kSwiglu>(a, st);
  }
  return launch_status("gemm_f32_few");
}

}  // extern "C"
