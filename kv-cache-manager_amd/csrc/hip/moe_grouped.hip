// The routed feed-forward for steps with many rows (bfloat16): the (row, slot) pairs are grouped by their expert and
// every expert's group is multiplied with that expert's matrices in tiles on the matrix cores, so that an expert's
// weights are read once per tile of pairs and not once per pair.
//
//   moe_group      pairs p = row * top + slot, grouped by chosen[p]: order[] lists the pairs expert by expert; two lists, for the
//                  tiles of UP and of DOWN (which may be of different heights), hold (expert, its first place in order, its
//                  pairs, its first tile) for every tile, the tiles of an expert one after the other.  One workgroup; places inside
//                  a group are handed out by an atomic counter in LDS, so the order inside a group may differ from run to
//                  run, which changes no result: a pair's row of a tile is computed from that row alone.
//   moe_grouped    UP:   act[place, :] = square(relu(W_up[e] h[row of the pair])), or gelu of it (bfloat16, in grouped order)
//                  GATED UP: act[place, :] = silu(W_gate[e] h) * (W_up[e] h); the two matrices of an expert are stored as
//                        one of 2F rows, interleaved sixteen at a time (gate 0..15, up 0..15, gate 16..31, ...), so that a
//                        lane's neighbouring accumulators hold the gate and the up values of the same columns
//                  DOWN: y[pair, :]   = weight[pair] * W_down[e] act[place, :]               (32-bit, by pair)
//                  The pairs' weights may act on the other side instead: UP then reads weight * h (the factor is applied to
//                  its 32-bit sums) and DOWN weighs nothing.
//                  A tile of BM pairs x BN rows of the expert's matrix per workgroup, its operands in a ring of stages in LDS
//                  (tile_ring.h).
//   moe_combine    out[row, :] = (add[row, :] +) sum over the row's slots, in slot order, of y[row * top + slot, :]
//
// What bounds the products is what bounds those of gemm_tiles.hip.  All five launches, us,
// against 128 x 128 pairs and rows with two stages throughout: 8 experts of which a row uses 2, width 2,048, 1,408 columns an expert: 80
// rows 64.6 -> 44.2, 300 69.9 -> 52.0, 1,024 86.1 -> 84.2, 2,048 134 -> 113, 4,072 230 -> 208; width 4,096, 3,584 columns, 2,048 rows 487 -> 468.
#include <cmath>

#include "common.h"
#include "gemm_tiles.h"
#include "kvcm_hip.h"
#include "tile_pipe.h"

namespace kvcm {

constexpr int kLeastHigh = 64;      // pairs of the lowest tile

__host__ __device__ __forceinline__ int most_tiles(int n, int E) { return n / kLeastHigh + E; }

// lists: the numbers of tiles of UP and DOWN, two unused, then the two lists of `most` entries
__global__ void __launch_bounds__(1024)
    moe_group_kernel(const int* __restrict__ chosen, int n, int E, int* __restrict__ order, int* __restrict__ lists, int high_up, int high_down) {
  extern __shared__ int sh[];      // per expert: pairs (later a cursor), first place, first tile of UP, of DOWN
  int *cnt = sh, *first = sh + E, *up = sh + 2 * E, *down = sh + 3 * E;
  const int most = most_tiles(n, E);
  for (int e = threadIdx.x; e < E; e += blockDim.x) cnt[e] = 0;
  __syncthreads();
  for (int p = threadIdx.x; p < n; p += blockDim.x) {
    const int e = chosen[p];
    if (e >= 0 && e < E) atomicAdd(&cnt[e], 1);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int at = 0, nu = 0, nd = 0;
    for (int e = 0; e < E; ++e) {
      first[e] = at;
      up[e] = nu;
      down[e] = nd;
      at += cnt[e];
      nu += (cnt[e] + high_up - 1) / high_up;
      nd += (cnt[e] + high_down - 1) / high_down;
    }
    lists[0] = nu;
    lists[1] = nd;
  }
  __syncthreads();
  int4* entry = reinterpret_cast<int4*>(lists + 4);
  for (int e = threadIdx.x; e < E; e += blockDim.x) {
    for (int r = 0, i = up[e]; r < cnt[e]; r += high_up, ++i) entry[i] = int4{e, first[e], cnt[e], up[e]};
    for (int r = 0, i = down[e]; r < cnt[e]; r += high_down, ++i) entry[most + i] = int4{e, first[e], cnt[e], down[e]};
    cnt[e] = 0;      // (no other thread reads it before the barrier)
  }
  __syncthreads();
  for (int p = threadIdx.x; p < n; p += blockDim.x) {
    const int e = chosen[p];
    if (e >= 0 && e < E) order[first[e] + atomicAdd(&cnt[e], 1)] = p;
  }
}

enum : int { kDown = 0, kUp = 1, kUpGated = 2, kUpGelu = 3 };

// N: rows of an expert's matrix (2F for the gated form); the output has N columns (F for the gated form).  Offset: of an operand's
// pieces from its beginning, in bytes; uint64_t for rows that lie beyond 4 GB or far apart.
template <int BM, int BN, int WM, int WN, int STAGES, bool PIPE, int MODE, class Offset>
__global__ void __launch_bounds__(WM* WN* kWave)
    moe_grouped_kernel(const uint16_t* __restrict__ A, int lda, const uint16_t* __restrict__ W, const int* __restrict__ order,
                       const int* __restrict__ count, const int4* __restrict__ list, int top, void* __restrict__ out,
                       const float* __restrict__ weight, int N, int K, int col_blocks) {
  using Ring = std::conditional_t<PIPE, TilePipe<BM, BN, WM, WN, STAGES>, TileRing<BM, BN, WM, WN, STAGES>>;
  constexpr int TM = Ring::TM, TN = Ring::TN, R = Ring::R;
  static_assert(MODE != kUpGated || TN % 2 == 0, "gate and up accumulators in one wave");
  __shared__ __attribute__((aligned(1024))) unsigned char ring[Ring::kBytes];
  // Each XCD takes a contiguous stretch of the tiles there are, one expert after the other, an expert's tiles of one column block
  // side by side: neighbours read the same rows of the expert's matrix.
  const int total = count[0] * col_blocks, per = total / 8, more = total % 8, xcd = blockIdx.x % 8, turn = blockIdx.x / 8;
  if (turn >= per + (xcd < more ? 1 : 0)) return;
  const int id = xcd * per + (xcd < more ? xcd : more) + turn;
  const int4 x = list[id / col_blocks];      // some tile of the expert
  const int e = x.x, tiles = (x.z + BM - 1) / BM, local = id - x.w * col_blocks;
  const int r0 = local % tiles * BM, p0 = x.y + r0, rows = x.z - r0 < BM ? x.z - r0 : BM;
  const int n0 = local / tiles * BN;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int wm = wave % WM, wn = wave / WM, frow = lane % 16, fk = lane / 16;
  const uint64_t abase = reinterpret_cast<uint64_t>(A + (MODE == kDown ? static_cast<size_t>(p0) * lda : 0));
  const uint64_t wbase = reinterpret_cast<uint64_t>(W + (static_cast<size_t>(e) * N + n0) * K);
  // rows past the tile and columns past N repeat the last one (what they give is not stored)
  Offset offset[R];
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int req = Ring::request_of(q, wave), row = req * 8 + lane / 8;
    const int r = row < rows ? row : rows - 1, c = row - BM < N - n0 ? row - BM : N - 1 - n0;
    const uint32_t from = MODE != kDown ? static_cast<uint32_t>(order[p0 + (req < BM / 8 ? r : 0)]) / static_cast<uint32_t>(top) : static_cast<uint32_t>(r);
    offset[q] = (req < BM / 8 ? static_cast<Offset>(from) * static_cast<Offset>(lda) : static_cast<Offset>(c) * static_cast<Offset>(K)) * 2u +
                static_cast<Offset>(Ring::piece_of(lane)) * 16u;
  }
  int pair[TM];      // of this lane's rows
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = (wm * TM + i) * 16 + frow;
    pair[i] = order[p0 + (m < rows ? m : rows - 1)];
  }
  ring_f32x4 acc[TN][TM];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i) acc[j][i] = ring_f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = (K + kStepK - 1) / kStepK;
  Ring::multiply(ring, offset, [&](int req) { return req < BM / 8 ? abase : wbase; }, steps, 0, K - (steps - 1) * kStepK, wave, lane, acc, [] {},
                 wm * TM * 16 < rows);
  // acc[j][i][r]: pair wm * TM * 16 + i * 16 + frow of the tile, row wn * TN * 16 + j * 16 + fk * 4 + r of the matrix (from n0 on)
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = (wm * TM + i) * 16 + frow;
    if (m >= rows) continue;
    const float g = weight ? weight[pair[i]] : 1.f;
    if constexpr (MODE == kDown) {
      float* dst = static_cast<float*>(out) + static_cast<size_t>(pair[i]) * N;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int c = n0 + (wn * TN + j) * 16 + fk * 4;
        const ring_f32x4 v = acc[j][i] * g;
        if (c + 3 < N) {
          *reinterpret_cast<any_f32x4*>(dst + c) = any_f32x4{v[0], v[1], v[2], v[3]};
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (c + r < N) dst[c + r] = v[r];
        }
      }
    } else if constexpr (MODE == kUpGated) {
      uint16_t* dst = static_cast<uint16_t*>(out) + static_cast<size_t>(p0 + m) * (N / 2);
#pragma unroll
      for (int j = 0; j < TN; j += 2) {      // (the columns are a multiple of 16: a piece lies inside or outside)
        const int c = n0 / 2 + (wn * TN + j) * 8 + fk * 4;
        if (c >= N / 2) continue;
        float a[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) a[r] = silu<bf16_t>(g * acc[j][i][r]) * (g * acc[j + 1][i][r]);
        *reinterpret_cast<uint2*>(dst + c) = uint2{two_bf16(a[0], a[1]), two_bf16(a[2], a[3])};
      }
    } else {
      uint16_t* dst = static_cast<uint16_t*>(out) + static_cast<size_t>(p0 + m) * N;
#pragma unroll
      for (int j = 0; j < TN; ++j) {      // (the columns are a multiple of 8)
        const int c = n0 + (wn * TN + j) * 16 + fk * 4;
        if (c >= N) continue;
        float a[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float v = g * acc[j][i][r], z = fmaxf(v, 0.f);
          a[r] = MODE == kUpGelu ? gelu_exact<bf16_t>(v) : z * z;
        }
        *reinterpret_cast<uint2*>(dst + c) = uint2{two_bf16(a[0], a[1]), two_bf16(a[2], a[3])};
      }
    }
  }
}

// A workgroup adds up N * 256 columns of one row, N a thread.
template <int N>
__global__ void __launch_bounds__(256)
    moe_combine_kernel(const float* __restrict__ y, const float* __restrict__ add, float* __restrict__ out, int H, int top, int chunks) {
  typedef float Vec __attribute__((ext_vector_type(N)));
  const long long row = blockIdx.x / chunks;
  const int c = (blockIdx.x % chunks * 256 + threadIdx.x) * N;
  if (c >= H) return;
  Vec acc = 0.f;
  for (int s = 0; s < top; ++s) acc += *reinterpret_cast<const Vec*>(y + (row * top + s) * H + c);
  *reinterpret_cast<Vec*>(out + row * H + c) = add ? *reinterpret_cast<const Vec*>(add + row * H + c) + acc : acc;
}

// The tiles, of an even number of accumulators a wave, and what a launch of them takes (gemm_tiles.h).  The eight to twelve waves of tile_ring.h in large tiles
// but for 192 x 128: an expert's few tiles do not make up for the longer beginning and end of the four waves of tile_pipe.h.  Fitted to 6,200 timed
// launches of 13 tiles at 472 products (33 sizes of experts, 4 to 64 of them, 64 to 8,192 rows).  At 858 further products (65 sizes) the pick takes 0.967 of the time of these waves'
// by the constants of gemm_tiles.hip with half a tile lost an expert, and 0.945 of what that rule took with six of tile_pipe.h's tiles instead, which were slower than these
// by a tenth at a quarter of the products.  Up and down, us, six of tile_pipe.h / so: 5,632 columns of 2,048, 8 experts, one a row, 509 rows
// 117 / 94; 1,408 columns gated, two a row, 4,072 rows 198 / 187, 2,048 rows 94 / 96, 1,024 rows 62 / 66; 256 columns of 512, 64 experts, eight a row, 4,072 rows 66 / 57.
#define KVCM_GROUPED_TILES(T)                                      \
  T(64, 64, 2, 2, 4, false, 3.293f, 0.253f, 0.752f, 0.696f)        \
  T(128, 64, 4, 2, 6, false, 3.734f, 0.322f, 1.004f, 2.392f)       \
  T(128, 128, 2, 4, 4, false, 4.219f, 0.517f, 1.032f, 2.958f)      \
  T(192, 128, 2, 2, 3, true, 6.472f, 0.589f, 1.071f, 4.782f)       \
  T(256, 128, 4, 2, 3, false, 6.426f, 0.794f, 1.037f, 4.013f)      \
  T(256, 192, 4, 3, 2, false, 5.680f, 1.201f, 1.033f, 4.175f)      \
  T(256, 256, 2, 4, 2, false, 7.658f, 1.491f, 0.991f, 6.674f)

struct High {
  int bm, bn;
  TileTime time;
};
#define KVCM_HIGH(BM, BN, WM, WN, STAGES, PIPE, FIXED, STEP, SHARE, ROUND) {BM, BN, {FIXED, STEP, SHARE, ROUND}},
static constexpr High kHighs[] = {KVCM_GROUPED_TILES(KVCM_HIGH)};
#undef KVCM_HIGH
constexpr int kHighCount = sizeof(kHighs) / sizeof(kHighs[0]);
constexpr int kFarTile = 2;      // the one that is there with 64-bit offsets too
static_assert(kHighs[kFarTile].bm == 128 && kHighs[kFarTile].bn == 128, "launch_grouped names it");

// Tiles of bm pairs that n pairs over E experts make up, if each expert is as likely: the sum over j of P(an expert has more than j bm pairs)
static float expected_tiles(int n, int E, int bm) {
  const double mean = static_cast<double>(n) / E, sd = std::sqrt(mean);
  const int whole = mean > 6.0 * sd ? static_cast<int>((mean - 6.0 * sd) / bm) : 0;
  double sum = whole;
  for (int j = whole; static_cast<double>(j) * bm < mean + 6.0 * sd + 1.0; ++j) sum += 0.5 * std::erfc((static_cast<double>(j) * bm + 0.5 - mean) / (sd * 1.41421356));
  return static_cast<float>(E * sum);
}

// The tile for n pairs over E experts, N rows of K each.
static int best_grouped(int n, int E, int N, int K) {
  const float used = n < E ? static_cast<float>(n) : static_cast<float>(E), k = static_cast<float>(K);
  int best = 0;
  float best_t = 0.f;
  for (int i = 0; i < kHighCount; ++i) {
    const float cols = static_cast<float>((N + kHighs[i].bn - 1) / kHighs[i].bn);
    const float t = tile_time(kHighs[i].time, expected_tiles(n, E, kHighs[i].bm) * cols, (K + kStepK - 1) / kStepK, used * static_cast<float>(N) * k,
                              static_cast<float>(n) * k * cols);
    if (i == 0 || t < best_t) {
      best = i;
      best_t = t;
    }
  }
  return best;
}

struct GroupedCall {
  const void* A;
  int lda;
  const void* W;
  const int *order, *count;
  const int4* list;
  int top;
  void* out;
  const float* weight;
  int N, K, n, E;
  bool far;      // operands need offsets of 64 bits (the tile is kFarTile)
};

template <int MODE>
static int launch_grouped(int tile, const GroupedCall& c, hipStream_t s) {
  const int col_blocks = (c.N + kHighs[tile].bn - 1) / kHighs[tile].bn;
  const long long grid = (static_cast<long long>(c.n / kHighs[tile].bm + c.E) * col_blocks + 7) / 8 * 8;
  KVCM_REQUIRE(grid < (1ll << 31), "moe_grouped: too many tiles");
#define KVCM_GROUPED(BM, BN, WM, WN, STAGES, PIPE, OFFSET)                                                                                   \
  moe_grouped_kernel<BM, BN, WM, WN, STAGES, PIPE, MODE, OFFSET><<<static_cast<unsigned>(grid), WM * WN * kWave, 0, s>>>(                    \
      static_cast<const uint16_t*>(c.A), c.lda, static_cast<const uint16_t*>(c.W), c.order, c.count, c.list, c.top, c.out, c.weight,   \
      c.N, c.K, col_blocks)
  if (c.far) {
    KVCM_GROUPED(128, 128, 2, 4, 4, false, uint64_t);
    return launch_status("moe_grouped");
  }
  int i = 0;
#define KVCM_GROUPED_LAUNCH(BM, BN, WM, WN, STAGES, PIPE, FIXED, STEP, SHARE, ROUND) \
  if (tile == i++) KVCM_GROUPED(BM, BN, WM, WN, STAGES, PIPE, uint32_t);
  KVCM_GROUPED_TILES(KVCM_GROUPED_LAUNCH)
#undef KVCM_GROUPED_LAUNCH
#undef KVCM_GROUPED
  return launch_status("moe_grouped");
}

}  // namespace kvcm

using namespace kvcm;

extern "C" {

// Does the grouped form take these sizes?  (bfloat16; rows of 16-byte pieces)
int kvcm_moe_grouped_supported(int K, int F, int E) { return K > 0 && F > 0 && K % 8 == 0 && F % 8 == 0 && E > 0 && E <= 4096; }

// int32 values of work memory that a step of n pairs over E experts needs for its lists of tiles (16-byte aligned)
int kvcm_moe_grouped_lists(int n, int E) { return 4 + 8 * most_tiles(n, E); }
int kvcm_moe_grouped_tile_count() { return kHighCount; }
// the tile that the rule picks for n pairs over E experts and N rows of K each, as 1,000 x its pairs + its rows: for tests
int kvcm_moe_grouped_pick(int n, int E, int N, int K) {
  KVCM_REQUIRE(n > 0 && E > 0 && N > 0 && K > 0, "moe_grouped_pick: bad sizes");
  const High& tile = kHighs[best_grouped(n, E, N, K)];
  return tile.bm * 1000 + tile.bn;
}

// h [T, K] bfloat16; w_up [E, F, K], w_down [E, H, F] bfloat16; chosen [T * top], weight [T * top]; work memory:
// order [T * top] and lists [kvcm_moe_grouped_lists] (int32), act [T * top, F] (bfloat16), y [T * top, H] (32-bit); out [T, H] 32-bit.
// kind 0: act = square(relu(up)); 2: gelu(up); 1, gated: w_up [E, 2F, K] (gate and up rows interleaved sixteen at a time), act =
// silu(gate) * up.  weigh_input: the weights are factors on what the experts read, not on what they give.  add [T, H] 32-bit
// or null: out = add + the experts' sum.  tile_up, tile_down: which tiles (< 0: those the rule picks).
int kvcm_moe_grouped(const void* h, int ldh, const void* w_up, const void* w_down, const int* chosen, const float* weight,
                     int* order, int* lists, void* act, float* y, const float* add, float* out, int T, int K, int F, int H,
                     int top, int E, int kind, int weigh_input, int tile_up, int tile_down, hipStream_t s) {
  if (T == 0) return 0;
  KVCM_REQUIRE(T > 0 && top > 0 && H > 0 && ldh >= K, "moe_grouped: bad sizes");
  KVCM_REQUIRE(kvcm_moe_grouped_supported(K, F, E), "moe_grouped: sizes K=%d F=%d experts=%d are not supported", K, F, E);
  KVCM_REQUIRE(static_cast<long long>(T) * top < (1ll << 30), "moe_grouped: too many rows");
  KVCM_REQUIRE(ldh % 8 == 0 && reinterpret_cast<uintptr_t>(h) % 16 == 0 && reinterpret_cast<uintptr_t>(w_up) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(w_down) % 16 == 0 && reinterpret_cast<uintptr_t>(act) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(lists) % 16 == 0,
               "moe_grouped: operands must be 16-byte aligned");
  KVCM_REQUIRE(kind >= 0 && kind <= 2, "moe_grouped: unknown kind of experts %d (0 relu2, 1 silu gated, 2 gelu)", kind);
  KVCM_REQUIRE(kind != 1 || F % 16 == 0, "moe_grouped: gated experts of %d columns are not supported (a multiple of 16)", F);
  KVCM_REQUIRE(tile_up < kHighCount && tile_down < kHighCount, "moe_grouped: no such tile");
  const int n = T * top, up_rows = kind == 1 ? 2 * F : F;
  const bool far_up = static_cast<long long>(T) * ldh >= (1ll << 31) || K >= kFarRows, far_down = F >= kFarRows;
  tile_up = far_up ? kFarTile : tile_up < 0 ? best_grouped(n, E, up_rows, K) : tile_up;
  tile_down = far_down ? kFarTile : tile_down < 0 ? best_grouped(n, E, H, F) : tile_down;
  moe_group_kernel<<<1, 1024, 4 * E * sizeof(int), s>>>(chosen, n, E, order, lists, kHighs[tile_up].bm, kHighs[tile_down].bm);
  const int4* list = reinterpret_cast<const int4*>(lists + 4);
  const GroupedCall up{h, ldh, w_up, order, lists, list, top, act, weigh_input ? weight : nullptr, up_rows, K, n, E, far_up};
  int rc = kind == 1 ? launch_grouped<kUpGated>(tile_up, up, s) : kind == 2 ? launch_grouped<kUpGelu>(tile_up, up, s) : launch_grouped<kUp>(tile_up, up, s);
  if (rc) return rc;
  const GroupedCall down{act, F, w_down, order, lists + 1, list + most_tiles(n, E), top, y, weigh_input ? nullptr : weight, H, F, n, E, far_down};
  rc = launch_grouped<kDown>(tile_down, down, s);
  if (rc) return rc;
  // four columns a thread where rows are whole 16-byte pieces (2,048 rows of 2,048 columns, two experts each: 20 us a column at a
  // time with a long division for its row, 15 us so)
  const bool four = H % 4 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0 && reinterpret_cast<uintptr_t>(add) % 16 == 0 &&
                    reinterpret_cast<uintptr_t>(out) % 16 == 0;
  const int chunks = (H + (four ? 1023 : 255)) / (four ? 1024 : 256);
  KVCM_REQUIRE(static_cast<long long>(T) * chunks < (1ll << 31), "moe_grouped: too many rows");
  if (four) moe_combine_kernel<4><<<T * chunks, 256, 0, s>>>(y, add, out, H, top, chunks);
  else moe_combine_kernel<1><<<T * chunks, 256, 0, s>>>(y, add, out, H, top, chunks);
  return launch_status("moe_grouped");
}

}  // extern "C"
