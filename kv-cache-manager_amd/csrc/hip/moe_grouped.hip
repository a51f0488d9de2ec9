// The routed feed-forward for steps with many rows (bfloat16): the (row, slot) pairs are grouped by their expert and
// every expert's group is multiplied with that expert's matrices in tiles on the matrix cores, so that an expert's
// weights are read once per tile of 128 pairs and not once per pair.
//
//   moe_group      pairs p = row * top + slot, grouped by chosen[p]: order[] lists the pairs expert by expert, tiles[]
//                  lists (expert, first place in order, pairs) for every stretch of up to 128 pairs of one expert, with
//                  the number of tiles in front.  One workgroup; places inside a group are handed out by an atomic
//                  counter in LDS, so the order inside a group may differ from run to run, which changes no result: a
//                  pair's row of a tile is computed from that row alone.
//   moe_grouped    UP:   act[place, :] = square(relu(W_up[e] h[row of the pair])), or gelu of it (bfloat16, in grouped order)
//                  GATED UP: act[place, :] = silu(W_gate[e] h) * (W_up[e] h); the two matrices of an expert are stored as
//                        one of 2F rows, interleaved sixteen at a time (gate 0..15, up 0..15, gate 16..31, ...), so that a
//                        lane's neighbouring 16 x 16 tiles hold the gate and the up value of one column
//                  DOWN: y[pair, :]   = weight[pair] * W_down[e] act[place, :]               (32-bit, by pair)
//                  The pairs' weights may act on the other side instead: UP then reads weight * h (the factor is applied to
//                  its 32-bit sums) and DOWN weighs nothing.
//                  Tile 128 pairs x 128 columns per workgroup of four waves (64 x 64 each: 4 x 4 matrix instructions of
//                  16 x 16 x 32), K advanced 64 at a time through two halves of LDS: while one is multiplied the other fills.
//   moe_combine    out[row, :] = (add[row, :] +) sum over the row's slots, in slot order, of y[row * top + slot, :]
#include "common.h"
#include "kvcm_hip.h"

namespace kvcm {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

constexpr int kGM = 128, kGN = 128, kGK = 64;

union Frag {
  uint4 u;
  bf16x8 v;
};

// 64 k of both operands' 128 rows.  A row's eight 16-byte pieces are permuted by the row (piece p lies at place p ^ (row % 8)),
// so that eight rows of a fragment read meet no bank twice without any padding, which requests straight into LDS have no room for.
struct Stage {
  uint16_t a[kGM * kGK], b[kGN * kGK];
};

// 16 bytes a lane from memory straight into LDS: lane l's go to `to` + 16 l (the same `to` for the whole wave)
__device__ __forceinline__ void bring16(const uint16_t* from, uint16_t* to) {
  __builtin_amdgcn_global_load_lds(reinterpret_cast<const __attribute__((address_space(1))) void*>(reinterpret_cast<uintptr_t>(from)),
                                   reinterpret_cast<__attribute__((address_space(3))) void*>(reinterpret_cast<uintptr_t>(to)), 16, 0, 0);
}

// this wave's requests into LDS have arrived, and so have everybody else's of the workgroup
__device__ __forceinline__ void arrived_barrier() {
  __builtin_amdgcn_s_waitcnt(0x0f70);      // vmcnt(0)
  __syncthreads();
}

__global__ void __launch_bounds__(1024)
    moe_group_kernel(const int* __restrict__ chosen, int n, int E, int* __restrict__ order, int* __restrict__ tiles, int max_tiles) {
  extern __shared__ int sh[];      // count / cursor [E], base [E]
  int* cnt = sh;
  int* base = sh + E;
  for (int e = threadIdx.x; e < E; e += blockDim.x) cnt[e] = 0;
  __syncthreads();
  for (int p = threadIdx.x; p < n; p += blockDim.x) {
    const int e = chosen[p];
    if (e >= 0 && e < E) atomicAdd(&cnt[e], 1);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int at = 0, nt = 0;
    for (int e = 0; e < E; ++e) {
      base[e] = at;
      for (int r = 0; r < cnt[e] && nt < max_tiles; r += kGM) {
        tiles[1 + 3 * nt] = e;
        tiles[2 + 3 * nt] = at + r;
        tiles[3 + 3 * nt] = cnt[e] - r < kGM ? cnt[e] - r : kGM;
        ++nt;
      }
      at += cnt[e];
      cnt[e] = 0;
    }
    tiles[0] = nt;
  }
  __syncthreads();
  for (int p = threadIdx.x; p < n; p += blockDim.x) {
    const int e = chosen[p];
    if (e >= 0 && e < E) order[base[e] + atomicAdd(&cnt[e], 1)] = p;
  }
}

enum : int { kDown = 0, kUp = 1, kUpGated = 2, kUpGelu = 3 };

// A wave's requests for 64 k of 32 rows of each operand.  A piece past K is read from the row's start and left out of the products.
__device__ __forceinline__ void grouped_request(const uint16_t* const (&arow)[4], const uint16_t* const (&brow)[4], int k0, int piece, int K,
                                                int wave, Stage* to) {
  const int off = k0 + piece < K ? k0 + piece : 0;      // K is a multiple of 8: a piece lies inside or outside
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    bring16(arow[q] + off, &to->a[(wave * 32 + q * 8) * kGK]);
    bring16(brow[q] + off, &to->b[(wave * 32 + q * 8) * kGK]);
  }
}

// The wave's 64 x 64 results += 64 k (not WHOLE: the first `left` of them)
template <bool WHOLE>
__device__ __forceinline__ void grouped_multiply(int wm, int wn, int lane, const Stage* from, int left, f32x4 (&acc)[4][4]) {
  const int frow = lane % 16, fk = lane / 16;
#pragma unroll
  for (int ks = 0; ks < kGK / 32; ++ks) {
    const int at = ((ks * 4 + fk) ^ (frow % 8)) * 8;      // (rows 16 apart have the same permutation)
    const bool in = WHOLE || ks * 32 + fk * 8 < left;
    Frag a[4], b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i].u = *reinterpret_cast<const uint4*>(&from->a[(wm * 64 + i * 16 + frow) * kGK + at]);
#pragma unroll
    for (int j = 0; j < 4; ++j) b[j].u = *reinterpret_cast<const uint4*>(&from->b[(wn * 64 + j * 16 + frow) * kGK + at]);
    if constexpr (!WHOLE) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a[i].u = in ? a[i].u : uint4{0u, 0u, 0u, 0u};
        b[i].u = in ? b[i].u : uint4{0u, 0u, 0u, 0u};
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i].v, b[j].v, acc[i][j], 0, 0, 0);
  }
}

// One step: the next 64 k are asked for, then these are multiplied.  The two halves are told apart for the compiler (else it
// makes the first fragment read wait for the requests just made).
__device__ __forceinline__ void grouped_step(const uint16_t* const (&arow)[4], const uint16_t* const (&brow)[4], bool more, int k0, int piece,
                                             int K, int wave, int lane, const Stage* __restrict__ from, Stage* __restrict__ to,
                                             f32x4 (&acc)[4][4]) {
  if (more) grouped_request(arow, brow, k0, piece, K, wave, to);
  grouped_multiply<true>(wave / 2, wave % 2, lane, from, kGK, acc);
}

// N: rows of an expert's matrix (2F for the gated form); the output has N columns (F for the gated form)
template <int MODE>
__global__ void __launch_bounds__(256, 2)
    moe_grouped_kernel(const uint16_t* __restrict__ A, int lda, const uint16_t* __restrict__ W, const int* __restrict__ order,
                       const int* __restrict__ tiles, int top, void* __restrict__ out, const float* __restrict__ weight, int N,
                       int K, int col_blocks) {
  __shared__ __attribute__((aligned(16))) Stage staged[2];      // the results pass through it too
  __shared__ int pair_of[kGM];
  // The chip hands consecutive workgroups to its eight XCDs in turn, each with an L2 of its own.  Workgroup L goes to
  // XCD L % 8; it takes a column block that is congruent to its XCD and walks the tiles in order, so that the tiles of
  // one expert (neighbours in the list) meet the same blocks of that expert's matrix in the same L2.
  const int col_slots = (col_blocks + 7) / 8;
  const int xcd = blockIdx.x % 8, turn = blockIdx.x / 8;
  const int tile = turn / col_slots, col_block = (turn % col_slots) * 8 + xcd;
  if (col_block >= col_blocks || tile >= tiles[0]) return;
  const int e = tiles[1 + 3 * tile], p0 = tiles[2 + 3 * tile], rows = tiles[3 + 3 * tile];
  const int n0 = col_block * kGN;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
  if (tid < kGM) pair_of[tid] = order[p0 + (tid < rows ? tid : 0)];
  __syncthreads();
  // A wave brings 32 rows of each operand, 8 rows a request: lane l asks for row l / 8, and for the 16-byte piece of the
  // row's 64 k that belongs at place l % 8 of the permuted row.  Rows past the tile and columns past N repeat others of
  // their kind (what they give is not stored).
  const int piece = ((lane % 8) ^ (lane / 8)) * 8;
  const uint16_t* arow[4];
  const uint16_t* brow[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = wave * 32 + q * 8 + lane / 8;
    const long long src = MODE != kDown ? pair_of[r] / top : p0 + (r < rows ? r : 0);
    arow[q] = A + src * lda;
    const int c = n0 + r;
    brow[q] = W + (static_cast<long long>(e) * N + (c < N ? c : N - 1)) * K;
  }
  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int wm = wave / 2, wn = wave % 2;
  // One barrier a step: past it every wave's requests for this step are in LDS and nobody reads the other half any more.
  const int steps = (K + kGK - 1) / kGK, whole_steps = K / kGK;
  grouped_request(arow, brow, 0, piece, K, wave, &staged[0]);
  for (int t = 0; t < whole_steps; ++t) {
    arrived_barrier();
    grouped_step(arow, brow, t + 1 < steps, (t + 1) * kGK, piece, K, wave, lane, &staged[t & 1], &staged[(t + 1) & 1], acc);
  }
  if (whole_steps < steps) {
    arrived_barrier();
    grouped_multiply<false>(wm, wn, lane, &staged[whole_steps & 1], K - whole_steps * kGK, acc);
  }
  __syncthreads();
  // accumulator layout: a lane holds column lane % 16 and rows 4 * (lane / 16) + r of each 16 x 16 tile
  if constexpr (MODE == kDown) {
    // 32-bit results by pair: stored from the accumulators a wave's store would write 64-byte pieces of four rows.  Each
    // wave passes its 64 x 64 results through LDS instead, 32 rows at a time, and writes whole 256-byte stretches of
    // a row, 16 bytes a lane.
    constexpr int kPitch = 68;      // floats
    static_assert(4 * 32 * kPitch * sizeof(float) <= sizeof(staged), "the results of half a tile must fit the operands' space");
    float* mine = reinterpret_cast<float*>(&staged[0]) + wave * 32 * kPitch;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int ii = 0; ii < 2; ++ii)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            mine[(ii * 16 + (lane / 16) * 4 + r) * kPitch + j * 16 + lane % 16] = acc[half * 2 + ii][j][r];
      __syncthreads();
#pragma unroll
      for (int it = 0; it < 8; ++it) {
        const int idx = it * kWave + lane, rl = idx / 16, c4 = (idx % 16) * 4;
        const int m = wm * 64 + half * 32 + rl;
        const int c = n0 + wn * 64 + c4;
        if (m >= rows || c >= N) continue;
        const int pair = pair_of[m];
        const float g = weight ? weight[pair] : 1.f;
        const float4 v = *reinterpret_cast<const float4*>(mine + rl * kPitch + c4);
        float* dst = static_cast<float*>(out) + static_cast<long long>(pair) * N + c;
        if (c + 3 < N && N % 4 == 0) {
          *reinterpret_cast<float4*>(dst) = float4{g * v.x, g * v.y, g * v.z, g * v.w};
        } else {
          const float e4[4] = {v.x, v.y, v.z, v.w};
          for (int q = 0; q < 4 && c + q < N; ++q) dst[q] = g * e4[q];
        }
      }
      __syncthreads();
    }
    return;
  }
  // activations, in grouped order: a wave's 64 rows of them (32 columns where two accumulators make one, else 64) pass through
  // LDS as well and are written in whole 64- or 128-byte stretches of a row, 16 bytes a lane
  constexpr int kWide = MODE == kUpGated ? 32 : 64, kPitch = kWide + 8;
  static_assert(4 * 64 * kPitch * sizeof(uint16_t) <= sizeof(staged), "the activations of a tile must fit the operands' space");
  uint16_t* mine = reinterpret_cast<uint16_t*>(&staged[0]) + wave * 64 * kPitch;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int ml = i * 16 + (lane / 16) * 4 + r;
      const float g = weight ? weight[pair_of[wm * 64 + ml]] : 1.f;      // a factor on what the expert reads
      if constexpr (MODE == kUpGated) {
#pragma unroll
        for (int j = 0; j < 4; j += 2)      // tile j: sixteen gate columns, tile j + 1: the same sixteen up columns
          mine[ml * kPitch + j * 8 + lane % 16] = float_to_bf16_bits(silu<bf16_t>(g * acc[i][j][r]) * (g * acc[i][j + 1][r]));
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float v = g * acc[i][j][r], z = fmaxf(v, 0.f);
          mine[ml * kPitch + j * 16 + lane % 16] = float_to_bf16_bits(MODE == kUpGelu ? gelu_exact<bf16_t>(v) : z * z);
        }
      }
    }
  __syncthreads();
  const int cols = MODE == kUpGated ? N / 2 : N, c0 = (MODE == kUpGated ? n0 / 2 : n0) + wn * kWide;
#pragma unroll
  for (int it = 0; it < kWide / 8; ++it) {      // (the columns are a multiple of 8: a piece lies inside or outside)
    const int idx = it * kWave + lane, ml = idx / (kWide / 8), c8 = (idx % (kWide / 8)) * 8, c = c0 + c8;
    if (wm * 64 + ml >= rows || c >= cols) continue;
    *reinterpret_cast<uint4*>(static_cast<uint16_t*>(out) + static_cast<long long>(p0 + wm * 64 + ml) * cols + c) =
        *reinterpret_cast<const uint4*>(mine + ml * kPitch + c8);
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

}  // namespace kvcm

using namespace kvcm;

extern "C" {

// Does the grouped form take these sizes?  (bfloat16; rows of 16-byte pieces)
int kvcm_moe_grouped_supported(int K, int F, int E) { return K > 0 && F > 0 && K % 8 == 0 && F % 8 == 0 && E > 0 && E <= 4096; }

// Tiles a step of n pairs over E experts can have at most.
int kvcm_moe_grouped_max_tiles(int n, int E) { return (n + kGM - 1) / kGM + E; }

// h [T, K] bfloat16; w_up [E, F, K], w_down [E, H, F] bfloat16; chosen [T * top], weight [T * top]; work memory:
// order [T * top] and tiles [3 * max_tiles + 1] (int32), act [T * top, F] (bfloat16), y [T * top, H] (32-bit); out [T, H] 32-bit.
// kind 0: act = square(relu(up)); 2: gelu(up); 1, gated: w_up [E, 2F, K] (gate and up rows interleaved sixteen at a time), act =
// silu(gate) * up.  weigh_input: the weights are factors on what the experts read, not on what they give.  add [T, H] 32-bit
// or null: out = add + the experts' sum.
int kvcm_moe_grouped(const void* h, int ldh, const void* w_up, const void* w_down, const int* chosen, const float* weight,
                     int* order, int* tiles, void* act, float* y, const float* add, float* out, int T, int K, int F, int H,
                     int top, int E, int kind, int weigh_input, hipStream_t s) {
  if (T == 0) return 0;
  KVCM_REQUIRE(T > 0 && top > 0 && H > 0 && ldh >= K, "moe_grouped: bad sizes");
  KVCM_REQUIRE(kvcm_moe_grouped_supported(K, F, E), "moe_grouped: sizes K=%d F=%d experts=%d are not supported", K, F, E);
  KVCM_REQUIRE(static_cast<long long>(T) * top < (1ll << 30), "moe_grouped: too many rows");
  KVCM_REQUIRE(ldh % 8 == 0 && reinterpret_cast<uintptr_t>(h) % 16 == 0 && reinterpret_cast<uintptr_t>(w_up) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(w_down) % 16 == 0 && reinterpret_cast<uintptr_t>(act) % 16 == 0,
               "moe_grouped: operands must be 16-byte aligned");
  const int n = T * top, max_tiles = kvcm_moe_grouped_max_tiles(n, E);
  KVCM_REQUIRE(kind >= 0 && kind <= 2, "moe_grouped: unknown kind of experts %d (0 relu2, 1 silu gated, 2 gelu)", kind);
  KVCM_REQUIRE(kind != 1 || F % 16 == 0, "moe_grouped: gated experts of %d columns are not supported (a multiple of 16)", F);
  const int up_rows = kind == 1 ? 2 * F : F;
  const float *up_weight = weigh_input ? weight : nullptr, *down_weight = weigh_input ? nullptr : weight;
  const int up_blocks = (up_rows + kGN - 1) / kGN, down_blocks = (H + kGN - 1) / kGN;
  const long long up_grid = static_cast<long long>(max_tiles) * ((up_blocks + 7) / 8) * 8;
  const long long down_grid = static_cast<long long>(max_tiles) * ((down_blocks + 7) / 8) * 8;
  KVCM_REQUIRE(up_grid < (1ll << 31) && down_grid < (1ll << 31), "moe_grouped: too many tiles");
  moe_group_kernel<<<1, 1024, 2 * E * sizeof(int), s>>>(chosen, n, E, order, tiles, max_tiles);
#define KVCM_GROUPED_UP(MODE)                                                                                              \
  moe_grouped_kernel<MODE><<<static_cast<unsigned>(up_grid), 256, 0, s>>>(static_cast<const uint16_t*>(h), ldh,            \
                                                                          static_cast<const uint16_t*>(w_up), order, tiles, \
                                                                          top, act, up_weight, up_rows, K, up_blocks)
  if (kind == 1) KVCM_GROUPED_UP(kUpGated);
  else if (kind == 2) KVCM_GROUPED_UP(kUpGelu);
  else KVCM_GROUPED_UP(kUp);
#undef KVCM_GROUPED_UP
  moe_grouped_kernel<kDown><<<static_cast<unsigned>(down_grid), 256, 0, s>>>(
      static_cast<const uint16_t*>(act), F, static_cast<const uint16_t*>(w_down), order, tiles, top, y, down_weight, H, F, down_blocks);
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
