// Routed experts' products in bfloat16 on MFMA, without the host in between.
//
// Pair p = (token t = p / top, its j-th expert e = index[p], j = p % top). The first product of all
// pairs, act = activation(G_e x, U_e x) (or of U_e x alone), and the second, w[p] * D_e act, written as
// float32 plane j of the result: out[j, t] is one pair's, so that no sum needs atomics and the norm that
// comes next adds the planes up in the pass in which it reads them. Sums, activation and weights stay
// float32 from the first product to `act` (bfloat16, as it always was) and from there to the planes.
//
// Two forms, by the number of pairs an expert has on average (see HipOps.moe_for_residual):
// * few: `experts_rows_kernel`, a stream of the chosen experts' weights. A block owns 16 weight rows (and
//   the 16 up rows that go with them) of one expert and finds that expert's pairs in `index` itself, by
//   ballots: no grouping kernel, no count that reaches the host. Weights and tokens come to LDS by direct
//   loads of whole cache lines, as in the few-row dense products. More than 16 pairs of an expert are taken 16 at a
//   time, the weights coming again from the caches.
// * many: `experts_tile_kernel`, tiles of the products of many rows (tiles.h) over an expert's pairs;
//   `experts_group_kernel` puts the pairs in their experts' order and lists the tiles.
//
// What they replace (MI355X, 16 experts of 2,560 x 1,536, 2 a token; us): a kernel of scalar products on LDS
// copies of a few rows, 58 + 27 and a grouping and a combining kernel of 4.5 + 8.9 for 8 tokens (now 28 + 17); one library
// product per expert and matrix behind a wait of the host, about 430 for 2,041 tokens, with the device idle for a
// sixth of the step.
#include "common.h"
#include "direct.h"
#include "tiles.h"

#define EXPERTS_DOWN 0   // second product: input rows by place, weighted float32 planes out
#define EXPERTS_GATED 1  // first product with a gate
#define EXPERTS_RELU2 2  // first product without one
#define QRT_ACT_RELU2 2

struct ExpertArgs {
  const bf16_t* in;      // MODE > 0: x [T, K]; MODE 0: act [pairs, K], by pair (rows kernel) or by place (tile kernel)
  const bf16_t* w;       // [E, N or 2N, K]
  const int* index;      // [pairs]
  const float* weight;   // [pairs] or null: 1. MODE 0: on the output; MODE > 0: on the input, in front of the activation
  void* out;             // MODE > 0: act [pairs, N] bfloat16, by pair / place; MODE 0: float32 [top, T, N]
  const int* order;      // tile kernel: the pair at every place
  const int* offsets;    // tile kernel: first place of every expert, [E + 1]
  const int* tiles;      // tile kernel: [1 + 2 n]: how many, then (expert, first place) of each
  int tokens, top, experts, K, N, act_kind;
  float limit;
};

template <int MODE>
__device__ __forceinline__ float expert_value(const ExpertArgs& a, float g, float u) {
  if (MODE == EXPERTS_RELU2) {
    g = fmaxf(g, 0.f);
    return g * g;
  }
  return gated_act(g, u, a.act_kind, a.limit);
}

// ------------------------------------------------------------------ few pairs an expert
// blockIdx.y: the expert, or (BY_PAIR: fewer pairs than experts) the pair that is its expert's first. The weight rows are
// blockIdx.x: blocks go to the eight XCDs in turn, and with the experts there an XCD had the work of experts e and e + 8
// (of 16), two, one or none of which are chosen (16 x 2,560 x 1,536, 8 tokens, some 10 of 16 chosen: 34.9 + 22.2 us, now 31.0 +
// 19.6). The weights are loaded as data used once, as in the few-row dense products (27.7 + 16.6 with that and the smallest rings:
// 16 rows and two pieces in flight a wave, three or four blocks a compute unit; 80 tokens, where an expert's weights come
// again from the caches: 49.1 + 29.4 -> 42.5 + 26.9).
template <int NW, int NT, int U, int MODE, bool BY_PAIR>
__global__ __launch_bounds__(64 * NW) void experts_rows_kernel(ExpertArgs a) {
  constexpr bool GATED = MODE == EXPERTS_GATED;
  constexpr int WT = GATED ? 2 * NT : NT, UNITS = WT + 1, LOADS = 2 * UNITS, SLOT = UNITS * 2048;
  static_assert((U - 1) * LOADS < 64, "the loads' counter holds 63");
  extern __shared__ __align__(16) unsigned char lds[];  // [NW][U][UNITS] x 2 KB, then the partial sums; behind: the expert's pairs
  int* list = (int*)(lds + NW * U * SLOT);
  const int lane = threadIdx.x & 63, wave = uniform_wave_number();
  const int pairs = a.tokens * a.top, K = a.K, N = a.N;
  const int e = BY_PAIR ? a.index[blockIdx.y] : blockIdx.y;
  // the expert's pairs in ascending order; every wave writes the same list
  int count = 0;
  for (int p0 = 0; p0 < pairs; p0 += 64) {
    const int p = p0 + lane;
    const bool hit = p < pairs && a.index[min(p, pairs - 1)] == e;
    const unsigned long long mask = __ballot(hit);
    if (hit) list[count + __popcll(mask & ((1ull << lane) - 1))] = p;
    count += __popcll(mask);
  }
  __syncthreads();
  count = __builtin_amdgcn_readfirstlane(count);
  if (count == 0 || (BY_PAIR && list[0] != (int)blockIdx.y)) return;  // the whole block alike
  const int r16 = lane & 15, quad = lane >> 4, n0 = blockIdx.x * 16 * NT;
  unsigned char* ring = lds + (size_t)wave * U * SLOT;
  const int sub = lane >> 3, piece = (lane & 7) ^ sub;
  const bf16_t* we = a.w + (size_t)e * (GATED ? 2 : 1) * N * K;
  const int all_pairs = K >> 6, mine = max(0, (all_pairs - wave + NW - 1) / NW);  // 64-wide pieces of K of this wave
  const int read_at[2] = {r16 * 128 + 16 * (quad ^ (r16 & 7)), r16 * 128 + 16 * ((4 + quad) ^ (r16 & 7))};
  for (int m0 = 0; m0 < count; m0 += 16) {
    const bf16_t* src[UNITS][2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int n = min(n0 + 16 * t + 8 * j + sub, N - 1);  // rows past the end repeat the last; not stored
        src[t][j] = we + (size_t)n * K + 8 * piece;
        if (GATED) src[NT + t][j] = we + (size_t)(N + n) * K + 8 * piece;
      }
      const int p = list[min(m0 + 8 * j + sub, count - 1)];
      src[WT][j] = a.in + (size_t)(MODE ? p / a.top : p) * K + 8 * piece;
    }
    auto fetch = [&](int i, int slot) {
      const size_t at = (size_t)(wave + i * NW) * 64;
      unsigned char* dst = ring + slot * SLOT;
#pragma unroll
      for (int un = 0; un < UNITS; ++un)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          if (un < WT)
            __builtin_amdgcn_global_load_lds((global_ptr_t)(src[un][j] + at), (lds_ptr_t)(dst + un * 2048 + j * 1024), 16, 0, 2);
          else
            __builtin_amdgcn_global_load_lds((global_ptr_t)(src[un][j] + at), (lds_ptr_t)(dst + un * 2048 + j * 1024), 16, 0, 0);
        }
    };
    f32x4_t acc[WT];
#pragma unroll
    for (int t = 0; t < WT; ++t) acc[t] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    int fetched = 0, slot = 0;
    for (; fetched < U && fetched < mine; ++fetched) fetch(fetched, fetched);
    for (int i = 0; i < mine; ++i) {
      if (fetched - i == U) QRT_WAIT_LOADS((U - 1) * LOADS);
      else QRT_WAIT_LOADS(0);
      const unsigned char* at = ring + slot * SLOT;
      bf16x8_t w[WT][2], x[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int t = 0; t < WT; ++t) w[t][h] = *(const bf16x8_t*)(at + t * 2048 + read_at[h]);
        x[h] = *(const bf16x8_t*)(at + WT * 2048 + read_at[h]);
      }
      QRT_WAIT_LDS();  // the slot is in registers: the next piece may overwrite it
      if (fetched < mine) {
        fetch(fetched, slot);
        ++fetched;
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < WT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[t][h], x[h], acc[t], 0, 0, 0);
      slot = slot + 1 == U ? 0 : slot + 1;
    }
    __syncthreads();  // every wave has read its last slot: the rings' room now takes the partial sums
    float* red = (float*)lds;  // [NW][WT][64][4]
#pragma unroll
    for (int t = 0; t < WT; ++t) *(f32x4_t*)(red + ((wave * WT + t) * 64 + lane) * 4) = acc[t];
    __syncthreads();
    for (int i = threadIdx.x; i < NT * 64; i += 64 * NW) {
      const int l = i & 63, t = i >> 6, m = m0 + (l & 15), n = n0 + 16 * t + 4 * (l >> 4);
      f32x4_t g = {0.f, 0.f, 0.f, 0.f}, u = g;
      for (int w = 0; w < NW; ++w) {  // the waves' parts in order
        g += *(const f32x4_t*)(red + ((w * WT + t) * 64 + l) * 4);
        if (GATED) u += *(const f32x4_t*)(red + ((w * WT + NT + t) * 64 + l) * 4);
      }
      if (m >= count) continue;
      const int p = list[m];
      const float by = a.weight ? a.weight[p] : 1.0f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (n + r >= N) break;
        if (MODE) ((bf16_t*)a.out)[(size_t)p * N + n + r] = from_f32<bf16_t>(expert_value<MODE>(a, g[r] * by, u[r] * by));
        else ((float*)a.out)[((size_t)(p % a.top) * a.tokens + p / a.top) * N + n + r] = g[r] * by;
      }
    }
    __syncthreads();  // before the next 16 pairs' pieces overwrite the sums
  }
}

// ------------------------------------------------------------------ many pairs an expert
// order[i] = the pair at place i (experts one after the other), offsets[e] = expert e's first place,
// tiles = how many, then (expert, first place) for every BM places of an expert. One block. Which of an
// expert's pairs gets which of its places is left to the order of the atomics; no result depends on it.
__global__ __launch_bounds__(1024) void experts_group_kernel(const int* __restrict__ index, int* __restrict__ order,
                                                             int* __restrict__ offsets, int* __restrict__ tiles, int pairs,
                                                             int experts, int bm) {
  extern __shared__ int smem[];  // [experts] counts, then [experts] first places
  int* count = smem;
  int* at = smem + experts;
  for (int e = threadIdx.x; e < experts; e += blockDim.x) count[e] = 0;
  __syncthreads();
  for (int p = threadIdx.x; p < pairs; p += blockDim.x) atomicAdd(&count[index[p]], 1);
  __syncthreads();
  if (threadIdx.x == 0) {
    int place = 0, n = 0;
    for (int e = 0; e < experts; ++e) {
      const int c = count[e];
      at[e] = place;
      offsets[e] = place;
      for (int first = 0; first < c; first += bm) {
        tiles[1 + 2 * n] = e;
        tiles[2 + 2 * n] = place + first;
        ++n;
      }
      place += c;
    }
    offsets[experts] = place;
    tiles[0] = n;
  }
  __syncthreads();
  for (int p = threadIdx.x; p < pairs; p += blockDim.x) order[atomicAdd(&at[index[p]], 1)] = p;
}

// BM places of one expert x BN weight rows (GATED: 8 gate rows and the 8 up rows that go with them in turn, BN / 2
// outputs). What bounds it is what bounds the dense products, and the places that an expert's last tile leaves empty:
// which tile is the best goes by how many pairs an expert has (HipOps.choose_experts_tiles). With one loop of 128 x 128
// tiles behind two barriers a stage, as it was, 2,041 tokens took 125 + 75 us in a prompt step of 16 experts of 2,560 x
// 1,536 with 2 a token.
template <int BM, int BN, int WM, int WN, int S, int MODE>
__global__ __launch_bounds__(64 * WM * WN, 2) void experts_tile_kernel(ExpertArgs a) {
#ifdef __HIP_DEVICE_COMPILE__  // the host's compiler knows no buffer resources
  typedef Tile<BM, BN, WM, WN, S> T;
  constexpr bool GATED = MODE == EXPERTS_GATED;
  constexpr int TM = T::TM, TN = T::TN, WIDTH = GATED ? BN / 2 : BN;
  extern __shared__ __align__(16) unsigned char lds[];  // [S] stages, then the result
  const int K = a.K, N = a.N, row_tiles = a.tiles[0], col_tiles = (N + WIDTH - 1) / WIDTH;
  // blocks go to the eight XCDs in turn: each takes a stretch of neighbouring tiles, an expert's row tiles
  // of the same weight rows first
  const int total = row_tiles * col_tiles, per = (total + 7) >> 3;
  const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || tile >= total) return;
  const int row_tile = tile % row_tiles, n0 = tile / row_tiles * WIDTH;
  const int e = __builtin_amdgcn_readfirstlane(a.tiles[1 + 2 * row_tile]);
  const int first = __builtin_amdgcn_readfirstlane(a.tiles[2 + 2 * row_tile]);
  const int rows = min(BM, __builtin_amdgcn_readfirstlane(a.offsets[e + 1]) - first);
  const int lane = threadIdx.x & 63, wave = uniform_wave_number();
  const int r16 = lane & 15, quad = lane >> 4, wm = wave / WN, wn = wave % WN;
  unsigned aoff[T::AL], woff[T::WL];
#pragma unroll
  for (int j = 0; j < T::AL; ++j) {
    const int r = min(T::row_of(j, T::AU, wave, lane), rows - 1);  // beyond the expert's last pair: that one again, not stored
    aoff[j] = (unsigned)(MODE ? a.order[first + r] / a.top : r) * (unsigned)(2 * K) + T::piece_of(lane);
  }
#pragma unroll
  for (int j = 0; j < T::WL; ++j) {
    const int r = T::row_of(j, T::WU, wave, lane);
    const int row = GATED ? min(n0 + 8 * (r >> 4) + (r & 7), N - 1) + ((r & 8) ? N : 0) : min(n0 + r, N - 1);
    woff[j] = (unsigned)row * (unsigned)(2 * K) + T::piece_of(lane);
  }
  const bf16_t* in = MODE ? a.in : a.in + (size_t)first * K;  // by token, or by place
  const size_t matrix = (size_t)(GATED ? 2 : 1) * N * K;
  f32x4_t acc[TM][TN];
  T::products(T::buffer(in, (size_t)(MODE ? a.tokens : rows) * K * 2), T::buffer(a.w + e * matrix, matrix * 2), aoff, woff, 0, K >> 6,
              lds, 0, acc);
  // acc[i][j][r]: place first + m + 16 i + r16, row 16 j + 4 quad + r of the wave's weights
  constexpr int ROWS = BM / WM, COLS = (GATED ? 8 : 16) * TN;
  const int mw = wm * ROWS, nw = n0 + wn * COLS;
  if (MODE == EXPERTS_DOWN) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = mw + 16 * i + r16;
      if (m >= rows) continue;
      const int p = a.order[first + m];
      const float by = a.weight ? a.weight[p] : 1.0f;
      float* out = (float*)a.out + ((size_t)(p % a.top) * a.tokens + p / a.top) * N;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = nw + 16 * j + 4 * quad;
        if (n < N) *(f32x4_t*)(out + n) = acc[i][j] * by;
      }
    }
    return;
  }
  // through LDS, so that rows are stored in whole lines
  constexpr int PITCH = 2 * COLS + 16, PIECES = COLS / 8;
  __syncthreads();  // nobody reads the ring any more
  unsigned char* own = lds + wave * ROWS * PITCH;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    unsigned char* row = own + (16 * i + r16) * PITCH;
    const float by = a.weight ? a.weight[a.order[first + min(mw + 16 * i + r16, rows - 1)]] : 1.0f;
#pragma unroll
    for (int j = 0; j < TN; j += GATED ? 2 : 1) {
      const bool pair = j + 1 < TN;  // GATED: two tiles change halves, a last single one leaves the upper half idle
      float g[4], u[4], o[4];
      bf16x4_t v;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        g[r] = acc[i][j][r], u[r] = GATED ? acc[i][pair ? j + 1 : j][r] : 0.f;
        if (GATED) swap_halves(g[r], u[r]);
        g[r] *= by, u[r] *= by;
      }
      if (GATED) gated_act4(g, u, a.act_kind, a.limit, o);
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = from_f32<bf16_t>(GATED ? o[r] : expert_value<MODE>(a, g[r], u[r]));
      if (!GATED) *(bf16x4_t*)(row + 32 * j + 8 * quad) = v;
      else if (pair || quad < 2) *(bf16x4_t*)(row + 16 * (j + (quad >> 1)) + 8 * (quad & 1)) = v;
    }
  }
#pragma unroll
  for (int c0 = 0; c0 < ROWS * PIECES; c0 += 64) {
    const int c = c0 + lane, row = c / PIECES, at = c % PIECES;
    if (ROWS * PIECES % 64 && c >= ROWS * PIECES) break;
    const u32x4_t v = *(const u32x4_t*)(own + row * PITCH + 16 * at);
    const int m = mw + row, n = nw + 8 * at;  // N is a multiple of 8: all or none
    if (m < rows && n < N) *(u32x4_t*)((bf16_t*)a.out + (size_t)(first + m) * N + n) = v;
  }
#endif
}

static bool lds_allowed(const void* kernel, size_t bytes) {
  return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) == hipSuccess;
}

template <int NT, int U, int MODE, bool BY_PAIR>
static int experts_rows_launch(const ExpertArgs& a, hipStream_t stream) {
  constexpr int NW = 4;
  const int pairs = a.tokens * a.top;
  const size_t smem = (size_t)NW * U * ((MODE == EXPERTS_GATED ? 2 : 1) * NT + 1) * 2048 + (size_t)pairs * 4;
  auto kernel = experts_rows_kernel<NW, NT, U, MODE, BY_PAIR>;
  static bool allowed = false;  // once per kernel: not inside a stream capture again and again
  if (!allowed && !lds_allowed((const void*)kernel, 160 * 1024)) return qrt_fail("experts: cannot get 160 KB of LDS");
  allowed = true;
  kernel<<<dim3((a.N + 16 * NT - 1) / (16 * NT), BY_PAIR ? pairs : a.experts), 64 * NW, smem, stream>>>(a);
  return 0;
}
template <int NT, int U, int MODE>
static int experts_rows(const ExpertArgs& a, hipStream_t stream) {
  return a.tokens * a.top < a.experts ? experts_rows_launch<NT, U, MODE, true>(a, stream) : experts_rows_launch<NT, U, MODE, false>(a, stream);
}

template <int BM, int BN, int WM, int WN, int S, int MODE>
static int experts_tile_launch(const ExpertArgs& a, hipStream_t stream) {
  constexpr size_t ring = Tile<BM, BN, WM, WN, S>::RING;
  constexpr size_t result = MODE == EXPERTS_DOWN ? 0 : (size_t)BM * ((MODE == EXPERTS_GATED ? BN : 2 * BN) + 16 * WN);
  constexpr size_t smem = ring > result ? ring : result;
  static_assert(smem <= 160 * 1024, "the result of this tile does not fit LDS");
  auto kernel = experts_tile_kernel<BM, BN, WM, WN, S, MODE>;
  static bool allowed = false;
  if (!allowed && !lds_allowed((const void*)kernel, smem)) return qrt_fail("experts: cannot get %zu bytes of LDS", smem);
  allowed = true;
  const int pairs = a.tokens * a.top, bn = MODE == EXPERTS_GATED ? BN / 2 : BN;
  const long row_tiles = pairs / BM + (pairs < a.experts ? pairs : a.experts);  // at most: one ragged tile an expert
  const long blocks = (row_tiles * ((a.N + bn - 1) / bn) + 7) / 8 * 8;
  QRT_CHECK(blocks < (1l << 31), "experts: too many tiles");
  kernel<<<(unsigned)blocks, 64 * WM * WN, smem, stream>>>(a);
  return 0;
}

// The tiles that experts take, by their numbers in TILES of ops/hip.py (plus EXPERTS_TWO_BLOCKS: with half the stages, so that
// two blocks share a compute unit); rows of each, or 0.
#define EXPERTS_TWO_BLOCKS 16
static int experts_tile_rows(int tile) {
  switch (tile) {
    case 3: case 4: case 5: return 192;
    case 7: case 7 + EXPERTS_TWO_BLOCKS: return 128;
    case 12: case 13: return 64;
    default: return 0;
  }
}
template <int MODE>
static int experts_tile(const ExpertArgs& a, int tile, hipStream_t stream) {
  switch (tile) {
    case 3: return experts_tile_launch<192, 192, 4, 2, 3, MODE>(a, stream);
    case 4: return experts_tile_launch<192, 160, 4, 2, 3, MODE>(a, stream);
    case 5: return experts_tile_launch<192, 128, 4, 2, 3, MODE>(a, stream);
    case 7: return experts_tile_launch<128, 128, 2, 2, 4, MODE>(a, stream);
    case 7 + EXPERTS_TWO_BLOCKS: return experts_tile_launch<128, 128, 2, 2, 2, MODE>(a, stream);
    case 12: return experts_tile_launch<64, 64, 1, 4, 4, MODE>(a, stream);
    case 13: return experts_tile_launch<64, 128, 1, 4, 3, MODE>(a, stream);
    default: return qrt_fail("experts: no tile %d", tile);
  }
}

// x [T, H], gate_up [E, 2I or I, H], down [E, H, I], index and weight [T, top] -> act [pairs, I] (scratch), out [top, T, H]
// float32 planes. `scratch`: null for the few-pairs form; else int32 [pairs + E + 1 + 1 + 2 (pairs / BM + E)], and `tile` and
// `tile_down` the two products' tiles, both of BM rows.
extern "C" int qrt_experts(const void* x, const void* gate_up, const void* down, const int* index, const float* weight,
                           void* act, float* out, int* scratch, int tokens, int hidden, int inter, int experts, int top,
                           int act_kind, float limit, int weight_on_input, int tile, int tile_down, hipStream_t stream) {
  QRT_CHECK(tokens >= 0 && hidden > 0 && inter > 0 && experts >= 1 && experts <= 1024 && top >= 1, "experts: bad sizes");
  QRT_CHECK(hidden % 64 == 0 && inter % 64 == 0, "experts: widths %d and %d are no multiples of 64", hidden, inter);
  QRT_CHECK(act_kind == QRT_ACT_SWIGLU || act_kind == QRT_ACT_CLAMPED || act_kind == QRT_ACT_RELU2, "experts: unknown activation %d", act_kind);
  QRT_CHECK(!weight_on_input || act_kind != QRT_ACT_RELU2, "experts: weights on the input go with gated experts");
  QRT_CHECK((long)tokens * top < (1l << 30), "experts: too many pairs");
  QRT_CHECK(((uintptr_t)x | (uintptr_t)gate_up | (uintptr_t)down | (uintptr_t)act | (uintptr_t)out) % 16 == 0, "experts: operands begin at multiples of 16 bytes");
  if (tokens == 0) return 0;
  const int pairs = tokens * top;
  QRT_CHECK(scratch || (size_t)pairs * 4 <= 32 * 1024, "experts: %d pairs are too many for the form of few", pairs);
  const uint64_t limit_bytes = (1ull << 32) - 128;  // tiles' offsets are 32 bits
  const int bm = experts_tile_rows(tile);
  QRT_CHECK(!scratch || (bm > 0 && bm == experts_tile_rows(tile_down)), "experts: no two tiles %d and %d of as many rows", tile, tile_down);
  QRT_CHECK(!scratch || ((uint64_t)tokens * hidden * 2 <= limit_bytes && (uint64_t)4 * inter * hidden <= limit_bytes),
            "experts: tiles take operands of less than 4 GiB (%d tokens of %d, %d wide)", tokens, hidden, inter);
  ExpertArgs a{};
  a.index = index; a.tokens = tokens; a.top = top; a.experts = experts; a.act_kind = act_kind; a.limit = limit;
  if (scratch) {
    int* order = scratch;
    int* offsets = order + pairs;
    int* tiles = offsets + experts + 1;
    experts_group_kernel<<<1, 1024, (size_t)experts * 8, stream>>>(index, order, offsets, tiles, pairs, experts, bm);
    a.order = order; a.offsets = offsets; a.tiles = tiles;
  }
  a.in = (const bf16_t*)x; a.w = (const bf16_t*)gate_up; a.weight = weight_on_input ? weight : nullptr; a.out = act;
  a.K = hidden; a.N = inter;
  int rc;
  if (act_kind == QRT_ACT_RELU2) rc = scratch ? experts_tile<EXPERTS_RELU2>(a, tile, stream) : experts_rows<2, 3, EXPERTS_RELU2>(a, stream);
  else rc = scratch ? experts_tile<EXPERTS_GATED>(a, tile, stream) : experts_rows<1, 2, EXPERTS_GATED>(a, stream);
  if (rc != 0) return rc;
  a.in = (const bf16_t*)act; a.w = (const bf16_t*)down; a.weight = weight_on_input ? nullptr : weight; a.out = out;
  a.K = inter; a.N = hidden;
  rc = scratch ? experts_tile<EXPERTS_DOWN>(a, tile_down, stream) : experts_rows<1, 2, EXPERTS_DOWN>(a, stream);
  if (rc != 0) return rc;
  QRT_LAUNCH_CHECK("experts");
  return 0;
}
