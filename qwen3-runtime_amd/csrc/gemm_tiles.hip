// bfloat16 matrix product for many rows by tiles through LDS: C[M, N] = A[M, K] * W[N, K]^T on
// MFMA, float32 accumulation, output bfloat16 or float32, optionally gated (W is [2N, K], gate rows
// and then up rows, and C the activation of the two) or cut along K into planes of float32 that the
// caller adds. tiles.h has the loop over K and what bounds it.
//
// The result goes through LDS so that rows are stored in whole lines: 64 -> 59 us for 2,048 x 6,144
// x 2,560, whose blocks all end at once. Blocks that make several tiles ask for the next one's first
// stages before they store the last one's result: 186 -> 179 us for gate/up at 2,048 rows, 976 tiles.
// Every output is a sum over K in the order of k, so its bits depend neither on M nor on the tile,
// only on the number of planes.
// Against the library's product (and gated_act behind it) at the 4B sizes, called in turn with it, weights of several
// layers, q/k/v, output, gate/up and down at 512 rows: 27 (27), 19 (24), 52 (69) and 34 us (51); at 2,048
// rows: 60 (58), 43 (51), 183 (195) and 85 us (107), output and down as float32 planes. See HipOps.choose_tile for which tile is taken.
#include "common.h"
#include "direct.h"
#include "gemm_epilogue.h"
#include "tiles.h"

struct TileArgs {
  const bf16_t* A;
  const bf16_t* W;
  void* C;
  int M, N, K;
  int mtiles, ntiles, parts;
  GatedEpilogue ep;
};

// Bytes of LDS that a tile's bfloat16 result passes through, and of LDS in all: the ring, and one stage more than the result
// where both fit (the first stage of the next tile has then a place beside it).
template <int BM, int BN, int WN, int GATED, typename TO>
constexpr int tile_result_bytes() {
  return sizeof(TO) == 4 ? 0 : BM * ((GATED ? BN : 2 * BN) + 16 * WN);
}
template <int BM, int BN, int WM, int WN, int S, int GATED, typename TO>
constexpr size_t tile_lds_bytes() {
  typedef Tile<BM, BN, WM, WN, S> T;
  constexpr size_t result = tile_result_bytes<BM, BN, WN, GATED, TO>(), both = result + T::STAGE;
  constexpr size_t least = T::RING > result ? T::RING : result;
  static_assert(least <= 160 * 1024, "the result of this tile does not fit LDS");
  return result > 0 && both > least && both <= 160 * 1024 ? both : least;
}

// WM x WN waves, each with BM / WM rows and BN / WN columns of the tile. GATED: 16 rows of the tile's
// weights are 8 gate rows and the 8 up rows that belong to them, so any BN makes BN / 2 columns.
template <int BM, int BN, int WM, int WN, int S, int GATED, typename TO, int POLICY = 0>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_bf16_tiles_kernel(TileArgs p) {
#ifdef __HIP_DEVICE_COMPILE__  // the host's compiler knows no buffer resources
  typedef Tile<BM, BN, WM, WN, S> T;
  constexpr int TM = T::TM, TN = T::TN;
  extern __shared__ __align__(16) unsigned char tiles_lds[];  // [S] stages, then the result
  const int lane = threadIdx.x & 63, wave = uniform_wave_number();
  const int wm = wave / WN, wn = wave % WN;
  const int r16 = lane & 15, quad = lane >> 4;
  const int K = p.K;

  // A tile of the launch by its number. Blocks reach the XCDs in turn: each gets a run of neighbouring tiles, so that its
  // L2 holds the rows they share. Runs go down bands of some 2,048 rows, column by column.
  const int total = p.mtiles * p.ntiles * p.parts;
  int part, m0, n0, s0, stages;
  unsigned aoff[T::AL], woff[T::WL];  // rows past the end repeat the last one and are not stored
  auto locate = [&](int tile) {
    const int xcd = tile & 7;
    int id = xcd * (total >> 3) + min(xcd, total & 7) + (tile >> 3);
    part = id / (p.mtiles * p.ntiles);
    id -= part * p.mtiles * p.ntiles;
    constexpr int BAND = 2048 / BM;
    const int band = id / (BAND * p.ntiles), in_band = id - band * BAND * p.ntiles;
    const int high = min(BAND, p.mtiles - band * BAND);
    m0 = (band * BAND + in_band % high) * BM;
    n0 = in_band / high * (GATED ? BN / 2 : BN);
    const int all = K >> 6, each = (all + p.parts - 1) / p.parts;
    s0 = min(all, part * each);
    stages = min(all, s0 + each) - s0;
#pragma unroll
    for (int j = 0; j < T::AL; ++j)
      aoff[j] = (unsigned)min(m0 + T::row_of(j, T::AU, wave, lane), p.M - 1) * (unsigned)(2 * K) + T::piece_of(lane);
#pragma unroll
    for (int j = 0; j < T::WL; ++j) {
      const int in_tile = T::row_of(j, T::WU, wave, lane);
      const int row = GATED ? min(n0 + 8 * (in_tile >> 4) + (in_tile & 7), p.N - 1) + ((in_tile & 8) ? p.N : 0)
                            : min(n0 + in_tile, p.N - 1);
      woff[j] = (unsigned)row * (unsigned)(2 * K) + T::piece_of(lane);
    }
  };
  const __amdgpu_buffer_rsrc_t a_buf = T::buffer(p.A, (size_t)p.M * K * 2);
  const __amdgpu_buffer_rsrc_t w_buf = T::buffer(p.W, (size_t)(GATED ? 2 : 1) * p.N * K * 2);

  // Where tiles are more than the compute units hold, a block makes several, gridDim.x apart (a multiple of 8: of the same
  // XCD), and asks for the first stages of the next one before it stores the last one's result: the stages whose
  // slots the result leaves free (FIRST of them; it lies at the end of LDS).
  constexpr int RESULT = tile_result_bytes<BM, BN, WN, GATED, TO>();
  constexpr int FIRST = RESULT == 0 ? S : ((int)tile_lds_bytes<BM, BN, WM, WN, S, GATED, TO>() - RESULT) / T::STAGE;
  unsigned char* const result = tiles_lds + tile_lds_bytes<BM, BN, WM, WN, S, GATED, TO>() - RESULT;
  int tile = blockIdx.x, fetched = 0;
  locate(tile);
  while (true) {
    f32x4_t acc[TM][TN];
    T::template products<POLICY>(a_buf, w_buf, aoff, woff, s0, stages, tiles_lds, fetched, acc);
    QRT_WAIT_LDS();
    QRT_BARRIER();  // nobody reads the ring any more
    // acc[i][j][r]: row 16 i + r16 of the wave's result, row 16 j + 4 quad + r of its weights
    TO* C = (TO*)p.C + (size_t)part * p.M * p.N;
    constexpr int ROWS = BM / WM, COLS = (GATED ? 8 : 16) * TN;
    const int mw = m0 + wm * ROWS, nw = n0 + wn * COLS;
    const bool more = tile + (int)gridDim.x < total;
    tile += gridDim.x;
    if (more) {
      locate(tile);
      T::template fetch_first<POLICY>(a_buf, w_buf, aoff, woff, s0, stages, tiles_lds, 0, FIRST);
    }
    if constexpr (sizeof(TO) == 4) {
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int m = mw + 16 * i + r16;
        if (m >= p.M) continue;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int n = nw + 16 * j + 4 * quad;
          if (n < p.N) *(f32x4_t*)(C + (size_t)m * p.N + n) = acc[i][j];
        }
      }
    } else {
      constexpr int PITCH = 2 * COLS + 16;
      unsigned char* own = result + wave * ROWS * PITCH;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        unsigned char* row = own + (16 * i + r16) * PITCH;
        if constexpr (GATED) {
          // the lower half of the lanes holds gate values and the upper half the up values that belong to
          // them: two tiles change halves, and every lane has a gate and an up value
          const int m = min(mw + 16 * i + r16, p.M - 1);
#pragma unroll
          for (int j = 0; j < TN; j += 2) {
            const bool pair = j + 1 < TN;  // a last single tile leaves the upper half idle
            float g[4], u[4], o[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              g[r] = acc[i][j][r], u[r] = acc[i][pair ? j + 1 : j][r];
              swap_halves(g[r], u[r]);
              // both rounded to bfloat16 first, as the unfused kernels see them
              g[r] = (float)(bf16_t)g[r], u[r] = (float)(bf16_t)u[r];
            }
            gated_act4(g, u, GATED == 1 ? QRT_ACT_SWIGLU : p.ep.kind, p.ep.limit, o);
            if (GATED == 2 && p.ep.row_scale) {
              const float by = p.ep.row_scale[m];
#pragma unroll
              for (int r = 0; r < 4; ++r) o[r] *= by;
            }
            if (pair || quad < 2) store4((bf16_t*)(row + 16 * (j + (quad >> 1)) + 8 * (quad & 1)), o);
          }
        } else {
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            float o[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] = p.ep.whole(acc[i][j][r]);
            store4((bf16_t*)(row + 32 * j + 8 * quad), o);
          }
        }
      }
      constexpr int PIECES = COLS / 8;  // of 16 bytes in a row
#pragma unroll
      for (int c0 = 0; c0 < ROWS * PIECES; c0 += 64) {
        const int c = c0 + lane, row = c / PIECES, at = c % PIECES;
        if (ROWS * PIECES % 64 && c >= ROWS * PIECES) break;
        const u32x4_t v = *(const u32x4_t*)(own + row * PITCH + 16 * at);
        const int m = mw + row, n = nw + 8 * at;
        if (m < p.M && n < p.N) *(u32x4_t*)(C + (size_t)m * p.N + n) = v;
      }
    }
    if (!more) break;
    fetched = FIRST < S ? FIRST : S;
    QRT_WAIT_LDS();
    QRT_BARRIER();  // the result's room is the ring's again
  }
#endif
}

template <int BM, int BN, int WM, int WN, int S, int GATED, typename TO, int POLICY = 0>
static int launch_tiles(TileArgs p, hipStream_t stream) {
  constexpr size_t smem = tile_lds_bytes<BM, BN, WM, WN, S, GATED, TO>();
  const int width = GATED ? BN / 2 : BN;
  p.mtiles = (p.M + BM - 1) / BM;
  p.ntiles = (p.N + width - 1) / width;
  const int64_t blocks = (int64_t)p.mtiles * p.ntiles * p.parts;
  QRT_CHECK(blocks < (1 << 30), "gemm_tiles: too many tiles for one launch (M=%d N=%d)", p.M, p.N);
  auto kernel = gemm_bf16_tiles_kernel<BM, BN, WM, WN, S, GATED, TO, POLICY>;
  static bool allowed = false;  // once per kernel: not inside a stream capture again and again
  if (smem > 64 * 1024 && !allowed) {
    if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess)
      return qrt_fail("gemm_tiles: cannot get %zu bytes of LDS", smem);
    allowed = true;
  }
  constexpr int64_t resident = 256 * (160 * 1024 / smem);  // blocks that the compute units hold
  kernel<<<(unsigned)(blocks < resident ? blocks : resident), 64 * WM * WN, smem, stream>>>(p);
  QRT_LAUNCH_CHECK("gemm_tiles");
  return 0;
}

template <int BM, int BN, int WM, int WN, int S>
static int by_result(const TileArgs& p, int out_dtype, int gated, hipStream_t stream) {
  if (gated == 1) return launch_tiles<BM, BN, WM, WN, S, 1, bf16_t>(p, stream);
  if (gated) return launch_tiles<BM, BN, WM, WN, S, 2, bf16_t>(p, stream);
  if (out_dtype == QRT_F32) return launch_tiles<BM, BN, WM, WN, S, 0, float>(p, stream);
  return launch_tiles<BM, BN, WM, WN, S, 0, bf16_t>(p, stream);
}

// C [M, N], or with parts > 1 (not gated, float32) planes [parts, M, N]; tile: a number of TILES in ops/hip.py.
// act_kind < 0: no gate; QRT_ACT_RELU2: none, but an activation of the whole result in bfloat16. Needs N a multiple of 16, K of 64, and operands at multiples of 16 bytes and of less
// than 4 GiB each (their offsets are 32 bits).
extern "C" int qrt_gemm_tiles(const void* a, const void* w, void* c, int out_dtype, int M, int N, int K, int tile, int parts,
                              int act_kind, float limit, const float* row_scale, hipStream_t stream) {
  const bool gated = act_kind >= 0 && act_kind != QRT_ACT_RELU2;
  QRT_CHECK(M >= 0 && N > 0 && K > 0, "gemm_tiles: bad sizes M=%d N=%d K=%d", M, N, K);
  QRT_CHECK(N % 16 == 0 && K % 64 == 0, "gemm_tiles: needs N %% 16 == 0 and K %% 64 == 0 (N=%d K=%d)", N, K);
  QRT_CHECK(out_dtype == QRT_BF16 || (out_dtype == QRT_F32 && !gated), "gemm_tiles: unknown output dtype %d", out_dtype);
  QRT_CHECK(parts >= 1 && parts <= 64, "gemm_tiles: bad number of K parts %d", parts);
  QRT_CHECK(parts == 1 || (!gated && out_dtype == QRT_F32), "gemm_tiles: K parts need no gate and float32 output");
  QRT_CHECK(act_kind <= QRT_ACT_RELU2, "gemm_tiles: unknown activation %d", act_kind);
  QRT_CHECK(act_kind != QRT_ACT_RELU2 || (out_dtype == QRT_BF16 && !row_scale), "gemm_tiles: an activation without a gate is of whole bfloat16 rows");
  QRT_CHECK(((uintptr_t)a | (uintptr_t)w | (uintptr_t)c) % 16 == 0, "gemm_tiles: operands must begin at multiples of 16 bytes");
  const uint64_t limit_bytes = (1ull << 32) - 128;
  QRT_CHECK((uint64_t)M * K * 2 <= limit_bytes && (uint64_t)(gated ? 2 : 1) * N * K * 2 <= limit_bytes,
            "gemm_tiles: an operand of 4 GiB or more (M=%d N=%d K=%d)", M, N, K);
  if (M == 0) return 0;
  const TileArgs p{(const bf16_t*)a, (const bf16_t*)w, c, M, N, K, 0, 0, parts, GatedEpilogue{act_kind, limit, row_scale}};
  const int mode = !gated ? 0 : act_kind == QRT_ACT_SWIGLU && !row_scale ? 1 : 2;
  switch (tile) {
    case 0: return by_result<256, 192, 4, 2, 2>(p, out_dtype, mode, stream);
    case 1: return by_result<256, 160, 4, 2, 3>(p, out_dtype, mode, stream);
    case 2: return by_result<256, 128, 4, 2, 3>(p, out_dtype, mode, stream);
    case 3: return by_result<192, 192, 4, 2, 3>(p, out_dtype, mode, stream);
    case 4: return by_result<192, 160, 4, 2, 3>(p, out_dtype, mode, stream);
    case 5: return by_result<192, 128, 4, 2, 3>(p, out_dtype, mode, stream);
    case 6: return by_result<128, 160, 2, 2, 4>(p, out_dtype, mode, stream);
    case 7: return by_result<128, 128, 2, 2, 4>(p, out_dtype, mode, stream);
    case 8: return by_result<128, 96, 2, 2, 4>(p, out_dtype, mode, stream);
    case 9: return by_result<96, 160, 2, 2, 4>(p, out_dtype, mode, stream);
    case 10: return by_result<96, 96, 2, 2, 6>(p, out_dtype, mode, stream);
    case 11: return by_result<128, 64, 2, 2, 6>(p, out_dtype, mode, stream);
    case 12:
      // One row tile: no block reads another's weights, so they come as data used once. As plain loads they put out of the L2s what the
      // kernels around the product read again, and every one of those took longer (the router of a 2,048-wide model 6.6 -> 8.1 us): decoding
      // 48 requests of the 2B size with latent attention took 2.52 ms a step with the kernel that shares the activations, 2.61 with
      // plain tiles and 2.50 so; the 4B size 3.71, 3.65 and 3.56.
      if (M <= 64 && mode == 0 && out_dtype == QRT_F32) return launch_tiles<64, 64, 1, 4, 4, 0, float, 2>(p, stream);
      return by_result<64, 64, 1, 4, 4>(p, out_dtype, mode, stream);
    case 13: return by_result<64, 128, 1, 4, 3>(p, out_dtype, mode, stream);
    default: return qrt_fail("gemm_tiles: no tile %d", tile);
  }
}
