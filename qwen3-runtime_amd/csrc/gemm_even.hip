// Few rows by a weight whose tiles of 16 rows do not share out: C[M, N] = A[M, K] W[N, K]^T in bfloat16, M <= 16, with as many weight rows for
// one compute unit as for the next.
//
// What bounds a few-row product is the stream of the weights into the busiest compute unit. 6,144 rows are 384 tiles, so some of 256 units get two
// and some one; 10,240 are 640, three or two. Here unit b has rows b N / 256 to (b + 1) N / 256 (24, 40), in units of eight as a direct load brings them. Loads,
// ring, and four waves that take the pairs of k-steps round-robin and meet in LDS are the few-row product's (gemm_bf16.hip), so the sums are its
// sums, bit by bit. us, weights of 24 layers in turn from a graph, by tiles and by this kernel at 1, 8 and 16 rows:
//   6,144 x 2,560   7.1, 7.75, 8.5 and 7.0, 7.2, 7.9;  of scaled rows 7.2, 7.8, 8.7 and 6.9, 7.15, 8.1
//   4,608 x 2,560   6.7, 7.6, 9.1 and 6.0, 6.2, 6.9;    6,144 x 4,096  10.4, 11.1, 12.9 and 10.3, 10.3, 10.55
//   9,728 x 2,560  10.6, 11.6, 13.4 and 9.9, 10.2, 10.7; 10,240 x 2,560  10.7, 11.75, 13.7 and 10.4, 10.55, 11.1 (5 TB/s);  10,240 x 5,120  19.1, 21.2, 24.2 and 18.2,
//   18.6, 19.2;  12,288 x 2,560  11.7, 12.4, 14.4 and 11.9, 12.1, 12.6
// Three pairs in flight a wave with three units (two 7.4 and four 7.3 at 8 rows of 6,144 x 2,560), two with five and six (10.55, three 10.7, four 10.8 at
// 10,240 x 2,560); eight waves of two pairs 7.25 and 10.5, with other bits.
// A decode pass of eight requests 19.07 -> 18.96 ms, with experts 25.04 -> 24.81.
#include "common.h"
#include "direct.h"
#include "gemm_even.h"

// U pairs in flight; UW units of eight weight rows and AR rows of activations are fetched.
template <int NW, int U, int AR, int UW, bool SCALED>
__global__ __launch_bounds__(64 * (NW + SCALED)) void gemm_bf16_even_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                                            bf16_t* __restrict__ C, int M, int N, int K, GatedEpilogue ep, RowNorm norm) {
  constexpr int AL = AR / 8, LOADS = UW + AL, SLOT = LOADS * 1024, TILES = (UW + 1) / 2;
  constexpr int ONCE = 2;  // the cache policy of a non-temporal load
  static_assert(AR <= 16 && (U - 1) * LOADS < 64, "one MFMA tile of activations, the loads' counter");
  extern __shared__ __align__(16) unsigned char even_lds[];  // [NW][U][SLOT], then the partial sums
  const int lane = threadIdx.x & 63, wave = uniform_wave_number();
  const int r16 = lane & 15, quad = lane >> 4;
  const int n0 = (int)((unsigned)blockIdx.x * (unsigned)N / EVEN_BLOCKS), n1 = (int)((blockIdx.x + 1u) * (unsigned)N / EVEN_BLOCKS);
  unsigned char* ring = even_lds + (size_t)wave * U * SLOT;
  const int sub = lane >> 3, piece = (lane & 7) ^ sub;
  const bf16_t *wsrc[UW], *asrc[AL];
  bool wthere[UW], athere[AL];
#pragma unroll
  for (int j = 0; j < UW; ++j) {
    wthere[j] = 8 * j + sub < max(n1 - n0, 8 * j + 1);  // a block without a unit's rows fetches one: see fetch
    wsrc[j] = W + (size_t)min(n0 + 8 * j + sub, N - 1) * K + 8 * piece;
  }
#pragma unroll
  for (int j = 0; j < AL; ++j) {
    athere[j] = 8 * j + sub < max(M, 8 * j + 1);
    asrc[j] = A + (size_t)min(8 * j + sub, M - 1) * K + 8 * piece;
  }
  const int pairs = K >> 6;
  const int mine = wave < NW ? max(0, (pairs - wave + NW - 1) / NW) : 0;
  // The wave's i-th pair of k-steps into a slot of its ring. Lanes of rows that are not there sit out (results of columns that are not stored), but
  // the waits below count LOADS loads a pair, so each has a lane that takes part: a load without any could be jumped over.
  auto fetch = [&](int i, int slot) {
    const size_t at = (size_t)(wave + i * NW) * 64;
    unsigned char* dst = ring + slot * SLOT;
#pragma unroll
    for (int j = 0; j < UW; ++j)
      if (wthere[j]) __builtin_amdgcn_global_load_lds((global_ptr_t)(wsrc[j] + at), (lds_ptr_t)(dst + j * 1024), 16, 0, ONCE);
#pragma unroll
    for (int j = 0; j < AL; ++j)
      if (athere[j]) __builtin_amdgcn_global_load_lds((global_ptr_t)(asrc[j] + at), (lds_ptr_t)(dst + (UW + j) * 1024), 16, 0, 0);
  };
  f32x4_t acc[TILES];
#pragma unroll
  for (int t = 0; t < TILES; ++t) acc[t] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  __shared__ float factor[SCALED ? AR : 1];
  int fetched = 0;
  for (; fetched < U && fetched < mine; ++fetched) fetch(fetched, fetched);
  if (SCALED && wave == NW) {  // a wave of its own, as in the few-row product
    f32x4_t parts[AR];
#pragma unroll
    for (int m = 0; m < AR; ++m) parts[m] = *(const f32x4_t*)(norm.squares + (size_t)min(m, M - 1) * SQUARE_PARTS + 4 * lane);
    float f[AR];
#pragma unroll
    for (int m = 0; m < AR; ++m) f[m] = norm.factor(parts[m]);
    if (lane == 0)
#pragma unroll
      for (int m = 0; m < AR; ++m) factor[m] = f[m];
  }
  const int ar = AR == 8 ? r16 & 7 : r16;
  int slot = 0;
  for (int i = 0; i < mine; ++i) {
    // pair i has landed when at most the U - 1 pairs behind it are on their way
    if (fetched - i == U) QRT_WAIT_LOADS((U - 1) * LOADS);
    else QRT_WAIT_LOADS(0);
    const unsigned char* at = ring + slot * SLOT;
    bf16x8_t w[TILES][2], a[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int in_row = 16 * ((4 * h + quad) ^ (r16 & 7));
#pragma unroll
      for (int t = 0; t < TILES; ++t) w[t][h] = *(const bf16x8_t*)(at + t * 2048 + (2 * t + 1 < UW ? r16 : r16 & 7) * 128 + in_row);
      a[h] = *(const bf16x8_t*)(at + UW * 1024 + ar * 128 + in_row);
    }
    QRT_WAIT_LDS();  // the slot is in registers: the next pair may overwrite it
    if (fetched < mine) {
      fetch(fetched, slot);
      ++fetched;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int t = 0; t < TILES; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[t][h], a[h], acc[t], 0, 0, 0);
    slot = slot + 1 == U ? 0 : slot + 1;
  }
  __syncthreads();  // every wave has read its last slot: the rings' room now takes the partial sums
  float* red = (float*)even_lds;  // [NW][TILES][4][64]
  if (wave < NW) {
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[((wave * TILES + t) * 4 + r) * 64 + lane] = acc[t][r];
  }
  __syncthreads();
  for (int i = threadIdx.x; i < TILES * 16 * AR; i += 64 * (NW + SCALED)) {
    const int c = i & 15, m = (i >> 4) % AR, t = (i >> 4) / AR, n = n0 + 16 * t + c;
    float sum = 0.f;  // the waves' parts in order
#pragma unroll
    for (int w = 0; w < NW; ++w) sum += red[((w * TILES + t) * 4 + (c & 3)) * 64 + (c >> 2) * 16 + m];
    if (SCALED) sum *= factor[m];
    if (m < M && n < n1) C[(size_t)m * N + n] = (bf16_t)ep.whole(sum);
  }
}

template <int NW, int U, int AR, int UW, bool SCALED>
static int launch(const bf16_t* a, const bf16_t* w, bf16_t* c, int M, int N, int K, const GatedEpilogue& ep, const RowNorm& norm,
                  hipStream_t stream) {
  constexpr size_t ring = (size_t)NW * U * (AR / 8 + UW) * 1024, meet = (size_t)NW * ((UW + 1) / 2) * 1024, smem = ring > meet ? ring : meet;
  static_assert(smem + 64 <= 160 * 1024, "the rings of this configuration do not fit LDS");
  auto kernel = gemm_bf16_even_kernel<NW, U, AR, UW, SCALED>;
  static bool allowed = false;  // once per kernel: not inside a stream capture again and again
  if (smem + 64 > 64 * 1024 && !allowed) {  // with the factors
    if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess)
      return qrt_fail("gemm_even: cannot get %zu bytes of LDS", smem);
    allowed = true;
  }
  kernel<<<EVEN_BLOCKS, 64 * (NW + SCALED), smem, stream>>>(a, w, c, M, N, K, ep, norm);
  QRT_LAUNCH_CHECK("gemm_even");
  return 0;
}

template <int U, int UW>
static int by_rows(const bf16_t* a, const bf16_t* w, bf16_t* c, int M, int N, int K, const GatedEpilogue& ep, const RowNorm* norm, hipStream_t stream) {
  if (norm) return M <= 8 ? launch<4, U, 8, UW, true>(a, w, c, M, N, K, ep, *norm, stream) : launch<4, U, 16, UW, true>(a, w, c, M, N, K, ep, *norm, stream);
  return M <= 8 ? launch<4, U, 8, UW, false>(a, w, c, M, N, K, ep, RowNorm{}, stream) : launch<4, U, 16, UW, false>(a, w, c, M, N, K, ep, RowNorm{}, stream);
}

int even_product(const bf16_t* a, const bf16_t* w, bf16_t* c, int M, int N, int K, const GatedEpilogue& ep, const RowNorm* norm, hipStream_t stream) {
  QRT_CHECK(even_takes(M, N, K) && M > 0 && M <= 16 && K > 0 && K % 64 == 0, "gemm_even: bad sizes M=%d N=%d K=%d", M, N, K);
  switch (even_units(N)) {
    case 3: return by_rows<3, 3>(a, w, c, M, N, K, ep, norm, stream);
    case 5: return by_rows<2, 5>(a, w, c, M, N, K, ep, norm, stream);
    default: return by_rows<2, 6>(a, w, c, M, N, K, ep, norm, stream);
  }
}

// For tests: whether few rows of a bfloat16 result are shared evenly.
extern "C" int qrt_gemm_even_takes(int M, int N, int K) { return even_takes(M, N, K); }
