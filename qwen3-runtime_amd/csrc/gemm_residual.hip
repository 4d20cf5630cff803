// Few rows: a product that is only added to the residual stream, the addition, and the RMS norm behind it.
//
// residual[M, N] += A[M, K] W[N, K]^T in float32; out[M, N] = residual * weight in bfloat16, the norm's rows but for their factor
// 1 / rms, which the products that read them multiply their sums by (gemm_bf16.hip, SCALED): a factor of a whole row passes through
// a product, and a rounding to bfloat16 is as large in relation to its value before it as behind it. What the factor is made of leaves
// as squares[M, SQUARE_PARTS]: each block's part of the rows' sums of squares, which every consumer adds up in an order of its own (few-row products
// as RowNorm::factor has it, the product that shares activations a quad of lanes at a time), whatever the other rows.
//
// Until there was this kernel K was cut over blocks, whose planes a kernel of a block a row added up and normed: 3 to 4 us of a
// boundary and two trips to memory for 40 KB a row. Here K stays whole in a block and the 256 compute units share the weight rows
// evenly instead (2,560 are 10 each), so a block has the row's elements of its columns complete. What bounds it is the stream of the
// weights and a kernel's start and end. Eight waves take the pairs of k-steps round-robin, as in the few-row product, through rings of
// U pairs by direct loads to LDS; a load fetches 8 rows x 128 bytes, lanes of rows that are not there sit out (their places in LDS hold
// what was there: results of columns that are not stored). us, the product in planes and the norm against this
// kernel, weights of 36 layers in turn, from a graph, 1, 8 and 16 rows:
//   2,560 x 4,096  9.0, 9.4, 10.5 and 6.2, 6.6, 7.6;  2,560 x 9,728  13.5, 14.2, 15.6 and 10.3, 11.3, 13.6.
// Narrower and wider residuals, with the product that reads the rows behind it, in planes and by this kernel: 256 x 256 (and 768 x 256) 6.6, 6.9, 6.9 and 5.2, 5.6,
// 6.2; 1,024 x 3,072 (4,096) 9.8, 10.1, 13.1 and 7.8, 8.2, 9.8; 2,048 x 6,144 (4,096) 14.1, 14.6, 16.7 and 11.9, 12.8, 14.5; 4,096 x 14,336 (6,144) 33.5, 34.4, 34.9 and
// 30.4, 30.9, 34.6; least at 16 rows of 4,096 x 12,288, in front of a gated product of 12,288 outputs 54.4 and 54.7.
// Four waves of eight pairs 6.7, 7.2 and 10.7, 11.6; sixteen of two 6.3, 6.8 and 10.6, 11.7; tiles of 16 rows on 160 compute units 6.6, 7.4
// and 11.0, 13.1; of eight rows on 320 7.4, 8.2 and 12.8, 15.6.
#include "common.h"
#include "direct.h"
#include "row_norm.h"

// AR rows of activations and WR weight rows, in units of eight, are fetched.
template <int NW, int U, int AR, int WR>
__global__ __launch_bounds__(64 * NW) void gemm_residual_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, int M, int N,
                                                                 int K, float* __restrict__ residual, const float* __restrict__ weight,
                                                                 bf16_t* __restrict__ out, float* __restrict__ squares) {
  constexpr int WL = WR / 8, AL = AR / 8, LOADS = WL + AL, SLOT = LOADS * 1024;
  constexpr int ONCE = 2;  // the cache policy of a non-temporal load
  static_assert(WR <= 16 && AR <= 16 && NW >= 4 && (U - 1) * LOADS < 64, "one MFMA tile, a thread an element, the loads' counter");
  extern __shared__ __align__(16) unsigned char ring_lds[];  // [NW][U][SLOT], then the partial sums
  const int lane = threadIdx.x & 63, wave = uniform_wave_number();
  const int r16 = lane & 15, quad = lane >> 4;
  const int n0 = (int)((unsigned)blockIdx.x * (unsigned)N / SQUARE_PARTS), n1 = (int)((blockIdx.x + 1u) * (unsigned)N / SQUARE_PARTS);
  unsigned char* ring = ring_lds + (size_t)wave * U * SLOT;
  const int sub = lane >> 3, piece = (lane & 7) ^ sub;
  const bf16_t *wsrc[WL], *asrc[AL];
  bool wthere[WL], athere[AL];
#pragma unroll
  for (int j = 0; j < WL; ++j) {
    wthere[j] = 8 * j + sub < max(n1 - n0, 8 * j + 1);  // a block of eight rows fetches a ninth: see fetch
    wsrc[j] = W + (size_t)min(n0 + 8 * j + sub, N - 1) * K + 8 * piece;
  }
#pragma unroll
  for (int j = 0; j < AL; ++j) {
    athere[j] = 8 * j + sub < M;
    asrc[j] = A + (size_t)min(8 * j + sub, M - 1) * K + 8 * piece;
  }
  const int pairs = K >> 6;
  const int mine = max(0, (pairs - wave + NW - 1) / NW);
  // The wave's i-th pair into a slot of its ring. The waits below count LOADS loads a pair, so each has a lane that takes part: a load
  // without any could be jumped over (AR and WR are the least that hold the most rows there are).
  auto fetch = [&](int i, int slot) {
    const size_t at = (size_t)(wave + i * NW) * 64;
    unsigned char* dst = ring + slot * SLOT;
#pragma unroll
    for (int j = 0; j < WL; ++j)
      if (wthere[j]) __builtin_amdgcn_global_load_lds((global_ptr_t)(wsrc[j] + at), (lds_ptr_t)(dst + j * 1024), 16, 0, ONCE);
#pragma unroll
    for (int j = 0; j < AL; ++j)
      if (athere[j]) __builtin_amdgcn_global_load_lds((global_ptr_t)(asrc[j] + at), (lds_ptr_t)(dst + (WL + j) * 1024), 16, 0, 0);
  };
  // thread t of the first 256 ends up with row t / 16, column t % 16 of the block's
  const int m = threadIdx.x >> 4, c = threadIdx.x & 15, n = n0 + c;
  const bool mine_out = threadIdx.x < 256 && m < M && n < n1;
  float res = 0.f, wn = 0.f;
  if (mine_out) {
    res = residual[(size_t)m * N + n];
    wn = weight[n];
  }
  f32x4_t acc = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  int fetched = 0;
  for (; fetched < U && fetched < mine; ++fetched) fetch(fetched, fetched);
  const int wr = WR == 8 ? r16 & 7 : r16, ar = AR == 8 ? r16 & 7 : r16;
  int slot = 0;
  for (int i = 0; i < mine; ++i) {
    // as in the few-row product: pair i has landed when at most the U - 1 pairs behind it are on their way
    if (fetched - i == U) QRT_WAIT_LOADS((U - 1) * LOADS);
    else QRT_WAIT_LOADS(0);
    const unsigned char* at = ring + slot * SLOT;
    bf16x8_t w[2], a[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      w[h] = *(const bf16x8_t*)(at + wr * 128 + 16 * ((4 * h + quad) ^ (r16 & 7)));
      a[h] = *(const bf16x8_t*)(at + WL * 1024 + ar * 128 + 16 * ((4 * h + quad) ^ (r16 & 7)));
    }
    QRT_WAIT_LDS();  // the slot is in registers: the next pair may overwrite it
    if (fetched < mine) {
      fetch(fetched, slot);
      ++fetched;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[h], a[h], acc, 0, 0, 0);
    slot = slot + 1 == U ? 0 : slot + 1;
  }
  __syncthreads();  // every wave has read its last slot: the rings' room now takes the partial sums
  float* red = (float*)ring_lds;  // [NW][4][64]
#pragma unroll
  for (int r = 0; r < 4; ++r) red[(wave * 4 + r) * 64 + lane] = acc[r];
  __syncthreads();
  if (threadIdx.x >= 256) return;
  float sum = 0.f;  // the waves' parts in order
#pragma unroll
  for (int w = 0; w < NW; ++w) sum += red[(w * 4 + (c & 3)) * 64 + (c >> 2) * 16 + m];
  float x = 0.f;
  if (mine_out) {
    x = res + sum;
    residual[(size_t)m * N + n] = x;
    out[(size_t)m * N + n] = (bf16_t)(x * wn);
  }
  float square = x * x;
#pragma unroll
  for (int o = 1; o < 16; o *= 2) square += __shfl_xor(square, o, 64);
  if (c == 0 && m < M) squares[(size_t)m * SQUARE_PARTS + blockIdx.x] = square;
}

template <int AR, int WR>
static int launch(const bf16_t* a, const bf16_t* w, float* residual, const float* weight, bf16_t* out, float* squares, int M, int N, int K,
                  hipStream_t stream) {
  constexpr int NW = 8, U = 4;
  constexpr size_t ring = (size_t)NW * U * (AR + WR) * 128, meet = NW * 1024, smem = ring > meet ? ring : meet;
  static_assert(smem <= 160 * 1024, "the rings of this configuration do not fit LDS");
  auto kernel = gemm_residual_kernel<NW, U, AR, WR>;
  static bool allowed = false;  // once per kernel: not inside a stream capture again and again
  if (smem > 64 * 1024 && !allowed) {
    if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess)
      return qrt_fail("gemm_residual: cannot get %zu bytes of LDS", smem);
    allowed = true;
  }
  kernel<<<SQUARE_PARTS, 64 * NW, smem, stream>>>(a, w, M, N, K, residual, weight, out, squares);
  QRT_LAUNCH_CHECK("gemm_residual");
  return 0;
}

// M <= 16 rows, 256 <= N <= 4,096 columns (at most 16 a block), K % 64 == 0, A and W on 16 bytes; squares [M, SQUARE_PARTS].
extern "C" int qrt_gemm_residual_bf16(const void* a, const void* w, float* residual, const float* weight, void* out, float* squares, int M,
                                      int N, int K, hipStream_t stream) {
  QRT_CHECK(M >= 0 && M <= 16 && N >= SQUARE_PARTS && N <= 16 * SQUARE_PARTS && K > 0 && K % 64 == 0,
            "gemm_residual: M=%d N=%d K=%d (up to 16 rows, 256 to 4,096 columns, K in multiples of 64)", M, N, K);
  QRT_CHECK(((uintptr_t)a | (uintptr_t)w) % 16 == 0, "gemm_residual: operands off 16 bytes");
  if (M == 0) return 0;
  const bf16_t *A = (const bf16_t*)a, *W = (const bf16_t*)w;
  bf16_t* o = (bf16_t*)out;
  if (N <= 8 * SQUARE_PARTS)
    return M <= 8 ? launch<8, 8>(A, W, residual, weight, o, squares, M, N, K, stream) : launch<16, 8>(A, W, residual, weight, o, squares, M, N, K, stream);
  return M <= 8 ? launch<8, 16>(A, W, residual, weight, o, squares, M, N, K, stream) : launch<16, 16>(A, W, residual, weight, o, squares, M, N, K, stream);
}
