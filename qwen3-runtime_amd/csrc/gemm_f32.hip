// True 32-bit matrix product: C[M, N] = A[M, K] * W[N, K]^T, float32 operands, float32 products and
// sums, no reduced-precision matrix mode (the float32 MFMA multiplies and adds whole float32 numbers).
//
// An output's value depends on neither M nor on which rows share the launch, whichever of the two
// MFMA kernels runs: both walk K in the same order. K is cut into PARTS contiguous parts (a function
// of K alone), within a part 16 k at a time by four MFMAs (MFMA c multiplies k = 4 q + c for q = 0 .. 3),
// and the parts' sums are added from the first to the last.
//
// * few rows (up to 64): `gemm_f32_rows_kernel` streams the weights. A block owns 16 weight rows, each
//   wave one part of K, and the parts meet in LDS. Bound by the weights' bytes.
// * more rows: `gemm_f32_tile_kernel`, tiles through LDS, bound by the float32 MFMA rate. A wave adds
//   its accumulators into a second set where a part ends.
// * K no multiple of 4 (rows that 16-byte loads cannot read): `gemm_f32_kernel`, one sequential sum
//   of fused multiply-adds per output, as every product had before: 64 x 64 outputs a block, one block per
//   64 weight rows however few the rows of A.
//
// Measured (MI355X, us; the 4B products q/k/v, output, gate/up, down; weights of six layers in turn). One row: 22, 14,
// 49, 36 (2.8 to 4.1 TB/s) against 262, 409, 326, 994 by the sequential kernel. 354 rows: 151, 98, 392, 235 (74 to 90
// TFLOP/s of 157) against 472, 443, 1,112, 1,080. Error against float64, relative: 3.3e-7 (K 2,560), 4.5e-7 (9,728); the
// sequential sums': 9.0e-7 and 1.8e-6.
#include "common.h"

#define TM 64
#define TN 64
#define TK 16

__global__ __launch_bounds__(256) void gemm_f32_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                        float* __restrict__ C, int M, int N, int K) {
  __shared__ float As[TK][TM + 4];
  __shared__ float Ws[TK][TN + 4];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;

  // loader: 256 threads bring 64 rows x 16 k of each operand; thread -> (row, 4 k)
  const int lrow = threadIdx.x >> 2, lk = (threadIdx.x & 3) * 4;
  for (int k0 = 0; k0 < K; k0 += TK) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int k = k0 + lk + e;
      const int am = m0 + lrow, wn = n0 + lrow;
      As[lk + e][lrow] = (am < M && k < K) ? A[(size_t)am * K + k] : 0.f;
      Ws[lk + e][lrow] = (wn < N && k < K) ? W[(size_t)wn * K + k] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < TK; ++kk) {
      float a[4], w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = Ws[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], w[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty * 4 + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n < N) C[(size_t)m * N + n] = acc[i][j];
    }
  }
}

// ------------------------------------------------------------ the MFMA kernels
// Parts of K (waves a block of the few-row kernel) and the length of one: more parts for a longer K, so
// that 160 blocks (the 2,560 rows of a 4B down projection) still keep enough loads in flight, and parts
// for a short one too, since a sum's error grows with the length of its chain: relative to float64 2.0e-7 in one
// chain and 1.1e-7 in four parts at K 128, 4.1e-7 and 1.6e-7 at 512 (equal up to 32, where there is one part).
static inline int f32_parts(int K) { return K >= 8192 ? 16 : K >= 256 ? 8 : K > 64 ? 4 : K > 32 ? 2 : 1; }
static inline int f32_part_len(int K, int parts) { return ((K + parts - 1) / parts + 31) / 32 * 32; }

__device__ __forceinline__ f32x4_t load_f32x4_below(const float* __restrict__ row, int k, int end) {
  const f32x4_t v = *(const f32x4_t*)(row + (k < end ? k : 0));
  return k < end ? v : f32x4_t{0.f, 0.f, 0.f, 0.f};  // K is a multiple of 4: all four or none
}

// 16 weight rows a block, PARTS waves of one part of K each, MB blocks of 16 rows of A. A lane holds
// weight row lane & 15 and, of 16 k, the four from 4 (lane >> 4) on: one 16-byte load feeds four MFMAs,
// and 64 k of a row are two whole cache lines.
template <int MB, int PARTS>
__global__ __launch_bounds__(64 * PARTS) void gemm_f32_rows_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                                   float* __restrict__ C, int M, int N, int K, int part_len) {
  extern __shared__ __align__(16) float sums[];  // [PARTS][MB][64 lanes][4]
  const int lane = threadIdx.x & 63, wave = uniform_wave_number();
  const int r = lane & 15, q = lane >> 4, n0 = blockIdx.x * 16;
  const int begin = wave * part_len, end = min(K, begin + part_len);
  const float* w = W + (size_t)min(n0 + r, N - 1) * K;  // rows beyond the matrix: its last one, dropped below
  const float* a[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b) a[b] = A + (size_t)min(16 * b + r, M - 1) * K;
  f32x4_t acc[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b) acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // 64 k a round, all of its loads asked for at once; what hides their latency is the number of waves (asking
  // for the next round's before this one's are multiplied costs as many registers and gains nothing:
  // 26.7 us against 21.6 for the 4B q/k/v weights and one row)
  auto round = [&](int at, bool whole) {
    f32x4_t wv[4], av[4][MB];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = at + 16 * u + 4 * q, from = whole || k < end ? k : 0;  // K is a multiple of 4: all four or none
      wv[u] = __builtin_nontemporal_load((const f32x4_t*)(w + from));
#pragma unroll
      for (int b = 0; b < MB; ++b) av[u][b] = *(const f32x4_t*)(a[b] + from);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool there = whole || at + 16 * u + 4 * q < end;
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int b = 0; b < MB; ++b)
          acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(there ? wv[u][c] : 0.f, there ? av[u][b][c] : 0.f, acc[b], 0, 0, 0);
    }
  };
  int at = begin;
  for (; at + 64 <= end; at += 64) round(at, true);
  if (at < end) round(at, false);
  f32x4_t* mine = (f32x4_t*)sums + ((size_t)wave * MB) * 64 + lane;
#pragma unroll
  for (int b = 0; b < MB; ++b) mine[b * 64] = acc[b];
  __syncthreads();
  for (int i = threadIdx.x; i < MB * 64; i += 64 * PARTS) {
    f32x4_t s = ((const f32x4_t*)sums)[i];
#pragma unroll
    for (int p = 1; p < PARTS; ++p) s += ((const f32x4_t*)sums)[p * MB * 64 + i];
    const int m = 16 * (i >> 6) + (i & 15), n = n0 + 4 * ((i & 63) >> 4);  // an accumulator: rows 4 q .., column r
    if (m >= M) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) C[(size_t)m * N + n + e] = s[e];
  }
}

// Tiles of T x T outputs, four waves of (T / 2) x (T / 2). 32 k of both operands at a time through LDS,
// two stages; the 32 k after the next come into registers during the products. Rows of 40 floats: 32 bytes
// modulo 64, with which operand reads meet no bank twice.
#define F32_LD 40
template <int T>
__global__ __launch_bounds__(256) void gemm_f32_tile_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                            float* __restrict__ C, int M, int N, int K, int part_len) {
  constexpr int B = T / 32;   // 16 x 16 blocks a wave and direction
  constexpr int L = T / 32;   // 16-byte pieces a thread brings per operand and stage
  __shared__ __align__(16) float as[2][T * F32_LD];
  __shared__ __align__(16) float ws[2][T * F32_LD];
  const int lane = threadIdx.x & 63, wave = uniform_wave_number();
  const int r = lane & 15, q = lane >> 4;
  const int m0 = blockIdx.y * T, n0 = blockIdx.x * T;
  const int wm = (wave >> 1) * (T / 2), wn = (wave & 1) * (T / 2);
  const int lrow = threadIdx.x >> 3, lk = (threadIdx.x & 7) * 4;
  const float* ar[L];
  const float* wr[L];
#pragma unroll
  for (int i = 0; i < L; ++i) {
    ar[i] = A + (size_t)min(m0 + lrow + 32 * i, M - 1) * K;
    wr[i] = W + (size_t)min(n0 + lrow + 32 * i, N - 1) * K;
  }
  f32x4_t acc[B][B], total[B][B];
#pragma unroll
  for (int i = 0; i < B; ++i)
#pragma unroll
    for (int j = 0; j < B; ++j) acc[i][j] = total[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  f32x4_t ga[2][L], gw[2][L];
  const int stages = (K + 31) / 32, per_part = part_len / 32;
  auto fetch = [&](int buf, int s) {
#pragma unroll
    for (int i = 0; i < L; ++i) {
      ga[buf][i] = load_f32x4_below(ar[i], 32 * s + lk, K);
      gw[buf][i] = load_f32x4_below(wr[i], 32 * s + lk, K);
    }
  };
  int left = per_part;
  bool first = true;
  auto stage = [&](int buf, int s) {
    float* da = as[buf];
    float* dw = ws[buf];
#pragma unroll
    for (int i = 0; i < L; ++i) {
      *(f32x4_t*)(da + (lrow + 32 * i) * F32_LD + lk) = ga[buf][i];
      *(f32x4_t*)(dw + (lrow + 32 * i) * F32_LD + lk) = gw[buf][i];
    }
    __syncthreads();  // the stage before last was read before the barrier of the last one: two stages suffice
    // unconditional (under a branch the compiler loses count of the loads in flight and waits for all of
    // them), and held up here (it would move them down to their use): 448 -> 234 us for 354 x 2,560 x 9,728
    fetch(buf, s + 2);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4_t av[B], wv[B];
#pragma unroll
      for (int i = 0; i < B; ++i) {
        av[i] = *(const f32x4_t*)(da + (wm + 16 * i + r) * F32_LD + 16 * h + 4 * q);
        wv[i] = *(const f32x4_t*)(dw + (wn + 16 * i + r) * F32_LD + 16 * h + 4 * q);
      }
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int i = 0; i < B; ++i)
#pragma unroll
          for (int j = 0; j < B; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[j][c], av[i][c], acc[i][j], 0, 0, 0);
    }
    if (--left == 0 || s + 1 == stages) {  // a part of K ends (sums of nothing but zeros may follow the last)
#pragma unroll
      for (int i = 0; i < B; ++i)
#pragma unroll
        for (int j = 0; j < B; ++j) {
          total[i][j] = first ? acc[i][j] : total[i][j] + acc[i][j];
          acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
      first = false;
      left = per_part;
    }
  };
  fetch(0, 0);
  fetch(1, 1);
  for (int s = 0; s < stages; s += 2) {  // an odd number of stages ends with one of zeros
    stage(0, s);
    stage(1, s + 1);
  }
#pragma unroll
  for (int i = 0; i < B; ++i) {
    const int m = m0 + wm + 16 * i + r;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < B; ++j) {
      const int n = n0 + wn + 16 * j + 4 * q;
      float* c = C + (size_t)m * N + n;
      if (N % 4 == 0 && n < N) *(f32x4_t*)c = total[i][j];
      else
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) c[e] = total[i][j][e];
    }
  }
}

template <int MB, int PARTS>
static void f32_rows(const float* a, const float* w, float* c, int M, int N, int K, hipStream_t stream) {
  gemm_f32_rows_kernel<MB, PARTS><<<(N + 15) / 16, 64 * PARTS, (size_t)PARTS * MB * 64 * 16, stream>>>(a, w, c, M, N, K, f32_part_len(K, PARTS));
}
template <int MB>
static void f32_rows_parts(const float* a, const float* w, float* c, int M, int N, int K, hipStream_t stream) {
  switch (f32_parts(K)) {
    case 16: return f32_rows<MB, 16>(a, w, c, M, N, K, stream);
    case 8: return f32_rows<MB, 8>(a, w, c, M, N, K, stream);
    case 4: return f32_rows<MB, 4>(a, w, c, M, N, K, stream);
    case 2: return f32_rows<MB, 2>(a, w, c, M, N, K, stream);
    default: return f32_rows<MB, 1>(a, w, c, M, N, K, stream);
  }
}

extern "C" int qrt_gemm_f32(const float* a, const float* w, float* c, int M, int N, int K, hipStream_t stream) {
  QRT_CHECK(M >= 0 && N > 0 && K > 0, "gemm_f32: bad sizes M=%d N=%d K=%d", M, N, K);
  if (M == 0) return 0;
  const bool wide = K % 4 == 0 && ((uintptr_t)a | (uintptr_t)w | (uintptr_t)c) % 16 == 0;
  if (!wide) {
    dim3 grid((N + TN - 1) / TN, (M + TM - 1) / TM), block(256);
    QRT_CHECK(grid.y <= 65535, "gemm_f32: M=%d is too large for one launch", M);
    gemm_f32_kernel<<<grid, block, 0, stream>>>(a, w, c, M, N, K);
  } else if (M <= 16) {
    f32_rows_parts<1>(a, w, c, M, N, K, stream);
  } else if (M <= 32) {
    f32_rows_parts<2>(a, w, c, M, N, K, stream);
  } else if (M <= 64) {
    f32_rows_parts<4>(a, w, c, M, N, K, stream);
  } else {
    // tiles of 128 only where they fill the 256 compute units several times: 2,048 x 2,560 x 9,728 is 320 of them, two
    // rounds for 1.25, 2,090 us; in 1,280 tiles of 64 it takes 946
    const int part_len = f32_part_len(K, f32_parts(K));
    const int t = (long)((N + 127) / 128) * ((M + 127) / 128) >= 1024 ? 128 : 64;
    dim3 grid((N + t - 1) / t, (M + t - 1) / t);
    QRT_CHECK(grid.y <= 65535, "gemm_f32: M=%d is too large for one launch", M);
    if (t == 128) gemm_f32_tile_kernel<128><<<grid, 256, 0, stream>>>(a, w, c, M, N, K, part_len);
    else gemm_f32_tile_kernel<64><<<grid, 256, 0, stream>>>(a, w, c, M, N, K, part_len);
  }
  QRT_LAUNCH_CHECK("gemm_f32");
  return 0;
}
