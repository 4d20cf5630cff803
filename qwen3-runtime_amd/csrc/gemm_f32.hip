// True 32-bit matrix product: C[M, N] = A[M, K] * W[N, K]^T, float32 operands, float32 products and
// sums, no reduced-precision matrix mode (the float32 MFMA multiplies and adds whole float32 numbers).
//
// An output's value depends on neither M nor on which rows share the launch, whichever of the two
// MFMA kernels runs: both walk K in the same order. K is cut into PARTS contiguous parts (a function
// of K alone), within a part 16 k at a time by four MFMAs (MFMA c multiplies k = 4 q + c for q = 0 .. 3),
// and the parts' sums are added from the first to the last.
//
// * few rows (up to 32, or 64): `gemm_f32_rows_kernel` streams the weights. A block owns 16 weight rows, each
//   wave one part of K, and the parts meet in LDS. Bound by the weights' bytes.
// * more rows: `gemm_f32_tile_kernel`, tiles through LDS, bound by the float32 MFMA rate. A wave adds
//   its accumulators into a second set where a part ends.
// * K no multiple of 4 (rows that 16-byte loads cannot read): `gemm_f32_kernel`, one sequential sum
//   of fused multiply-adds per output, as every product had before: 64 x 64 outputs a block, one block per
//   64 weight rows however few the rows of A.
//
// Either MFMA kernel may leave a product for the residual in four planes, the sums of groups of neighbouring parts, or add
// those up itself.
// Error against float64, relative: 3.3e-7 (K 2,560), 4.5e-7 (9,728); the sequential sums': 9.0e-7 and 1.8e-6.
#include "common.h"
#include <type_traits>
#include "direct.h"
#include <limits.h>
#include <algorithm>

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
// For the residual a product may leave four planes that its reader adds, each the sum of a group of
// neighbouring parts (8 or 16 parts, from K 256 on), so that blocks can share K whatever the number of rows.
#define F32_GROUPS 4

__device__ __forceinline__ f32x4_t load_f32x4_below(const float* __restrict__ row, int k, int end) {
  const f32x4_t v = *(const f32x4_t*)(row + (k < end ? k : 0));
  return k < end ? v : f32x4_t{0.f, 0.f, 0.f, 0.f};  // K is a multiple of 4: all four or none
}

// Few rows (up to 64), a stream of the weights. A block owns 16 weight rows (GATED: 8 gate rows and the 8 up rows that
// go with them), each wave one part of K, MB blocks of 16 rows of A. Operands reach LDS by direct loads of 8 rows x 128
// bytes, whole cache lines: lane l fetches piece (l & 7) ^ (l / 8) of row l / 8, so piece c of row r lies at
// 128 r + 16 (c ^ (r & 7)) and the operand reads (row lane & 15, piece 4 h + lane / 16 for the h-th 16 k) touch every bank
// once. A slot of the wave's ring holds 32 k of all units (16 rows x 32 k, 2 KB), U slots are in flight, and the waits on the
// loads' counter are counted by hand. Weights are loaded as data used once. FEW: up to 8 rows of A, whose unit is half as
// long (operand rows 8 to 15 repeat them, and are not stored).
// Loads straight to registers (a lane 16 bytes of its row, sixteen half lines an instruction) made the same products at one row
// in 22, 14, 49, 36 us (4B q/k/v, output, gate/up, down, weights of six layers in turn); this takes 13.8, 9.7, 31.4, 19.9 (4.4 to
// 6.4 TB/s), and at 16 rows 17, 12, 40, 28 instead of 29, 18, 71, 51.
template <int MB, int PARTS, int U, bool FEW, int GATED>
__global__ __launch_bounds__(64 * PARTS) void gemm_f32_rows_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                                   float* __restrict__ C, int M, int N, int K, int part_len, float limit, bool by_groups) {
  constexpr int SLOT = (1 + MB) * 2048 - (FEW ? 1024 : 0), LOADS = 2 + (FEW ? 1 : 2 * MB);
  constexpr int ONCE = 2;  // the cache policy of a non-temporal load
  static_assert(!FEW || MB == 1, "up to 8 rows are one block of rows");
  static_assert((U - 1) * LOADS < 64, "the loads' counter holds 63");
  extern __shared__ __align__(16) unsigned char f32_lds[];  // [PARTS][U] slots, then the parts' sums
  const int lane = threadIdx.x & 63, wave = uniform_wave_number();
  const int r = lane & 15, q = lane >> 4, n0 = blockIdx.x * (GATED ? 8 : 16);
  const int begin = (blockIdx.y * PARTS + wave) * part_len, end = min(K, begin + part_len);
  C += (size_t)blockIdx.y * M * N;
  const int mine = max(0, (end - begin + 31) >> 5);  // slots of this wave
  unsigned char* ring = f32_lds + (size_t)wave * U * SLOT;
  const int sub = lane >> 3, col = 4 * ((lane & 7) ^ sub);
  const float* src[1 + MB][2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    // rows beyond the matrix: its last one, dropped below
    src[0][j] = W + ((size_t)(GATED ? j * N : 0) + min(n0 + (GATED ? 0 : 8 * j) + sub, N - 1)) * K;
#pragma unroll
    for (int b = 0; b < MB; ++b) src[1 + b][j] = A + (size_t)min(16 * b + 8 * j + sub, M - 1) * K;
  }
  auto fetch = [&](int i, int slot) {
    const int k = begin + 32 * i + col, at = k < end ? k : 0;  // K is a multiple of 4: all four or none
    unsigned char* dst = ring + slot * SLOT;
#pragma unroll
    for (int j = 0; j < 2; ++j)
      __builtin_amdgcn_global_load_lds((global_ptr_t)(src[0][j] + at), (lds_ptr_t)(dst + j * 1024), 16, 0, ONCE);
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
      for (int j = 0; j < (FEW ? 1 : 2); ++j)
        __builtin_amdgcn_global_load_lds((global_ptr_t)(src[1 + b][j] + at), (lds_ptr_t)(dst + (1 + b) * 2048 + j * 1024), 16, 0, 0);
  };
  f32x4_t acc[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b) acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  int fetched = 0;
  for (; fetched < U && fetched < mine; ++fetched) fetch(fetched, fetched);
  const int read_at[2] = {r * 128 + 16 * (q ^ (r & 7)), r * 128 + 16 * ((4 + q) ^ (r & 7))};
  const int ra = FEW ? r & 7 : r, a_at[2] = {2048 + ra * 128 + 16 * (q ^ (r & 7)), 2048 + ra * 128 + 16 * ((4 + q) ^ (r & 7))};
  int slot = 0;
  for (int i = 0; i < mine; ++i) {
    // slot i has landed when at most the U - 1 fetched after it are on their way; near the end the wave waits for all
    if (fetched - i == U) QRT_WAIT_LOADS((U - 1) * LOADS);
    else QRT_WAIT_LOADS(0);
    const unsigned char* at = ring + slot * SLOT;
    f32x4_t w[2], a[MB][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      w[h] = *(const f32x4_t*)(at + read_at[h]);
#pragma unroll
      for (int b = 0; b < MB; ++b) a[b][h] = *(const f32x4_t*)(at + b * 2048 + a_at[h]);
    }
    QRT_WAIT_LDS();  // the slot is in registers: the next one may overwrite it
    if (fetched < mine) {
      fetch(fetched, slot);
      ++fetched;
    }
    const int k = begin + 32 * i + 4 * q;
    if (begin + 32 * i + 32 > end)  // the end of K inside a slot: what lies beyond counts as zero
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const bool there = k + 16 * h < end;
        w[h] = there ? w[h] : f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int b = 0; b < MB; ++b) a[b][h] = there ? a[b][h] : f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int b = 0; b < MB; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[h][c], a[b][h][c], acc[b], 0, 0, 0);
    slot = slot + 1 == U ? 0 : slot + 1;
  }
  __syncthreads();  // every wave has read its last slot: the rings' room now takes the parts' sums
  f32x4_t* sums = (f32x4_t*)f32_lds;  // [PARTS][MB][64 lanes]
#pragma unroll
  for (int b = 0; b < MB; ++b) sums[(wave * MB + b) * 64 + lane] = acc[b];
  __syncthreads();
  auto total = [&](int i) {
    if (PARTS >= 2 * F32_GROUPS && by_groups) {  // the whole sum as a reader of the planes adds it
      constexpr int EACH = PARTS >= 2 * F32_GROUPS ? PARTS / F32_GROUPS : 1;
      f32x4_t s;
#pragma unroll
      for (int g = 0; g < F32_GROUPS; ++g) {
        f32x4_t of_group = sums[i + g * EACH * MB * 64];
#pragma unroll
        for (int p = 1; p < EACH; ++p) of_group += sums[i + (g * EACH + p) * MB * 64];
        s = g ? s + of_group : of_group;
      }
      return s;
    }
    f32x4_t s = sums[i];
#pragma unroll
    for (int p = 1; p < PARTS; ++p) s += sums[p * MB * 64 + i];
    return s;
  };
  // an accumulator: rows 4 q .., column r; gated: the gate rows' in lanes 0 to 31, their up rows' in the others
  for (int i = threadIdx.x; i < MB * 64; i += 64 * PARTS) {
    const int m = 16 * (i >> 6) + (i & 15), n = n0 + 4 * ((i & 63) >> 4);
    if (m >= M || (GATED && (i & 32))) continue;
    f32x4_t s = total(i);
    if (GATED) {
      const f32x4_t up = total(i + 32);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = gated_act(s[e], up[e], GATED - 1, limit);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) C[(size_t)m * N + n + e] = s[e];
  }
}

// Tiles of TM x TN outputs, four waves of (TM / 2) x (TN / 2). 32 k of both operands at a time through LDS,
// two stages; the 32 k after the next come into registers during the products. Rows of 40 floats: 32 bytes
// modulo 64, with which operand reads meet no bank twice. The result is all parts, from the first to the last (F32_WHOLE);
// plane blockIdx.z of it, the sum of that group of parts (F32_PLANES); or the sum of all groups, as a reader of the planes
// adds them (F32_GROUPS_SUM).
#define F32_LD 40
enum { F32_WHOLE, F32_PLANES, F32_GROUPS_SUM };
template <int TM_, int TN_, int FORM>
__global__ __launch_bounds__(256) void gemm_f32_tile_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                            float* __restrict__ C, int M, int N, int K, int part_len, int group) {
  constexpr bool PLANES = FORM == F32_PLANES, GROUPS_SUM = FORM == F32_GROUPS_SUM;
  constexpr int BI = TM_ / 32, BJ = TN_ / 32;  // 16 x 16 blocks a wave, rows of A by rows of W
  // square whole tiles move a piece of either operand in turn, the others all of A's and then W's: 64 x 64, 2,560 x 9,728 at
  // 4,096 rows 1,780 us in turn, 1,803 apart; 64 x 32 at 1,024 rows 496 and 487
  constexpr int IN_TURN = !PLANES && BI == BJ ? BI : BI + BJ;
  __shared__ __align__(16) float as[2][TM_ * F32_LD];
  __shared__ __align__(16) float ws[2][TN_ * F32_LD];
  const int lane = threadIdx.x & 63, wave = uniform_wave_number();
  const int r = lane & 15, q = lane >> 4;
  const int m0 = blockIdx.y * TM_, n0 = blockIdx.x * TN_;
  const int wm = (wave >> 1) * (TM_ / 2), wn = (wave & 1) * (TN_ / 2);
  const int lrow = threadIdx.x >> 3, lk = (threadIdx.x & 7) * 4;
  // BI (BJ) pieces of 16 bytes a thread brings per operand and stage
  const float* ar[BI];
  const float* wr[BJ];
#pragma unroll
  for (int i = 0; i < BI; ++i) ar[i] = A + (size_t)min(m0 + lrow + 32 * i, M - 1) * K;
#pragma unroll
  for (int i = 0; i < BJ; ++i) wr[i] = W + (size_t)min(n0 + lrow + 32 * i, N - 1) * K;
  f32x4_t acc[BI][BJ], total[BI][BJ];
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j) acc[i][j] = total[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  f32x4_t of_groups[GROUPS_SUM ? BI : 1][GROUPS_SUM ? BJ : 1];
  f32x4_t ga[2][BI], gw[2][BJ];
  const int per_part = part_len / 32, all = (K + 31) / 32;
  const int s_first = PLANES ? blockIdx.z * group * per_part : 0, stages = PLANES ? min(all, s_first + group * per_part) : all;
  auto fetch = [&](int buf, int s) {
#pragma unroll
    for (int i = 0; i < IN_TURN; ++i) {
      const int j = i - (IN_TURN - BJ);
      if (i < BI) ga[buf][i] = load_f32x4_below(ar[i], 32 * s + lk, K);
      if (j >= 0) gw[buf][j] = load_f32x4_below(wr[j], 32 * s + lk, K);
    }
  };
  int left = per_part, parts_left = group;
  bool first = true, first_group = true;
  auto stage = [&](int buf, int s) {
    float* da = as[buf];
    float* dw = ws[buf];
#pragma unroll
    for (int i = 0; i < IN_TURN; ++i) {
      const int j = i - (IN_TURN - BJ);
      if (i < BI) *(f32x4_t*)(da + (lrow + 32 * i) * F32_LD + lk) = ga[buf][i];
      if (j >= 0) *(f32x4_t*)(dw + (lrow + 32 * j) * F32_LD + lk) = gw[buf][j];
    }
    __syncthreads();  // the stage before last was read before the barrier of the last one: two stages suffice
    // unconditional (under a branch the compiler loses count of the loads in flight and waits for all of
    // them), and held up here (it would move them down to their use): 448 -> 234 us for 354 x 2,560 x 9,728
    fetch(buf, s + 2);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4_t av[BI], wv[BJ];
#pragma unroll
      for (int i = 0; i < IN_TURN; ++i) {
        const int j = i - (IN_TURN - BJ);
        if (i < BI) av[i] = *(const f32x4_t*)(da + (wm + 16 * i + r) * F32_LD + 16 * h + 4 * q);
        if (j >= 0) wv[j] = *(const f32x4_t*)(dw + (wn + 16 * j + r) * F32_LD + 16 * h + 4 * q);
      }
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int i = 0; i < BI; ++i)
#pragma unroll
          for (int j = 0; j < BJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[j][c], av[i][c], acc[i][j], 0, 0, 0);
    }
    // a part of K ends. An odd number of stages is followed by one that counts for nothing (zeros; in planes the next
    // group's first, whose products are dropped)
    if (--left == 0 || (PLANES ? s + 1 >= stages : s + 1 == stages)) {
#pragma unroll
      for (int i = 0; i < BI; ++i)
#pragma unroll
        for (int j = 0; j < BJ; ++j) {
          if (!PLANES || s < stages) total[i][j] = first ? acc[i][j] : total[i][j] + acc[i][j];
          acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
      first = false;
      left = per_part;
      if (GROUPS_SUM && (--parts_left == 0 || s + 1 == stages)) {
#pragma unroll
        for (int i = 0; i < BI; ++i)
#pragma unroll
          for (int j = 0; j < BJ; ++j) {
            f32x4_t& sum = of_groups[GROUPS_SUM ? i : 0][GROUPS_SUM ? j : 0];
            sum = first_group ? total[i][j] : sum + total[i][j];
          }
        first = true;
        first_group = false;
        parts_left = group;
      }
    }
  };
  fetch(0, s_first);
  fetch(1, s_first + 1);
  for (int s = s_first; s < stages; s += 2) {
    stage(0, s);
    stage(1, s + 1);
  }
  if (PLANES) C += (size_t)blockIdx.z * M * N;
#pragma unroll
  for (int i = 0; i < BI; ++i) {
    const int m = m0 + wm + 16 * i + r;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < BJ; ++j) {
      const int n = n0 + wn + 16 * j + 4 * q;
      float* c = C + (size_t)m * N + n;
      const f32x4_t v = GROUPS_SUM ? of_groups[GROUPS_SUM ? i : 0][GROUPS_SUM ? j : 0] : total[i][j];
      if (N % 4 == 0 && n < N) *(f32x4_t*)c = v;
      else
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) c[e] = v[e];
    }
  }
}

// The same tiles, parts and sums (the same bits) where rows are whole stages of 32 k and offsets fit 32 bits: operands come to LDS by direct loads,
// S stages of 32 k in a ring, piece c (16 bytes) of row r at 128 r + 16 (c ^ (r & 7)), so that operand reads meet no bank twice. What bounded
// the kernel above beside its matrix instructions were the others, which do not overlap with them on a SIMD: addresses, a row's end and the way
// through registers were 1.9 vector instructions an MFMA; here a load costs its wave two scalar ones. Blocks of one stretch of
// weight rows follow one another on an XCD, whose L2 then has it for all of them.
#ifdef __HIP_DEVICE_COMPILE__
__device__ __forceinline__ __amdgpu_buffer_rsrc_t f32_buffer(const void* p, unsigned bytes) {
  constexpr int RAW = 0x00020000;  // a buffer of bytes
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)bytes, RAW);
}
#endif
template <int TM_, int TN_, int S, int FORM>
__global__ __launch_bounds__(256) void gemm_f32_ring_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C, int M,
                                                            int N, int K, int part_len, int group, int tiles, int row_tiles) {
#ifdef __HIP_DEVICE_COMPILE__
  constexpr bool PLANES = FORM == F32_PLANES, GROUPS_SUM = FORM == F32_GROUPS_SUM;
  constexpr int BI = TM_ / 32, BJ = TN_ / 32;  // 16 x 16 blocks a wave, and its loads of 8 rows of A and of W a stage
  constexpr int LOADS = BI + BJ, STAGE = (TM_ + TN_) * 128;
  static_assert((S - 1) * LOADS < 64, "the loads' counter holds 63");
  extern __shared__ __align__(16) unsigned char ring[];
  const int per_xcd = (tiles + 7) >> 3, tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (tile >= tiles) return;
  const int lane = threadIdx.x & 63, wave = uniform_wave_number();
  const int r = lane & 15, q = lane >> 4;
  const int m0 = tile % row_tiles * TM_, n0 = tile / row_tiles * TN_;
  const int wm = (wave >> 1) * (TM_ / 2), wn = (wave & 1) * (TN_ / 2);
  const unsigned piece = 16 * ((lane & 7) ^ (lane >> 3));
  const __amdgpu_buffer_rsrc_t a_buf = f32_buffer(A, (unsigned)M * (unsigned)K * 4u), w_buf = f32_buffer(W, (unsigned)N * (unsigned)K * 4u);
  unsigned aoff[BI], woff[BJ];  // rows past the end repeat the last; not stored
#pragma unroll
  for (int i = 0; i < BI; ++i) aoff[i] = (unsigned)min(m0 + 8 * (wave + 4 * i) + (lane >> 3), M - 1) * (unsigned)K * 4u + piece;
#pragma unroll
  for (int j = 0; j < BJ; ++j) woff[j] = (unsigned)min(n0 + 8 * (wave + 4 * j) + (lane >> 3), N - 1) * (unsigned)K * 4u + piece;
  const int per_part = part_len / 32, all = K / 32;
  const int s_first = PLANES ? blockIdx.z * group * per_part : 0, s_end = PLANES ? min(all, s_first + group * per_part) : all;
  const int stages = max(0, s_end - s_first);
  auto fetch = [&](int s, int slot) {
    unsigned char* dst = ring + slot * STAGE + wave * 1024;
#pragma unroll
    for (int i = 0; i < BI; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_buf, (lds_ptr_t)(dst + i * 4096), 16, aoff[i], (s_first + s) * 128, 0, 0);
#pragma unroll
    for (int j = 0; j < BJ; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(w_buf, (lds_ptr_t)(dst + TM_ * 128 + j * 4096), 16, woff[j], (s_first + s) * 128, 0, 0);
  };
  f32x4_t acc[BI][BJ], total[BI][BJ], of_groups[GROUPS_SUM ? BI : 1][GROUPS_SUM ? BJ : 1];
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j) acc[i][j] = total[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  int left = per_part, parts_left = group, slot = 0;
  bool first = true, first_group = true;
#pragma unroll
  for (int s = 0; s < S - 1; ++s)
    if (s < stages) fetch(s, s);
  const unsigned char* a_at = ring + (wm + r) * 128;
  const unsigned char* w_at = ring + (TM_ + wn + r) * 128;
  const int read_at[2] = {16 * (q ^ (r & 7)), 16 * ((4 + q) ^ (r & 7))};
  for (int s = 0; s < stages; ++s) {
    // stage s has landed when at most the S - 2 behind it are on their way; behind the barrier it has for every wave, and
    // every wave has the stage before in registers, whose slot takes the S - 1st from here
    if (s + S - 1 <= stages) QRT_WAIT_LOADS((S - 2) * LOADS);
    else QRT_WAIT_LOADS(0);
    QRT_WAIT_LDS();
    QRT_BARRIER();
    const int free_slot = slot == 0 ? S - 1 : slot - 1;
    if (s + S - 1 < stages) fetch(s + S - 1, free_slot);
    const int base = slot * STAGE;
    f32x4_t av[2][BI], wv[2][BJ];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int i = 0; i < BI; ++i) av[h][i] = *(const f32x4_t*)(a_at + base + i * 2048 + read_at[h]);
#pragma unroll
      for (int j = 0; j < BJ; ++j) wv[h][j] = *(const f32x4_t*)(w_at + base + j * 2048 + read_at[h]);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int i = 0; i < BI; ++i)
#pragma unroll
          for (int j = 0; j < BJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[h][j][c], av[h][i][c], acc[i][j], 0, 0, 0);
    if (--left == 0 || s + 1 == stages) {  // a part of K ends
#pragma unroll
      for (int i = 0; i < BI; ++i)
#pragma unroll
        for (int j = 0; j < BJ; ++j) {
          total[i][j] = first ? acc[i][j] : total[i][j] + acc[i][j];
          acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
      first = false;
      left = per_part;
      if (GROUPS_SUM && (--parts_left == 0 || s + 1 == stages)) {
#pragma unroll
        for (int i = 0; i < BI; ++i)
#pragma unroll
          for (int j = 0; j < BJ; ++j) {
            f32x4_t& sum = of_groups[GROUPS_SUM ? i : 0][GROUPS_SUM ? j : 0];
            sum = first_group ? total[i][j] : sum + total[i][j];
          }
        first = true;
        first_group = false;
        parts_left = group;
      }
    }
    slot = slot + 1 == S ? 0 : slot + 1;
  }
  if (PLANES) C += (size_t)blockIdx.z * M * N;
#pragma unroll
  for (int i = 0; i < BI; ++i) {
    const int m = m0 + wm + 16 * i + r;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < BJ; ++j) {
      const int n = n0 + wn + 16 * j + 4 * q;
      float* c = C + (size_t)m * N + n;
      const f32x4_t v = GROUPS_SUM ? of_groups[GROUPS_SUM ? i : 0][GROUPS_SUM ? j : 0] : total[i][j];
      if (N % 4 == 0 && n < N) *(f32x4_t*)c = v;
      else
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) c[e] = v[e];
    }
  }
#endif
}

// A block's waves: all parts of K, or those of one group (gridDim.y of them, each a plane of the result).
template <int MB, int PARTS, int U, bool FEW, int GATED>
static int f32_rows(const float* a, const float* w, float* c, int M, int N, int K, float limit, hipStream_t stream, bool by_groups, int groups = 1) {
  constexpr size_t smem = (size_t)PARTS * U * ((1 + MB) * 2048 - (FEW ? 1024 : 0));  // the parts' sums fit in it
  static_assert(smem <= 160 * 1024, "the rings of this configuration do not fit LDS");
  auto kernel = gemm_f32_rows_kernel<MB, PARTS, U, FEW, GATED>;
  static bool allowed = false;  // once per kernel: not inside a stream capture again and again
  if (smem > 64 * 1024 && !allowed) {
    if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess)
      return qrt_fail("gemm_f32: cannot get %zu bytes of LDS", smem);
    allowed = true;
  }
  kernel<<<dim3(GATED ? (N + 7) / 8 : (N + 15) / 16, groups), 64 * PARTS, smem, stream>>>(a, w, c, M, N, K, f32_part_len(K, PARTS * groups), limit, by_groups);
  return 0;
}
template <int MB, bool FEW, int GATED>
static int f32_rows_parts(const float* a, const float* w, float* c, int M, int N, int K, float limit, hipStream_t stream, bool by_groups) {
  constexpr int MANY = MB > 1 ? 1 : 2;  // sixteen rings and their slots have to fit LDS
  switch (f32_parts(K)) {
    case 16: return f32_rows<MB, 16, MANY, FEW, GATED>(a, w, c, M, N, K, limit, stream, by_groups);
    case 8: return f32_rows<MB, 8, 2, FEW, GATED>(a, w, c, M, N, K, limit, stream, by_groups);
    case 4: return f32_rows<MB, 4, 2, FEW, GATED>(a, w, c, M, N, K, limit, stream, by_groups);
    case 2: return f32_rows<MB, 2, 2, FEW, GATED>(a, w, c, M, N, K, limit, stream, by_groups);
    default: return f32_rows<MB, 1, 2, FEW, GATED>(a, w, c, M, N, K, limit, stream, by_groups);
  }
}
template <int MB, bool FEW>
static int f32_rows_planes(const float* a, const float* w, float* c, int M, int N, int K, hipStream_t stream) {
  return f32_parts(K) == 16 ? f32_rows<MB, 4, 2, FEW, 0>(a, w, c, M, N, K, 0.f, stream, false, F32_GROUPS)
                            : f32_rows<MB, 2, 2, FEW, 0>(a, w, c, M, N, K, 0.f, stream, false, F32_GROUPS);
}
template <int GATED>
static int f32_few_rows(const float* a, const float* w, float* c, int M, int N, int K, float limit, hipStream_t stream, bool by_groups = false) {
  if constexpr (!GATED)
    if (M > 32) return f32_rows_parts<4, false, 0>(a, w, c, M, N, K, limit, stream, by_groups);
  if (M <= 8) return f32_rows_parts<1, true, GATED>(a, w, c, M, N, K, limit, stream, by_groups);
  if (M <= 16) return f32_rows_parts<1, false, GATED>(a, w, c, M, N, K, limit, stream, by_groups);
  return f32_rows_parts<2, false, GATED>(a, w, c, M, N, K, limit, stream, by_groups);
}

// Which tile: the fewest rounds of blocks over the 256 compute units times what a round takes, us for 32 k: a unit's blocks
// share its matrix cores, so a tile costs its area and little more (113, 107, 98 TFLOP/s of the 157 where rounds are whole, 24,
// 12 and 6 of them), but alone on its unit a block waits for its own loads: no fewer than 1.3, 1.8 and 2.5 rounds' time.
// 4B sizes, us, by 64 x 64, 64 x 32, 32 x 32: q/k/v at 64, 180, 354, 1,024 rows 62 47 42, 101 81 76, 146 131 144, 291 309 340;
// down in planes at 64, 180, 354, 1,024 rows 62 59 49, 97 101 108, 189 195 203, 455 478 521 (whole: 230, 224, 223, 543 by
// 64 x 64). 128 x 128 where that makes four rounds and more, one block to a unit (its two stages are 80 KB of LDS): 6 % less work a
// round, but a round is four times as long. By 64 x 64 and 128 x 128, us: 2,560 x 4,096 at 8,192 rows 1,506 and 1,434, 2,560 x 9,728 3,557 and
// 3,385, 6,144 x 2,560 at 4,096 1,141 and 1,103, 5,120 x 8,192 3,002 and 2,863; 19,456 x 2,560 at 2,048 (9.5 rounds) 1,799 and 1,831, at
// 1,024 (4.75) 906 and 917; 96 x 64 at 2,048 1,854. From 65 to 128 rows they read the weights once: 151,936 x 1,024 at 96 rows 428 and 394.
//
// Where the ring takes the product (f32_ring) a round costs less and its start more; 64 x 64 run four to a unit (two slots), and a lone fifth takes
// longer than a share of four. us, through registers and by the ring, 64 x 64, 64 x 32 and 32 x 32 each, weights of eight layers in turn:
//   19,456 x 2,560 at 128 rows 146 131 144 and 133 118 117, at 354 378 378 391 and 331 318 316 (on another device 336 329 341), at 512 476 480 510
//     and 416 402 412 (418 424 461), at 2,048 1,788 1,884 2,008 and 1,542 1,684 1,691 (132, 121, 121 TFLOP/s);
//   6,144 x 2,560 at 128 61 60 49 and 66 51 42, at 354 146 130 139 and 131 118 105, at 512 147 160 165 and 131 133 136, at 2,048 571 604 639 and
//     496 533 541;
//   2,560 x 9,728 in planes at 128 98 78 70 and 88 66 60, at 354 186 192 193 and 160 162 159, at 512 230 239 256 and 209 202 208, at 2,048
//     889 937 1,003 and 768 842 857.
// A round of n blocks to a unit takes next to the same whatever the sizes, us for 32 k at 1, 2, 3, 4, 5, 8, 16 and 38 rounds: 64 x 64 0.78, 1.17, 1.67,
// 2.13, 2.79, 4.2, 8.2, 19.7; 64 x 32 0.47, 0.62, 0.90, 1.15, 1.49, 2.20, 4.45, 10.4; 32 x 32 0.3, 0.38, 0.53, 0.66, 0.79, 1.23, 2.35, 5.7: the costs below. Over 477
// products, 24 weights of 768 to 19,456 rows at 65 to 2,048 rows, the tile they choose takes 0.4 % longer than the best of the three
// on average. Most where short K or a last round that is half empty counts: 1,024 x 3,072 in planes at 600 rows 43.0, 32 x 32 38.8;
// 5,120 x 5,120 at 480 251 and 232; 3,584 x 18,944 in planes at 101 173, 64 x 32 162.
// 128 x 128 tiles do not pay beside them (19,456 x 2,560 at 2,048 rows 1,918 by a ring, 1,809 through registers). Slots of a ring: two for
// 64 x 64 (four blocks a compute unit in place of three: 1,542 and 1,597), three otherwise; four are slower everywhere (1,673). In sums of groups two
// where a unit's blocks make fewer fours than threes, by two and by three: 2,048 x 768 at 2,048 rows (4 rounds) 56.5 and 70.2, 2,560 x
// 4,096 at 1,300 (4) 265 and 285, 5,120 x 2,048 at 1,300 (7) 238 and 245, 2,560 x 9,728 at 1,300 (4) 623 and 669; else three: at 2,048 (5) 834 and 800, 512 (2) 336 and 329.
static long f32_rounds(int M, int N, int groups, int tm, int tn) { return ((long)((M + tm - 1) / tm) * ((N + tn - 1) / tn) * groups + 255) / 256; }
// A block alone on its unit waits for its stages one after the other, through the ring longer where they come from L2. So weights of up to 4 MB, which may
// be there from the pass before, go through registers where 32 x 32 tiles are no more than the units: us through registers and by the ring from L2 and from
// beyond, 1,024 x 1,024 at 65 rows 10.3, 12.4 and 13.2, 12.7; 256 x 512 at 300 6.5, 7.5 and 7.1, 7.2; 16 x 2,048 at 300 18.3, 24.3 and 23.8, 23.8 (K of 96 and less level or
// better by the ring); 2,048 x 2,048 at 65 18.4, 22.9 and 30.6, 23.8.
static bool f32_ring(int M, int N, int K, int groups) {
  if (K % 32 != 0 || (long)M * K >= 1 << 29 || (long)N * K >= 1 << 29) return false;
  return K < 128 || (long)N * K > 1 << 20 || f32_rounds(M, N, groups, 32, 32) > 1;
}
static long f32_tile_cost(int M, int N, int groups, int tm, int tn, int round, int least) {  // in units of 1 / 100 of 1 / 1000 us
  return std::max(f32_rounds(M, N, groups, tm, tn) * 100, (long)least) * round;
}
static long f32_cost_64x64(int M, int N, int groups, bool ring) {
  if (!ring) return f32_tile_cost(M, N, groups, 64, 64, 606, 130);
  const long rounds = f32_rounds(M, N, groups, 64, 64);
  return 100 * (515 * rounds + (rounds % 4 == 1 ? 280 : 150));
}
static long f32_cost_64x32(int M, int N, int groups, bool ring) {
  return ring ? 100 * std::max(278 * f32_rounds(M, N, groups, 64, 32) + 55, 480l) : f32_tile_cost(M, N, groups, 64, 32, 329, 180);
}
static long f32_cost_32x32(int M, int N, int groups, bool ring) {
  return ring ? 100 * std::max(147 * f32_rounds(M, N, groups, 32, 32) + 62, 340l) : f32_tile_cost(M, N, groups, 32, 32, 190, 250);
}
static long f32_cost_128x128(int M, int N, bool ring) {
  return ring || (long)((M + 127) / 128) * ((N + 127) / 128) < 1024 ? LONG_MAX : f32_tile_cost(M, N, 1, 128, 128, 2324, 0);
}
enum { F32_128x128, F32_64x64, F32_64x32, F32_32x32 };
static int f32_tile_of(int M, int N, int K, int form) {
  const int groups = form == F32_PLANES ? F32_GROUPS : 1;
  const bool ring = f32_ring(M, N, K, groups);
  const long c64 = f32_cost_64x64(M, N, groups, ring), c32 = f32_cost_64x32(M, N, groups, ring), c16 = f32_cost_32x32(M, N, groups, ring);
  if (form != F32_PLANES && f32_cost_128x128(M, N, ring) < (M > 64 && M <= 128 ? LONG_MAX : c64)) return F32_128x128;
  if (form == F32_GROUPS_SUM || (c64 <= c32 && c64 <= c16)) return F32_64x64;
  return c32 <= c16 || (!ring && (M + 31) / 32 > 65535) ? F32_64x32 : F32_32x32;
}
template <int TM_, int TN_, int FORM>
static int f32_tile_launch(const float* a, const float* w, float* c, int M, int N, int K, hipStream_t stream) {
  const int parts = f32_parts(K);
  if constexpr (TM_ < 128)
    if (f32_ring(M, N, K, FORM == F32_PLANES ? F32_GROUPS : 1)) {
      const long tiles = (long)((N + TN_ - 1) / TN_) * ((M + TM_ - 1) / TM_);
      QRT_CHECK(tiles < 1l << 28, "gemm_f32: %ld tiles", tiles);  // a result of 2^38 elements
      auto go = [&](auto slots) {
        constexpr int S = decltype(slots)::value;
        constexpr size_t smem = (size_t)S * (TM_ + TN_) * 128;
        static_assert(smem <= 64 * 1024, "what a block gets without asking");
        gemm_f32_ring_kernel<TM_, TN_, S, FORM><<<dim3((unsigned)((tiles + 7) / 8 * 8), 1, FORM == F32_PLANES ? F32_GROUPS : 1), 256, smem, stream>>>(
            a, w, c, M, N, K, f32_part_len(K, parts), parts / F32_GROUPS, (int)tiles, (M + TM_ - 1) / TM_);
      };
      if constexpr (FORM == F32_GROUPS_SUM) {
        const long rounds = f32_rounds(M, N, 1, TM_, TN_);
        if ((rounds + 3) / 4 < (rounds + 2) / 3) go(std::integral_constant<int, 2>{});
        else go(std::integral_constant<int, 3>{});
      } else go(std::integral_constant<int, TM_ == 64 && TN_ == 64 ? 2 : 3>{});
      return 0;
    }
  gemm_f32_tile_kernel<TM_, TN_, FORM><<<dim3((N + TN_ - 1) / TN_, (M + TM_ - 1) / TM_, FORM == F32_PLANES ? F32_GROUPS : 1), 256, 0, stream>>>(
      a, w, c, M, N, K, f32_part_len(K, parts), parts / F32_GROUPS);
  return 0;
}
template <int FORM>
static int f32_tiles(const float* a, const float* w, float* c, int M, int N, int K, hipStream_t stream) {
  // a grid holds 65,535 rows of tiles: a result of more rows than that many of 64 is made in two calls (planes are of fewer)
  constexpr int MOST = 65535 * 64;
  QRT_CHECK(M <= (FORM == F32_PLANES ? MOST : 2 * MOST), "gemm_f32: M=%d is too large", M);
  if (M > MOST) {
    if (const int rc = f32_tiles<FORM>(a, w, c, MOST, N, K, stream)) return rc;
    a += (size_t)MOST * K, c += (size_t)MOST * N, M -= MOST;
  }
  const int tile = f32_tile_of(M, N, K, FORM);
  if constexpr (FORM != F32_PLANES)
    if (tile == F32_128x128) return f32_tile_launch<128, 128, FORM>(a, w, c, M, N, K, stream);
  if constexpr (FORM != F32_GROUPS_SUM) {
    if (tile == F32_64x32) return f32_tile_launch<64, 32, FORM>(a, w, c, M, N, K, stream);
    if (tile == F32_32x32) return f32_tile_launch<32, 32, FORM>(a, w, c, M, N, K, stream);
  }
  return f32_tile_launch<64, 64, FORM>(a, w, c, M, N, K, stream);
}
// For tests: the tile of a product by tiles, its whole result, its planes or their sum (4, 1 planes; else 0), as rows * 1000 + columns, and
// whether it goes through the ring.
extern "C" int qrt_gemm_f32_tile_of(int M, int N, int K, int planes) {
  const int sizes[] = {128128, 64064, 64032, 32032};
  return sizes[f32_tile_of(M, N, K, planes == 0 ? F32_WHOLE : planes == 1 ? F32_GROUPS_SUM : F32_PLANES)];
}
extern "C" int qrt_gemm_f32_ring_of(int M, int N, int K, int planes) { return f32_ring(M, N, K, planes == F32_GROUPS ? F32_GROUPS : 1); }

extern "C" int qrt_gemm_f32(const float* a, const float* w, float* c, int M, int N, int K, hipStream_t stream) {
  QRT_CHECK(M >= 0 && N > 0 && K > 0, "gemm_f32: bad sizes M=%d N=%d K=%d", M, N, K);
  if (M == 0) return 0;
  const bool wide = K % 4 == 0 && ((uintptr_t)a | (uintptr_t)w | (uintptr_t)c) % 16 == 0;
  if (!wide) {
    dim3 grid((N + TN - 1) / TN, (M + TM - 1) / TM), block(256);
    QRT_CHECK(grid.y <= 65535, "gemm_f32: M=%d is too large for one launch", M);
    gemm_f32_kernel<<<grid, block, 0, stream>>>(a, w, c, M, N, K);
  } else {
    // 33 to 64 rows: tiles of 32 x 32 where they give every compute unit one and a half (4B gate/up 85 us, as a stream 100;
    // q/k/v 42 either way)
    const bool few = M <= 32 || (M <= 64 && (long)((M + 31) / 32) * ((N + 31) / 32) < 384);
    if (const int rc = few ? f32_few_rows<0>(a, w, c, M, N, K, 0.f, stream) : f32_tiles<F32_WHOLE>(a, w, c, M, N, K, stream)) return rc;
  }
  QRT_LAUNCH_CHECK("gemm_f32");
  return 0;
}

// The product for the residual (K in multiples of 4 from 256 on), the groups of K's parts added from the first to the last whatever
// the number of rows: in planes [4, M, N], whose reader adds them, or as their sum [M, N]. Blocks of their own make each plane, which
// fills the chip where the weight has few rows. Up to 32 rows as a stream (4B output and down projections at 1, 16, 32 rows 9.5, 10.4,
// 14.7 and 18.1, 22.9, 31.5 us; all parts in a block 9.7, 12.3, 17.2 and 19.9, 28.1, 40.6), beyond by tiles.
//
// How many planes. By tiles three more of them are written and read, 150 / K of the product's time (of the ring's, which is shorter, 300), so from a
// round of 64 x 64 tiles on they have to save more than that in part-filled rounds (product and norm at 181 sizes of 360 to 2,048 rows by 1,024 to 5,120
// columns: 0.5 % above the best of both forms and all tiles on average, most at 2,048 x 2,048 and 710 rows, 70.9 and 66.3 us). As a stream: where 16 weight rows a block leave compute units idle, under
// 4,096 rows (product and norm, us at 1, 8 and 32 rows, whole and by planes: 2,560 x 4,096 14.4, 14.1, 20.7 and 14.0, 13.9, 19.6; 4,096 x 4,096
// 17.1, 17.5, 22.4 and 17.5, 18.3, 23.9; 8,192 x 4,096 32.0, 32.3, 47.0 and 35.4, 36.2, 55.8; 8,192 x 256 9.0, 9.5, 12.3 and 11.2, 12.3, 16.9).
extern "C" int qrt_gemm_f32_planes_of(int M, int N, int K) {
  if (M <= 32) return N < 4096 ? F32_GROUPS : 1;
  if (N <= 0 || K <= 0 || (long)((M + 63) / 64) * ((N + 63) / 64) < 256) return F32_GROUPS;
  const bool ring = f32_ring(M, N, K, 1);
  const long cut = std::min({f32_cost_64x64(M, N, F32_GROUPS, ring), f32_cost_64x32(M, N, F32_GROUPS, ring), f32_cost_32x32(M, N, F32_GROUPS, ring)}) / F32_GROUPS;
  if (M > 65535 * 64) return 1;  // two calls
  return cut + cut * (ring ? 300 : 150) / K < std::min(f32_cost_64x64(M, N, 1, ring), f32_cost_128x128(M, N, ring)) ? F32_GROUPS : 1;
}
extern "C" int qrt_gemm_f32_planes(const float* a, const float* w, float* c, int M, int N, int K, int planes, hipStream_t stream) {
  QRT_CHECK(M >= 0 && N > 0 && K >= 256 && K % 4 == 0, "gemm_f32_planes: bad sizes M=%d N=%d K=%d", M, N, K);
  QRT_CHECK(planes == F32_GROUPS || planes == 1, "gemm_f32_planes: %d planes", planes);
  QRT_CHECK(((uintptr_t)a | (uintptr_t)w | (uintptr_t)c) % 16 == 0, "gemm_f32_planes: operands are read 16 bytes at a time");
  if (M == 0) return 0;
  if (const int rc = planes == 1 ? (M <= 32 ? f32_few_rows<0>(a, w, c, M, N, K, 0.f, stream, true) : f32_tiles<F32_GROUPS_SUM>(a, w, c, M, N, K, stream))
                     : M <= 8    ? f32_rows_planes<1, true>(a, w, c, M, N, K, stream)
                     : M <= 16   ? f32_rows_planes<1, false>(a, w, c, M, N, K, stream)
                     : M <= 32   ? f32_rows_planes<2, false>(a, w, c, M, N, K, stream)
                                 : f32_tiles<F32_PLANES>(a, w, c, M, N, K, stream))
    return rc;
  QRT_LAUNCH_CHECK("gemm_f32_planes");
  return 0;
}

// The gated product of few rows: W is [2N, K] (gate rows, then up rows), C[M, N] = act(A Wg^T, A Wu^T) as gated_act makes it
// of the product's columns, with the same bits.
extern "C" int qrt_gated_gemm_f32(const float* a, const float* w, float* c, int M, int N, int K, int act_kind, float limit,
                                  hipStream_t stream) {
  QRT_CHECK(M >= 0 && M <= 32 && N > 0 && N <= 1 << 30 && K > 0, "gated_gemm_f32: bad sizes M=%d N=%d K=%d", M, N, K);
  QRT_CHECK(act_kind == QRT_ACT_SWIGLU || act_kind == QRT_ACT_CLAMPED, "gated_gemm_f32: unknown activation %d", act_kind);
  QRT_CHECK(K % 4 == 0 && ((uintptr_t)a | (uintptr_t)w) % 16 == 0, "gated_gemm_f32: operands are read 16 bytes at a time (K=%d)", K);
  if (M == 0) return 0;
  const int rc = act_kind == QRT_ACT_SWIGLU ? f32_few_rows<1 + QRT_ACT_SWIGLU>(a, w, c, M, N, K, limit, stream)
                                            : f32_few_rows<1 + QRT_ACT_CLAMPED>(a, w, c, M, N, K, limit, stream);
  if (rc) return rc;
  QRT_LAUNCH_CHECK("gated_gemm_f32");
  return 0;
}
