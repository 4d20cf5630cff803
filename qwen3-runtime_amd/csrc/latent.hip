// Steps of attention through a latent, each over packed tokens:
//
// * the RMS norm of some columns of a wider matrix (a latent that a fused product left beside
//   other things), float32 inside, out in the matrix's type;
// * the write of the cached row: columns [first, first + rank) RMS-normed are the latent c, the
//   rot_dim columns behind them, rotated, the key part all heads share; the key row of the one
//   key/value head is [c | k_rot], its value row [c | 0] (keys [page, 1, offset, W], values
//   [page, 1, W, offset], W = rank + rot_dim);
// * a copy of `width` elements per (token, head) from one strided layout to another with the
//   first 2 n of them turned, element i against element i + n (the "rotate half" layout), or,
//   with `neighbours`, element 2i against element 2i + 1, by position * freq[i] (angles, sines
//   and cosines float32; sines and cosines times `magnitude`); the cached row's rotated part
//   takes the same two options;
// * a product per head, out[t, h, :] = W[h] x[t, h, :], on strided rows: W [heads, N, K].
#include "common.h"
#include "direct.h"
#include <math.h>

// Element i of a vector whose first 2 `pairs` elements turn: its partner and the pair's number.
// Half layout: i against i + pairs; neighbours: 2j against 2j + 1. `first` says whether i is the
// pair's first element (x cos - other sin) or its second (x cos + other sin).
__device__ __forceinline__ void rotation_partner(int i, int pairs, int neighbours, int* pair, int* other, bool* first) {
  if (neighbours) {
    *pair = i >> 1;
    *first = (i & 1) == 0;
    *other = i ^ 1;
  } else {
    *first = i < pairs;
    *pair = *first ? i : i - pairs;
    *other = *first ? i + pairs : i - pairs;
  }
}

// ---------------------------------------------------------------- norm of some columns
template <typename T>
__global__ __launch_bounds__(256) void rmsnorm_columns_kernel(const T* __restrict__ y, long stride, int first, int width,
                                                              const float* __restrict__ weight, float eps,
                                                              T* __restrict__ out) {
  __shared__ float red[32];
  const T* row = y + (size_t)blockIdx.x * stride + first;
  float ss = 0.f;
  for (int i = threadIdx.x; i < width; i += 256) {
    const float v = to_f32<T>(row[i]);
    ss += v * v;
  }
  ss = block_sum(ss, red);
  const float inv = 1.0f / sqrtf(ss / (float)width + eps);
  for (int i = threadIdx.x; i < width; i += 256)
    out[(size_t)blockIdx.x * width + i] = from_f32<T>(to_f32<T>(row[i]) * inv * weight[i]);
}

extern "C" int qrt_rmsnorm_columns(const void* y, long stride, int first, int width, const float* weight, float eps,
                                   void* out, int dtype, int num_tokens, hipStream_t stream) {
  QRT_CHECK(num_tokens >= 0 && width > 0 && first >= 0 && (long)first + width <= stride, "rmsnorm_columns: bad sizes");
  if (num_tokens == 0) return 0;
  if (dtype == QRT_F32)
    rmsnorm_columns_kernel<float><<<num_tokens, 256, 0, stream>>>((const float*)y, stride, first, width, weight, eps, (float*)out);
  else if (dtype == QRT_BF16)
    rmsnorm_columns_kernel<bf16_t><<<num_tokens, 256, 0, stream>>>((const bf16_t*)y, stride, first, width, weight, eps, (bf16_t*)out);
  else return qrt_fail("rmsnorm_columns: unknown dtype %d", dtype);
  QRT_LAUNCH_CHECK("rmsnorm_columns");
  return 0;
}

// ---------------------------------------------------------------- the cached row
template <typename T>
__global__ __launch_bounds__(256) void latent_store_kernel(const T* __restrict__ y, long stride, int first, int rank,
                                                           int rot_dim, const float* __restrict__ weight, float eps,
                                                           const int* __restrict__ positions, const float* __restrict__ freq,
                                                           int pairs, const int* __restrict__ slots, T* __restrict__ k_cache,
                                                           T* __restrict__ v_cache, int page_size, int neighbours,
                                                           float magnitude) {
  __shared__ float red[32];
  const int t = blockIdx.x;
  const T* row = y + (size_t)t * stride + first;
  const int slot = slots[t];
  const int page = slot / page_size, off = slot - page * page_size;
  const int w = rank + rot_dim;
  T* kr = k_cache + (size_t)slot * w;
  T* vr = v_cache + (size_t)page * w * page_size + off;
  float ss = 0.f;
  for (int i = threadIdx.x; i < rank; i += 256) {
    const float v = to_f32<T>(row[i]);
    ss += v * v;
  }
  ss = block_sum(ss, red);
  const float inv = 1.0f / sqrtf(ss / (float)rank + eps);
  for (int i = threadIdx.x; i < rank; i += 256) {
    const T c = from_f32<T>(to_f32<T>(row[i]) * inv * weight[i]);
    kr[i] = c;
    vr[(size_t)i * page_size] = c;
  }
  const float pos = (float)positions[t];
  const T* rot = row + rank;
  for (int i = threadIdx.x; i < rot_dim; i += 256) {
    float x = to_f32<T>(rot[i]);
    if (i < 2 * pairs) {
      int j, o;
      bool first;
      rotation_partner(i, pairs, neighbours, &j, &o, &first);
      float sn, cs;
      sincos_angle(pos * freq[j], &sn, &cs);
      sn *= magnitude;
      cs *= magnitude;
      const float other = to_f32<T>(rot[o]);
      x = first ? x * cs - other * sn : x * cs + other * sn;
    }
    kr[rank + i] = from_f32<T>(x);
    vr[(size_t)(rank + i) * page_size] = from_f32<T>(0.f);
  }
}

extern "C" int qrt_latent_store(const void* y, long stride, int first, int rank, int rot_dim, const float* weight, float eps,
                                const int* positions, const float* freq, int pairs, const int* slots, void* k_cache,
                                void* v_cache, int page_size, long num_pages, int dtype, int num_tokens, int neighbours,
                                float magnitude, hipStream_t stream) {
  QRT_CHECK(num_tokens >= 0 && rank > 0 && rot_dim >= 0 && first >= 0 && (long)first + rank + rot_dim <= stride,
            "latent_store: bad sizes");
  QRT_CHECK(pairs >= 0 && 2 * pairs <= rot_dim && (pairs == 0 || freq), "latent_store: %d pairs in %d elements", pairs, rot_dim);
  QRT_CHECK(page_size > 0 && num_pages > 0 && slots && positions, "latent_store: no cache");
  if (num_tokens == 0) return 0;
  if (dtype == QRT_F32)
    latent_store_kernel<float><<<num_tokens, 256, 0, stream>>>((const float*)y, stride, first, rank, rot_dim, weight, eps, positions,
                                                               freq, pairs, slots, (float*)k_cache, (float*)v_cache, page_size, neighbours, magnitude);
  else if (dtype == QRT_BF16)
    latent_store_kernel<bf16_t><<<num_tokens, 256, 0, stream>>>((const bf16_t*)y, stride, first, rank, rot_dim, weight, eps, positions,
                                                                freq, pairs, slots, (bf16_t*)k_cache, (bf16_t*)v_cache, page_size, neighbours, magnitude);
  else return qrt_fail("latent_store: unknown dtype %d", dtype);
  QRT_LAUNCH_CHECK("latent_store");
  return 0;
}

// ---------------------------------------------------------------- rotate half, from one layout to another
struct RotateArgs {
  const void* x; long x_row; int in_stride, in_offset;
  void* out; long out_row; int out_stride, out_offset;
  int heads, width, pairs;
  const int* positions; const float* freq;
  int scale_from_head; float scale;  // heads from this one on are multiplied by `scale` after turning
  int neighbours; float magnitude;   // pairs of neighbours instead of halves; what multiplies sines and cosines
};

template <typename TI, typename TO>
__global__ __launch_bounds__(256) void rotate_half_kernel(RotateArgs a) {
  const int t = blockIdx.x;
  const float pos = a.pairs ? (float)a.positions[t] : 0.f;
  const TI* xr = (const TI*)a.x + (size_t)t * a.x_row + a.in_offset;
  TO* orow = (TO*)a.out + (size_t)t * a.out_row + a.out_offset;
  const int total = a.heads * a.width;
  for (int e = blockIdx.y * 256 + threadIdx.x; e < total; e += 256 * gridDim.y) {
    const int h = e / a.width, i = e - h * a.width;
    const TI* src = xr + (size_t)h * a.in_stride;
    float x = to_f32<TI>(src[i]);
    if (i < 2 * a.pairs) {
      int j, o;
      bool first;
      rotation_partner(i, a.pairs, a.neighbours, &j, &o, &first);
      float sn, cs;
      sincos_angle(pos * a.freq[j], &sn, &cs);
      sn *= a.magnitude;
      cs *= a.magnitude;
      const float other = to_f32<TI>(src[o]);
      x = first ? x * cs - other * sn : x * cs + other * sn;
    }
    if (h >= a.scale_from_head) x *= a.scale;
    orow[(size_t)h * a.out_stride + i] = from_f32<TO>(x);
  }
}

// The rotation of halves by pieces of 8 elements, a token's sines and cosines made once for all its heads (the kernel
// above makes them for every element, in float64 up to the reduced angle, which is what it takes its time for): 2,047
// tokens, 64 heads of 128 into float32 44 -> 19 us. A few tokens of which little turns are spread wider by the kernel above
// (8 tokens, 32 heads of 192, 64 of them turned: 2.5 us there, 3.1 here).
#define ROTATE_MAX_PAIRS 512
template <typename TI, typename TO>
__global__ __launch_bounds__(256) void rotate_half_wide_kernel(RotateArgs a) {
  typedef TI ivec_t __attribute__((ext_vector_type(8), aligned(16)));
  typedef TO ovec_t __attribute__((ext_vector_type(8), aligned(16)));
  __shared__ float cosines[ROTATE_MAX_PAIRS], sines[ROTATE_MAX_PAIRS];
  const int t = blockIdx.x;
  if (a.pairs) {
    const float pos = (float)a.positions[t];
    for (int j = threadIdx.x; j < a.pairs; j += 256) {
      float sn, cs;
      sincos_angle(pos * a.freq[j], &sn, &cs);
      sines[j] = sn * a.magnitude;
      cosines[j] = cs * a.magnitude;
    }
    __syncthreads();
  }
  const TI* xr = (const TI*)a.x + (size_t)t * a.x_row + a.in_offset;
  TO* orow = (TO*)a.out + (size_t)t * a.out_row + a.out_offset;
  const int turning = a.pairs / 8, per_head = a.width / 8 - turning, total = a.heads * per_head;
  for (int e = blockIdx.y * 256 + threadIdx.x; e < total; e += 256 * gridDim.y) {
    const int h = e / per_head, c = e - h * per_head;
    const TI* src = xr + (size_t)h * a.in_stride;
    TO* dst = orow + (size_t)h * a.out_stride;
    const float by = h >= a.scale_from_head ? a.scale : 1.0f;
    if (c < turning) {
      const ivec_t u = *(const ivec_t*)(src + 8 * c), v = *(const ivec_t*)(src + 8 * c + a.pairs);
      ovec_t p, q;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float x = to_f32<TI>(u[k]), y = to_f32<TI>(v[k]), cs = cosines[8 * c + k], sn = sines[8 * c + k];
        p[k] = from_f32<TO>((x * cs - y * sn) * by);
        q[k] = from_f32<TO>((y * cs + x * sn) * by);
      }
      *(ovec_t*)(dst + 8 * c) = p;
      *(ovec_t*)(dst + 8 * c + a.pairs) = q;
    } else {
      const int i = 8 * (turning + c);  // the pairs' second halves lie between
      const ivec_t u = *(const ivec_t*)(src + i);
      ovec_t p;
#pragma unroll
      for (int k = 0; k < 8; ++k) p[k] = from_f32<TO>(to_f32<TI>(u[k]) * by);
      *(ovec_t*)(dst + i) = p;
    }
  }
}

extern "C" int qrt_rotate_half(const RotateArgs* args, int in_dtype, int out_dtype, int num_tokens, hipStream_t stream) {
  RotateArgs a = *args;
  QRT_CHECK(num_tokens >= 0 && a.heads > 0 && a.width > 0 && a.pairs >= 0 && 2 * a.pairs <= a.width, "rotate_half: bad sizes");
  QRT_CHECK(a.in_offset >= 0 && a.in_offset + a.width <= a.in_stride && (long)a.heads * a.in_stride <= a.x_row &&
            a.out_offset >= 0 && a.out_offset + a.width <= a.out_stride && (long)a.heads * a.out_stride <= a.out_row,
            "rotate_half: heads of %d at %d in rows of %ld, to heads of %d at %d in rows of %ld", a.in_stride, a.in_offset,
            a.x_row, a.out_stride, a.out_offset, a.out_row);
  QRT_CHECK(a.pairs == 0 || (a.freq && a.positions), "rotate_half: no angles");
  if (num_tokens == 0) return 0;
  const int total = a.heads * a.width;
  const dim3 grid(num_tokens, num_tokens >= 512 ? 1 : min((total + 255) / 256, 64));
  const bool pieces = !a.neighbours && a.pairs <= ROTATE_MAX_PAIRS && (num_tokens > 8 || 2 * a.pairs == a.width) &&
                      (a.pairs | a.width | a.in_stride | a.in_offset | a.out_stride | a.out_offset) % 8 == 0 &&
                      a.x_row % 8 == 0 && a.out_row % 8 == 0 && ((uintptr_t)a.x | (uintptr_t)a.out) % 16 == 0;
  if (pieces && in_dtype <= QRT_BF16 && out_dtype <= QRT_BF16 && !(in_dtype == QRT_F32 && out_dtype == QRT_BF16)) {
    const dim3 wide(num_tokens, num_tokens >= 512 ? 1 : min((total / 8 + 255) / 256, 64));
    if (in_dtype == QRT_F32) rotate_half_wide_kernel<float, float><<<wide, 256, 0, stream>>>(a);
    else if (out_dtype == QRT_BF16) rotate_half_wide_kernel<bf16_t, bf16_t><<<wide, 256, 0, stream>>>(a);
    else rotate_half_wide_kernel<bf16_t, float><<<wide, 256, 0, stream>>>(a);
  } else if (in_dtype == QRT_F32 && out_dtype == QRT_F32) rotate_half_kernel<float, float><<<grid, 256, 0, stream>>>(a);
  else if (in_dtype == QRT_BF16 && out_dtype == QRT_BF16) rotate_half_kernel<bf16_t, bf16_t><<<grid, 256, 0, stream>>>(a);
  else if (in_dtype == QRT_BF16 && out_dtype == QRT_F32) rotate_half_kernel<bf16_t, float><<<grid, 256, 0, stream>>>(a);
  else return qrt_fail("rotate_half: no form for types %d -> %d", in_dtype, out_dtype);
  QRT_LAUNCH_CHECK("rotate_half");
  return 0;
}

// ---------------------------------------------------------------- a product per head
// One block of four waves per (token, head): the head's input in LDS as float32, each wave takes
// outputs wave, wave + 4, ...; an output is one wave's sum over K in a fixed order, whatever else is
// in the batch. For float32 (few tokens: the kernel below).
template <typename T>
__global__ __launch_bounds__(256) void heads_linear_kernel(const T* __restrict__ x, long x_row, int in_stride, int in_offset,
                                                           const T* __restrict__ w, int n, int k, T* __restrict__ out,
                                                           long out_row, int out_stride, int out_offset) {
  extern __shared__ float xs[];
  const int t = blockIdx.x, h = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const T* xr = x + (size_t)t * x_row + (size_t)h * in_stride + in_offset;
  for (int i = threadIdx.x; i < k; i += 256) xs[i] = to_f32<T>(xr[i]);
  __syncthreads();
  const T* wh = w + (size_t)h * n * k;
  T* o = out + (size_t)t * out_row + (size_t)h * out_stride + out_offset;
  for (int j = wave; j < n; j += 4) {
    const T* wr = wh + (size_t)j * k;
    float acc = 0.f;
    for (int c = lane; c < k; c += 64) acc = fmaf(xs[c], to_f32<T>(wr[c]), acc);
    acc = wave_sum(acc);
    if (lane == 0) o[j] = from_f32<T>(acc);
  }
}

// Few tokens: one block per (64 outputs of a head), all tokens of the step at once, so that the
// head's weights are read once a step. Lane j of every wave owns output j of the block's 64 and
// walks its weight row; the four waves take a quarter of K each, and their partial sums meet in
// LDS in a fixed order. A token's sum is the same sequence of operations whatever else is in the
// batch. Tokens go in groups of HL_TOKENS with the inputs in LDS as float32.
#define HL_TOKENS 8
template <typename T>
__global__ __launch_bounds__(256) void heads_linear_rows_kernel(const T* __restrict__ x, long x_row, int in_stride, int in_offset,
                                                                const T* __restrict__ w, int n, int k, T* __restrict__ out,
                                                                long out_row, int out_stride, int out_offset, int num_tokens) {
  extern __shared__ float sm[];
  float* xs = sm;                        // [HL_TOKENS][k]
  float* red = sm + HL_TOKENS * k;       // [4][HL_TOKENS][64]
  const int h = blockIdx.y, j0 = blockIdx.x * 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int j = min(j0 + lane, n - 1);
  const T* wr = w + ((size_t)h * n + j) * k;
  const int per = (k + 3) / 4, c0 = min(wave * per, k), c1 = min(k, c0 + per);
  for (int t0 = 0; t0 < num_tokens; t0 += HL_TOKENS) {
    const int nt = min(HL_TOKENS, num_tokens - t0);
    __syncthreads();
    for (int i = threadIdx.x; i < HL_TOKENS * k; i += 256) {
      const int t = i / k, c = i - t * k;
      xs[i] = t < nt ? to_f32<T>(x[(size_t)(t0 + t) * x_row + (size_t)h * in_stride + in_offset + c]) : 0.f;
    }
    __syncthreads();
    float acc[HL_TOKENS];
#pragma unroll
    for (int t = 0; t < HL_TOKENS; ++t) acc[t] = 0.f;
    if (sizeof(T) == 2 && (k & 31) == 0 && ((uintptr_t)w & 15) == 0) {
      // bfloat16 rows whose quarters are whole 16-byte pieces: eight weights a load
      for (int c = c0; c < c1; c += 8) {
        const bf16x8_t w8 = *(const bf16x8_t*)((const bf16_t*)wr + c);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float wv = (float)w8[e];
#pragma unroll
          for (int t = 0; t < HL_TOKENS; ++t) acc[t] = fmaf(xs[t * k + c + e], wv, acc[t]);
        }
      }
    } else {
      for (int c = c0; c < c1; ++c) {
        const float wv = to_f32<T>(wr[c]);
#pragma unroll
        for (int t = 0; t < HL_TOKENS; ++t) acc[t] = fmaf(xs[t * k + c], wv, acc[t]);
      }
    }
#pragma unroll
    for (int t = 0; t < HL_TOKENS; ++t) red[(wave * HL_TOKENS + t) * 64 + lane] = acc[t];
    __syncthreads();
    for (int i = threadIdx.x; i < nt * 64; i += 256) {
      const int t = i >> 6, l = i & 63;
      if (j0 + l < n) {
        const float sum = ((red[(0 * HL_TOKENS + t) * 64 + l] + red[(1 * HL_TOKENS + t) * 64 + l]) +
                           red[(2 * HL_TOKENS + t) * 64 + l]) + red[(3 * HL_TOKENS + t) * 64 + l];
        out[(size_t)(t0 + t) * out_row + (size_t)h * out_stride + out_offset + j0 + l] = from_f32<T>(sum);
      }
    }
  }
}

// bfloat16 with K a multiple of 64 and rows in whole pieces of 16 bytes: tiles of 128 tokens x BN outputs of a head on
// MFMA, four waves, 64 k at a time in two LDS stages filled by direct loads of whole cache lines (piece c of row r at
// 128 r + 16 (c ^ (r & 7)), as in the other tile kernels). K is one head's width, so a tile is two to six stages and
// the pass is bound by its rows' way in and out: strided rows are read and written in place. A batched library
// product on transposed weights and a copy of its result into the strided rows took 61 and 33 us for 32 heads of
// 128 -> 384 and 384 -> 128 at 2,047 tokens; this kernel 26 and 16 (67 MB: 14 at the rate of a copy).
// Neighbouring blocks of an XCD share a head's weights and a stretch of tokens.
template <int BN>
__global__ __launch_bounds__(256, 2) void heads_linear_tile_kernel(const bf16_t* __restrict__ x, long x_row, int in_stride, int in_offset,
                                                                   const bf16_t* __restrict__ w, int heads, int n, int k,
                                                                   bf16_t* __restrict__ out, long out_row, int out_stride, int out_offset,
                                                                   int num_tokens) {
  constexpr int STAGE = (128 + BN) * 128, LOADS = (128 + BN) / 32, WN = BN / 2, JT = BN / 32;
  extern __shared__ __align__(16) unsigned char lds[];  // [2][128 tokens | BN weight rows] x 128 bytes
  const int col_tiles = (n + BN - 1) / BN, row_tiles = (num_tokens + 127) / 128;
  const int total = heads * col_tiles * row_tiles, per = (total + 7) >> 3;
  const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || tile >= total) return;
  const int h = tile / (col_tiles * row_tiles), rest = tile % (col_tiles * row_tiles);
  const int t0 = rest / col_tiles * 128, n0 = rest % col_tiles * BN;
  const int lane = threadIdx.x & 63, wave = uniform_wave_number();
  const int r16 = lane & 15, quad = lane >> 4, wm = (wave >> 1) * 64, wn = (wave & 1) * WN;
  const int sub = lane >> 3, piece = (lane & 7) ^ sub;
  // a wave's loads of a stage, 8 rows x 128 bytes each; rows past the end repeat the last and are not stored
  const bf16_t* src[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int r = (wave * LOADS + i) * 8 + sub;
    src[i] = r < 128 ? x + (size_t)min(t0 + r, num_tokens - 1) * x_row + (size_t)h * in_stride + in_offset + 8 * piece
                     : w + ((size_t)h * n + min(n0 + r - 128, n - 1)) * k + 8 * piece;
  }
  unsigned char* dst = lds + wave * LOADS * 1024;
  auto fetch = [&](int s) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      __builtin_amdgcn_global_load_lds((global_ptr_t)(src[i] + (size_t)s * 64), (lds_ptr_t)(dst + (s & 1) * STAGE + i * 1024), 16, 0, 0);
  };
  f32x4_t acc[4][JT];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < JT; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  const int stages = k >> 6;
  fetch(0);
  for (int s = 0; s < stages; ++s) {
    if (s + 1 < stages) {
      fetch(s + 1);
      QRT_WAIT_LOADS(LOADS);
    } else {
      QRT_WAIT_LOADS(0);
    }
    QRT_BARRIER();
    const unsigned char* at = lds + (s & 1) * STAGE;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int col = 16 * ((4 * e + quad) ^ (r16 & 7));
      bf16x8_t xv[4], wv[JT];
#pragma unroll
      for (int i = 0; i < 4; ++i) xv[i] = *(const bf16x8_t*)(at + (wm + 16 * i + r16) * 128 + col);
#pragma unroll
      for (int j = 0; j < JT; ++j) wv[j] = *(const bf16x8_t*)(at + (128 + wn + 16 * j + r16) * 128 + col);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < JT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[j], xv[i], acc[i][j], 0, 0, 0);
    }
    QRT_WAIT_LDS();  // read before the barrier behind which the stage may be overwritten
    QRT_BARRIER();
  }
  // acc[i][j]: token t0 + wm + 16 i + r16, four outputs from n0 + wn + 16 j + 4 quad on
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = t0 + wm + 16 * i + r16;
    if (t >= num_tokens) continue;
    bf16_t* o = out + (size_t)t * out_row + (size_t)h * out_stride + out_offset;
#pragma unroll
    for (int j = 0; j < JT; ++j) {
      const int c = n0 + wn + 16 * j + 4 * quad;
      if (c >= n) continue;  // n is a multiple of 4: four or none
      bf16x4_t v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = from_f32<bf16_t>(acc[i][j][r]);
      *(bf16x4_t*)(o + c) = v;
    }
  }
}

extern "C" int qrt_heads_linear(const void* x, long x_row, int in_stride, int in_offset, const void* w, int heads, int n, int k,
                                void* out, long out_row, int out_stride, int out_offset, int dtype, int num_tokens, int tiles,
                                hipStream_t stream) {
  QRT_CHECK(num_tokens >= 0 && heads > 0 && heads <= 65535 && n > 0 && k > 0 && k <= 16384, "heads_linear: bad sizes");
  QRT_CHECK(in_offset >= 0 && in_offset + k <= in_stride && (long)heads * in_stride <= x_row && out_offset >= 0 &&
            out_offset + n <= out_stride && (long)heads * out_stride <= out_row, "heads_linear: heads do not fit their rows");
  if (num_tokens == 0) return 0;
  if (tiles) {
    QRT_CHECK(dtype == QRT_BF16 && k % 64 == 0 && n % 4 == 0 && (x_row | in_stride | in_offset) % 8 == 0 &&
                  (out_row | out_stride | out_offset) % 4 == 0 && ((uintptr_t)x | (uintptr_t)w) % 16 == 0 && (uintptr_t)out % 8 == 0,
              "heads_linear: rows of the tile kernel are whole pieces of 16 bytes");
    const bool narrow = n <= 64;
    const long blocks = (long)heads * ((n + (narrow ? 63 : 127)) / (narrow ? 64 : 128)) * ((num_tokens + 127) / 128);
    QRT_CHECK(blocks < (1l << 30), "heads_linear: too many tiles");
    const unsigned grid = (unsigned)((blocks + 7) / 8 * 8);
    auto kernel = narrow ? heads_linear_tile_kernel<64> : heads_linear_tile_kernel<128>;
    kernel<<<grid, 256, narrow ? 48 * 1024 : 64 * 1024, stream>>>((const bf16_t*)x, x_row, in_stride, in_offset, (const bf16_t*)w, heads, n, k,
                                                                  (bf16_t*)out, out_row, out_stride, out_offset, num_tokens);
    QRT_LAUNCH_CHECK("heads_linear_tile");
    return 0;
  }
  if (num_tokens <= 64 && k <= 1024) {  // the head's weights once a step
    const dim3 rows_grid((n + 63) / 64, heads);
    const size_t rows_lds = (size_t)(HL_TOKENS * k + 4 * HL_TOKENS * 64) * sizeof(float);
    if (dtype == QRT_F32)
      heads_linear_rows_kernel<float><<<rows_grid, 256, rows_lds, stream>>>((const float*)x, x_row, in_stride, in_offset, (const float*)w,
                                                                            n, k, (float*)out, out_row, out_stride, out_offset, num_tokens);
    else if (dtype == QRT_BF16)
      heads_linear_rows_kernel<bf16_t><<<rows_grid, 256, rows_lds, stream>>>((const bf16_t*)x, x_row, in_stride, in_offset, (const bf16_t*)w,
                                                                             n, k, (bf16_t*)out, out_row, out_stride, out_offset, num_tokens);
    else return qrt_fail("heads_linear: unknown dtype %d", dtype);
    QRT_LAUNCH_CHECK("heads_linear_rows");
    return 0;
  }
  const dim3 grid(num_tokens, heads);
  const size_t lds = (size_t)k * sizeof(float);
  if (dtype == QRT_F32)
    heads_linear_kernel<float><<<grid, 256, lds, stream>>>((const float*)x, x_row, in_stride, in_offset, (const float*)w, n, k,
                                                           (float*)out, out_row, out_stride, out_offset);
  else if (dtype == QRT_BF16)
    heads_linear_kernel<bf16_t><<<grid, 256, lds, stream>>>((const bf16_t*)x, x_row, in_stride, in_offset, (const bf16_t*)w, n, k,
                                                            (bf16_t*)out, out_row, out_stride, out_offset);
  else return qrt_fail("heads_linear: unknown dtype %d", dtype);
  QRT_LAUNCH_CHECK("heads_linear");
  return 0;
}
