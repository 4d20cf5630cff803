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
#include <type_traits>
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

// ---------------------------------------------------------------- norm of some columns, and the cached row
struct LatentArgs {
  const void* y; long stride; int num_tokens;
  // the norm of columns [q_first, q_first + q_width)
  int q_first, q_width; const float* q_weight; float q_eps; void* q_out;
  // the cached row
  int first, rank, rot_dim; const float* weight; float eps;
  const int* positions; const float* freq; int pairs; const int* slots; void* k_cache; void* v_cache; int page_size;
  int neighbours; float magnitude;
};

// A row in pieces of 256 elements, one a thread each. KEEP, the first of up to four, stay in registers, asked for with their weights in one go;
// the rest of a row over 1,024 is read again, four pieces at a time (`put` stores, and no load would be moved up in front of a store).
// us at 8 and 2,048 rows by an element at a time, four always in registers and the rest one at a time, and this: rows of 64 2.5, 3.1 and 2.3, 3.3 and 2.3, 3.0;
// of 1,536 3.7, 5.7 and 3.1, 5.7 and 2.9, 5.3; of 2,560 4.6, 7.3 and 3.9, 8.2 and 3.3, 6.9; of 8,192 9.7, 23.0 and 9.0, 30.0 and 5.7, 18.7.
template <int N>
struct RowPieces {  // of which the last may be part of one: its threads beyond the row read the last element and count for nothing
  float v[N];
  template <typename T>
  __device__ __forceinline__ void load(const T* __restrict__ row, int from, int width) {
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const int i = from + 256 * k + (int)threadIdx.x;
      v[k] = to_f32<T>(row[k < N - 1 ? i : min(i, width - 1)]);
    }
  }
};
template <typename T, int KEEP, class Put>
__device__ __forceinline__ void rms_normed(const T* __restrict__ row, int width, const float* __restrict__ weight, float eps, float* red, Put put) {
  float ss = 0.f, inv;
  auto add = [&](auto& x, int from) {
    constexpr int N = sizeof(x.v) / sizeof(float);
#pragma unroll
    for (int k = 0; k < N; ++k) ss += k < N - 1 || from + 256 * k + (int)threadIdx.x < width ? x.v[k] * x.v[k] : 0.f;
  };
  auto store = [&](auto& x, auto& w, int from) {
    constexpr int N = sizeof(x.v) / sizeof(float);
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const int i = from + 256 * k + (int)threadIdx.x;
      if (k < N - 1 || i < width) put(i, from_f32<T>(x.v[k] * inv * w.v[k]));
    }
  };
  auto rest = [&](auto each) {  // four pieces at a time, then the one to four that are left; the same in the whole block
    int from = 1024;
    for (; width - from > 1024; from += 1024) each(std::integral_constant<int, 4>{}, from);
    switch ((width - from + 255) >> 8) {
      case 1: each(std::integral_constant<int, 1>{}, from); break;
      case 2: each(std::integral_constant<int, 2>{}, from); break;
      case 3: each(std::integral_constant<int, 3>{}, from); break;
      case 4: each(std::integral_constant<int, 4>{}, from); break;
    }
  };
  RowPieces<KEEP> kept, kept_weight;
  kept.load(row, 0, width);
  kept_weight.load(weight, 0, width);
  add(kept, 0);
  if (KEEP == 4)
    rest([&](auto count, int from) {
      RowPieces<decltype(count)::value> x;
      x.load(row, from, width);
      add(x, from);
    });
  ss = block_sum(ss, red);
  inv = 1.0f / sqrtf(ss / (float)width + eps);
  store(kept, kept_weight, 0);
  if (KEEP == 4)
    rest([&](auto count, int from) {
      RowPieces<decltype(count)::value> x, w;
      x.load(row, from, width);
      w.load(weight, from, width);
      store(x, w, from);
    });
}
template <typename T, class Put>
__device__ __forceinline__ void rms_normed(const T* __restrict__ row, int width, const float* __restrict__ weight, float eps, float* red, Put put) {
  if (width <= 256) rms_normed<T, 1>(row, width, weight, eps, red, put);  // the same branch in the whole block
  else if (width <= 512) rms_normed<T, 2>(row, width, weight, eps, red, put);
  else if (width <= 768) rms_normed<T, 3>(row, width, weight, eps, red, put);
  else rms_normed<T, 4>(row, width, weight, eps, red, put);
}

template <typename T>
__device__ __forceinline__ void store_latent(const LatentArgs& a, int t, float* red) {
  const T* row = (const T*)a.y + (size_t)t * a.stride + a.first;
  const int w = a.rank + a.rot_dim;
  const int slot = a.slots[t];
  const int page = slot / a.page_size, off = slot - page * a.page_size;
  T* kr = (T*)a.k_cache + (size_t)slot * w;
  T* vr = (T*)a.v_cache + (size_t)page * w * a.page_size + off;
  const float pos = (float)a.positions[t];
  const T* rot = row + a.rank;
  for (int i = threadIdx.x; i < a.rot_dim; i += 256) {
    float x = to_f32<T>(rot[i]);
    if (i < 2 * a.pairs) {
      int j, o;
      bool first;
      rotation_partner(i, a.pairs, a.neighbours, &j, &o, &first);
      const float other = to_f32<T>(rot[o]);
      float sn, cs;
      sincos_angle(pos * a.freq[j], &sn, &cs);
      sn *= a.magnitude;
      cs *= a.magnitude;
      x = first ? x * cs - other * sn : x * cs + other * sn;
    }
    kr[a.rank + i] = from_f32<T>(x);
    vr[(size_t)(a.rank + i) * a.page_size] = from_f32<T>(0.f);
  }
  rms_normed<T>(row, a.rank, a.weight, a.eps, red, [&](int i, T c) {
    kr[i] = c;
    vr[(size_t)i * a.page_size] = c;
  });
}

// Block row `jobs` + blockIdx.y: 0 the norm, 1 the cached row. Both in one launch where a layer wants both: 8 tokens 4.7 and 5.2 us
// apart in a traced step, 5.0 together.
template <typename T>
__global__ __launch_bounds__(256) void latent_rows_kernel(LatentArgs a, int jobs) {
  __shared__ float red[32];
  const int t = blockIdx.x;
  if (jobs + blockIdx.y == 0) {
    T* out = (T*)a.q_out + (size_t)t * a.q_width;
    rms_normed<T>((const T*)a.y + (size_t)t * a.stride + a.q_first, a.q_width, a.q_weight, a.q_eps, red, [&](int i, T c) { out[i] = c; });
  } else {
    store_latent<T>(a, t, red);
  }
}

static int latent_rows(const LatentArgs& a, bool norm, bool store, int dtype, hipStream_t stream) {
  if (norm)
    QRT_CHECK(a.num_tokens >= 0 && a.q_width > 0 && a.q_first >= 0 && (long)a.q_first + a.q_width <= a.stride, "rmsnorm_columns: bad sizes");
  if (store) {
    QRT_CHECK(a.num_tokens >= 0 && a.rank > 0 && a.rot_dim >= 0 && a.first >= 0 && (long)a.first + a.rank + a.rot_dim <= a.stride,
              "latent_store: bad sizes");
    QRT_CHECK(a.pairs >= 0 && 2 * a.pairs <= a.rot_dim && (a.pairs == 0 || a.freq), "latent_store: %d pairs in %d elements", a.pairs, a.rot_dim);
    QRT_CHECK(a.page_size > 0 && a.slots && a.positions && a.k_cache && a.v_cache, "latent_store: no cache");
  }
  QRT_CHECK(dtype == QRT_F32 || dtype == QRT_BF16, "latent rows: unknown dtype %d", dtype);
  if (a.num_tokens == 0) return 0;
  const dim3 grid(a.num_tokens, norm && store ? 2 : 1);
  if (dtype == QRT_F32) latent_rows_kernel<float><<<grid, 256, 0, stream>>>(a, norm ? 0 : 1);
  else latent_rows_kernel<bf16_t><<<grid, 256, 0, stream>>>(a, norm ? 0 : 1);
  QRT_LAUNCH_CHECK("latent_rows");
  return 0;
}

extern "C" int qrt_rmsnorm_columns(const void* y, long stride, int first, int width, const float* weight, float eps,
                                   void* out, int dtype, int num_tokens, hipStream_t stream) {
  LatentArgs a{};
  a.y = y, a.stride = stride, a.num_tokens = num_tokens;
  a.q_first = first, a.q_width = width, a.q_weight = weight, a.q_eps = eps, a.q_out = out;
  return latent_rows(a, true, false, dtype, stream);
}

// q_out null: the cached row alone
extern "C" int qrt_latent_store(const void* y, long stride, int first, int rank, int rot_dim, const float* weight, float eps,
                                const int* positions, const float* freq, int pairs, const int* slots, void* k_cache,
                                void* v_cache, int page_size, long num_pages, int dtype, int num_tokens, int neighbours,
                                float magnitude, int q_first, int q_width, const float* q_weight, void* q_out, hipStream_t stream) {
  QRT_CHECK(num_pages > 0, "latent_store: no cache");
  const LatentArgs a{y, stride, num_tokens, q_first, q_width, q_weight, eps, q_out, first, rank, rot_dim, weight, eps,
                     positions, freq, pairs, slots, k_cache, v_cache, page_size, neighbours, magnitude};
  return latent_rows(a, q_out != nullptr, true, dtype, stream);
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
__device__ __forceinline__ void rotate_token(const RotateArgs& a, int t, int y, int ys, float* cosines, float* sines) {
  typedef TI ivec_t __attribute__((ext_vector_type(8), aligned(16)));
  typedef TO ovec_t __attribute__((ext_vector_type(8), aligned(16)));
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
  for (int e = y * 256 + threadIdx.x; e < total; e += 256 * ys) {
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

template <typename TI, typename TO>
__global__ __launch_bounds__(256) void rotate_half_wide_kernel(RotateArgs a) {
  __shared__ float cosines[ROTATE_MAX_PAIRS], sines[ROTATE_MAX_PAIRS];
  rotate_token<TI, TO>(a, blockIdx.x, blockIdx.y, gridDim.y, cosines, sines);
}
// Two of them in one launch, one in each half of the grid: 8 tokens, 64 heads turned and 32 copied, 9.2 us in
// two in a traced step, 4.7 in one.
template <typename TI, typename TO>
__global__ __launch_bounds__(256) void rotate_half_two_kernel(RotateArgs a, RotateArgs b) {
  __shared__ float cosines[ROTATE_MAX_PAIRS], sines[ROTATE_MAX_PAIRS];
  rotate_token<TI, TO>(blockIdx.z == 0 ? a : b, blockIdx.x, blockIdx.y, gridDim.y, cosines, sines);
}

static bool rotate_in_pieces(const RotateArgs& a) {
  return !a.neighbours && a.pairs <= ROTATE_MAX_PAIRS && (a.pairs | a.width | a.in_stride | a.in_offset | a.out_stride | a.out_offset) % 8 == 0 &&
         a.x_row % 8 == 0 && a.out_row % 8 == 0 && ((uintptr_t)a.x | (uintptr_t)a.out) % 16 == 0;
}
static int rotate_check(const RotateArgs& a, int num_tokens) {
  QRT_CHECK(num_tokens >= 0 && a.heads > 0 && a.width > 0 && a.pairs >= 0 && 2 * a.pairs <= a.width, "rotate_half: bad sizes");
  QRT_CHECK(a.in_offset >= 0 && a.in_offset + a.width <= a.in_stride && (long)a.heads * a.in_stride <= a.x_row &&
            a.out_offset >= 0 && a.out_offset + a.width <= a.out_stride && (long)a.heads * a.out_stride <= a.out_row,
            "rotate_half: heads of %d at %d in rows of %ld, to heads of %d at %d in rows of %ld", a.in_stride, a.in_offset,
            a.x_row, a.out_stride, a.out_offset, a.out_row);
  QRT_CHECK(a.pairs == 0 || (a.freq && a.positions), "rotate_half: no angles");
  return 0;
}

extern "C" int qrt_rotate_half(const RotateArgs* args, int in_dtype, int out_dtype, int num_tokens, hipStream_t stream) {
  const RotateArgs a = *args;
  if (const int rc = rotate_check(a, num_tokens)) return rc;
  if (num_tokens == 0) return 0;
  const int total = a.heads * a.width;
  const dim3 grid(num_tokens, num_tokens >= 512 ? 1 : min((total + 255) / 256, 64));
  const bool pieces = rotate_in_pieces(a) && (num_tokens > 8 || 2 * a.pairs == a.width);
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

// Two copies of the same tokens and types, into places that do not overlap: in one launch where both go by pieces.
extern "C" int qrt_rotate_half_two(const RotateArgs* first, const RotateArgs* second, int in_dtype, int out_dtype, int num_tokens,
                                   hipStream_t stream) {
  const RotateArgs a = *first, b = *second;
  if (const int rc = rotate_check(a, num_tokens)) return rc;
  if (const int rc = rotate_check(b, num_tokens)) return rc;
  if (num_tokens == 0) return 0;
  if (in_dtype == QRT_BF16 && out_dtype == QRT_F32 && rotate_in_pieces(a) && rotate_in_pieces(b)) {
    const int most = max(a.heads * a.width, b.heads * b.width) / 8;
    rotate_half_two_kernel<bf16_t, float><<<dim3(num_tokens, num_tokens >= 512 ? 1 : min((most + 255) / 256, 64), 2), 256, 0, stream>>>(a, b);
    QRT_LAUNCH_CHECK("rotate_half_two");
    return 0;
  }
  if (const int rc = qrt_rotate_half(first, in_dtype, out_dtype, num_tokens, stream)) return rc;
  return qrt_rotate_half(second, in_dtype, out_dtype, num_tokens, stream);
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
//
// MORE = HL_GATE: the result, rounded, times the sigmoid of gate[t, its column in out] and rounded again, as a pass behind it would
// make it. HL_ROTATE: blocks behind those of the tiles turn and copy another part of the heads, as rotate_half does (`ys` a token).
// A launch less either way: 8 tokens of 32 heads in a traced step, 384 -> 128 and the gate 11.9 and 8.8 us, 128 -> 384 and the rotation
// of 64 elements 9.6 and 5.3.
//
// Few tokens: tiles of 32 tokens x 64 outputs with eight stages in the ring, while they are no more than one for each of 256 compute units. What
// bounds the pass then is a stage's latency after the other's, and few blocks: 512 columns of K come at one time here, 32 heads of 128 outputs are 64
// blocks. Same sums, same bits. us by tiles of 128 tokens and these, from a graph:
//   32 heads, 384 -> 128 and the gate, at 1, 8, 32, 64 and 128 tokens 8.9, 8.1, 9.8, 13.2, 13.2 and 5.3, 5.0, 5.25, 5.3, 5.4; without it 6.5, 6.6, 6.9, 7.6, 8.3
//   and 4.2, 4.3, 4.6, 4.7, 4.7; 128 -> 384 beside the rotation at 1, 8 and 32 4.5, 4.6, 5.0 and 3.6, 3.75, 4.0 (at 33, 384 tiles, 5.0 and 5.5);
//   128 heads, 512 -> 128 at 8 and 33 (512 tiles) 8.8, 9.3 and 6.4, 9.6.
enum { HL_PLAIN = 0, HL_GATE = 1, HL_ROTATE = 2 };
template <int BM, int BN, int S, int MORE>
__global__ __launch_bounds__(256, BM == 128 ? 2 : 1) void heads_linear_tile_kernel(const bf16_t* __restrict__ x, long x_row, int in_stride, int in_offset,
                                                                   const bf16_t* __restrict__ w, int heads, int n, int k,
                                                                   bf16_t* __restrict__ out, long out_row, int out_stride, int out_offset,
                                                                   int num_tokens, const bf16_t* __restrict__ gate, long gate_row,
                                                                   RotateArgs turn, int tile_blocks, int ys) {
  extern __shared__ __align__(16) unsigned char lds[];  // [S][BM tokens | BN weight rows] x 128 bytes
  if (MORE == HL_ROTATE && (int)blockIdx.x >= tile_blocks) {  // the whole block turns here, before any other barrier
    const int b = blockIdx.x - tile_blocks;
    rotate_token<bf16_t, bf16_t>(turn, b / ys, b % ys, ys, (float*)lds, (float*)lds + ROTATE_MAX_PAIRS);
    return;
  }
  constexpr int STAGE = (BM + BN) * 128, LOADS = (BM + BN) / 32, WM = BM / 2, WN = BN / 2, IT = BM / 32, JT = BN / 32;
  static_assert((S & (S - 1)) == 0 && (S - 1) * LOADS < 64, "slots by a mask, the loads' counter");
  const int col_tiles = (n + BN - 1) / BN, row_tiles = (num_tokens + BM - 1) / BM;
  const int total = heads * col_tiles * row_tiles, per = (total + 7) >> 3;
  const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || tile >= total) return;
  const int h = tile / (col_tiles * row_tiles), rest = tile % (col_tiles * row_tiles);
  const int t0 = rest / col_tiles * BM, n0 = rest % col_tiles * BN;
  const int lane = threadIdx.x & 63, wave = uniform_wave_number();
  const int r16 = lane & 15, quad = lane >> 4, wm = (wave >> 1) * WM, wn = (wave & 1) * WN;
  const int sub = lane >> 3, piece = (lane & 7) ^ sub;
  // a wave's loads of a stage, 8 rows x 128 bytes each; rows past the end repeat the last and are not stored
  const bf16_t* src[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int r = (wave * LOADS + i) * 8 + sub;
    src[i] = r < BM ? x + (size_t)min(t0 + r, num_tokens - 1) * x_row + (size_t)h * in_stride + in_offset + 8 * piece
                     : w + ((size_t)h * n + min(n0 + r - BM, n - 1)) * k + 8 * piece;
  }
  unsigned char* dst = lds + wave * LOADS * 1024;
  auto fetch = [&](int s) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      __builtin_amdgcn_global_load_lds((global_ptr_t)(src[i] + (size_t)s * 64), (lds_ptr_t)(dst + (s & (S - 1)) * STAGE + i * 1024), 16, 0, 0);
  };
  f32x4_t acc[IT][JT];
#pragma unroll
  for (int i = 0; i < IT; ++i)
#pragma unroll
    for (int j = 0; j < JT; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  const int stages = k >> 6;
#pragma unroll
  for (int s = 0; s < S - 1; ++s)
    if (s < stages) fetch(s);
  for (int s = 0; s < stages; ++s) {
    if (s + S - 1 < stages) {
      fetch(s + S - 1);
      QRT_WAIT_LOADS((S - 1) * LOADS);
    } else {
      QRT_WAIT_LOADS(0);
    }
    QRT_BARRIER();
    const unsigned char* at = lds + (s & (S - 1)) * STAGE;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int col = 16 * ((4 * e + quad) ^ (r16 & 7));
      bf16x8_t xv[IT], wv[JT];
#pragma unroll
      for (int i = 0; i < IT; ++i) xv[i] = *(const bf16x8_t*)(at + (wm + 16 * i + r16) * 128 + col);
#pragma unroll
      for (int j = 0; j < JT; ++j) wv[j] = *(const bf16x8_t*)(at + (BM + wn + 16 * j + r16) * 128 + col);
#pragma unroll
      for (int i = 0; i < IT; ++i)
#pragma unroll
        for (int j = 0; j < JT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[j], xv[i], acc[i][j], 0, 0, 0);
    }
    QRT_WAIT_LDS();  // read before the barrier behind which the stage may be overwritten
    QRT_BARRIER();
  }
  // acc[i][j]: token t0 + wm + 16 i + r16, four outputs from n0 + wn + 16 j + 4 quad on
#pragma unroll
  for (int i = 0; i < IT; ++i) {
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
      if (MORE == HL_GATE) {
        const bf16x4_t g = *(const bf16x4_t*)(gate + (size_t)t * gate_row + (size_t)h * out_stride + out_offset + c);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = (bf16_t)((float)v[r] / (1.0f + expf(-(float)g[r])));
      }
      *(bf16x4_t*)(o + c) = v;
    }
  }
}

// `gate` [num_tokens, gate_row] or null, `turn` or null: with `tiles` only.
extern "C" int qrt_heads_linear(const void* x, long x_row, int in_stride, int in_offset, const void* w, int heads, int n, int k,
                                void* out, long out_row, int out_stride, int out_offset, int dtype, int num_tokens, int tiles,
                                const void* gate, long gate_row, const RotateArgs* turn, hipStream_t stream) {
  QRT_CHECK(num_tokens >= 0 && heads > 0 && heads <= 65535 && n > 0 && k > 0 && k <= 16384, "heads_linear: bad sizes");
  QRT_CHECK(in_offset >= 0 && in_offset + k <= in_stride && (long)heads * in_stride <= x_row && out_offset >= 0 &&
            out_offset + n <= out_stride && (long)heads * out_stride <= out_row, "heads_linear: heads do not fit their rows");
  QRT_CHECK((!gate && !turn) || (tiles && !(gate && turn)), "heads_linear: a gate or a rotation goes with the tile kernel");
  if (turn)
    if (const int rc = rotate_check(*turn, num_tokens)) return rc;
  if (num_tokens == 0) return 0;
  if (tiles) {
    QRT_CHECK(dtype == QRT_BF16 && k % 64 == 0 && n % 4 == 0 && (x_row | in_stride | in_offset) % 8 == 0 &&
                  (out_row | out_stride | out_offset) % 4 == 0 && ((uintptr_t)x | (uintptr_t)w) % 16 == 0 && (uintptr_t)out % 8 == 0,
              "heads_linear: rows of the tile kernel are whole pieces of 16 bytes");
    QRT_CHECK(!gate || (gate_row >= (long)heads * out_stride && gate_row % 4 == 0 && (uintptr_t)gate % 8 == 0),
              "heads_linear: gate rows of %ld elements in pieces of 8 bytes", gate_row);
    QRT_CHECK(!turn || rotate_in_pieces(*turn), "heads_linear: the rotation beside it goes by pieces of 16 bytes");
    const bool few = (long)heads * ((n + 63) / 64) * ((num_tokens + 31) / 32) <= 256, narrow = few || n <= 64;
    const int rows = few ? 32 : 128, columns = narrow ? 64 : 128;
    const long blocks = (long)heads * ((n + columns - 1) / columns) * ((num_tokens + rows - 1) / rows);
    const int ys = turn ? (num_tokens >= 512 ? 1 : min((turn->heads * turn->width / 8 + 255) / 256, 64)) : 0;
    QRT_CHECK(blocks < (1l << 30) && (long)num_tokens * ys < (1l << 30), "heads_linear: too many tiles");
    const unsigned grid = (unsigned)((blocks + 7) / 8 * 8);
#define GO(BM, BN, S, MORE)                                                                                                          \
  do {                                                                                                                               \
    auto kernel = heads_linear_tile_kernel<BM, BN, S, MORE>;                                                                         \
    constexpr int smem = S * (BM + BN) * 128;                                                                                        \
    static bool allowed = false; /* once per kernel: not inside a stream capture again and again */                                 \
    if (smem > 64 * 1024 && !allowed) {                                                                                              \
      if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, smem) != hipSuccess)                  \
        return qrt_fail("heads_linear: cannot get %d bytes of LDS", smem);                                                           \
      allowed = true;                                                                                                                \
    }                                                                                                                                \
    kernel<<<grid + (unsigned)(num_tokens * ys), 256, smem, stream>>>(                                                               \
        (const bf16_t*)x, x_row, in_stride, in_offset, (const bf16_t*)w, heads, n, k, (bf16_t*)out, out_row, out_stride, out_offset, \
        num_tokens, (const bf16_t*)gate, gate_row, turn ? *turn : RotateArgs{}, (int)grid, ys);                                      \
  } while (0)
#define BY_SIZE(MORE)                       \
  do {                                      \
    if (few) GO(32, 64, 8, MORE);           \
    else if (narrow) GO(128, 64, 2, MORE);  \
    else GO(128, 128, 2, MORE);             \
  } while (0)
    if (gate) BY_SIZE(HL_GATE);
    else if (turn) BY_SIZE(HL_ROTATE);
    else BY_SIZE(HL_PLAIN);
#undef BY_SIZE
#undef GO
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
