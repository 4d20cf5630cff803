// Paged attention in true 32-bit: a kernel by tiles (below) for the usual sizes in float32, and one for
// any head size and either type.
//
// The latter: one wave per (query token, query head). The wave walks the keys its query may
// see in chunks of 64 (one key per lane for the scores), keeps a running
// maximum and sum (online softmax, float32), and accumulates the context with
// each lane owning head elements lane, lane + 64, ... Query head h reads key
// head h / g. The query at position p sees keys j <= p, and j > p - window when
// a window is set, or j >= p - p % chunk when a chunk size is. Scores are
// dot * scale, then, with a cap, cap * tanh(score / cap). Values may have another
// size Dv than keys; with a gate the output is multiplied by sigmoid(gate). Beside a window the
// first keep_first keys of the sequence stay visible to every later query (their pages stay in the
// table; the pages between them and the window may be gone and are not touched). With a sink the
// softmax's denominator has one more term of score 0: p_j = exp(s_j) / (1 + sum exp(s_j)). Cache
// layout: keys [page, head, offset, D], values [page, head, Dv, offset].
#include "common.h"
#include <math.h>
#include <type_traits>

struct AttnArgs {
  const void* q;         // [T, nq * D]
  void* out;             // [T, nq * D]
  const void* k_cache;
  const void* v_cache;
  const int* positions;  // [T] position of each query token
  const int* seq_of_token;  // [T]
  const int* block_table;   // [S, table_width]
  int table_width;
  int num_tokens, nq, nkv, head_dim, page_size, window;  // window 0: none
  float scale;
  int chunk;       // 0: none
  float softcap;   // 0: none
  int value_dim;   // 0: head_dim
  const void* gate;  // [T, gate_stride] with nq * Dv columns used, or null
  long gate_stride;
  int keep_first;  // with a window: keys j < keep_first are seen too
  int sink;        // 1: one more term exp(0) in the denominator
  const float* turn;  // [T, Dv] or null: cosines of the token's Dv / 2 angles, then their sines; the output is turned back by them
  const int* cu_q;    // [S + 1] or null: first token of every sequence (the tile kernel goes by it)
  int num_seqs, max_q_len;  // sequences, and the most tokens one brings
  int min_q_len;            // the fewest (0: not known)
};

#define MAX_D 1024

// What a wave wrote to its own LDS is there for all of its lanes.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One token's head, by one wave; `qs`: MD floats of LDS of its own (heads and values of up to MD elements).
template <typename T, int MD>
__device__ __forceinline__ void attend_row(const AttnArgs& a, int t, int h, float* qs) {
  const int lane = threadIdx.x & 63;
  const int D = a.head_dim, ps = a.page_size, Dv = a.value_dim;
  const int kvh = h / (a.nq / a.nkv);
  const int pos = a.positions[t];
  const int* table = a.block_table + (size_t)a.seq_of_token[t] * a.table_width;
  const T* q = (const T*)a.q + ((size_t)t * a.nq + h) * D;
  for (int i = lane; i < D; i += 64) qs[i] = to_f32<T>(q[i]);
  wave_lds_fence();

  const int lo = a.window > 0 ? max(0, pos - a.window + 1) : (a.chunk > 0 ? pos - pos % a.chunk : 0);
  float m = -INFINITY, l = 0.f;
  float acc[(MD + 63) / 64];
#pragma unroll
  for (int i = 0; i < (MD + 63) / 64; ++i) acc[i] = 0.f;

  const T* kc = (const T*)a.k_cache;
  const T* vc = (const T*)a.v_cache;
  // two stretches of keys: the kept first ones that lie before the window, then the window
  const int kept_end = a.window > 0 ? min(a.keep_first, lo) : 0;
  for (int seg = kept_end > 0 ? 0 : 1; seg < 2; ++seg) {
  const int seg_begin = seg == 0 ? 0 : lo, seg_last = seg == 0 ? kept_end - 1 : pos;
  for (int j0 = seg_begin; j0 <= seg_last; j0 += 64) {
    const int j = j0 + lane;
    const bool valid = j <= seg_last;
    float s = -INFINITY;
    int page = 0, off = 0;
    if (valid) {
      page = table[j / ps];
      off = j % ps;
      const T* kr = kc + (((size_t)page * a.nkv + kvh) * ps + off) * D;
      float dot = 0.f;
      for (int d = 0; d < D; ++d) dot = fmaf(qs[d], to_f32<T>(kr[d]), dot);
      s = dot * a.scale;
      if (a.softcap > 0.f) s = a.softcap * tanhf(s / a.softcap);
    }
    const float m_new = fmaxf(m, wave_max(s));
    const float p = valid ? expf(s - m_new) : 0.f;
    const float corr = expf(m - m_new);  // m = -inf at the first chunk: exp(-inf) = 0
    l = l * corr + wave_sum(p);
    m = m_new;
#pragma unroll
    for (int i = 0; i < (MD + 63) / 64; ++i) acc[i] *= corr;
    const int n = min(64, seg_last - j0 + 1);
    for (int jj = 0; jj < n; ++jj) {
      const float pj = __shfl(p, jj, 64);
      const int pg = __shfl(page, jj, 64);
      const int of = __shfl(off, jj, 64);
      const T* vr = vc + ((size_t)pg * a.nkv + kvh) * Dv * ps + of;
#pragma unroll
      for (int i = 0; i < (MD + 63) / 64; ++i) {
        const int d = lane + 64 * i;
        if (d < Dv) acc[i] = fmaf(pj, to_f32<T>(vr[(size_t)d * ps]), acc[i]);
      }
    }
  }
  }
  if (a.sink) {  // the sink: a key of score 0 without a value
    const float m_new = fmaxf(m, 0.f);
    const float corr = expf(m - m_new);
    l = l * corr + expf(-m_new);
#pragma unroll
    for (int i = 0; i < (MD + 63) / 64; ++i) acc[i] *= corr;
  }
  T* o = (T*)a.out + ((size_t)t * a.nq + h) * Dv;
  const T* gate = a.gate ? (const T*)a.gate + (size_t)t * a.gate_stride + (size_t)h * Dv : nullptr;
  const float inv = l > 0.f ? 1.0f / l : 0.f;
  const float* angles = a.turn ? a.turn + (size_t)t * Dv : nullptr;
  if (angles) {  // partners meet in LDS, which the queries no longer need
    wave_lds_fence();
#pragma unroll
    for (int i = 0; i < (MD + 63) / 64; ++i)
      if (lane + 64 * i < Dv) qs[lane + 64 * i] = acc[i];
    wave_lds_fence();
  }
#pragma unroll
  for (int i = 0; i < (MD + 63) / 64; ++i) {
    const int d = lane + 64 * i;
    if (d < Dv) {
      float v = acc[i] * inv;
      if (angles) {
        const int half = Dv >> 1;
        const bool low = d < half;
        const int j = low ? d : d - half;
        const float p = qs[low ? d + half : j] * inv, c = angles[j], s = angles[half + j];
        v = low ? v * c + p * s : v * c - p * s;
      }
      if (gate) v *= 1.0f / (1.0f + expf(-to_f32<T>(gate[d])));
      o[d] = from_f32<T>(v);
    }
  }
}

template <typename T>
__global__ __launch_bounds__(64) void attention_f32_kernel(AttnArgs a) {
  __shared__ float qs[MAX_D];
  attend_row<T, MAX_D>(a, blockIdx.x, blockIdx.y, qs);
}

// ---------------------------------------------------------------- float32 by tiles
// A block takes 16 rows (token * g + head in group) of one sequence and key head, its W waves the
// sequence's blocks of 16 keys in turn, each with a maximum, a sum and an accumulator of its own, which
// meet in LDS at the end. Scores are formed transposed, S^T = K Q^T, on the float32 MFMA (whole float32
// products and sums): a lane then holds four neighbouring keys of its row, exactly the operand that
// O^T = V^T P^T takes against one 16-byte read of the transposed value page, so nothing crosses lanes but
// the row's maximum. The kernel before it (a wave per token and head, a key's dot product per lane,
// uncoalesced) is bound by load latency: 354 tokens of 2 sequences with 32 heads of 128 took 798 us, two
// decoded tokens behind 267 keys 170 us; this one 49 and 19 us.
// A sequence of few rows has eight waves a tile (its keys are what there is to share: a token behind 2,049 keys with
// 32 heads of 128 on 8 takes 78 us, with four 161), any other four (16 prompts of 64 tokens 60 us, with eight 105); heads wider than
// 128 always eight (2,048 tokens, 16 heads of 256 on 4: 910 us, with four 1,440). That goes by
// the sequence's own rows, and a block of keys goes to the wave of its number in the sequence, so that neither what shares
// a step nor a tile changes a sum's order.
// A row takes nothing from keys it does not see, whatever they hold; but 0 times an infinity is no number, and the tile's rows
// share the products. A tile with a result that is not finite is therefore made again row by row, as in the kernel above.
// Head sizes in multiples of 16 up to 256, pages of a multiple of 4 keys; other sizes keep the kernel above.
// The keys and values of a wave's next block are on their way while one is multiplied (asked for together, under no branch: heads of
// 32, 64 and 128, FULL, have instances of their own): prompts of 93 and 261 tokens and 6 more tokens of each at the 4B size 56.6 -> 54.5 ms,
// 252 launches, most of them two tokens behind some 300 keys.
#define F32_FEW_ROWS 64
template <int ND, int W, bool FULL>
__global__ __launch_bounds__(64 * W) void attention_f32_tile_kernel(AttnArgs a) {
  __shared__ __align__(16) f32x4_t hand[W > 1 ? W / 2 : 1][ND * 64];  // accumulators on their way from wave to wave
  __shared__ float hand_m[W][16], hand_l[W][16];
  __shared__ int odd;  // whether a result is not finite
  const int lane = threadIdx.x & 63, wave = uniform_wave_number();
  const int r = lane & 15, q = lane >> 4;
  const int s = blockIdx.z, kvh = blockIdx.y, g = a.nq / a.nkv;
  const int t0 = a.cu_q[s], rows = (a.cu_q[s + 1] - t0) * g, row0 = blockIdx.x * 16;
  if (row0 >= rows || (ND < 16 && (rows <= F32_FEW_ROWS) != (W == 8))) return;  // the whole block alike
  const int D = a.head_dim, Dv = a.value_dim, ps = a.page_size, nd = D >> 4, nv = Dv >> 4;
  const int last_row = min(row0 + 15, rows - 1), rr = min(row0 + r, last_row);
  const int t = t0 + rr / g, h = kvh * g + rr % g;
  const int pos = a.positions[t], hi = a.positions[t0 + last_row / g], pos0 = a.positions[t0 + row0 / g];
  const int* table = a.block_table + (size_t)s * a.table_width;
  const int lo = a.window > 0 ? max(0, pos - a.window + 1) : (a.chunk > 0 ? pos - pos % a.chunk : 0);
  const int lo0 = a.window > 0 ? max(0, pos0 - a.window + 1) : (a.chunk > 0 ? pos0 - pos0 % a.chunk : 0);
  const int keep = a.window > 0 ? a.keep_first : 0;
  // blocks of 16 keys: the kept first ones that lie before the window's, then from the first row's first key on
  const int main0 = __builtin_amdgcn_readfirstlane(lo0 >> 4), kept = min((keep + 15) >> 4, main0);
  const int last_block = __builtin_amdgcn_readfirstlane(hi >> 4);

  f32x4_t qv[ND], acc[ND];
  const float* qr = (const float*)a.q + ((size_t)t * a.nq + h) * D + 4 * q;
#pragma unroll
  for (int j = 0; j < ND; ++j) {
    if (FULL || j < nd) qv[j] = *(const f32x4_t*)(qr + 16 * j);
    acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  float m = -INFINITY, l = 0.f;
  const float* kc = (const float*)a.k_cache;
  const float* vc = (const float*)a.v_cache;
  // K: the lane's key j0 + r; V: its keys j0 + 4 q .. + 3 (one page). Places after the last key, and pages
  // that were given back, are read as the sequence's last key (its page is there) and count for nothing
  const int last_page = table[hi / ps];
  auto key_row = [&](int b) {
    const int kj = min(16 * b + r, hi);
    int kp = table[kj / ps];
    kp = kp < 0 ? last_page : kp;
    return kc + (((size_t)kp * a.nkv + kvh) * ps + kj % ps) * D + 4 * q;
  };
  auto value_row = [&](int b, bool& there) {
    const int vj = 16 * b + 4 * q;
    int vp = table[min(vj, hi) / ps];
    there = vj <= hi && vp >= 0;
    vp = there ? vp : last_page;
    return vc + ((size_t)vp * a.nkv + kvh) * Dv * ps + (there ? vj % ps : 0) + (FULL ? (size_t)r * ps : 0);
  };
  struct Block { f32x4_t k[ND], v[ND]; bool v_there; };
  auto load = [&](int b, Block& blk) {
    const float* kr = key_row(b);
    const float* vr = value_row(b, blk.v_there);
#pragma unroll
    for (int j = 0; j < ND; ++j) blk.k[j] = *(const f32x4_t*)(kr + 16 * j);
#pragma unroll
    for (int j = 0; j < ND; ++j) blk.v[j] = *(const f32x4_t*)(vr + (size_t)(16 * j) * ps);
  };
  // a wave's blocks are those of its number modulo W
  auto after = [&](int b) { return b + W < kept || b >= main0 ? b + W : main0 + ((wave - main0) & (W - 1)); };
  int b = wave < kept ? wave : main0 + ((wave - main0) & (W - 1));
  Block now, next;
  if (FULL && b <= last_block) load(b, now);
  while (b <= last_block) {
    const int j0 = 16 * b, vj = j0 + 4 * q, b_next = after(b);
    const float *kr = nullptr, *vr = nullptr;
    if (FULL) {
      load(min(b_next, last_block), next);  // behind the wave's last block: one that nobody needs
    } else {  // the block's page numbers together: one round trip
      kr = key_row(b);
      vr = value_row(b, now.v_there);
    }
    f32x4_t sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < ND; ++j)
      if (FULL || j < nd) {
        const f32x4_t kv = FULL ? now.k[j] : *(const f32x4_t*)(kr + 16 * j);
#pragma unroll
        for (int c = 0; c < 4; ++c) sc = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[c], qv[j][c], sc, 0, 0, 0);
      }
    float mx = m;
    bool seen[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int j = j0 + 4 * q + e;
      sc[e] *= a.scale;
      if (a.softcap > 0.f) sc[e] = a.softcap * tanhf(sc[e] / a.softcap);
      seen[e] = j <= pos && (j >= lo || j < keep);
      if (seen[e]) mx = fmaxf(mx, sc[e]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    if (mx > -INFINITY) {  // false only for rows that have seen no key yet
      const float corr = expf(m - mx);
      l *= corr;
#pragma unroll
      for (int j = 0; j < ND; ++j) acc[j] *= corr;
      m = mx;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      sc[e] = seen[e] ? expf(sc[e] - m) : 0.f;
      l += sc[e];
    }
#pragma unroll
    for (int j = 0; j < ND; ++j)
      if (FULL || j < nv) {
        const f32x4_t vv = FULL ? now.v[j] : *(const f32x4_t*)(vr + (size_t)(16 * j + r) * ps);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float value = (now.v_there && vj + e <= hi) ? vv[e] : 0.f;  // never written: not a number, perhaps
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(value, sc[e], acc[j], 0, 0, 0);
        }
      }
    if (FULL) now = next;
    b = b_next;
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  // waves that had a block: of a sequence of few keys the first ones alone, and there is nothing to add from the others
  // (one token behind 5 keys, 32 heads of 128 on 8, launched in a row: 10.5 us, with all eight 14.4)
  const int busy = main0 == 0 ? min(last_block + 1, W) : W;
  if (W > 1 && busy > 1) {
    if (q == 0) {
      hand_m[wave][r] = m;
      hand_l[wave][r] = l;
    }
    __syncthreads();
    float top = -INFINITY, sum = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) top = w < busy ? fmaxf(top, hand_m[w][r]) : top;
#pragma unroll
    for (int w = 0; w < W; ++w)
      if (w < busy) sum += hand_m[w][r] > -INFINITY ? hand_l[w][r] * expf(hand_m[w][r] - top) : 0.f;
    const float corr = m > -INFINITY ? expf(m - top) : 0.f;
#pragma unroll
    for (int j = 0; j < ND; ++j) acc[j] *= corr;
    m = top;
    l = sum;
#pragma unroll
    for (int half = W / 2; half > 0; half >>= 1) {
      if (half >= busy) continue;  // the whole block alike
      if (wave >= half && wave < min(2 * half, busy))
#pragma unroll
        for (int j = 0; j < ND; ++j) hand[wave - half][j * 64 + lane] = acc[j];
      __syncthreads();
      if (wave < half && wave + half < busy)
#pragma unroll
        for (int j = 0; j < ND; ++j) acc[j] += hand[wave][j * 64 + lane];
      __syncthreads();
    }
  }
  if (a.sink) {  // a key of score 0 without a value
    const float top = fmaxf(m, 0.f), corr = m > -INFINITY ? expf(m - top) : 0.f;
    l = l * corr + expf(-top);
#pragma unroll
    for (int j = 0; j < ND; ++j) acc[j] *= corr;
  }
  // rows into LDS in order, then out with the block's threads (a turned value's partner lies half a row away)
  float* out_rows = (float*)hand;
  if (threadIdx.x == 0) odd = 0;
  if (wave == 0) {
    const float inv = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
    for (int j = 0; j < ND; ++j)
      if (j < nv) *(f32x4_t*)(out_rows + r * Dv + 16 * j + 4 * q) = acc[j] * inv;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < (last_row - row0 + 1) * Dv; i += 64 * W)
    if (!(fabsf(out_rows[i]) < INFINITY)) odd = 1;
  __syncthreads();
  if (odd) {
    for (int i = row0 + wave; i <= last_row; i += W) attend_row<float, 16 * ND>(a, t0 + i / g, kvh * g + i % g, out_rows + 16 * ND * wave);
    return;
  }
  for (int i = threadIdx.x; i < (last_row - row0 + 1) * Dv; i += 64 * W) {
    const int ri = row0 + i / Dv, d = i % Dv, ti = t0 + ri / g, hq = kvh * g + ri % g;
    float v = out_rows[i];
    if (a.turn) {
      const float* angles = a.turn + (size_t)ti * Dv;
      const int half = Dv >> 1, j = d < half ? d : d - half;
      const float p = out_rows[d < half ? i + half : i - half], c = angles[j], sn = angles[half + j];
      v = d < half ? v * c + p * sn : v * c - p * sn;
    }
    if (a.gate) v *= 1.0f / (1.0f + expf(-((const float*)a.gate)[(size_t)ti * a.gate_stride + (size_t)hq * Dv + d]));
    ((float*)a.out)[((size_t)ti * a.nq + hq) * Dv + d] = v;
  }
}

template <int ND>
static void attention_f32_tiles(const AttnArgs& a, hipStream_t stream) {
  const long g = a.nq / a.nkv;
  const auto grid = [&](long rows) { return dim3((unsigned)((rows + 15) / 16), a.nkv, a.num_seqs); };
  const auto launch = [&](auto full) {
    constexpr bool FULL = decltype(full)::value;
    if constexpr (ND >= 16) {
      attention_f32_tile_kernel<ND, 8, FULL><<<grid(a.max_q_len * g), 512, 0, stream>>>(a);
    } else {  // sequences of both kinds: both kernels, each leaves the other's alone
      if (a.min_q_len * g <= F32_FEW_ROWS) attention_f32_tile_kernel<ND, 8, FULL><<<grid(min(a.max_q_len * g, (long)F32_FEW_ROWS)), 512, 0, stream>>>(a);
      if (a.max_q_len * g > F32_FEW_ROWS) attention_f32_tile_kernel<ND, 4, FULL><<<grid(a.max_q_len * g), 256, 0, stream>>>(a);
    }
  };
  if (ND <= 8 && a.head_dim == 16 * ND && a.value_dim == 16 * ND) launch(std::bool_constant<(ND <= 8)>{});
  else launch(std::false_type{});
}

extern "C" int qrt_attention_f32(const AttnArgs* args, int dtype, hipStream_t stream) {
  AttnArgs a = *args;
  QRT_CHECK(a.num_tokens >= 0 && a.nq > 0 && a.nkv > 0 && a.nq % a.nkv == 0,
            "attention: %d query heads do not divide into %d key heads", a.nq, a.nkv);
  QRT_CHECK(a.head_dim > 0 && a.head_dim <= MAX_D, "attention: head size %d is above %d", a.head_dim, MAX_D);
  QRT_CHECK(a.page_size > 0 && a.table_width > 0 && a.window >= 0, "attention: bad page size, table width or window");
  if (a.value_dim == 0) a.value_dim = a.head_dim;
  QRT_CHECK(a.value_dim > 0 && a.value_dim <= MAX_D, "attention: value size %d is above %d", a.value_dim, MAX_D);
  QRT_CHECK(a.chunk >= 0 && !(a.chunk > 0 && a.window > 0), "attention: a window or a chunk size, not both");
  QRT_CHECK(a.softcap >= 0.f, "attention: negative score cap");
  QRT_CHECK(a.keep_first >= 0 && (a.keep_first == 0 || a.window > 0), "attention: first keys are kept beside a window");
  QRT_CHECK(!a.turn || a.value_dim % 2 == 0, "attention: turned values of odd size %d", a.value_dim);
  QRT_CHECK(a.nq <= 65535, "attention: too many heads");
  if (a.num_tokens == 0) return 0;
  const int widest = a.head_dim > a.value_dim ? a.head_dim : a.value_dim;
  if (dtype == QRT_F32 && a.cu_q && a.head_dim % 16 == 0 && a.value_dim % 16 == 0 && widest <= 256 && a.page_size % 4 == 0 &&
      a.num_seqs <= 65535 && a.nkv <= 65535 && a.max_q_len > 0 &&
      ((uintptr_t)a.q | (uintptr_t)a.k_cache | (uintptr_t)a.v_cache) % 16 == 0) {
    if (widest <= 32) attention_f32_tiles<2>(a, stream);
    else if (widest <= 64) attention_f32_tiles<4>(a, stream);
    else if (widest <= 128) attention_f32_tiles<8>(a, stream);
    else attention_f32_tiles<16>(a, stream);
    QRT_LAUNCH_CHECK("attention_f32_tiles");
    return 0;
  }
  dim3 grid(a.num_tokens, a.nq), block(64);
  if (dtype == QRT_F32) attention_f32_kernel<float><<<grid, block, 0, stream>>>(a);
  else if (dtype == QRT_BF16) attention_f32_kernel<bf16_t><<<grid, block, 0, stream>>>(a);
  else return qrt_fail("attention: unknown dtype %d", dtype);
  QRT_LAUNCH_CHECK("attention_f32");
  return 0;
}
