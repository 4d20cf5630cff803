// Tiles of bfloat16 products through LDS: the loop over K that the products of many rows share.
//
// A block makes a tile of BM x BN from stages of 64 columns of K. Both operands come by direct
// loads: a unit is 8 rows x 128 bytes, whole cache lines, and lies in LDS with piece c (16 bytes) of
// row r at 128 r + 16 (c ^ (r & 7)), so that the operand reads (row lane & 15, piece 4 h + lane / 16
// for k-step h of the stage) touch every bank once. S stages are in flight in a ring. What bounds it:
//   - LDS and the vector memory pipe rather than the matrix cores: a compute unit takes a line
//     (64 bytes) a cycle, so a tile of 128 x 160 wants nine tenths of that at full MFMA rate and one
//     of 256 x 160 two thirds; large tiles win where there are enough of them for 256 compute units;
//   - the memory's latency: two stages in flight behind the one in use (S = 3, some 100 KB a compute
//     unit) load at 20 TB/s out of the L2s, one (S = 2) at 13. That is why 256 x 160 with three
//     stages beats 256 x 256 with two (the 4B gate/up product at 2,048 rows: 187 us against 221),
//     and why rows of 32 columns with twice the stages do not pay (half lines: 224);
//   - instructions between the MFMAs: offsets of a buffer load sit in one register a unit and one
//     scalar a stage, so a load costs the wave two instructions (a 64-bit address and a branch a
//     load: 216 us against 200 for 4,096 x 4,096 x 8,192).
// Eight waves (two a SIMD) fill each other's waits; four waves with twice the tile each have the same
// MFMAs and fewer operand reads, but stand still at every load they issue (258 against 211 us).
// A stage's two k-steps are two phases: operands of the next k-step leave LDS between the rows of
// products of this one; half of a stage's loads are issued in the second phase, behind the one
// barrier a stage needs, and half in the first phase of the next stage, where S allows it.
#pragma once
#include "common.h"
#include "direct.h"
#include <type_traits>

// The upper half of the lanes of g changes places with the lower half of u.
__device__ __forceinline__ void swap_halves(float& g, float& u) {
  typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));
  const u32x2_t v = __builtin_amdgcn_permlane32_swap(__float_as_uint(g), __float_as_uint(u), false, false);
  g = __uint_as_float(v[0]);
  u = __uint_as_float(v[1]);
}

// Four times gated_act of common.h, for results that are rounded to bfloat16 at once. A tile of 256 x 160 forms 40 of them
// a lane at its end, where the matrix cores wait: with expf and an IEEE division that is some 31 issues each, here 19 (the
// 4B gate/up product at 2,048 rows 195 -> 188 us when it was taken). The exponential is the hardware's power of two of a
// product whose rounding error is made good to first order, the quotient the product with the hardware's reciprocal and one step
// that makes good what this leaves of g. That holds while everything on the way is a normal number; where the exponential's argument is
// beyond 87 in size, or NaN, the result is gated_act's own, element by element: none depends on its neighbours. Against
// float64, in 2^-24 of the result, largest and rms over four million gates within 8: 3.6 and 0.83 (gated_act 3.3 and 0.79),
// within 87: 4.2 and 0.71 (3.5 and 0.65); rounded to bfloat16, the two rms errors are the same to ten digits.
template <bool CLAMPED>
__device__ __forceinline__ void gated_act4_of(const float (&g)[4], const float (&u)[4], float limit, float (&o)[4]) {
  constexpr float LOG2E = 1.44269502f, LOG2E_REST = 1.92596299e-8f, LN2 = 0.693147181f, FAR = 87.0f;
  float x[4];
  bool far = false;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float gr = CLAMPED ? fminf(g[r], limit) : g[r];
    const float ur = CLAMPED ? fminf(fmaxf(u[r], -limit), limit) + 1.0f : u[r];
    x[r] = CLAMPED ? -1.702f * gr : -gr;
    far |= !(fabsf(x[r]) <= FAR);
    const float t = x[r] * LOG2E, rest = fmaf(x[r], LOG2E_REST, fmaf(x[r], LOG2E, -t));
    const float e = __builtin_amdgcn_exp2f(t);
    const float d = 1.0f + fmaf(e, rest * LN2, e), by = __builtin_amdgcn_rcpf(d);
    const float q = gr * by;
    o[r] = fmaf(fmaf(-d, q, gr), by, q) * ur;
  }
  if (__builtin_amdgcn_ballot_w64(far) != 0) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (!(fabsf(x[r]) <= FAR)) o[r] = gated_act(g[r], u[r], CLAMPED ? QRT_ACT_CLAMPED : QRT_ACT_SWIGLU, limit);
  }
}
__device__ __forceinline__ void gated_act4(const float (&g)[4], const float (&u)[4], int kind, float limit, float (&o)[4]) {
  if (kind == QRT_ACT_CLAMPED) gated_act4_of<true>(g, u, limit, o);
  else gated_act4_of<false>(g, u, limit, o);
}

// WM x WN waves, each with BM / WM rows and BN / WN columns of the tile, S stages in flight.
template <int BM, int BN, int WM, int WN, int S>
struct Tile {
  static constexpr int WAVES = WM * WN, TM = BM / WM / 16, TN = BN / WN / 16;
  static constexpr int AU = BM / 8, WU = BN / 8;  // units of a stage; where they are no multiple of the waves, the last is loaded twice
  static constexpr int AL = (AU + WAVES - 1) / WAVES, WL = (WU + WAVES - 1) / WAVES, LOADS = AL + WL;
  static constexpr int STAGE = (BM + BN) * 128;
  static constexpr size_t RING = (size_t)S * STAGE;
  static_assert(BM % (16 * WM) == 0 && BN % (16 * WN) == 0, "waves own whole MFMA tiles");
  static_assert(S >= 2 && (S - 1) * LOADS < 64, "the loads' counter holds 63");
  static_assert(RING <= 160 * 1024, "the ring of this tile does not fit LDS");

  // the row of the tile (of its weights) that load j of this lane brings 16 bytes of, and which 16 of a stage's 128
  static __device__ __forceinline__ int row_of(int j, int units, int wave, int lane) {
    return 8 * min(wave + WAVES * j, units - 1) + (lane >> 3);
  }
  static __device__ __forceinline__ unsigned piece_of(int lane) { return 16 * ((lane & 7) ^ (lane >> 3)); }

#ifdef __HIP_DEVICE_COMPILE__  // the host's compiler knows no buffer resources
  static __device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer(const void* p, size_t bytes) {
    constexpr int RAW = 0x00020000;  // a buffer of bytes
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)bytes, RAW);
  }

  // POLICY: the cache policy of the weights' loads (2: non-temporal, for weights that no other block reads).
  // Load j of the stage that begins at byte `at` of every row, into the slot that begins at `dst`. aoff, woff: where each
  // load of this lane begins, in bytes from its buffer, without the stage's.
  template <int POLICY>
  static __device__ __forceinline__ void fetch_one(const __amdgpu_buffer_rsrc_t a_buf, const __amdgpu_buffer_rsrc_t w_buf,
                                                   const unsigned (&aoff)[AL], const unsigned (&woff)[WL], int at,
                                                   unsigned char* dst, int j, int wave) {
    if (j < AL) {
      const int unit = AU % WAVES && j == AL - 1 ? min(wave + WAVES * j, AU - 1) : wave + WAVES * j;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_buf, (lds_ptr_t)(dst + unit * 1024), 16, aoff[j], at, 0, 0);
    } else {
      const int unit = WU % WAVES && j == LOADS - 1 ? min(wave + WAVES * (j - AL), WU - 1) : wave + WAVES * (j - AL);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(w_buf, (lds_ptr_t)(dst + (AU + unit) * 1024), 16, woff[j - AL], at, 0, POLICY);
    }
  }
  // stages `from` to `to` - 1 of a tile of `stages`, each into the slot of its number
  template <int POLICY = 0>
  static __device__ __forceinline__ void fetch_first(const __amdgpu_buffer_rsrc_t a_buf, const __amdgpu_buffer_rsrc_t w_buf,
                                                     const unsigned (&aoff)[AL], const unsigned (&woff)[WL], int s0, int stages,
                                                     unsigned char* lds, int from, int to) {
    const int wave = uniform_wave_number();
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (s >= from && s < to && s < stages) {
#pragma unroll
        for (int j = 0; j < LOADS; ++j) fetch_one<POLICY>(a_buf, w_buf, aoff, woff, (s0 + s) * 128, lds + s * STAGE, j, wave);
      }
  }

  // acc[i][j] of a wave, from zero: row 16 i + (lane & 15) of its rows, rows 16 j + 4 (lane / 16) + 0..3 of its
  // weights. `fetched`: how many first stages have been asked for already; whatever else the wave has on its way to memory
  // since (stores) only makes the waits longer, since loads land in order.
  template <int POLICY = 0>
  static __device__ __forceinline__ void products(const __amdgpu_buffer_rsrc_t a_buf, const __amdgpu_buffer_rsrc_t w_buf,
                                                  const unsigned (&aoff)[AL], const unsigned (&woff)[WL], int s0, int stages,
                                                  unsigned char* lds, int fetched, f32x4_t (&acc)[TM][TN]) {
    const int lane = threadIdx.x & 63, wave = uniform_wave_number();
    const int wm = wave / WN, wn = wave % WN, r16 = lane & 15, quad = lane >> 4;
    auto stage_at = [&](int it) { return (s0 + it) * 128; };

#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    const int read_at[2] = {r16 * 128 + 16 * (quad ^ (r16 & 7)), r16 * 128 + 16 * ((4 + quad) ^ (r16 & 7))};
    const int a_at = wm * (BM / WM) * 128, w_at = (BM + wn * (BN / WN)) * 128;
    bf16x8_t a[2][TM], w[2][TN];
    constexpr int READS = TM + TN;
    auto read_one = [&](int slot, int h, int r) {  // operand r of k-step h: first the weights', then the activations'
      const unsigned char* src = lds + slot * STAGE + read_at[h];
      if (r < TN) w[h][r] = *(const bf16x8_t*)(src + w_at + r * 2048);
      else a[h][r - TN] = *(const bf16x8_t*)(src + a_at + (r - TN) * 2048);
    };
    auto row_of_products = [&](int h, int i) {
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[h][j], a[h][i], acc[i][j], 0, 0, 0);
    };
    // operands of the next k-step asked for behind each row of products, none behind the last
    constexpr int READS_A_ROW = TM > 1 ? (READS + TM - 2) / (TM - 1) : READS;
    // of a stage's loads, those that are left to the next stage's first phase
    constexpr int LATE = S >= 3 ? LOADS / 2 : 0, SOON = LOADS - LATE;
    constexpr int SOON_A_ROW = (SOON + TM - 1) / TM, LATE_A_ROW = (LATE + TM - 1) / TM;

    // Stage `it`, whose first operands are in registers, from `slot`; `before` and `next` are the slots of its
    // neighbours. MORE: a stage `it + S` follows. Loads land in the order of issue, so stage it + 1 has landed
    // when at most the S - 2 stages issued behind it are on their way. The barrier says that this holds for
    // every wave's share, and that every wave has this stage's last operands in registers: its slot is free.
    auto step = [&](int it, int slot, int before, int next, auto follows) {
      constexpr bool MORE = decltype(follows)::value;
      const bool owed = LATE > 0 && it > 0 && it - 1 + S < stages;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        row_of_products(0, i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = i * READS_A_ROW; r < (i + 1) * READS_A_ROW && r < READS; ++r) read_one(slot, 1, r);
        if (owed) {
#pragma unroll
          for (int j = i * LATE_A_ROW; j < (i + 1) * LATE_A_ROW && j < LATE; ++j)
            fetch_one<POLICY>(a_buf, w_buf, aoff, woff, stage_at(it - 1 + S), lds + before * STAGE, SOON + j, wave);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (MORE || it - 1 + S < stages) QRT_WAIT_LOADS((S - 2) * LOADS);
      else QRT_WAIT_LOADS(0);
      QRT_WAIT_LDS();
      QRT_BARRIER();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        row_of_products(1, i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = i * READS_A_ROW; r < (i + 1) * READS_A_ROW && r < READS; ++r) read_one(next, 0, r);
        if (MORE) {
#pragma unroll
          for (int j = i * SOON_A_ROW; j < (i + 1) * SOON_A_ROW && j < SOON; ++j)
            fetch_one<POLICY>(a_buf, w_buf, aoff, woff, stage_at(it + S), lds + slot * STAGE, j, wave);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };

    if (stages > 0) {  // the same in every wave of the block
      fetch_first<POLICY>(a_buf, w_buf, aoff, woff, s0, stages, lds, fetched, S);
      if (stages >= S) QRT_WAIT_LOADS((S - 1) * LOADS);
      else QRT_WAIT_LOADS(0);
      QRT_BARRIER();
#pragma unroll
      for (int r = 0; r < READS; ++r) read_one(0, 0, r);
      int slot = 0, before = 0, it = 0;
      auto walk = [&](int end, auto follows) {
        for (; it < end; ++it) {
          const int next = slot + 1 == S ? 0 : slot + 1;
          step(it, slot, before, next, follows);  // behind the last stage it reads a slot that nobody needs
          before = slot;
          slot = next;
        }
      };
      walk(stages - S, std::true_type{});
      walk(stages, std::false_type{});
    }
  }
#endif
};
