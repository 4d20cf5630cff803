// Recurrences of linear attention with one decay per head, float32.
//
//   S <- d S + k v^T;   o = S^T q                (S [dim, vdim] per sequence and head)
//
// Retention: d is a constant of the head. State-space form (STEP): a step size per token and head,
// D = softplus(logit + bias), makes both the decay d = exp(-exp(a_log) D) and the written value v = D x,
// the read-out has a skip, o = S^T q + skip x, and neighbouring heads share keys and queries (head h has
// those of h / share).
// Matrix memory (GATES): what a token keeps of the state and what its write weighs come per token and
// head as logarithms, and the state has one more column, whose value is always 1: the sum of the weighted
// keys, whose read-out goes to a place of its own.
//
// over each sequence's tokens of the step, from the state in the sequence's slot, which is left
// there for the next step: [slots, heads, vdim, dim], a value channel's column of S contiguous.
// q, k, v come as float32 [T, 2 heads dim + heads vdim] (queries, keys, values; rotated and
// scaled by whoever made them). A block of 256 threads owns 16 columns of one head's state for
// one sequence; 16 neighbouring lanes share a column, each holding its rows in registers four
// neighbours at a time (rows 4 (lane + 16 g) .. + 3 of group g), so that state, keys and queries
// move 16 bytes a lane and the sum over rows that a read-out needs ends in a DPP sum inside a row
// of 16 lanes. Tokens are staged through LDS 16 at a time; the next tile's global loads are in
// flight while a tile is walked, the walk has no global access and no branch between tokens, and
// the tile's read-outs leave together afterwards. The order of the float32 operations per token
// does not depend on how the tokens are cut into steps, tiles or batches. (Retention over long spans goes
// by chunks instead: see retention_chunk_kernel.)
#include "common.h"
#include <math.h>
#include <type_traits>

struct RetentionArgs {
  const void* qkv;        // [T, channels] float32, or (STEP) bfloat16
  int channels, q_first, k_first, v_first;
  const float* decay;     // [heads]
  float* state;           // [slots, heads, vdim, dim]
  float* out;             // [T, heads, vdim]
  const int* cu_q; const int* state_slots;
  int heads, dim, vdim;
  int share;              // heads that have one key and query in common (1: each its own)
  const void* step; long step_stride; int step_code;   // [T, heads] step logits, float32 or bfloat16; null: retention
  const float* step_bias; const float* a_log; const float* skip;  // [heads]
  int qkv_code;
  const int* seq_ids;     // the sequences of this launch; null: all of the step's
  const float* gates;     // [T, 3, heads] (GATES): log keep, log write (a third row is not read here)
  float* last_out;        // [T, heads] (GATES): the read-out of the state's last column
  // Retention: sequences of at least `chunk_from` tokens go by chunks (0: none does). It goes by the sequence's own
  // tokens, not the step's, so that a request's results do not depend on what shares its step. `shortest`, `longest`:
  // bounds of the step's lengths, as the caller knows them, that say whether a form has any work.
  int chunk_from, shortest, longest;
};

constexpr int RT_CONSTANT = 0, RT_STEP = 1, RT_GATES = 2;  // where decays and writes come from

#define RT_COLS 16   // columns of the state per block

// the sum over the 16 lanes of a row (every lane gets it)
__device__ __forceinline__ float row16_sum(float x) {
  int v = __builtin_bit_cast(int, x);
  x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, true));   // quad_perm [1,0,3,2]
  v = __builtin_bit_cast(int, x);
  x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, true));   // quad_perm [2,3,0,1]
  v = __builtin_bit_cast(int, x);
  x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, true));  // row_half_mirror
  v = __builtin_bit_cast(int, x);
  x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, v, 0x140, 0xF, 0xF, true));  // row_mirror
  return x;
}

// G groups of four rows a lane: heads of up to 64 G key elements (padded with zero rows). RT_TILE
// tokens a tile: 16 (8 for the widest heads: what fits 64 KB), or 4 for steps of single tokens,
// whose blocks then are all resident at once with a quarter of the LDS and of the loads.
template <int G, int RT_TILE, int MODE, typename TI>
__global__ __launch_bounds__(256) void retention_kernel(RetentionArgs a) {
  constexpr bool STEP = MODE == RT_STEP, GATES = MODE == RT_GATES, PER_TOKEN = STEP || GATES;
  constexpr int DP = 64 * G;                          // rows staged
  constexpr int NQK = 2 * RT_TILE * DP / 256;         // q and k elements a thread fetches per tile
  __shared__ __attribute__((aligned(16))) float qs[RT_TILE * DP];
  __shared__ __attribute__((aligned(16))) float ks[RT_TILE * DP];
  __shared__ float vs[RT_TILE * RT_COLS];
  __shared__ float os[RT_TILE * RT_COLS];
  __shared__ float ds[RT_TILE], steps[RT_TILE];  // a token's decay and what its value is multiplied by (PER_TOKEN)
  const int seq = a.seq_ids ? a.seq_ids[blockIdx.x] : blockIdx.x, head = blockIdx.y, col0 = blockIdx.z * RT_COLS;
  const int t0 = a.cu_q[seq], t1 = a.cu_q[seq + 1];
  if (t1 <= t0 || (!PER_TOKEN && a.chunk_from > 0 && t1 - t0 >= a.chunk_from)) return;
  const int dim = a.dim, vdim = a.vdim;
  const int cols = GATES ? vdim + 1 : vdim;  // columns of the state
  const TI* qkv = (const TI*)a.qkv;
  const int sub = threadIdx.x & 15, colg = threadIdx.x >> 4;  // lane within its column, column of the block
  const int col = col0 + colg;
  const bool col_ok = col < cols;
  const float decay = PER_TOKEN ? 0.f : a.decay[head];
  const float rate = STEP ? expf(a.a_log[head]) : 0.f, bias = STEP ? a.step_bias[head] : 0.f, skip = STEP ? a.skip[head] : 0.f;
  const int qk_head = head / a.share;
  float* st = a.state + (((size_t)a.state_slots[seq] * a.heads + head) * cols + min(col, cols - 1)) * dim;
  const bool vec = (dim & 3) == 0;  // a lane's four rows are 16 aligned bytes of the column
  float s[G][4];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int d = 4 * (sub + 16 * g);
    if (vec && d < dim && col_ok) {
      const float4 x = *(const float4*)(st + d);
      s[g][0] = x.x; s[g][1] = x.y; s[g][2] = x.z; s[g][3] = x.w;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) s[g][j] = (d + j < dim && col_ok) ? st[d + j] : 0.f;
    }
  }
  // what this thread fetches of a tile: elements threadIdx.x + 256 i of q | k ([which][token][row]), one of v
  float pre[NQK], pre_v, pre_step = 0.f, pre_write = 0.f;
  auto fetch = [&](int base) {
    const int n = min(RT_TILE, t1 - base);
#pragma unroll
    for (int i = 0; i < NQK; ++i) {
      const int e = threadIdx.x + 256 * i;
      const int which = e / (RT_TILE * DP), tok = (e / DP) % RT_TILE, d = e % DP;
      const bool ok = tok < n && d < dim;
      const TI* row = qkv + (size_t)(base + min(tok, n - 1)) * a.channels + (which ? a.k_first : a.q_first) + qk_head * dim;
      pre[i] = ok ? to_f32<TI>(row[d]) : 0.f;
    }
    const int tok = min((int)threadIdx.x / RT_COLS, RT_TILE - 1), c = threadIdx.x % RT_COLS;
    if (STEP && (int)threadIdx.x < n) {
      const size_t at = (size_t)(base + threadIdx.x) * a.step_stride + head;
      pre_step = a.step_code == QRT_F32 ? ((const float*)a.step)[at] : (float)((const bf16_t*)a.step)[at];
    }
    if (GATES && (int)threadIdx.x < n) {
      const float* row = a.gates + (size_t)(base + threadIdx.x) * 3 * a.heads + head;
      pre_step = row[0];
      pre_write = row[a.heads];
    }
    pre_v = GATES && col0 + c == vdim ? 1.f : (tok < n && col0 + c < vdim) ? to_f32<TI>(qkv[(size_t)(base + tok) * a.channels + a.v_first + head * vdim + col0 + c]) : 0.f;
  };
  fetch(t0);
  for (int base = t0; base < t1; base += RT_TILE) {
    const int n = min(RT_TILE, t1 - base);
    __syncthreads();  // the tile before has been walked and its read-outs have left
#pragma unroll
    for (int i = 0; i < NQK; ++i) {
      const int e = threadIdx.x + 256 * i;
      if (e < RT_TILE * DP) qs[e] = pre[i];
      else ks[e - RT_TILE * DP] = pre[i];
    }
    if (threadIdx.x < RT_TILE * RT_COLS) vs[threadIdx.x] = pre_v;
    if (STEP && threadIdx.x < RT_TILE) {
      const float z = pre_step + bias;
      const float sp = z > 20.f ? z : log1pf(expf(z));
      steps[threadIdx.x] = sp;
      ds[threadIdx.x] = expf(-rate * sp);
    }
    if (GATES && threadIdx.x < RT_TILE) {
      ds[threadIdx.x] = expf(pre_step);
      steps[threadIdx.x] = expf(pre_write);
    }
    __syncthreads();
    if (base + RT_TILE < t1) fetch(base + RT_TILE);  // on its way during the walk
    auto token = [&](int i) {
      const float x = vs[i * RT_COLS + colg];
      const float d = PER_TOKEN ? ds[i] : decay, v = PER_TOKEN ? x * steps[i] : x;
      float acc = 0.f;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const float4 kd = *(const float4*)(ks + i * DP + 4 * (sub + 16 * g));
        const float4 qd = *(const float4*)(qs + i * DP + 4 * (sub + 16 * g));
        s[g][0] = fmaf(d, s[g][0], kd.x * v); acc = fmaf(s[g][0], qd.x, acc);
        s[g][1] = fmaf(d, s[g][1], kd.y * v); acc = fmaf(s[g][1], qd.y, acc);
        s[g][2] = fmaf(d, s[g][2], kd.z * v); acc = fmaf(s[g][2], qd.z, acc);
        s[g][3] = fmaf(d, s[g][3], kd.w * v); acc = fmaf(s[g][3], qd.w, acc);
      }
      acc = row16_sum(acc);
      if (STEP) acc = fmaf(skip, x, acc);
      if (sub == 0) os[i * RT_COLS + colg] = acc;
    };
    if (n == RT_TILE) {
#pragma unroll 4
      for (int i = 0; i < RT_TILE; ++i) token(i);
    } else {
      for (int i = 0; i < n; ++i) token(i);
    }
    __syncthreads();
    {  // the tile's read-outs: thread (token, column)
      const int tok = threadIdx.x / RT_COLS, c = threadIdx.x % RT_COLS;
      if (tok < n && tok < RT_TILE && col0 + c < vdim) a.out[((size_t)(base + tok) * a.heads + head) * vdim + col0 + c] = os[threadIdx.x];
      if (GATES && tok < n && tok < RT_TILE && col0 + c == vdim) a.last_out[(size_t)(base + tok) * a.heads + head] = os[threadIdx.x];
    }
  }
  if (col_ok) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int d = 4 * (sub + 16 * g);
      if (vec && d < dim) {
        *(float4*)(st + d) = make_float4(s[g][0], s[g][1], s[g][2], s[g][3]);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (d + j < dim) st[d + j] = s[g][j];
      }
    }
  }
}

// Prompts under a constant decay, in chunks of 32 tokens on float32 MFMA. With S the state in front of the
// chunk, i and j tokens of the chunk and n how many it has:
//
//   o_i = d^(i+1) S^T q_i + sum over j <= i of d^(i-j) (k_j . q_i) v_j
//   S  <- d^n S + sum over j of d^(n-1-j) k_j v_j^T
//
// Walked token by token the recurrence was bound by its chain: one wave a SIMD, 187 ns a token (32 heads of 128 x
// 128, 2,047 tokens: 386 us). In chunks that case takes 155 us, 2.4 us a chunk, of which 1.1 are matrix products and the
// rest the way from LDS through them and back to it (4 heads of 32: 315 -> 116; 16 of 256: 590 -> 257).
// Error against 64 bits of the same case: 1.1e-7 to 1.4e-7 by the head's decay, walked 1.1e-7 to 3.9e-7.
// A block owns 16 columns of one head's state, as above; each of its NW waves owns 16 G of the state's rows
// in accumulators, and because all of o is linear in the sums over rows, a wave carries its share of both terms
// through to the end (its scores are its rows' part of k . q), so that the waves meet once a chunk, in LDS. Operands
// need no rearrangement: register r of an accumulator holds rows 4 (lane / 16) + r at column lane % 16, which as an operand is
// the k-slice {r, 4 + r, 8 + r, 12 + r}; whoever meets it takes the same slice. Scores are formed as
// K Q^T for that reason. Rows of 128 are 132 apart in LDS: 16-byte reads of 16 neighbouring rows and
// 4-byte reads of 16 neighbouring elements of every fourth row both meet the banks evenly.
// A sum that is masked must not meet an infinity of a later token (0 x inf), nor a sum overflow whose decay, taken
// afterwards here, would have kept it finite: a chunk with a value that is not finite or over 10^12, or with a state over 10^24
// in front of it, goes through the same products one token at a time, each read out of the state after it.
// Powers are products of repeated squares, so any decay goes (negative, none at all), in double and kept in two
// floats: a rounded d^32 would be off by the same part every chunk, which over a memory of 500 tokens made ten
// times the error of the walk (3e-6 against 4e-7).
// LEAN: the same operations with a quarter fewer registers (one chunk on its way, powers read where they are used), so that
// one more block shares a compute unit: for launches of more blocks than one (256 threads: three) a unit. 2 sequences of 1,000
// tokens, 32 heads of 128: 157 -> 145 us, 8 of 128 103 -> 78 (walked 73); a lone one of 2,047 155 and 170.
constexpr int RC_TOKENS = 32, RC_VROW = 20;

template <int G, int NW, bool LEAN>
__global__ __launch_bounds__(64 * NW, LEAN ? 4 : 1) void retention_chunk_kernel(RetentionArgs a) {
  constexpr int DP = 16 * G * NW, ROW = DP + 4, THREADS = 64 * NW, AHEAD = LEAN ? 1 : 2;
  constexpr int PIECES = RC_TOKENS * DP / 4 / THREADS;       // 16-byte pieces of q, and of k, a thread
  constexpr int OWN = RC_TOKENS * RT_COLS / THREADS;         // values, and read-outs, a thread
  __shared__ __attribute__((aligned(16))) float qs[RC_TOKENS * ROW];
  __shared__ __attribute__((aligned(16))) float ks[RC_TOKENS * ROW];
  __shared__ __attribute__((aligned(16))) float vs[RC_TOKENS * RC_VROW];
  __shared__ __attribute__((aligned(16))) float red[NW][2][64 * 4];
  __shared__ float powers[RC_TOKENS + 1], powers_rest[RC_TOKENS + 1];
  __shared__ int odd[2];  // whether the chunk (of even, of odd number) holds a value for single tokens
  const int seq = a.seq_ids ? a.seq_ids[blockIdx.x] : blockIdx.x, head = blockIdx.y, col0 = blockIdx.z * RT_COLS;
  const int t0 = a.cu_q[seq], t1 = a.cu_q[seq + 1];
  if (t1 - t0 < a.chunk_from) return;
  const int dim = a.dim, vdim = a.vdim, qk_head = head / a.share;
  const int lane = threadIdx.x & 63, wave = uniform_wave_number(), r16 = lane & 15, quad = lane >> 4;
  const float* qkv = (const float*)a.qkv;
  if (threadIdx.x <= RC_TOKENS) {
    double by = a.decay[head], p = 1.0;
    for (int e = threadIdx.x; e; e >>= 1, by *= by)
      if (e & 1) p *= by;
    powers[threadIdx.x] = (float)p;
    powers_rest[threadIdx.x] = (float)(p - (double)(float)p);
  }
  if (threadIdx.x < 2) odd[threadIdx.x] = 0;
  float* st = a.state + (((size_t)a.state_slots[seq] * a.heads + head) * vdim + min(col0 + r16, vdim - 1)) * dim;
  const bool col_ok = col0 + r16 < vdim;
  f32x4_t s[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int d = 16 * (G * wave + g) + 4 * quad;
    s[g] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    if (d < dim && col_ok) s[g] = *(const f32x4_t*)(st + d);
  }
  // the pieces of the next two chunks (LEAN: of the next), on their way while one is walked (2.4 us a chunk; a load takes about one); what lies beyond the head or the tokens becomes
  // zero only on its way to LDS: a choice here would wait for the loads
  struct Ahead {
    f32x4_t q[PIECES], k[PIECES];
    float v[OWN];
  };
  auto fetch = [&](Ahead& to, int base) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int e = threadIdx.x + THREADS * i, tok = e / (DP / 4), d = 4 * (e % (DP / 4));
      const float* row = qkv + (size_t)min(base + tok, t1 - 1) * a.channels + qk_head * dim + min(d, dim - 4);
      to.q[i] = *(const f32x4_t*)(row + a.q_first);
      to.k[i] = *(const f32x4_t*)(row + a.k_first);
    }
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
      const int e = threadIdx.x + THREADS * i, tok = e >> 4, c = col0 + (e & 15);
      to.v[i] = qkv[(size_t)min(base + tok, t1 - 1) * a.channels + a.v_first + head * vdim + min(c, vdim - 1)];
    }
    __builtin_amdgcn_sched_barrier(0);  // asked for here, not where they are used
  };
  __syncthreads();
  // d^(i+1); d^(i-j) by how many tiles apart; d^(n-1-j): kept in registers or (LEAN) read where they are used
  struct Powers {
    float by[2][4], rest[2][4];
  };
  auto load_powers = [&](Powers& to, auto exponent) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int e = max(exponent(i, 4 * quad + r), 0);
        to.by[i][r] = powers[e];
        to.rest[i][r] = powers_rest[e];
      }
  };
  Powers to_row, back, to_end;
  auto rows_powers = [&] { load_powers(to_row, [](int i, int row) { return 16 * i + row + 1; }); };
  auto back_powers = [&] { load_powers(back, [&](int i, int row) { return 16 * i + r16 - row; }); };
  auto end_powers = [&](int n) { load_powers(to_end, [&](int i, int row) { return n - 1 - (16 * i + row); }); };
  if (!LEAN) {
    rows_powers();
    back_powers();
    end_powers(RC_TOKENS);
  }
  auto times = [](float x, const Powers& p, int i, int r) { return fmaf(x, p.by[i][r], x * p.rest[i][r]); };
  // one chunk from LDS: rows off .. off + n - 1; SINGLE: one row (n = 1), the others taken as zeros
  f32x4_t o[2];
  auto walk = [&](auto single, int off, int n) {
    constexpr bool SINGLE = decltype(single)::value;
    constexpr int TILES = SINGLE ? 1 : 2;
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    // all of the wave's operands first, and no further apart than that: left alone the compiler waits for LDS 14 times
    f32x4_t q[TILES][G], k[TILES][G], kt[TILES][G], v[TILES], scores[TILES][TILES];
#pragma unroll
    for (int j = 0; j < TILES; ++j)
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const int at = (off + (SINGLE ? 0 : 16 * j + r16)) * ROW + 16 * (G * wave + g) + 4 * quad;
        q[j][g] = *(const f32x4_t*)(qs + at);
        k[j][g] = *(const f32x4_t*)(ks + at);
      }
#pragma unroll
    for (int j = 0; j < TILES; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = off + (SINGLE ? 0 : 16 * j + 4 * quad + r);
        v[j][r] = vs[row * RC_VROW + r16];
#pragma unroll
        for (int g = 0; g < G; ++g) kt[j][g][r] = ks[row * ROW + 16 * (G * wave + g) + r16];
      }
    __builtin_amdgcn_sched_barrier(0);
    if (SINGLE) {  // S <- d S + k v^T, o = S^T q: nothing is multiplied that the recurrence does not multiply
      const bool first = quad == 0;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        f32x4_t acc = __builtin_amdgcn_mfma_f32_16x16x4f32(first ? kt[0][g][0] : 0.f, first ? v[0][0] : 0.f, zero, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) s[g][r] = fmaf(s[g][r], powers[1], acc[r]);
        acc = zero;
#pragma unroll
        for (int r = 0; r < 4; ++r) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(r16 ? 0.f : q[0][g][r], s[g][r], acc, 0, 0, 0);
        o[0] = g ? o[0] + acc : acc;
      }
      return;
    }
#pragma unroll
    for (int j = 0; j < TILES; ++j) {  // scores[i][j]: rows are keys, columns queries
#pragma unroll
      for (int i = j; i < TILES; ++i) {
        f32x4_t sum = zero;
#pragma unroll
        for (int g = 0; g < G; ++g) {
          f32x4_t acc = zero;
#pragma unroll
          for (int r = 0; r < 4; ++r) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(k[j][g][r], q[i][g][r], acc, 0, 0, 0);
          sum = g ? sum + acc : acc;
        }
        scores[i][j] = sum;
      }
    }
    if (LEAN) rows_powers();
#pragma unroll
    for (int i = 0; i < TILES; ++i) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        f32x4_t acc = zero;
#pragma unroll
        for (int r = 0; r < 4; ++r) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(q[i][g][r], s[g][r], acc, 0, 0, 0);
        o[i] = g ? o[i] + acc : acc;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) o[i][r] = times(o[i][r], to_row, i, r);
    }
    if (LEAN) back_powers();
#pragma unroll
    for (int i = 0; i < TILES; ++i)
#pragma unroll
      for (int j = 0; j <= i; ++j) {
        f32x4_t acc = zero;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float p = i == j && r16 < 4 * quad + r ? 0.f : times(scores[i][j][r], back, i - j, r);
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(p, v[j][r], acc, 0, 0, 0);
        }
        o[i] += acc;
      }
    const float all = powers[n], rest = powers_rest[n];
    if (LEAN) end_powers(n);
#pragma unroll
    for (int j = 0; j < TILES; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[j][r] = times(v[j][r], to_end, j, r);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      f32x4_t add[TILES];
#pragma unroll
      for (int j = 0; j < TILES; ++j) {
        add[j] = zero;
#pragma unroll
        for (int r = 0; r < 4; ++r) add[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(kt[j][g][r], v[j][r], add[j], 0, 0, 0);
      }
      add[0] += add[TILES - 1];
#pragma unroll
      for (int r = 0; r < 4; ++r) s[g][r] = fmaf(s[g][r], all, fmaf(s[g][r], rest, add[0][r]));
    }
  };
  auto leave = [&](int base, int n) {  // the waves' sums meet, and the read-outs leave
#pragma unroll
    for (int i = 0; i < 2; ++i) *(f32x4_t*)(red[wave][i] + lane * 4) = o[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
      // token tok, column c: register tok % 4 of lane 16 (tok % 16 / 4) + c in tile tok / 16
      const int e = threadIdx.x + THREADS * i, tok = e >> 4, c = e & 15, at = (16 * ((tok & 15) >> 2) + c) * 4 + (tok & 3);
      double sum = 0.0;  // rounded once
#pragma unroll
      for (int w = 0; w < NW; ++w) sum += red[w][tok >> 4][at];
      if (tok < n && col0 + c < vdim) a.out[((size_t)(base + tok) * a.heads + head) * vdim + col0 + c] = (float)sum;
    }
  };
  auto chunk = [&](Ahead& from, int base, int turn) {
    const int n = min(RC_TOKENS, t1 - base);
    bool large = false;
    auto look = [&](float x) { large |= !(fabsf(x) < 1e12f); };
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int e = threadIdx.x + THREADS * i, tok = e / (DP / 4), d = 4 * (e % (DP / 4));
      if (tok >= n || d >= dim) from.q[i] = from.k[i] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
      *(f32x4_t*)(qs + tok * ROW + d) = from.q[i];
      *(f32x4_t*)(ks + tok * ROW + d) = from.k[i];
#pragma unroll
      for (int r = 0; r < 4; ++r) look(from.q[i][r]), look(from.k[i][r]);
    }
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
      const int e = threadIdx.x + THREADS * i;
      if ((e >> 4) >= n || col0 + (e & 15) >= vdim) from.v[i] = 0.f;
      vs[(e >> 4) * RC_VROW + (e & 15)] = from.v[i];
      look(from.v[i]);
    }
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r) large |= !(fabsf(s[g][r]) < 1e24f);
    if (large) odd[turn] = 1;
    __syncthreads();
    const bool one_by_one = odd[turn];
    if (threadIdx.x == 0) odd[turn ^ 1] = 0;  // read last before the barrier in `leave` of the chunk before
    if (base + AHEAD * RC_TOKENS < t1) fetch(from, base + AHEAD * RC_TOKENS);
    if (!one_by_one) {
      if (!LEAN && n < RC_TOKENS) end_powers(n);  // the last chunk
      walk(std::false_type{}, 0, n);
      leave(base, n);
    } else {
      for (int i = 0; i < n; ++i) {
        o[1] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
        walk(std::true_type{}, i, 1);
        leave(base + i, 1);
        __syncthreads();
      }
    }
  };
  Ahead first;
  fetch(first, t0);
  if (LEAN) {
    for (int base = t0, turn = 0; base < t1; base += RC_TOKENS, turn ^= 1) chunk(first, base, turn);
  } else {
    Ahead second;
    if (t0 + RC_TOKENS < t1) fetch(second, t0 + RC_TOKENS);
    for (int base = t0; base < t1; base += 2 * RC_TOKENS) {
      chunk(first, base, 0);
      if (base + RC_TOKENS < t1) chunk(second, base + RC_TOKENS, 1);
    }
  }
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int d = 16 * (G * wave + g) + 4 * quad;
    if (d < dim && col_ok) *(f32x4_t*)(st + d) = s[g];
  }
}

extern "C" int qrt_retention(const RetentionArgs* args, int num_tokens, int num_seqs, int num_slots, hipStream_t stream) {
  RetentionArgs a = *args;
  QRT_CHECK(num_tokens >= 0 && num_seqs >= 0 && num_slots > 0, "retention: bad counts");
  QRT_CHECK(a.heads > 0 && a.heads <= 65535 && a.dim > 0 && a.dim <= 512 && a.vdim > 0, "retention: %d heads of %d x %d", a.heads, a.dim, a.vdim);
  if (a.share == 0) a.share = 1;
  QRT_CHECK(a.qkv_code == QRT_F32 || (a.qkv_code == QRT_BF16 && (a.step || a.gates)), "retention: unknown input type %d", a.qkv_code);
  QRT_CHECK(a.share > 0 && a.heads % a.share == 0, "retention: %d heads, %d of which share a key", a.heads, a.share);
  QRT_CHECK(a.channels >= 2 * (a.heads / a.share) * a.dim + a.heads * a.vdim, "retention: %d channels hold no q, k and v", a.channels);
  QRT_CHECK(!a.gates || (a.last_out && !a.step), "retention: gates without a place for the last column's read-out, or beside step logits");
  QRT_CHECK(a.gates ? true : a.step ? a.step_bias && a.a_log && a.skip && a.step_stride >= a.heads : a.decay != nullptr,
            "retention: neither constant decays nor step logits with their bias, rate and skip");
  if (num_tokens == 0 || num_seqs == 0) return 0;
  const dim3 grid(num_seqs, a.heads, (a.vdim + (a.gates ? 1 : 0) + RT_COLS - 1) / RT_COLS);
  const int groups = (a.dim + 63) / 64;
  if (a.chunk_from > 0) {
    QRT_CHECK(!a.gates && !a.step && groups <= 4 && a.dim % 4 == 0 && a.channels % 4 == 0 && a.q_first % 4 == 0 && a.k_first % 4 == 0 &&
                  ((uintptr_t)a.qkv | (uintptr_t)a.state) % 16 == 0,
              "retention: chunks go with constant decays and heads of up to 256 elements in whole pieces of 16 bytes");
    if (a.longest >= a.chunk_from) {
      const long blocks = (long)grid.x * grid.y * grid.z;
      if (groups == 1 && blocks > 768) retention_chunk_kernel<1, 4, true><<<grid, 256, 0, stream>>>(a);
      else if (groups == 1) retention_chunk_kernel<1, 4, false><<<grid, 256, 0, stream>>>(a);
      else if (groups == 2 && blocks > 256) retention_chunk_kernel<1, 8, true><<<grid, 512, 0, stream>>>(a);
      else if (groups == 2) retention_chunk_kernel<1, 8, false><<<grid, 512, 0, stream>>>(a);
      else retention_chunk_kernel<2, 8, false><<<grid, 512, 0, stream>>>(a);
      QRT_LAUNCH_CHECK("retention (chunks)");
      if (a.shortest >= a.chunk_from) return 0;
    }
  }
#define GO(G, TILE)                                                                 \
  do {                                                                              \
    if (a.gates && a.qkv_code == QRT_BF16) retention_kernel<G, TILE, RT_GATES, bf16_t><<<grid, 256, 0, stream>>>(a); \
    else if (a.gates) retention_kernel<G, TILE, RT_GATES, float><<<grid, 256, 0, stream>>>(a); \
    else if (a.step && a.qkv_code == QRT_BF16) retention_kernel<G, TILE, RT_STEP, bf16_t><<<grid, 256, 0, stream>>>(a); \
    else if (a.step) retention_kernel<G, TILE, RT_STEP, float><<<grid, 256, 0, stream>>>(a); \
    else retention_kernel<G, TILE, RT_CONSTANT, float><<<grid, 256, 0, stream>>>(a);      \
  } while (0)
  if (num_tokens <= 2 * num_seqs || (a.chunk_from > 0 && a.longest >= a.chunk_from && a.shortest <= 4)) {  // decoded tokens, mostly
    if (groups <= 1) GO(1, 4);
    else if (groups <= 2) GO(2, 4);
    else if (groups <= 4) GO(4, 4);
    else GO(8, 4);
  } else if (groups <= 1) GO(1, 16);
  else if (groups <= 2) GO(2, 16);
  else if (groups <= 4) GO(4, 16);
  else GO(8, 8);
#undef GO
  QRT_LAUNCH_CHECK("retention");
  return 0;
}
