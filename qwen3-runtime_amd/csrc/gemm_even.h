// Few rows by a weight whose rows are shared out evenly (gemm_even.hip).
#pragma once
#include "common.h"
#include "gemm_epilogue.h"
#include "row_norm.h"

constexpr int EVEN_BLOCKS = 256;  // a compute unit each
// Units of eight weight rows that the block with the most rows fetches.
constexpr int even_units(int N) { return ((N + EVEN_BLOCKS - 1) / EVEN_BLOCKS + 7) / 8; }
// Up to 4,096 rows a tile a unit is even already; from 6,145 to 8,192 two tiles a unit are as fast (7,168 x 2,560 at 1 and 8 rows 7.7, 8.1 by
// tiles and 8.0, 8.2 evenly; 8,192 8.3, 8.7 and 8.65, 8.9). Beyond 12,288 a unit's rows are many tiles, of which one more or less matters little. Within, not
// - where K is under 640: a block's start and end are what counts, and the units' loads one by one cost more (5,120 x 64 at 16 rows 2.8 and 2.9, 9,000 x 192 3.45 and 3.65,
//   12,000 x 320 4.15 and 4.4; level at 512);
// - just above two tiles a unit, and four where K is a multiple of 4,096, whose rows lie at the same channels of the memory: a few units would fetch
//   a load more for a row or two (4,104 x 1,024 at 9 rows 4.2 and 4.35, level up to 2,048; 8,200 x 4,096 at 1 and 8 rows 13.6, 14.8 and 16.0, 16.05; 8,320 and on level or faster);
// - three tiles a unit, of which some have two, up to 7 rows (12,288 x 2,560 at 1 and 5 rows 11.7, 12.0 and 11.9, 12.0), where K is under 1,024 (level) or a multiple of 2,048
//   over that (11,264 x 6,144 at 8 and 16 rows 9 % slower and 2 % faster, 12,288 x 4,096 3 and -8).
// - up to 7 rows where K is such a multiple, and none of 8,192: tiles are at their best there (10,240 x 6,144 at 1 and 8 rows 23.6, 24.8 and 25.0, 25.0; 6,144 x 12,288 4 % slower and
//   6 % faster).
// Elsewhere 1 to 35 % faster, at 16 rows and large K most.
constexpr bool even_takes(int M, int N, int K) {
  if (K < 640 || (M < 8 && K > 4096 && K % 2048 == 0 && K % 8192 != 0)) return false;
  if (even_units(N) == 3) return N >= 4160;
  if (even_units(N) == 5) return N >= 8320 || K % 4096 != 0;
  return even_units(N) == 6 && M >= 8 && K >= 1024 && (K <= 2048 || K % 2048 != 0);
}

// Operands on 16 bytes, 0 < M <= 16, K % 64 == 0; ep.whole() of the sums, which `norm` (or null) multiplies by its factors first.
int even_product(const bf16_t* a, const bf16_t* w, bf16_t* c, int M, int N, int K, const GatedEpilogue& ep, const RowNorm* norm, hipStream_t stream);
