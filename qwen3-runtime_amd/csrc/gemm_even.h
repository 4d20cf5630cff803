// Few rows by a weight whose rows are shared out evenly (gemm_even.hip).
#pragma once
#include "common.h"
#include "gemm_epilogue.h"
#include "row_norm.h"

constexpr int EVEN_BLOCKS = 256;  // a compute unit each
// Units of eight weight rows that the block with the most rows fetches.
constexpr int even_units(int N) { return ((N + EVEN_BLOCKS - 1) / EVEN_BLOCKS + 7) / 8; }
// Up to 4,096 rows a tile a unit is even already; from 6,145 to 8,192 two tiles a unit are as fast (7,168 x 2,560 at 1 and 8 rows 7.7, 8.1 by
// tiles and 8.0, 8.2 evenly; 8,192 8.3, 8.7 and 8.65, 8.9); up to 12,288 three are at up to 4 rows (12,288 x 2,560 11.7 and 11.9), and 16 rows gain
// 1 to 24 %, short K least. Beyond, a unit's rows are many tiles, of which one more or less matters little.
constexpr bool even_takes(int M, int N) { return even_units(N) == 3 || even_units(N) == 5 || (even_units(N) == 6 && M > 4); }

// Operands on 16 bytes, 0 < M <= 16, K % 64 == 0; ep.whole() of the sums, which `norm` (or null) multiplies by its factors first.
int even_product(const bf16_t* a, const bf16_t* w, bf16_t* c, int M, int N, int K, const GatedEpilogue& ep, const RowNorm* norm, hipStream_t stream);
