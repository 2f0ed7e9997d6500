// Matmuls of a few tokens (2 to 16 a tile) on the matrix cores.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "gemm.h"

namespace th {

// Most parts few_ksplit asks for.
constexpr int kFewMaxSplitK = 4;

// Whether launch_few takes rows of `cols` columns for n tokens: whole 16-byte
// chunks, and offsets that fit its buffer descriptors.
bool few_supported(size_t n, size_t rows, size_t cols);

// out[t * rows + r] = w[r] . x[t] for t < n, for 1-3 matrices of `cols`
// columns that share x. With ksplit > 1 (one matrix) the partial products go
// to part[ksplit][n][rows], to be summed in order.
hipError_t launch_few(hipStream_t s, const float *x, size_t n, size_t cols, const GemmOut *outs, int n_outs,
                      float *part, int ksplit);

// Ways launch_few's caller should split K for one [rows, cols] matrix, when
// the consumer sums the partials (1: no split), at most kFewMaxSplitK.
int few_ksplit(size_t n, size_t rows, size_t cols);

// Whether launch_few (and launch_few_silu) is the faster one for 1-3 matrices
// of `rows` rows in all that the GEMM would take too.
bool few_preferred(size_t n, size_t rows, size_t cols, int n_outs);

// Whether launch_few (or, two, launch_few_silu) for n_outs matrices together is
// faster than each through launch_matmul (and, two, a silu_mul launch), where
// the GEMM does not take them.
bool few_together(size_t n, const size_t *rows, int n_outs, size_t cols);

// About how long launch_few takes for one [rows, cols] matrix, K in ksplit
// parts that are summed. At more than a few tokens it reads the weights again
// for every 16 (and, past 2560 columns a part, x for every 16 rows), so
// matrices that are not whole GEMM tiles go to launch_gemm_ragged where that is
// faster (us a call, this kernel against that: 64 tokens x 5003 x 2968 51.3 and
// 19.0, 700 535 and 98.8, 2000 x 7003 x 4552 2439 and 530; but 20 x 1003 x 1096
// 6.2 and 9.3, 200 8.8 and 10.8).
double few_us(size_t n, size_t rows, size_t cols, int ksplit = 1);

// h[t * inter + j] = silu(gate[j] . x[t]) * (up[j] . x[t]) (model/cpu.rs:151-155).
hipError_t launch_few_silu(hipStream_t s, const float *x, size_t n, size_t cols, const uint16_t *gate,
                           const uint16_t *up, size_t inter, float *h);

}  // namespace th
