// The prefill GEMM (tile_gemm.hip): tiles of 64 rows, 80 in the merged list.

#pragma once

#include "lk_gemm.hpp"

namespace lk {

// Launches the prefill GEMM over `tiles` row tiles (an upper bound in schedule
// modes) for a weight format kFmt*: Gather (two
// matrices), Scatter or Dense (one). The caller has checked the operands and
// set a_pair / a_neg (W4A16) and a_rows; with g.part (device memory of
// tile_gemm_split_bytes) a dense product too small to fill the chip runs in
// several runs of k.
int tile_gemm_launch(int fmt, int mats, GemmArgs g, Mode mode, int64_t tiles, hipStream_t s,
                     const char* what);

// Bytes of the fp32 sums of a dense [m, k] x [k, outputs * n] product that is
// worth splitting over k in weight format kFmt*; 0 where it is not.
int64_t tile_gemm_split_bytes(int fmt, int64_t m, int64_t n, int64_t k, int64_t outputs);

}  // namespace lk
