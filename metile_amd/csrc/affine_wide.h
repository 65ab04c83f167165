// Host-visible launch interface of the wide affine GEMM kernel (more rows than one small-row
// dispatch takes).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace mt {

struct WideParams {
  const uint16_t* x;        // [M, K] activations
  const uint32_t* w[2];     // packed codes of each projection (gate, up for SwiGLU)
  const uint16_t* s[2];     // [N, K/G] scales
  const uint16_t* b[2];     // [N, K/G] biases
  const uint16_t* residual;  // [M, N], added before the output rounding, or null
  uint16_t* y;              // [M, N]
  float* partial;           // split K: [split][tile][wave][accumulator registers]
  uint32_t* counters;       // split K: one per (tile, wave), zero between calls
  int M, K, N;
  int group_shift;          // log2 of the group size
  int tile_m;               // 32, 64, 96 or 128 rows a workgroup
  int tile_n;               // 64, 128 or 256 code columns a workgroup (of both projections)
  int ksplit;
  int steps_per_split;      // 64-wide K steps, a multiple of wide_split_unit
  uint32_t col_stride;      // bytes from one column's codes to the next's
  uint32_t step_stride;     // bytes from one K step's codes to the next's
};

// bits 4 (groups of 64 or more) or 8 (groups of 32 or more); N a multiple of 32; the codes,
// activations and outputs each below 2 GiB.
hipError_t launch_affine_wide(const WideParams& p, int bits, int dtype, int nproj,
                              hipStream_t stream);

// K splits start on whole groups and whole iterations of the four-step loop.
constexpr int wide_split_unit(int group_size) {
  return group_size > 256 ? group_size / 64 : 4;
}

// Bytes of one projection's codes: below 2 GiB for every call, but not so the number of its bits, which
// 32 bits do not hold from 512 MiB of codes on (K is a multiple of 64, so the row's bytes are whole).
constexpr uint32_t wide_code_bytes(int N, int K, int bits) {
  return (uint32_t)N * ((uint32_t)K * (uint32_t)bits / 8u);
}
static_assert(wide_code_bytes(152064, 3584, 8) == 544997376u, "a vocabulary head in 8 bits");
static_assert(wide_code_bytes(131072, 8192, 4) == (512u << 20), "in 4 bits, 2^32 bits of codes");
static_assert(wide_code_bytes(32, (1 << 26) - 64, 8) == (1u << 31) - 2048u, "the largest codes");

// Bytes of one split's partial sums of one tile.
constexpr size_t wide_part_bytes(int tile_m, int tile_n) { return (size_t)tile_m * tile_n * 4; }

}  // namespace mt
