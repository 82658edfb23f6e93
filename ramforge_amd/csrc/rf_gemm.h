// rf_gemm.h — the tiled prefill GEMM behind launch_matmul_packed (internal).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rf {

struct MmTileSeg {
  const uint8_t* reg[4];  // packed regions at the segment's first row
  uint64_t bytes[4];      // and their sizes (each below 2^31)
  uint64_t rows;
};
// Where a launch leaves its split-K partials: [nsplit][n][all rows].
struct MmTileOut {
  const float* part;
  uint32_t nsplit;
};
constexpr uint64_t MM_TILE_ROWS = 256;  // weight rows of a workgroup (one segment's)
// Workspace floats (x planes, block sums, partials) of a launch of exactly n
// tokens; groups: the sum of each segment's rows over MM_TILE_ROWS, rounded up.
uint64_t mm_tile_ws_floats(uint64_t groups, uint64_t mtot, uint64_t K, uint64_t n);
// K a whole number of the type's blocks, ws 16-byte aligned; x of any float alignment.
hipError_t launch_mm_tile(uint32_t t, const MmTileSeg* segs, int nseg, const float* x, uint64_t ldx, uint64_t n,
                          uint64_t K, float* ws, uint64_t ws_floats, hipStream_t st, MmTileOut* out);
hipError_t load_module_gemm();

}  // namespace rf
