// Expert-grouped GEMM with large route tiles (uqm_prefill.hip), for calls with
// many routes per expert.
#pragma once

#include "uqm_internal.h"

namespace uqm {

// Largest route tile of the kernel. An expert's routes are cut into as few
// tiles as that allows, of equal size up to a multiple of 16.
constexpr int kPrefillTileTokens = 144;

// Routes per tile when n routes are split evenly over `tiles` tiles: a multiple
// of 16.
__host__ __device__ inline int even_step(int n, int tiles) { return ((n + tiles - 1) / tiles + 15) / 16 * 16; }

// Routes per tile of an expert with n routes, over ceil(n / most) tiles (none
// of which is empty).
__host__ __device__ inline int route_tile_step(int n, int most) {
  const int tiles = (n + most - 1) / most;
  return tiles <= 1 ? most : even_step(n, tiles);
}

// Shapes the kernel takes: rows (per expert) x K weights, activations of at
// most x_rows rows of ldx elements.
bool prefill_supported(int enc, int64_t rows, int64_t K, int64_t group, int64_t x_rows, int64_t ldx);
// nmat 2: gate/up with the SiLU epilogue (kModeSilu); 1: kModeF32 or kModeBF16
// rows. Tiles split by route_tile_step(., kPrefillTileTokens): the device list
// built with that tile size. With tiles == null: the n_routes rows of one
// matrix in tile_bound tiles of even_step routes (at most kPrefillTileTokens).
// No K split.
hipError_t launch_prefill_mfma(int enc, int nmat, int mode, const MfmaArgs& a, hipStream_t stream);

}  // namespace uqm
