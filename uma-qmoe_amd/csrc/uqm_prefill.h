// Expert-grouped GEMM with large route tiles (uqm_prefill.hip), for calls with
// many routes per expert.
#pragma once

#include "uqm_internal.h"

namespace uqm {

// Largest route tile of the kernel. An expert's routes are cut into as few
// tiles as that allows, of equal size up to a multiple of 16.
constexpr int kPrefillTileTokens = 144;

// Routes per tile of an expert with n routes: the multiple of 16 that splits
// them evenly over ceil(n / most) tiles (none of which is empty).
__host__ __device__ inline int route_tile_step(int n, int most) {
  const int tiles = (n + most - 1) / most;
  if (tiles <= 1) return most;
  return ((n + tiles - 1) / tiles + 15) / 16 * 16;
}

// Shapes the kernel takes: rows (per expert) x K weights, activations of at
// most x_rows rows of ldx elements.
bool prefill_supported(int enc, int64_t rows, int64_t K, int64_t group, int64_t x_rows, int64_t ldx);
// nmat 2: gate/up with the SiLU epilogue (kModeSilu); 1: kModeF32 or kModeBF16
// rows. Tiles of kPrefillTileTokens split by route_tile_step: the device list
// built with that tile size, or with tiles == null the n_routes rows of one
// matrix. No K split.
hipError_t launch_prefill_mfma(int enc, int nmat, int mode, const MfmaArgs& a, hipStream_t stream);

}  // namespace uqm
