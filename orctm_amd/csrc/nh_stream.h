// nh_stream.h -- the inner iteration of launches of many columns (nh_stream.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "nh_device.h"
#include "nh_kernels.h"

namespace onh {

// Levels up to which the column update keeps a column on chip.
constexpr int kStreamLevels = 64;

struct StreamLaunch {
  bool fp32 = true;
  bool tab = false;   // every system reads ZW/ZP from its table
  bool wrap = false;  // some system is periodic along x
  const Sys* d_sys = nullptr;
  const Tile* d_tiles = nullptr;  // tiles of 64 x kOuterRows columns
  int ntiles = 0;
  const Tile* d_pairs = nullptr;  // pairs of them (pair_tiles)
  int npairs = 0;
};

hipError_t stream_update(hipStream_t st, const StreamLaunch& l, bool init);
hipError_t stream_matvec(hipStream_t st, const StreamLaunch& l);

}  // namespace onh
