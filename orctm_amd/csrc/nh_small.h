// nh_small.h -- the inner iteration of launches of few columns (nh_small.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "nh_device.h"

namespace onh {

// One block works on `wc` columns of a row and all their levels, held in LDS.
constexpr size_t kSmallLds = size_t(160) * 1024 - 8192;  // of a block's columns; the rest for the sums
constexpr int kSmallBatch = 8;                           // levels are padded to whole batches
constexpr int kSmallColumns = 8192;                      // columns (whole rows of 64) of a system at most, wc < 64

// Whether a system of nz levels fits the blocks' LDS (4 planes a level) and registers (levels per thread: 13, 9
// and 5 at 64, 32 and 16 columns).
inline bool small_fits(int nz, bool fp32, int wc) {
  const size_t levels = (size_t)(nz + kSmallBatch - 1) / kSmallBatch * kSmallBatch;
  return levels <= (wc == 64 ? 13 * 12 : wc == 32 ? 9 * 24 : 5 * 48) && levels * 4 * wc * (fp32 ? 4 : 8) <= kSmallLds;
}

struct SmallLaunch {
  bool fp32 = true;
  int wc = 64;     // columns per block: 64, or 32 or 16 (one system)
  bool one = true; // one system, by value
  int nsys = 0;
  int nblocks = 0;
  int nz = 0;      // most levels of a system
  Sys sys{};       // the system (one)
  const Sys* d_sys = nullptr;
  const Tile* d_rows = nullptr;  // (sys, bx, by = row j) of each block (several systems)
};

// Raises the kernels' LDS limits on the current device; before the first launch on it.
hipError_t small_setup(const SmallLaunch& l);
// The first column update of an inner solve (x = 0) and its scalars.
hipError_t small_begin(hipStream_t st, const SmallLaunch& l);
// n iterations and their scalars: 2 n + 1 launches.
hipError_t small_iterations(hipStream_t st, const SmallLaunch& l, int n);
// One matvec without scalars (verification).
hipError_t small_matvec(hipStream_t st, const SmallLaunch& l);
hipError_t small_update(hipStream_t st, const SmallLaunch& l);
hipError_t small_finish(hipStream_t st, const SmallLaunch& l);

}  // namespace onh
