// Modelled times of the persistent kernel's tile shapes and of the tiles that they are compared with; how they were fitted: plan_tile_shape in msco_gmm.hip.
#pragma once

#include "gmm_kernels.h"

#include <cstdint>

namespace msco {

struct TileTime { double launch, idle, slab, fixed, read, unaligned; };
struct TileTimes { double launch, idle, read, unaligned, empty, slab[T4M_SHAPES], fixed[T4M_SHAPES]; TileTime tall, small, low; };   // 128 x 256, 128 x 128, 64 x 128 tiles
constexpr TileTimes kTileTimes[3] = {   // [E,K,N], [E,N,K], packed; 0: no such shape
    {4.73, 0.303, 0.251, 0.042, 0.128, {1.457, 1.283, 1.128, 1.019, 0.876, 0.0, 0.755, 0.870}, {7.15, 6.74, 5.99, 5.09, 4.30, 0.0, 3.28, 3.85},
     {4.88, 0.313, 1.004, 2.76, 0.205, 0.058}, {4.40, 0.396, 0.585, 1.92, 0.212, 0.147}, {4.65, 0.414, 0.385, 0.72, 0.225, 0.178}},
    {4.37, 0.314, 0.208, 0.144, 0.135, {1.367, 1.229, 1.080, 0.982, 0.859, 1.305, 0.685, 0.776}, {7.61, 6.71, 5.95, 5.08, 4.27, 7.61, 3.24, 3.83},
     {4.00, 0.326, 1.124, 2.97, 0.249, 0.154}, {3.58, 0.501, 0.639, 1.87, 0.225, 0.182}, {4.16, 0.642, 0.447, 0.52, 0.251, 0.205}},
    {5.00, 0.325, 0.197, 0.042, 0.150, {1.378, 1.205, 1.051, 0.939, 0.805, 1.313, 0.663, 0.738}, {7.90, 7.19, 6.38, 5.53, 4.51, 8.01, 3.34, 4.23},
     {4.64, 0.386, 0.990, 2.98, 0.197, 0.045}, {4.53, 0.463, 0.568, 1.90, 0.146, 0.084}, {4.83, 0.542, 0.342, 0.70, 0.194, 0.060}}};

// What the device picks by (t4m_pick).  layout: an index into kTileTimes.
inline void tile_shape_times(int layout, int64_t k, T4mPick &pick) {
  const TileTimes &t = kTileTimes[layout];
  const double slabs = (double)(2 * ((k + 255) / 256)) * (k % 128 != 0 ? 1.0 + t.unaligned : 1.0);
  for (int j = 0; j < T4M_SHAPES; ++j) pick.us[j] = (float)(slabs * t.slab[j] + t.fixed[j]);
  pick.idle = (float)t.idle;
  pick.empty = (float)t.empty;
}

}  // namespace msco
