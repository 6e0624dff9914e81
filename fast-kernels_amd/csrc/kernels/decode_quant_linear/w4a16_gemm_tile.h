// Host side of the row-tile GEMM (w4a16_gemm_tile.hip): tile shape, work split and workspace of a
// launch over any number of activation rows.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>

#include "w4a16_device.h"
#include "w4a16_gemv.h"

namespace fk {

// Rows of one launch; more are run as several launches over the same workspace, which keeps the
// prepared activations (2 bytes per value and 16 per (row, group)) bounded.
constexpr int kTileMaxRows = 1024;
constexpr int kTileThreads = 512;
constexpr int kTileWaves = kTileThreads / 64;
// k values a wave takes per unit (two groups of 128 or four of 64).
constexpr int kTileWaveK = 256;

struct TileShape {
  int rows = 0;         // activation rows of the launch
  double us = 0;        // estimated time on MI355X
  bool direct = false;  // the workgroups stage x themselves: no prepare launch, no fused neighbour
  int bm = 0, bn = 0;   // rows and columns of a workgroup's tile
  int mtiles = 0, col_tiles = 0;
  int unit_groups = 0;  // groups of a unit, the grain of the K splits
  int units = 0;        // units per tile
  int splits = 1;       // workgroups sharing a tile
  int per = 0;          // units per workgroup
  int grid = 0;
  // Workspace layout, in bytes from its start (the counters come first).
  size_t partials = 0, sums = 0, xs = 0, end = 0;
};

struct TileLaunch {
  const void* x = nullptr;
  const void* packets = nullptr;
  void* out = nullptr;
  void* workspace = nullptr;
  int M = 0, N = 0, K = 0;
  int group_size = 128;
  Act act = Act::kF16;
  PacketFormat format = PacketFormat::kArc;
  bool silu = false;                  // out[M, N/2] = silu(gate) * up
  const void* norm_weight = nullptr;  // RMSNorm before the product
  float eps = 0.0f;
};

// Work split and workspace for `rows` (at most kTileMaxRows) on cu_count CUs; the workspace starts
// with counter_bytes of counters. direct: at most 32 rows.
TileShape tile_shape(int rows, int n, int k, int group_size, bool direct, int cu_count,
                     size_t counter_bytes);

hipError_t launch_w4a16_gemm_tile(const TileLaunch& l, const TileShape& s, hipStream_t stream);

}  // namespace fk
