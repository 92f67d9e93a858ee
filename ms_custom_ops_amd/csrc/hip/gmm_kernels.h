// Host-side declarations of the kernel launchers (one translation unit per kernel family).
#ifndef MSCO_GMM_KERNELS_H_
#define MSCO_GMM_KERNELS_H_

#include <hip/hip_runtime.h>
#include "gmm_common.h"

namespace msco {

// Tile shapes of the persistent four-wave kernel: 32 xb rows x 32 wb columns.
struct T4mShape { int xb, wb; };
constexpr int T4M_SHAPES = 8;
constexpr T4mShape kT4mShape[T4M_SHAPES] = {{8, 8}, {7, 8}, {6, 8}, {5, 8}, {4, 8}, {9, 7}, {4, 6}, {5, 6}};
constexpr bool t4m_has(int shape, int layout) { return layout != 2 || kT4mShape[shape].wb != 7; }   // layout 0 [E,N,K], 1 packed, 2 [E,K,N]
// The shape of a launch: an index into kT4mShape, or negative: by the groups, which the device counts, and these modelled times
// (t4m_pick in gmm_tile4m_kernel.h).  (Not part of GmmParams: every kernel would request them.)
struct T4mPick {
  int shape;
  float us[T4M_SHAPES];   // of a round (0: no such shape)
  float idle, empty;      // the share of a round that is free where a CU has no tile; of a tile, where its rows do not exist
};

enum TileCfg : int {
  TILE_256x256 = 0, TILE_128x128 = 1, TILE_64x128 = 2, TILE_128x256 = 3,
  TILE_256x256_W4 = 4,   // persistent, four wavefronts with accumulators for a quarter of the tile each: gmm_tile4m_kernel.h (16 x 16 x 64 MFMAs); T4mPick
  TILE_256x256_W4_MFMA32 = 5,   // the same on 32 x 32 x 32 MFMAs: gmm_tile4_w8a8.hip (never planned; kept to be measured against)
  TILE_ROWS256 = 6,   // packed weights only: chunks of up to 256 rows x strips of 256 columns, x through LDS, weights straight into MFMA operands: gmm_rows_w8a8.hip
  TILE_ROWS128 = 7,   // the same with chunks of up to 128 rows and two workgroups per CU
  TILE_ROWS160 = 8,   // ... of up to 160 rows, two workgroups per CU, two K blocks of weights in flight
  TILE_64x256_W4B = 9,    // 4-bit weights [E,K,N/2]
  TILE_128x256_W4B = 10,
  TILE_32x128 = 11,   // a few rows on [E,K,N] and [E,N,K] weights, two waves side by side, two workgroups per CU
  TILE_32x256 = 12,   // ... on [E,K,N] weights, four waves side by side
  TILE_CFG_COUNT = 13
};

// MFMA tile kernel for W8A8 (prefill shapes).  nk: weights stored [E,N,K]; packed: the packed layout (nk is ignored).
hipError_t launch_tile_w8a8(const GmmParams &p, int tile_cfg, bool nk, bool packed, const T4mPick &pick, hipStream_t stream);   // pick: TILE_256x256_W4 only
hipError_t launch_tile_a8w4(const GmmParams &p, int tile_cfg, hipStream_t stream);   // int8 x, 4-bit weights [E,K,N/2]
const char *tile_cfg_name(int tile_cfg);
hipError_t launch_tile4m_w8a8(const GmmParams &p, const T4mPick &pick, int layout, hipStream_t stream);  // layout 0 [E,N,K], 1 packed, 2 [E,K,N] (N % 16 == 0)
hipError_t launch_tile4_w8a8(const GmmParams &p, int layout, hipStream_t stream);   // layout 0 [E,N,K], 1 packed, 2 [E,K,N] (N % 16 == 0)
void tile_cfg_dims(int tile_cfg, int *bm, int *bn);
// packed weights, several groups of a few dozen to a few hundred rows: chunks of 16 rbmax rows (rbmax = 8, 10 or 16), see gmm_rows_w8a8.hip;
// p.w_nontemporal as for the tiles
hipError_t launch_rows_w8a8(const GmmParams &p, int rbmax, hipStream_t stream);
// K split across workgroups (p.split_k > 1; four-wave tile shapes only): partial tiles and arrival counters
size_t tile_count_bound(int tile_cfg, int64_t m, int64_t n, int64_t e);
size_t tile_workspace_bytes(int tile_cfg, int64_t m, int64_t n, int64_t e, int split_k);

// grid.y of the decode kernels: an upper bound, for any group_list, of the number of chunks of rows_per_chunk rows that
// hold rows (see chunk_of_slot in gmm_common.h)
inline unsigned chunk_slots(const GmmParams &p, int rows_per_chunk) {
  const long long per_group = ((long long)p.m + rows_per_chunk - 1) / rows_per_chunk;
  const long long all = (long long)p.e * (per_group > 1 ? per_group : 1);
  const long long held = (p.m < p.e ? p.m : p.e) + p.m / rows_per_chunk;
  const long long slots = all < held ? all : held;
  return (unsigned)(slots > 1 ? slots : 1);
}

// workgroups of a launch that finds its work with chunk_of_xcd_slot: an XCD holds at most ceil(strips / 8) strips of a group
inline long long xcd_slots(const GmmParams &p, int rows_per_chunk) {
  return (long long)kNumXcd * ((p.n_strips + kNumXcd - 1) / kNumXcd) * chunk_slots(p, rows_per_chunk);
}

// Skinny (decode) kernels: one workgroup streams a 128-column weight strip of one group over a K
// range; waves split K and reduce through LDS, workgroups split K and reduce through the workspace.
// wide16: the 16-wave / 128-column-strip variant for small weight sets, else 4 waves / 256-column strips
hipError_t launch_skinny_w8a8(const GmmParams &p, bool nk, bool wide16, hipStream_t stream);
size_t decode_tiles(int64_t m, int64_t n, int64_t e, int rows_per_chunk, int cols);   // partial tiles (per K slice) and counters of the decode kernels

// Decode kernels for weights in the packed layout (gmm_stream.hip): 4 waves, strips of up to 256 columns, K slices of
// at most 128 blocks of 64 bytes (split_k chosen accordingly).
hipError_t launch_stream_w8a8(const GmmParams &p, hipStream_t stream);
hipError_t launch_stream_a16w8(const GmmParams &p, hipStream_t stream);   // K slices of at most 64 blocks
// more than 16 rows per group on packed weights: chunks of 16 tch rows (tch = 2, 4, 8), strips of 64 columns
hipError_t launch_streamm_w8a8(const GmmParams &p, int tch, hipStream_t stream);
hipError_t launch_streamm_a16w8(const GmmParams &p, int tch, bool packed, hipStream_t stream);   // weight-only, 32 / 64 / 128 rows per chunk (tch = 2, 4, 8), packed or [E,K,N] weights, no K split
// weight-only, packed or [E,K,N] weights: equal chunks of up to 128 rows x strips of 512 or 256 columns, p.split_k slices of K, one or two sets of waves (gmm_rows_a16w8_kernel.h)
hipError_t launch_rows_a16w8(const GmmParams &p, bool packed, bool w4, int strip_cols, int sets, hipStream_t stream);
size_t rows_a16w8_slice_bytes();   // workspace bytes of one (chunk, strip, K slice) partial tile
size_t streamm_tile_bytes(int tch);   // workspace bytes of one (chunk, strip, K slice) partial tile
size_t rows32_a16w8_slice_bytes(int strip_groups);   // workspace bytes of one (chunk, strip, K slice) partial tile of the 128-row weight-only kernel
size_t stream_a16w8_tile_bytes();   // workspace bytes of one (strip, K slice) partial tile of the weight-only kernel
int stream_blocks_per_wave(int64_t k, int split_k);
size_t packed_weight_bytes(int64_t k, int64_t n);   // bytes of one group's weights in the packed layout
hipError_t launch_pack_weight(const void *src, void *dst, long long e, long long k, long long n, bool src_nk,
                              hipStream_t stream);

// Row-major [E,K,N] weights of 4 or 8 bits transposed and converted in registers (gmm_regt.hip): chunks of 16 row_blocks rows
// (1 or 2), strips of strip_cols columns (256 or 512), p.split_k slices of K; shallow (16-bit x on 8-bit weights): more workgroups per CU
hipError_t launch_regt(const GmmParams &p, int weight_bits, int row_blocks, int strip_cols, bool shallow, hipStream_t stream);
size_t regt_slice_bytes(int row_blocks, int strip_cols);   // workspace bytes of one (chunk, strip, K slice) partial tile
// 4-bit values widened to int8 (gmm_w4.hip)
hipError_t launch_unpack_int4(const void *src, void *dst, long long src_bytes, hipStream_t stream);

// Shape-agnostic fallback kernels (one output element per thread), any K / N.
// layout: 0 [E,K,N], 1 [E,N,K], 2 packed
hipError_t launch_generic_w8a8(const GmmParams &p, int layout, hipStream_t stream);
hipError_t launch_generic_a16w8(const GmmParams &p, int layout, hipStream_t stream);

// Batched 2-D transpose, src [batch, rows, cols] -> dst [batch, cols, rows].
hipError_t launch_transpose_2d(const void *src, void *dst, long long batch, long long rows, long long cols,
                               int elem_bytes, hipStream_t stream);

}  // namespace msco
#endif  // MSCO_GMM_KERNELS_H_
