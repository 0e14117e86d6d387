// The quantized matmuls of the prefill path as their callers see them.
#pragma once

#include <algorithm>

#include "mf_device.h"
#include "mf_internal.h"

namespace mf {

constexpr int kMaxLds = 160 * 1024;    // LDS of a CU
constexpr uint32_t kTileTokens = 64;   // tokens of one expert a workgroup handles
constexpr uint32_t kSmallTile = 32;    // ... where few tokens meet an expert
constexpr uint32_t kQmmWaves = 4;      // waves per workgroup, 32 weight rows each
constexpr uint32_t kQmmRows = kQmmWaves * 32;

struct Tile {
  uint32_t expert, pair_start, count, list_tiles;  // list_tiles: how many the list has
};
// What the grouping leaves for the two matmuls of a layer call: runs of at most `tokens` routes of one expert, in expert order, room for
// `slots` (a multiple of 8).  A list of no tiles has a first record of zeros.  list[1] null: both read list[0].
struct TileLists {
  Tile* list[2];
  uint32_t slots[2], tokens[2];
};

struct QmmArgs {
  // weights: routed = blobs of the expert pool, dense = one projection set
  const uint8_t* expert_base;
  size_t expert_stride;
  uint32_t w_off[2], s_off[2], b_off[2];
  mf_qtensor dense[2];
  int pair_rows;        // 1: the NPROJ blocks of a wave are consecutive 32-row blocks of projection 0
  int tiled;            // 1: the routed experts' codes are in the matmul's own order (tile_codes_kernel), not row by row
  int dense_mode;       // 1: the "expert" is dense[], tiles are runs of consecutive rows
  uint32_t dense_rows;  // number of x rows in dense mode
  // activations: rows of kdim bf16 as matmul_row8 leaves them + their group sums (store_group_sum)
  const uint16_t* x;
  const uint16_t* sumx;
  // largest magnitude of every token's row of the first product, times kRowScale (dense mode: of every row); the rows' scale follows
  // from it (row_scale, or act_scale where act_rows is set), and so does that of the activations epilogue 0 leaves
  const float* row_max;
  int act_rows;
  uint32_t x_stride;
  int gather;           // 1: x row = sorted[pair].token, 0: x row = pair index
  const mf_pair* sorted;
  const Tile* tiles;
  uint32_t rows, kdim;  // weight rows (output width) and contraction length
  // a launch may take a window of the contraction (long K is cut into windows whose fp32 results are
  // added afterwards): rows of weights, tables and group sums are ng_ld groups apart (0: kdim / 64)
  // and the window starts at group g_off (a multiple of 8)
  uint32_t ng_ld, g_off;
  // several windows in one launch (dense mode): window w covers the groups from
  // dense_window_start(ng_ld, n_win, w) on and writes its fp32 result out_win_stride elements behind the
  // previous window's
  uint32_t n_win;
  size_t out_win_stride;
  // epilogue
  int epi;              // 0 swiglu -> bf16 [pair, rows] as matmul_row8 leaves rows, group sums to out_sums; 1 fp32 [token*K+rank, rows]; 2 bf16 [pair, rows];
                        // 3 bf16 [token*K+rank, rows]
  int narrow;           // shared-expert rounding points (dequant_int4.metal:240-245)
  int ternary;          // 2-bit codes {0,1,2} with bias = -scale: b_off / dense[].biases name the SCALE table
  int maple;            // MapleMoE's bf16-stepped activation in the SwiGLU epilogue
  void* out;
  uint16_t* out_sums;
  void* out2;           // epi 1 / 2 with two projections that are not row blocks of one: where projection 1 goes (null: dropped)
  uint32_t top_k;
  float limit;
  // dense mode: number of 64-row tiles and of work items; every XCD gets an eighth of the items however few
  // tiles there are.  With few tiles (tile_major = 0: x is small, the weights are not) work item w is tile
  // w % dense_tiles of row slice (w / dense_tiles) % slices: the items that read the same weight rows follow
  // one another (same XCD, same moment).  With many tiles (tile_major = 1) the slices of one tile follow one
  // another and an XCD's L2 holds the x rows of the few tiles it works on.  The window is w / (tiles * slices).
  uint32_t dense_tiles, dense_items;
  int tile_major;
  // optional stage stamps: 8 per work item, 100 MHz clock
  unsigned long long* trace;
  uint32_t trace_items;
};

// first K group of window wdx when ng groups are cut into n_win windows (multiples of 8 groups)
__host__ __device__ __forceinline__ uint32_t dense_window_start(uint32_t ng, uint32_t n_win, uint32_t wdx) {
  if (wdx >= n_win) return ng;
  return static_cast<uint32_t>(static_cast<uint64_t>(ng) * wdx / n_win) & ~7u;
}

// bits: 4, 2 (2-bit and ternary codes), or kMixedBits: the routed problem 2-bit, the dense one 4-bit
constexpr int kMixedBits = 24;
inline int part_bits(int bits, const QmmArgs& q) { return bits != kMixedBits ? bits : q.dense_mode ? 4 : 2; }

// tile_slots: entries of the tile list (routed; a multiple of 8) or number of tiles (dense), tiles of TT rows (kTileTokens or
// kSmallTile) in both.  `b` (optional) is a second problem for the same instantiation, run behind `a` in the same launch.  few: the
// form for few work items (tiles of 32 only).
template <int TT>
hipError_t launch_qmm_tiles(hipStream_t s, int bits, const QmmArgs& a, int nproj, uint32_t tile_slots, const QmmArgs* b,
                            uint32_t b_tile_slots, bool few);
template <int TT>
hipError_t launch_kres_tiles(hipStream_t s, int bits, const QmmArgs& a, uint32_t tile_slots, const QmmArgs* b,
                             uint32_t b_tile_slots);
}  // namespace mf
