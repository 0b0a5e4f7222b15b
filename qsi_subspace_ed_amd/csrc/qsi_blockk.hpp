// Block apply shared by qsi_op_apply_block, the FTLM block Lanczos and the
// solve engine: many columns (start vectors or requests) over one or more
// operators, rows cut into 64-row tiles walked by a persistent grid of
// wavefronts.  The kernels live in qsi_block.hip.
#pragma once

#include <hip/hip_runtime.h>

#include "qsi_device.hpp"
#include "qsi_internal.hpp"
#include "qsi_reduce.hpp"

namespace qsi {

constexpr int kBlkThreads = 256;
constexpr int kBlkWaves = kBlkThreads / 64;
constexpr int kTileRows = 64;  // at most
constexpr int kMaxSectors = 8;

struct BlkSector {
  BasisView b;
  const OffTerm* off;
  TermPlanes tp;
  const DiagTerm* dg;
  const double* coeffs;  // n_slots x R, or null
  const CoefClass* cls;  // coefficient classes of the off-diagonal terms
  int n_cls;             // 0: per-term coefficients
  int n_off;
  int n_diag;
  int64_t tile_begin;  // first global tile of this sector, a multiple of kBlkWaves (blk_set_tiles)
  int64_t row_off;     // first row of this sector in the concatenated blocks
  // cached connectivity of the operator, or null (see qsi_op_s)
  const uint64_t* rowptr;
  const uint32_t* cj;
  const uint8_t* cm;
};

struct BlkArgs {
  BlkSector sec[kMaxSectors];
  int n_sec;
  int64_t n_tiles;  // tiles of all sectors (blk_set_tiles)
  int tile_rows;    // rows per tile: a power of two, at most 64 (blk_set_tiles)
  int R;
  int G;            // lanes per row: a power of two >= R (launch_blk_apply sets
                    // its own)
  int64_t ldx, ldy; // row strides of the X and Y blocks (>= R)
  int accumulate;   // Y += H X instead of Y = H X (apply kernel)
  int y_colmajor;   // Y stored column-major: Y[col * ldy + row] (apply kernel)
  int cfg;          // kernel configuration (blk_cfg_*), chosen by the autotuner
};

// Block-apply configuration: bits 0-1 pick the kernel (cached connectivity:
// 4 / 8 / 16 gathers in flight per lane; searching: 6 or 4 lookups in flight
// by the state's words, or 2), bit 2 halves the persistent grid, bit 3 lets the
// cached kernel serve several columns per lane (16-byte gathers; blk_cpl); the
// searching kernel always does.
constexpr int kBlkCfgDefault = 1;
inline int blk_cfg_kernel(int cfg) { return cfg & 3; }
inline bool blk_cfg_half(int cfg) { return (cfg >> 2) & 1; }
inline bool blk_cfg_pairs(int cfg) { return (cfg >> 3) & 1; }

// True when every sector of `a` has its connectivity cached: the block
// apply then gathers through the cached ranks instead of searching.
inline bool blk_cached(const BlkArgs& a) {
  for (int k = 0; k < a.n_sec; ++k)
    if (!a.sec[k].rowptr) return false;
  return a.n_sec > 0;
}

// Columns per lane of a block apply (1, 2 or 4, at most R): one without the
// configuration's bit over cached connectivity, else two, or four in wide cached
// applies of large bases.
int blk_cpl(const BlkArgs& a);

// Cuts the sectors (bases, R and G set) into tiles, one wavefront's work each:
// tile_rows, every tile_begin and n_tiles.
void blk_set_tiles(BlkArgs& a);

// Blocks of a persistent block-apply grid over the tiles of `a`: all resident
// at once (occupancy x compute units), never more than the tiles need.
int blk_apply_blocks(const BlkArgs& a, int nw);

// Y (+)= H X over the sectors of `a` (the block-apply kernels; see
// qsi_block.hip).  partials: n_sec x n_blocks x R, or null.
int launch_blk_apply(const BlkArgs& a, int nw, int n_blocks, const double* X, double* Y,
                     double* partials, hipStream_t s);

// Builds (enable != 0) or frees the operator's cached connectivity.
int op_cache_connectivity(qsi_op_s* op, bool enable, bool allow_pad = true);

}  // namespace qsi
