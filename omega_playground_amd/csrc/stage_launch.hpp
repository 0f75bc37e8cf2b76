// Parameter blocks of the stage kernels (kernels_stage.hip), passed by value
// to a single model's launches and kept in tables for an ensemble's.
#pragma once

#include "internal.hpp"

namespace omega_hip {

// momentum and thickness: rows cells of lx lanes per block, ncb such blocks
// per level chunk, tiles = ncb * chunks
struct StageLaunch {
  HexCoef q;
  const int *rec; // neighbourhood records
  int nc, L, lx, rows, ncb, tiles;
  int swz;    // each XCD takes a contiguous range of entries
  int block0; // first block in an ensemble's launch
  StageArgs a;
  DiagOut d;
  const double *x; // momentum del4: the edge field a Laplacian launch reads
  double *y;       // and writes; the del4 term for the momentum launch
  PreOut pre;      // rows for the tendency VJP at this stage input
};

// tracers: work = tiles * level chunks
struct TileLaunch {
  HexCoef q;
  const int *ids; // [tiles][(th + 4)(tw + 4)] cell at each place, row-major
  int nx, ny, tiles_x, nch, work, nc, L, per_block;
  int lx; // lanes of a tile, and with them its cells (TileView)
  int swz, block0;
  StageArgs a;
  DiagOut d;
};

// Fills a stage's parameter blocks (t where a.ntr > 0) for N levels per lane.
void stage_launch(const MeshView &m, const Launch &lc, int N, const HexCoef &q, const StageArgs &a,
                  const DiagOut &d, StageLaunch &p, TileLaunch &t);
int stage_levels(const MeshView &m, const Launch &lc); // N of a model's launches

// Momentum blocks for a kernel that has 256 threads whatever the model's cells
// per block (4 cells of 64 levels would leave three of its wavefronts idle).
inline void whole_blocks(StageLaunch &p) {
  const int nch = p.tiles / p.ncb;
  p.rows = 256 / p.lx;
  p.ncb = (p.nc + p.rows - 1) / p.rows;
  p.tiles = p.ncb * nch;
}

// Fewer tiles than this (two blocks per CU) leave the chip short of blocks, so
// each tracer has blocks of its own; us per RK4 step with del4, a block for all
// tracers of a tile or for each: one layer, 4 tracers 50 against 36 at 144
// tiles, 69 against 66 at 400, but 81 against 98 at 576; 64 layers 60 against
// 48 at 128 tiles, 71 against 62 at 200, 89 against 98 at 288 (2 tracers 69
// against 63), 116 against 123 at 512.
constexpr int kFewTiles = 512;

// Both in one launch, where that is the faster one (kernels_stage_both.hip);
// false: nothing launched.
bool stage_one_launch(int N, const StageLaunch &p, const TileLaunch &t);
// whether the stages of a model take it
bool stage_shares_launch(const MeshView &m, const Launch &lc, int terms, int ntr);
bool launch_stage_both(int N, int lx, const StageLaunch &p, const TileLaunch &t, bool emit, bool pre,
                       hipStream_t s);

// What an ensemble's launches over members with N levels per lane have compiled
// in: the tile shape and terms where the members share them, which is 1 to 3 %
// faster than branching to them (16 mixed members 968 against 978 us per
// step), otherwise every body (kAny).
constexpr int kAny = -1;
struct StageKind {
  int N = 0;
  int v2 = kAny;            // momentum del2
  int lx = kAny, d2 = kAny; // tile lanes and tracer del2, both or neither kAny
  bool d4 = false;          // tracer del4: all members (lx set), or some
};
// One launch of n blocks; block b belongs to the member with parameter block
// desc[who[b]], to none if that is negative.
void launch_stage_batch(const StageKind &k, const StageLaunch *desc, const int *who, int n, bool emit,
                        hipStream_t s);
void launch_tile_batch(const StageKind &k, const TileLaunch *desc, const int *who, int n, bool emit,
                       hipStream_t s);

} // namespace omega_hip
