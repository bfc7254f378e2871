// Tiles of the fused flux / draining / update kernel: host-built static
// tables (swe_tiles.cpp) and their device view (swe_fused.hip).
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <vector>

namespace swe {

#ifndef SWE_TILE_CELLS
#define SWE_TILE_CELLS 256
#endif
constexpr int kTileCells = SWE_TILE_CELLS;      // cells per tile (the tables also build at 512; the stage kernels' local indices hold 256)
constexpr int kTileMaxLocal = 2 * kTileCells;  // tile cells + ring
constexpr int kTileMaxEval = 3 * kTileCells;   // edge evaluations per tile (LDS flux slots)
static_assert(kTileCells == 256 || kTileCells == 512, "tile size");
constexpr uint32_t kNbWall = 0xffffu, kNbFree = 0xfffeu, kNbOut = 0xfffdu;

// one evaluated edge: its cells and nodes (one 16-byte load)
struct alignas(16) EdgeRec {
  int et0, et1, ep0, ep1;
};

struct TileTables {
  int64_t ntiles = 0;
  std::vector<uint32_t> code;       // [3][T] tile cells: slot << 16 | neighbour code
  std::vector<int> ring_off;        // [ntiles + 1]
  std::vector<int> ring_cell;       // ring cells (global ids), tile by tile
  std::vector<uint32_t> ring_code;  // [ring entry][3] codes of the ring cells
  std::vector<int> ev_off;          // [ntiles + 1]
  std::vector<uint16_t> ev;         // evaluations: local cell << 2 | k
  std::vector<EdgeRec> evrec;       // per evaluation: the edge's et0, et1, ep0, ep1
  std::vector<int> evedge;          // per evaluation: the edge
  int max_eval = 0, max_ring = 0;
};

// false when a tile exceeds the kernel's LDS capacity (a mesh far from a
// cell-local order) or the tables are inconsistent: the fused kernel is
// then not used
bool build_tiles(int64_t T, const int* tt, const int* te, const uint32_t* cflag, const int* et0, const int* et1,
                 const int* ep0, const int* ep1, TileTables& out);

// The stage kernels' view of the tiles: a tile keeps the data of its cells,
// of the ring and of the cells beyond the ring (the other side of the ring
// cells' outer edges), and of the nodes of every evaluated edge in LDS, and
// the tables name them by local index: cells 0 .. kTileCells - 1 the tile's
// own, then the ring, then the cells beyond; nodes those of the tile's own
// cells first.  Indices take 10 bits.
constexpr uint32_t kLocalBits = 10, kLocalMask = (1u << kLocalBits) - 1u;
constexpr uint32_t kLocalWall = kLocalMask, kLocalFree = kLocalMask - 1u;  // in the place of a neighbour
constexpr uint32_t kLocalMax = kLocalFree;  // local indices are below
// Every list of a tile starts at tile * stride (the longest of any tile), so
// that its loads wait for nothing but the tile's number; entries past a
// tile's counts hold valid indices.
struct alignas(16) TileHead {
  uint16_t nr, nx;   // ring cells; ring and beyond
  uint16_t nn0, nn;  // nodes of the own cells; all
  // evaluations: of edges the tile owns (et0 is its cell), which come first;
  // of all edges of its cells, which come before those the ring alone has (a
  // draining step needs the mass flux only); all
  uint16_t ne0, na, ne;
  uint16_t pad;
};
// three local indices per word: vertices, neighbours across edge k (or
// kLocalWall / kLocalFree), flux slots of edge k; and the cell's flags
struct alignas(16) TileCell {
  uint32_t nodes, nbs, slots, flags;
};
struct alignas(8) RingCode {
  uint32_t slots, flags;
};
// an evaluation: local cells et0 | et1 << 10 (or a boundary code), local
// nodes ep0 | ep1 << 10
struct alignas(8) EvalCode {
  uint32_t cells, nodes;
};
struct StageTables {
  int64_t ntiles = 0;
  std::vector<TileHead> head;
  std::vector<TileCell> cell;   // [T]
  int sx = 0, sr = 0, sn = 0, se = 0;  // strides: the largest nx, nr, nn, ne
  int max_own_nodes = 0, max_own_ev = 0;  // the largest nn0, na
  std::vector<int> xcell;       // [tile][sx] global ids of ring and beyond
  std::vector<RingCode> xcode;  // [tile][sr] of the ring cells
  std::vector<int> node;        // [tile][sn] global node ids
  std::vector<EvalCode> ev;     // [tile][se]
  std::vector<int> evedge;      // [tile][se] the edge of each evaluation
};
// build_tiles' tables in this form, built by several threads; false where
// build_tiles refuses the mesh or a local index does not fit
bool build_stage_tables(int64_t T, const int* tp, const int* tt, const int* te, const uint32_t* cflag, const int* et0,
                        const int* et1, const int* ep0, const int* ep1, StageTables& out);

// whether the edges' geometry needs none of the special cases of the IEEE
// square root and division (PlainGeometry): every edge's coordinate
// differences are zero or of magnitude 2^-400 .. 2^400, and not both zero
bool plain_geometry(const double* px, const double* py, int64_t E, const int* ep0, const int* ep1);

struct DevTiles {
  const TileHead* head;
  const TileCell* cell;
  const int* xcell;
  const RingCode* xcode;
  const int* node;
  const EvalCode* ev;
  const int* evedge;
  // static geometry in the tiles' order (the setup kernels): node
  // coordinates [tile][3][sn], centroids [tile][sx][2] of ring and beyond,
  // bathymetry and area [tile][sr][2] of the ring
  double* tnode;
  double* txc;
  double* tring;
  int64_t ntiles;
  int sx, sr, sn, se;  // strides
  int lo, la;          // the most nodes of a tile's own cells, evaluations of its cells' edges
};

constexpr size_t kTileMaxLds = 64 * 1024;  // of one workgroup
constexpr size_t kCuLds = 160 * 1024;
constexpr int kCus = 256;

// Bytes of LDS of a stage kernel's tile, arrays of doubles one after the
// other: the reconstruction of the local cells (w0, gx, gy, u, v, centroid)
// where the fluxes are evaluated (far: without the cells beyond the ring), the
// nodes (x, y, z; those of the own cells alone where that will do), the
// fluxes.  The draining steps take the place of the cells' w0, which nothing
// reads after the fluxes.  ff: the fluxes are read, not evaluated; len:
// SWE_OPT_DRAIN_LENGTH.
inline size_t stage_lds(const DevTiles& P, bool ff, bool far, bool len) {
  const int cells = ff ? kTileCells + P.sr : 7 * (kTileCells + (far ? P.sr : P.sx));
  const int nodes = (ff && !len) || far ? P.lo : P.sn;
  return sizeof(double) * size_t(cells + 3 * nodes + P.se + 2 * P.la);
}
// Whether a launch of n tiles leaves the cells beyond the ring out of LDS:
// where all of them would not fit, or leave a CU two workgroups and there are
// more tiles than that.  At three to a CU the two forms are alike (4M cells,
// us per fused stage staged whole / far: 272 / 268, 311 / 305; with edge
// lengths 301 / 312, 350 / 360), at two far is the faster one (335 / 265), but
// not while all tiles are on the chip at once (307 of them: 17.3 / 18.7).
inline bool stage_far(const DevTiles& P, bool len, int64_t n) {
  const size_t whole = stage_lds(P, false, false, len);
  return whole > kTileMaxLds || (3 * whole > kCuLds && n > 2 * kCus);
}

}  // namespace swe
