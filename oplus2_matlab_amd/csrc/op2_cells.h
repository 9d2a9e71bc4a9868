// Cell tiles: the form of the Runge-Kutta stage kernel in which a thread
// evaluates all the edges of one cell (op2_cells.hip).
#pragma once

#include <cmath>
#include <limits>

#include "op2_kernels.h"

namespace op2 {

// The tiles of one owner-gather res_calc plan and one cell -> 4 nodes map.
// Per tile: its owned cells, rings of halo cells around them (ring 1 the
// cells across an edge of an owned cell, ring 2 those across an edge of ring
// 1, ...; listed) and the nodes of its owned cells and of all rings but the
// last (the longest run of consecutive ones of the owned cells, most of them
// on a renumbered mesh, and a list of the others, ring by ring).  Per owned
// cell and per cell of all rings but the last a record of eight 16-bit
// halves: four neighbours, in the order the cell's increments are summed (the
// plan's), then the four nodes, round the cell as in the map.  A node is its
// byte offset in the tile's LDS; a neighbour has its local number (cells: owned
// first, then the rings; kNoCell after the last) from bit 6, from bit 2 the
// side of the cell its edge is (2 bits, side i from node i to i + 1) and
// whether the increment takes the side vector reversed (1), and in bit 0
// whether the cell is the edge's second.  (What a thread unpacks costs it
// instructions, the bound of large meshes: 12 bytes of 10-bit numbers took
// 12 more for each edge.)
constexpr unsigned kNoCell = 1023;
constexpr int kMaxLocal = 1023;  // local cells and local nodes of a tile
constexpr int kMaxRings = 2;
constexpr int kMaxStages = 64;   // of one launch

// The tiles are the plan's blocks, except that a block is cut in halves until
// its parts have no more cells to finish than 1.5 times the plan's tile size
// with two rings (a square tile of 256 cells has 64 cells in its first ring),
// and no more cells and nodes in all than 1.5 times, or twice with two rings
// (ragged blocks with many halo cells, which would otherwise set the threads
// and the LDS of every workgroup).
constexpr int kCellWaves = 24;             // wavefronts per CU: 6 per SIMD
constexpr int kCus = 256;

// Two rings, hence two stages per launch, where the tiles fit on the chip all
// at once.  A launch is then bound by latency: the second stage saves a launch
// and the loads before it, and the quarter of cells finished twice runs on
// idle units.  Larger FP64 meshes are bound by memory as much as by the
// instructions that a cell takes (about 520 a stage; 470 in the FP32 form):
// on tiles of two plan blocks, where a sixth of the cells is finished twice,
// two stages a launch win what the second need not read; the FP32 form keeps
// one stage a launch on single blocks.  us per iteration, one ring on single
// blocks, two rings on single blocks, two rings on pairs:
//   cells        FP64               FP32
//   45k     11.9  10.1  12.4   10.8   8.4   9.5
//   180k    18.0  16.2  18.4   13.8  11.9  12.9
//   361k    28.7  29.3  26.2   19.0  21.0  18.0
//   721k    44.7  48.9  46.8   29.6  36.4  33.2
//   2.88M   165.6 178.3 148.4  82.3  123.5 98.0
// (The rule is not the best everywhere: at 361k FP32 pairs are 5% faster, at
// 721k FP64 single blocks are.)
struct CellForm {
  int rings;
  bool wide;
};
inline CellForm cell_form(int nblocks, int part_size, size_t real_bytes) {
  const int waves = (part_size * 3 / 2 + kWave - 1) / kWave;
  if (nblocks <= kCus * std::max(kCellWaves / waves, 1)) return {2, false};
  if (real_bytes == 8 && part_size == 256) return {2, true};
  return {1, false};
}

// A mesh of at most kWholeCells cells is one tile, without rings, and runs as
// many stages per launch as there are (24x12 cells FP64: 9.7 us an iteration
// against 12.7 with a launch per stage on two tiles).
constexpr int kWholeCells = 512;
// Per tile: first owned cell, owned cells, first list entry, first node of
// the run, nodes in it, first record, then the number of cells up to each
// ring, from 1, and the number of listed nodes of the cells inside it (rings
// that the tiles do not have: as the last).
constexpr int kTileInts = 6 + 2 * kMaxRings;

struct CellTiles {
  op_map pcell = nullptr;
  bool whole = false;                // one tile of all cells
  int depth = 1;                     // rings (whole: none is needed)
  int ntiles = 0;
  // for launches of 1, 2, ... stages: the largest numbers of cells that a
  // tile finishes in the first stage, of its cells and of its nodes
  int max_done[kMaxRings] = {}, max_cells[kMaxRings] = {}, max_nodes[kMaxRings] = {};
  int *d_tile = nullptr;             // kTileInts per tile
  int *d_list = nullptr;             // per tile: ring cells, then nodes outside its run
  unsigned *d_rec = nullptr;         // 4 words per finished cell
  double *partials[2] = {nullptr, nullptr};  // rms partials per stage and tile, as StageBufs'
  // first tile of each plan block, and the end; -1: the block is the second of
  // its tile's pair
  std::vector<int> first_of_block;
  std::vector<std::pair<op_map, int *>> tile_off;  // first tile of each mesh, as StageBufs'
  int stages() const { return whole ? kMaxStages : depth; }  // most per launch
  int rings(int nstages) const { return std::min(nstages, kMaxRings) - 1; }  // index above
};

// The same on the host; empty `rec` when a cell or a tile does not fit the
// form (an increment whose edge is no side of its cell, two increments on
// one side, a wavefront of cells with more than kMaxLocal cells or nodes).
struct CellTilesHost {
  bool whole = false;
  int max_done[kMaxRings] = {}, max_cells[kMaxRings] = {}, max_nodes[kMaxRings] = {};
  std::vector<int> tile, list, first_of_block;
  std::vector<unsigned> rec;
  int ntiles() const { return (int)(tile.size() / kTileInts); }
};
CellTilesHost build_cell_tiles(const Plan &p, op_map pcell, size_t real_bytes, bool whole,
                               bool wide, int depth);

template <typename T>
struct CellArgs {
  const int *tile, *list, *owned;  // owned: null when tiles own consecutive cells
  const uint4 *rec;
  int nblk, nfold;  // tiles; leading workgroups that fold (a multiple of kXcds)
  int cells;        // length of the LDS rows (cells_cap)
  int stages;       // the Runge-Kutta stages to run
  unsigned long long saves;  // bit s: the next iteration's save_soln follows stage s
  const T *x, *adt_in;
  T *q_in;        // (written by save_soln between the stages: one tile only)
  const T *qold;  // null: the state before the first stage is q_in itself
  T *res, *q_out, *adt_out, *qold_out;  // qold_out: null unless save_soln stores a copy
  double *partials;                     // one per tile, stage by stage
  double *out, *log;                    // one tile: it logs its sums itself
  unsigned *log_count, *log_base;       // batched form: log slots of the stages' nseg results
  int nseg;
  bool bres;
  bool adt;                  // adt_calc follows the last stage (it follows all others)
  bool zero_res, store_res;  // of the first stage, of the last
  bool stream;               // the new q bypasses the caches (cells_stream)
  T rcfl;                    // 1 / cfl rounded to nearest; 0: not to be used
};

// LDS of a tile (TileLds): rows of 16-byte vectors for cells_cap cells, and 2
// reals per node.  The rows' length is a constant of the kernel.
constexpr int cells_row_bytes(int real_bytes) { return real_bytes == 8 ? 64 : 32; }
inline int cells_cap(int cells) {
  for (int cap : {256, 384, 512, 768})
    if (cells <= cap) return cap;
  return 1024;
}
inline size_t cells_lds(size_t real_bytes, int cap, int nodes) {
  return (size_t)cells_row_bytes((int)real_bytes) * cap + 2 * real_bytes * (size_t)nodes;
}

// Whether a march's stages write the new q past the caches: when the buffers
// that they alternate between (three states, two adt, x and the records)
// exceed 4/3 of the 256 MB last-level cache, a q kept there would be gone
// before the next stage reads it, and takes the place of data that would
// still be found.  us per iteration, cached and past the caches: FP64 1.45M
// cells (206 MB) 79.2 and 81.4, 2.0M (284 MB) 104.6 and 107.5, 2.88M (409 MB)
// 155.8 and 148.7; FP32 2.88M (226 MB) 82.2 and 86.3, 3.9M (306 MB) 118.2 and
// 113.8, 5.4M (421 MB) 176.5 and 170.8.  (FP64 changes over between 284 and
// 409 MB; the FP32 form already between 226 and 306, by 4%.)
inline bool cells_stream(size_t real_bytes, size_t cells, size_t nodes) {
  return (14 * real_bytes + 16) * cells + 2 * real_bytes * nodes > (size_t)256 * 1000000 / 3 * 4;
}

// Workgroups that fold the previous stages' partials, ahead of the tiles.
inline int cells_fold_blocks(int nseg) { return (std::max(nseg, 1) + kXcds - 1) / kXcds * kXcds; }

// 1 / d for a quotient by d (CellArgs::rcfl), 0 where that cannot be used: d
// not a positive number of moderate size, or with a mantissa of ones alone
// (Markstein's exception).
template <typename T>
T near_reciprocal(T d) {
  int e = 0;
  const T m = std::frexp(d, &e);
  return d > T(0) && std::isfinite(d) && std::abs(e) < 40 &&
                 m != T(1) - std::numeric_limits<T>::epsilon() / 2
             ? T(1) / d
             : T(0);
}

template <typename T>
void launch_cells(int threads, const CellArgs<T> &a, const BresIdx<T> &bi,
                  const AirfoilConsts<T> &k, const CarriedFold &fold, size_t lds,
                  hipStream_t stream);

}  // namespace op2
