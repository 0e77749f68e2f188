// sg_plan_host.hpp -- the host side of a plan: tilings, band windows, LDS
// budgets, the adjoint's gather lists, the transposed band lists and the
// batch's work queues.  Everything here is index arithmetic on host vectors
// (the spans of every dimension); nothing calls the HIP runtime, so the
// same code is built on its own under the address and undefined-behaviour
// sanitizers and driven on the CPU by tests/native/plan_check.cpp.
#pragma once

#include <algorithm>
#include <functional>
#include <vector>

#include "sg_queue.hpp"

namespace sg {

// ---- environment knobs (positive integers; anything else: fallback) ----
int env_int(const char* name, int fallback);

// ---- tilings of the streaming kernels (sg_api.cpp builds the plan) ----

// Band windows of a tiling: tiles of kLanes * wx samples along dimension 1
// (or t.tile_w), chunks of kWaves / wx * rows_per_wave rows (or t.chunk_h)
// along dimension 2.
void compute_tiling(const Plan& pl, Tiling& t, int rows_per_wave, int wx = 1);
// Samples of dimension 3 per workgroup (0: about 1024 workgroups) and the
// widest k3 window of those groups.
void compute_ztiling(const Plan& pl, Tiling& t, int j3_per_block);
// Largest LDS claim of a forward launch (FP64, widest channel block).
size_t forward_lds_worst(const Plan& pl, const Tiling& t);
// LDS of an adjoint streaming launch of nc channels of elem bytes.
size_t adjoint_stream_lds(const Plan& pl, int nc, size_t elem);
// LDS of an MFMA forward launch: nch window channels, nf fields.
size_t mma_lds(const Plan& pl, int nch, int nf);
// NURBS adjoint in FP32: three channels share a workgroup and its weight field
// (else every channel is a workgroup of its own).  Their rings and the
// field's fit 256 registers, two waves per SIMD, up to p3 = kSharedMaxP3.
constexpr int kSharedMaxP3 = 2;
bool adjoint_shares_weights(const Plan& pl);
// Threads one launch may have per grid dimension: HIP refuses 2^32 and more.
constexpr long long kMaxLaunch = (1LL << 32) - 1;
// Parts of `threads` threads each that one launch takes, at least one.
inline long long launch_groups(long long threads) {
  return threads < kMaxLaunch ? kMaxLaunch / threads : 1;
}
// Workgroup numbering of a plan's launches (see xcd_logical_block).
int default_xcd_map(const Plan& pl);

// Every tiling of a plan whose dimensions carry their host spans and
// monotone flags: stream_ok, fwd, mma, and with want_adjoint adj and (when
// adjm_shape_ok) adjm and adjm64, whose runs use resident_waves(plan) -- the
// waves of the matrix-core adjoint the device holds at once for the plan's
// tiling of that type as chosen so far (resident_waves64: FP64, if it differs).
void plan_tilings(Plan& pl, bool want_adjoint, bool adjm_shape_ok,
                  const std::function<int(const Plan&)>& resident_waves,
                  const std::function<int(const Plan&)>& resident_waves64 = nullptr);

// For dimension d and control point k, the element offsets (in the partial
// windows of tiling t, w1 x w2 x t.w3max per channel) of the windows that
// hold k: ptr[d][k] .. ptr[d][k + 1] index off[d].  gchan: offset between
// channels.
struct GatherLists {
  std::vector<int32_t> ptr[3];
  std::vector<long long> off[3];
  long long gchan = 0;
};
GatherLists gather_lists(const Plan& pl, const Tiling& t, int w1, int w2);
// Dimension d's lists as rows of kGatherRow entries, one per control point:
// the list's length, then the list itself where it fits the row, so that both
// come from one cache line; a longer list follows the rows, from the index in
// the row's second entry.  most: the longest list.
std::vector<long long> gather_table(const GatherLists& g, int d, int& most);

// Lanes per control point of the gather (1 or 4), for control points of up to
// `windows` windows and `outputs` control points times channels.  A lane alone
// where its windows are one batch of loads, or where the points fill the chip
// before their windows count: one window in 16 384 points (64 x 64 x 32 x 3: 18
// us with four lanes, 10 with one; 100^3, 12 windows: a whole call 70 and 52).
// Else four (20^3 x 3, up to 75 windows: 14 us with one lane, 7 with four; 73 x 9
// x 26 x 4, 94 windows: a whole call 96 and 72; 30 x 30 x 40 x 2, 152: 122, 78).
constexpr int kGatherBatch = 4;  // loads of windows in flight per lane
inline int gather_lanes(long long windows, long long outputs) {
  return windows > std::max<long long>(kGatherBatch, outputs >> 14) ? 4 : 1;
}

// Transposed band lists of a dimension: the (sample, term) pairs whose band
// holds control point k, j * (p + 1) + a, in sample order, at
// js[ptr[k] .. ptr[k + 1]).
void band_lists(const DimDev& D, std::vector<int32_t>& ptr, std::vector<int32_t>& js);

// Threads per control point and channel of the general adjoint (adj_csr): 1,
// kLanes or kCsrBlock, for `outputs` control points times channels whose band
// lists have `entries` entries on average, in nin dimensions.
constexpr int kCsrBlock = 1024;  // one workgroup per control point
int csr_threads(long long outputs, double entries, int nin);

// ---- the batch's launch (sg_batch.hip) ----

constexpr int kBC = 4;  // value channels per pass; the weight is slab 4
// 3-D tiles' plane list: entries of kEntry floats, weights then k3 at
// kEntryK; entry 0 holds the list's length at kEntryN
constexpr int kEntry = 8;
constexpr int kEntryK = 4;
constexpr int kEntryN = 5;
__host__ __device__ constexpr int plane_list_floats(int p3) {
  return (kWaves * (p3 + 1) + 1) * kEntry;
}

// The plane list of the 3-D batch tile whose kWaves samples j3 start at j3_0
// (`planes` <= kWaves of them inside the grid): one entry per control-point
// plane k3 in the union of their dimension-3 bands, in increasing k3,
// {w[0..kWaves), k3}, where w[pz] is B3 of sample j3_0 + pz at k3 (0 outside
// its band), then one padding entry with zero weights and the last k3, so
// that entries can be taken in pairs.  span3 / tab3: the dimension's spans
// and FP32 order-0 table [m3][p3 + 1].  Writes plane_list_floats(p3) floats
// (the rest zero) and returns the length.
int plane_list_host(const int32_t* span3, const float* tab3, int p3, int j3_0, int planes,
                    float* list);

// LDS one workgroup may take when blocks_per_cu of them share a CU.
size_t lds_cap(int blocks_per_cu);

// Samples j1 per lane a grid's batch tiles may take: 2 for grids of degrees
// p1, p2 <= kVec2MaxDegree whose rows are longer than one wave (tiles of
// 2 kLanes samples, rows stored in 8-byte pairs: half the store
// instructions, and a row of up to 128 samples in one tile), else 1.  Such
// tiles take channel blocks of at most kVec2Slabs window slabs.
constexpr int kVec2MaxDegree = 4;
constexpr int kVec2Slabs = 4;
int batch_vec(const Plan& pl);

// Window sizes of a grid's batch tiles (kLanes * vec samples j1) for a
// rows-per-wave choice.
struct GridTiling {
  int rows, ntx, nty, w1, w2;
  size_t lds;  // bytes of LDS one tile of this grid needs
  int tw;      // samples j1 per tile
};
GridTiling grid_tiling(const Plan& pl, int rows, int vec = 1);

// The tiling of a grid in a batch of `rows_per_wave` under an LDS cap: rows
// halve from rows_per_wave until the window fits; two samples per lane
// where batch_vec allows them and their wider window fits at some number of
// rows (on C5 that beats one sample per lane even with fewer rows), else
// one.  lds > cap when nothing fits (the grid then needs its own launch).
GridTiling batch_grid_tiling(const Plan& pl, int rows_per_wave, size_t cap);

// Workgroups per CU a batch is tiled for (its LDS share; the kernel's 128
// registers allow four waves per SIMD), and its rows per wave by the number of
// tiles that 16 rows give: 8 below one tile per resident workgroup (16 grids,
// 444 tiles: 19.5 us with 16 rows, 18.3 with 8), 32 from six on, where the
// window staging weighs more than the last tiles (1024 grids, 30 785 tiles: 701
// and 649 us; 256 grids, 7 171 tiles, near the line: 167 and 172), else 16 (100
// grids, 3 024 tiles: 57.1, 55.8, 56.7 us with 8, 16, 32; 64 grids, 1 523 tiles:
// 37.7, 41.4, 40.4).
constexpr int kBatchPerCu = 4;
int batch_default_rows(const std::vector<const Plan*>& plans, int cus);

// Cost of a tile of tiling t with `samples` samples in `planes` planes, in
// outputs: what a tile costs at all, its outputs and its windows.  From batches
// of 8 to 400 copies of one grid (66 grids of 16 to 128 samples in 3-D, 32 to 512
// in 2-D, degrees 1 to 4): 4.5 ns, 0.55 ns per 1000 outputs and 1.0 per 1000
// window elements, with 20 % left over per grid.
inline long long batch_tile_cost(const Plan& pl, const GridTiling& t, long long samples,
                                 long long planes) {
  const long long nch = pl.nout + (pl.nurbs ? 1 : 0);
  return 8192 + samples * pl.nout + 2 * planes * t.w1 * t.w2 * nch;
}

// The queues of a tile list.  Grids go to the least loaded queue, largest first,
// whole where that leaves the queues even (their control points then sit in one
// XCD's L2) and else cut into ranges of tiles: no other XCD takes over the tiles
// of a long queue.  Writes the tiles in queue order and the queue starts (host_q:
// zero counters, then starts).
void pack_queues(const std::vector<std::vector<BTile>>& grid_tiles,
                 const std::vector<long long>& grid_cost, std::vector<BTile>& sorted,
                 int* host_q);

}  // namespace sg
