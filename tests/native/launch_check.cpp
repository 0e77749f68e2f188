// launch_check.cpp -- the launch shapes that the host plan code
// (splinegrids.jl_amd/csrc/sg_plan_host.hip) chooses, on the CPU under the
// address and undefined-behaviour sanitizers: what a launch may ask of the
// runtime, at sizes no test allocates.  The argument names the check; prints
// "launch_check ok <name>" and exits 0, or names the first failure.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <string>
#include <vector>

#include "sg_plan_host.hpp"

using namespace sg;

namespace {

void require(bool ok, const std::string& what) {
  if (!ok) {
    std::fprintf(stderr, "launch_check FAILED: %s\n", what.c_str());
    std::exit(1);
  }
}

// The general adjoint: blocks of max(G, 256) threads over outputs * G threads
// stay below 2^32 for every number of outputs that one thread each can take.
void check_csr_limit() {
  const double entries[] = {1, 48, 49, 100, 300, 1000, 1025, 4096, 4097, 6000, 1e5, 1e7};
  for (long long outputs = 1; outputs < (1LL << 32) - 512; outputs = outputs * 9 / 8 + 1)
    for (int k = 0; k < 12 * 4; ++k) {
      const double e = entries[k / 4];
      const int g = csr_threads(outputs, e, 1 + k % 4);
      require(g == 1 || g == kLanes || g == kCsrBlock, "threads per control point");
      const long long block = g > 256 ? g : 256;
      const long long threads = (outputs * g + block - 1) / block * block;
      require(threads < (1LL << 32), std::to_string(outputs) + " outputs of " + std::to_string(e) +
                                         " entries: " + std::to_string(threads) + " threads");
    }
  // cubic volumes of 120^3 control points x 3 with 4.5 samples per control
  // point and dimension, unsorted; quadratic 4-D grids of 64^4 points x 4
  require(csr_threads(3LL * 120 * 120 * 120, 18.0 * 18 * 18, 3) == kLanes, "5 million outputs");
  require(csr_threads(4LL << 24, 81.0, 4) == 1, "67 million outputs");
}

// Where many outputs fill the chip a thread walks each list: shapes on which a
// wave each took two to three times as long.
void check_csr_many() {
  require(csr_threads(995328, 52.8, 4) == 1, "24^4 x 3 linear control points");
  require(csr_threads(270000, 66.7, 2) == 1, "300^2 x 3 control points of degree 6");
  require(csr_threads(128000, 50.0, 3) == 1, "64 000 x 2 control points of degree 6");
  // and the waves and workgroups that pay
  require(csr_threads(600000, 52.0, 1) == kLanes, "a curve of 200 000 x 3 control points");
  require(csr_threads(131072, 410.0, 3) == kLanes, "131 072 outputs of 410 entries");
  require(csr_threads(11858, 6000.0, 2) == kLanes, "11 858 outputs of 6 000 entries");
  require(csr_threads(1458, 6000.0, 2) == kCsrBlock, "1 458 outputs of 6 000 entries");
  require(csr_threads(20, 8000.0, 1) == kCsrBlock, "20 outputs of 8 000 entries");
}

// A launch of launch_groups(t) parts of t threads is below 2^32, and one more
// part would not be.
void check_groups() {
  for (long long t = 64; t < (1LL << 32); t = t * 3 / 2 + 64) {
    const long long n = launch_groups(t);
    require(n >= 1 && n * t < (1LL << 32) && (n + 1) * t >= (1LL << 32),
            "parts of " + std::to_string(t) + " threads");
  }
}

// Four lanes of the gather share a point's windows where there are many, also
// past 65 536 control points.
void check_gather_lanes() {
  require(gather_lanes(94, 68328) == 4, "73 x 9 x 26 x 4 control points of 94 windows");
  require(gather_lanes(152, 72000) == 4, "30 x 30 x 40 x 2 of 152 windows");
  require(gather_lanes(88, 128000) == 4, "40 x 40 x 40 x 2 of 88 windows");
  require(gather_lanes(75, 24000) == 4, "20^3 x 3 of 75 windows");
  require(gather_lanes(4, 8148) == 1, "four windows are one batch");
  require(gather_lanes(12, 393216) == 1, "64 x 64 x 32 x 3 control points");
  require(gather_lanes(12, 1000000) == 1, "100^3 control points");
}

// A plan's host part for clamped uniform knots and uniform samples: the spans.
Plan make_plan(const std::vector<int>& n, const std::vector<int>& p, const std::vector<int>& m,
               int nout, bool nurbs) {
  Plan pl;
  pl.nin = static_cast<int>(n.size());
  pl.nout = nout;
  pl.nurbs = nurbs ? 1 : 0;
  pl.dims.resize(n.size());
  for (size_t d = 0; d < n.size(); ++d) {
    DimDev& D = pl.dims[d];
    D.n = n[d];
    D.p = p[d];
    D.m = m[d];
    D.h_span.resize(m[d]);
    const int cells = n[d] - p[d];
    for (int j = 0; j < m[d]; ++j) {
      const double t = m[d] > 1 ? static_cast<double>(j) / (m[d] - 1) : 0.0;
      D.h_span[j] = p[d] + std::min(static_cast<int>(t * cells), cells - 1);
    }
  }
  return pl;
}

Plan tiled(const std::vector<int>& n, const std::vector<int>& p, const std::vector<int>& m,
           int nout, bool nurbs) {
  Plan pl = make_plan(n, p, m, nout, nurbs);
  plan_tilings(pl, true, true, [](const Plan&) { return 2048; });
  require(pl.stream_ok, "streaming plan");
  return pl;
}

// The NURBS gradient's rows where they differ from the evaluation's, and where not.
void check_gradient() {
  const Plan dense = tiled({60, 103, 66}, {1, 2, 3}, {99, 270, 159}, 1, true);
  require(dense.fwd.rows_per_wave == 32 && dense.grad.rows_per_wave == 16, "windows crowd the LDS");
  require(tiled({40, 40, 20}, {3, 3, 2}, {333, 301, 157}, 1, true).grad.rows_per_wave == 32,
          "windows that do not");
  const Plan full = tiled({124, 19, 4}, {3, 3, 2}, {167, 264, 31}, 3, true);
  require(full.grad64.rows_per_wave == 16 && full.grad.rows_per_wave == 8, "two workgroups per CU");
  require(tiled({60, 60, 30}, {2, 2, 2}, {300, 300, 300}, 4, true).grad.rows_per_wave == 8,
          "a large volume");
  require(tiled({40, 40, 20}, {3, 3, 2}, {333, 301, 157}, 1, false).grad.n_tiles1 == 0, "no weights");
}

std::string name_of(const Plan& pl) {
  std::string s;
  for (const DimDev& D : pl.dims)
    s += "n" + std::to_string(D.n) + " p" + std::to_string(D.p) + " m" + std::to_string(D.m) + ", ";
  return s + std::to_string(pl.nout) + (pl.nurbs ? " nurbs" : "");
}

// Every block of `len` samples: its window inside the control points, and
// within `widest`.
void check_windows(const DimDev& D, int blocks, int len, int widest, const std::string& what) {
  require(blocks == (D.m + len - 1) / len, what + ": blocks");
  for (int a = 0; a < D.m; a += len) {
    const int lo = D.h_span[a] - D.p, hi = D.h_span[std::min(a + len, D.m) - 1];
    require(lo >= 0 && hi < D.n && hi - lo + 1 <= widest, what + ": window");
  }
}

// The swept forward's tiles: every sample in one, the windows of every tile
// within the LDS that the launch takes.
void check_sweep(const Plan& pl, int k, const std::string& what) {
  const Sweep& t = pl.sweep[k];
  if (t.threads_x == 0) return;
  const DimDev &d1 = pl.dims[0], &d2 = pl.dims[1], &d3 = pl.dims[2];
  const size_t elem = k ? sizeof(double) : sizeof(float);
  const int tw = t.threads_x * (16 / static_cast<int>(elem));
  require(t.threads_x * t.rows <= kThreads, what + ": threads");
  require(t.ntx == (d1.m + tw - 1) / tw && t.nty == (d2.m + t.rows - 1) / t.rows &&
              t.nz == (d3.m + t.run - 1) / t.run,
          what + ": tiles");
  require(t.lds_elements * elem <= static_cast<size_t>(kMaxLds), what + ": LDS");
  require(static_cast<long long>(t.ntx) * t.nty * t.nz * kThreads < (1LL << 32), what + ": grid");
  for (int a = 0; a < d1.m; a += tw)
    for (int z = 0; z < d3.m; z += t.run) {
      const int w1 = d1.h_span[std::min(a + tw, d1.m) - 1] - d1.h_span[a] + d1.p + 1;
      const int planes = d3.h_span[std::min(z + t.run, d3.m) - 1] - d3.h_span[z] + d3.p + 1;
      require(static_cast<size_t>(planes) * t.rows * w1 <= t.lds_elements, what + ": windows");
    }
}

// The gather of a matrix-core tiling as the library lays it out: for every
// control point the tables list the windows that hold it, whose element is the
// one that the workgroup of that window writes.
void check_gather(const Plan& pl, const Tiling& t, const std::string& what) {
  const GatherLists g = gather_lists(pl, t, t.w1max, t.w2max);
  const int nb[3] = {t.n_tiles1, t.n_chunks2, pl.nin == 3 ? t.n_z : 1};
  const int len[3] = {t.tile_width(), t.chunk_rows(), t.j3_per_block};
  const long long plane = static_cast<long long>(t.w1max) * t.w2max;
  const long long block = plane * t.w3max * pl.nout;
  const long long per_block[3] = {block, block * nb[0], block * nb[0] * nb[1]};
  const long long per_point[3] = {1, t.w1max, plane * pl.nout};
  require(g.gchan == plane, what + ": channels");
  for (int d = 0; d < 3; ++d) {
    int most = 0;
    const std::vector<long long> table = gather_table(g, d, most);
    const int n = d < pl.nin ? pl.dims[d].n : 1;
    require(table.size() >= static_cast<size_t>(n) * kGatherRow, what + ": rows");
    for (int k = 0; k < n; ++k) {
      std::vector<long long> want;
      for (int b = 0; b < nb[d]; ++b) {
        if (d >= pl.nin) {
          want.push_back(0);
          continue;
        }
        const DimDev& D = pl.dims[d];
        const int a = b * len[d], lo = D.h_span[a] - D.p, hi = D.h_span[std::min(a + len[d], D.m) - 1];
        if (lo <= k && k <= hi) want.push_back(b * per_block[d] + (k - lo) * per_point[d]);
      }
      const long long* row = table.data() + static_cast<size_t>(k) * kGatherRow;
      require(row[0] == static_cast<long long>(want.size()) && row[0] <= most, what + ": count");
      size_t at = static_cast<size_t>(row - table.data()) + 2;
      if (row[0] > kGatherRow - 2) at = static_cast<size_t>(row[1]);
      require(at + want.size() <= table.size(), what + ": list");
      require(std::equal(want.begin(), want.end(), table.begin() + at), what + ": offsets");
    }
  }
}

// Every tiling of plans over degrees, sizes and densities: the four forward
// tilings, the gradient's, the swept forward's, both adjoints' and the batch's.
void check_tilings() {
  std::mt19937_64 rng(0x711E5);
  const auto pick = [&](int a, int b) { return std::uniform_int_distribution<int>(a, b)(rng); };
  std::vector<Plan> plans;
  const auto add = [&](const std::vector<int>& n, const std::vector<int>& p, const std::vector<int>& m,
                       int nout, bool nurbs) {
    Plan pl = make_plan(n, p, m, nout, nurbs);
    plan_tilings(pl, true, pl.nin == 2 || pl.dims[2].p <= kMaxStreamDegree,
                 [](const Plan&) { return 4096; }, [](const Plan&) { return 1024; });
    plans.push_back(pl);
  };
  add({64, 64, 32}, {3, 3, 2}, {512, 512, 256}, 3, true);
  add({64, 64, 32}, {3, 3, 2}, {512, 512, 256}, 1, false);
  add({40, 40, 20}, {3, 3, 3}, {400, 400, 200}, 3, false);
  add({40, 40, 20}, {3, 3, 3}, {400, 401, 203}, 1, false);
  add({128, 128}, {3, 3}, {4096, 4096}, 1, false);
  add({200, 150}, {5, 5}, {210, 160}, 4, true);
  add({9, 8, 30}, {2, 1, 1}, {700, 9, 901}, 1, false);
  for (int i = 0; i < 400; ++i) {
    const int nin = 2 + i % 2;
    std::vector<int> n, p, m;
    for (int d = 0; d < nin; ++d) {
      const int limit = nin == 2 ? 2500 : i % 5 ? 90 : 260;
      m.push_back(static_cast<int>(std::exp(std::uniform_real_distribution<double>(0.0, std::log(limit))(rng))));
      p.push_back(pick(0, 5));
      n.push_back(p[d] + 1 + pick(0, std::max(1, m[d])));
    }
    add(n, p, m, pick(1, 5), i % 3 == 0);
  }
  for (const Plan& pl : plans) {
    const std::string nm = name_of(pl);
    if (!pl.stream_ok) continue;
    const long long m3 = pl.nin == 3 ? pl.dims[2].m : 1;
    const Tiling* forward[] = {&pl.fwd, &pl.fwd64, &pl.fields, &pl.fields64, &pl.grad, &pl.grad64};
    for (int k = 0; k < 6; ++k) {
      const Tiling& t = *forward[k];
      const std::string what = nm + " forward tiling " + std::to_string(k);
      if (k >= 4 && !pl.nurbs) continue;
      check_windows(pl.dims[0], t.n_tiles1, t.tile_width(), t.w1max, what);
      check_windows(pl.dims[1], t.n_chunks2, t.chunk_rows(), t.w2max, what);
      require(forward_lds_worst(pl, t) <= static_cast<size_t>(kMaxLds), what + ": LDS");
      require(m3 * t.n_tiles1 * t.n_chunks2 * kThreads < (1LL << 32), what + ": grid");
    }
    for (int k = 0; k < 2; ++k) check_sweep(pl, k, nm + " sweep " + std::to_string(k));
    for (const Tiling* t : {&pl.adjm, &pl.adjm64}) {
      if (t->n_tiles1 == 0) continue;
      const std::string what = nm + (t == &pl.adjm ? " adjm" : " adjm64");
      require(t->w1max <= kAdjMmaWin && t->w2max <= kAdjMmaWin, what + ": window edge");
      const int waves = t->chunk_rows() / t->rows_per_wave;
      require((waves == 1 || waves == 2 || waves == 4) && waves * t->rows_per_wave == t->chunk_rows(),
              what + ": waves");
      check_windows(pl.dims[0], t->n_tiles1, t->tile_width(), t->w1max, what);
      check_windows(pl.dims[1], t->n_chunks2, t->chunk_rows(), t->w2max, what);
      if (pl.nin == 3) check_windows(pl.dims[2], t->n_z, t->j3_per_block, t->w3max, what);
      check_gather(pl, *t, what);
    }
    require((pl.adjm.n_tiles1 > 0) == (pl.adjm64.n_tiles1 > 0), nm + ": both types or none");
  }
  // the batch's rows, and its longest queue
  for (size_t count : {size_t(1), size_t(5), plans.size()}) {
    std::vector<const Plan*> some;
    for (size_t i = 0; i < count; ++i)
      if (plans[i].stream_ok) some.push_back(&plans[i]);
    const int rows = batch_default_rows(some, 256);
    require(rows == 8 || rows == 16 || rows == 32, "batch rows");
  }
  std::vector<int> q(kQueueInts, 0);
  for (int i = 0; i <= kXcds; ++i) q[kXcds * kQueueStride + i] = i < 3 ? 0 : 7 * i - 5;
  require(longest_queue(q.data()) == 16, "longest queue");
}

struct Packed {
  std::vector<BTile> tiles;
  std::vector<int> q;
  double longest = 0.0, mean = 0.0;  // queue costs
  const int* start() const { return q.data() + kXcds * kQueueStride; }
};

// The queues of a batch at 16 rows; checks that they hold each grid's tiles
// once, and in each queue as ranges of neighbours.
Packed pack(const std::vector<Plan>& plans, const std::string& what) {
  std::vector<std::vector<BTile>> grid_tiles;
  std::vector<long long> cost;
  for (size_t g = 0; g < plans.size(); ++g) {
    const Plan& pl = plans[g];
    const GridTiling t = batch_grid_tiling(pl, 16, lds_cap(kBatchPerCu));
    const int nz = pl.nin == 3 ? (pl.dims[2].m + kWaves - 1) / kWaves : 1;
    std::vector<BTile> tiles;
    long long sum = 0;
    for (int z = 0; z < nz; ++z)
      for (int y = 0; y < t.nty; ++y)
        for (int x = 0; x < t.ntx; ++x) {
          tiles.push_back(BTile{static_cast<int>(g), x, y, z});
          sum += batch_tile_cost(pl, t, 64LL * 64 * (pl.nin == 3 ? kWaves : 1), pl.nin == 3 ? kWaves : 1);
        }
    grid_tiles.push_back(tiles);
    cost.push_back(sum);
  }
  Packed out;
  out.q.assign(kQueueInts, -1);
  pack_queues(grid_tiles, cost, out.tiles, out.q.data());
  std::vector<size_t> held(plans.size(), 0);
  for (int q = 0; q < kXcds; ++q) {
    double load = 0.0;
    std::vector<char> seen(plans.size(), 0);
    for (int i = out.start()[q]; i < out.start()[q + 1]; ++i) {
      const BTile& t = out.tiles[i];
      const std::vector<BTile>& of = grid_tiles[t.grid];
      load += static_cast<double>(cost[t.grid]) / of.size();
      ++held[t.grid];
      if (i > out.start()[q] && out.tiles[i - 1].grid == t.grid) {
        const Plan& pl = plans[t.grid];
        const GridTiling gt = batch_grid_tiling(pl, 16, lds_cap(kBatchPerCu));
        const auto at = [&](const BTile& b) { return (static_cast<long long>(b.bz) * gt.nty + b.by) * gt.ntx + b.bx; };
        require(at(t) > at(out.tiles[i - 1]), what + ": tiles in order");
      } else {
        require(!seen[t.grid], what + ": a queue holds one range of a grid");
        seen[t.grid] = 1;
      }
    }
    out.longest = std::max(out.longest, load);
    out.mean += load / kXcds;
  }
  for (size_t g = 0; g < plans.size(); ++g)
    require(held[g] == grid_tiles[g].size(), what + ": every tile once");
  return out;
}

// No workgroup takes a tile of another XCD's queue, so the queues themselves
// have to be even: single grids, a large one among small ones, uneven ones.
void check_queues() {
  std::mt19937_64 rng(0x0DD);
  const auto pick = [&](int a, int b) { return std::uniform_int_distribution<int>(a, b)(rng); };
  const auto even = [&](const std::vector<Plan>& plans, const std::string& what) {
    const Packed q = pack(plans, what);
    if (q.tiles.size() < 32 * kXcds) return;  // a tile is more than 1/32 of a queue
    require(q.longest <= 1.1 * q.mean, what + ": longest queue " + std::to_string(q.longest / q.mean) +
                                           " of the mean");
  };
  even({make_plan({40, 40, 20}, {3, 3, 2}, {256, 255, 200}, 3, false)}, "one volume");
  even({make_plan({64, 64}, {3, 3}, {2000, 1500}, 3, true)}, "one surface");
  for (int count : {1, 2, 3, 4, 8, 9, 16, 32, 64, 256})
    for (int rep = 0; rep < 20; ++rep) {
      std::vector<Plan> plans;
      for (int i = 0; i < count; ++i) {
        const int nin = i < count / 2 ? 2 : 3;
        std::vector<int> n, p, m;
        for (int d = 0; d < nin; ++d) {
          n.push_back(pick(8, 64));
          p.push_back(pick(1, 4));
          m.push_back(nin == 2 ? pick(32, 512) : pick(16, 128));
        }
        plans.push_back(make_plan(n, p, m, i % 2 ? 3 : 1, i % 4 == 0));
      }
      const std::string what = std::to_string(count) + " grids";
      even(plans, what);
      plans.push_back(make_plan({40, 40, 20}, {3, 3, 2}, {256, 255, 200}, 3, false));
      even(plans, what + " and a large one");
    }
}

}  // namespace

int main(int argc, char** argv) {
  const std::string name = argc > 1 ? argv[1] : "";
  if (name == "csr_limit")
    check_csr_limit();
  else if (name == "csr_many")
    check_csr_many();
  else if (name == "groups")
    check_groups();
  else if (name == "queues")
    check_queues();
  else if (name == "gather_lanes")
    check_gather_lanes();
  else if (name == "gradient")
    check_gradient();
  else if (name == "tilings")
    check_tilings();
  else
    require(false, "no check named '" + name + "'");
  std::printf("launch_check ok %s\n", name.c_str());
  return 0;
}
