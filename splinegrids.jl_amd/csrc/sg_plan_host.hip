// sg_plan_host.hip -- host-side plan arithmetic (sg_plan_host.hpp): no HIP
// runtime calls, no kernels.  Built into the library, and on its own under
// the sanitizers by the CPU test of tests/native/plan_check.cpp.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <numeric>

#include "sg_plan_host.hpp"

namespace sg {

constexpr size_t kLdsPerCu = 160 * 1024;

int env_int(const char* name, int fallback) {
  const char* v = std::getenv(name);
  if (!v || !*v) return fallback;
  const int x = std::atoi(v);
  return x > 0 ? x : fallback;
}

// Rows of dimension 1 whose length is not a multiple of 128 bytes make
// neighbouring tiles share a cache line; keep such tiles on one XCD.
int default_xcd_map(const Plan& pl) {
  return (pl.dims[0].m * sizeof(float)) % 128 == 0 ? 0 : 2;
}

void compute_tiling(const Plan& pl, Tiling& t, int rows_per_wave, int wx) {
  const DimDev& d1 = pl.dims[0];
  const DimDev& d2 = pl.dims[1];
  const std::vector<int32_t>& s1 = d1.h_span;
  const std::vector<int32_t>& s2 = d2.h_span;
  t.rows_per_wave = rows_per_wave;
  t.wx = wx;
  const int tw = t.tile_width();
  t.n_tiles1 = (d1.m + tw - 1) / tw;
  t.w1max = 0;
  for (int i = 0; i < t.n_tiles1; ++i) {
    const int a = i * tw, b = std::min(a + tw, d1.m) - 1;
    t.w1max = std::max(t.w1max, s1[b] - s1[a] + d1.p + 1);
  }
  const int chunk = t.chunk_rows();
  t.n_chunks2 = (d2.m + chunk - 1) / chunk;
  t.w2max = 0;
  t.w2wave_max = 0;
  for (int c = 0; c < t.n_chunks2; ++c) {
    const int a = c * chunk, b = std::min(a + chunk, d2.m) - 1;
    t.w2max = std::max(t.w2max, s2[b] - s2[a] + d2.p + 1);
    for (int w = 0; w < kWaves / wx; ++w) {
      const int ra = a + w * rows_per_wave;
      const int rb = std::min(ra + rows_per_wave, b + 1) - 1;
      if (ra > rb) continue;
      t.w2wave_max = std::max(t.w2wave_max, s2[rb] - s2[ra] + d2.p + 1);
    }
  }
}

// the band window of fwd_stream; the MFMA kernels add their chunk's B2 rows
size_t forward_lds_worst(const Plan& pl, const Tiling& t) {
  const int nc = std::min(pl.nout, 4) + (pl.nurbs ? 1 : 0);
  const size_t p2 = static_cast<size_t>(pl.dims[1].p);
  return (static_cast<size_t>(nc) * t.w1max * t.w2max + t.chunk_rows() * (p2 + 1)) *
             sizeof(double) +
         static_cast<size_t>(t.chunk_rows()) * sizeof(int);
}

// Samples of dimension 3 per adjoint workgroup: enough workgroups to fill
// the chip (about 8 per CU), as few as possible beyond that so that each
// k3 window is shared by many j3.
void compute_ztiling(const Plan& pl, Tiling& t, int j3_per_block) {
  if (pl.nin != 3) {
    t.j3_per_block = 1;
    t.n_z = 1;
    t.w3max = 1;
    return;
  }
  const DimDev& d3 = pl.dims[2];
  if (j3_per_block <= 0) {
    const long long xy = static_cast<long long>(t.n_tiles1) * t.n_chunks2;
    const long long target = 1024;
    j3_per_block = static_cast<int>(std::max<long long>(1, (xy * d3.m) / target));
  }
  t.j3_per_block = std::min(j3_per_block, d3.m);
  t.n_z = (d3.m + t.j3_per_block - 1) / t.j3_per_block;
  t.w3max = 0;
  for (int z = 0; z < t.n_z; ++z) {
    const int a = z * t.j3_per_block, b = std::min(a + t.j3_per_block, d3.m) - 1;
    t.w3max = std::max(t.w3max, d3.h_span[b] - d3.h_span[a] + d3.p + 1);
  }
}

// adj_stream: each wave's partial window of its rows, the dimension-1 B
// rows, the (p3 + 1)-slab ring of the workgroup's window, the chunk's B2
// rows and the row / span bookkeeping
size_t adjoint_stream_lds(const Plan& pl, int nc, size_t elem) {
  const Tiling& t = pl.adj;
  const int p3 = pl.nin == 3 ? pl.dims[2].p : 0;
  const size_t ls = kLanes + 16 / elem;
  const size_t chunk = static_cast<size_t>(t.chunk_rows());
  return static_cast<size_t>(kWaves) * t.w2wave_max * nc * ls * elem +
         static_cast<size_t>(t.w1max) * ls * elem +
         static_cast<size_t>(p3 + 1) * t.w1max * t.w2max * nc * elem +
         chunk * (pl.dims[1].p + 1) * elem +
         (chunk + 2 * kWaves + 2 * t.w1max) * sizeof(int);
}

// mma_stream: G for nch channels, the chunk's B2 rows of nf fields and its
// spans
size_t mma_lds(const Plan& pl, int nch, int nf) {
  const Tiling& t = pl.mma;
  return (static_cast<size_t>(nch) * t.w1max * t.w2max +
          static_cast<size_t>(nf) * t.chunk_rows() * (pl.dims[1].p + 1)) * sizeof(float) +
         static_cast<size_t>(t.chunk_rows()) * sizeof(int);
}

bool adjoint_shares_weights(const Plan& pl) {
  return pl.nurbs && pl.nout > 1 && (pl.nin == 2 || pl.dims[2].p <= kSharedMaxP3);
}

namespace {

size_t adjoint_lds_min(const Plan& pl) {  // one channel, FP64
  return adjoint_stream_lds(pl, 1, sizeof(double));
}

// Rows of a wave when `waves` waves of at most `most` rows share a chunk: the
// chunks of dimension 2 as even as whole rows allow (a last chunk of a few
// rows would leave most of its workgroup idle).
void balanced_rows(const Plan& pl, Tiling& t, int most, int waves) {
  const int m2 = pl.dims[1].m;
  const int chunks = (m2 + most * waves - 1) / (most * waves);
  const int rows = (m2 + chunks * waves - 1) / (chunks * waves);
  t.chunk_h = rows * waves;
  compute_tiling(pl, t, rows);
}

// Matrix-core adjoint: tiles of 64 (or 32) samples j1 and workgroups of 4, 2
// or 1 waves of up to 16 rows j2 (2-D: up to 128) whose band windows fit one
// 16 x 16 MFMA tile, and runs of samples j3 (see below).  Leaves the tiling t
// (pl.adjm or pl.adjm64) empty when the bands do not fit.
void plan_adjoint_mma(Plan& pl, Tiling& t, size_t elem,
                      const std::function<int(const Plan&)>& resident_waves) {
  // workgroups per tile, chunk and run: the channels, or with NURBS weights in
  // FP32 the groups of three that share a weight field
  const long long groups =
      elem == sizeof(float) && adjoint_shares_weights(pl) ? (pl.nout + 2) / 3 : pl.nout;
  const auto fit = [&](int tile, int most) {  // most waves per workgroup that fit
    t = Tiling();
    t.tile_w = tile;
    for (int waves : {4, 2, 1}) {
      balanced_rows(pl, t, most, waves);
      if (t.w1max > kAdjMmaWin) return false;
      if (t.w2max <= kAdjMmaWin) return true;
    }
    t.chunk_h = 16;  // every chunk of a multiple of 16 rows that fits holds these
    compute_tiling(pl, t, 16);
    return t.w2max <= kAdjMmaWin;
  };
  const int tile = fit(64, 16) ? 64 : fit(32, 16) ? 32 : 0;
  if (tile == 0) {
    t = Tiling();
    return;
  }
  if (pl.nin == 2) {
    // more rows per wave amortise a wave's set-up, as long as every CU keeps
    // two workgroups and the chunk's window fits
    const Tiling one = t;
    if (one.chunk_rows() == 4 * one.rows_per_wave) {
      for (int most : {128, 64, 32}) {
        t = Tiling();
        t.tile_w = tile;
        balanced_rows(pl, t, most, 4);
        if (t.w2max <= kAdjMmaWin && groups * t.n_tiles1 * t.n_chunks2 >= 512) break;
        t = one;
      }
    }
    compute_ztiling(pl, t, 1);
    return;
  }
  int j3 = env_int("SG_ADJM_J3", 0);
  if (j3 <= 0) {
    // Runs of j3: the number that minimises a fit to measured times (14
    // grids of 2 to 805 MB, FP32 and FP64, every run length; furthest from the
    // best since: NURBS 230 x 281 x 132, 47 us in its 12 runs, 42 in 22).  Few
    // long runs leave
    // few partial windows; what costs is a last round of workgroups that
    // leaves CUs idle (400 x 400 x 200 samples: 88 us with 735 workgroups,
    // 100 us with 588), and less than 32 KB of ebar in flight per CU (one
    // unit per wave).  Runs shorter than 16 samples are never cut so short that
    // not all workgroups are resident at once: their prologues would not overlap
    // (FP64 NURBS, one wave per SIMD, 51 x 11 x 286 samples x 4: 40 us in 384
    // workgroups of 3 samples, 27 in 192 of 6).  Longer ones may take what four
    // waves per SIMD hold, in several rounds (FP64 NURBS 300 x 301 x 150 x 4: 191
    // us in 500 workgroups, 254 in 200).
    const long long xy = groups * t.n_tiles1 * t.n_chunks2;
    const int m3 = pl.dims[2].m;
    const int waves = t.chunk_rows() / t.rows_per_wave;
    const long long most = std::max<long long>(resident_waves(pl) / waves, 1);
    const long long rounds = std::max<long long>(most, 16 * kCus / waves);
    const double unit = 16.0 * t.tile_w * 4 * waves, window = t.w1max * t.w2max;
    const double samples = 1.0 * pl.dims[0].m * pl.dims[1].m * m3;
    double best = 0.0;
    for (int runs = 1, last = 0; runs <= m3; ++runs) {
      const int len = (m3 + runs - 1) / runs, n = (m3 + len - 1) / len;
      if (runs > 1 && xy * runs > (len < 16 ? most : rounds)) break;
      if (len == last) continue;
      last = len;
      compute_ztiling(pl, t, len);
      const double per_cu = static_cast<double>(xy) * n / kCus;
      const double idle = std::ceil(per_cu) / per_cu - 1.0;
      const double hungry = std::max(32768.0 / (unit * per_cu) - 1.0, 0.0);
      const double partial = 1.0 * t.n_tiles1 * t.n_chunks2 * n * t.w3max * window / samples;
      const double cost = 1.0 * len * n / m3 * (1.0 + 0.2 * idle) * (1.0 + 0.15 * hungry) +
                          4.0 * partial;
      if (j3 <= 0 || cost < best) {
        best = cost;
        j3 = len;
      }
    }
  }
  compute_ztiling(pl, t, j3);
}

// Forward tiles.  What bounds these kernels is the rate of their stores, and
// that is set by how close together in time the pieces of one line and of one
// DRAM page are written; so the waves of a workgroup stand side by side along
// dimension 1 (unless that leaves over 11 % more of their lanes past the row's
// end: 439x111x60, 3 channels, four fields 56.5 us with four, 55 with one), few
// rows deep:
//   - rows of whole 64-byte sectors: no sector is shared; the launch order is
//     kept, or by rows where a 128-byte line is shared.  16 rows: 512x512x256,
//     3 channels, NURBS 145 us (32 rows of one wave 156).
//   - other rows: the sector at a tile's edge waits in L2 for its other half,
//     so workgroups are numbered in contiguous ranges per XCD.  16 rows too,
//     but 8 for volumes of 100 MB and more and of 12 bytes per sample (16 where
//     two waves span the row): the wider a row of the volume, the fewer rows
//     may pass before that half comes.  300x300x300, 4 channels 98 us (128; 16
//     rows 130); 603x301x99, 3 channels 54 (67; 16 rows 60).  Smaller outputs
//     stay in the last-level cache, where the columns that 8 rows compute
//     again weigh more (362x32x240, 4 channels: 16.7 us in 8 rows, 14.8);
//     2-D grids have 16 (8001x6001, 3 channels 114 us, 8 rows 129; 171).
//   - several fields in a launch are several streams of stores at one sample
//     each: 16 rows (4096x4096, four fields 45 us, 57 with 32 rows; 203x311x160,
//     2 channels, four fields 83 us, 8 rows 100).
//   - one FP32 channel: a wave writes so little per row that its first columns
//     (stage 1, first band) weigh more than the stores: 32 rows.  3001x3001
//     14.6 us (16 rows 14.9), 251x250x251 22 (16 rows 26).
// Small grids take fewer rows, to two workgroups per CU: 1027x773, 3 channels
// 7.4 us at 8 rows, 7.8 at 16.  (Earlier figures in brackets.)
// The NURBS gradient takes the tiles of one field (three fields of 333x301x157,
// 3 channels: 144 us, with those of several 175; 300x300x300, 4 channels 358,
// 431), but FP64 kernels of three channels, which fill a CU with two workgroups,
// take no fewer rows for a second round of them (167x264x31: 465 workgroups of
// 16 rows 26 us, 837 of 8 rows 32), and no 32 rows where the windows, twice the
// channels', crowd the LDS (99x270x159 of 60x103x66, scalar: 39 us, 16 rows 29).
struct ForwardShape {
  int rows = 16, wx = 1, xcd_map = 0;
};

ForwardShape forward_shape(const Plan& pl, size_t elem, bool several, bool gradient = false) {
  const DimDev& d1 = pl.dims[0];
  const int m1 = d1.m, m2 = pl.dims[1].m;
  const long long m3 = pl.nin == 3 ? pl.dims[2].m : 1;
  const size_t sample = elem * std::max(pl.nout, 1);
  const bool thin = sample <= sizeof(float) && !several;
  ForwardShape s;
  auto tiles = [&](int wx) { return (m1 + kLanes * wx - 1) / (kLanes * wx); };
  for (int wx : {2, 4})
    if (tiles(wx / 2) > 1 && tiles(1) >= 0.89 * wx * tiles(wx)) s.wx = wx;
  auto chunks = [&](int rows) {
    const int h = rows * (kWaves / s.wx);
    return (m2 + h - 1) / h;
  };
  const bool whole = m1 * elem % 64 == 0;
  s.xcd_map = !whole || thin ? 1 : m1 * elem % 128 == 0 ? 0 : 2;
  if (thin) {
    const int h = 32 * (kWaves / s.wx);
    if (m2 >= 0.8 * h * chunks(32)) s.rows = 32;
  } else if (!several && !whole && pl.nin == 3 && tiles(1) > 1 &&
             sample >= (m1 > 2 * kLanes ? 12 : 16) && 1.0 * m1 * m2 * m3 * sample >= 1e8) {
    s.rows = 8;
  }
  auto groups = [&](int rows) { return m3 * tiles(s.wx) * chunks(rows); };
  // (two per CU is all that the FP64 gradient's kernels of three channels hold)
  const bool full = gradient && elem == sizeof(double) && pl.nin == 3 && pl.nout >= 3;
  while (s.rows > 8 && groups(s.rows) < 2 * kCus &&
         !(full && groups(s.rows / 2) > 2 * kCus))
    s.rows /= 2;
  while (s.rows < 32 && groups(s.rows) > (1 << 23)) s.rows *= 2;  // grid limit: 2^24
  s.wx = env_int("SG_FWD_WX", s.wx);
  if (s.wx != 1 && s.wx != 2 && s.wx != 4) s.wx = 1;
  s.rows = env_int("SG_FWD_ROWS", s.rows);
  if (const char* xm = std::getenv("SG_XCD_MAP"); xm && *xm) s.xcd_map = std::atoi(xm);
  return s;
}

// The swept forward's tiles, where it is the faster kernel: one channel (its
// kernels take degrees 1 to 4 in dimensions 1 and 3), and
// enough samples to pay for its longer prologue (1.5 M; 115x64x53 is launch
// time in both).  Runs are as long as leaves two workgroups per CU: 200x200x200
// 15.5 us in runs of 8 (1000 workgroups), 16.9 in 16, 19.0 in 4.  With two
// channels the ring takes the registers that hide the prologue (500x500x100:
// 57.8 us, streamed 46.3; 256x256x200 quartic: 39, 34; 40x700x700: 41, 45), and
// where stage 1 computes more than 0.75 of the samples' number it is the larger
// part (200x200x80 of 160x160x64 control points: 35.2, 35.3).
void plan_sweep(const Plan& pl, size_t elem, Sweep& t) {
  const DimDev &d1 = pl.dims[0], &d2 = pl.dims[1];
  auto in_range = [](const DimDev& d) { return d.p >= 1 && d.p <= 4; };
  if (pl.nin != 3 || pl.nout != 1 || pl.nurbs || pl.nt_stores || !in_range(d1) ||
      !in_range(pl.dims[2]))
    return;
  const DimDev& d3 = pl.dims[2];
  const double samples = 1.0 * d1.m * d2.m * d3.m;
  if (samples < 1000.0 * env_int("SG_SWEEP_MIN", 1500)) return;  // thousands
  const int vec = 16 / static_cast<int>(elem);
  const int across = (d1.m + vec - 1) / vec;  // threads that a row takes
  const int ntx = (across + kThreads - 1) / kThreads;
  const int tx = (across + ntx - 1) / ntx;
  // rows: the tile that leaves the fewest lanes of its waves idle, larger
  // tiles where that is equal to 2 %
  int rows = 1;
  double best = 0.0;
  for (int r = 1; r * tx <= kThreads && r <= d2.m; ++r) {
    const int waves = (r * tx + kLanes - 1) / kLanes;
    const double full = 1.0 * r * tx / (kLanes * waves) + 0.01 * waves;
    if (full > best + 0.02) {
      best = full;
      rows = r;
    }
  }
  const int nty = (d2.m + rows - 1) / rows;
  int w1 = 0;
  for (int i = 0; i < ntx; ++i) {
    const int a = i * tx * vec, b = std::min(a + tx * vec, d1.m) - 1;
    w1 = std::max(w1, d1.h_span[b] - d1.h_span[a] + d1.p + 1);
  }
  for (int run = 16; run >= 4; run /= 2) {
    const int nz = (d3.m + run - 1) / run;
    if (run > 4 && 1.0 * ntx * nty * nz < 2 * kCus) continue;
    int planes = 0;
    for (int a = 0; a < d3.m; a += run)
      planes = std::max(planes, d3.h_span[std::min(a + run, d3.m) - 1] - d3.h_span[a] + d3.p + 1);
    const size_t elements = static_cast<size_t>(planes) * rows * w1;
    if (elements * elem > static_cast<size_t>(kMaxLds) / 2) continue;
    if (1.0 * elements > 0.75 * rows * tx * vec * run) continue;
    if (1.0 * ntx * nty * nz > (1 << 23)) continue;  // grid limit
    t.threads_x = tx;
    t.rows = rows;
    t.ntx = ntx;
    t.nty = nty;
    t.run = run;
    t.nz = nz;
    t.lds_elements = elements;
    t.xcd_map = d1.m * elem % 64 == 0 ? 0 : 1;  // as the streaming kernel's rows
    return;
  }
}

}  // namespace

void plan_tilings(Plan& pl, bool want_adjoint, bool adjm_shape_ok,
                  const std::function<int(const Plan&)>& resident_waves,
                  const std::function<int(const Plan&)>& resident_waves64) {
  // streaming kernels: Nin 2-3, monotone spans, p1, p2 <= 5, non-empty grid
  bool ok = (pl.nin == 2 || pl.nin == 3);
  for (int d = 0; ok && d < pl.nin; ++d) ok = pl.dims[d].monotone && pl.dims[d].m > 0;
  ok = ok && pl.dims[0].p <= kMaxStreamDegree && pl.dims[1].p <= kMaxStreamDegree;
  pl.nt_stores = env_int("SG_NT_STORES", 0) ? 1 : 0;
  if (ok) {
    const char* xm = std::getenv("SG_XCD_MAP");
    const int xcd = (xm && *xm) ? std::atoi(xm) : default_xcd_map(pl);
    Tiling* const tilings[6] = {&pl.fwd, &pl.fields, &pl.grad, &pl.fwd64, &pl.fields64, &pl.grad64};
    for (int k = 0; k < 6; ++k) {
      const size_t elem = k / 3 ? sizeof(double) : sizeof(float);
      const bool gradient = k % 3 == 2;
      if (gradient && !pl.nurbs) continue;
      ForwardShape f = forward_shape(pl, elem, k % 3 == 1, gradient);
      Tiling& fwd = *tilings[k];
      compute_tiling(pl, fwd, f.rows, f.wx);
      // four windows of one channel: the NURBS gradient's least (two fields of
      // numerator and denominator), which a wider tile must not push out
      auto fits = [&]() {
        const size_t four = 4 * sizeof(double) * fwd.w1max * fwd.w2max;
        return std::max(forward_lds_worst(pl, fwd), f.wx > 1 ? four : 0) <=
               static_cast<size_t>(kMaxLds);
      };
      while (!fits() && (f.rows > 1 || f.wx > 1)) {
        if (f.wx > 1)
          f.wx /= 2;
        else
          f.rows /= 2;
        compute_tiling(pl, fwd, f.rows, f.wx);
      }
      // the gradient's windows, twice the channels', leave eight workgroups per CU
      if (gradient && f.rows > 16 && 4 * elem * fwd.w1max * fwd.w2max > kLdsPerCu / 8)
        compute_tiling(pl, fwd, 16, f.wx);
      fwd.xcd_map = f.xcd_map;
      ok = ok && forward_lds_worst(pl, fwd) <= static_cast<size_t>(kMaxLds);
    }
    for (int k = 0; k < 2; ++k)
      if (ok) plan_sweep(pl, k ? sizeof(double) : sizeof(float), pl.sweep[k]);
    // MFMA tiers: 64-sample tiles, each wave 16 samples of dimension 1
    // (LDS: the widest channel block, or four fields of one channel)
    const int mnch = std::max(std::min(pl.nout, 4) + (pl.nurbs ? 1 : 0), 1);
    auto mma_worst = [&]() {
      return std::max(mma_lds(pl, mnch, 1), mma_lds(pl, 1, SG_MAX_FIELDS));
    };
    int mrows = 32;
    compute_tiling(pl, pl.mma, mrows, 1);
    while (mma_worst() > static_cast<size_t>(kMaxLds) && mrows > 4) {
      mrows /= 2;
      compute_tiling(pl, pl.mma, mrows, 1);
    }
    if (mma_worst() > static_cast<size_t>(kMaxLds)) pl.mma = Tiling();
    pl.mma.xcd_map = xcd;
  }
  // adjoint tilings for NURBS plans too: the rational adjoint runs the
  // B-spline adjoint on the same dimensions
  if (ok && want_adjoint) {
    int rows = env_int("SG_ADJ_ROWS", 16);
    const int j3 = env_int("SG_ADJ_J3", 0);
    compute_tiling(pl, pl.adj, rows);
    compute_ztiling(pl, pl.adj, j3);
    while (adjoint_lds_min(pl) > static_cast<size_t>(kMaxLds) && rows > 1) {
      rows /= 2;
      compute_tiling(pl, pl.adj, rows);
      compute_ztiling(pl, pl.adj, j3);
    }
    if (adjoint_lds_min(pl) > static_cast<size_t>(kMaxLds)) pl.adj = Tiling();
    const char* xm = std::getenv("SG_XCD_MAP");
    pl.adj.xcd_map = (xm && *xm) ? std::atoi(xm) : default_xcd_map(pl);
  }
  pl.stream_ok = ok;
  const char* adj_mma_env = std::getenv("SG_ADJ_MMA");  // "0": streaming kernel only
  if (ok && want_adjoint && !(adj_mma_env && std::strcmp(adj_mma_env, "0") == 0) &&
      adjm_shape_ok) {
    plan_adjoint_mma(pl, pl.adjm, sizeof(float), resident_waves);
    plan_adjoint_mma(pl, pl.adjm64, sizeof(double),
                     resident_waves64 ? resident_waves64 : resident_waves);
    pl.adjm.xcd_map = pl.adjm64.xcd_map = pl.adj.xcd_map;
  }
}

// Gather lists of a tiling whose partial windows are w1 x w2 x w3max per
// channel, laid out [block3][block2][block1][k3 - lo3][channel][k2 - lo2]
// [k1 - lo1]: the element offset of control point k in a window is the sum
// of one entry per dimension and channel * gchan.
GatherLists gather_lists(const Plan& pl, const Tiling& tl, int w1, int w2) {
  GatherLists g;
  const long long plane = static_cast<long long>(w1) * w2;
  const long long win = static_cast<long long>(tl.w3max) * pl.nout * plane;  // one block
  // (block, offset in window) of dimension d -> its part of the element offset
  const long long stride1 = win, stride2 = win * tl.n_tiles1,
                  stride3 = win * tl.n_tiles1 * tl.n_chunks2;
  auto lists = [&](int nblocks, int block_len, const DimDev& D, long long bstride,
                   long long ostride, std::vector<int32_t>& ptr, std::vector<long long>& off) {
    std::vector<std::vector<long long>> per(D.n);
    for (int b = 0; b < nblocks; ++b) {
      const int a = b * block_len, e = std::min(a + block_len, D.m) - 1;
      const int lo = D.h_span[a] - D.p;
      for (int k = lo; k <= D.h_span[e]; ++k) per[k].push_back(b * bstride + (k - lo) * ostride);
    }
    ptr.assign(D.n + 1, 0);
    off.clear();
    for (int k = 0; k < D.n; ++k) {
      off.insert(off.end(), per[k].begin(), per[k].end());
      ptr[k + 1] = static_cast<int32_t>(off.size());
    }
  };
  lists(tl.n_tiles1, tl.tile_width(), pl.dims[0], stride1, 1, g.ptr[0], g.off[0]);
  lists(tl.n_chunks2, tl.chunk_rows(), pl.dims[1], stride2, w1, g.ptr[1], g.off[1]);
  if (pl.nin == 3) {
    lists(tl.n_z, tl.j3_per_block, pl.dims[2], stride3, pl.nout * plane, g.ptr[2], g.off[2]);
  } else {
    g.ptr[2] = {0, 1};
    g.off[2] = {0};
  }
  g.gchan = plane;
  return g;
}

std::vector<long long> gather_table(const GatherLists& g, int d, int& most) {
  const size_t n = g.ptr[d].size() - 1;
  std::vector<long long> table(n * kGatherRow, 0);
  most = 0;
  for (size_t k = 0; k < n; ++k) {
    const auto first = g.off[d].begin() + g.ptr[d][k], last = g.off[d].begin() + g.ptr[d][k + 1];
    const int count = static_cast<int>(last - first);
    most = std::max(most, count);
    table[k * kGatherRow] = count;
    if (count <= kGatherRow - 2) {
      std::copy(first, last, table.begin() + k * kGatherRow + 2);
    } else {
      table[k * kGatherRow + 1] = static_cast<long long>(table.size());
      table.insert(table.end(), first, last);
    }
  }
  return table;
}

void band_lists(const DimDev& D, std::vector<int32_t>& ptr, std::vector<int32_t>& js) {
  ptr.assign(D.n + 1, 0);
  js.assign(static_cast<size_t>(D.m) * (D.p + 1), 0);
  for (int j = 0; j < D.m; ++j)
    for (int a = 0; a <= D.p; ++a) ptr[D.h_span[j] - D.p + a + 1]++;
  for (int k = 0; k < D.n; ++k) ptr[k + 1] += ptr[k];
  std::vector<int32_t> fill(ptr.begin(), ptr.end() - 1);
  for (int j = 0; j < D.m; ++j)
    for (int a = 0; a <= D.p; ++a) js[fill[D.h_span[j] - D.p + a]++] = j * (D.p + 1) + a;
}

// One thread each walks short lists, and longer ones the more outputs there
// are: they fill the chip by themselves, neighbouring threads read neighbouring
// entries of ebar, and a wave's set-up and its reduction (0.6 to 0.9 ns per
// output) are not paid.  A wave each overtook a thread at, in entries, on 2-D /
// 3-D (degree 6) / 4-D (degree 2) grids: 45 / below 30 / below 30 at 50 000
// outputs, 140 / 75 / 55 at 130 000, 240 / 200 / 120 at 270 000, 250 / 500 / 240
// to 500 above a million (1.4 M outputs of 52 entries, 4-D: a thread 287 us, a
// wave 1 386; 265 000 of 252, 3-D: 439 and 365).  Curves take a wave from 48
// entries at any size: 600 000 outputs of 52, 1 278 and 181 us (a thread's
// samples lie far from its neighbour's).  A workgroup pays where the lists are
// long and the outputs few (1 458 outputs of 6 000: a wave 93, a workgroup 45
// us; 11 858: 224 and 380).  And never more threads than a launch takes.
int csr_threads(long long outputs, double entries, int nin) {
  const double most = nin == 1 ? 48.0 : nin == 2 ? 256.0 : 512.0;
  const double lone = std::max(std::min(outputs / (400.0 * nin), most), 48.0);
  if (entries <= lone || outputs > (kMaxLaunch - kCsrBlock) / kLanes) return 1;
  return (entries > 64.0 * kLanes && outputs <= 8192) ||
                 (entries > 16.0 * kLanes && outputs <= 2048)
             ? kCsrBlock
             : kLanes;
}

// A launch meant to keep `bpc` workgroups per CU gives each at most a bpc-th of
// its LDS, or fewer workgroups than asked are resident.

size_t lds_cap(int blocks_per_cu) {
  const size_t share = kLdsPerCu / static_cast<size_t>(std::max(1, blocks_per_cu));
  return std::min(static_cast<size_t>(kMaxLds), (share & ~size_t(511)) - 512);
}

int batch_vec(const Plan& pl) {
  const int m1 = pl.dims[0].m;
  return m1 > kLanes && pl.dims[0].p <= kVec2MaxDegree &&
                 pl.dims[1].p <= kVec2MaxDegree
             ? 2
             : 1;
}

GridTiling grid_tiling(const Plan& pl, int rows, int vec) {
  const DimDev& d1 = pl.dims[0];
  const DimDev& d2 = pl.dims[1];
  const int tw = kLanes * vec;
  GridTiling t{rows, (d1.m + tw - 1) / tw, 0, 0, 0, 0, tw};
  const int chunk = rows * kWaves;
  t.nty = (d2.m + chunk - 1) / chunk;
  for (int i = 0; i < t.ntx; ++i) {
    const int a = i * tw, e = std::min(a + tw, d1.m) - 1;
    t.w1 = std::max(t.w1, d1.h_span[e] - d1.h_span[a] + d1.p + 1);
  }
  for (int c = 0; c < t.nty; ++c) {
    const int a = c * chunk, e = std::min(a + chunk, d2.m) - 1;
    t.w2 = std::max(t.w2, d2.h_span[e] - d2.h_span[a] + d2.p + 1);
  }
  const size_t nch = std::min(pl.nout, kBC) + (pl.nurbs ? 1 : 0);
  const size_t planes = pl.nin == 3 ? kWaves : 1;
  t.lds = planes * nch * t.w1 * t.w2 * sizeof(float);  // the window slabs
  return t;
}

GridTiling batch_grid_tiling(const Plan& pl, int rows_per_wave, size_t cap) {
  auto fit = [&](int vec) {
    int rows = rows_per_wave;
    GridTiling t = grid_tiling(pl, rows, vec);
    while (t.lds > cap && rows > 1) t = grid_tiling(pl, rows /= 2, vec);
    return t;
  };
  const GridTiling t1 = fit(1);
  if (batch_vec(pl) != 2) return t1;
  const GridTiling t2 = fit(2);
  return t2.lds <= cap ? t2 : t1;
}

int batch_default_rows(const std::vector<const Plan*>& plans, int cus) {
  long long tiles = 0;  // at 16 rows
  for (const Plan* pl : plans) {
    const GridTiling t = batch_grid_tiling(*pl, 16, lds_cap(kBatchPerCu));
    const int nz = pl->nin == 3 ? (pl->dims[2].m + kWaves - 1) / kWaves : 1;
    tiles += static_cast<long long>(t.ntx) * t.nty * nz;
  }
  const long long slots = static_cast<long long>(kBatchPerCu) * cus;
  return tiles < slots ? 8 : tiles < 6 * slots ? 16 : 32;
}

int plane_list_host(const int32_t* span3, const float* tab3, int p3, int j3_0, int planes,
                    float* list) {
  const int cap = plane_list_floats(p3);
  std::fill(list, list + cap, 0.f);
  std::vector<int> ks;
  for (int pz = 0; pz < planes; ++pz)
    for (int d = 0; d <= p3; ++d) ks.push_back(span3[j3_0 + pz] - p3 + d);
  std::sort(ks.begin(), ks.end());
  ks.erase(std::unique(ks.begin(), ks.end()), ks.end());
  const int nk = static_cast<int>(ks.size());
  auto put_k = [&](int i, int k3) { std::memcpy(list + i * kEntry + kEntryK, &k3, sizeof(int)); };
  for (int i = 0; i < nk; ++i) {
    put_k(i, ks[i]);
    for (int pz = 0; pz < planes; ++pz) {
      const int d = ks[i] - (span3[j3_0 + pz] - p3);
      if (d >= 0 && d <= p3) list[i * kEntry + pz] = tab3[static_cast<size_t>(j3_0 + pz) * (p3 + 1) + d];
    }
  }
  put_k(nk, ks.back());  // padding: zero weights, a plane of the grid
  std::memcpy(list + kEntryN, &nk, sizeof(int));
  return nk;
}

void pack_queues(const std::vector<std::vector<BTile>>& grid_tiles,
                 const std::vector<long long>& grid_cost, std::vector<BTile>& sorted,
                 int* host_q) {
  std::vector<size_t> order(grid_tiles.size());
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(),
                   [&](size_t a, size_t c) { return grid_cost[a] > grid_cost[c]; });
  struct Piece {  // tiles [first, last) of a grid
    size_t grid, first, last;
  };
  const auto tile_cost = [&](size_t g) {
    return static_cast<double>(grid_cost[g]) / std::max<size_t>(1, grid_tiles[g].size());
  };
  // What a queue should hold.  A grid that would take the least loaded queue
  // 1/20 past it is cut into ranges of neighbouring tiles over several.
  double mean = 0.0;
  for (size_t g : order) mean += static_cast<double>(grid_cost[g]) / kXcds;
  std::vector<std::vector<Piece>> queue(kXcds);
  double load[kXcds] = {};
  for (size_t g : order) {
    const size_t n = grid_tiles[g].size();
    const double each = tile_cost(g);
    for (size_t first = 0; first < n;) {
      const int q = static_cast<int>(std::min_element(load, load + kXcds) - load);
      const double room = mean - load[q];
      size_t last = n;
      if (each * static_cast<double>(n - first) > room + 0.05 * mean)
        last = first + std::min(std::max<size_t>(static_cast<size_t>(std::max(room, 0.0) / each), 1),
                                n - first);
      queue[q].push_back(Piece{g, first, last});
      load[q] += each * static_cast<double>(last - first);
      first = last;
    }
  }
  // a queue hands out its costly tiles first, so that the last to start are
  // short
  for (std::vector<Piece>& q : queue)
    std::stable_sort(q.begin(), q.end(), [&](const Piece& a, const Piece& c) {
      return tile_cost(a.grid) > tile_cost(c.grid);
    });
  sorted.clear();
  std::fill(host_q, host_q + kQueueInts, 0);
  int* start = host_q + kXcds * kQueueStride;
  for (int q = 0; q < kXcds; ++q) {
    start[q] = static_cast<int>(sorted.size());
    for (const Piece& piece : queue[q])
      sorted.insert(sorted.end(), grid_tiles[piece.grid].begin() + piece.first,
                    grid_tiles[piece.grid].begin() + piece.last);
  }
  start[kXcds] = static_cast<int>(sorted.size());
}

}  // namespace sg
