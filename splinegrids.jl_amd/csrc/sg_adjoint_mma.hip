// sg_adjoint_mma.hip -- evaluate_adjoint!(grid) on matrix cores, FP32 and
// FP64: Pbar = M^T ebar without atomics (src/adjoint.jl:1-40, :52-83), and
// the adjoint of a NURBS grid's evaluate! in its control points.
//
// The two innermost contractions of the adjoint are small matrix products.
// For a tile of 16 NQ samples j1 whose bands cover at most 16 control points
// k1 (from lo1), 16 rows j2 and one sample j3:
//
//   T1[j2][k1] = sum_j1 ebar[j1, j2, j3] * B1[j1, k1]     (16 x 16 NQ) (16 NQ x 16)
//   T2[k2][k1] = sum_j2 B2[j2, k2] * T1[j2][k1]           (16 x 16) (16 x 16)
//
// Both run on v_mfma_f32_16x16x4f32 or v_mfma_f64_16x16x4f64 (products and
// sums of the array's own type).  With lane l = 16 g + i, these take A[i][g]
// and B[g][i] from lane l and leave D[drow(g, r)][i] in register r, where
// drow is 4 g + r (FP32) or g + 4 r (FP64).  So:
//   GEMM1, K-step s (4 NQ steps): A = ebar[j1_0 + samp(g, s), row i]
//                                 B = B1[j1_0 + samp(g, s)][lo1 + i]
//     (samp: lane l reads 16-byte pieces of its row, and the four lanes of a
//     row read 64 contiguous bytes per load instruction)
//   GEMM2, K-step r (4 steps, row j2 = drow(g, r) of the 16):
//                                 A = B2[drow(g, r)][lo2 + i]
//                                 B = T1[drow(g, r)][i] = register r of GEMM1
//   D2: T2[lo2 + drow(g, r)][lo1 + i].
//
// 3-D: a wave holds 16 rows and walks a run of samples j3; T2 of each j3 is
// weighted by B3[j3, d] into a register ring of p3 + 1 slabs of k3.  2-D: a
// wave walks 16-row blocks and T2 accumulates.  The NW waves of a workgroup
// (4, 2 or 1) hold neighbouring rows whose bands share one window of 16
// control points k2, so a slab that is final (its k3 leaves the band of the
// next j3) is summed over the waves through LDS, in wave order, and one
// partial window per workgroup goes to HBM; adj_gather (sg_adjoint.hip) then
// sums the few partial windows that hold each control point.
//
// Bound: HBM reads of ebar (a kernel that only reads ebar in this tile pattern
// takes 76 us of the 82 here on 400 x 400 x 200 samples x 3, 147 of 154 on
// 512 x 512 x 256 x 3).  With the gather: FP32 400 x 400 x 200 x 3 87 us (91
// with the channels and 64 rows in one wave); FP32 251 x 197 x 123 x 3 24 us
// (50: rows of odd length took 4-byte loads); FP64 200 x 201 x 99 x 3 32 us
// (154 with a sliding window of FMAs and LDS); NURBS 512 x 512 x 256 x 3 179 us
// (327 with 1 / w(x) written by a pass of its own and read back).  What the
// layout is for:
//  - a wave holds one unit (16 rows x 16 NQ samples, 4 KB in FP32, 8 in FP64 at
//    NQ = 4) and has the next in flight, three to five waves per SIMD;
//  - the channels are workgroups of their own (plain adjoint), so small grids
//    fill the chip with fewer, longer runs of j3 and fewer partial windows;
//  - ebar is read with raw buffer loads: one descriptor per (j3, channel)
//    plane and per-lane byte offsets.  Any element-aligned row takes the
//    16-byte loads (gfx950 loads need dword alignment only), the hardware
//    returns 0 for every dword past the plane, and offsets past it mask rows
//    past the chunk and samples past m1 without a branch (branches around
//    loads make the compiler wait for every load in flight at the merge).
#include <algorithm>

#include "sg_mma_ops.hpp"
#include "sg_plan_host.hpp"

namespace sg {

namespace {

constexpr int kWin = kAdjMmaWin;  // control points per MFMA tile edge
constexpr int kSlab = kWin * kWin;

template <typename T>
struct Mfma;
template <>
struct Mfma<float> {
  typedef float D __attribute__((ext_vector_type(4)));
  typedef float Ld __attribute__((ext_vector_type(4)));  // one 16-byte load
  static constexpr int VW = 4;                           // elements per load
  __device__ static constexpr int drow(int g, int r) { return 4 * g + r; }
  // sample (of 16) of element r of lane group g, and of A row / B column i
  __device__ static constexpr int samp(int g, int r) { return 4 * g + r; }
  __device__ static constexpr int column(int i) { return i; }
  __device__ static D mma(float a, float b, D c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mfma<double> {
  typedef double D __attribute__((ext_vector_type(4)));
  typedef double Ld __attribute__((ext_vector_type(2)));
  static constexpr int VW = 2;
  __device__ static constexpr int drow(int g, int r) { return g + 4 * r; }
  __device__ static constexpr int samp(int g, int r) { return 8 * (r >> 1) + 2 * g + (r & 1); }
  // D row rho = drow(g, r) holds sample samp(g, r)
  __device__ static constexpr int column(int i) { return samp(i & 3, i >> 2); }
  __device__ static D mma(double a, double b, D c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};

template <typename T>
struct AdjMmaArgs {
  const T* E;
  const T* W;  // NURBS: weights [n3][n2][n1]
  T* part;
  const T* tab1;  // [m1][p1+1]
  const T* tab2;  // [m2][p2+1]
  const T* tab3;  // [m3][P3+1] (3-D)
  const int32_t* span1;
  const int32_t* span2;
  const int32_t* span3;
  int m1, m2, m3, p1, p2, n1, n2, n3;
  int nout, group0;  // group0: the launch's first group of NC channels
  int rows, chunk, j3_per_block;
  int ntx, nty, nz, w1max, w2max, w3max, xcd_map;
  long long m12, nsamp;
};

// Byte offsets at or past a plane's size read 0 (planes are < 2 GiB).
constexpr unsigned kOff = 0x80000000u;
constexpr int kRsrcWord3 = 0x00020000;  // raw buffer, 32-bit elements (gfx9)

// Units per unrolled group, one register buffer each: KB - 1 are in flight.
// One unit ahead and three to five waves per SIMD read faster than five ahead
// and three waves (400 x 400 x 200 samples x 3: 92 us with six buffers, 90
// with four, 88 with two; 512 x 512 x 256 x 3: 173, 173, 164 us).
template <int NC>
constexpr int unit_buffers() {
  return NC == 1 ? 2 : NC;
}

__device__ inline bool finite(float x) { return __builtin_isfinite(x); }
__device__ inline bool finite(double x) { return __builtin_isfinite(x); }

// The kernel's arguments, read again: what the cold path below takes from here
// the hot one need not hold (held, they spilled 50 scalars and cost 1.2 us of 33
// on 200 x 201 x 99 x 3 FP64).
template <typename T>
using Global = __attribute__((address_space(1))) T;
template <typename T>
using AdjArgsAgain = Constant<const AdjMmaArgs<T>>;
template <typename T>
__device__ inline AdjArgsAgain<T>* kernel_args() {
  auto at = reinterpret_cast<uintptr_t>(__builtin_amdgcn_kernarg_segment_ptr());
  asm volatile("" : "+s"(at));
  return reinterpret_cast<AdjArgsAgain<T>*>(at);
}

// The workgroup's tile, chunk, run and first channel.
struct AdjBlock {
  int bx, by, bz, c0;
};
template <typename Args>
__device__ inline AdjBlock adj_block(const Args& a, int nc) {
  int rest = xcd_logical_block(a.xcd_map, a.ntx);
  AdjBlock b;
  b.bx = rest % a.ntx;
  rest /= a.ntx;
  b.by = rest % a.nty;
  rest /= a.nty;
  b.bz = rest % a.nz;
  b.c0 = (a.group0 + rest / a.nz) * nc;
  return b;
}

// A workgroup's run of one channel (c), every value over its own bands alone:
// what adj_mma takes back to where Inf or NaN entered its products, whose zeros
// off the bands make NaN of the whole window.  Same partial windows, plain sums
// through LDS (banded_lds elements).  Slow, and seldom: 200 x 201 x 99 x 3 FP64
// with one Inf 185 us, all NaN 222 (clean 33); 400 x 400 x 200 x 3 743 and 1367
// (88); NURBS 512 x 512 x 256 x 3 3.8 and 5.3 ms (0.18).  What it costs a clean
// call: 0.2 to 0.4 us.  (A check of each unit in the loop: 0.6 us.)
template <typename T, int NIN, int P3, int NQ, bool NURBS>
__device__ __attribute__((always_inline)) void banded_run(AdjArgsAgain<T>& a, T* lds, int bx, int by, int bz, int c) {
  constexpr int TW = 16 * NQ;
  // (the compiler knows no address space of a pointer that it reads from memory)
  const auto span1 = (Global<const int32_t>*)a.span1;
  const auto span2 = (Global<const int32_t>*)a.span2;
  const auto span3 = (Global<const int32_t>*)a.span3;
  const auto tab1 = (Global<const T>*)a.tab1;
  const auto tab2 = (Global<const T>*)a.tab2;
  const auto tab3 = (Global<const T>*)a.tab3;
  const auto part = (Global<T>*)a.part;
  const int tid = static_cast<int>(threadIdx.x), threads = static_cast<int>(blockDim.x);
  const int rows = threads / 4;           // rows j2 at a time
  T* T1 = lds;                            // [rows][kWin]
  T* G = T1 + 4 * threads;                // NURBS: [kWin][kWin] weights at j3
  T* winv = G + kSlab;                    // NURBS: [rows][TW] 1 / w
  const int p1 = a.p1, p2 = a.p2;
  const int j1_0 = bx * TW, x1 = min(j1_0 + TW, a.m1);
  const int r0 = by * a.chunk, r1 = min(r0 + a.chunk, a.m2);
  const int lo1 = span1[j1_0] - p1, lo2 = span2[r0] - p2;
  const int W1 = span1[x1 - 1] - lo1 + 1, W2 = span2[r1 - 1] - lo2 + 1;
  const int j3a = NIN == 3 ? bz * a.j3_per_block : 0;
  const int j3e = NIN == 3 ? min(j3a + a.j3_per_block, a.m3) : 1;
  const int lo3 = NIN == 3 ? span3[j3a] - P3 : 0;
  const size_t block = (static_cast<size_t>(bz) * a.nty + by) * a.ntx + bx;
  // the samples whose bands hold a control point are one range
  const auto range = [](Global<const int32_t>* span, int p, int from, int to, int k, int& first, int& last) {
    first = last = from;
    for (int j = from; j < to; ++j) {
      first += span[j] < k ? 1 : 0;
      last += span[j] - p <= k ? 1 : 0;
    }
  };
  const int q1 = tid % kWin;
  int ja, jb;
  range(span1, p1, j1_0, x1, lo1 + q1, ja, jb);
  for (int t0 = 0; t0 < kSlab; t0 += threads) {  // the thread's window entry
    const int q2 = (t0 + tid) / kWin;
    int ra, rb;
    range(span2, p2, r0, r1, lo2 + q2, ra, rb);
    const auto store = [&](T v, int k3) {
      if (q2 < W2 && q1 < W1)
        part[((block * a.w3max + (k3 - lo3)) * a.nout + c) *
                   (static_cast<size_t>(a.w1max) * a.w2max) + q2 * a.w1max + q1] = v;
    };
    T R[P3 + 1];
#pragma unroll
    for (int d = 0; d <= P3; ++d) R[d] = T(0);
    int cur3 = lo3 + P3;
    for (int j3 = j3a; j3 < j3e; ++j3) {
      const int s3 = NIN == 3 ? span3[j3] : 0;
      T b3[P3 + 1];
#pragma unroll
      for (int d = 0; d <= P3; ++d)
        b3[d] = NIN == 3 ? tab3[static_cast<size_t>(j3) * (P3 + 1) + d] : T(1);
      for (; NIN == 3 && cur3 < s3; ++cur3) {
        store(R[0], cur3 - P3);
#pragma unroll
        for (int d = 0; d < P3; ++d) R[d] = R[d + 1];
        R[P3] = T(0);
      }
      if constexpr (NURBS) {
        for (int x = tid; x < kSlab; x += threads) {
          const auto W = (Global<const T>*)a.W + (static_cast<long long>(NIN == 3 ? s3 - P3 : 0) * a.n2 +
                              lo2 + x / kWin) * a.n1 + lo1 + x % kWin;
          T v = T(0);
          if (x / kWin < W2 && x % kWin < W1)
#pragma unroll
            for (int d = 0; d <= P3; ++d) v += b3[d] * W[static_cast<long long>(d) * a.n2 * a.n1];
          G[x] = v;
        }
        __syncthreads();
      }
      const auto E = (Global<const T>*)a.E + a.m12 * j3 + a.nsamp * c;
      T t2 = T(0);
      for (int row0 = r0; row0 < r1; row0 += rows) {
        const int n = min(rows, r1 - row0);
        if constexpr (NURBS) {
          for (int x = tid; x < n * TW; x += threads) {
            const int j1 = j1_0 + x % TW, j2 = row0 + x / TW;
            if (j1 >= x1) continue;
            const T* g = G + (span2[j2] - p2 - lo2) * kWin + span1[j1] - p1 - lo1;
            T w = T(0);
            for (int d = 0; d <= p2; ++d, g += kWin) {
              T u = T(0);
              for (int q = 0; q <= p1; ++q) u += tab1[static_cast<size_t>(j1) * (p1 + 1) + q] * g[q];
              w += tab2[static_cast<size_t>(j2) * (p2 + 1) + d] * u;
            }
            winv[x] = T(1) / w;
          }
          __syncthreads();
        }
        for (int x = tid; x < n * kWin; x += threads) {
          const int r = x / kWin;
          const auto row = E + static_cast<long long>(row0 + r) * a.m1;
          T s = T(0);
#pragma unroll 4
          for (int j1 = ja; j1 < jb; ++j1)
            s += tab1[static_cast<size_t>(j1) * (p1 + 1) + lo1 + q1 + p1 - span1[j1]] *
                 (NURBS ? row[j1] * winv[r * TW + j1 - j1_0] : row[j1]);
          T1[x] = s;
        }
        __syncthreads();
        for (int j2 = max(ra, row0); j2 < min(rb, row0 + n); ++j2)
          t2 += tab2[static_cast<size_t>(j2) * (p2 + 1) + lo2 + q2 + p2 - span2[j2]] *
                T1[(j2 - row0) * kWin + q1];
        __syncthreads();
      }
#pragma unroll
      for (int d = 0; d <= P3; ++d) R[d] += b3[d] * t2;
    }
#pragma unroll
    for (int d = 0; d <= P3; ++d) store(R[d], cur3 - P3 + d);
  }
}
constexpr size_t banded_lds(int nw, int nq, bool nurbs) {
  return static_cast<size_t>(nw) * kSlab * (nurbs ? 1 + nq : 1) + (nurbs ? kSlab : 0);
}

// NURBS: ebar is multiplied by 1 / w(x) as its units arrive.  The weight
// field of a unit is two more small products with the same operand trick,
//   V[k2][j1] = sum_k1 Gw[k2][k1] B1[j1][k1],  w^T[j1][j2] = sum_k2 V[k2][j1] B2[j2][k2],
// Gw a plane of the window of weights; w^T lands in the lanes and registers
// that hold ebar's samples.  3-D: a register ring keeps w^T of the p3 + 1
// planes k3 of the band, so the products run once per plane and a sample j3
// takes p3 + 1 FMAs per value (the products once per j3 took 32 MFMA of 92).
// The NC channels of a workgroup share it (units go sample j3 by sample,
// the channels of a sample together, each channel with a ring of its own).
template <typename T, int NIN, int P3, int NQ, int NC, int TIER, bool NURBS>
__global__ __launch_bounds__(kThreads, NURBS && sizeof(T) == 8 ? 1 : 2) void adj_mma(
    AdjMmaArgs<T> a) {
  using M = Mfma<T>;
  using D = typename M::D;
  using Ld = typename M::Ld;
  constexpr int VW = M::VW;
  constexpr int NL = 16 * NQ / 4 / VW;  // 16-byte loads per unit and lane
  constexpr int KB = unit_buffers<NC>();
  constexpr int NS = 4 * NQ;  // K-steps of GEMM1, samples per lane
  static_assert(KB % NC == 0, "the channel of a buffer position must be constant");
  extern __shared__ __align__(16) unsigned char smem[];
  T* red = reinterpret_cast<T*>(smem);  // [2][NW][kSlab]

  const int lane = threadIdx.x & (kLanes - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes);
  const int nw = static_cast<int>(blockDim.x) / kLanes;
  const int g = lane >> 4, i = lane & 15;
  const AdjBlock at = adj_block(a, NC);
  const int bx = at.bx, by = at.by, bz = at.bz, c0 = at.c0;
  const int nc = NC == 1 ? 1 : min(NC, a.nout - c0);
  const int j1_0 = bx * 16 * NQ;
  const int r0 = by * a.chunk, r1 = min(r0 + a.chunk, a.m2);
  const int rb = min(r0 + wave * a.rows, r1), re = min(rb + a.rows, r1);
  const int p1 = a.p1, p2 = a.p2;
  const int lo1 = a.span1[j1_0] - p1;
  const int lo2 = a.span2[r0] - p2;
  const int W1 = a.span1[min(j1_0 + 16 * NQ, a.m1) - 1] - lo1 + 1;  // <= 16
  const int W2 = a.span2[r1 - 1] - lo2 + 1;                          // <= 16
  const int left = a.m1 - j1_0;             // samples j1 from the tile's first
  const bool tail = left < 16 * NQ && (left & (VW - 1)) != 0;  // a load crosses the row's end

  // Operand tables.  Every load below is unconditional, at a clamped index,
  // and masked afterwards (table values are finite), so that each group of
  // loads is issued at once and costs one memory latency.
  auto b1_at = [&](int j1, int sp, int k1) {
    const int off = lo1 + k1 - (sp - p1);
    const T v = a.tab1[static_cast<size_t>(min(j1, a.m1 - 1)) * (p1 + 1) + min(max(off, 0), p1)];
    return v * ((j1 < a.m1 && off >= 0 && off <= p1) ? T(1) : T(0));
  };
  auto b2_at = [&](int j2, int sp, int k2) {
    const int off = lo2 + k2 - (sp - p2);
    const T v = a.tab2[static_cast<size_t>(min(j2, r1 - 1)) * (p2 + 1) + min(max(off, 0), p2)];
    return v * ((j2 < re && off >= 0 && off <= p2) ? T(1) : T(0));
  };
  // GEMM1 B operand: B1 at (j1_0 + sample, lo1 + i), 0 off the band
  T b1[NS];
  {
    int sp[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s)
      sp[s] = a.span1[min(j1_0 + 16 * (s >> 2) + M::samp(g, s & 3), a.m1 - 1)];
#pragma unroll
    for (int s = 0; s < NS; ++s) b1[s] = b1_at(j1_0 + 16 * (s >> 2) + M::samp(g, s & 3), sp[s], i);
  }
  // MFMA tiers: GEMM1 on 16x16x32 FP16 / BF16 products.  K block h of a
  // unit holds samples j1_0 + 32 h + 0..31; element e of a lane is its
  // K-step 8 h + e of the FP32 path in both operands.  B1 is scaled by 2^-eb
  // (split FP16: max|B1| of the wave's tile below 1) and converted once.
  constexpr bool MT = TIER != SG_TIER_NATIVE;
  Operand8<MT ? TIER : SG_TIER_BF16> b1op[MT ? NQ / 2 : 1];
  int eb = 0;
  if constexpr (MT) {
    float sb = 1.f;
    if constexpr (TIER == SG_TIER_SPLIT_F16) {
      float m = 0.f;
#pragma unroll
      for (int s = 0; s < NS; ++s) m = fmaxf(m, fabsf(static_cast<float>(b1[s])));
      eb = scale_exponent(wave_max(m));
      sb = ldexpf(1.f, -eb);
    }
#pragma unroll
    for (int h = 0; h < NQ / 2; ++h)
#pragma unroll
      for (int e = 0; e < 8; ++e) b1op[h].set(e, static_cast<float>(b1[8 * h + e]) * sb);
  }
  // GEMM2 A operand of the 16 rows from row0, K-step r: B2 at
  // (row0 + drow(g, r), lo2 + i); NURBS also B2 at (row0 + i, lo2 + drow(g, r))
  T b2[4], b2t[NURBS ? 4 : 1];
  auto load_b2 = [&](int row0) {
    int sp[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) sp[r] = a.span2[min(row0 + M::drow(g, r), r1 - 1)];
    const int spi = NURBS ? a.span2[min(row0 + i, r1 - 1)] : 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) b2[r] = b2_at(row0 + M::drow(g, r), sp[r], i);
    if constexpr (NURBS) {
#pragma unroll
      for (int r = 0; r < 4; ++r) b2t[r] = b2_at(row0 + i, spi, M::drow(g, r));
    }
  };
  load_b2(rb);

  const int j3a = NIN == 3 ? bz * a.j3_per_block : 0;
  const int J = NIN == 3 ? min(a.j3_per_block, a.m3 - j3a) : 1;
  // steps of NC units: samples j3 (3-D) or blocks of 16 rows (2-D)
  const int steps = NIN == 3 ? J : (re - rb + 15) / 16;
  const bool any = rb < re;

  // Load cursor: the plane (3-D) and row offset (2-D) of the next unit, kept
  // as running state; units past the last read nothing (no records).
  const unsigned plane_bytes = static_cast<unsigned>(a.m12 * static_cast<long long>(sizeof(T)));
  int lc = 0, lstep = 0;
  const T* lplane = a.E + static_cast<long long>(j3a) * a.m12 + a.nsamp * c0;
  auto load = [&](Ld (&e)[NL]) {
    const int row = (NIN == 2 ? rb + 16 * lstep : rb) + i;
    const unsigned base = static_cast<unsigned>(
        (static_cast<long long>(row) * a.m1 + j1_0) * static_cast<long long>(sizeof(T)));
    const bool live = any && lstep < steps && (NC == 1 || lc < nc);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<T*>(lplane), 0, static_cast<int>(live ? plane_bytes : 0u), kRsrcWord3);
#pragma unroll
    for (int q = 0; q < NL; ++q) {
      const int s = 4 * VW * q + VW * g;  // the load's first sample
      const unsigned o = row < re && s < left
                             ? base + static_cast<unsigned>(s * static_cast<int>(sizeof(T)))
                             : kOff;
      // the b128 loads return raw 32-bit words: reinterpret, not convert
      e[q] = __builtin_bit_cast(Ld, __builtin_amdgcn_raw_buffer_load_b128(rs, static_cast<int>(o), 0, 0));
    }
    if (NC == 1) {
      ++lstep;
      if (NIN == 3) lplane += a.m12;
    } else {
      lplane += a.nsamp;
      if (++lc == NC) {
        lc = 0;
        ++lstep;
        lplane += (NIN == 3 ? a.m12 : 0) - NC * a.nsamp;
      }
    }
  };

  // At position k of a group the unit KB - 1 ahead is loaded into the buffer
  // that position k - 1 has just used, so KB - 1 units are in flight and no
  // buffer is ever copied (a copy of a register whose load is in flight
  // waits for that load).
  Ld buf[KB][NL];
#pragma unroll
  for (int k = 0; k < KB - 1; ++k) load(buf[k]);

  // NURBS: rw[d] holds w^T of plane k3 = cur3 - P3 + d at the lane's samples
  // (2-D: the one plane of the current row block), wn the window of weights of
  // the next plane, lane (g, i) at (k2 = lo2 + i, k1 = lo1 + 4 g + s), and b1t
  // B1 at (sample column(i) of block q, lo1 + 4 g + s)
  T rw[NURBS ? P3 + 1 : 1][NURBS ? NS : 1], b1t[NURBS ? NQ : 1][4], wn[4], inv[NURBS ? NS : 1];
  const int lo3 = NIN == 3 ? a.span3[j3a] - P3 : 0;
  int cur3 = lo3 + P3;
  auto load_w = [&](int k3) {
    if constexpr (NURBS) {
      const T* src = a.W + (static_cast<long long>(min(k3, a.n3 - 1)) * a.n2 +
                            min(lo2 + i, a.n2 - 1)) * a.n1;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const T v = src[min(lo1 + 4 * g + s, a.n1 - 1)];
        wn[s] = i < W2 && 4 * g + s < W1 ? v : T(0);
      }
    }
  };
  // the plane in wn at the tile's samples of the rows in b2t
  auto plane_w = [&](T (&out)[NURBS ? NS : 1]) {
    if constexpr (NURBS) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        D v = {T(0), T(0), T(0), T(0)}, w = {T(0), T(0), T(0), T(0)};
#pragma unroll
        for (int s = 0; s < 4; ++s) v = M::mma(wn[s], b1t[q][s], v);
#pragma unroll
        for (int r = 0; r < 4; ++r) w = M::mma(v[r], b2t[r], w);
#pragma unroll
        for (int r = 0; r < 4; ++r) out[4 * q + r] = w[r];
      }
    }
  };
  // 1 / w; rows and samples outside the grid have w = 0, and their ebar reads 0
  auto recip_w = [&](const T (&w)[NURBS ? NS : 1], int row0) {
    const bool rowok = row0 + i < re;
#pragma unroll
    for (int s = 0; s < (NURBS ? NS : 1); ++s)
      inv[s] = rowok && 16 * (s >> 2) + M::samp(g, s & 3) < left ? T(1) / w[s] : T(0);
  };
  if constexpr (NURBS) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int j1 = j1_0 + 16 * q + M::column(i);
      const int sp = a.span1[min(j1, a.m1 - 1)];
#pragma unroll
      for (int s = 0; s < 4; ++s) b1t[q][s] = b1_at(j1, sp, 4 * g + s);
    }
    load_w(lo3);
    if constexpr (NIN == 3) {
#pragma unroll
      for (int d = 0; d <= P3; ++d) {
        plane_w(rw[d]);
        load_w(lo3 + d + 1);
      }
    }
  }

  // R[ch][d]: slab k3 = cur3 - P3 + d of channel c0 + ch (2-D: T2 itself)
  D R[NC][P3 + 1];
#pragma unroll
  for (int ch = 0; ch < NC; ++ch)
#pragma unroll
    for (int d = 0; d <= P3; ++d) R[ch][d] = D{T(0), T(0), T(0), T(0)};

  // Slab k3 of channel c0 + ch is final: summed over the waves in order, it
  // goes to part[block][k3 - lo3][channel] inside the W2 x W1 window (the
  // gather reads no other entry).  Two LDS slots in turn: a wave reaches the
  // next use of a slot only past the barrier that follows every wave's reads
  // of it.
  int par = 0;
  T seen = T(0);  // not finite once a slab was not (all its entries then are)
  const size_t block = (static_cast<size_t>(bz) * a.nty + by) * a.ntx + bx;
  auto flush = [&](const D& slab, int ch, int k3) {
    T* dst = a.part + ((block * a.w3max + (k3 - lo3)) * a.nout + c0 + ch) *
                          (static_cast<size_t>(a.w1max) * a.w2max);
    seen += slab[0];
    if (nw == 1) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (M::drow(g, r) < W2 && i < W1) dst[M::drow(g, r) * a.w1max + i] = slab[r];
      return;
    }
    T* slot = red + static_cast<size_t>(par) * nw * kSlab;
#pragma unroll
    for (int r = 0; r < 4; ++r) slot[wave * kSlab + r * kLanes + lane] = slab[r];
    __syncthreads();
    for (int t = threadIdx.x; t < kSlab; t += nw * kLanes) {
      T s = slot[t];
      for (int w = 1; w < nw; ++w) s += slot[w * kSlab + t];
      const int row = M::drow((t >> 4) & 3, t >> 6), col = t & 15;
      if (row < W2 && col < W1) dst[row * a.w1max + col] = s;
    }
    par ^= 1;
  };

  // B3 rows and spans through the constant address space: the index is
  // uniform, so they are scalar loads and wait for no ebar load
  Constant<const T>* tab3 = constant_ptr(a.tab3);
  Constant<const int32_t>* span3 = constant_ptr(a.span3);
  T b3[P3 + 1];
  for (int s0 = 0; s0 < steps; s0 += KB / NC) {
#pragma unroll
    for (int k = 0; k < KB; ++k) {
      const int ch = k % NC;          // the unit's channel
      const int step = s0 + k / NC;   // its sample j3 - j3a, or row block
      load(buf[(k + KB - 1) % KB]);
      if (step < steps) {
        if (ch == 0) {
          if constexpr (NIN == 3) {
            const int j3 = j3a + step;
#pragma unroll
            for (int d = 0; d <= P3; ++d) b3[d] = tab3[static_cast<size_t>(j3) * (P3 + 1) + d];
            const int s3 = span3[j3];
            while (cur3 < s3) {  // every ring moves to the sample's band
#pragma unroll
              for (int cc = 0; cc < NC; ++cc) {
                if (cc < nc) flush(R[cc][0], cc, cur3 - P3);
#pragma unroll
                for (int d = 0; d < P3; ++d) R[cc][d] = R[cc][d + 1];
                R[cc][P3] = D{T(0), T(0), T(0), T(0)};
              }
              ++cur3;
              if constexpr (NURBS) {
#pragma unroll
                for (int d = 0; d < P3; ++d)
#pragma unroll
                  for (int s = 0; s < NS; ++s) rw[d][s] = rw[d + 1][s];
                plane_w(rw[P3]);
                load_w(cur3 + 1);
              }
            }
            if constexpr (NURBS) {
              T w[NS];
#pragma unroll
              for (int s = 0; s < NS; ++s) {
                w[s] = T(0);
#pragma unroll
                for (int d = 0; d <= P3; ++d) w[s] += b3[d] * rw[d][s];
              }
              recip_w(w, rb);
            }
          } else {
            if (step > 0) load_b2(rb + 16 * step);
            if constexpr (NURBS) {
              plane_w(rw[0]);
              recip_w(rw[0], rb + 16 * step);
            }
          }
        }
        if (any && (NC == 1 || ch < nc)) {
          T e[NS];
#pragma unroll
          for (int s = 0; s < NS; ++s) e[s] = buf[k][s / VW][s % VW];
          if (tail) {  // elements past the row's end are the next row's
#pragma unroll
            for (int s = 0; s < NS; ++s)
              e[s] = 16 * (s >> 2) + M::samp(g, s & 3) < left ? e[s] : T(0);
          }
          if constexpr (NURBS) {
#pragma unroll
            for (int s = 0; s < NS; ++s) e[s] *= inv[s];
          }
          D d1 = {T(0), T(0), T(0), T(0)};
          if constexpr (!MT) {
#pragma unroll
            for (int s = 0; s < NS; ++s) d1 = M::mma(e[s], b1[s], d1);
          } else {
            // split FP16: the unit's ebar scaled by 2^-eu (max below 1), and
            // T1 scaled back by 2^(eu + eb); BF16 needs no scaling
            int eu = 0;
            float su = 1.f;
            if constexpr (TIER == SG_TIER_SPLIT_F16) {
              float m = 0.f;
#pragma unroll
              for (int s = 0; s < NS; ++s) m = fmaxf(m, fabsf(e[s]));
              eu = scale_exponent(wave_max(m));
              su = ldexpf(1.f, -eu);
            }
#pragma unroll
            for (int h = 0; h < NQ / 2; ++h) {
              Operand8<TIER> op;
#pragma unroll
              for (int x = 0; x < 8; ++x) op.set(x, e[8 * h + x] * su);
              d1 = Operand8<TIER>::mma(op, b1op[h], d1);
            }
            if constexpr (TIER == SG_TIER_SPLIT_F16) {
#pragma unroll
              for (int r = 0; r < 4; ++r) d1[r] = ldexpf(d1[r], eu + eb);
            }
          }
          if constexpr (NIN == 2) {
#pragma unroll
            for (int r = 0; r < 4; ++r) R[ch][0] = M::mma(b2[r], d1[r], R[ch][0]);
          } else {
            D t2 = {T(0), T(0), T(0), T(0)};
#pragma unroll
            for (int r = 0; r < 4; ++r) t2 = M::mma(b2[r], d1[r], t2);
#pragma unroll
            for (int d = 0; d <= P3; ++d)
#pragma unroll
              for (int r = 0; r < 4; ++r) R[ch][d][r] += b3[d] * t2[r];
          }
        }
      }
    }
  }
  // the run's last band is final; the waves tell each other what they have seen
  // before its last barrier
  T* flags = red + 2 * static_cast<size_t>(nw) * kSlab;  // [nw]
#pragma unroll
  for (int d = 0; d <= P3; ++d)
#pragma unroll
    for (int cc = 0; cc < NC; ++cc)
      if (cc < nc) {
        if (!MT && d == P3 && cc == nc - 1 && lane == 0) {
          T all = seen;
#pragma unroll
          for (int c = 0; c < NC; ++c) all += R[c][P3][0];
          flags[wave] = all;
        }
        flush(R[cc][d], cc, cur3 - P3 + d);
      }
  if constexpr (!MT) {
    T all = flags[0];
    for (int w = 1; w < nw; ++w) all += flags[w];
    if (__builtin_expect(!finite(wave_uniform(all)), 0)) {
      __syncthreads();
      AdjArgsAgain<T>& again = *kernel_args<T>();
      const AdjBlock here = adj_block(again, NC);
      for (int c = here.c0; c < min(here.c0 + NC, again.nout); ++c)
        banded_run<T, NIN, P3, NQ, NURBS>(again, red, here.bx, here.by, here.bz, c);
    }
  }
}

template <typename T>
using AdjMmaKernel = void (*)(AdjMmaArgs<T>);

template <typename T, int NIN, int P3, int NQ>
AdjMmaKernel<T> pick_tier(int tier, int nurbs_nc) {
  if constexpr (sizeof(T) == 4) {
    if constexpr (P3 <= kSharedMaxP3)
      if (nurbs_nc == 3) return adj_mma<T, NIN, P3, NQ, 3, SG_TIER_NATIVE, true>;
    if (nurbs_nc == 1) return adj_mma<T, NIN, P3, NQ, 1, SG_TIER_NATIVE, true>;
    switch (tier) {
      case SG_TIER_NATIVE: return adj_mma<T, NIN, P3, NQ, 1, SG_TIER_NATIVE, false>;
      case SG_TIER_SPLIT_F16: return adj_mma<T, NIN, P3, NQ, 1, SG_TIER_SPLIT_F16, false>;
      case SG_TIER_BF16: return adj_mma<T, NIN, P3, NQ, 1, SG_TIER_BF16, false>;
    }
    return nullptr;
  } else {
    return nurbs_nc ? adj_mma<T, NIN, P3, NQ, 1, SG_TIER_NATIVE, true>
                    : adj_mma<T, NIN, P3, NQ, 1, SG_TIER_NATIVE, false>;
  }
}

template <typename T, int NIN, int P3>
AdjMmaKernel<T> pick_nq(int tile_width, int tier, int nurbs_nc) {
  return tile_width == 64 ? pick_tier<T, NIN, P3, 4>(tier, nurbs_nc)
                          : pick_tier<T, NIN, P3, 2>(tier, nurbs_nc);
}

template <typename T>
AdjMmaKernel<T> pick_adj_mma(const Plan& pl, int tier, int nurbs_nc) {
  const int tw = pl.adjoint(sizeof(T)).tile_width();
  if (pl.nin == 2) return pick_nq<T, 2, 0>(tw, tier, nurbs_nc);
  switch (pl.dims[2].p) {
    case 0: return pick_nq<T, 3, 0>(tw, tier, nurbs_nc);
    case 1: return pick_nq<T, 3, 1>(tw, tier, nurbs_nc);
    case 2: return pick_nq<T, 3, 2>(tw, tier, nurbs_nc);
    case 3: return pick_nq<T, 3, 3>(tw, tier, nurbs_nc);
    case 4: return pick_nq<T, 3, 4>(tw, tier, nurbs_nc);
    case 5: return pick_nq<T, 3, 5>(tw, tier, nurbs_nc);
  }
  return nullptr;
}

long long plane_samples(const Plan& pl) {
  return static_cast<long long>(pl.dims[0].m) * pl.dims[1].m;
}

// Channels that share a workgroup and its weight field (NURBS).
template <typename T>
int weight_channels(const Plan& pl) {
  return sizeof(T) == 4 && adjoint_shares_weights(pl) ? 3 : 1;
}

template <typename T>
int resident_waves(const Plan& pl) {
  AdjMmaKernel<T> k = pick_adj_mma<T>(pl, SG_TIER_NATIVE, pl.nurbs ? weight_channels<T>(pl) : 0);
  if (!k) return 0;
  int blocks = 0, cus = 0, dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, reinterpret_cast<const void*>(k),
                                                   kThreads, 0) != hipSuccess)
    return 0;
  return blocks * kWaves * cus;
}

template <typename T>
hipError_t launch_mma(const Plan& pl, int tier, const int32_t* orders, const T* E, const T* W,
                      T* Pbar, int accumulate, hipStream_t s) {
  const Tiling& tl = pl.adjoint(sizeof(T));
  const DimDev& d1 = pl.dims[0];
  const DimDev& d2 = pl.dims[1];
  const auto table = [](const DimDev& d, int order) {
    const size_t at = static_cast<size_t>(order) * d.m * (d.p + 1);
    if constexpr (sizeof(T) == 4)
      return static_cast<const T*>(d.ktab32 + at);
    else
      return static_cast<const T*>(d.ktab64 + at);
  };
  AdjMmaArgs<T> a{};
  a.E = E;
  a.W = W;
  a.part = static_cast<T*>(pl.work);
  a.tab1 = table(d1, orders[0]);
  a.tab2 = table(d2, orders[1]);
  a.span1 = d1.span;
  a.span2 = d2.span;
  a.m1 = d1.m;
  a.m2 = d2.m;
  a.m3 = 1;
  a.p1 = d1.p;
  a.p2 = d2.p;
  a.n1 = d1.n;
  a.n2 = d2.n;
  a.n3 = 1;
  if (pl.nin == 3) {
    const DimDev& d3 = pl.dims[2];
    a.tab3 = table(d3, orders[2]);
    a.span3 = d3.span;
    a.m3 = d3.m;
    a.n3 = d3.n;
  }
  a.nout = pl.nout;
  a.rows = tl.rows_per_wave;
  a.chunk = tl.chunk_rows();
  a.j3_per_block = tl.j3_per_block;
  a.ntx = tl.n_tiles1;
  a.nty = tl.n_chunks2;
  a.nz = tl.n_z;
  a.xcd_map = tl.xcd_map;
  a.w1max = tl.w1max;
  a.w2max = tl.w2max;
  a.w3max = tl.w3max;
  a.m12 = plane_samples(pl);
  a.nsamp = a.m12 * a.m3;
  const int nurbs_nc = W ? weight_channels<T>(pl) : 0;
  const int per = std::max(nurbs_nc, 1);
  AdjMmaKernel<T> k = pick_adj_mma<T>(pl, tier, nurbs_nc);
  if (!k) return hipErrorInvalidValue;
  const int nw = tl.chunk_rows() / tl.rows_per_wave;
  const long long blocks = static_cast<long long>(tl.n_tiles1) * tl.n_chunks2 * tl.n_z;
  // the waves' sums and flags, or what banded_run keeps there
  const size_t lds = std::max(2 * static_cast<size_t>(nw) * kSlab + nw,
                              banded_lds(nw, tl.tile_width() / 16, W != nullptr)) * sizeof(T);
  // a plane's tiles are below 2^32 threads by its size (adjoint_mma_shape_ok),
  // those of every channel need not be
  const int groups = (pl.nout + per - 1) / per;
  const int at_once =
      static_cast<int>(std::min<long long>(launch_groups(blocks * nw * kLanes), groups));
  for (a.group0 = 0; a.group0 < groups; a.group0 += at_once) {
    const int n = std::min(at_once, groups - a.group0);
    hipLaunchKernelGGL(k, dim3(static_cast<unsigned>(blocks * n)), dim3(nw * kLanes), lds, s, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return launch_adjoint_gather(pl, tl, pl.work, Pbar, sizeof(T) == 4 ? SG_F32 : SG_F64,
                               accumulate, s, W);
}

}  // namespace

bool adjoint_mma_shape_ok(const Plan& pl, int dtype) {
  // one (sample j3, channel) plane of ebar must stay below the out-of-range
  // offset of the buffer loads
  return (pl.nin == 2 || pl.nin == 3) && (pl.nin == 2 || pl.dims[2].p <= kMaxStreamDegree) &&
         plane_samples(pl) * (dtype == SG_F32 ? 4 : 8) < static_cast<long long>(kOff) - 64;
}

int adjoint_mma_resident_waves(const Plan& pl) { return resident_waves<float>(pl); }
int adjoint_mma_resident_waves64(const Plan& pl) { return resident_waves<double>(pl); }

size_t adjoint_mma_work_bytes(const Plan& pl) {
  size_t most = 0;
  for (size_t elem : {sizeof(float), sizeof(double)}) {
    const Tiling& t = pl.adjoint(elem);
    if (t.n_tiles1 == 0) continue;
    const size_t units = static_cast<size_t>(t.n_tiles1) * t.n_chunks2 * t.n_z;
    most = std::max(most, units * t.w3max * pl.nout * t.w1max * t.w2max * elem);
  }
  return most;
}

hipError_t launch_adjoint_mma(const Plan& pl, int tier, const int32_t* orders, const void* E,
                              const void* W, void* Pbar, int dtype, int accumulate,
                              hipStream_t s) {
  if (dtype == SG_F32)
    return launch_mma<float>(pl, tier, orders, static_cast<const float*>(E),
                             static_cast<const float*>(W), static_cast<float*>(Pbar), accumulate,
                             s);
  return launch_mma<double>(pl, tier, orders, static_cast<const double*>(E),
                            static_cast<const double*>(W), static_cast<double*>(Pbar), accumulate,
                            s);
}

}  // namespace sg
