// sg_forward_sweep.hip -- evaluate!(grid) of large scalar volumes, swept along
// dimension 3.
//
// One channel gives the streaming kernel (sg_forward.hip) little to store per
// row, so its per-plane stage 1 and first columns weigh as much as the stores.
// Here one thread holds 16 bytes of neighbouring samples of dimension 1 and
// walks a run of j3.  Per control plane k3 its samples' values, contracted
// along dimensions 1 and 2, sit in a register ring of p3 + 1 planes, so a
// sample costs p3 + 1 multiply-adds and one 16-byte store serves V samples:
//   stage 1 (workgroup, LDS): every plane of the run contracted along
//            dimension 2 for the tile's rows,
//            G[k3][row][k1] = sum_b B2[j2, b] * P[k1, s2-p2+b, k3]
//   stage 2 (thread): O[k3][v] = sum_a B1[j1+v, a] * G[k3][row][s1-p1+a]
//            when the span of dimension 3 advances, and for every j3
//            eval[j1+v, j2, j3] = sum_d B3[j3, d] * O[s3-p3+d][v]
// Threads are numbered through the rows of a tile, so rows of any length fill
// the waves.  512x512x256 FP32 54 us (4.9 TB/s; streaming 65), 200x200x200
// 15.5 (20.5), 360x466x133 21 (34), 400x400x200 FP64 48 (58).  What is left
// over the bare stores (42 us at 512x512x256) is the prologue's loads, which
// wait behind other workgroups' stores.
#include "sg_internal.hpp"

namespace sg {

namespace {

template <typename T>
constexpr int kVec = 16 / static_cast<int>(sizeof(T));  // samples per thread

template <typename T>
struct SweepArgs {
  const T* P;
  const int32_t *span1, *span2;
  const T *tab1, *tab2;  // [m][p+1] at the field's order
  int n1, n2, m1, m2, m3, p2;
  int threads_x, rows;   // a tile: threads_x threads along dimension 1, rows of dimension 2
  unsigned rcp_x;        // udiv_rcp(threads_x)
  int ntx, nty, run, xcd_map;
};

template <typename T, int P1, int P3>
__global__ __launch_bounds__(kThreads) void fwd_sweep(
    SweepArgs<T> a, const int32_t* __restrict__ span3, const T* __restrict__ tab3,
    T* __restrict__ out) {
  extern __shared__ __align__(16) unsigned char smem[];
  T* G = reinterpret_cast<T*>(smem);
  constexpr int V = kVec<T>;
  typedef T Vec __attribute__((ext_vector_type(V), aligned(sizeof(T))));

  const int L = xcd_logical_block(a.xcd_map, a.ntx);
  const int bx = L % a.ntx, by = (L / a.ntx) % a.nty;
  const int j3b = L / (a.ntx * a.nty) * a.run, j3e = min(j3b + a.run, a.m3);
  const int row0 = by * a.rows, nrows = min(a.rows, a.m2 - row0);
  const int x0 = bx * a.threads_x * V, x1 = min(x0 + a.threads_x * V, a.m1) - 1;
  const int lo1 = a.span1[x0] - P1, W1 = a.span1[x1] - lo1 + 1;
  const int lo3 = span3[j3b] - P3, planes = span3[j3e - 1] - lo3 + 1;
  const int cs = W1 * nrows;  // LDS elements of a plane

  // what stage 2 needs of dimension 1, loaded ahead of stage 1
  const int r = udiv_fast(threadIdx.x, a.threads_x, a.rcp_x);
  const int x = x0 + V * (static_cast<int>(threadIdx.x) - r * a.threads_x);
  int q1[V];
  T b1[V][P1 + 1];
#pragma unroll
  for (int v = 0; v < V; ++v) {
    const int j1 = min(x + v, x1);
    q1[v] = a.span1[j1] - P1 - lo1;
#pragma unroll
    for (int d = 0; d <= P1; ++d) b1[v][d] = a.tab1[static_cast<size_t>(j1) * (P1 + 1) + d];
  }

  // ---- stage 1 ----
  const long long plane = static_cast<long long>(a.n1) * a.n2;
  for (int idx = threadIdx.x; idx < planes * cs; idx += blockDim.x) {
    const int k = idx / cs, i = idx - k * cs;
    const int row = i / W1;
    const int j2 = row0 + row;
    const T* b2 = a.tab2 + static_cast<size_t>(j2) * (a.p2 + 1);
    long long off = lo1 + i - row * W1 +
                    static_cast<long long>(a.n1) * (a.span2[j2] - a.p2) + plane * (lo3 + k);
    T s = T(0);
#pragma unroll 4
    for (int d = 0; d <= a.p2; ++d, off += a.n1) s += b2[d] * a.P[off];
    G[idx] = s;
  }
  __syncthreads();

  // ---- stage 2 ----
  if (r >= nrows || x > x1) return;  // no barrier follows
  T O[P3 + 1][V];
  const T* g = G + r * W1;
  auto next_plane = [&](T(&o)[V]) {
#pragma unroll
    for (int v = 0; v < V; ++v) {
      T s = T(0);
#pragma unroll
      for (int d = 0; d <= P1; ++d) s += b1[v][d] * g[q1[v] + d];
      o[v] = s;
    }
    g += cs;
  };
#pragma unroll
  for (int q = 0; q <= P3; ++q) next_plane(O[q]);

  int cur = lo3 + P3;
  const bool whole = x + V <= a.m1;
  const long long step = static_cast<long long>(a.m1) * a.m2;
  T* dst = out + x + static_cast<long long>(a.m1) * (row0 + r) + step * j3b;
  int s3 = span3[j3b];
  T b3[P3 + 1];
#pragma unroll
  for (int q = 0; q <= P3; ++q) b3[q] = tab3[static_cast<size_t>(j3b) * (P3 + 1) + q];
  for (int j3 = j3b; j3 < j3e; ++j3, dst += step) {
    while (cur < s3) {
#pragma unroll
      for (int q = 0; q < P3; ++q)
#pragma unroll
        for (int v = 0; v < V; ++v) O[q][v] = O[q + 1][v];
      ++cur;
      next_plane(O[P3]);
    }
    // span and B3 of the next j3: scalar loads, one step ahead
    const int jn = min(j3 + 1, j3e - 1);
    s3 = span3[jn];
    T bn[P3 + 1];
#pragma unroll
    for (int q = 0; q <= P3; ++q) bn[q] = tab3[static_cast<size_t>(jn) * (P3 + 1) + q];
    Vec u;
#pragma unroll
    for (int v = 0; v < V; ++v) {
      T s = T(0);
#pragma unroll
      for (int q = 0; q <= P3; ++q) s += b3[q] * O[q][v];
      u[v] = s;
    }
    if (whole) {
      *reinterpret_cast<Vec*>(dst) = u;
    } else {
#pragma unroll
      for (int v = 0; v < V - 1; ++v)
        if (x + v < a.m1) dst[v] = u[v];
    }
#pragma unroll
    for (int q = 0; q <= P3; ++q) b3[q] = bn[q];
  }
}

template <typename T>
using SweepKernel = void (*)(SweepArgs<T>, const int32_t*, const T*, T*);

template <typename T, int P1>
SweepKernel<T> pick_p3(int p3) {
  switch (p3) {
    case 1: return fwd_sweep<T, P1, 1>;
    case 2: return fwd_sweep<T, P1, 2>;
    case 3: return fwd_sweep<T, P1, 3>;
    case 4: return fwd_sweep<T, P1, 4>;
  }
  return nullptr;
}

template <typename T>
SweepKernel<T> pick_sweep(int p1, int p3) {
  switch (p1) {
    case 1: return pick_p3<T, 1>(p3);
    case 2: return pick_p3<T, 2>(p3);
    case 3: return pick_p3<T, 3>(p3);
    case 4: return pick_p3<T, 4>(p3);
  }
  return nullptr;
}

template <typename T>
const T* table(const DimDev& d, int order);
template <>
const float* table<float>(const DimDev& d, int order) {
  return d.ktab32 + static_cast<size_t>(order) * d.m * (d.p + 1);
}
template <>
const double* table<double>(const DimDev& d, int order) {
  return d.ktab64 + static_cast<size_t>(order) * d.m * (d.p + 1);
}

template <typename T>
hipError_t launch(const Plan& pl, const int32_t* orders, const T* P, T* out, hipStream_t s) {
  const DimDev &d1 = pl.dims[0], &d2 = pl.dims[1], &d3 = pl.dims[2];
  const Sweep& t = pl.sweep[sizeof(T) == sizeof(double)];
  SweepArgs<T> a{};
  a.P = P;
  a.span1 = d1.span;
  a.span2 = d2.span;
  a.tab1 = table<T>(d1, orders[0]);
  a.tab2 = table<T>(d2, orders[1]);
  a.n1 = d1.n;
  a.n2 = d2.n;
  a.m1 = d1.m;
  a.m2 = d2.m;
  a.m3 = d3.m;
  a.p2 = d2.p;
  a.threads_x = t.threads_x;
  a.rcp_x = udiv_rcp(static_cast<unsigned>(t.threads_x));
  a.rows = t.rows;
  a.ntx = t.ntx;
  a.nty = t.nty;
  a.run = t.run;
  a.xcd_map = t.xcd_map;
  const SweepKernel<T> k = pick_sweep<T>(d1.p, d3.p);
  if (!k) return hipErrorInvalidValue;
  const int threads = (t.threads_x * t.rows + kLanes - 1) / kLanes * kLanes;
  hipLaunchKernelGGL(k, dim3(static_cast<unsigned>(t.ntx) * t.nty * t.nz), dim3(threads),
                     t.lds_elements * sizeof(T), s, a, d3.span, table<T>(d3, orders[2]), out);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_forward_sweep(const Plan& pl, const int32_t* orders, const void* P, void* out,
                                int dtype, hipStream_t s) {
  if (dtype == SG_F32)
    return launch(pl, orders, static_cast<const float*>(P), static_cast<float*>(out), s);
  return launch(pl, orders, static_cast<const double*>(P), static_cast<double*>(out), s);
}

}  // namespace sg
