// rcg_plain.hip -- the FP64 "plain" gridder and degridder.
//
// One launch covers every point.  Gridding: one wavefront handles one point at
// a time, its lanes cover the point's S x S window (rows of min(S,64) lanes)
// and add every tap to HBM with a native FP64 atomic (global_atomic_add_f64).
// Degridding: 16 or 64 lanes a point, summed across them with shuffles.  Arithmetic follows the reference's
// complex product (scatter_gridder_w_dependent_dyn_1p.cpp:169 grid,
// :171 degrid) in FP64 with contraction switched off.  This is the
// straightforward GPU gridder and the denominator the tiled FP32 path is
// measured against.
#include "rcg_internal.h"

namespace rcg {

__device__ __forceinline__ void window_lanes(int S, int lane, int *r0,
                                             int *c0, int *rows, int *cols)
{
  const int c = S < 64 ? (S > 0 ? S : 1) : 64;
  *cols = c;
  *rows = 64 / c;
  *r0 = lane / c;
  *c0 = lane - (lane / c) * c;
}

__global__ void __launch_bounds__(256)
k_grid_plain_f64(const rcg_pg *__restrict__ pg,
                 const double2 *__restrict__ vis,
                 const double2 *__restrict__ taps, double2 *__restrict__ grid,
                 int pitch, long long n)
{
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const long long wave = ((long long)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const long long nwaves = ((long long)gridDim.x * blockDim.x) >> 6;
  for (long long i = wave; i < n; i += nwaves) {
    const rcg_pg r = pg[i];
    if (r.cell < 0) continue;
    const double2 v = vis[i];
    const int S = r.supp, st = r.stride;
    int r0, c0, rows, cols;
    window_lanes(S, lane, &r0, &c0, &rows, &cols);
    if (r0 >= rows) continue;
    const double sgn = (r.flags & PG_CONJ) ? -1.0 : 1.0;
    for (int su = r0; su < S; su += rows) {
      const double2 *trow = taps + r.tap0 + su * st;
      double *grow = reinterpret_cast<double *>(grid + r.cell + (long long)su * pitch);
      for (int sv = c0; sv < S; sv += cols) {
        double2 t = trow[sv];
        t.y *= sgn;
        const double pr = v.x * t.x - v.y * t.y;
        const double pi = v.x * t.y + v.y * t.x;
        unsafeAtomicAdd(grow + 2 * sv, pr);
        unsafeAtomicAdd(grow + 2 * sv + 1, pi);
      }
    }
  }
}

// PL lanes per point: they take the taps of its window in row order, PL apart,
// U steps' loads together.  Of many points, 16 lanes each: four share a
// wavefront and the latency of its chain (record, taps and cells, sums,
// store): 500,310 points of supports 8..24 on 1024^2 0.092 against 0.167 ms
// with a wavefront per point, 2,496,960 of 8..48 on 2048^2 0.41 against 0.81.
// Of few, up to FEW_POINTS, a wavefront each: there are lanes enough, and the
// S^2 / 16 steps of a large window would be the time (100 points of 64 x 64:
// 11 against 33 us, 1000 of 128 x 128: 89 against 149, 4096: 125 against 155;
// 8000 of 32, 64, 128: 24, 81, 349 against 21, 65, 229).  More of their steps
// together help only where the caches do not bound (3000 of 256 x 256: 366 us
// with one, 433 with two, 514 with four).  A lane sums each of its U steps
// apart, so that either way a window is 64 sums, added in the same order: 16
// chains would be four times as long and their errors up to 1.8 times as large
// (64 x 64 normal deviates, relative L2: 5.5e-16 against 3.2e-16).
template <int PL, int U>
__global__ void __launch_bounds__(256)
k_degrid_plain_f64(const rcg_pg *__restrict__ pg,
                   const double2 *__restrict__ grid,
                   const double2 *__restrict__ taps,
                   double2 *__restrict__ vis, int pitch, long long n)
{
#pragma clang fp contract(off)
  const int sub = threadIdx.x & (PL - 1);
  const long long first = ((long long)blockIdx.x * blockDim.x + threadIdx.x) / PL;
  const long long step = (long long)gridDim.x * blockDim.x / PL;
  // every lane of a wavefront makes as many turns as its first point
  const long long turns = (n - (first - (threadIdx.x & 63) / PL) + step - 1) / step;
  rcg_pg next = pg[min(first, n - 1)];
  for (long long k = 0; k < turns; k++) {
    const long long i = first + k * step;
    const rcg_pg r = next;
    next = pg[min(i + step, n - 1)];
    double ar[U] = {}, ai[U] = {};
    if (i < n && r.cell >= 0 && r.supp > 0) {
      const int S = r.supp, st = r.stride, total = S * S;
      const double sgn = (r.flags & PG_CONJ) ? -1.0 : 1.0;
      // quotients by the approximate reciprocal: (x + 0.5) / S lies at least
      // 0.5 / S >= 1/512 from an integer, far above its error
      const float inv = __builtin_amdgcn_rcpf((float)S);
      const int row = (int)(((float)sub + 0.5f) * inv), dr = (int)(((float)PL + 0.5f) * inv);
      int col = sub - row * S;
      const int dc = PL - dr * S;
      const double2 *t = taps + r.tap0 + (long long)row * st + col;
      const double2 *g = grid + r.cell + (long long)row * pitch + col;
      const long long dt = (long long)dr * st + dc, dg = (long long)dr * pitch + dc;
      for (int q = sub; q < total; q += U * PL) {
        double2 tt[U], gg[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
          const bool act = q + u * PL < total;
          tt[u] = act ? *t : make_double2(0.0, 0.0);
          gg[u] = act ? *g : make_double2(0.0, 0.0);
          col += dc;
          t += dt;
          g += dg;
          if (col >= S) {
            col -= S;
            t += st - S;
            g += pitch - S;
          }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
          const double ty = tt[u].y * sgn;
          const double pr = gg[u].x * tt[u].x - gg[u].y * ty;
          const double pi = gg[u].x * ty + gg[u].y * tt[u].x;
          ar[u] += pr;
          ai[u] += pi;
        }
      }
    }
#pragma unroll
    for (int h = U / 2; h > 0; h >>= 1)
#pragma unroll
      for (int u = 0; u < h; u++) {
        ar[u] += ar[u + h];
        ai[u] += ai[u + h];
      }
#pragma unroll
    for (int off = PL / 2; off > 0; off >>= 1) {
      ar[0] += __shfl_xor(ar[0], off);
      ai[0] += __shfl_xor(ai[0], off);
    }
    if (sub == 0 && i < n) vis[i] = make_double2(ar[0], ai[0]);
  }
}

__global__ void k_zero_f64(double *__restrict__ p, long long n)
{
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    p[i] = 0.0;
}

constexpr long long FEW_POINTS = 6144;

static int plain_blocks(long long n)
{
  // four wavefronts per block, grid-stride beyond 64k blocks
  long long b = (n + 3) / 4;
  if (b > 65536) b = 65536;
  return (int)(b < 1 ? 1 : b);
}

}  // namespace rcg

extern "C" rcg_status rcg_grid_plain_f64(const rcg_geom *geom,
                                         const rcg_gcf *gcf,
                                         const rcg_pg *pg,
                                         const rcg_c128 *vis, rcg_c128 *grid,
                                         void *stream)
{
  using namespace rcg;
  clear_error();
  if (!geom || !gcf || !pg || !vis || !grid) {
    set_error(RCG_ERR_ARG, "rcg_grid_plain_f64: null argument");
    return RCG_ERR_ARG;
  }
  rcg_status s = check_geom(geom);
  if (s != RCG_OK) return s;
  hipStream_t st = (hipStream_t)stream;
  // zeroed by a kernel rather than a memset node, so the call can be
  // captured into a graph
  const long long nd = 2LL * geom->grid_size * geom->grid_pitch;
  hipLaunchKernelGGL(k_zero_f64, dim3(2048), dim3(256), 0, st,
                     reinterpret_cast<double *>(grid), nd);
  const long long n = (long long)geom->n_chunks * geom->ts_ch;
  if (n == 0) return RCG_OK;
  hipLaunchKernelGGL(k_grid_plain_f64, dim3(plain_blocks(n)), dim3(256), 0, st,
                     pg, reinterpret_cast<const double2 *>(vis),
                     reinterpret_cast<const double2 *>(gcf->data),
                     reinterpret_cast<double2 *>(grid), geom->grid_pitch, n);
  RCG_HIP_TRY(hipGetLastError());
  return RCG_OK;
}

extern "C" rcg_status rcg_degrid_plain_f64(const rcg_geom *geom,
                                           const rcg_gcf *gcf,
                                           const rcg_pg *pg,
                                           const rcg_c128 *grid,
                                           rcg_c128 *vis, void *stream)
{
  using namespace rcg;
  clear_error();
  if (!geom || !gcf || !pg || !vis || !grid) {
    set_error(RCG_ERR_ARG, "rcg_degrid_plain_f64: null argument");
    return RCG_ERR_ARG;
  }
  rcg_status s = check_geom(geom);
  if (s != RCG_OK) return s;
  const long long n = (long long)geom->n_chunks * geom->ts_ch;
  if (n == 0) return RCG_OK;
  const bool few = n <= FEW_POINTS;
  hipLaunchKernelGGL(few ? (k_degrid_plain_f64<64, 1>) : (k_degrid_plain_f64<16, 4>),
                     dim3(plain_blocks(few ? n : (n + 3) / 4)), dim3(256), 0, (hipStream_t)stream,
                     pg, reinterpret_cast<const double2 *>(grid),
                     reinterpret_cast<const double2 *>(gcf->data),
                     reinterpret_cast<double2 *>(vis), geom->grid_pitch, n);
  RCG_HIP_TRY(hipGetLastError());
  return RCG_OK;
}
