// rcg_gcf.hip -- w-projection GCF (gridding convolution function) taps on
// the GPU.
//
// Restates the reference's generator, MS4/kernel/cpu/gcf/GCF.cpp:16-219,
// and the per-plane loop of its caller, MS4/dna-programs/Kernel/CPU/GCF.hs:
// 36-89:
//
//  calcAccums   per w-plane sum of w and point count, plane = round(w/wstep)
//               (C rounding, half away from zero), planes centred at
//               n_planes / 2 (GCF.cpp:148-219);
//  mkGCFLayer   one plane's 64 oversampled layers: the w screen
//               exp(-2 pi i w (1 - sqrt(1 - x^2 - y^2))) on a max_support^2
//               block at the centre of an (8 max_support)^2 arena (row
//               pitch 8 max_support + src_pad), zero elsewhere; the backward
//               transform with fftshifts (fft_inplace_even, sign +1); the
//               sum of real parts over each of the 8 x 8 oversampling
//               sub-lattices; the support^2 window of every sub-lattice
//               divided by its sum -> dst[over_u][over_v][support][support]
//               (GCF.cpp:16-120).
//
// The reference's sums walk the padded arena as if it were contiguous
// (GCF.cpp:28-32), which reads the wrong elements when src_pad != 0 (the MS4
// Haskell caller uses src_pad = 4).  The default here is the pad-correct
// sum; `pad_quirk` selects the reference's walk.
//
// GPU structure.  Only max_support^2 cells of the arena differ from zero and
// only support^2 samples per sub-lattice are kept, so the transform is two
// small matrix products, out = E X E^T with E[u][a] = exp(2 pi i (u - L/2)
// (a - R) / L) (L = 8 max_support, R = max_support / 2, X the screen): FP64
// matrix instructions on 16 x 16 blocks, the terms of equal cells of X (which
// is even in both coordinates) together, one launch for all planes of a table
// (k_gcf_layers).  The sum over a sub-lattice needs no samples: the sum over
// its max_support^2 places of E's products is max_support^2 for the cell
// a = b = R, where the screen is 1, and 0 for every other.  With pad_quirk the
// sums need the whole padded arena: screen, rocFFT (rcg_fft plan), 64
// workgroups for the sums, one kernel for the window.
// calcAccums uses per-workgroup LDS histograms and one FP64 atomic per
// touched plane per workgroup.
#include <algorithm>
#include <climits>
#include <cmath>

#include "rcg_internal.h"

constexpr int GCF_OVER = 8;  // MS4/kernel/common/metrix.h:5
constexpr int ACC_MAX_PLANES = 8192;

struct rcg_gcf_gen {
  int max_support, src_pad, L, pitch;
  bool held = false;         // counted as a user of the FFT library state
  // pad_quirk only: made with the generator, or on first use where its maker
  // asked for that (rcg_gcf_gen_create_ex)
  double2 *arena = nullptr;  // L rows x pitch complex
  double *sums = nullptr;    // 64 sub-lattice sums
  rcg_fft_plan *fft = nullptr;
};

namespace rcg {
// rcg_fft.hip: counts a user of the FFT library state (+1, -1).
void fft_hold(int n);

namespace {

__global__ void __launch_bounds__(256)
k_wscreen(double2 *__restrict__ arena, int L, int pitch, int ms, double t2, double w)
{
#pragma clang fp contract(off)
  const int radius = ms / 2;
  const double normer = t2 / (double)radius;
  const int r0 = L / 2 - radius;
  const long long n = (long long)L * pitch;
  for (long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x; k < n;
       k += (long long)gridDim.x * blockDim.x) {
    const int r = (int)(k / pitch), c = (int)(k - (long long)r * pitch);
    double2 v = make_double2(0.0, 0.0);
    const int a = r - r0, b = c - r0;
    if (a >= 0 && a < ms && b >= 0 && b < ms) {
      const double x = (double)(a - radius) * normer;
      const double y = (double)(b - radius) * normer;
      const double ph = w * (1.0 - sqrt(1.0 - x * x - y * y));
      double s, co;
      sincos(2.0 * M_PI * ph, &s, &co);
      v = make_double2(co, -s);
    }
    arena[k] = v;
  }
}

// One cell of the screen, (a, b) places from its centre.
__device__ __forceinline__ double2 screen_cell(int a, int b, double normer, double w)
{
#pragma clang fp contract(off)
  const double x = (double)a * normer, y = (double)b * normer;
  const double ph = w * (1.0 - sqrt(1.0 - x * x - y * y));
  double s, co;
  sincos(2.0 * M_PI * ph, &s, &co);
  return make_double2(co, -s);
}

// Planes of one launch.
constexpr int GCF_PLANES = 64;
struct GcfPlanes {
  int n;
  int support[GCF_PLANES];
  int first[GCF_PLANES + 1];  // first workgroup of each plane
  long long off[GCF_PLANES];  // element offset of its layers in dst
  double w[GCF_PLANES];
};

constexpr int GCF_ROWS = 32;  // output rows of a workgroup
constexpr int GCF_THREADS = 1024, GCF_WAVES = GCF_THREADS / 64;

// LDS of k_gcf_layers: the L roots of unity, Y (GCF_ROWS x (R + 1), padded to
// whole blocks; a row one more than a multiple of 16 cells, so that the 16
// rows of an operand start in different banks) and, where it fits, the
// screen's quadrant.
__host__ __device__ inline int gcf_ypitch(int ms)
{
  return ((ms / 2 + 1 + 15) & ~15) + 1;
}
size_t gcf_lds(int ms, bool quad)
{
  const size_t q = quad ? (size_t)(ms / 2 + 1) * (ms / 2 + 1) : 0;
  return (8 * (size_t)ms + (size_t)GCF_ROWS * gcf_ypitch(ms) + q) * sizeof(double2);
}
constexpr size_t GCF_LDS = 160 * 1024;

typedef double d4 __attribute__((ext_vector_type(4)));

// acc += a b on 16 x 16 blocks, four products deep: A's row lane % 16, B's
// column lane % 16, term lane / 16; the result's column lane % 16, rows
// 4 i + lane / 16.
__device__ __forceinline__ void mfma_d(d4 &acc, double a, double b)
{
  acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
}

// 32 rows u of one plane: Y = E X, then Y E^T, each wavefront a share of the
// blocks of 16 x 16.  X is even in both coordinates, and so is Y in its
// second: the terms a and -a from the centre go together, with the real
// coefficient 2 cos, over a = 0..R.  Of an even max_support the last, a = R,
// stands for -R alone: coefficient exp(-i phi R), its imaginary part added
// by itself.  Output columns are taken in the order (over_v, sv), so that 16
// lanes write consecutive taps.  Bound by the matrix units and, for small
// supports, by the screen and the roots, which every workgroup computes (1089
// + 512 sincos at max_support 64).  One plane has few workgroups (64 at
// support 256) and from max_support 100 on a CU holds one, so the workgroup is
// as large as can be.  Measured, one plane of support = max_support 64 / 128 /
// 256, and 63 planes of it: 31 / 85 / 288 us and 0.24 / 0.82 / 4.7 ms; with 512
// threads 34 / 95 / 327 us, with 256 57 / 172 / 638; with all max_support^2
// terms, complex coefficients and 256 threads 79 / 283 / 1099 us; by rocFFT
// 65 / 122 / 302 us and, with the making of its plan, 6 / 12 / 23 ms.
template <class T, bool QUAD>
__global__ void __launch_bounds__(GCF_THREADS)
k_gcf_layers(GcfPlanes pl, int ms, double t2, T *__restrict__ out)
{
  extern __shared__ __attribute__((aligned(16))) char smem[];
  double2 *root = reinterpret_cast<double2 *>(smem);
  double2 *Y = root + 8 * ms;
  const int yp = gcf_ypitch(ms), R = ms / 2, L = 8 * ms, even = 1 - (ms & 1);
  double2 *quad = Y + GCF_ROWS * yp;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l16 = lane & 15, l4 = lane >> 4;
  int p = 0;
  while (p + 1 < pl.n && (int)blockIdx.x >= pl.first[p + 1]) p++;
  const int S = pl.support[p];
  const double w = pl.w[p], normer = t2 / (double)R;
  T *dst = out + pl.off[p];
  for (int k = threadIdx.x; k < L; k += GCF_THREADS) {
    double s, c;
    sincospi(2.0 * (double)k / (double)L, &s, &c);
    root[k] = make_double2(c, s);
  }
  if (QUAD) {
    const int qs = R + 1;
    for (int k = threadIdx.x; k < qs * qs; k += GCF_THREADS)
      quad[k] = screen_cell(k / qs, k % qs, normer, w);
  }
  __syncthreads();
  auto screen = [&](int a, int b) {  // a, b in [0, R], else 0
    if (a > R || b > R) return make_double2(0.0, 0.0);
    return QUAD ? quad[a * (R + 1) + b] : screen_cell(a, b, normer, w);
  };
  auto mod = [&](int k) {  // into [0, L)
    k %= L;
    return k < 0 ? k + L : k;
  };
  // coefficient of term a (root index e = u a mod L)
  auto coef = [&](int a, int e) {
    const double c = a > R ? 0.0 : root[e].x;
    return a == 0 || (even && a == R) ? c : 2.0 * c;
  };
  const int n8 = 8 * S;                           // output rows and columns
  const int start = (ms / 2 - S / 2) * GCF_OVER;  // of the window in the arena
  const int row0 = ((int)blockIdx.x - pl.first[p]) * GCF_ROWS;
  // this wavefront's 16 of the rows, and its first block of 16 columns
  const int h = wave & 1, c0 = (wave >> 1) * 16;
  constexpr int CSTEP = GCF_WAVES / 2 * 16;
  auto row_of = [&](int r) { return mod(start + min(row0 + 16 * h + r, n8 - 1) - L / 2); };
  // this lane's A row of E: root index at a = l4, and its step for a + 4
  const int u = row_of(l16);
  const int e0 = mod(u * l4), de = mod(4 * u);
  for (int b0 = c0; b0 <= R; b0 += CSTEP) {
    d4 re = {}, im = {};
    int e = e0;
    for (int a = l4; a <= R + l4; a += 4) {
      const double2 x = screen(a, b0 + l16);
      const double c = coef(a, e);
      mfma_d(re, c, x.x);
      mfma_d(im, c, x.y);
      e += de;
      e -= e >= L ? L : 0;
    }
    const double2 x = even ? screen(R, b0 + l16) : make_double2(0.0, 0.0);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int r = 4 * i + l4;
      const double s = root[mod(row_of(r) * R)].y;
      Y[(16 * h + r) * yp + b0 + l16] = make_double2(fma(s, x.y, re[i]), fma(-s, x.x, im[i]));
    }
  }
  __syncthreads();
  const double sum = (double)ms * (double)ms;
  for (int f0 = c0; f0 < n8; f0 += CSTEP) {
    const int f = min(f0 + l16, n8 - 1);
    const int ov = f / S, sv = f - ov * S;
    const int v = mod(start + 8 * sv + ov - L / 2);
    int e = mod(v * l4);
    const int d = mod(4 * v);
    d4 re = {}, im = {};
    for (int b = l4; b <= R + l4; b += 4) {
      const double2 y = Y[(16 * h + l16) * yp + min(b, R)];
      const double c = coef(b, e);
      mfma_d(re, y.x, c);
      mfma_d(im, y.y, c);
      e += d;
      e -= e >= L ? L : 0;
    }
    if (f0 + l16 >= n8) continue;
    const double s = even ? root[mod(v * R)].y : 0.0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int r = row0 + 16 * h + 4 * i + l4;
      if (r >= n8) continue;
      const double2 y = Y[(16 * h + 4 * i + l4) * yp + R];
      T o;
      o.x = fma(s, y.y, re[i]) / sum;
      o.y = fma(-s, y.x, im[i]) / sum;
      dst[((long long)((r & 7) * GCF_OVER + ov) * S + (r >> 3)) * S + sv] = o;
    }
  }
}

// Sum of real parts over sub-lattice (over_u, over_v) = blockIdx.x: the
// elements at contiguous offset ((su*8 + over_u)*ms + sv)*8 + over_v, su, sv <
// ms (the reference's walk, which takes the padded arena for a contiguous one).
__global__ void __launch_bounds__(256)
k_gcf_sums(const double2 *__restrict__ arena, int pitch, int ms,
           double *__restrict__ sums)
{
  __shared__ double sh[4];
  const int ou = blockIdx.x / GCF_OVER, ov = blockIdx.x % GCF_OVER;
  double acc = 0.0;
  for (int e = threadIdx.x; e < ms * ms; e += 256) {
    const int su = e / ms, sv = e - (e / ms) * ms;
    const long long k = ((long long)(su * GCF_OVER + ou) * ms + sv) * GCF_OVER + ov;
    acc += arena[k].x;
  }
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) sums[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

template <class T>
__global__ void __launch_bounds__(256)
k_gcf_extract(const double2 *__restrict__ arena, int pitch, int ms, int support,
              const double *__restrict__ sums, T *__restrict__ dst)
{
  const int start = (ms / 2 - support / 2) * GCF_OVER;
  const long long per = (long long)support * support;
  const long long n = 64 * per;
  for (long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x; k < n;
       k += (long long)gridDim.x * blockDim.x) {
    const int layer = (int)(k / per);
    const int e = (int)(k - layer * per);
    const int ou = layer / GCF_OVER, ov = layer % GCF_OVER;
    const int su = e / support, sv = e - (e / support) * support;
    const double2 a = arena[(long long)(start + ou + su * GCF_OVER) * pitch + start + ov +
                            sv * GCF_OVER];
    const double s = sums[layer];
    T o;
    o.x = a.x / s;
    o.y = a.y / s;
    dst[k] = o;
  }
}

// C round() of w / wstep + centre; LDS histogram per workgroup.
__global__ void __launch_bounds__(256)
k_accums(const rcg_double3 *__restrict__ uvw, long long n, double wstep, int n_planes,
         double *__restrict__ sums, int *__restrict__ npts, int *__restrict__ err)
{
#pragma clang fp contract(off)
  extern __shared__ double lds[];
  double *hs = lds;
  int *hn = reinterpret_cast<int *>(lds + n_planes);
  for (int p = threadIdx.x; p < n_planes; p += 256) {
    hs[p] = 0.0;
    hn[p] = 0;
  }
  __syncthreads();
  const int centre = n_planes / 2;
  int bad = 0;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const double w = uvw[i].w;
    const double q = round(w / wstep);
    if (!(q >= -centre && q < n_planes - centre)) {
      bad = 1;
      continue;
    }
    const int p = (int)q + centre;
    atomicAdd(&hs[p], w);
    atomicAdd(&hn[p], 1);
  }
  if (bad) atomicOr(err, ERR_RANGE);
  __syncthreads();
  for (int p = threadIdx.x; p < n_planes; p += 256) {
    if (hn[p]) {
      unsafeAtomicAdd(&sums[p], hs[p]);
      atomicAdd(&npts[p], hn[p]);
    }
  }
}

__global__ void k_zero_acc(double *__restrict__ sums, int *__restrict__ npts, int *err, int n)
{
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
    sums[p] = 0.0;
    npts[p] = 0;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0 && err) *err = 0;
}

}  // namespace
}  // namespace rcg

using namespace rcg;

extern "C" rcg_status rcg_gcf_gen_destroy(rcg_gcf_gen *g)
{
  if (!g) return RCG_OK;
  if (g->fft) rcg_fft_plan_destroy(g->fft);
  if (g->held) fft_hold(-1);
  if (g->arena) (void)hipFree(g->arena);
  if (g->sums) (void)hipFree(g->sums);
  delete g;
  return RCG_OK;
}

namespace {

// The arena, sums and FFT plan of the pad_quirk path.
rcg_status gen_arena(rcg_gcf_gen *g)
{
  if (g->fft) return RCG_OK;
  const size_t bytes = (size_t)g->L * g->pitch * sizeof(double2);
  if ((!g->arena && dev_malloc(reinterpret_cast<void **>(&g->arena), bytes) != hipSuccess) ||
      (!g->sums &&
       dev_malloc(reinterpret_cast<void **>(&g->sums), 64 * sizeof(double)) != hipSuccess)) {
    set_error(RCG_ERR_NOMEM, "rcg_gcf_gen: device arena of %zu bytes", bytes);
    return RCG_ERR_NOMEM;
  }
  return rcg_fft_plan_create(1, 1, g->L, g->pitch, &g->fft);
}

}  // namespace

extern "C" rcg_status rcg_gcf_gen_create(int max_support, int src_pad, rcg_gcf_gen **out)
{
  return rcg_gcf_gen_create_ex(max_support, src_pad, 1, out);
}

extern "C" rcg_status rcg_gcf_gen_create_ex(int max_support, int src_pad, int arena,
                                            rcg_gcf_gen **out)
{
  clear_error();
  if (!out || max_support < 2 || max_support > MAX_SUPPORT || src_pad < 0 || src_pad > 4096) {
    set_error(RCG_ERR_ARG, "rcg_gcf_gen_create: max_support %d / src_pad %d out of range",
              max_support, src_pad);
    return RCG_ERR_ARG;
  }
  *out = nullptr;
  rcg_gcf_gen *g = new (std::nothrow) rcg_gcf_gen();
  if (!g) {
    set_error(RCG_ERR_NOMEM, "host allocation failed");
    return RCG_ERR_NOMEM;
  }
  g->max_support = max_support;
  g->src_pad = src_pad;
  g->L = max_support * GCF_OVER;
  g->pitch = g->L + src_pad;
  fft_hold(1);
  g->held = true;
  const rcg_status s = arena ? gen_arena(g) : RCG_OK;
  if (s != RCG_OK) {
    rcg_gcf_gen_destroy(g);
    return s;
  }
  *out = g;
  return RCG_OK;
}

namespace {

rcg_status quirk_layer(rcg_gcf_gen *g, void *dst, int f64, int support, double t2, double w,
                       hipStream_t st)
{
  rcg_status s = gen_arena(g);
  if (s != RCG_OK) return s;
  const long long cells = (long long)g->L * g->pitch;
  const int nb = (int)std::min<long long>((cells + 255) / 256, 2048);
  hipLaunchKernelGGL(k_wscreen, dim3(nb), dim3(256), 0, st, g->arena, g->L, g->pitch,
                     g->max_support, t2, w);
  RCG_HIP_TRY(hipGetLastError());
  s = rcg_fft_execute(g->fft, g->arena, st);
  if (s != RCG_OK) return s;
  hipLaunchKernelGGL(k_gcf_sums, dim3(64), dim3(256), 0, st, g->arena, g->pitch, g->max_support,
                     g->sums);
  const long long n = 64LL * support * support;
  const int nb2 = (int)std::min<long long>((n + 255) / 256, 1024);
  if (f64)
    hipLaunchKernelGGL(k_gcf_extract<double2>, dim3(nb2), dim3(256), 0, st, g->arena, g->pitch,
                       g->max_support, support, g->sums, static_cast<double2 *>(dst));
  else
    hipLaunchKernelGGL(k_gcf_extract<float2>, dim3(nb2), dim3(256), 0, st, g->arena, g->pitch,
                       g->max_support, support, g->sums, static_cast<float2 *>(dst));
  RCG_HIP_TRY(hipGetLastError());
  return RCG_OK;
}

template <class T, bool QUAD>
rcg_status launch_layers(const GcfPlanes &pl, int ms, double t2, void *dst, hipStream_t st)
{
  const size_t lds = gcf_lds(ms, QUAD);
  RCG_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_gcf_layers<T, QUAD>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)GCF_LDS));
  hipLaunchKernelGGL((k_gcf_layers<T, QUAD>), dim3(pl.first[pl.n]), dim3(GCF_THREADS), lds, st, pl, ms, t2,
                     static_cast<T *>(dst));
  RCG_HIP_TRY(hipGetLastError());
  return RCG_OK;
}

}  // namespace

extern "C" rcg_status rcg_gcf_gen_layers(rcg_gcf_gen *g, void *dst, int f64, int n,
                                         const int *supports, const long long *offsets, double t2,
                                         const double *w, int pad_quirk, void *stream)
{
  clear_error();
  if (!g || !dst || n < 1 || !supports || !offsets || !w) {
    set_error(RCG_ERR_ARG, "rcg_gcf_gen_layers: null argument or no plane");
    return RCG_ERR_ARG;
  }
  for (int k = 0; k < n; k++)
    if (supports[k] < 1 || supports[k] > g->max_support || offsets[k] < 0) {
      set_error(RCG_ERR_ARG, "plane %d: support %d outside [1, %d] or offset %lld", k, supports[k],
                g->max_support, offsets[k]);
      return RCG_ERR_ARG;
    }
  hipStream_t st = (hipStream_t)stream;
  if (pad_quirk) {
    for (int k = 0; k < n; k++) {
      char *to = static_cast<char *>(dst) + offsets[k] * (f64 ? sizeof(double2) : sizeof(float2));
      const rcg_status s = quirk_layer(g, to, f64, supports[k], t2, w[k], st);
      if (s != RCG_OK) return s;
    }
    return RCG_OK;
  }
  const int ms = g->max_support;
  const bool quad = gcf_lds(ms, true) <= GCF_LDS;
  for (int k0 = 0; k0 < n; k0 += GCF_PLANES) {
    GcfPlanes pl;
    pl.n = std::min(GCF_PLANES, n - k0);
    pl.first[0] = 0;
    for (int k = 0; k < pl.n; k++) {
      pl.support[k] = supports[k0 + k];
      pl.off[k] = offsets[k0 + k];
      pl.w[k] = w[k0 + k];
      pl.first[k + 1] = pl.first[k] + (8 * pl.support[k] + GCF_ROWS - 1) / GCF_ROWS;
    }
    const rcg_status s = f64 ? (quad ? launch_layers<double2, true>(pl, ms, t2, dst, st)
                                     : launch_layers<double2, false>(pl, ms, t2, dst, st))
                             : (quad ? launch_layers<float2, true>(pl, ms, t2, dst, st)
                                     : launch_layers<float2, false>(pl, ms, t2, dst, st));
    if (s != RCG_OK) return s;
  }
  return RCG_OK;
}

extern "C" rcg_status rcg_gcf_gen_layer(rcg_gcf_gen *g, void *dst, int f64, int support,
                                        double t2, double w, int pad_quirk, void *stream)
{
  clear_error();
  if (!g || !dst || support < 1 || support > g->max_support) {
    set_error(RCG_ERR_ARG, "rcg_gcf_gen_layer: support %d outside [1, %d]", support,
              g ? g->max_support : 0);
    return RCG_ERR_ARG;
  }
  const long long off = 0;
  return rcg_gcf_gen_layers(g, dst, f64, 1, &support, &off, t2, &w, pad_quirk, stream);
}

extern "C" rcg_status rcg_calc_accums(const rcg_double3 *uvw, long long n, double wstep,
                                      int n_planes, double *sums, int *npts, int *err_dev,
                                      void *stream)
{
  clear_error();
  if ((n > 0 && !uvw) || !sums || !npts || !err_dev || n < 0 || n_planes < 1 ||
      n_planes > ACC_MAX_PLANES || !(wstep > 0.0)) {
    set_error(RCG_ERR_ARG, "rcg_calc_accums: bad argument (n %lld, planes %d, wstep %g)", n,
              n_planes, wstep);
    return RCG_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(k_zero_acc, dim3(std::max(1, (n_planes + 255) / 256)), dim3(256), 0, st,
                     sums, npts, err_dev, n_planes);
  RCG_HIP_TRY(hipGetLastError());
  if (n == 0) return RCG_OK;
  const int nb = (int)std::min<long long>((n + 255) / 256, 1024);
  const size_t lds = (size_t)n_planes * (sizeof(double) + sizeof(int));
  if (lds > 64 * 1024) {
    RCG_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_accums),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
  }
  hipLaunchKernelGGL(k_accums, dim3(nb), dim3(256), lds, st, uvw, n, wstep, n_planes, sums,
                     npts, err_dev);
  RCG_HIP_TRY(hipGetLastError());
  return RCG_OK;
}

// ---------------------------------------------------------------------------
// The reference's host entry points (host memory; GCF.cpp:123-146, 148-152)

namespace {
thread_local bool t_pad_quirk = false;
}

extern "C" void rcg_gcf_pad_quirk(int enable) { t_pad_quirk = enable != 0; }

extern "C" void *mkGCFLayer(void *p, rcg_c128 dst[], rcg_c128 *table[], rcg_c128 arena[],
                            int support, int max_support, int src_pad, double t2, double w)
{
  (void)arena;  // the work buffer lives on the device
  clear_error();
  if (!dst || !table) {
    set_error(RCG_ERR_ARG, "mkGCFLayer: null argument");
    return p;
  }
  rcg_gcf_gen *g = static_cast<rcg_gcf_gen *>(p);
  if (g && (g->max_support != max_support || g->src_pad != src_pad)) {
    set_error(RCG_ERR_ARG, "mkGCFLayer: generator made for max_support %d / pad %d",
              g->max_support, g->src_pad);
    return p;
  }
  if (!g && rcg_gcf_gen_create_ex(max_support, src_pad, t_pad_quirk ? 1 : 0, &g) != RCG_OK)
    return nullptr;
  const size_t bytes = 64ull * support * support * sizeof(rcg_c128);
  hipStream_t st = nullptr;
  void *d = nullptr;
  if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess ||
      dev_malloc(&d, bytes) != hipSuccess) {
    set_error(RCG_ERR_NOMEM, "mkGCFLayer: device buffers");
  } else if (rcg_gcf_gen_layer(g, d, 1, support, t2, w, t_pad_quirk, st) == RCG_OK) {
    if (hipMemcpyAsync(dst, d, bytes, hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
      set_error(RCG_ERR_HIP, "mkGCFLayer: copy out");
    for (int i = 0; i < 64; i++) table[i] = dst + (size_t)i * support * support;
  }
  if (st) (void)hipStreamSynchronize(st);
  if (d) (void)hipFree(d);
  if (st) (void)hipStreamDestroy(st);
  return g;
}

extern "C" void calcAccums(const rcg_double3 uvw[], double sums[], int npts[], double wstep,
                           int numDataPoints, int numOfWPlanes)
{
  clear_error();
  if (!uvw || !sums || !npts || numDataPoints < 0 || numOfWPlanes < 1) {
    set_error(RCG_ERR_ARG, "calcAccums: bad argument");
    return;
  }
  hipStream_t st = nullptr;
  void *du = nullptr, *ds = nullptr, *dn = nullptr, *de = nullptr;
  const size_t ub = (size_t)numDataPoints * sizeof(rcg_double3);
  if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess ||
      dev_malloc(&du, ub ? ub : 1) != hipSuccess ||
      dev_malloc(&ds, numOfWPlanes * sizeof(double)) != hipSuccess ||
      dev_malloc(&dn, numOfWPlanes * sizeof(int)) != hipSuccess ||
      dev_malloc(&de, sizeof(int)) != hipSuccess) {
    set_error(RCG_ERR_NOMEM, "calcAccums: device buffers");
  } else if ((ub && hipMemcpyAsync(du, uvw, ub, hipMemcpyHostToDevice, st) != hipSuccess)) {
    set_error(RCG_ERR_HIP, "calcAccums: copy in");
  } else if (rcg_calc_accums(static_cast<rcg_double3 *>(du), numDataPoints, wstep, numOfWPlanes,
                             static_cast<double *>(ds), static_cast<int *>(dn),
                             static_cast<int *>(de), st) == RCG_OK) {
    int e = 0;
    if (hipMemcpyAsync(sums, ds, numOfWPlanes * sizeof(double), hipMemcpyDeviceToHost, st) !=
            hipSuccess ||
        hipMemcpyAsync(npts, dn, numOfWPlanes * sizeof(int), hipMemcpyDeviceToHost, st) !=
            hipSuccess ||
        hipMemcpyAsync(&e, de, sizeof(int), hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
      set_error(RCG_ERR_HIP, "calcAccums: copy out");
    else if (e)
      set_error(RCG_ERR_RANGE, "calcAccums: points with a w-plane outside the %d planes "
                "(skipped)", numOfWPlanes);
  }
  if (st) (void)hipStreamSynchronize(st);
  void *bufs[] = {du, ds, dn, de};
  for (void *b : bufs)
    if (b) (void)hipFree(b);
  if (st) (void)hipStreamDestroy(st);
}
