// rcg_clean.hip -- Hogbom CLEAN minor cycle on the GPU.
//
// Interface of the reference's deconvolve (MS4/kernel/common/hogbom.h:7-16,
// body MS4/kernel/cpu/hogbom/hogbom.cpp:94-121) with textbook semantics:
//   model = 0; p = argmax |psf|, pv = psf[p]
//   repeat niters: r = argmax |res| (first index on ties), v = res[r];
//     stop if |v| < threshold; a = gain * v / pv;
//     res[x] -= a * psf[x - r + p] where x - r + p lies in the image;
//     model[r] += a.
// (The reference's own findPeak reads past the array and returns |x|, so its
// results are not reproduced; see the oracle.)
//
// GPU structure.  Subtracting a component changes every pixel, but the peak
// moves among few: the image is cut into at most 4096 square tiles, and a
// tile is brought up to date (the components since its last visit subtracted,
// in their order, its maximum found) only when it can hold the peak.  For
// every tile the maximum e at its last visit and a slack s are kept, s the
// sum of |a| times the largest |psf| over the part of the PSF that covered the
// tile, for the components since.  Its maximum now is at most e + s, and the
// image's at least the largest e - s; the tiles with e + s not below that are
// visited, and more while one not visited could still exceed the best found.
// So each iteration finds the same peak as a pass over the whole image, and
// every pixel sees the same subtractions in the same order: the results are
// bit for bit those of the passes.
//
//   k_clean_tiles   one workgroup per tile: all pending components subtracted,
//                   the tile's maximum (also the PSF's, with none pending);
//   k_clean_prep    the PSF's peak and its tile maxima over 2 x 2 tiles;
//   k_clean_minor   one workgroup, up to CK iterations: 4 tiles per thread in
//                   registers, candidates visited by quarters, a
//                   wavefront each;
// then k_clean_tiles again.
//
// How many tiles can hold the peak is a matter of the PSF and the image: with
// the sidelobes of a short snapshot, or on a flat image, the slacks soon let in
// hundreds, all visited by one CU (100 points on 2048^2: 93 an iteration, 87
// us; a zero image: all, 6.7 ms).  So k_clean_minor stops before it visits more
// than a budget (visit_budget, below), and the rest is done by passes over the
// whole image, one launch per iteration (k_clean_pass: every block reduces the
// last pass's 512 block maxima, subtracts the component and leaves its own
// maximum): 12 us an iteration at 2048^2 FP32 whatever the image.  The host has
// to see that, so rcg_hogbom_run waits for the result; rcg_hogbom, which
// queues everything at once, is passes only.
//
// What bounds it: k_clean_minor the latency of an iteration on one CU (three
// barriers, one round of loads per visit), k_clean_tiles the reads of the PSF
// beyond the L2 (16 MB a component at 2048^2 FP32, 10 TB/s), k_clean_pass its
// launch and the image's and PSF's bytes.  Measured, FP32, an iteration on
// tiles and by a pass: dense uv coverage 10.0 and 12.7 us at 2048^2, 7.7 and
// 10.3 at 1024^2; 2000 points 16.9 and 12.3, 10.0 and 10.2; 100 points 87 and
// 12, 48 and 10.  Passes whose reductions shuffled value, sign and place took
// 16.9 us at 2048^2, 13 at 256^2 (6.7 now).  CK iterations between two rounds of
// k_clean_tiles: a tile seldom visited has up to CK components to catch up on,
// a round costs 10 us besides them; 12 and 24 are within 1% of 16, 32 takes
// 10.4, 64 11.4, 128 15.3 ms.  A visit's pixels four to a lane, loaded
// together: 13 us an iteration at CK = 128, against 18 us one to a lane.
#include <algorithm>

#include "rcg_internal.h"

namespace rcg {
namespace {

constexpr int CT = 1024;       // threads of the one-workgroup kernels
constexpr int CTILES = 4096;   // tiles of an image at most
constexpr int PER = CTILES / CT;
constexpr int CK = 16;         // iterations (components) between two rounds of k_clean_tiles
constexpr int CAND = 128;      // tiles visited at a time
constexpr int NP = 4;          // parts of a tile, a wavefront each
constexpr int MSIDE = 65;      // side of the table of PSF maxima at most
constexpr int PBLOCKS = 512;   // blocks of a pass over the whole image
constexpr int PB = 8;          // pixels of a thread whose loads are issued together

struct CleanState {
  long long pos;    // residual peak (row*pitch + col)
  long long ppos;   // PSF peak
  double val;       // signed residual peak value
  double pval;      // signed PSF peak value
  int done;
  int iters;
  int passes;       // too many tiles can hold the peak: passes from here on
};

// A tile's maximum: |value|, the signed value, its place in the tile (row-major).
struct TileMax {
  double a, v;
  int p, pad;
};

struct Comp {
  double a;    // amplitude times gain, as the image's type holds it
  int dr, dc;  // row and column of the PSF over pixel (0, 0)
};

// Block maxima of a pass: |value|, signed value, row-major place in the image.
struct Partials {
  double a[PBLOCKS], v[PBLOCKS];
  long long p[PBLOCKS];
};

struct Scratch {
  CleanState st;
  int nc;                    // pending components
  int prow, pcol;            // PSF peak
  Comp comp[CK];
  unsigned char applied[CTILES];  // of the pending, how many a tile has had
  TileMax psf[CTILES], res[CTILES];
  float m2[MSIDE * MSIDE];   // largest |psf| over tiles (i-1, i) x (j-1, j)
  Partials part[2];          // of the last pass and of the one before it
};

// Tile geometry: nb x nb tiles of 2^lb pixels a side.
struct Tiling {
  int siz, pitch, lb, nb;
};

Tiling tiling_of(int siz, int pitch)
{
  Tiling t{siz, pitch, 5, 0};
  while (true) {
    t.nb = (int)(((long long)siz + (1LL << t.lb) - 1) >> t.lb);
    if ((long long)t.nb * t.nb <= CTILES) return t;
    t.lb++;
  }
}

// Larger |value| first, then the lower place (a NaN is never larger).
template <class T>
__device__ __forceinline__ void take(T &a, T &v, long long &p, T a2, T v2, long long p2)
{
  if (a2 > a || (a2 == a && p2 < p)) {
    a = a2;
    v = v2;
    p = p2;
  }
}

// One DPP step of a maximum over lanes: x and the lane that `CTRL` names.
template <int CTRL, class T>
__device__ __forceinline__ T dpp_max(T x)
{
  if constexpr (sizeof(T) == 8) {
    const long long w = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp((int)w, (int)w, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(w >> 32), (int)(w >> 32), CTRL, 0xf, 0xf, false);
    return fmax(x, __longlong_as_double((long long)hi << 32 | (unsigned)lo));
  } else {
    const int w = __float_as_int(x);
    return fmaxf(x, __int_as_float(__builtin_amdgcn_update_dpp(w, w, CTRL, 0xf, 0xf, false)));
  }
}
__device__ __forceinline__ long long lane_word(long long w, int l)
{
  const unsigned lo = __builtin_amdgcn_readlane((int)w, l);
  const int hi = __builtin_amdgcn_readlane((int)(w >> 32), l);
  return (long long)hi << 32 | lo;
}
__device__ __forceinline__ double lane_value(double x, int l)
{
  return __longlong_as_double(lane_word(__double_as_longlong(x), l));
}
__device__ __forceinline__ float lane_value(float x, int l)
{
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}
// Maximum over the wavefront (row_shr 1, 2, 4, 8, row_bcast 15, 31: in the
// last lane) or, ROW, over each row of 16 lanes that hold the same values.
// (Shuffles of the value, its sign and its place through LDS took 4 us a
// workgroup; a few hundred cycles like this.)
template <bool ROW, class T>
__device__ __forceinline__ T lanes_max(T x)
{
  x = dpp_max<0x111>(x);
  x = dpp_max<0x112>(x);
  x = dpp_max<0x114>(x);
  x = dpp_max<0x118>(x);
  if (ROW) return lane_value(x, 15);
  x = dpp_max<0x142>(x);
  x = dpp_max<0x143>(x);
  return lane_value(x, 63);
}
// The same for the lowest of whole numbers (a lane without a source keeps its own).
template <int CTRL>
__device__ __forceinline__ long long dpp_min(long long w)
{
  const int lo = __builtin_amdgcn_update_dpp((int)w, (int)w, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(w >> 32), (int)(w >> 32), CTRL, 0xf, 0xf, false);
  const long long x = (long long)hi << 32 | (unsigned)lo;
  return x < w ? x : w;
}
template <bool ROW>
__device__ __forceinline__ long long lanes_min(long long w)
{
  w = dpp_min<0x111>(w);
  w = dpp_min<0x112>(w);
  w = dpp_min<0x114>(w);
  w = dpp_min<0x118>(w);
  if (ROW) return lane_word(w, 15);
  w = dpp_min<0x142>(w);
  w = dpp_min<0x143>(w);
  return lane_word(w, 63);
}
// The largest a (>= 0) of the lanes, the lowest place p on ties, and its v; a
// = -1 when there is none.  (On a flat image all lanes tie: one by one they
// took 3 us a reduction.)
template <bool ROW, class T>
__device__ __forceinline__ void lanes_best(T &a, T &v, long long &p)
{
  const T m = lanes_max<ROW>(a);
  unsigned long long eq = m >= 0 ? __ballot(a == m) : 0;
  long long bp = 0x7fffffffffffffffLL;
  T bv = 0;
  if (eq & (eq - 1)) {
    bp = lanes_min<ROW>(a == m ? p : bp);
    eq &= __ballot(p == bp);
  }
  if (eq) {
    const int l = __ffsll(eq) - 1;
    bp = lane_word(p, l);
    bv = lane_value(v, l);
  }
  a = m;
  v = bv;
  p = bp;
}

// Quarter q (by rows) of a tile, by one wavefront: components [k0, nc)
// subtracted from its pixels, the largest of them (every lane gets it).  A
// component lies over all of the part, over some of it, or not over it at
// all; lane l finds out for the l-th of 64.  Those over all of it are taken
// PC at a time: their loads are issued together, each from a scalar base (the
// component's) and a lane offset (the pixel's), so that a pixel and component
// cost one load and two operations.  (With the range tests of every pixel and
// component instead, a visit was bound by instruction issue on its one CU.)
template <int PC, class T>
__device__ __forceinline__ TileMax visit(T *__restrict__ img, const T *__restrict__ psf,
                                         const Tiling &g, int tile, int q, const Comp *comp, int k0,
                                         int nc)
{
#pragma clang fp contract(off)
  // four pixels of a row per lane, one load of the image's own alignment
  typedef T Quad __attribute__((ext_vector_type(4), aligned(sizeof(T))));
  const int lane = threadIdx.x & 63;
  const int B = 1 << g.lb, rows = B / NP;
  const int tr = tile / g.nb, tc = tile - tr * g.nb;
  const int r0 = tr * B + q * rows, c0 = tc * B;
  // the part's last row and column in the image
  const int r1 = min(r0 + rows, g.siz) - 1, c1 = min(c0 + B, g.siz) - 1;
  const bool wide = c0 + B <= g.siz;
  T ba = -1, bv = 0;
  int bp = 0x7fffffff;
  for (int i = 0; i < rows << g.lb && r0 < g.siz; i += 256) {
    const int p0 = i + lane * 4;
    const int r = r0 + (p0 >> g.lb), c = c0 + (p0 & (B - 1));
    // a lane past the edge works on the part's last pixels and drops them
    const long long row = (long long)min(r, r1) * g.pitch;
    auto load = [&](const T *src) {
      Quad x;
      if (wide) {
        x = *reinterpret_cast<const Quad *>(src + (row + c));
      } else {
#pragma unroll
        for (int u = 0; u < 4; u++) x[u] = src[row + min(c + u, c1)];
      }
      return x;
    };
    Quad x = load(img);
    for (int k = k0; k < nc; k += 64) {
      const Comp mine = comp[min(k + lane, nc - 1)];
      const T ma = (T)mine.a;
      const bool live = k + lane < nc;
      const bool some = live && r1 + mine.dr >= 0 && r0 + mine.dr < g.siz && c1 + mine.dc >= 0 &&
                        c0 + mine.dc < g.siz;
      const bool all = some && r0 + mine.dr >= 0 && r1 + mine.dr < g.siz && c0 + mine.dc >= 0 &&
                       c1 + mine.dc < g.siz;
      unsigned long long todo = __ballot(some);
      const unsigned long long whole = __ballot(all);
      while (todo) {
        int l[PC];
        unsigned long long left = todo, these = 0;
#pragma unroll
        for (int j = 0; j < PC; j++) {
          l[j] = left ? __ffsll(left) - 1 : -1;
          if (left) these |= left & -left;
          left &= left - 1;
        }
        if ((these & ~whole) == 0) {
          Quad y[PC];
#pragma unroll
          for (int j = 0; j < PC; j++) {
            const int m = l[j] < 0 ? l[0] : l[j];
            y[j] = load(psf + ((long long)__builtin_amdgcn_readlane(mine.dr, m) * g.pitch +
                               __builtin_amdgcn_readlane(mine.dc, m)));
          }
#pragma unroll
          for (int j = 0; j < PC; j++) {
            if (l[j] < 0) break;
            const T a = lane_value(ma, l[j]);
#pragma unroll
            for (int u = 0; u < 4; u++) x[u] -= a * y[j][u];
          }
          todo = left;
        } else {
          // one component, pixel by pixel
          const int dr = __builtin_amdgcn_readlane(mine.dr, l[0]);
          const int dc = __builtin_amdgcn_readlane(mine.dc, l[0]);
          const T a = lane_value(ma, l[0]);
#pragma unroll
          for (int u = 0; u < 4; u++) {
            const int sr = r + dr, sc = c + u + dc;
            if (r <= r1 && c + u <= c1 && sr >= 0 && sr < g.siz && sc >= 0 && sc < g.siz)
              x[u] -= a * psf[(long long)sr * g.pitch + sc];
          }
          todo &= todo - 1;
        }
      }
    }
    if (r <= r1) {
      if (k0 < nc) {
        if (wide) {
          *reinterpret_cast<Quad *>(img + (row + c)) = x;
        } else {
#pragma unroll
          for (int u = 0; u < 4; u++)
            if (c + u <= c1) img[row + c + u] = x[u];
        }
      }
#pragma unroll
      for (int u = 0; u < 4; u++)
        if (c + u <= c1 && fabs(x[u]) > ba) {
          ba = fabs(x[u]);
          bv = x[u];
          bp = (q * rows << g.lb) + p0 + u;
        }
    }
  }
  long long p = bp;
  lanes_best<false>(ba, bv, p);
  return TileMax{(double)ba, (double)bv, ba >= 0 ? (int)p : 0x7fffffff, 0};
}

// One workgroup of 4 wavefronts per tile.  sc->nc pending components (which
// == 0: the residual) or none (1: the PSF, read only).
template <class T>
__global__ void __launch_bounds__(256)
k_clean_tiles(T *__restrict__ img, const T *__restrict__ psf, Tiling g, Scratch *__restrict__ sc,
              int which, int pending)
{
  __shared__ Comp comp[CK];
  __shared__ TileMax best[4];
  const int nc = pending ? sc->nc : 0;
  if (pending && nc == 0) return;  // stopped: nothing has changed
  for (int k = threadIdx.x; k < nc; k += 256) comp[k] = sc->comp[k];
  __syncthreads();
  const int tile = blockIdx.x, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int k0 = nc ? sc->applied[tile] : 0;
  const TileMax m = visit<8>(img, psf, g, tile, wave, comp, k0, nc);
  if ((threadIdx.x & 63) == 0) best[wave] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double a = best[0].a, v = best[0].v;
    long long p = best[0].p;
    for (int w = 1; w < 4; w++) take(a, v, p, best[w].a, best[w].v, (long long)best[w].p);
    (which ? sc->psf : sc->res)[tile] = TileMax{a, v, (int)p, 0};
  }
}

// The best of a workgroup's (a, v, p), in every thread.
template <class T>
struct BlockBest {
  T a[CT / 64], v[CT / 64];
  long long p[CT / 64];
};
template <class T>
__device__ __forceinline__ void block_take(T &a, T &v, long long &p, BlockBest<T> &sh)
{
  lanes_best<false>(a, v, p);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    sh.a[wave] = a;
    sh.v[wave] = v;
    sh.p[wave] = p;
  }
  __syncthreads();
  const int w = lane & ((blockDim.x >> 6) - 1);  // 8 or 16 wavefronts
  a = sh.a[w];
  v = sh.v[w];
  p = sh.p[w];
  lanes_best<true>(a, v, p);
}

constexpr long long NOWHERE = 0x7fffffffffffffffLL;

// Row-major place in the image of place p of a tile.
__device__ __forceinline__ long long image_place(const Tiling &g, int tile, int p)
{
  const int tr = tile / g.nb, tc = tile - tr * g.nb;
  return (long long)((tr << g.lb) + (p >> g.lb)) * g.siz + (tc << g.lb) + (p & ((1 << g.lb) - 1));
}

// The PSF's peak and the table of its maxima; the state of a new cycle.
__global__ void __launch_bounds__(CT)
k_clean_prep(Tiling g, Scratch *__restrict__ sc)
{
  __shared__ BlockBest<double> sh;
  const int nt = g.nb * g.nb;
  double a = -1.0, v = 0.0;
  long long p = NOWHERE;
  for (int t = threadIdx.x; t < nt; t += CT) {
    const TileMax m = sc->psf[t];
    if (m.a >= 0.0) take(a, v, p, m.a, m.v, image_place(g, t, m.p));
  }
  block_take(a, v, p, sh);
  if (threadIdx.x == 0) {
    const bool any = p != NOWHERE;
    const int pr = any ? (int)(p / g.siz) : 0, pc = any ? (int)(p % g.siz) : 0;
    sc->st = CleanState{0, (long long)pr * g.pitch + pc, 0.0, any ? v : 0.0, 0, 0, 0};
    sc->prow = pr;
    sc->pcol = pc;
    sc->nc = 0;
  }
  const int side = g.nb + 1;
  for (int k = threadIdx.x; k < side * side; k += CT) {
    const int i = k / side, j = k - i * side;
    float m = 0.f;
    for (int di = -1; di <= 0; di++)
      for (int dj = -1; dj <= 0; dj++) {
        const int r = i + di, c = j + dj;
        // rounded up
        if (r >= 0 && r < g.nb && c >= 0 && c < g.nb)
          m = fmaxf(m, (float)sc->psf[r * g.nb + c].a * 1.000001f);
      }
    sc->m2[k] = m;
  }
}

// Up to `iters` (<= CK) iterations.  Three barriers an iteration: after the
// candidates' list, the visits, and the new component.  The run ends, and with
// it the work on tiles, before it visits more than `budget` of them.  The
// state goes to the host's copy too.
template <class T>
__global__ void __launch_bounds__(CT)
k_clean_minor(T *__restrict__ img, const T *__restrict__ psf, T *__restrict__ model, Tiling g,
              Scratch *__restrict__ sc, double gain, double threshold, int iters, int budget,
              CleanState *__restrict__ seen)
{
#pragma clang fp contract(off)
  __shared__ float m2[MSIDE * MSIDE];
  __shared__ Comp comp[CK];
  __shared__ unsigned char applied[CTILES];
  __shared__ int cand[CAND];
  __shared__ TileMax found[CAND * NP];
  __shared__ float sh_lb[CT / 64];
  __shared__ int n_cand[2];  // the round's count; the other is cleared for the next
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (sc->st.done || sc->st.passes) {
    if (tid == 0) sc->nc = 0;
    return;
  }
  const int nt = g.nb * g.nb, side = g.nb + 1, prow = sc->prow, pcol = sc->pcol;
  const double pval = sc->st.pval;
  const int iter0 = sc->st.iters;
  for (int k = tid; k < side * side; k += CT) m2[k] = sc->m2[k];
  for (int t = tid; t < CTILES; t += CT) applied[t] = 0;
  // Slacks in float, each step rounded up by more than the float operations
  // and the rounding of the pixels' own subtractions can lose; above 0, so
  // that a peak is always found by a visit.
  constexpr float UP = 1.000001f, TINY = 5e-7f, LEAST = 1e-37f;
  float e[PER], s[PER];
  int at[PER], slot[PER];  // tile row << 16 | column (-1: no tile)
#pragma unroll
  for (int j = 0; j < PER; j++) {
    const int t = tid + j * CT;
    at[j] = t < nt ? (t / g.nb) << 16 | t % g.nb : -1;
    e[j] = t < nt ? (float)sc->res[t].a * UP : -1.f;
    s[j] = LEAST;
  }
  if (tid < 2) n_cand[tid] = 0;
  int nc = 0, done = 0, passes = 0, flip = 0, visits = 0;
  long long pos = 0;
  double val = 0.0;
  // A bound from below on the image's maximum: the largest e - s.
  auto offer_lb = [&]() {
    float lb = -1.f;
#pragma unroll
    for (int j = 0; j < PER; j++) lb = fmaxf(lb, e[j] * (1.f - 4.f * TINY) - s[j]);
    lb = lanes_max<false>(lb);
    if (lane == 0) sh_lb[wave] = lb;
  };
  offer_lb();
  __syncthreads();
  while (nc < iters) {
    float lb = lanes_max<true>(sh_lb[lane & 15]);
    T ba = -1, bv = 0;
    long long bp = NOWHERE;
    while (true) {
      // tiles that can reach lb (a NaN slack: looked at)
#pragma unroll
      for (int j = 0; j < PER; j++) {
        slot[j] = -1;
        if (at[j] >= 0 && s[j] != 0.f && !(e[j] + s[j] < lb)) {
          const int k = atomicAdd(&n_cand[flip], 1);
          if (k < CAND) {
            slot[j] = k;
            cand[k] = tid + j * CT;
          }
        }
      }
      __syncthreads();
      const int all = __builtin_amdgcn_readfirstlane(n_cand[flip]), n = min(all, CAND);
      visits += all;
      if (visits > budget) {
        passes = 1;
        break;
      }
      if (tid == 0) n_cand[flip ^ 1] = 0;
      flip ^= 1;
      for (int job = wave; job < n * NP; job += CT / 64) {
        const int t = __builtin_amdgcn_readfirstlane(cand[job / NP]);
        const TileMax m = visit<sizeof(T) == 4 ? 8 : 4>(
            img, psf, g, t, job % NP, comp, __builtin_amdgcn_readfirstlane((int)applied[t]), nc);
        if (lane == 0) found[job] = m;
      }
      __syncthreads();
      // every wavefront: the best of the visits
      for (int k = 0; k < n * NP; k += 64) {
        T a = -1, v = 0;
        long long p = NOWHERE;
        if (k + lane < n * NP) {
          const TileMax m = found[k + lane];
          if (m.a >= 0.0) {
            a = (T)m.a;
            v = (T)m.v;
            p = image_place(g, cand[(k + lane) / NP], m.p);
          }
        }
        lanes_best<false>(a, v, p);
        take(ba, bv, bp, a, v, p);
      }
#pragma unroll
      for (int j = 0; j < PER; j++)
        if (slot[j] >= 0) {
          const TileMax *f = found + slot[j] * NP;
          e[j] = (float)fmax(fmax(f[0].a, f[1].a), fmax(f[2].a, f[3].a)) * UP;
          s[j] = 0.f;
          applied[tid + j * CT] = (unsigned char)nc;
        }
      // Tiles not visited lie below lb: unless the list was full, or the best
      // below lb (NaNs took pixels away), nothing can exceed the best found.
      if (all <= CAND && ba >= lb) break;
      if (all == 0) break;
      lb = (float)ba * (1.f - 4.f * TINY);
      __syncthreads();  // the list and the visits have been read
    }
    if (passes) break;
    if (bp == NOWHERE || fabs((double)bv) < threshold || pval == 0.0) {
      done = 1;
      pos = bp == NOWHERE ? 0 : bp / g.siz * g.pitch + bp % g.siz;
      val = bv;
      break;
    }
    const int r = (int)(bp / g.siz), c = (int)(bp - (long long)r * g.siz);
    const double w = gain * (double)bv / pval;
    pos = (long long)r * g.pitch + c;
    val = bv;
    if (tid == 0) {
      comp[nc] = Comp{(double)(T)w, prow - r, pcol - c};
      model[pos] += (T)w;
    }
    nc++;
    const float aw = fabsf((float)w) * UP;
#pragma unroll
    for (int j = 0; j < PER; j++)
      if (at[j] >= 0) {
        // the tile's first row and column in the PSF, and the PSF tiles there
        const int i = ((((at[j] >> 16) << g.lb) + prow - r) >> g.lb) + 1;
        const int k = ((((at[j] & 0xffff) << g.lb) + pcol - c) >> g.lb) + 1;
        const float m = i >= 0 && i < side && k >= 0 && k < side ? m2[i * side + k] : 0.f;
        s[j] = (s[j] + aw * m + TINY * e[j] + LEAST) * UP;
      }
    offer_lb();
    __syncthreads();
  }
  for (int k = tid; k < nc; k += CT) sc->comp[k] = comp[k];
  for (int t = tid; t < nt; t += CT) sc->applied[t] = applied[t];
  if (tid == 0) {
    sc->nc = nc;
    sc->st.pos = pos;
    sc->st.val = val;
    sc->st.done = done;
    sc->st.iters = iter0 + nc;
    sc->st.passes = passes;
    *seen = sc->st;
  }
}

// Pass `it` over the whole image.  it >= 1: reduce the last pass's block maxima
// (pin) to the peak of iteration base + it - 1; stop below the threshold; else
// block 0 adds gain * peak / psf peak to the model, and every block subtracts
// that times the PSF shifted onto the peak.  find: leave this block's maximum
// of the (updated) image in pout.  it = 0: find only.  The kernel boundary
// orders the passes: no block waits for another.
template <class T>
__global__ void __launch_bounds__(CT)
k_clean_pass(T *__restrict__ img, const T *__restrict__ psf, T *__restrict__ model, Tiling g,
             Scratch *__restrict__ sc, double gain, double threshold, int base, int it, int find,
             const Partials *__restrict__ pin, Partials *__restrict__ pout)
{
#pragma clang fp contract(off)
  __shared__ BlockBest<double> sh_peak, sh_out;
  CleanState *st = &sc->st;
  if (st->done) return;
  const int siz = g.siz, pitch = g.pitch;
  long long dr = 0, dc = 0;
  T a = 0;
  const bool subtract = it > 0;
  if (subtract) {
    double pa = -1.0, pv = 0.0;
    long long pp = NOWHERE;
    for (int k = threadIdx.x; k < PBLOCKS; k += blockDim.x) take(pa, pv, pp, pin->a[k], pin->v[k], pin->p[k]);
    block_take(pa, pv, pp, sh_peak);
    const long long r = pp == NOWHERE ? 0 : pp / siz, c = pp == NOWHERE ? 0 : pp % siz;
    const long long pos = r * pitch + c;
    const double pval = st->pval;
    if (pp == NOWHERE || fabs(pv) < threshold || pval == 0.0) {
      if (blockIdx.x == 0 && threadIdx.x == 0) {
        st->pos = pos;
        st->val = pv;
        st->done = 1;
      }
      return;
    }
    const double w = gain * pv / pval;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      st->pos = pos;
      st->val = pv;
      st->iters = base + it;
      model[pos] += (T)w;
    }
    dr = sc->prow - r;
    dc = sc->pcol - c;
    a = (T)w;
  }
  // A thread's pixels are rows blockIdx.x + k * gridDim.x, columns
  // threadIdx.x + j * blockDim.x, taken PB at a time in (k, j) order.  Every
  // load of a batch (image, and PSF where the shifted PSF covers the pixel)
  // is issued before any is used, so a batch costs one memory latency: at
  // 2048^2 a thread's 8 pixels are one batch.  The pixels of a batch are
  // distinct and img and psf do not alias, so the stores may follow all the
  // loads.  The thread's running maximum: its pixels come in increasing
  // order, so a strict > keeps the first on ties, as take() does.
  T ba = -1, bv = 0;
  int br = -1, bc = 0;
  const int tx = threadIdx.x, bx = blockIdx.x, nb = gridDim.x, nt = blockDim.x;
  const int nj = tx < siz ? (siz - 1 - tx) / nt + 1 : 0;
  const int nk = bx < siz ? (siz - 1 - bx) / nb + 1 : 0;
  const int ne = nj * nk;
  int k = 0, j = 0;
  for (int e0 = 0; e0 < ne; e0 += PB) {
    T x[PB], p[PB];
    int rr[PB], cc[PB];
    bool sb[PB];
#pragma unroll
    for (int u = 0; u < PB; u++) {
      const int r = bx + k * nb, c = tx + j * nt;
      const bool ok = e0 + u < ne;
      const long long sr = r + dr, sc = c + dc;
      rr[u] = r;
      cc[u] = c;
      sb[u] = ok && subtract && sr >= 0 && sr < siz && sc >= 0 && sc < siz;
      x[u] = ok ? img[(long long)r * pitch + c] : T(0);
      p[u] = sb[u] ? psf[sr * pitch + sc] : T(0);
      if (++j == nj) {
        j = 0;
        k++;
      }
    }
#pragma unroll
    for (int u = 0; u < PB; u++) {
      if (sb[u]) {
        x[u] -= a * p[u];
        img[(long long)rr[u] * pitch + cc[u]] = x[u];
      }
      if (find && e0 + u < ne && fabs(x[u]) > ba) {
        ba = fabs(x[u]);
        bv = x[u];
        br = rr[u];
        bc = cc[u];
      }
    }
  }
  if (!find) return;
  double ma = br >= 0 ? (double)ba : -1.0, mv = (double)bv;
  long long mp = br >= 0 ? (long long)br * siz + bc : NOWHERE;
  block_take(ma, mv, mp, sh_out);
  if (tx == 0) {
    pout->a[blockIdx.x] = ma;
    pout->v[blockIdx.x] = mv;
    pout->p[blockIdx.x] = mp;
  }
}

template <class T>
__global__ void k_zero(T *__restrict__ p, long long n)
{
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    p[i] = 0;
}

// The model cleared, the PSF's peak and maxima, the state.
template <class T>
void begin(T *model, const T *psf, const Tiling &g, Scratch *sc, hipStream_t st)
{
  hipLaunchKernelGGL(k_zero<T>, dim3(1024), dim3(256), 0, st, model, (long long)g.siz * g.pitch);
  hipLaunchKernelGGL(k_clean_tiles<T>, dim3(g.nb * g.nb), dim3(256), 0, st, const_cast<T *>(psf),
                     psf, g, sc, 1, 0);
  hipLaunchKernelGGL(k_clean_prep, dim3(1), dim3(CT), 0, st, g, sc);
}

// Iterations [base, niters), one launch each after the first that finds the
// peak only.
template <class T>
void passes(T *model, T *res, const T *psf, const Tiling &g, unsigned base, unsigned niters,
            double gain, double threshold, Scratch *sc, hipStream_t st)
{
  // FP64 passes need more registers per thread: 512 threads keep two blocks
  // per CU resident
  const int nt = sizeof(T) == 8 ? 512 : CT;
  Partials *pp = sc->part;
  const unsigned n = niters - base;
  for (unsigned it = 0; n && it <= n; it++)
    hipLaunchKernelGGL(k_clean_pass<T>, dim3(PBLOCKS), dim3(nt), 0, st, res, psf, model, g, sc, gain,
                       threshold, (int)base, (int)it, it < n ? 1 : 0, pp + ((it + 1) & 1),
                       pp + (it & 1));
}

template <class T>
rcg_status hogbom(T *model, T *res, const T *psf, int siz, int pitch, unsigned niters,
                  double gain, double threshold, Scratch *sc, hipStream_t st)
{
  const Tiling g = tiling_of(siz, pitch);
  begin(model, psf, g, sc, st);
  passes(model, res, psf, g, 0, niters, gain, threshold, sc, st);
  RCG_HIP_TRY(hipGetLastError());
  return RCG_OK;
}

// Tiles a run of CK iterations may visit before passes are the faster way (0:
// from the start).  A pass takes 6.5 us and 0.37 us a MB of the image; an
// iteration on tiles about half of that a MB, 5 to 13 us by the tiles' side,
// and for each visit 0.85, 3 and 14 us with tiles of 32, 64 and 128 pixels.
// They break even at a number of visits an iteration that grows as the image's
// bytes over a tile's pixels, as the number of tiles times a pixel's bytes:
// measured 3.8 and 9.5 at 4096^2 (FP32, FP64; 4.7 and 9.4 by the rule), 2.7 and
// 5.3 at 3000^2 (2.6, 5.2), 5 and 11 at 8192^2 (4.7, 9.4), 9.5 at 2048^2 FP64.
// Tiles of 32 pixels, where both sides are bound by latency, break even at 4.2
// to 6.4 from 400^2 to 2048^2 (5).  Four tiles are always faster than passes
// (5.6 against 6.9 us at 64^2), from there to 400^2 a pass is (6.8 against 8.7
// us at 256^2), and below two visits an iteration nothing is left.
int visit_budget(const Tiling &g, size_t elem)
{
  if (g.nb <= 2) return 1 << 30;
  if (g.siz < 400) return 0;
  const int rule = (int)(g.nb * g.nb * elem / 218);
  if (g.lb == 5) return std::max(rule, 5 * CK);
  return rule < 2 * CK ? 0 : rule;
}

// What the host keeps of a running call: given back when the stream is done.
struct Watch {
  hipStream_t st;
  CleanState *seen = nullptr;  // pinned host memory
  hipEvent_t ev[2] = {};
  ~Watch()
  {
    (void)hipStreamSynchronize(st);
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
    if (seen) pool_pin_put(seen);
  }
};

// On tiles while that pays, then by passes.  Rounds are queued in groups, each
// up to twice as large as the last, and before the next group the host looks
// at where the group before this one has got: the device never waits for it.
template <class T>
rcg_status hogbom_run(T *model, T *res, const T *psf, int siz, int pitch, unsigned niters,
                      double gain, double threshold, Scratch *sc, unsigned *iters, hipStream_t st)
{
  const Tiling g = tiling_of(siz, pitch);
  const int nt = g.nb * g.nb, budget = visit_budget(g, sizeof(T));
  Watch w{st};
  RCG_HIP_TRY(pool_pin(reinterpret_cast<void **>(&w.seen)));
  for (hipEvent_t &e : w.ev) RCG_HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  volatile CleanState *seen = w.seen;
  seen->done = seen->passes = 0;
  begin(model, psf, g, sc, st);
  if (!budget) {
    passes(model, res, psf, g, 0, niters, gain, threshold, sc, st);
  } else if (niters > 0) {
    hipLaunchKernelGGL(k_clean_tiles<T>, dim3(nt), dim3(256), 0, st, res, psf, g, sc, 0, 0);
  }
  unsigned queued = 0, group = 1;
  for (int k = 0; budget && queued < niters; k++) {
    for (unsigned r = 0; r < group && queued < niters; r++) {
      const unsigned n = std::min(niters - queued, (unsigned)CK);
      hipLaunchKernelGGL(k_clean_minor<T>, dim3(1), dim3(CT), 0, st, res, psf, model, g, sc, gain,
                         threshold, (int)n, budget, w.seen);
      hipLaunchKernelGGL(k_clean_tiles<T>, dim3(nt), dim3(256), 0, st, res, psf, g, sc, 0, 1);
      queued += n;
    }
    RCG_HIP_TRY(hipGetLastError());
    RCG_HIP_TRY(hipEventRecord(w.ev[k & 1], st));
    if (k > 0) {
      RCG_HIP_TRY(hipEventSynchronize(w.ev[(k - 1) & 1]));
      if (seen->done || seen->passes) break;
    }
    group = std::min(2 * group, 32u);
  }
  auto state = [&]() {
    hipError_t e = hipMemcpyAsync(w.seen, &sc->st, sizeof(CleanState), hipMemcpyDeviceToHost, st);
    return e == hipSuccess ? hipStreamSynchronize(st) : e;
  };
  RCG_HIP_TRY(state());
  if (seen->passes && !seen->done) {
    passes(model, res, psf, g, (unsigned)seen->iters, niters, gain, threshold, sc, st);
    RCG_HIP_TRY(hipGetLastError());
    RCG_HIP_TRY(state());
  }
  *iters = (unsigned)seen->iters;
  return RCG_OK;
}

rcg_status check_hogbom(const void *model, const void *res, const void *psf, int siz, int pitch,
                        const void *scratch)
{
  if (!model || !res || !psf || !scratch || siz <= 0 || pitch < siz ||
      (long long)siz * siz > 0x7fffffffffffLL) {
    set_error(RCG_ERR_ARG, "rcg_hogbom: bad arguments");
    return RCG_ERR_ARG;
  }
  return RCG_OK;
}

}  // namespace
}  // namespace rcg

using namespace rcg;

extern "C" size_t rcg_hogbom_scratch_bytes(void)
{
  return sizeof(Scratch);
}

extern "C" rcg_status rcg_hogbom(void *model, void *res, const void *psf, int f64, int siz,
                                 int pitch, unsigned niters, double gain, double threshold,
                                 void *scratch, void *stream)
{
  clear_error();
  const rcg_status s = check_hogbom(model, res, psf, siz, pitch, scratch);
  if (s != RCG_OK) return s;
  hipStream_t st = (hipStream_t)stream;
  Scratch *sc = static_cast<Scratch *>(scratch);
  if (f64)
    return hogbom<double>(static_cast<double *>(model), static_cast<double *>(res),
                          static_cast<const double *>(psf), siz, pitch, niters, gain,
                          threshold, sc, st);
  return hogbom<float>(static_cast<float *>(model), static_cast<float *>(res),
                       static_cast<const float *>(psf), siz, pitch, niters, gain, threshold, sc,
                       st);
}

extern "C" rcg_status rcg_hogbom_run(void *model, void *res, const void *psf, int f64, int siz,
                                     int pitch, unsigned niters, double gain, double threshold,
                                     void *scratch, unsigned *iters, void *stream)
{
  clear_error();
  const rcg_status s = check_hogbom(model, res, psf, siz, pitch, scratch);
  if (s != RCG_OK) return s;
  unsigned n = 0;
  if (!iters) iters = &n;
  hipStream_t st = (hipStream_t)stream;
  Scratch *sc = static_cast<Scratch *>(scratch);
  if (f64)
    return hogbom_run<double>(static_cast<double *>(model), static_cast<double *>(res),
                              static_cast<const double *>(psf), siz, pitch, niters, gain,
                              threshold, sc, iters, st);
  return hogbom_run<float>(static_cast<float *>(model), static_cast<float *>(res),
                           static_cast<const float *>(psf), siz, pitch, niters, gain, threshold,
                           sc, iters, st);
}

// Iterations the last rcg_hogbom on this scratch performed (synchronises).
extern "C" rcg_status rcg_hogbom_iterations(const void *scratch, unsigned *iters, void *stream)
{
  clear_error();
  if (!scratch || !iters) {
    set_error(RCG_ERR_ARG, "rcg_hogbom_iterations: null argument");
    return RCG_ERR_ARG;
  }
  CleanState cs;
  RCG_HIP_TRY(hipMemcpyAsync(&cs, scratch, sizeof(cs), hipMemcpyDeviceToHost,
                             (hipStream_t)stream));
  RCG_HIP_TRY(hipStreamSynchronize((hipStream_t)stream));
  *iters = (unsigned)cs.iters;
  return RCG_OK;
}

extern "C" void deconvolve(double *mod_p, double *res_p, double *psf_p, int siz, int pitch,
                           unsigned int niters, double gain, double threshold)
{
  clear_error();
  if (!mod_p || !res_p || !psf_p || siz <= 0 || pitch < siz) {
    set_error(RCG_ERR_ARG, "deconvolve: bad arguments");
    return;
  }
  const size_t bytes = (size_t)siz * pitch * sizeof(double);
  hipStream_t st = nullptr;
  void *dm = nullptr, *dr = nullptr, *dp = nullptr, *ds = nullptr;
  if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess ||
      dev_malloc(&dm, bytes) != hipSuccess || dev_malloc(&dr, bytes) != hipSuccess ||
      dev_malloc(&dp, bytes) != hipSuccess ||
      dev_malloc(&ds, rcg_hogbom_scratch_bytes()) != hipSuccess) {
    set_error(RCG_ERR_NOMEM, "deconvolve: device buffers");
  } else if (hipMemcpyAsync(dr, res_p, bytes, hipMemcpyHostToDevice, st) != hipSuccess ||
             hipMemcpyAsync(dp, psf_p, bytes, hipMemcpyHostToDevice, st) != hipSuccess) {
    set_error(RCG_ERR_HIP, "deconvolve: copy in");
  } else if (rcg_hogbom_run(dm, dr, dp, 1, siz, pitch, niters, gain, threshold, ds, nullptr, st) ==
             RCG_OK) {
    if (hipMemcpyAsync(mod_p, dm, bytes, hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipMemcpyAsync(res_p, dr, bytes, hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
      set_error(RCG_ERR_HIP, "deconvolve: copy out");
  }
  if (st) (void)hipStreamSynchronize(st);
  void *bufs[] = {dm, dr, dp, ds};
  for (void *b : bufs)
    if (b) (void)hipFree(b);
  if (st) (void)hipStreamDestroy(st);
}
