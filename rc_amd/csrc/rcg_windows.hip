// rcg_windows.hip -- FP32 degridding of whole windows.
//
// Same sums as the reference's degridder (MS4/kernel/cpu/scatter_grid/
// scatter_gridder_w_dependent_dyn_1p.cpp:146-176, :171), one visibility per
// point: v = sum over the S x S window of grid * tap.  A workgroup takes a
// work item of a tile and degrids the points whose window starts in that
// tile (the records of tile slot 0), each whole: the tile and the
// max_support - 1 cells after it in both directions are staged in LDS, which
// all its wavefronts read.
//
// A wavefront takes 8 points at a time, 8 lanes each.  A point's lanes walk
// its window two columns per step: column pairs q = sub, sub + 8, ... in row
// order (CP = ceil(S / 2) pairs a row), one 16-byte tap load and one pair of
// LDS cells per lane and step.  The points of an item are sorted by support
// first (a counting sort in LDS), so the eight of a wavefront take nearly
// the same number of steps, the longest first.
//
// What bounds it: the vector-memory path moves about 32 to 50 bytes a cycle
// per CU and takes 8 cycles for any load instruction, so lanes must be full
// and loads wide.  A window cut at tile edges (k_degrid_tiles) fills 40 of 64
// lanes with 8 bytes each, and leaves per-tile partial sums to store and add.
// Measured on the 4096^2 w-projection workload (9,987,840 points, 3.2e9 taps):
// 1.32 ms, 19 TB/s of taps, against 2.35 + 0.08 ms for k_degrid_tiles and its
// sums; 16 snapshots of 2048^2 (6.3 M points): 0.87 against 1.65 ms.  With
// FP32 sums (1.26 and 0.82 ms) 0.85 of the former's were the steps, bound by
// instruction issue and the two workgroups per CU more than by the loads; the
// rest was the sorts and staging of an item.  Variants on the former workload:
// 16 lanes a point 5% slower, 32 lanes 24% (small windows leave them idle); U
// = 2 4% slower, 3 equal there and 5% slower on the latter; 4 wavefronts per
// workgroup 35% slower (32% on the latter); blocks that all lanes need without
// the range mask 5% slower; the region staged for the plan's largest support
// rather than the batch's 12% slower (23% on the latter); supports from the
// points' pregrid records rather than in the pair records, and staging after
// the sort, 7% slower.
#include <algorithm>

#include "rcg_internal.h"
#include "rcg_tiled.h"
#include "rcg_tiledev.h"

namespace rcg {
namespace {

constexpr int WIN_SCAN = 1024;     // records looked at together
constexpr int WIN_BUCKETS = 128;   // supports below this
constexpr int WIN_LDS = 80 * 1024; // two workgroups per CU
constexpr int U = 4;               // steps whose loads are issued together
constexpr int G = 8;               // lanes per point
constexpr int PW = 64 / G;         // points a wavefront takes at a time
// Points a full item holds (chunk over the tiles that a window meets) from
// which whole windows are taken: with fewer, most of the 64 points that a
// workgroup's wavefronts walk at a time are missing, and the region is staged
// for little.  400,000 points on 2048^2, tile 32, pairs against windows: 31 x 31
// windows with 17, 34, 51 points an item 330 / 555, 307 / 333, 305 / 266 us, 63
// x 63 with 15, 30, 59 902 / 1815, 891 / 1003, 912 / 678; 60,000 on 1024^2 with
// 17, 26 and 7, 30, 45: 98 / 95, 93 / 70 and 189 / 512, 183 / 192, 195 / 160.
constexpr int ITEM_POINTS = 30;
// Points of a tile's item up to which each takes a wavefront and reads the grid
// where it lies.  Uniform points on 4096^2, 16 x 16 and 63 x 63 windows, 0.3
// points a tile: 89 -> 40 and 456 -> 124 us; 3.7: 187 -> 106 and 1017 -> 450.
// With up to 4 alike, but 670 us for the last; with up to 16, tiles that hold
// so many lose (5000 points of 48 x 48 on 512^2, 20 a tile: 22 -> 38 us).
constexpr int FEW = 6;

// Side of the staged region and its row stride (odd, so that rows start in
// different banks).
__host__ __device__ inline int win_side(int T, int max_support) { return T + max_support - 1; }
__host__ __device__ inline int win_stride(int side) { return side | 1; }

// LDS of a workgroup that sorts up to `cap` points at a time, and the cap:
// all records of a scan when that leaves room for two workgroups per CU.
size_t win_lds(int T, int max_support, int cap)
{
  const int side = win_side(T, max_support);
  return ((size_t)side * win_stride(side) + 3) * sizeof(float2) + 16 + cap * sizeof(int4) +
         (WIN_BUCKETS + 4) * sizeof(int);
}
int win_cap(int T, int max_support)
{
  return win_lds(T, max_support, WIN_SCAN) <= WIN_LDS ? WIN_SCAN : WIN_SCAN / 2;
}
size_t win_lds(int T, int max_support)
{
  return win_lds(T, max_support, win_cap(T, max_support));
}

struct Steps {
  float2 a[U], b[U];  // taps of the pair's two columns
  int la[U];          // LDS byte address of its first cell (odd windows: bit 0 set in a row's
                      // last pair, whose second column lies outside)
};

// Where a lane is in its window.  pos holds the pair's index in its row
// (from bit POS_BITS) above the LDS byte offset of its first cell, so that one
// register is stepped and compared for both.
constexpr int POS_BITS = 20;
struct Walk {
  int tap, pos;           // byte offset of the current pair's first tap; see above
  int wrap;               // pos at and above which the next pair lies past the row's end
  int tstep, pstep;       // steps within a row
  int twrap, pwrap;       // steps past its end
  int half;               // pos from which a pair's second column lies outside (odd windows)
  int k, n;               // step and steps of this lane
};

// The next U steps; past its last a lane reads zeros.  The second half of an
// odd row's last load lies past the row, and of the table's very last row past
// the buffer's end: each dword is checked against the end by itself, so that
// the tap in the first half is read (observed for loads 1 to 4 dwords before
// the end; the last tap of a table is tested).
template <bool ODD>
__device__ __forceinline__ void win_load(Steps &s, Walk &w, int dummy, __amdgpu_buffer_rsrc_t rsrc)
{
#pragma unroll
  for (int u = 0; u < U; u++) {
    const bool act = w.k + u < w.n;
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, act ? (unsigned)w.tap : TAP_OOB, 0, 0);
    s.a[u] = make_float2(__int_as_float(v[0]), __int_as_float(v[1]));
    s.b[u] = make_float2(__int_as_float(v[2]), __int_as_float(v[3]));
    int la = w.pos & ((1 << POS_BITS) - 1);
    if (ODD) la |= w.pos >= w.half ? 1 : 0;
    s.la[u] = act ? la : dummy;
    const bool wrap = w.pos >= w.wrap;
    w.tap += wrap ? w.twrap : w.tstep;
    w.pos += wrap ? w.pwrap : w.pstep;
  }
  w.k += U;
}

// P = sum gx tx, Q = sum gy ty, R = sum gx ty, V = sum gy tx: the 2 U products
// of a call in FP32, the calls' sums and the lanes' in FP64.  In FP32 a lane's
// chain over the window would be S^2 / 8 long, eight times that of a wavefront
// per window: relative L2 error of the 4096^2 workload's visibilities, six sets
// of points, 0.67-2.9e-7 with FP32 sums per call, 0.68-2.2e-7 a wavefront per
// window, 0.37-1.8e-7 this way, for 1.26 -> 1.32 ms.
struct Acc {
  double P, Q, R, V;
};
template <bool ODD>
__device__ __forceinline__ void win_add(const Steps &s, const char *reg, Acc &acc)
{
  float2 g[U], h[U];
#pragma unroll
  for (int u = 0; u < U; u++) {
    const float2 *c = reinterpret_cast<const float2 *>(reg + (ODD ? s.la[u] & ~1 : s.la[u]));
    g[u] = c[0];
    h[u] = c[1];
  }
  float P = 0.f, Q = 0.f, R = 0.f, V = 0.f;
#pragma unroll
  for (int u = 0; u < U; u++) {
    float2 b = s.b[u], c = h[u];
    if (ODD && (s.la[u] & 1)) {
      b = make_float2(0.f, 0.f);
      c = make_float2(0.f, 0.f);
    }
    P = u ? fmaf(g[u].x, s.a[u].x, P) : g[u].x * s.a[u].x;
    Q = u ? fmaf(g[u].y, s.a[u].y, Q) : g[u].y * s.a[u].y;
    R = u ? fmaf(g[u].x, s.a[u].y, R) : g[u].x * s.a[u].y;
    V = u ? fmaf(g[u].y, s.a[u].x, V) : g[u].y * s.a[u].x;
    P = fmaf(c.x, b.x, P);
    Q = fmaf(c.y, b.y, Q);
    R = fmaf(c.x, b.y, R);
    V = fmaf(c.y, b.x, V);
  }
  acc.P += P;
  acc.Q += Q;
  acc.R += R;
  acc.V += V;
}

// Sum over a point's G lanes, in the last of them (fixed order).
template <int CTRL>
__device__ __forceinline__ double dpp_add(double x)
{
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, false);
  return x + __hiloint2double(hi, lo);
}
__device__ __forceinline__ float lane_sum(double x)
{
  static_assert(G == 8, "three steps");
  return (float)dpp_add<0x114>(dpp_add<0x112>(dpp_add<0x111>(x)));
}

// A sorted point in LDS: x = tap offset of its window (elements), y = r0 |
// c0 << 6 | S << 12 | conj << 30 (first cell relative to the tile), z = layer
// row stride, w = point.
__device__ __forceinline__ void win_start(Walk &w, const int4 &q, int S, int sub, int LS)
{
  const int r0 = q.y & 63, c0 = (q.y >> 6) & 63, stride = q.z;
  const int CP = max(1, (S + 1) >> 1);
  // quotients by the approximate reciprocal: (x + 0.5) / CP lies at least
  // 0.5 / CP >= 1/128 from an integer, far above its error
  const float inv = __builtin_amdgcn_rcpf((float)CP);
  const int row = (int)(((float)sub + 0.5f) * inv);
  const int dr = (int)(((float)G + 0.5f) * inv);
  const int cp = sub - row * CP, dc = G - dr * CP;
  w.tap = (q.x + row * stride + 2 * cp) * 8;
  w.pos = cp << POS_BITS | ((r0 + row) * LS + c0 + 2 * cp) * 8;
  w.tstep = (dr * stride + 2 * dc) * 8;
  w.pstep = (dc << POS_BITS) + (dr * LS + 2 * dc) * 8;
  w.twrap = w.tstep + (stride - 2 * CP) * 8;
  w.pwrap = w.pstep + (LS - 2 * CP) * 8 - (CP << POS_BITS);
  w.wrap = (CP - dc) << POS_BITS;
  w.half = S & 1 ? (CP - 1) << POS_BITS : 0x7fffffff;
  w.k = 0;
  w.n = (S * CP - sub + G - 1) / G;
}

// A wavefront's groups of PW points (wave, wave + W, ... of the batch's ng),
// as one stream of blocks of U steps: while a block is added, the next one's
// taps are in flight, the next group's first after a group's last.  The loads
// stand outside every branch, so that the waits count exactly what is behind
// them; past the end they are sent out of range.
template <bool ODD, int W>
__device__ __forceinline__ void win_stream(const int4 *pts, int total, int wave, int lane, int LS,
                                           int dummy, const char *reg,
                                           __amdgpu_buffer_rsrc_t rsrc, float2 *vis)
{
  const int sub = lane & (G - 1);
  const int ng = (total + PW - 1) / PW;
  int left = ng > wave ? (ng - wave + W - 1) / W : 0;  // groups not yet finished
  if (!left) return;
  int grp = wave;       // the group whose taps are loaded
  Walk w;
  int lb, cb;           // blocks to load of group grp, to add of the current one
  int point, conj, npoint, nconj, nb;
  auto start = [&]() {
    const int j = grp * PW + lane / G;
    const int4 q = pts[min(j, total - 1)];
    const int S = j < total ? (q.y >> 12) & 127 : 0;
    win_start(w, q, S, sub, LS);
    npoint = S ? q.w : -1;
    nconj = q.y;
    // the first point has the largest support, its first lane the most steps
    nb = lb = (__builtin_amdgcn_readfirstlane(w.n) + U - 1) / U;
  };
  auto load = [&](Steps &s) {
    win_load<ODD>(s, w, dummy, rsrc);
    lb--;
  };
  start();
  point = npoint;
  conj = nconj;
  cb = nb;
  Steps s0, s1;
  load(s0);
  Acc acc = {};
  auto body = [&](Steps &cur, Steps &nxt) {
    if (lb == 0) {
      grp += W;
      if (grp < ng) {
        start();
      } else {
        w.n = 0;
        lb = 1 << 30;
      }
    }
    load(nxt);
    __builtin_amdgcn_sched_barrier(0);
    win_add<ODD>(cur, reg, acc);
    if (--cb == 0) {
      // tap (tx, sg ty): re = P - sg Q, im = sg R + V
      const double sg = (conj >> 30) & 1 ? -1.0 : 1.0;
      const float re = lane_sum(fma(-sg, acc.Q, acc.P));
      const float im = lane_sum(fma(sg, acc.R, acc.V));
      if (sub == G - 1 && point >= 0) vis[point] = make_float2(re, im);
      acc = {};
      point = npoint;
      conj = nconj;
      left--;
      cb = left ? nb : 1 << 30;
    }
  };
  do {
    body(s0, s1);
    body(s1, s0);
  } while (left);
}

// One point by a wavefront, the grid read where it lies: g0 its first cell, tap0
// its first tap (element).  Lanes take the taps of the window in row order, 64
// apart, U steps' loads together; sums as in win_add.
__device__ __forceinline__ float2 win_point(const float2 *__restrict__ g0, int pitch,
                                            __amdgpu_buffer_rsrc_t rsrc, int tap0, int stride,
                                            int S, bool conj, int lane)
{
  // quotients by the approximate reciprocal: (x + 0.5) / S lies at least 0.5 /
  // S >= 1/512 from an integer, far above its error
  const float inv = __builtin_amdgcn_rcpf((float)S);
  const int row = (int)(((float)lane + 0.5f) * inv), dr = (int)(64.5f * inv);
  const int dc = 64 - dr * S, total = S * S;
  int col = lane - row * S;
  int t = tap0 + row * stride + col, g = row * pitch + col;
  const int dt = dr * stride + dc, dg = dr * pitch + dc;
  Acc acc = {};
  for (int q = lane; q < total + lane; q += 64 * U) {
    float2 tt[U], gg[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const bool act = q + 64 * u < total;
      tt[u] = tap_load(rsrc, act ? (unsigned)t * 8u : TAP_OOB, 0);
      gg[u] = act ? g0[g] : make_float2(0.f, 0.f);
      const bool wrap = col + dc >= S;
      col += wrap ? dc - S : dc;
      t += wrap ? dt + stride - S : dt;
      g += wrap ? dg + pitch - S : dg;
    }
    float P = 0.f, Q = 0.f, R = 0.f, V = 0.f;
#pragma unroll
    for (int u = 0; u < U; u++) {
      P = fmaf(gg[u].x, tt[u].x, P);
      Q = fmaf(gg[u].y, tt[u].y, Q);
      R = fmaf(gg[u].x, tt[u].y, R);
      V = fmaf(gg[u].y, tt[u].x, V);
    }
    acc.P += P;
    acc.Q += Q;
    acc.R += R;
    acc.V += V;
  }
  const double sg = conj ? -1.0 : 1.0;
  double re = fma(-sg, acc.Q, acc.P), im = fma(sg, acc.R, acc.V);
  for (int off = 32; off > 0; off >>= 1) {
    re += __shfl_xor(re, off);
    im += __shfl_xor(im, off);
  }
  return make_float2((float)re, (float)im);
}

// The points whose support lies above the plan's max_support but whose window
// meets no more tiles than the plan allows (they are gridded too): one
// wavefront per point.  Kept out of the staged region, whose size is the
// plan's; a plan made for its points has none.
__device__ __forceinline__ void win_above(const TiledDev &d, const rcg_pg *__restrict__ pg,
                                          const float2 *__restrict__ grid,
                                          __amdgpu_buffer_rsrc_t rsrc, float2 *__restrict__ vis,
                                          int lane)
{
  const long long nw = (long long)gridDim.x * (blockDim.x >> 6);
  int inst = 0;
  for (long long i = (long long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); i < d.npts;
       i += nw) {
    const rcg_pg r = pg[i];
    if (r.cell < 0 || r.supp <= d.windows) continue;
    int u0, v0, tu0, tu1, tv0, tv1;
    point_tiles(r, d.pitch, d.inv_pitch, d.lt, &u0, &v0, &tu0, &tu1, &tv0, &tv1);
    if ((tu1 - tu0 + 1) * (tv1 - tv0 + 1) > d.mpp) continue;
    while (i >= d.pt_off[inst + 1]) inst++;
    const float2 v = win_point(grid + inst * d.gstride + r.cell, d.pitch, rsrc, r.tap0, r.stride,
                               r.supp, r.flags & PG_CONJ, lane);
    if (lane == 0) vis[i] = v;
  }
}

template <int W>
__global__ void __launch_bounds__(64 * W, 4)  // four wavefronts per SIMD
k_degrid_windows(TiledDev d, int side, int cap, const rcg_pg *__restrict__ pg,
                 const float2 *__restrict__ grid, const float2 *__restrict__ taps,
                 long long n_taps, float2 *__restrict__ vis)
{
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int LS = win_stride(side);
  const int dummy = side * LS * (int)sizeof(float2);  // two cells that stay zero
  float2 *reg = reinterpret_cast<float2 *>(smem);
  int4 *pts = reinterpret_cast<int4 *>(smem + ((dummy + 31) & ~15));
  int *hist = reinterpret_cast<int *>(pts + cap);
  int *misc = hist + WIN_BUCKETS;  // of the batch: points, any odd support, largest support
  const __amdgpu_buffer_rsrc_t rsrc = tap_rsrc(taps, n_taps);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int guess = 0;  // side of the region the last batch needed
  if (threadIdx.x < 2) reg[side * LS + threadIdx.x] = make_float2(0.f, 0.f);
  // points a record
  const float share = (float)d.npts / (float)max(d.totals[0], 1);
  for_each_item(d, d.queue + Q_DEGRID, [&](const ItemRange &ir) {
    const int gsz = d.grid_size;
    const float2 *gi = grid + ir.goff;
    // Of a tile with few points: each by a wavefront (the whole tile alike, so
    // that a point's sums do not hang on the item its record fell in).
    if ((float)ir.most * share <= (float)FEW) {
      for (int k = ir.begin + wave; k < ir.end; k += W) {
        const int4 rec = uniform_record(d.pairs, k);
        if (rec.z >= 0) continue;  // not the point's first tile
        const int S = ((rec.x >> 24) & 63) | ((rec.z >> 24) & 64);
        const float2 v =
            win_point(gi + (long long)(ir.tu0 + (rec.x & 63)) * d.pitch + ir.tv0 + ((rec.x >> 6) & 63),
                      d.pitch, rsrc, rec.y, rec.z & 0xffff, S, (rec.x >> 30) & 1, lane);
        if (lane == 0) vis[rec.w] = v;
      }
      __syncthreads();  // for_each_item's next draw overwrites this one
      return;
    }
    // the square of side `to`, without that of side `from`
    auto stage = [&](int from, int to) {
      for (int r = wave; r < to; r += W) {
        const int gu = ir.tu0 + r;
        for (int c = lane + (r < from ? from : 0); c < to; c += 64) {
          const int gv = ir.tv0 + c;
          reg[r * LS + c] = gu < gsz && gv < gsz ? gi[(long long)gu * d.pitch + gv]
                                                 : make_float2(0.f, 0.f);
        }
      }
    };
    int staged = 0;  // side of the region in LDS
    int n = 0;
    for (int b0 = ir.begin; b0 < ir.end; b0 += n) {
      n = min(WIN_SCAN, ir.end - b0);
      // The records of the batch, and while they are on their way the part of
      // the tile and its surroundings that the last batch needed: a tile's
      // neighbour rarely needs more.
      constexpr int PT = WIN_SCAN / (64 * W);
      int4 rec[PT];
      int key[PT];
#pragma unroll
      for (int u = 0; u < PT; u++)
        rec[u] = d.pairs[min(b0 + u * 64 * W + (int)threadIdx.x, ir.end - 1)];
      for (int q = threadIdx.x; q < WIN_BUCKETS; q += 64 * W) hist[q] = 0;
      if (threadIdx.x == 0) misc[1] = misc[2] = 0;
      if (staged < guess) {
        stage(staged, guess);
        staged = guess;
      }
      __syncthreads();
      // Counting sort by support, largest first.  A thread keeps its records
      // and their ranks between the passes.
      auto count = [&]() {
#pragma unroll
        for (int u = 0; u < PT; u++) {
          const int k = u * 64 * W + (int)threadIdx.x;
          key[u] = 0;
          if (k < n && rec[u].z < 0) {  // the point's first tile
            const int S = ((rec[u].x >> 24) & 63) | ((rec[u].z >> 24) & 64);
            key[u] = S << 16 | atomicAdd(&hist[S], 1);
            if (S & 1) misc[1] = 1;
          }
        }
      };
      // exclusive sums from the largest support down, two buckets a lane
      auto scan = [&]() {
        const int hi = WIN_BUCKETS - 1 - 2 * lane;
        const int x = hist[hi], y = hist[hi - 1];
        int t = x + y;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
          const int z = __shfl_up(t, off);
          if (lane >= off) t += z;
        }
        hist[hi] = t - x - y;
        hist[hi - 1] = t - y;
        if (lane == 63) misc[0] = t;
        const unsigned long long some = __ballot(x + y > 0);
        if (some && lane == __ffsll(some) - 1) misc[2] = x ? hi : hi - 1;
      };
      count();
      __syncthreads();
      if (wave == 0) scan();
      __syncthreads();
      int total = __builtin_amdgcn_readfirstlane(misc[0]);
      if (total > cap) {  // half the records hold no more points than fit
        n = cap;
        __syncthreads();
        for (int q = threadIdx.x; q < WIN_BUCKETS; q += 64 * W) hist[q] = 0;
        __syncthreads();
        count();
        __syncthreads();
        if (wave == 0) scan();
        __syncthreads();
        total = __builtin_amdgcn_readfirstlane(misc[0]);
      }
      if (total) {
        guess = d.T + __builtin_amdgcn_readfirstlane(misc[2]) - 1;
        if (staged < guess) {
          stage(staged, guess);
          staged = guess;
        }
      }
#pragma unroll
      for (int u = 0; u < PT; u++)
        if (key[u])
          pts[hist[key[u] >> 16] + (key[u] & 0xffff)] =
              make_int4(rec[u].y, (rec[u].x & 0x40000fff) | key[u] >> 16 << 12, rec[u].z & 0xffff,
                        rec[u].w);
      __syncthreads();
      if (__builtin_amdgcn_readfirstlane(misc[1]))
        win_stream<true, W>(pts, total, wave, lane, LS, dummy, smem, rsrc, vis);
      else
        win_stream<false, W>(pts, total, wave, lane, LS, dummy, smem, rsrc, vis);
      __syncthreads();
    }
  });
  if (d.totals[3]) win_above(d, pg, grid, rsrc, vis, lane);
}

const void *win_kernel(int waves)
{
  switch (waves) {
    case 2: return reinterpret_cast<const void *>(&k_degrid_windows<2>);
    case 4: return reinterpret_cast<const void *>(&k_degrid_windows<4>);
    default: return reinterpret_cast<const void *>(&k_degrid_windows<8>);
  }
}

}  // namespace

bool windows_fit(int T, int max_support, int chunk)
{
  const double tiles = (double)(max_support - 1) / T + 1;
  return max_support < WIN_BUCKETS && win_lds(T, max_support) <= WIN_LDS &&
         chunk >= ITEM_POINTS * tiles * tiles;
}

hipError_t windows_blocks(int T, int max_support, int waves, int *blocks)
{
  const void *k = win_kernel(waves);
  int dev = 0, cus = 0, per_cu = 0;
  hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, WIN_LDS);
  if (e == hipSuccess) e = hipGetDevice(&dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (e == hipSuccess)
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k, 64 * waves,
                                                     win_lds(T, max_support));
  if (e != hipSuccess) return e;
  *blocks = std::max(8, (std::max(1, per_cu) * std::max(1, cus)) & ~7);
  return hipSuccess;
}

rcg_status windows_degrid(const TiledDev &d, int max_support, int waves, int blocks,
                          const rcg_pg *pg, const float2 *grid, const float2 *taps,
                          long long n_taps, float2 *vis, hipStream_t st)
{
  int side = win_side(d.T, max_support), cap = win_cap(d.T, max_support);
  TiledDev dd = d;
  void *args[] = {&dd, &side, &cap, &pg, &grid, &taps, &n_taps, &vis};
  RCG_HIP_TRY(hipLaunchKernel(win_kernel(waves), dim3(blocks), dim3(64 * waves), args,
                              win_lds(d.T, max_support), st));
  return RCG_OK;
}

}  // namespace rcg
