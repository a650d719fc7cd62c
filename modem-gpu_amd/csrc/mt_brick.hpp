// Brick layout of the inner solves of the mixed-precision solver.
//
// The FP32 inner BiCGStab (red-black tile DILU, multi-system SpMV) keeps its
// vectors, couplings and pivots tile by tile: the 8x8x8 tiles of the three
// interior edge lattices of the red-black tile plan, numbered as the plan
// numbers them (lattice tbase + ti + ntx*(tj + nty*tk)), each tile's 512
// points contiguous (i fastest, then j, then k), points past a partial tile's
// extent held at zero.  In the lattice order a tile row is 8 points (64 bytes
// of FP32 complex), half of a 128-byte line whose other half belongs to the
// neighbouring tile of the other colour: the red-black sweeps fetched about
// twice the bytes they used, in short pieces.  Bricked, a tile is 4 KB
// contiguous per system, and the SpMV's k-1 and k+1 neighbours of 7 of a
// tile's 8 planes lie in the tile itself.
//
// The preconditioned vectors p-hat and s-hat, which the SpMV gathers, can be
// kept with the systems of a pair (2m, 2m+1) side by side, entry
// (s/2)*2nB + 2*point + s%2: the SpMV then reads both systems of a pair with
// one 16-byte gather per neighbour (k_spmv_btp), the DILU writes them so
// (DiluArgs::zout), and every other inner vector stays system-major.
//
// The outer FP64 defect correction stays in the all-edge layout: its scaled
// residual is permuted into bricks before an inner solve and the inner
// correction permuted back after it (k_bk_to_brick / k_bk_from_brick, once
// per outer iteration).
#pragma once

#include "mt_dilu.hpp"
#include "mt_sweep.hpp"

namespace mt {

constexpr int kBkPts = 512;
// chunks of tiles of the brick SpMV (at most; a multiple of the 8 XCDs)
constexpr int kBtChunks = 2048;

// Tile geometry of the bricks (the red-black tile plan's lattices).
struct BrickGeom {
  int A[3], B[3], C[3];        // interior lattice dims per edge component
  int oi[3], oj[3], ok[3];     // offset of the interior lattice in the full lattice
  int ntx[3], nty[3], ntz[3];  // tiles per direction
  int tbase[4];                // first tile of each lattice; tbase[3] = all tiles
  int64_t nB;                  // points per system: tiles * 512
};

// (component, di, dj, dk) of stencil slot s for a row of component c, in
// full-lattice index steps (the order of stencil_neighbours)
struct NbS { int cb, di, dj, dk; };
__host__ __device__ constexpr NbS bk_nb(int c, int s) {
  if (s == 0) return {c, 0, 0, 0};
  if (s <= 6) {
    const int d = (s & 1) ? -1 : 1, ax = (s - 1) >> 1;
    return {c, ax == 0 ? d : 0, ax == 1 ? d : 0, ax == 2 ? d : 0};
  }
  if (c == 0) {
    switch (s) {
      case 7: return {1, 0, -1, 0};  case 8: return {1, 1, -1, 0};
      case 9: return {1, 0, 0, 0};   case 10: return {1, 1, 0, 0};
      case 11: return {2, 0, 0, -1}; case 12: return {2, 1, 0, -1};
      case 13: return {2, 0, 0, 0};  default: return {2, 1, 0, 0};
    }
  }
  if (c == 1) {
    switch (s) {
      case 7: return {0, -1, 0, 0};  case 8: return {0, 0, 0, 0};
      case 9: return {0, -1, 1, 0};  case 10: return {0, 0, 1, 0};
      case 11: return {2, 0, 0, -1}; case 12: return {2, 0, 1, -1};
      case 13: return {2, 0, 0, 0};  default: return {2, 0, 1, 0};
    }
  }
  switch (s) {
    case 7: return {0, -1, 0, 0};  case 8: return {0, 0, 0, 0};
    case 9: return {0, -1, 0, 1};  case 10: return {0, 0, 0, 1};
    case 11: return {1, 0, -1, 0}; case 12: return {1, 0, 0, 0};
    case 13: return {1, 0, -1, 1}; default: return {1, 0, 0, 1};
  }
}

// Brick index of the interior edge of component C at full-lattice (I, J, K),
// or -1 when that edge is not interior (a boundary edge, whose coupling is
// zero, or past the lattice).
template <int C>
__device__ __forceinline__ int bk_at(const BrickGeom& g, int I, int J, int K) {
  const int i = I - g.oi[C], j = J - g.oj[C], k = K - g.ok[C];
  const bool in = (unsigned)i < (unsigned)g.A[C] && (unsigned)j < (unsigned)g.B[C] &&
                  (unsigned)k < (unsigned)g.C[C];
  const int t = g.tbase[C] + (i >> 3) + g.ntx[C] * ((j >> 3) + g.nty[C] * (k >> 3));
  const int q = t * kBkPts + (i & 7) + 8 * (j & 7) + 64 * (k & 7);
  return in ? q : -1;
}

// Lattice and tile position of tile t.
__device__ __forceinline__ void bk_tile(const BrickGeom& g, int t, int& c, int& ti, int& tj,
                                        int& tk) {
  c = t >= g.tbase[2] ? 2 : (t >= g.tbase[1] ? 1 : 0);
  int q = t - g.tbase[c];
  ti = q % g.ntx[c];
  q /= g.ntx[c];
  tj = q % g.nty[c];
  tk = q / g.nty[c];
}

// Tiles [t0, t1) of chunk g of G, the chunks dealt to the three lattices in
// turn (chunk g is part g/3 of lattice g%3): an XCD's G/8 consecutive chunks
// are then the same k-slab fraction of all three lattices, whose rows gather
// each other's values.
__device__ __forceinline__ void bk_tile_range3(const BrickGeom& g, int G, int gi, int& t0,
                                               int& t1) {
  const int c = gi % 3, j = gi / 3;
  const int cnt = (G - c + 2) / 3;
  const int64_t n = g.tbase[c + 1] - g.tbase[c];
  // balanced: every chunk gets floor or ceil of n / cnt tiles
  t0 = g.tbase[c] + int(n * j / cnt);
  t1 = g.tbase[c] + int(n * (j + 1) / cnt);
}

// ------------------------------------------------------------ permutations
// dst[q][b] = src[q][bmap[b]] (0 where bmap[b] < 0), q < nq
template <class T>
__global__ __launch_bounds__(BS) void k_bk_gather(const int* __restrict__ bmap, int64_t nB, int nq,
                                                  int64_t sstride, int64_t dstride,
                                                  const C2<T>* __restrict__ src,
                                                  C2<T>* __restrict__ dst) {
  for (int64_t idx = blockIdx.x * int64_t(BS) + threadIdx.x; idx < nB * nq;
       idx += int64_t(gridDim.x) * BS) {
    const int q = int(idx / nB);
    const int64_t b = idx - q * nB;
    const int e = bmap[b];
    dst[q * dstride + b] = e >= 0 ? src[q * sstride + e] : C2<T>{T(0), T(0)};
  }
}

// Row-major couplings [n][16] (15 slots and vms1) into brick order.
template <class V>
__global__ __launch_bounds__(BS) void k_bk_rows(const int* __restrict__ bmap, int64_t nB,
                                                const V* __restrict__ src, V* __restrict__ dst) {
  for (int64_t idx = blockIdx.x * int64_t(BS) + threadIdx.x; idx < nB * 16;
       idx += int64_t(gridDim.x) * BS) {
    const int64_t b = idx >> 4;
    const int e = bmap[b];
    dst[idx] = e >= 0 ? src[int64_t(e) * 16 + (idx & 15)] : V(0);
  }
}

// Slots 1..6 (the same-component couplings the DILU sweeps use) of the
// slot-major stencil [15][nE] into [6][nB].
template <class V>
__global__ __launch_bounds__(BS) void k_bk_slots(const int* __restrict__ bmap, int64_t nB,
                                                 int64_t nE, const V* __restrict__ coef,
                                                 V* __restrict__ dst) {
  for (int64_t idx = blockIdx.x * int64_t(BS) + threadIdx.x; idx < nB * 6;
       idx += int64_t(gridDim.x) * BS) {
    const int s = int(idx / nB);
    const int64_t b = idx - s * nB;
    const int e = bmap[b];
    dst[idx] = e >= 0 ? coef[(1 + s) * nE + e] : V(0);
  }
}

// Inner right-hand sides: r (bricks) = r32 (all-edge layout) of the active
// systems, the inner correction d (bricks) = 0.
__global__ __launch_bounds__(BS) void k_bk_to_brick(const int* __restrict__ act, int nact,
                                                    const int* __restrict__ bmap, int64_t nB,
                                                    int64_t nE, const C2<float>* __restrict__ r32,
                                                    C2<float>* __restrict__ rb,
                                                    C2<float>* __restrict__ db) {
  for (int64_t idx = blockIdx.x * int64_t(BS) + threadIdx.x; idx < nB * nact;
       idx += int64_t(gridDim.x) * BS) {
    const int q = int(idx / nB);
    const int64_t b = idx - q * nB;
    const int64_t s = act[q];
    const int e = bmap[b];
    rb[s * nB + b] = e >= 0 ? r32[s * nE + e] : C2<float>{0.f, 0.f};
    db[s * nB + b] = {0.f, 0.f};
  }
}

// The inner corrections back into the all-edge layout.
__global__ __launch_bounds__(BS) void k_bk_from_brick(const int* __restrict__ act, int nact,
                                                      const int* __restrict__ bmap, int64_t nB,
                                                      int64_t nE, const C2<float>* __restrict__ db,
                                                      C2<float>* __restrict__ d32) {
  for (int64_t idx = blockIdx.x * int64_t(BS) + threadIdx.x; idx < nB * nact;
       idx += int64_t(gridDim.x) * BS) {
    const int q = int(idx / nB);
    const int64_t b = idx - q * nB;
    const int64_t s = act[q];
    const int e = bmap[b];
    if (e >= 0) d32[s * nE + e] = db[s * nB + b];
  }
}

// FP64 <-> FP32 copies of complex vectors (n entries)
__global__ __launch_bounds__(BS) void k_bk_narrow(const Z* __restrict__ x, C2<float>* __restrict__ y,
                                                  int64_t n) {
  for (int64_t q = blockIdx.x * int64_t(BS) + threadIdx.x; q < n; q += int64_t(gridDim.x) * BS)
    y[q] = {float(x[q].x), float(x[q].y)};
}
__global__ __launch_bounds__(BS) void k_bk_widen(const C2<float>* __restrict__ x, Z* __restrict__ y,
                                                 int64_t n) {
  for (int64_t q = blockIdx.x * int64_t(BS) + threadIdx.x; q < n; q += int64_t(gridDim.x) * BS)
    y[q] = {double(x[q].x), double(x[q].y)};
}

// Point p of tile t for the brick SpMV: whether it is an interior edge, its
// brick index e, its 14 neighbours' brick indices (a neighbour that is not an
// interior edge has a zero coupling and the row's own index) and its 16
// couplings (the brick-ordered row-major copy: 15 slots and the omega-free
// diagonal).
template <class V>
__device__ __forceinline__ void bt_point(const BrickGeom& bg, const V* __restrict__ rowc, int t,
                                         int p, bool& valid, int& e, V (&cf)[16], int (&nb)[15]) {
  int c, ti, tj, tk;
  bk_tile(bg, t, c, ti, tj, tk);
  const int li = p & 7, lj = (p >> 3) & 7, lk = p >> 6;
  const int i = ti * 8 + li, j = tj * 8 + lj, k = tk * 8 + lk;
  valid = i < bg.A[c] && j < bg.B[c] && k < bg.C[c];
  e = t * kBkPts + p;
  const int ee = e;
  auto setup = [&](auto cc) {
    constexpr int C = decltype(cc)::value;
    const int I = i + bg.oi[C], J = j + bg.oj[C], K = k + bg.ok[C];
#pragma unroll
    for (int q = 1; q < 15; ++q) {
      const NbS d = bk_nb(C, q);
      int r;
      if (d.cb == 0) r = bk_at<0>(bg, I + d.di, J + d.dj, K + d.dk);
      else if (d.cb == 1) r = bk_at<1>(bg, I + d.di, J + d.dj, K + d.dk);
      else r = bk_at<2>(bg, I + d.di, J + d.dj, K + d.dk);
      nb[q] = r < 0 ? ee : r;
    }
  };
  if (c == 0) setup(Comp<0>());
  else if (c == 1) setup(Comp<1>());
  else setup(Comp<2>());
  using V4 = typename std::conditional<std::is_same<V, float>::value, float4, double2>::type;
  constexpr int PER = sizeof(V4) / sizeof(V);
  const V4* __restrict__ rp = reinterpret_cast<const V4*>(rowc + int64_t(e) * 16);
#pragma unroll
  for (int q = 0; q < 16 / PER; ++q) {
    const V4 v4 = rp[q];   // pads hold zero couplings
    if constexpr (PER == 4) {
      cf[4 * q] = v4.x; cf[4 * q + 1] = v4.y; cf[4 * q + 2] = v4.z; cf[4 * q + 3] = v4.w;
    } else {
      cf[2 * q] = v4.x; cf[2 * q + 1] = v4.y;
    }
  }
}

// ------------------------------------------------------------------ SpMV
// y_s = A x_s on bricks with the dot products of k_spmv_ms (WHICH=1:
// v = A ph, <rt,v>; WHICH=2: t = A sh, <t,t>, <t,s>), one block per chunk of
// tiles and group of sg active systems (four systems' sums per thread, as
// k_spmv_ms keeps them, cap a brick kernel at two or three waves per SIMD by
// registers): a thread owns one point of the tile, forms its 14 neighbours'
// brick indices and loads its 16 couplings (the brick-ordered row-major copy)
// once, then runs the group's systems one after another, two at a time.  A
// neighbour that is not an interior edge has a zero coupling and the row's
// own index.  The row sums run in k_spmv_ms's order.  Each wave reduces its
// lanes' dot contributions per system (wave_sum63) into LDS; the block then
// sums its waves in order into the per-(system, chunk) partials.
constexpr int kBtThreads = 512, kBtWaves = kBtThreads / 64, kBtMaxSys = 64;
template <class T, class V, int WHICH>
__global__ __launch_bounds__(kBtThreads) void k_spmv_bt(IterArgs<T, V> a, BrickGeom bg,
                                                        const V* __restrict__ rowc, int sg) {
  constexpr int NQ = WHICH == 1 ? 2 : 3;   // doubles per system: <rt,v>; <t,t>, <t,s>
  __shared__ double red[kBtWaves][kBtMaxSys][NQ];
  const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
  // blocks (chunk g, group of sg active systems), the groups of a chunk
  // consecutive inside an XCD (they read the same couplings)
  const int ngrp = (a.nact + sg - 1) / sg;
  const int w = blockIdx.x >> 3, grp = w % ngrp;
  const int g = (blockIdx.x & 7) * (a.G >> 3) + w / ngrp;
  const int s0 = grp * sg, nact = min(a.nact, s0 + sg);
  for (int q = tid; q < kBtWaves * kBtMaxSys * NQ; q += kBtThreads) (&red[0][0][0])[q] = 0.0;
  __syncthreads();
  // the <t,s> partner: s stored by the preconditioner, else r - alpha v
  const bool fz = WHICH == 2 && a.fused && !a.s_ok;
  int t0, t1;
  bk_tile_range3(bg, a.G, g, t0, t1);
  for (int t = t0; t < t1; ++t) {
    const int p = tid;
    bool valid;
    int e;
    V cf[16];
    int nb[15];
    bt_point(bg, rowc, t, p, valid, e, cf, nb);
    // one system: y = A x at this point, its dot contributions
    auto one = [&](int si, double* dq) {
      const int sys = a.act[si];
      const SysScal& sc0 = a.sc[sys];
#pragma unroll
      for (int q = 0; q < NQ; ++q) dq[q] = 0.0;
      if (sc0.status != ST_RUN) return false;
      const int64_t o = (int64_t)sys * a.nE;
      const C2<T>* __restrict__ x = (WHICH == 1 ? a.ph : a.sh) + o;
      const C2<T> xe = x[e];
      C2<T> y = cscale(T(cf[0]), xe);
#pragma unroll
      for (int q = 1; q < 15; ++q) {
        const C2<T> xv = x[nb[q]];
        const T cq = T(cf[q]);
        y.x += cq * xv.x;
        y.y += cq * xv.y;
      }
      const T d = T(kIsignD * sc0.freq_omega) * T(cf[15]);
      y.x += -d * xe.y;
      y.y += d * xe.x;
      if (valid) (WHICH == 1 ? a.v : a.t)[o + e] = y;
      if (!valid) y = {T(0), T(0)};
      C2<T> wv = (WHICH == 1 ? a.rt : (fz ? a.r : a.s))[o + e];
      if (fz) wv = csub(wv, cmul(ccast<T>(sc0.alpha), a.v[o + e]));
      if (WHICH == 1) {
        dq[0] = double(wv.x) * y.x + double(wv.y) * y.y;
        dq[1] = double(wv.x) * y.y - double(wv.y) * y.x;
      } else {
        dq[0] = double(y.x) * y.x + double(y.y) * y.y;
        dq[1] = double(y.x) * wv.x + double(y.y) * wv.y;
        dq[2] = double(y.x) * wv.y - double(y.y) * wv.x;
      }
      return true;
    };
    for (int si = s0; si < nact; si += 2) {
      double d0[NQ], d1[NQ];
      const bool r0 = one(si, d0);
      const bool r1 = si + 1 < nact ? one(si + 1, d1) : false;
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        d0[q] = wave_sum63(d0[q]);
        if (si + 1 < nact) d1[q] = wave_sum63(d1[q]);
      }
      if (lane == 63) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          if (r0) red[wv][si][q] += d0[q];
          if (r1) red[wv][si + 1][q] += d1[q];
        }
      }
    }
  }
  __syncthreads();
  for (int si = s0 + tid; si < nact; si += kBtThreads) {
    double v[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      v[q] = 0.0;
      for (int w = 0; w < kBtWaves; ++w) v[q] += red[w][si][q];
    }
    Z* out = a.partials + ((int64_t)si * a.G + g) * 2;
    if (WHICH == 1) {
      out[0] = {v[0], v[1]};
      out[1] = {0.0, 0.0};
    } else {
      out[0] = {v[0], 0.0};
      out[1] = {v[1], v[2]};
    }
  }
}

// k_spmv_bt for the FP32 inner solves with paired x: ph (WHICH=1) or sh
// (WHICH=2) holds the two systems of a pair interleaved, so one 16-byte
// gather per neighbour serves both (the addressers, which bound the
// single-system kernel, process half the gather instructions).  A block
// takes a chunk of tiles and a group of spg entries of the pair list
// {system 2m, system 2m+1, active index of each or -1}; a pair with one
// system stopped reads both halves and keeps only the running one.  Per
// system the arithmetic, its order and the partial sums (per active index,
// over the block's tiles and waves in order) are k_spmv_bt's.
template <int WHICH>
__global__ __launch_bounds__(kBtThreads, 4) void k_spmv_btp(IterArgs<float, float> a, BrickGeom bg,
                                                         const float* __restrict__ rowc,
                                                         const int4* __restrict__ pairs, int npair,
                                                         int spg) {
  constexpr int NQ = WHICH == 1 ? 2 : 3;
  __shared__ double red[kBtWaves][kBtMaxSys][NQ];
  const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
  const int ngrp = (npair + spg - 1) / spg;
  const int w = blockIdx.x >> 3, grp = w % ngrp;
  const int g = (blockIdx.x & 7) * (a.G >> 3) + w / ngrp;
  const int p0 = grp * spg, p1 = min(npair, p0 + spg);
  for (int q = tid; q < kBtWaves * kBtMaxSys * NQ; q += kBtThreads) (&red[0][0][0])[q] = 0.0;
  __syncthreads();
  // the <t,s> partner: s stored by the preconditioner, else r - alpha v
  const bool fz = WHICH == 2 && a.fused && !a.s_ok;
  const float4* __restrict__ xi = reinterpret_cast<const float4*>(WHICH == 1 ? a.phi : a.shi);
  const int64_t xpair = a.ppair >> 1;   // float4 entries per pair
  int t0, t1;
  bk_tile_range3(bg, a.G, g, t0, t1);
  for (int t = t0; t < t1; ++t) {
    bool valid;
    int e;
    float cf[16];
    int nb[15];
    bt_point(bg, rowc, t, tid, valid, e, cf, nb);
    for (int pi = p0; pi < p1; ++pi) {
      const int4 pr = pairs[pi];   // {2m, 2m+1, active index of 2m, of 2m+1}
      // both systems' records up front (status, omega, alpha)
      bool ra = false, rb = false;
      float wa = 0.f, wb = 0.f;
      C2<float> ala = {0.f, 0.f}, alb = {0.f, 0.f};
      if (pr.z >= 0) {
        const SysScal& sc0 = a.sc[pr.x];
        ra = sc0.status == ST_RUN;
        wa = float(kIsignD * sc0.freq_omega);
        ala = ccast<float>(sc0.alpha);
      }
      if (pr.w >= 0) {
        const SysScal& sc1 = a.sc[pr.y];
        rb = sc1.status == ST_RUN;
        wb = float(kIsignD * sc1.freq_omega);
        alb = ccast<float>(sc1.alpha);
      }
      if (!ra && !rb) continue;   // uniform over the block
      const float4* __restrict__ x = xi + (int64_t)(pr.x >> 1) * xpair;
      const float4 xe = x[e];
      C2<float> y0 = cscale(cf[0], C2<float>{xe.x, xe.y});
      C2<float> y1 = cscale(cf[0], C2<float>{xe.z, xe.w});
#pragma unroll
      for (int q = 1; q < 15; ++q) {
        const float4 xv = x[nb[q]];
        const float cq = cf[q];
        y0.x += cq * xv.x;
        y0.y += cq * xv.y;
        y1.x += cq * xv.z;
        y1.y += cq * xv.w;
      }
      // one system: the diagonal term, y stored (on: running), its dot
      // contributions.  Both systems of the pair are finished whether running
      // or not (a stopped or absent second one reads the first's partner):
      // were the second one's work in a branch, the compiler would sink its
      // half of every gather into it, splitting each 16-byte gather in two.
      auto fin = [&](int sys, bool on, float wsc, C2<float> al, C2<float> y, float xr, float xim,
                     double* dq) {
        const float d = wsc * cf[15];
        y.x += -d * xim;
        y.y += d * xr;
        const int64_t o = (int64_t)sys * a.nE;
        if (valid && on) (WHICH == 1 ? a.v : a.t)[o + e] = y;
        if (!valid) y = {0.f, 0.f};
        C2<float> pw = (WHICH == 1 ? a.rt : (fz ? a.r : a.s))[o + e];
        if (fz) pw = csub(pw, cmul(al, a.v[o + e]));
        if (WHICH == 1) {
          dq[0] = double(pw.x) * y.x + double(pw.y) * y.y;
          dq[1] = double(pw.x) * y.y - double(pw.y) * y.x;
        } else {
          dq[0] = double(y.x) * y.x + double(y.y) * y.y;
          dq[1] = double(y.x) * pw.x + double(y.y) * pw.y;
          dq[2] = double(y.x) * pw.y - double(y.y) * pw.x;
        }
      };
      double d0[NQ], d1[NQ];
      fin(pr.x, ra, wa, ala, y0, xe.x, xe.y, d0);
      fin(rb ? pr.y : pr.x, rb, wb, alb, y1, xe.z, xe.w, d1);
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        d0[q] = wave_sum63(d0[q]);
        d1[q] = wave_sum63(d1[q]);
      }
      if (lane == 63) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          if (ra) red[wv][pr.z][q] += d0[q];
          if (rb) red[wv][pr.w][q] += d1[q];
        }
      }
    }
  }
  __syncthreads();
  // the per-(system, chunk) partials of every active index of the group
  for (int k = tid; k < 2 * (p1 - p0); k += kBtThreads) {
    const int4 pr = pairs[p0 + (k >> 1)];
    const int si = (k & 1) ? pr.w : pr.z;
    if (si < 0) continue;
    double v[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      v[q] = 0.0;
      for (int w2 = 0; w2 < kBtWaves; ++w2) v[q] += red[w2][si][q];
    }
    Z* out = a.partials + ((int64_t)si * a.G + g) * 2;
    if (WHICH == 1) {
      out[0] = {v[0], v[1]};
      out[1] = {0.0, 0.0};
    } else {
      out[0] = {v[0], 0.0};
      out[1] = {v[1], v[2]};
    }
  }
}

// ------------------------------------------------- red-black DILU on bricks
// One tile of one colour for NW systems per workgroup, one wave per system:
// the tile's right-hand sides, pivots and the six couplings it uses are
// contiguous runs, swept in registers (mt_sweep.hpp).  The red forward sweep
// leaves w = dinv*y of the red tiles in the output: that is what the black
// tiles take from their red neighbours, and the red backward sweep forms
// z = w - dinv*(sum of the upper terms), as the black backward sweep does.  A
// tile reads its neighbours' k- and j-faces from their bricks (a k-face is 512
// contiguous bytes, a j-face eight runs of 64) and their i-faces, one value
// per 64 bytes there, from the packed i-faces (DiluArgs::xf) the other colour
// wrote: w of the red tiles, z of the black tiles.  What the neighbouring
// tiles contribute (black: all six faces before the forward sweep; red: all
// six before the backward one, the forward one has none) is folded into the
// right-hand side first, so the sweeps' couplings out of the tile are zero.
// PU: the forward sweeps of the first application form the BiCGStab
// p = r + beta (p - omega v) for their tiles as they load them.
// DiluArgs on bricks: coef = the [6][nB] couplings (slots 1..6), cstride =
// nB, vstride = nB, dinv = [nfreq][nB].
// What bounds it: memory at many systems (100x100x60+10, 16 systems: red
// forward 404 MB in 94 us, black 568 MB in 132 us, red backward 511 MB in 106
// us, 4.3-4.8 TB/s of a copy's 4.9-5.4; per application 330 us, where sweeps
// out of an LDS box took 461 with persistent workgroups that loaded their next
// tile meanwhile), one tile's chain of loads, sweep and stores at few (two
// systems 56 us against 116; 40x40x30+10 19 against 41).  The sweeps are short
// enough that four or five workgroups per CU hide the loads without
// prefetching; the p-update variant needs 98 registers and spills at five.
template <class T, class V, int MODE, int NW, bool ZP = false, bool PU = false>
__global__ __launch_bounds__(64 * NW, NW == 4 ? (PU ? 4 : 5) : 1) void k_dilu_bc(DiluArgs<T, V> a) {
  constexpr int TX = 8, NP = kRbNP, NU = 8;
  static_assert(!PU || MODE != RB_RED_BWD, "the p-update is folded into the forward sweeps");
  constexpr bool FWDP = MODE != RB_RED_BWD;   // has a forward sweep
  constexpr bool BWDP = MODE != RB_RED_FWD;   // has a backward sweep
  constexpr bool HALO = MODE != RB_RED_FWD;   // reads face neighbours
  constexpr int CPT = NP / (64 * NW);         // tile points per thread for the couplings
  __shared__ C2<T> Pall[NW][NP];              // per system: the tile, point order
  __shared__ C2<T> Xall[NW][64];              // per system: cross-row words of the sweeps
  // couplings inside the tile (0 across its faces), and across its faces
  __shared__ V CL[FWDP ? 3 : 1][FWDP ? NP : 1], CH[BWDP ? 3 : 1][BWDP ? NP : 1];
  __shared__ V FC[HALO ? 6 : 1][64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ngrp = (a.nact + NW - 1) / NW;
  const int nwork = a.ntiles * ngrp;
  const int xcd = blockIdx.x & 7, lb = blockIdx.x >> 3;
  const int chunk = (nwork + 7) / 8;
  const int w = xcd * chunk + lb;
  if (lb >= chunk || w >= nwork) return;   // uniform over the workgroup
  const int tix = w / ngrp, grp = w - tix * ngrp;
  const int si = grp * NW + wv;
  const int sys = a.act[si < a.nact ? si : 0];
  const int4 tl = a.tiles[tix];
  const SysScal& sc = a.sc[sys];
  const bool mine = si < a.nact && sc.status == a.status_req;   // uniform over the wave
  const int fidx = sc.fidx;
  const LatticeInfo L = a.lat[tl.x];
  const int gi0 = tl.y * TX, gj0 = tl.z * TX, gk0 = tl.w * TX;
  const int ex = min(TX, L.A - gi0), ey = min(TX, L.B - gj0), ez = min(TX, L.C - gk0);
  const int tself = L.tbase + tl.y + L.ntx * (tl.z + L.nty * tl.w);
  const int tb = tself * kBkPts;   // the tile's first brick index
  const V* __restrict__ cfs = a.coef;
  const int64_t cst = a.cstride;
  const int64_t o = (int64_t)sys * a.vstride;
  const int fa = lane & 7, fb = lane >> 3;
  constexpr bool zp = ZP && MODE != RB_RED_FWD;
  constexpr int zs = zp ? 2 : 1;
  C2<T>* __restrict__ P = Pall[wv];
  // ---- every load of the item
  V cl[CPT][3], ch[CPT][3];
#pragma unroll
  for (int c = 0; c < CPT; ++c) {
    const int p = tid + 64 * NW * c;
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      cl[c][s] = FWDP ? cfs[(int64_t)(2 * s) * cst + tb + p] : V(0);
      ch[c][s] = BWDP ? cfs[(int64_t)(2 * s + 1) * cst + tb + p] : V(0);
    }
  }
  // the tile point next to face f (dir = f/2, low or high) for this lane
  auto face_point = [&](int f) {
    const int dir = f >> 1, t = (f & 1) ? TX - 1 : 0;
    if (dir == 0) return t + TX * (fa + TX * fb);
    if (dir == 1) return fa + TX * (t + TX * fb);
    return fa + TX * (fb + TX * t);
  };
  constexpr int FPW = HALO ? (6 + NW - 1) / NW : 1;   // faces per wave
  V fcv[FPW];
  if (HALO) {
#pragma unroll
    for (int q = 0; q < FPW; ++q) {
      const int f = wv + NW * q;
      fcv[q] = f < 6 ? cfs[(int64_t)f * cst + tb + face_point(f)] : V(0);
    }
  }
  C2<T> rv[NU], v2[NU], r3[PU ? NU : 1], dd[NU], fv[6];
  if (mine) {
    const C2<T>* __restrict__ pin = (FWDP ? a.in : a.out) + o + tb;
    const C2<T>* __restrict__ pin2 = a.in2 ? a.in2 + o + tb : nullptr;
    const C2<T>* __restrict__ dinv = a.dinv + (int64_t)fidx * cst + tb;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int p = lane + 64 * u;
      rv[u] = pin[p];   // points past a partial tile's extent hold zeros
      if constexpr (PU) {
        v2[u] = a.pu_v[o + tb + p];
        r3[u] = a.pu_r[o + tb + p];
      } else {
        v2[u] = (FWDP && pin2) ? pin2[p] : C2<T>{T(0), T(0)};
      }
      dd[u] = dinv[p];
    }
    if (HALO) {
      // the other colour's results (red backward with zout: the black tiles'
      // z, pair-interleaved)
      constexpr bool zr = ZP && MODE == RB_RED_BWD;   // (ZP: the launch has a.zout)
      const C2<T>* __restrict__ pout =
          zr ? a.zout + (int64_t)(sys >> 1) * a.zpair + (sys & 1) : a.out + o;
      const C2<T>* __restrict__ xfi =
          a.xf + (MODE == RB_BLACK_FB ? 0 : a.xfhalf) + (int64_t)sys * a.xfsys;
#pragma unroll
      for (int f = 0; f < 6; ++f) {
        const int dir = f >> 1, d = (f & 1) ? 1 : -1;
        const int ni = tl.y + (dir == 0 ? d : 0), nj = tl.z + (dir == 1 ? d : 0),
                  nk = tl.w + (dir == 2 ? d : 0);
        fv[f] = {T(0), T(0)};
        // (uniform) the neighbouring tile exists
        if (ni >= 0 && nj >= 0 && nk >= 0 && ni * TX < L.A && nj * TX < L.B && nk * TX < L.C) {
          const int tn = L.tbase + ni + L.ntx * (nj + L.nty * nk);
          // its facing layer: i-faces packed (entry lj + 8*lk = lane), j- and
          // k-faces from its brick
          if (!(fa < (dir == 0 ? ey : ex) && fb < (dir == 2 ? ey : ez))) continue;
          if (dir == 0) {
            fv[f] = xfi[(int64_t)tn * kRbFaces + ((f & 1) ? 0 : 64) + lane];
          } else {
            const int fl = (f & 1) ? 0 : TX - 1;
            const int pn = dir == 1 ? fa + TX * (fl + TX * fb) : fa + TX * (fb + TX * fl);
            fv[f] = pout[(zr ? 2 : 1) * ((int64_t)tn * kBkPts + pn)];
          }
        }
      }
    }
  }
  // ---- the couplings into LDS, those across the tile's faces apart
#pragma unroll
  for (int c = 0; c < CPT; ++c) {
    const int p = tid + 64 * NW * c;
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      const int q = s == 0 ? (p & 7) : (s == 1 ? ((p >> 3) & 7) : (p >> 6));
      if (FWDP) CL[s][p] = q == 0 ? V(0) : cl[c][s];
      if (BWDP) CH[s][p] = q == TX - 1 ? V(0) : ch[c][s];
    }
  }
  if (HALO) {
#pragma unroll
    for (int q = 0; q < FPW; ++q) {
      const int f = wv + NW * q;
      if (f < 6) FC[f][lane] = fcv[q];
    }
  }
  __syncthreads();   // the shared couplings; the rest is per wave
  if (!mine) return;
  const int skew = sw_skew(lane);
  const C2<T> zero = {T(0), T(0)};
  // ---- pivots, through the tile buffer into skewed registers
  C2<T> D[NU], R[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) P[lane + 64 * u] = dd[u];
  Xall[wv][lane] = zero;
  sw_order();
#pragma unroll
  for (int u = 0; u < NU; ++u) D[u] = P[sw_point(lane, skew, u)];
  if (HALO) {
#pragma unroll
    for (int f = 0; f < 6; ++f) {
      const T c = T(FC[f][lane]);
      fv[f] = {c * fv[f].x, c * fv[f].y};
      // (the red tiles' buffer will hold w = dinv*y)
      if (MODE == RB_RED_BWD) fv[f] = cmul(P[face_point(f)], fv[f]);
    }
  }
  sw_order();
  // ---- right-hand sides, with the neighbouring tiles' terms taken off
  const C2<T> al = ccast<T>(sc.alpha);
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    C2<T> r = rv[u];
    const int64_t pe = o + tb + lane + 64 * u;
    if constexpr (PU) {
      // k_pupdate's p, stored for the colour's tiles
      if (sc.restart_due) {
        a.pu_rt[pe] = r3[u];
        r = r3[u];
      } else {
        r = cadd(r3[u], cmul(ccast<T>(sc.beta), csub(r, cmul(ccast<T>(sc.omg), v2[u]))));
      }
      a.pu_p[pe] = r;
    } else if (FWDP && a.in2) {
      r = csub(r, cmul(al, v2[u]));
      if (a.sout) a.sout[pe] = r;
    }
    P[lane + 64 * u] = r;
  }
  sw_order();
  if (HALO) {
    // one direction after another: a tile edge lies on two faces
#pragma unroll
    for (int s = 0; s < 3; ++s) {
#pragma unroll
      for (int f = 2 * s; f < 2 * s + 2; ++f) {
        const int q = face_point(f);
        P[q] = csub(P[q], fv[f]);
      }
      sw_order();
    }
  }
#pragma unroll
  for (int u = 0; u < NU; ++u) R[u] = P[sw_point(lane, skew, u)];
  // ---- sweeps
  V cc[NU][3];
  if (FWDP) {
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
      for (int s = 0; s < 3; ++s) cc[u][s] = CL[s][sw_point(lane, skew, u)];
    sw_run<false>(lane, skew, Xall[wv], [&](int u, C2<T> vi, C2<T> vj, C2<T> vk, bool act) {
      C2<T> y = R[u];
      y.x -= T(cc[u][0]) * vi.x;
      y.y -= T(cc[u][0]) * vi.y;
      y.x -= T(cc[u][1]) * vj.x;
      y.y -= T(cc[u][1]) * vj.y;
      y.x -= T(cc[u][2]) * vk.x;
      y.y -= T(cc[u][2]) * vk.y;
      const C2<T> x = cmul(D[u], y);
      R[u] = {act ? x.x : R[u].x, act ? x.y : R[u].y};
      return x;
    });
  }
  if (BWDP) {
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
      for (int s = 0; s < 3; ++s) cc[u][s] = CH[s][sw_point(lane, skew, u)];
    sw_run<true>(lane, skew, Xall[wv], [&](int u, C2<T> vi, C2<T> vj, C2<T> vk, bool act) {
      C2<T> y;
      y.x = T(cc[u][0]) * vi.x;
      y.y = T(cc[u][0]) * vi.y;
      y.x += T(cc[u][1]) * vj.x;
      y.y += T(cc[u][1]) * vj.y;
      y.x += T(cc[u][2]) * vk.x;
      y.y += T(cc[u][2]) * vk.y;
      const C2<T> x = csub(R[u], cmul(D[u], y));
      R[u] = {act ? x.x : R[u].x, act ? x.y : R[u].y};
      return x;
    });
  }
  // ---- back into point order and out (red forward: w; otherwise z), with
  // the packed i-faces the other colour reads next
  sw_order();
#pragma unroll
  for (int u = 0; u < NU; ++u) P[sw_point(lane, skew, u)] = R[u];
  sw_order();
  C2<T>* __restrict__ dst =
      zp ? a.zout + (int64_t)(sys >> 1) * a.zpair + (sys & 1) + 2 * (int64_t)tb : a.out + o + tb;
  C2<T>* __restrict__ xfo = a.xf + (MODE == RB_RED_FWD ? 0 : a.xfhalf) + (int64_t)sys * a.xfsys +
                            (int64_t)tself * kRbFaces;
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    if (!(fa < ex && fb < ey && u < ez)) continue;
    const C2<T> zv = P[lane + 64 * u];
    dst[zs * (lane + 64 * u)] = zv;
    if (MODE != RB_RED_BWD && (fa == 0 || fa == TX - 1)) xfo[(fa == 0 ? 0 : 64) + fb + 8 * u] = zv;
  }
}

}  // namespace mt
