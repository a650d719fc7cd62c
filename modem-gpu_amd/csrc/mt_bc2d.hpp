// The boundary values and initial guess of a forward solve from 2-D TE slice
// solves (BC_x0_WS, 3D_MT/FWD/boundary_ws.f90:21-171), on the device.
//
// For mode 1 (Ey polarisation) the reference solves one 2-D TE problem per
// y-slice over the (x, z) cells of the slice and writes it to the y-edges;
// for mode 2 (Ex) one per x-slice over (y, z), written to the x-edges.  Each
// problem (Siripunvaraporn's code, 3D_MT/FWD/Mod2d/) has (nh-1)(nz-1)
// interior nodes, 1 at the top of the air, and on the sides and bottom the
// values of 1-D TE columns (Fwd1D_TE, WSfwd1Dmod.f90:79-141).  Its 5-point
// system is band-factored by LAPACK (FormAII -> ZGBTRF, WSfwd2Dmod.f90:31-85)
// and solved (Fwd2DsolveTE -> ZGBTRS, FwdTEmod.f90:110-169), bandwidth nz-1
// on both sides of the diagonal.
//
// k_bc_te1d solves every 1-D column, one thread each.  k_bc_te2d solves one
// slice per workgroup: the band's active (nz x nz) window stays in registers
// as a circular buffer over rows and columns, the right-hand side is
// eliminated as the factorisation proceeds, the rows of U go to a
// per-workgroup scratch in HBM, and one wave back-substitutes from staged
// chunks of U.
//
// Every complex product and quotient is formed as the reference's BLAS and
// LAPACK form it (textbook products, C99 Annex G division as __divdc3 does
// it, no contraction) and every entry receives its updates in the same
// order, so the fields equal the reference's bit for bit while its partial
// pivoting keeps the diagonal.  (ZGERU's a + x*(-1*y) is formed as
// a - x*y: negation is exact and round-to-nearest symmetric, so the two
// agree in value and differ at most in the sign of a zero.)  A column where it would interchange rows (or
// a zero pivot) is flagged, and the entry point reports it.
#pragma once

#include "mt_device.hpp"
#include "mt_dilu.hpp"
#include "mt_internal.h"
#include "mt_sweep.hpp"

namespace mt {

constexpr int kBcChunk = 128;  // factorisation steps per staged chunk of entering coefficients
constexpr int kBcBack = 16;    // back-substitution steps per staged chunk of U

// A node's diagonal, right-hand side and couplings to the next node in z and
// in the horizontal.
struct BcCoef { double2 d, r; double a2, a3; };

struct BcArgs {
  int nx, ny, nz, nza;          // 3-D grid; nz counts the air layers
  int64_t nXe, nE;              // x-edges, all edges
  const double *dx, *dy, *dz;   // cell sizes
  const double *cx, *cy, *cz;   // DistanceBetweenBlocks of dx, dy, dz (n+1 entries each)
  const double* sig;            // earth cell conductivity [nzEarth][ny][nx]
  const double* omega;          // [nsys]
  const int* mode;              // [nsys] 1 or 2
  const int2* item;             // [nitem] (system, slice), slice 1-based
  int nitem;
  int ncolMax;                  // max(nx, ny) + 1: 1-D columns per item, padded
  int mmbMax;                   // boundary vector length per item (1-based, index 0 unused)
  double2* exb;                 // [nitem][mmbMax] boundary values of each slice (EXB)
  double2* side;                // [nitem][2][nz][2] factors of the two side columns
  int* flag;                    // [nitem] 1 if the reference's LU would pivot (or a zero pivot)
  double2* e;                   // [nsys][nE] out: E0 inside, the boundary conditions outside
};

// Per-workgroup scratch of k_bc_te2d: urow [nmax][M], urow[j-1][c] = U(j, j+c) (M >= nz slots);
// yx [nmax], the eliminated rhs, then the solution; coef [nmax], the slice's
// matrix and rhs by node.
struct BcScratch {
  double2 *urow, *yx;
  BcCoef* coef;
  int64_t nmax;
  int nz, nitem;
};

struct BcSlice {
  int sys, s, mode, nh;
  const double *dh, *ch;
  double omue;
};

__device__ __forceinline__ BcSlice bc_slice(const BcArgs& a, int it) {
#pragma clang fp contract(off)
  const int2 q = a.item[it];
  BcSlice S;
  S.sys = q.x;
  S.s = q.y;
  S.mode = a.mode[q.x];
  S.nh = S.mode == 2 ? a.ny : a.nx;
  S.dh = S.mode == 2 ? a.dy : a.dx;
  S.ch = S.mode == 2 ? a.cy : a.cx;
  // ComputeBC passes period = 2 PI / omega; the 2-D and 1-D codes take
  // omega = 2 PI / period back and omega mu0 from it
  const double per = (2.0 * kPi) / a.omega[q.x];
  S.omue = ((2.0 * kPi) / per) * kMu0;
  return S;
}

__device__ __forceinline__ double2 bz_mul(double2 a, double2 b) {
#pragma clang fp contract(off)
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// complex quotient, C99 Annex G (G.5.1) for finite operands: the divisor
// scaled by 2^-logb(max(|c|, |d|)).  In two steps, so that what depends on the
// divisor alone can be formed ahead: den = |scaled divisor|^2 lies in [1, 8)
// and inv is 1/den to the last bit or so; a quotient n/den is n*inv with one
// correction from its exact remainder, which is the correctly rounded one (the
// steps of the hardware's own division without its rescaling) while neither
// n nor the remainder leaves the normal range; else n/den is divided as such.
struct BzDen { double c, e, den, inv; int il; };
__device__ __forceinline__ BzDen bz_den(double2 d) {
#pragma clang fp contract(off)
  BzDen q;
  q.c = d.x;
  q.e = d.y;
  q.il = 0;
  const double mx = fmax(fabs(q.c), fabs(q.e));
  if (mx > 0.0 && mx < HUGE_VAL) {   // logb(mx) is finite
    q.il = __builtin_amdgcn_frexp_exp(mx) - 1;
    q.c = scalbn(q.c, -q.il);
    q.e = scalbn(q.e, -q.il);
  }
  q.den = q.c * q.c + q.e * q.e;
  double r = __builtin_amdgcn_rcp(q.den);
  r = __builtin_fma(r, __builtin_fma(-q.den, r, 1.0), r);
  q.inv = __builtin_fma(r, __builtin_fma(-q.den, r, 1.0), r);
  return q;
}
__device__ __forceinline__ double2 bz_div(double2 n, const BzDen& q) {
#pragma clang fp contract(off)
  const double nx = n.x * q.c + n.y * q.e, ny = n.y * q.c - n.x * q.e;
  double x = nx * q.inv, y = ny * q.inv;
  x = __builtin_fma(__builtin_fma(-q.den, x, nx), q.inv, x);
  y = __builtin_fma(__builtin_fma(-q.den, y, ny), q.inv, y);
  // 2^-900 .. 2^900, or zero over a den in its range
  const double lo = 0x1p-900, hi = 0x1p900, ax = fabs(nx), ay = fabs(ny);
  const bool ok = q.den >= 1.0 && q.den < 8.0 && (ax == 0.0 || ax > lo) && ax < hi &&
                  (ay == 0.0 || ay > lo) && ay < hi;
  if (!ok) {
    x = nx / q.den;
    y = ny / q.den;
  }
  return make_double2(scalbn(x, -q.il), scalbn(y, -q.il));
}
__device__ __forceinline__ double2 bz_div(double2 n, double2 d) { return bz_div(n, bz_den(d)); }

__device__ __forceinline__ bool bz_nz(double2 v) { return v.x != 0.0 || v.y != 0.0; }
__device__ __forceinline__ double bz_abs1(double2 v) { return fabs(v.x) + fabs(v.y); }

// cell conductivity of the slice, 1-based (ih, iz); the air is SIGMA_AIR
__device__ __forceinline__ double bc_sig(const BcArgs& a, const BcSlice& S, int ih, int iz) {
  if (iz <= a.nza) return kSigmaAir;
  const int i = S.mode == 2 ? S.s : ih, j = S.mode == 2 ? ih : S.s;
  return a.sig[(i - 1) + int64_t(a.nx) * ((j - 1) + int64_t(a.ny) * (iz - a.nza - 1))];
}

// node q (1-based) of the slice's interior, iz fastest
__device__ __forceinline__ void bc_node(int b, int q, int& iy, int& iz) {
  iy = 2 + (q - 1) / b;
  iz = 2 + (q - 1) % b;
}

// SetupA_TE (WSfwd2Dmod.f90:345-438) + FormAII's diagonal
__device__ __forceinline__ double2 bc_diag(const BcArgs& a, const BcSlice& S, int iy, int iz) {
#pragma clang fp contract(off)
  const double s00 = bc_sig(a, S, iy, iz), s10 = bc_sig(a, S, iy, iz - 1);
  const double s01 = bc_sig(a, S, iy - 1, iz), s11 = bc_sig(a, S, iy - 1, iz - 1);
  const double dzi = a.dz[iz - 1], dzm = a.dz[iz - 2], dyi = S.dh[iy - 1], dym = S.dh[iy - 2];
  const double s2d = (s00 * dzi * dyi + s01 * dzi * dym + s10 * dzm * dyi + s11 * dzm * dym) /
                     (dzi * dyi + dzi * dym + dzm * dyi + dzm * dym);
  const double cz = a.cz[iz - 1], cy = S.ch[iy - 1];
  const double ar = 2.0 * cz / dyi, al = 2.0 * cz / dym, ad = 2.0 * cy / dzi, au = 2.0 * cy / dzm;
  const double a1 = -ar - al - ad - au;
  const double a4 = cy * cz * s2d;
  return make_double2(a1, S.omue * a4);
}
// coupling to the next node in z (0 at the bottom row)
__device__ __forceinline__ double bc_a2(const BcArgs& a, const BcSlice& S, int iy, int iz) {
#pragma clang fp contract(off)
  return iz == a.nz ? 0.0 : 2.0 * S.ch[iy - 1] / a.dz[iz - 1];
}
// coupling to the next node in the horizontal (0 in the last column)
__device__ __forceinline__ double bc_a3(const BcArgs& a, const BcSlice& S, int iy, int iz) {
#pragma clang fp contract(off)
  return iy < S.nh ? 2.0 * a.cz[iz - 1] / S.dh[iy - 1] : 0.0;
}

// MulAibWithXb (WSfwd2Dmod.f90:89-140) for one node: the sides assign (the
// right after the left), then the top and the bottom subtract
__device__ __forceinline__ double2 bc_rhs(const BcArgs& a, const BcSlice& S, const double2* exb,
                                          int iy, int iz) {
#pragma clang fp contract(off)
  const int Nz = a.nz, Ny = S.nh;
  double2 r = make_double2(0.0, 0.0);
  if (iy == 2) {
    const double c = 2.0 * a.cz[iz - 1] / S.dh[0];
    const double2 x = exb[iz];
    r = make_double2(-(c * x.x), -(c * x.y));
  }
  if (iy == Ny) {
    const double c = 2.0 * a.cz[iz - 1] / S.dh[Ny - 1];
    const double2 x = exb[Nz + 2 * Ny - 1 + iz];
    r = make_double2(-(c * x.x), -(c * x.y));
  }
  if (iz == 2) {
    const double c = 2.0 * S.ch[iy - 1] / a.dz[0];
    const double2 x = exb[Nz + iy];
    r = make_double2(r.x - c * x.x, r.y - c * x.y);
  }
  if (iz == Nz) {
    const double c = 2.0 * S.ch[iy - 1] / a.dz[Nz - 1];
    const double2 x = exb[Nz + Ny + iy - 1];
    r = make_double2(r.x - c * x.x, r.y - c * x.y);
  }
  return r;
}

// conductivity of the 1-D column col at layer iz (1..nz+1; nz+1 repeats nz):
// the side columns of the slice, or the dh-weighted mean of the two cells
// over an interior bottom node (SetBound2D_TE, WSfwd2Dmod.f90:262-341)
__device__ __forceinline__ double bc_col_sig(const BcArgs& a, const BcSlice& S, int col, int iz) {
#pragma clang fp contract(off)
  const int z = iz > a.nz ? a.nz : iz;
  if (z <= a.nza) return kSigmaAir;
  if (col == 0) return bc_sig(a, S, 1, z);
  if (col == S.nh) return bc_sig(a, S, S.nh, z);
  const int iy = col + 1;
  return (bc_sig(a, S, iy - 1, z) * S.dh[iy - 2] + bc_sig(a, S, iy, z) * S.dh[iy - 1]) /
         (S.dh[iy - 2] + S.dh[iy - 1]);
}

// Fwd1D_TE + Solve1D for every column of every slice: the tridiagonal LU
// (ZGBTF2 with kl = ku = 1, which never pivots here: every pivot exceeds its
// real subdiagonal in modulus) and ZGBTRS.  Interior columns keep only the
// bottom value; the two side columns keep their whole profile.
__global__ void k_bc_te1d(BcArgs a) {
#pragma clang fp contract(off)
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int it = int(t / a.ncolMax), col = int(t % a.ncolMax);
  if (it >= a.nitem) return;
  const BcSlice S = bc_slice(a, it);
  if (col > S.nh) return;
  const int Nz = a.nz;
  const bool sidecol = col == 0 || col == S.nh;
  double2* exb = a.exb + (int64_t)it * a.mmbMax;
  double2* sd = a.side + ((int64_t)it * 2 + (col == 0 ? 0 : 1)) * Nz * 2;
  const double skd = sqrt(2.0 / (bc_col_sig(a, S, col, Nz + 1) * S.omue));
  // ac(jj) = i omue (s(jj+1) dz1(jj+1) + s(jj) dz1(jj)) - 2/dz1(jj) - 2/dz1(jj+1)
  double dprev = a.dz[0], sprev = bc_col_sig(a, S, col, 1);
  const double au1 = 2.0 / dprev;
  double dcur = Nz >= 2 ? a.dz[1] : skd, scur = bc_col_sig(a, S, col, 2);
  double adv = 2.0 / dcur;
  double2 p = make_double2((0.0 - au1) - adv, S.omue * (scur * dcur + sprev * dprev));
  double2 bj = make_double2(-au1, 0.0);
  for (int j = 1; j < Nz; ++j) {
    if (sidecol) {
      sd[2 * (j - 1)] = p;
      sd[2 * (j - 1) + 1] = bj;
    }
    const double2 r = bz_div(make_double2(1.0, 0.0), p);
    const double2 l = bz_mul(r, make_double2(adv, 0.0));
    const double2 tt = bz_mul(make_double2(-1.0, 0.0), make_double2(adv, 0.0));
    // next row: au(j+1) = 2/dz1(j+1) is this adv
    dprev = dcur;
    sprev = scur;
    dcur = j + 2 <= Nz ? a.dz[j + 1] : skd;
    scur = bc_col_sig(a, S, col, j + 2);
    const double au = adv;
    adv = 2.0 / dcur;
    const double2 ac = make_double2((0.0 - au) - adv, S.omue * (scur * dcur + sprev * dprev));
    const double2 lt = bz_mul(l, tt);
    p = make_double2(ac.x + lt.x, ac.y + lt.y);
    if (bz_nz(bj)) {
      const double2 lb = bz_mul(l, bz_mul(make_double2(-1.0, 0.0), bj));
      bj = make_double2(0.0 + lb.x, 0.0 + lb.y);
    } else {
      bj = make_double2(0.0, 0.0);
    }
  }
  double2 x = bz_nz(bj) ? bz_div(bj, p) : bj;
  if (!sidecol) {
    exb[Nz + S.nh - 1 + (col + 1)] = x;   // X1D(nz+1) under interior node column col+1
    return;
  }
  // back substitution of the side column: x(j-1) from b(j-1) - x(j) ad(j-1)
  const int base = col == 0 ? 1 : Nz + 2 * S.nh;   // EXB position of X1D(1)
  exb[base] = make_double2(1.0, 0.0);
  exb[base + Nz] = x;
  for (int j = Nz - 1; j >= 1; --j) {
    const double2 pj = sd[2 * (j - 1)];
    double2 b = sd[2 * (j - 1) + 1];
    if (bz_nz(x)) {
      const double ad = 2.0 / a.dz[j];          // A(j, j+1) = 2/dz1(j+1)
      const double2 u = bz_mul(x, make_double2(ad, 0.0));
      b = make_double2(b.x - u.x, b.y - u.y);
    }
    x = bz_nz(b) ? bz_div(b, pj) : b;
    exb[base + j] = x;
  }
  if (col == 0)
    for (int ii = Nz + 2; ii <= Nz + S.nh; ++ii) exb[ii] = make_double2(1.0, 0.0);   // the surface
}

// A workgroup barrier that orders LDS only: the factorisation's global
// stores (rows of U, the eliminated rhs) are not read back until after a full
// barrier, so the steps need not wait for them (__syncthreads would).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Largest nz mt_bc_x0_dev takes (the largest window, 16 x 7 slots, would hold 112).
constexpr int kBcMaxNz = 100;

// The arguments as if met for the first time: what one phase of a slice reads
// of them is not kept in registers over the others.
__device__ __forceinline__ const BcArgs* bc_reload(const BcArgs* p) {
  asm volatile("" : "+s"(p));
  return p;
}

// v of a wave's lane `l` (uniform)
__device__ __forceinline__ double bc_lane(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                          __builtin_amdgcn_readlane(__double2loint(v), l));
}
__device__ __forceinline__ double2 bc_lane(double2 v, int l) {
  return make_double2(bc_lane(v.x, l), bc_lane(v.y, l));
}

// One slice per workgroup of TG x TG threads, persistent over the items.
//
// The window: node r has slot r mod M, M = TG*R >= nz (the nodes j .. j+nz-1
// of step j hold distinct slots); thread (tr, tc) keeps A(r, c) of the R x R
// slots (tr + TG*ii, tc + TG*jj) in registers, 0 where the slots hold no node.
// A step j is
//   export  (at the end of step j-1): the wave that holds column j forms the
//           multipliers l = A(:, j) (1/p) and the rhs update, the threads of
//           row j store U(j, :); both go to LDS vectors by slot (two sets,
//           alternating) and the slot's row and column become zero;
//   barrier;
//   the entering node's coefficients are placed, then every thread updates
//   its R x R entries with the R multipliers and R row values it reads.
// What bounds it: with many slices the issue of FP64 products and sums
// without contraction, eight per entry and step (three slices per CU at nz =
// 70: 3,530 cycles a step, 3 x 1,200 of issue), and the rounds (1,600 slices of
// 100 x 70 on 768 resident workgroups leave 64 for a third); with few the
// chain of a step (1/p 440 cycles, multipliers 450, update 570 at nz = 35).
// With the window in LDS a step moved 290 KB there and took two barriers:
// 1,600 slices of 100 x 70 97 ms, now 43; 78 of 45 x 35 3.4 ms, now 2.1.
template <int TG, int R>
struct BcShape {
  static constexpr int M = TG * R, NT = TG * TG;
  // waves per SIMD the register window leaves room for
  static constexpr int WAVES = R <= 4 ? 4 : (R == 5 ? 3 : (R == 6 ? 2 : 1));
};

__host__ __device__ inline size_t bc_back_bytes(int nz) {
  return (size_t(kBcBack) * nz + 2 * kBcBack) * sizeof(double2) + kBcBack * sizeof(BzDen);
}

template <int TG, int R>
__global__ __launch_bounds__(TG * TG, (BcShape<TG, R>::WAVES)) void k_bc_te2d(const BcArgs* __restrict__ ap, BcScratch w) {
#pragma clang fp contract(off)
  constexpr int M = BcShape<TG, R>::M, NT = BcShape<TG, R>::NT;
  static_assert(NT % 64 == 0 && 64 % TG == 0, "a column's threads lie in one wave");
  extern __shared__ double2 lds[];   // back substitution: kBcBack columns of U, as many rhs entries
  __shared__ double2 Lv[2][M], Uv[2][M], Pv[2], Bv[M];
  __shared__ double2 Ed[2][kBcChunk], Er[2][kBcChunk];
  __shared__ double Ea2[2][kBcChunk], Ea3[2][kBcChunk];
  __shared__ int sflag;
  const int b = w.nz - 1, B1 = w.nz;
  const int tid = threadIdx.x, tr = tid % TG, tc = tid / TG, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  double2* __restrict__ U = w.urow + (int64_t)blockIdx.x * w.nmax * M;
  double2* __restrict__ Y = w.yx + (int64_t)blockIdx.x * w.nmax;
  BcCoef* __restrict__ C = w.coef + (int64_t)blockIdx.x * w.nmax;

  for (int it = blockIdx.x; it < w.nitem; it += gridDim.x) {
    if (tid == 0) sflag = 0;
    int n;
    {
      const BcArgs a = *bc_reload(ap);
      const BcSlice S = bc_slice(a, it);
      const double2* exb = a.exb + (int64_t)it * a.mmbMax;
      n = __builtin_amdgcn_readfirstlane((S.nh - 1) * b);
      for (int q = 1 + tid; q <= n; q += NT) {
        int iy, iz;
        bc_node(b, q, iy, iz);
        BcCoef v;
        v.d = bc_diag(a, S, iy, iz);
        v.r = bc_rhs(a, S, exb, iy, iz);
        v.a2 = bc_a2(a, S, iy, iz);
        v.a3 = bc_a3(a, S, iy, iz);
        C[q - 1] = v;
      }
    }
    __syncthreads();
    // the window of step 1: nodes 1 .. b (n >= b) in the slots of their numbers
    double Ax[R][R], Ay[R][R];
#pragma unroll
    for (int ii = 0; ii < R; ++ii)
#pragma unroll
      for (int jj = 0; jj < R; ++jj) {
        const int r = tr + TG * ii, c = tc + TG * jj, lo = min(r, c);
        Ax[ii][jj] = Ay[ii][jj] = 0.0;
        if (lo >= 1 && max(r, c) <= b) {
          if (r == c) {
            Ax[ii][jj] = C[lo - 1].d.x;
            Ay[ii][jj] = C[lo - 1].d.y;
          } else if (r - c == 1 || c - r == 1) {
            Ax[ii][jj] = C[lo - 1].a2;
          }
        }
      }
    for (int q = tid; q < M; q += NT) {
      double2 v = make_double2(0.0, 0.0);
      if (q >= 1 && q <= b) v = C[q - 1].r;
      Bv[q] = v;
    }
    // the coefficients of steps j0 .. j0+kBcChunk-1: node step+b's diagonal and
    // rhs, its z-coupling to the node before, the step's own horizontal coupling
    auto stage = [&](int j0, int buf) {
      for (int t = tid; t < kBcChunk; t += NT) {
        const int jj = j0 + t, q = jj + b;
        if (q <= n) {
          Ed[buf][t] = C[q - 1].d;
          Er[buf][t] = C[q - 1].r;
          Ea2[buf][t] = C[q - 2].a2;
        }
        if (jj <= n) Ea3[buf][t] = C[jj - 1].a3;
      }
    };
    stage(1, 0);
    __syncthreads();

    // (the window is in registers here: with its loads still pending at the
    // loop, every step would wait for its own stores of U)
#pragma unroll
    for (int ii = 0; ii < R; ++ii)
#pragma unroll
      for (int jj = 0; jj < R; ++jj) asm volatile("" : "+v"(Ax[ii][jj]), "+v"(Ay[ii][jj]));
    // the steps, slot by slot of the pivot: sj = ts + TG*ip with ip a constant
    int j = 1, ts = 1 % TG, sj = 1, sq = (1 + b) % M;
    // step jn's entering coefficients: read a step ahead where there are
    // registers for them (R = 5 spills with eight more)
    constexpr bool AHEAD = R <= 4;
    double2 ed;
    double e2, e3;
    auto entering = [&](int jn) {
      const int c1 = (jn - 1) % kBcChunk, b1 = ((jn - 1) / kBcChunk) & 1;
      ed = Ed[b1][c1];
      e2 = Ea2[b1][c1];
      e3 = Ea3[b1][c1];
    };
    entering(1);
    while (j <= n) {
#pragma unroll
      for (int ip = 0; ip < R; ++ip) {
        for (; ts < TG && j <= n; ++ts, ++j) {
          // (opaque: nothing a step derives from the grid position is kept in
          // registers over the steps.  A spilled register's reload would wait
          // for the step's stores of U)
          int r0 = tr, c0 = tc;
          asm volatile("" : "+v"(r0), "+v"(c0));
          const int par = j & 1, cs = (j - 1) % kBcChunk, buf = ((j - 1) / kBcChunk) & 1;
          const bool own = wave == (ts * TG) >> 6;   // this wave's threads c0 == ts hold column j
          if (j + b <= n) {
            if constexpr (!AHEAD) entering(j);
            // node q = j+b enters: its diagonal, its couplings to q-1 and to j
            // (slot sq, empty until here)
            const int iq = sq / TG, tq = sq % TG, t1 = (tq + TG - 1) % TG;
            const bool wq = wave == (tq * TG) >> 6;
            if (own || wq || wave == (t1 * TG) >> 6) {
#pragma unroll
              for (int ii = 0; ii < R; ++ii) {
                if (ii != iq) continue;   // uniform
                const int im = (ii + R - 1) % R;
                if (wq && c0 == tq) {
                  if (r0 == tq) {
                    Ax[ii][ii] = ed.x;
                    Ay[ii][ii] = ed.y;
                  }
                  if (r0 == t1) {
                    if (tq > 0) Ax[ii][ii] = e2;
                    else Ax[im][ii] = e2;
                  }
                  if (r0 == ts) Ax[ip][ii] = e3;
                }
                if (c0 == t1 && r0 == tq) {
                  if (tq > 0) Ax[ii][ii] = e2;
                  else Ax[ii][im] = e2;
                }
                if (own && c0 == ts && r0 == tq) Ax[ii][ip] = e3;
              }
            }
          }
          if (own) {
            __builtin_amdgcn_s_setprio(1);   // the others wait for this wave
            // thread r0 == c0 == ts holds the pivot
            const double2 p =
                bc_lane(make_double2(Ax[ip][ip], Ay[ip][ip]), (ts * TG + ts) & 63);
            const double2 rp = bz_div(make_double2(1.0, 0.0), p);
            if (c0 == ts) {
              const double pa = bz_abs1(p);
              bool bad = !bz_nz(p);
#pragma unroll
              for (int ii = 0; ii < R; ++ii) {
                const double2 v = make_double2(Ax[ii][ip], Ay[ii][ip]);
                const bool piv = ii == ip && r0 == ts;   // (multiplier 0 in the pivot's own slot)
                const double2 l = bz_mul(rp, v);
                Lv[par][r0 + TG * ii] = make_double2(piv ? 0.0 : l.x, piv ? 0.0 : l.y);
                if (piv) Pv[par] = v;
                bad |= !(bz_abs1(v) <= pa);
                Ax[ii][ip] = Ay[ii][ip] = 0.0;
              }
              if (bad) sflag = 1;
            }
            __builtin_amdgcn_s_setprio(0);
          }
          if (r0 == ts) {
#pragma unroll
            for (int jj = 0; jj < R; ++jj) {
              // (the pivot's own slot: zero, as above or by the column's threads)
              const bool piv = jj == ip && c0 == ts;
              Uv[par][c0 + TG * jj] = make_double2(piv ? 0.0 : Ax[ip][jj], piv ? 0.0 : Ay[ip][jj]);
              Ax[ip][jj] = Ay[ip][jj] = 0.0;
            }
          }
          lds_barrier();
          if constexpr (AHEAD) entering(j + 1);
          double2 l[R];
#pragma unroll
          for (int ii = 0; ii < R; ++ii) l[ii] = Lv[par][r0 + TG * ii];
          // (a column's row value is read one column ahead, not all at once:
          // registers)
          double2 u = Uv[par][c0];
#pragma unroll
          for (int jj = 0; jj < R; ++jj) {
            const double2 un = Uv[par][c0 + TG * (jj + 1 < R ? jj + 1 : jj)];
#pragma unroll
            for (int ii = 0; ii < R; ++ii) {
              const double2 t = bz_mul(l[ii], u);
              Ax[ii][jj] -= t.x;
              Ay[ii][jj] -= t.y;
            }
            u = un;
            __builtin_amdgcn_sched_barrier(0);
          }
          // row j of U, entry c (node j+c, slot s = sj + c mod M, zero in empty
          // slots), and the rhs of row j+c: by threads of the waves that do not
          // hold the next columns
          const int t = (tid - 64 * ((ts * TG >> 6) + 2)) & (NT - 1);
          if (t < M) {
            int s = sj + t;
            if (s >= M) s -= M;
            const double2 yv = Bv[sj], ls = Lv[par][s];
            double2 u = Uv[par][s], base = Bv[s];
            if (s == sq && j + b <= n) base = Er[buf][cs];
            if (t == 0) {
              u = Pv[par];
              Y[j - 1] = yv;
            } else {
              if (bz_nz(yv)) {
                const double2 d = bz_mul(ls, yv);
                base = make_double2(base.x - d.x, base.y - d.y);
              }
              Bv[s] = base;
            }
            U[(int64_t)(j - 1) * M + t] = u;
          }
          // (read from step j0+kBcChunk on, barriers later)
          if (cs == 0 && j + kBcChunk <= n) stage(j + kBcChunk, buf ^ 1);
          if (++sj == M) sj = 0;
          if (++sq == M) sq = 0;
        }
        if (ts == TG) ts = 0;
      }
    }
    __syncthreads();
    if (tid == 0) ap->flag[it] = sflag;

    // back substitution with U (ZTBSV order): x_j = y_j / U(j,j), then
    // y_{j-o} -= x_j U(j-o, j) for o = 1..b.  Wave 0 keeps the open rows, row
    // i in lane i mod 64 (ra the lane's highest open row, ya its value, yb row
    // ra-64's); the columns of U are staged by chunk, the next chunk's loads
    // in flight meanwhile.
    double2* SU = lds;                   // [k][o] = U(j-o, j), j = j0+k
    double2* SY = lds + kBcBack * B1;    // [k] = y of row j-128
    double2* SX = SY + kBcBack;          // [k] = x_j
    BzDen* SD = reinterpret_cast<BzDen*>(SX + kBcBack);   // [k]: U(j,j) as a divisor
    constexpr int NE = ((kBcBack + M) * kBcBack + NT - 1) / NT;
    double2 st[NE], sy = make_double2(0.0, 0.0);
    auto back_load = [&](int j1) {
      const int j0 = max(1, j1 - kBcBack + 1);
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const int x = tid + NT * e, k = x % kBcBack, o = b - x / kBcBack + k;
        const int i = j0 + k - o;
        st[e] = make_double2(0.0, 0.0);
        if (o >= 0 && o <= b && j0 + k <= j1 && i >= 1) st[e] = U[(int64_t)(i - 1) * M + o];
      }
      sy = make_double2(0.0, 0.0);
      if (tid < kBcBack && j0 + tid - 128 >= 1) sy = Y[j0 + tid - 128 - 1];
    };
    double2 ya = make_double2(0.0, 0.0), yb = ya;
    if (wave == 0) {
      const int ra = n - ((n - lane) & 63);
      if (ra >= 1) ya = Y[ra - 1];
      if (ra > 64) yb = Y[ra - 65];
    }
    // (arrived here: pending at the steps, they would make each step wait for
    // the next chunk's loads too)
    asm volatile("" : "+v"(ya.x), "+v"(ya.y), "+v"(yb.x), "+v"(yb.y));
    back_load(n);
    for (int j1 = n; j1 >= 1; j1 -= kBcBack) {
      const int j0 = max(1, j1 - kBcBack + 1);
      __syncthreads();
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const int x = tid + NT * e, k = x % kBcBack, o = b - x / kBcBack + k;
        if (o >= 0 && o <= b) SU[k * B1 + o] = st[e];
      }
      if (tid < kBcBack) SY[tid] = sy;
      __syncthreads();
      if (wave == 0 && lane < kBcBack) SD[lane] = bz_den(SU[lane * B1]);
      sw_order();
      if (j1 - kBcBack >= 1) back_load(j1 - kBcBack);
      if (wave == 0) {
        // a step's reads a step ahead; column entry o past the band or above
        // row 1 is taken as 0 (subtracting x*0 changes nothing)
        double2 ua, ub, ys;
        BzDen p;
        auto fetch = [&](int j) {
          const int k = j - j0, o = (j - lane) & 63;
          const double2* Uc = SU + k * B1;
          p = SD[k];
          ys = SY[k];
          const double2 va = Uc[min(o, b)], vb = Uc[min(o + 64, b)];
          const bool oa = o >= 1 && o <= b, ob = o + 64 <= b;
          ua = make_double2(oa ? va.x : 0.0, oa ? va.y : 0.0);
          ub = make_double2(ob ? vb.x : 0.0, ob ? vb.y : 0.0);
        };
        fetch(j1);
        for (int j = j1; j >= j0; --j) {
          const BzDen pj = p;
          const double2 uaj = ua, ubj = ub, ysj = ys;
          fetch(max(j - 1, j0));
          const int lj = j & 63;
          const double2 yj = bc_lane(ya, lj);
          double2 xj = yj;
          if (bz_nz(yj)) {   // uniform
            xj = bz_div(yj, pj);
            const double2 da = bz_mul(xj, uaj), db = bz_mul(xj, ubj);
            ya = make_double2(ya.x - da.x, ya.y - da.y);
            yb = make_double2(yb.x - db.x, yb.y - db.y);
          }
          if (lane == lj) {
            SX[j - j0] = xj;
            ya = yb;
            yb = ysj;
          }
        }
        if (lane <= j1 - j0) Y[j0 + lane - 1] = SX[lane];
      }
    }
    __syncthreads();
    // Esol into the edge field (mode 2: x-edges of x-slice s; mode 1: y-edges
    // of y-slice s); the bottom face carries the zeroed xZMax / yZMax
    const BcArgs a = *bc_reload(ap);
    const BcSlice S = bc_slice(a, it);
    const double2* exb = a.exb + (int64_t)it * a.mmbMax;
    const int Ny = S.nh, nzp = a.nz + 1, nhp = Ny + 1;
    double2* E = a.e + (int64_t)S.sys * a.nE;
    for (int e = tid; e < nhp * nzp; e += NT) {
      const int iz = 1 + e % nzp, ih = 1 + e / nzp;
      double2 v;
      if (iz == nzp) v = make_double2(0.0, 0.0);
      else if (ih == 1) v = exb[iz];
      else if (ih == nhp) v = exb[a.nz + 2 * Ny - 1 + iz];
      else if (iz == 1) v = exb[a.nz + ih];
      else v = Y[(ih - 2) * b + (iz - 2)];
      const int64_t idx =
          S.mode == 2 ? (S.s - 1) + int64_t(a.nx) * ((ih - 1) + int64_t(a.ny + 1) * (iz - 1))
                      : a.nXe + (ih - 1) + int64_t(a.nx + 1) * ((S.s - 1) + int64_t(a.ny) * (iz - 1));
      E[idx] = v;
    }
    __syncthreads();
  }
}

}  // namespace mt
