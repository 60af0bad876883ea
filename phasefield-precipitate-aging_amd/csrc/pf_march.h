// pf_march.h -- device code shared by the plain and the batched step kernels:
// the per-strip "march" that advances one wave's strip of one row chunk by one
// explicit Euler step.  Both kernels run exactly this arithmetic, so a
// simulation gives the same bits whether it runs alone or inside a batch.
//
// One wave64 owns a strip of 64 columns (62 output columns + one halo column
// each side) and marches down a chunk of rows.  Each lane keeps a three-row
// window (y-1, y, y+1) of what the stencil needs -- phi_delta, phi_Laves and
// the two diffusion potentials mu -- in registers, so each cell
// is loaded once per strip and its KKS solve is done once.  x-neighbours come
// from adjacent lanes through DPP wave shifts (no LDS round trip).  Loads run DEPTH
// rows ahead of the row being computed (a register ring), so a wave keeps
// several rows of HBM requests in flight; the row loop is unrolled by 6 so the
// window and the ring rotate by register renaming instead of moves.
//
// Boundary conditions are index maps (no ghost reads): no-flux reflects about
// the domain faces, which at the one ghost layer the one-step march reads is
// exactly the reference's ghost copy (src/discretization.cu:360-394); periodic
// wraps.
// Ghost cells of the outputs are written with the value of the cell they
// mirror.  Storage T is double or float; all arithmetic is FP64.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "pf_internal.h"
#include "pf_thermo.h"

// Every fused multiply-add of the step is written as fma(): the kernels that
// inline this arithmetic (one to four steps per launch, plain and batched) must
// give the same bits, and the compiler's own contraction depends on what it
// sees around an expression.
#pragma clang fp contract(off)

namespace pf {

constexpr int WAVE = 64;
constexpr int STRIP = WAVE - 2;   // output columns per strip
constexpr int STRIP3 = WAVE - 6;  // and of the three-step march (the batched form's strips)
constexpr int WPB = 4;           // waves (strips) per block: adjacent strips of one row chunk
constexpr int UNROLL = 6;        // multiple of the 3-row window and of every ring depth

// a pointer into LDS (address space 3), for the multi-step march's row windows
typedef double __attribute__((address_space(3)))* LdsPtr;

__device__ __forceinline__ int xcd_remap(int b, int nb) {
  // Hardware dispatches block b to XCD b % 8.  Give XCD x the contiguous
  // logical range [x*per + min(x, rem), ... + count_x).
  const int per = nb >> 3, rem = nb & 7;
  const int x = b & 7, k = b >> 3;
  return x * per + min(x, rem) + k;
}

// Interior index map.  No-flux (BC 0): even reflection about the domain
// faces (-1 -> 0, -2 -> 1, ..., n -> n-1, n+1 -> n-2, ...).  At the one
// ghost layer (i = -1, n) this is the reference's ghost copy
// (src/discretization.cu:360-394); deeper halo cells (the multi-step march)
// are the mirror images that make every intermediate level's halo equal,
// bit for bit, to the ghost copy of that level (see marchk_impl).  Periodic
// (BC 1): wrap.  Both for i in [-n, 2n); any other i maps into [0, n) too
// (lanes past the last strip's halo, unused).  No division: the march maps a
// row index per iteration.
template <int BC>
__device__ __forceinline__ int bc_map(int i, int n) {
  if (i < 0) return BC == 0 ? min(-1 - i, n - 1) : i + n;
  if (i >= n) return BC == 0 ? max(2 * n - 1 - i, 0) : ((i - n) < n ? i - n : n - 1);
  return i;
}

// DPP wave shifts (GFX9 wave_shr:1 / wave_shl:1): lane i receives lane i-1 /
// lane i+1.  With bound_ctrl set, lanes 0 and 63 (no source lane) receive 0;
// their results are never stored.
__device__ __forceinline__ double from_left(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x138, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x138, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double from_right(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x130, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x130, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

struct Point {       // what the neighbours of a cell need
  double pd, pl;     // phase fields
  double mu0, mu1;   // common diffusion potential
};
struct Centre {      // extra state of a cell when it is the stencil centre
  double xCr, xNb;   // compositions as stored (x - StepParams::xoff)
};
template <typename T>
struct Raw {
  T cr, nb, pd, pl;
};

// Field access as a wave-uniform row byte offset (scalar registers) plus a
// 32-bit per-lane byte offset.  The compiler forms each address with one
// 64-bit multiply-add of the row index onto a hoisted per-lane base; forcing
// a scalar row base instead costs more in scalar-register spills than the
// add it saves.
template <typename T>
__device__ __forceinline__ T ld_at(const T* base, size_t row_bytes, uint32_t lane_bytes) {
  return *(const T*)((const char*)base + row_bytes + lane_bytes);
}
template <typename T>
__device__ __forceinline__ void st_at(T* base, size_t row_bytes, uint32_t lane_bytes, T v) {
  *(T*)((char*)base + row_bytes + lane_bytes) = v;
}
template <typename T>
__device__ __forceinline__ void load_row(Raw<T>& r, const T* iCr, const T* iNb, const T* ipd,
                                         const T* ipl, size_t row_bytes, uint32_t lane_bytes) {
  r.cr = ld_at(iCr, row_bytes, lane_bytes);
  r.nb = ld_at(iNb, row_bytes, lane_bytes);
  r.pd = ld_at(ipd, row_bytes, lane_bytes);
  r.pl = ld_at(ipl, row_bytes, lane_bytes);
}
template <typename T>
__device__ __forceinline__ void store_row(T* oCr, T* oNb, T* opd, T* opl, size_t row_bytes,
                                          uint32_t lane_bytes, double a, double b, double c,
                                          double d) {
  st_at(oCr, row_bytes, lane_bytes, (T)a);
  st_at(oNb, row_bytes, lane_bytes, (T)b);
  st_at(opd, row_bytes, lane_bytes, (T)c);
  st_at(opl, row_bytes, lane_bytes, (T)d);
}

// 1/d to within an ulp or so: hardware reciprocal r and one third-order step
// r (1 + e + e^2), e = 1 - d r.  Measured on 4M random doubles over 200
// binades, the hardware reciprocal is good to 2^-24.4, so the e^3 left out is
// below 2^-73; a Newton step (r + r e) leaves up to 2.2e-15 relative.
__device__ __forceinline__ double recip(double d) {
  const double r = __builtin_amdgcn_rcp(d);
  const double e = fma(-d, r, 1.0);
  return fma(r, fma(e, e, e), r);
}
// One Newton step (relative error <= 2.2e-15): for FP32 storage, whose every
// stored value is rounded to 2^-24 relative, so the second step changes no
// stored result beyond that rounding; 2 FP64 operations less per cell
// (the FP32-storage kernels are bound by FP64 arithmetic).
__device__ __forceinline__ double recip1(double d) {
  const double r = __builtin_amdgcn_rcp(d);
  return fma(r, fma(-d, r, 1.0), r);
}

// Interpolator p(x) = x^3 (6x^2 - 15x + 10), returned less one half:
// p - 1/2 = (x - 1/2) (1 + 2u + 6u^2), u = x (1 - x).  The halves are folded
// into the constants p multiplies.  Five operations, as the power form takes;
// for |x| < TINY this gives exactly -1/2 (u = x, x - 1/2 and 1 + 2u round to
// -1/2 and 1), which is what lets matrix cells share one set of coefficients
// (Coef).  It is good to 2^-54 absolute, what the sums of order one it enters
// hold of it; the power form's terms cancel near x = 1.  Error of one step's
// composition increments against long double, power form / this: quiet matrix
// 2.6e-21 / 2.7e-21 (x_Cr) and 1.8e-20 / 1.6e-20 (x_Nb), two particles per kind
// 5.5e-20 / 1.5e-20 and 1.5e-19 / 4.6e-20, phi random 1.5e-16 / 1.4e-17 and
// 3.8e-16 / 3.5e-17.
constexpr double TINY = 0x1p-56;
__device__ __forceinline__ double p_less_half(double x) {
  const double u = fma(-x, x, x);
  return (x - 0.5) * fma(u, fma(6.0, u, 2.0), 1.0);
}

// KKS solve of a cell (src/parabola625.cu:245-297 restated): with
// p_gamma = 1 - p_delta - p_Laves eliminated and q = p - 1/2,
// M = M_mid + q_d (A_d - A_g) + q_l (A_l - A_g), M_mid = (A_d + A_l) / 2, and
// r = x - xe_mid - q_d (xe_d - xe_g) - q_l (xe_l - xe_g), xe_mid = (xe_d + xe_l) / 2
// less the storage offset (StepParams::xe_mid); mu = M^-1 r, and the
// neighbours need mu (x_g = xe_g + A_g mu is linear in it).
constexpr double DA_DEL[3] = {A[1][0] - A[0][0], A[1][1] - A[0][1], A[1][2] - A[0][2]};
constexpr double DA_LAV[3] = {A[2][0] - A[0][0], A[2][1] - A[0][1], A[2][2] - A[0][2]};
constexpr double A_MID[3] = {0.5 * (A[1][0] + A[2][0]), 0.5 * (A[1][1] + A[2][1]),
                             0.5 * (A[1][2] + A[2][2])};
constexpr double DXE_DEL[2] = {XE[1][0] - XE[0][0], XE[1][1] - XE[0][1]};
constexpr double DXE_LAV[2] = {XE[2][0] - XE[0][0], XE[2][1] - XE[0][1]};

// Addends of FMAs whose multiplicand is a constant too.  A VOP3 instruction
// reads one scalar register pair at most, so one of the two constants has to
// be in vector registers; keeping these there for the whole march saves a
// move before each use (the empty asm stops the compiler from rebuilding them
// from scalars every time).
struct Addends {
  double A[3];          // A_MID
  double xe[2];         // -StepParams::xe_mid
  double qs[2];         // StepParams::qs
  double g3[2], g4[2];  // StepParams::g[.][3], [4]
  double w[2];          // -StepParams::w
};
__device__ __forceinline__ double in_vgpr(double x) {
  asm("" : "+v"(x));
  return x;
}
__device__ __forceinline__ Addends addends(const StepParams& P) {
  Addends a;
#pragma unroll
  for (int i = 0; i < 3; i++) a.A[i] = in_vgpr(A_MID[i]);
#pragma unroll
  for (int i = 0; i < 2; i++) {
    a.xe[i] = in_vgpr(-P.xe_mid[i]);
    a.qs[i] = in_vgpr(P.qs[i]);
    a.g3[i] = in_vgpr(P.g[i][3]);
    a.g4[i] = in_vgpr(P.g[i][4]);
    a.w[i] = in_vgpr(-P.w[i]);
  }
  return a;
}

// What the phase fields of a cell determine of its solve: M, 1/det M and the
// composition-free part t of r = x + t.
struct Coef {
  double M0, M1, M2, t0, t1, inv;
};
template <typename T>
__device__ __forceinline__ Coef coefficients(const Addends& ad, double pd, double pl) {
  const double qD = p_less_half(pd);
  const double qL = p_less_half(pl);
  Coef k;
  k.M0 = fma(qD, DA_DEL[0], fma(qL, DA_LAV[0], ad.A[0]));
  k.M1 = fma(qD, DA_DEL[1], fma(qL, DA_LAV[1], ad.A[1]));
  k.M2 = fma(qD, DA_DEL[2], fma(qL, DA_LAV[2], ad.A[2]));
  k.t0 = fma(-qD, DXE_DEL[0], fma(-qL, DXE_LAV[0], ad.xe[0]));
  k.t1 = fma(-qD, DXE_DEL[1], fma(-qL, DXE_LAV[1], ad.xe[1]));
  const double det = fma(k.M0, k.M2, -(k.M1 * k.M1));
  k.inv = sizeof(T) == sizeof(float) ? recip1(det) : recip(det);
  return k;
}
__device__ __forceinline__ void solve(const Coef& k, const Centre& c, Point& v) {
  const double r0 = c.xCr + k.t0, r1 = c.xNb + k.t1;
  v.mu0 = fma(k.M2, r0, -(k.M1 * r1)) * k.inv;
  v.mu1 = fma(k.M0, r1, -(k.M1 * r0)) * k.inv;
}

template <typename T>
__device__ __forceinline__ void derive(const Addends& ad, const Raw<T>& r, Point& v, Centre& c) {
  v.pd = (double)r.pd;
  v.pl = (double)r.pl;
  c.xCr = (double)r.cr;
  c.xNb = (double)r.nb;
  solve(coefficients<T>(ad, v.pd, v.pl), c, v);
}

__device__ __forceinline__ Point shift_left(const Point& a) {
  return Point{from_left(a.pd), from_left(a.pl), from_left(a.mu0), from_left(a.mu1)};
}
__device__ __forceinline__ Point shift_right(const Point& a) {
  return Point{from_right(a.pd), from_right(a.pl), from_right(a.mu0), from_right(a.mu1)};
}

// Nucleation of one cell from its new values (centre-only scan; the caller
// guarantees R_scan < 1).  Mirrors src/discretization.cu:1104-1176 with the
// event order delta then Laves on the pre-embed composition.
__device__ __forceinline__ void nucleate_cell(const NucParams& N, uint32_t cell, double& xCr,
                                           double& xNb, double& pd, double& pl,
                                           const Scratch& S) {
  const double phi_pre = p(pd) + p(pl);
  if (!(phi_pre < 1e-10)) return;
  double u1, u2;
  nuc_uniforms(N.seed, N.call, N.instance, cell, u1, u2);
  const double cCr = xCr, cNb = xNb;
  const double dG = g(0, cCr, cNb);
  const double DCrCr = D(0, 0, cCr, cNb);
  const double DNbNb = D(1, 1, cCr, cNb);
#pragma unroll
  for (int ph = 0; ph < 2; ph++) {
    double Rstar, Pn;
    nucleation_probability(cCr, cNb, dG, DCrCr, DNbNb, ph == 0 ? N.sigma_del : N.sigma_lav,
                           N.Vatom, N.n_gam, N.dV, N.dt, Rstar, Pn);
    if (Rstar > 0.) {
      const double u = ph == 0 ? u1 : u2;
      if (Pn - u > 0) {
        const double R = Rstar / N.dx_arg;
        if (R < 1.0) {
          // embed loop collapses to the centre (r = 0 <= R)
          xCr = XE[1 + ph][0];
          xNb = XE[1 + ph][1];
          if (ph == 0)
            pd = 1.0;
          else
            pl = 1.0;
        } else {
          const uint32_t slot = atomicAdd(&S.counters[0], 1u);
          atomicAdd(&S.counters[2], 1u);
          if (slot < S.event_capacity) {
            S.events[slot] = Event{cell, (uint32_t)ph, cCr, cNb, R};
          } else {
            atomicOr(&S.counters[1], 1u);
          }
        }
      }
    }
  }
}

// Laplacians of the four stencil quantities with the reference's masks
// (src/discretization.cu:589-595): rows y-1, y, y+1; columns x-1, x, x+1.
// FIVE: a folded symmetric five-point mask (m[1] = m[7] = 1, m[3] = m[5]; the
// factor the caller's mask had at m[1] is in q and k).  A Laplacian is
// (S + N) + m[3] (W + E) + m[4] C.
// NINE: a mask symmetric in x and y (the reference's nine-point one).  Its
// west and east columns are alike, so a lane forms its column's share of its
// neighbours' Laplacians, m[0] (S + N) + m[3] C, and only that is exchanged:
// 7 operations and one shift each way per value, 9 and three rows' shifted
// neighbours kept in registers for ANY.
// Both add mirror images in the same order, which the multi-step march's
// no-flux halo rests on.
// ANY: the nine-term sum in mask order.
enum Mask { FIVE, NINE, ANY };

__device__ __forceinline__ double five_point(const double* m, double s, double w, double c,
                                             double e, double n) {
  return fma(m[4], c, fma(m[3], w + e, s + n));
}
template <Mask MASK>
__device__ __forceinline__ double stencil(const double* m, double s, double c, double n) {
  if constexpr (MASK == FIVE) {
    return five_point(m, s, from_left(c), c, from_right(c), n);
  } else {
    const double sn = s + n, column = fma(m[0], sn, m[3] * c);
    return (from_left(column) + from_right(column)) + fma(m[4], c, m[1] * sn);
  }
}
template <Mask MASK>
__device__ __forceinline__ void laplacians(const double* m, const Point& S, const Point& C,
                                           const Point& N, double lap[4]) {
  lap[0] = stencil<MASK>(m, S.pd, C.pd, N.pd);
  lap[1] = stencil<MASK>(m, S.pl, C.pl, N.pl);
  lap[2] = stencil<MASK>(m, S.mu0, C.mu0, N.mu0);
  lap[3] = stencil<MASK>(m, S.mu1, C.mu1, N.mu1);
}
__device__ __forceinline__ double nine_terms(const double* m, double sw, double s, double se,
                                             double w, double c, double e, double nw, double n,
                                             double ne) {
  double v = m[0] * sw;
  v = fma(m[1], s, v);
  v = fma(m[2], se, v);
  v = fma(m[3], w, v);
  v = fma(m[4], c, v);
  v = fma(m[5], e, v);
  v = fma(m[6], nw, v);
  v = fma(m[7], n, v);
  return fma(m[8], ne, v);
}
// ANY: win, winW, winE hold rows y-1, y, y+1 in slots p, c, n
__device__ __forceinline__ void laplacians_any(const double* m, const Point* win,
                                               const Point* winW, const Point* winE, int p,
                                               int c, int n, double lap[4]) {
#define PF_TERMS(F)                                                                          \
  nine_terms(m, winW[p].F, win[p].F, winE[p].F, winW[c].F, win[c].F, winE[c].F, winW[n].F,   \
             win[n].F, winE[n].F)
  lap[0] = PF_TERMS(pd);
  lap[1] = PF_TERMS(pl);
  lap[2] = PF_TERMS(mu0);
  lap[3] = PF_TERMS(mu1);
#undef PF_TERMS
}

// The explicit Euler update of one cell from its stencil Laplacians:
// Cahn-Hilliard (src/discretization.cu:859-863) and Allen-Cahn
// (src/discretization.cu:888-942) with the closed-form grand-potential
// difference at the solved potential, as the quadratic form of StepParams.
// The composition increment is formed on its own from the Laplacians of the
// potential and added to x once, as the reference adds dt D lap(x_g): where
// the increment is ~0 (the uniform matrix) x comes back unchanged, so rounding
// adds no drift there.  The kernels are bound by the FP64 operations they
// issue, so the sums are nested to take the fewest: the Laplacians of mu (not
// of dt D x_gamma) save the two products of q per cell and two doubles of
// state per level, the quadratic form is evaluated in two brackets with no
// squares, and u (G u + w (2 phi - 1)) and c phi phi_o^2 are folded into
// FMAs: 33 operations after the Laplacians, 41 with the terms written out.
__device__ __forceinline__ void update_compositions(const StepParams& P, const Addends& ad,
                                                    const double lap_mu[2], const Centre& cc,
                                                    double& nCr, double& nNb) {
  nCr = cc.xCr + fma(P.qCr[0], lap_mu[0], fma(P.qCr[1], lap_mu[1], ad.qs[0]));
  nNb = cc.xNb + fma(P.qNb[0], lap_mu[0], fma(P.qNb[1], lap_mu[1], ad.qs[1]));
}
__device__ __forceinline__ void update_cell(const StepParams& P, const Addends& ad,
                                            const double lap[4], const Point& cur,
                                            const Centre& cc, double& nCr, double& nNb,
                                            double& npd, double& npl) {
  update_compositions(P, ad, lap + 2, cc, nCr, nNb);
  const double fd = cur.pd, fl = cur.pl;
  const double Gd = fma(cur.mu0, fma(P.g[0][0], cur.mu0, fma(P.g[0][1], cur.mu1, ad.g3[0])),
                        cur.mu1 * fma(P.g[0][2], cur.mu1, ad.g4[0]));
  const double Gl = fma(cur.mu0, fma(P.g[1][0], cur.mu0, fma(P.g[1][1], cur.mu1, ad.g3[1])),
                        cur.mu1 * fma(P.g[1][2], cur.mu1, ad.g4[1]));
  const double ud = fma(-fd, fd, fd), ul = fma(-fl, fl, fl);  // phi (1 - phi)
  const double td = fma(ud, Gd, fma(P.w2[0], fd, ad.w[0]));
  const double tl = fma(ul, Gl, fma(P.w2[1], fl, ad.w[1]));
  const double z = fd * fl;
  npd = fma(-(P.c[0] * z), fl, fma(ud, td, fma(P.k[0], lap[0], fd)));
  npl = fma(-(P.c[1] * z), fd, fma(ul, tl, fma(P.k[1], lap[1], fl)));
}

template <typename T>
__device__ __forceinline__ void store4(T* oCr, T* oNb, T* opd, T* opl, size_t o, double a,
                                       double b, double c, double d) {
  oCr[o] = (T)a;
  oNb[o] = (T)b;
  opd[o] = (T)c;
  opl[o] = (T)d;
}

// Write the ghost-ring images of interior cell (gx, y) (0-based interior
// coordinates): no-flux mirrors edge cells onto the adjacent ghost cells,
// periodic onto the opposite side.  Corner ghosts get the corner cell's value.
template <typename T, int BC>
__device__ __forceinline__ void store_ghost_images(T* oCr, T* oNb, T* opd, T* opl, int gx, int y,
                                                   int Nx, int Ny, int pitch, double a, double b,
                                                   double c, double d) {
  const bool ex = (gx == 0) || (gx == Nx - 1);
  const bool ey = (y == 0) || (y == Ny - 1);
  if (!(ex || ey)) return;
  int cx[3], cy[3], ncx = 1, ncy = 1;
  cx[0] = 1 + gx;
  cy[0] = 1 + y;
  if (BC == 0) {
    if (gx == 0) cx[ncx++] = 0;
    if (gx == Nx - 1) cx[ncx++] = Nx + 1;
    if (y == 0) cy[ncy++] = 0;
    if (y == Ny - 1) cy[ncy++] = Ny + 1;
  } else {
    if (gx == Nx - 1) cx[ncx++] = 0;
    if (gx == 0) cx[ncx++] = Nx + 1;
    if (y == Ny - 1) cy[ncy++] = 0;
    if (y == 0) cy[ncy++] = Ny + 1;
  }
  for (int j = 0; j < ncy; j++)
    for (int i = 0; i < ncx; i++) {
      if (i == 0 && j == 0) continue;
      store4(oCr, oNb, opd, opl, (size_t)cy[j] * pitch + cx[i], a, b, c, d);
    }
}

// Advance strip `strip` of row chunk `chunk` (rows [chunk*rows, ...)) by one
// step, reading the old fields and writing the new ones.  Called by a whole
// wave; uses no barriers.  SW is the number of output columns per strip (62,
// or 60 where the strips are laid out for the two-step march).
template <typename T, int BC, Mask MASK, bool NUC, int DEPTH, int SW = STRIP>
__device__ __forceinline__ void march(
    const T* __restrict__ iCr, const T* __restrict__ iNb, const T* __restrict__ ipd,
    const T* __restrict__ ipl, T* __restrict__ oCr, T* __restrict__ oNb, T* __restrict__ opd,
    T* __restrict__ opl, int Nx, int Ny, int pitch, int strip, int chunk, int rows,
    const StepParams& P, const NucParams& N, const Scratch& S) {
  static_assert(UNROLL % DEPTH == 0, "ring depth must divide the unroll factor");
  const int lane = threadIdx.x & (WAVE - 1);

  static_assert(SW >= 1 && SW <= STRIP, "strip width");
  const int gx = strip * SW + lane - 1;   // interior column owned by this lane
  const int px = 1 + bc_map<BC>(gx, Nx);  // padded column it reads
  const bool out_lane = (lane >= 1) && (lane <= SW) && (gx < Nx);

  const int y0 = chunk * rows;
  const int y1 = min(y0 + rows, Ny);
  if (y0 >= Ny) return;

  const uint32_t in_lane = (uint32_t)px * (uint32_t)sizeof(T);
  const uint32_t out_lane_b = (uint32_t)(1 + gx) * (uint32_t)sizeof(T);
  const size_t row_b = (size_t)pitch * sizeof(T);
  auto load = [&](Raw<T>& r, int y) {
    load_row(r, iCr, iNb, ipd, ipl, (size_t)(1 + bc_map<BC>(y, Ny)) * row_b, in_lane);
  };

  const Addends ad = addends(P);
  // window slots (row y0 + k - 1 + 3j lives in slot k % 3 pattern below)
  Point win[3];
  Centre cen[3];
  Point winW[3], winE[3];  // DPP-shifted neighbours (ANY only)
  Raw<T> ring[DEPTH];

  {
    Raw<T> r;
    load(r, y0 - 1);
    derive<T>(ad, r, win[2], cen[2]);
    load(r, y0);
    derive<T>(ad, r, win[0], cen[0]);
  }
#pragma unroll
  for (int j = 0; j < DEPTH; j++) load(ring[j], min(y0 + 1 + j, y1));
  if (MASK == ANY) {
    winW[2] = shift_left(win[2]);
    winE[2] = shift_right(win[2]);
    winW[0] = shift_left(win[0]);
    winE[0] = shift_right(win[0]);
  }

  const double* m = P.m;
  for (int yb = y0;; yb += UNROLL) {
#pragma unroll
    for (int k = 0; k < UNROLL; k++) {
      const int y = yb + k;
      if (y >= y1) return;
      const int ps = (k + 2) % 3, cs = k % 3, ns = (k + 1) % 3;
      const int rs = k % DEPTH;
      derive<T>(ad, ring[rs], win[ns], cen[ns]);
      load(ring[rs], min(y + 1 + DEPTH, y1));

      double lap[4];
      if constexpr (MASK == ANY) {
        winW[ns] = shift_left(win[ns]);
        winE[ns] = shift_right(win[ns]);
        laplacians_any(m, win, winW, winE, ps, cs, ns, lap);
      } else {
        laplacians<MASK>(m, win[ps], win[cs], win[ns], lap);
      }

      double nCr, nNb, npd, npl;
      update_cell(P, ad, lap, win[cs], cen[cs], nCr, nNb, npd, npl);

      const int py = 1 + y;
      if (NUC && out_lane) {
        // decide on the stored (storage-rounded) values, as a separate pass
        // would, with the compositions in absolute units; an embed stores
        // xe - xoff, anything else the stored value unchanged
        const double sCr = (double)(T)nCr, sNb = (double)(T)nNb;
        const double aCr = sCr + P.xoff[0], aNb = sNb + P.xoff[1];
        double eCr = aCr, eNb = aNb;
        npd = (double)(T)npd;
        npl = (double)(T)npl;
        nucleate_cell(N, (uint32_t)(py * pitch + 1 + gx), eCr, eNb, npd, npl, S);
        const bool embedded = eCr != aCr || eNb != aNb;
        nCr = embedded ? eCr - P.xoff[0] : sCr;
        nNb = embedded ? eNb - P.xoff[1] : sNb;
      }

      if (out_lane) {
        store_row(oCr, oNb, opd, opl, (size_t)py * row_b, out_lane_b, nCr, nNb, npd, npl);
        store_ghost_images<T, BC>(oCr, oNb, opd, opl, gx, y, Nx, Ny, pitch, nCr, nNb, npd, npl);
      }
    }
  }
}


// ---------------------------------------------------------------------------
// K explicit steps per pass (temporal blocking, K = 2, 3 or 4).  The reference
// advances one step per sequence of launches and so reads and writes every
// field once per step; here a wave marches its strip through K time levels at
// once, so the old fields are read once and the fields K steps later written
// once: 1/K of the HBM traffic per step of the one-step march.
//
// A strip has 64 - 2K output columns and a K-column halo each side.  Level
// l (1..K) is computed on every lane and is valid on lanes l .. 63-l; level K
// is stored, on lanes K .. 63-K.  Level l reads level l-1 through the same DPP
// shifts as the one-step march.
//
// The levels form a pipeline along the march: at iteration t level 0 (the old
// fields, loaded) reaches row y0-K+t and level l computes row y0-K+t-l from
// level l-1's rows y0-K+t-l-1 .. y0-K+t-l+1, the last of which level l-1 has
// just produced.  Level l starts at iteration 2l, so the chunk reads old rows
// y0-K .. y1-1+K and level l covers rows y0-(K-l) .. y1-1+(K-l).  Each level
// keeps a window of rows in registers, the row computed at iteration t in slot
// t % SLOTS; the first 2K iterations (the prologue) are unrolled at compile
// time.
//
// With a window array `lw` in LDS (LW = true, the four-step kernel), each
// level's centre row goes to LDS at the end of an iteration and comes back at
// the next as the row behind: the register windows then hold two live rows
// per level, not three.  Each lane reads back only what it wrote itself, so no
// barrier is needed.  The array holds K levels x 4 values x 64 lanes.
//
// The intermediate levels are exactly what one-step launches would have
// stored: values are rounded to the storage type before the next level uses
// them, and values at positions outside the interior are the images the
// one-step kernel writes into the ghost ring.  Both come out of the index map
// of the old fields (bc_map):
//  - periodic: a halo lane at gx = -1 reads the neighbourhood of column Nx-1;
//  - no-flux: the old fields are read through the even reflection (column -1
//    is column 0, -2 is 1, ...).  The step is pointwise apart from the
//    five-point Laplacian, and the Laplacian of a cell and of its mirror
//    image add the same two values in x (W + E = u[1] + u[0] and u[0] + u[1])
//    and in y, in the same order otherwise; floating-point addition being
//    commutative, every level's value at -1 is its value at 0 bit for bit,
//    which is the ghost copy a one-step launch makes.  So no image needs a
//    fix-up.
// So K steps here give the same result as K one-step launches.  Symmetric
// masks (FIVE, NINE), no nucleation (the caller runs nucleation steps one at a
// time).
//
// Most of a domain is matrix, away from any interface, and the march is bound
// by the FP64 operations it issues (and the power they take), so an iteration
// runs in one of three modes, chosen by the old rows it depends on: the 2K+1
// newest, over the wave's 64 columns.
//  - MATRIX: every |phi| is below PHI_MATRIX.  No level's |phi| can then reach
//    TINY, so p - 1/2 is exactly -1/2 (p_less_half) and M, 1/det M and r - x
//    are the same for all cells of all levels: computed once per wave, by the
//    instructions a cell's own would be.  A solve is 8 operations, not 39.
//  - QUIET: besides, every phi is +0.  The phase updates then give +0 by their
//    own arithmetic, so only the compositions are updated and only the
//    potentials exchanged.
//  - DENSE: the general case, at the cost of the test (seven operations per
//    row of some 430).
// The rows of the prologue are dense or matrix; quiet ones begin behind it.
//
// With FAIR, a wave's priority within its SIMD falls by quarters of its chunk.
// The older of the two waves of a SIMD otherwise wins every issue slot, ends
// early and leaves the other to run alone at two thirds of the pair's rate.
//
// Every mode gives the bits of DENSE: StepParams::matrix_ok says (from bounds
// on the coefficients) that a step multiplies |phi| < TINY by 16 at most, that
// compositions below X_MATRIX keep every product finite (so 0 * G is 0), and
// the test fails on NaN and infinity.
enum Mode { DENSE, MATRIX, QUIET };

template <typename T>
__device__ __forceinline__ bool matrix_row(const Raw<T>& r) {
  return __all(fabs((double)r.pd) < PHI_MATRIX && fabs((double)r.pl) < PHI_MATRIX &&
               fabs((double)r.cr) < X_MATRIX && fabs((double)r.nb) < X_MATRIX);
}
__device__ __forceinline__ int set_bits(float v) { return __float_as_int(v); }
__device__ __forceinline__ int set_bits(double v) { return __double2loint(v) | __double2hiint(v); }

template <typename T, int BC, int K, int DEPTH, int SW, bool LW, bool MODES, Mask MASK,
          bool FAIR>
__device__ __forceinline__ void marchk_impl(
    const T* __restrict__ iCr, const T* __restrict__ iNb, const T* __restrict__ ipd,
    const T* __restrict__ ipl, T* __restrict__ oCr, T* __restrict__ oNb, T* __restrict__ opd,
    T* __restrict__ opl, int Nx, int Ny, int pitch, int strip, int chunk, int rows,
    const StepParams& P, LdsPtr lw) {
  static_assert(K >= 2 && K <= 4, "two to four steps per pass");
  static_assert(MASK == FIVE || MASK == NINE, "symmetric masks");
  // window rows in registers.  Two live rows suffice with the rows behind in
  // LDS; the plain march still rotates three names over six rows, which the
  // register allocator handles best, while the march with modes, three times
  // the code per row, takes the shortest unrolling.
  constexpr int SLOTS = LW && MODES ? 2 : 3;
  constexpr int UNROLL = LW && MODES ? (DEPTH % 2 ? 2 * DEPTH : DEPTH) : pf::UNROLL;
  static_assert(UNROLL % DEPTH == 0 && UNROLL % SLOTS == 0, "ring and window rotate by unrolling");
  // SW output columns per strip (64 - 2K, or fewer where the strips are laid
  // out for a deeper march); lanes K .. K+SW-1 store
  static_assert(SW >= 1 && SW <= WAVE - 2 * K, "strip width");
  const int lane = threadIdx.x & (WAVE - 1);

  const int gx = strip * SW + lane - K;  // interior column of this lane (may be a halo)
  const int px = 1 + bc_map<BC>(gx, Nx);
  const bool out_lane = (lane >= K) && (lane < K + SW) && (gx < Nx);

  const int y0 = chunk * rows;
  const int y1 = min(y0 + rows, Ny);
  if (y0 >= Ny) return;
  const int nrows = y1 - y0;
  const int y_last = y1 - 1 + K;  // last old row the chunk reads

  const uint32_t in_lane = (uint32_t)px * (uint32_t)sizeof(T);
  const uint32_t out_lane_b = (uint32_t)(1 + gx) * (uint32_t)sizeof(T);
  const size_t row_b = (size_t)pitch * sizeof(T);
  auto row_offset = [&](int y) { return (size_t)(1 + bc_map<BC>(y, Ny)) * row_b; };
  auto load = [&](Raw<T>& r, size_t offset) {
    load_row(r, iCr, iNb, ipd, ipl, offset, in_lane);
  };
  const double* m = P.m;
  const Addends ad = addends(P);
  int matrix_rows = 0, quiet_rows = 0;  // old rows of each kind, up to the newest
  auto inspect = [&](const Raw<T>& r) {
    if constexpr (!MODES) return;
    const bool mr = P.matrix_ok && matrix_row(r);
    const bool qr = mr && __all((set_bits(r.pd) | set_bits(r.pl)) == 0);
    matrix_rows = mr ? matrix_rows + 1 : 0;
    quiet_rows = qr ? quiet_rows + 1 : 0;
  };

  // windows: level l (0 = old fields) row of iteration t in slot t % SLOTS
  Point win[K][SLOTS];
  Centre cen[K][SLOTS];
  Raw<T> ring[DEPTH];

  // LDS copy of the row of level l that is behind at the next iteration
  auto put = [&](int l, const Point& v) {
    LdsPtr q = lw + (l * 4) * WAVE + lane;
    q[0] = v.pd;
    q[WAVE] = v.pl;
    q[2 * WAVE] = v.mu0;
    q[3 * WAVE] = v.mu1;
  };
  // level l's row behind (slot sb of the window; in LDS, the centre row of
  // the iteration before)
  auto behind = [&](int l, int sb) -> Point {
    if constexpr (LW) {
      const LdsPtr q = lw + (l * 4) * WAVE + lane;
      return Point{q[0], q[WAVE], q[2 * WAVE], q[3 * WAVE]};
    } else {
      return win[l][sb];
    }
  };

  // a row's values as stored -> its window entry
  Coef matrix;
  auto enter = [&](auto mode, const Raw<T>& r, Point& v, Centre& c) {
    v.pd = mode.value == QUIET ? 0.0 : (double)r.pd;
    v.pl = mode.value == QUIET ? 0.0 : (double)r.pl;
    c.xCr = (double)r.cr;
    c.xNb = (double)r.nb;
    if constexpr (mode.value == DENSE)
      solve(coefficients<T>(ad, v.pd, v.pl), c, v);
    else
      solve(matrix, c, v);
  };
  // the values one step after the centre row of level l's window (slots
  // behind / centre / ahead)
  auto advance = [&](auto mode, int l, int sa, int sc, int sb, double n[4]) {
    const Point S = behind(l, sb);
    const Point& C = win[l][sc];
    const Point& N = win[l][sa];
    if constexpr (mode.value == QUIET) {
      const double lap[2] = {stencil<MASK>(m, S.mu0, C.mu0, N.mu0),
                             stencil<MASK>(m, S.mu1, C.mu1, N.mu1)};
      update_compositions(P, ad, lap, cen[l][sc], n[0], n[1]);
      n[2] = n[3] = 0.0;
    } else {
      double lap[4];
      laplacians<MASK>(m, S, C, N, lap);
      update_cell(P, ad, lap, C, cen[l][sc], n[0], n[1], n[2], n[3]);
    }
  };

  // Levels 1..K-1 at iteration t (slots are compile-time in both callers):
  // level l computes row y0-K+t-l.
  auto middle_levels = [&](auto mode, int sa, int sc, int sb, int lmax_active) {
#pragma unroll
    for (int l = 1; l < K; l++) {
      if (l > lmax_active) break;
      double n[4];
      advance(mode, l - 1, sa, sc, sb, n);
      enter(mode, Raw<T>{(T)n[0], (T)n[1], (T)n[2], (T)n[3]}, win[l][sa], cen[l][sa]);
    }
  };
  // end of iteration t: the centre rows of the levels active before it to
  // LDS, over the rows behind that the iteration has read
  auto put_rows = [&](int sc, int levels) {
    if constexpr (LW) {
#pragma unroll
      for (int l = 0; l < K; l++) {
        if (l >= levels) break;
        put(l, win[l][sc]);
      }
    }
  };

  if constexpr (MODES) matrix = coefficients<T>(ad, 0.0, 0.0);

  // ---- prologue: iterations t = 0 .. 2K-1 (level K not yet active).  Every
  // row the prologue reads, and the ring, is requested before the first is
  // used, so a wave waits for one memory latency at its start, not 2K.
  {
    Raw<T> pro[2 * K];
#pragma unroll
    for (int t = 0; t < 2 * K; t++) load(pro[t], row_offset(y0 - K + t));
#pragma unroll
    for (int j = 0; j < DEPTH; j++) load(ring[j], row_offset(min(y0 + K + j, y_last)));
#pragma unroll
    for (int t = 0; t < 2 * K; t++) {
      const int sa = t % SLOTS, sc = (t + SLOTS - 1) % SLOTS, sb = (t + 1) % SLOTS;
      inspect(pro[t]);
      auto iteration = [&](auto mode) {
        enter(mode, pro[t], win[0][sa], cen[0][sa]);
        middle_levels(mode, sa, sc, sb, t / 2);
      };
      if (MODES && matrix_rows > t)
        iteration(std::integral_constant<Mode, MATRIX>());
      else
        iteration(std::integral_constant<Mode, DENSE>());
      put_rows(sc, (t + 1) / 2);
    }
  }

  // ---- main loop: iteration t = 2K + i, output row y = y0 + i
  for (int ib = 0;; ib += UNROLL) {
    if constexpr (FAIR) {
      if (4 * ib < nrows)
        __builtin_amdgcn_s_setprio(3);
      else if (2 * ib < nrows)
        __builtin_amdgcn_s_setprio(2);
      else if (4 * ib < 3 * nrows)
        __builtin_amdgcn_s_setprio(1);
      else
        __builtin_amdgcn_s_setprio(0);
    }
#pragma unroll
    for (int k = 0; k < UNROLL; k++) {
      if (ib + k >= nrows) return;
      const int y = y0 + ib + k;
      const int sa = (2 * K + k) % SLOTS, sc = (2 * K + k + SLOTS - 1) % SLOTS,
                sb = (2 * K + k + 1) % SLOTS;
      const int rs = k % DEPTH;
      double n[4];
      inspect(ring[rs]);
      auto iteration = [&](auto mode) {
        enter(mode, ring[rs], win[0][sa], cen[0][sa]);  // old row y + K
        load(ring[rs], row_offset(min(y + K + DEPTH, y_last)));
        middle_levels(mode, sa, sc, sb, K - 1);
        // level K: row y
        advance(mode, K - 1, sa, sc, sb, n);
      };
      if (MODES && quiet_rows > 2 * K)
        iteration(std::integral_constant<Mode, QUIET>());
      else if (MODES && matrix_rows > 2 * K)
        iteration(std::integral_constant<Mode, MATRIX>());
      else
        iteration(std::integral_constant<Mode, DENSE>());
      if (out_lane) {
        store_row(oCr, oNb, opd, opl, (size_t)(1 + y) * row_b, out_lane_b, n[0], n[1], n[2],
                  n[3]);
        store_ghost_images<T, BC>(oCr, oNb, opd, opl, gx, y, Nx, Ny, pitch, n[0], n[1], n[2],
                                  n[3]);
      }
      put_rows(sc, K);
    }
  }
}

template <typename T, int BC, int K, int DEPTH, int SW = WAVE - 2 * K, bool LW = false,
          bool MODES = false, Mask MASK = FIVE, bool FAIR = false>
__device__ __forceinline__ void marchk(
    const T* __restrict__ iCr, const T* __restrict__ iNb, const T* __restrict__ ipd,
    const T* __restrict__ ipl, T* __restrict__ oCr, T* __restrict__ oNb, T* __restrict__ opd,
    T* __restrict__ opl, int Nx, int Ny, int pitch, int strip, int chunk, int rows,
    const StepParams& P, LdsPtr lw = nullptr) {
  marchk_impl<T, BC, K, DEPTH, SW, LW, MODES, MASK, FAIR>(
      iCr, iNb, ipd, ipl, oCr, oNb, opd, opl, Nx, Ny, pitch, strip, chunk, rows, P, lw);
}

}  // namespace pf

#pragma clang fp contract(fast)  // the compiler's default for device code
