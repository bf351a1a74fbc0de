// Single-pass 2D MHD step (k_march2d): the program of one wave.
//
// A wave holds 64 / LW strips of LW columns (LW = 64: one strip, LW = 32: two strips side by
// side in its lanes) and marches along y, one row per pass.  The middle LW - 4 columns of a
// strip are its output, two columns of halo on each side are computed again by the
// neighbouring strips.  At row s a lane
//   - turns the prefetched row s+1 into primitives, and computes its corner electric field and
//     the half-step record of its cell at row s (half_step_2d),
//   - solves the EMF of the lower-left corner of its cell (records of rows s-1 and s of its own
//     and of the left column), the y face below it and the x face left of it,
//   - finishes the update + CT of row s-1 (its upper flux and corners are now known), writes it
//     and folds its CFL term, and starts the update of row s (the reference's order
//     +Fx(i) -Fx(i+1) +Fy(j) -Fy(j+1), one partial sum carried per variable).
// So the state is read once and written once, and no record, flux or EMF goes through memory;
// the three-kernel form moves about 900 bytes per cell and step.  A strip of H output rows
// takes H + 2 passes, the first only for the records of the row below it, the last without an
// x face.
//
// Data of other lanes: primitives of rows s and s+1 lie in a two-row LDS ring that belongs to
// the wave (its neighbours' x values are read there, and it keeps 30 registers per lane free
// during the solves); states and fluxes of the left / right column come by lane shifts.  Waves
// never wait for each other: there is no barrier.  The upper-side face values of a cell are
// bit for bit the lower-side values of its +1 neighbour (see fused_body.hpp), so the averages
// of the EMF solver of equal values are exact and the strict build equals the other forms.
//
// References: primitives and half step src/muscl/MHDBaseFunctor2D.h:774-1109, faces, EMF and
// update src/muscl/MHDRunFunctors2D.h:612-686, 1646-1699.
#pragma once

#include "fused_body.hpp"

namespace ppk {
namespace PPK_NS {
namespace march2k {

using namespace fusedk;

constexpr int kWaves = 4;          // waves per block (independent of each other)
constexpr int kRing = 2 * 8 * 64;  // doubles of LDS per wave: Q of rows s and s+1

// LDS writes of this wave before the call are seen by its lanes after it
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// the value of the lane to the left / right (lanes at a strip's edge get a value that no
// output depends on)
__device__ __forceinline__ double from_left(double x) { return __shfl_up(x, 1, 64); }
__device__ __forceinline__ double from_right(double x) { return __shfl_down(x, 1, 64); }

// Fix a value in its register, as a value read from memory is: the compiler neither contracts
// its product into the sums of its users nor keeps its operands alive for that.  Applied to the
// values that the three-kernel form passes through LDS and HBM, it rounds nearly as that form
// does and took the spills of k_march2d from 17 to 6 registers (2048^2: 364 -> 337 us; with the
// leaner solvers 2 are spilled).
__device__ __forceinline__ void settle(double &x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void settle(St<double> &s) {
#pragma unroll
  for (int v = 0; v < 8; ++v) settle(s[v]);
}
// the fields of a record (the lower-side ones)
__device__ __forceinline__ void settle(Half2D<double> &h) {
  for (double *x : {&h.r, &h.pp, &h.u, &h.v, &h.w, &h.A, &h.B, &h.C, &h.drx, &h.dpx, &h.dux,
                    &h.dvx, &h.dwx, &h.dBx, &h.dCx, &h.dry, &h.dpy, &h.duy, &h.dvy, &h.dwy,
                    &h.dAy, &h.dCy, &h.AL, &h.BL, &h.dALy, &h.dBLx})
    settle(*x);
}

// a row of a lane's column as loaded ahead: the state, A of the column to the right and B of
// the row above
struct Row {
  double u[8], ar, bu;
};
__device__ __forceinline__ void load_row(const double *__restrict__ U, const DevParams &p, int ic,
                                         int j, Row &r) {
  const int jc = min(j, p.jsize - 1);
  const long long vs = p.vstride, t = (long long)jc * p.isize + ic;
#pragma unroll
  for (int v = 0; v < 8; ++v) r.u[v] = U[t + v * vs];
  r.ar = U[(long long)jc * p.isize + min(ic + 1, p.isize - 1) + IA * vs];
  r.bu = U[(long long)min(j + 1, p.jsize - 1) * p.isize + ic + IB * vs];
}
__device__ __forceinline__ void row_prims(const Row &r, const DevParams &p, St<double> &q) {
  St<double> u;
#pragma unroll
  for (int v = 0; v < 8; ++v) u[v] = r.u[v];
  constoprim(u, r.ar, r.bu, 0.0, q, p);
  settle(q);
}

// The wave's program: rows [r0, r0 + n) of the strip of this lane (n may be 0 or differ between
// the strips of a wave), `passes` = the largest n of the wave + 2.  i: the lane's column; out:
// the lane is an output column.  Returns the lane's largest CFL term (0 without fold).
template <int RS>
__device__ __forceinline__ double march2d_wave(const double *__restrict__ Uin,
                                               double *__restrict__ Uout, const DevParams &p,
                                               int i, bool out, int r0, int n, int passes,
                                               double dt, bool fold, double *ring) {
  const int lane = threadIdx.x & 63;
  const int ic = min(i, p.isize - 1);  // lanes past the box: clamped, never output
  const int lm = max(lane - 1, 0), lp = min(lane + 1, 63);
  const long long vs = p.vstride;
  const double dtdx = dt / p.dx, dtdy = dt / p.dy;
  // Q of row s in ring slot s & 1 (of this strip's own numbering)
  auto Q = [&](int slot, int v, int l) -> double & { return ring[(slot * 8 + v) * 64 + l]; };

  double best = 0.0;
  Row nx;
  St<double> q;
  double A0, Am, AR0, B0, E0 = 0.0;
  {  // rows s-1 and s of the first pass (s = r0 - 1)
    load_row(Uin, p, ic, r0 - 2, nx);
    Am = nx.u[IA];
    row_prims(nx, p, q);
#pragma unroll
    for (int v = 0; v < 8; ++v) Q(1, v, lane) = q[v];
    Row r;
    load_row(Uin, p, ic, r0 - 1, r);
    load_row(Uin, p, ic, r0, nx);
    A0 = r.u[IA];
    B0 = r.u[IB];
    AR0 = r.ar;
    row_prims(r, p, q);
#pragma unroll
    for (int v = 0; v < 8; ++v) Q(0, v, lane) = q[v];
    wave_sync();
    E0 = elec_z_2d(Q(1, IU, lm), Q(0, IU, lm), Q(1, IU, lane), q[IU], Q(1, IV, lm), Q(0, IV, lm),
                   Q(1, IV, lane), q[IV], Am, A0, from_left(B0), B0);
    settle(E0);
  }
  // carried from row s-1: its cell's upper corner states (the left column's, and its own), the
  // face field part of both, the state at its upper y face; the update of its cell so far
  St<double> rt, lt, qmy;
  double top_a = 0.0, op[5], oc = 0.0, bn_prev = 0.0, ez_prev = 0.0, a_prev = 0.0;
#pragma unroll
  for (int v = 0; v < 8; ++v) rt[v] = lt[v] = qmy[v] = 0.0;
#pragma unroll
  for (int v = 0; v < 5; ++v) op[v] = 0.0;

#pragma unroll 1
  for (int t = 0; t < passes; ++t) {
    const int s = r0 - 1 + t, a = t & 1, b = a ^ 1;  // ring slots of rows s and s+1
    Half2D<double> h;
    double ap, bp, ar;
    {
      St<double> nb[3][3];
      double bf[4][4][3];
#pragma unroll
      for (int v = 0; v < 8; ++v) nb[1][0][v] = Q(b, v, lane);  // row s-1, before s+1 replaces it
      wave_sync();
      ap = nx.u[IA];
      bp = nx.u[IB];
      ar = nx.ar;
      row_prims(nx, p, nb[1][2]);
#pragma unroll
      for (int v = 0; v < 8; ++v) Q(b, v, lane) = nb[1][2][v];
      wave_sync();
      load_row(Uin, p, ic, s + 2, nx);  // a pass ahead
#pragma unroll
      for (int v = 0; v < 8; ++v) {
        nb[0][1][v] = Q(a, v, lm);
        nb[1][1][v] = Q(a, v, lane);
        nb[2][1][v] = Q(a, v, lp);
      }
      double E1 =
          elec_z_2d(nb[0][1][IU], Q(b, IU, lm), nb[1][1][IU], nb[1][2][IU], nb[0][1][IV],
                    Q(b, IV, lm), nb[1][1][IV], nb[1][2][IV], A0, ap, from_left(bp), bp);
      settle(E1);
      const double E0r = from_right(E0);
      bf[1][1][0] = A0;
      bf[1][1][1] = B0;
      bf[2][1][0] = AR0;
      bf[1][2][1] = bp;
      bf[1][2][0] = ap;
      bf[1][0][0] = Am;
      bf[2][1][1] = from_right(B0);
      bf[0][1][1] = from_left(B0);
      // the upper-side fields and their slopes (ERR, bf corners) are not used: they come from
      // the neighbours' lower sides
      bf[2][2][0] = bf[2][0][0] = bf[2][2][1] = bf[0][2][1] = 0.0;
      half_step_2d(nb, bf, E0, E1, E0r, 0.0, dtdx, dtdy, p, h);
      E0 = E1;
    }
    const double a0 = A0, b0 = B0;  // face fields of row s before the step
    Am = A0;
    A0 = ap;
    AR0 = ar;
    B0 = bp;
    settle(h);
    h.AR = h.BR = h.dARy = h.dBRx = 0.0;

    if (t > 0) {
      // corner (i, s): RT of the lower left cell, RB of the left one, LT of the lower one, LB
      double ez;
      {
        St<double> rb = edge_state_2d(h, IRB, p);
        rb[IB] = h.BL + h.dBLx;
#pragma unroll
        for (int v = 0; v < 8; ++v)
          if (v != IA) rb[v] = from_left(rb[v]);
        rb[IA] = h.AL + -h.dALy;
        const St<double> lb = edge_state_2d(h, ILB, p);
        rt[IA] = top_a;
        lt[IA] = top_a;
        rt[IB] = rb[IB];
        lt[IB] = lb[IB];
        ez = compute_emf<EMFZ>(rt, rb, lt, lb, p);
        settle(ez);
      }
      const double bn = b0 - (from_right(ez) - ez) * dtdx;  // new B of row s
      // y face below row s
      St<double> f;
      {
        St<double> ql = qmy, qr = face_state_2d(h, 1, -1, p);
        ql[IB] = h.BL;
        swap_dir(ql, IU, IV); swap_dir(ql, IA, IB);
        swap_dir(qr, IU, IV); swap_dir(qr, IA, IB);
        riemann_mhd_rs<RS>(ql, qr, f, p);
        settle(f);
      }
      if (t > 1) {  // finish row s-1
        St<double> u;
        u[ID] = op[0] - f[ID] * dtdy;
        u[IP] = op[1] - f[IP] * dtdy;
        u[IU] = op[2] - f[IV] * dtdy;
        u[IV] = op[3] - f[IU] * dtdy;
        u[IW] = op[4] - f[IW] * dtdy;
        u[IC] = oc - f[IC] * dtdy;
        u[IA] = a_prev + (ez - ez_prev) * dtdy;
        u[IB] = bn_prev;
        const double ax = from_right(u[IA]);
        if (out && t - 2 < n) {
          const long long c = (long long)(s - 1) * p.isize + i;
#pragma unroll
          for (int v = 0; v < 8; ++v) Uout[c + v * vs] = u[v];
          if (fold) {
            // new face fields of the +1 neighbours; past the last cell the next ghost fill's
            // (where both faces of a direction are periodic, a ghost column / row has its image's
            // records, hence its CT value; other periodic upper faces: march_folds_cfl)
            double mx = ax, my = bn;
            if (i + 1 == p.isize - p.gw && p.bc[1] != PPK_BC_PERIODIC)
              mx = p.bc[1] == PPK_BC_DIRICHLET ? -u[IA] : u[IA];
            if (s == p.jsize - p.gw && p.bc[3] != PPK_BC_PERIODIC)
              my = p.bc[3] == PPK_BC_DIRICHLET ? -u[IB] : u[IB];
            St<double> qn;
            constoprim(u, mx, my, 0.0, qn, p);
            best = fmax(best, inv_dt_cell(qn, p));
          }
        }
      }
      if (t + 1 < passes) {  // x face left of row s, start of its update
        const long long c = (long long)min(s, p.jsize - 1) * p.isize + ic;
        op[0] = Uin[c + ID * vs];
        op[1] = Uin[c + IP * vs];
        op[2] = Uin[c + IU * vs];
        op[3] = Uin[c + IV * vs];
        op[4] = Uin[c + IW * vs];
        oc = Uin[c + IC * vs];
        St<double> g, ql = face_state_2d(h, 0, +1, p), qr = face_state_2d(h, 0, -1, p);
#pragma unroll
        for (int v = 0; v < 8; ++v)
          if (v != IA) ql[v] = from_left(ql[v]);
        ql[IA] = h.AL;
        riemann_mhd_rs<RS>(ql, qr, g, p);
        settle(g);
        auto start = [&](double o, double fx, double fy) {
          o += fx * dtdx;
          o -= from_right(fx) * dtdx;
          o += fy * dtdy;
          return o;
        };
        op[0] = start(op[0], g[ID], f[ID]);
        op[1] = start(op[1], g[IP], f[IP]);
        op[2] = start(op[2], g[IU], f[IV]);
        op[3] = start(op[3], g[IV], f[IU]);
        op[4] = start(op[4], g[IW], f[IW]);
        oc = start(oc, g[IC], f[IC]);
        bn_prev = bn;
        ez_prev = ez;
        a_prev = a0;
      }
    }
    // upper states of row s
    rt = edge_state_2d(h, IRT, p);
#pragma unroll
    for (int v = 0; v < 8; ++v)
      if (v != IA && v != IB) rt[v] = from_left(rt[v]);
    lt = edge_state_2d(h, ILT, p);
    top_a = h.AL + h.dALy;
    qmy = face_state_2d(h, 1, +1, p);
  }
  return best;
}

// strip `t` of a grid (x fastest): its first column and rows
struct Geom {
  int lw, rows;   // columns per strip (lanes), output rows per strip
  int nsx, nsy;   // strips
  PPK_HD int waves() const { return (nsx * nsy + 64 / lw - 1) / (64 / lw); }
};
PPK_HD Geom geom_of(const DevParams &p) {
  Geom g;
  g.lw = p.march_lw;
  g.rows = p.march_rows;
  g.nsx = (p.nx + g.lw - 5) / (g.lw - 4);
  g.nsy = (p.ny + g.rows - 1) / g.rows;
  return g;
}

// wave w of a grid: its strips, marched; returns the wave's largest CFL term in every lane
template <int RS>
__device__ __forceinline__ double march2d(const double *__restrict__ Uin,
                                          double *__restrict__ Uout, const DevParams &p,
                                          const Geom &g, int w, double dt, bool fold,
                                          double *ring) {
  const int lane = threadIdx.x & 63, per = 64 / g.lw;
  const int strip = w * per + lane / g.lw, col = lane % g.lw;
  const int sy = strip / g.nsx, sx = strip - sy * g.nsx;
  const bool live = sy < g.nsy;
  const int i = p.gw + sx * (g.lw - 4) + col - 2;
  const int r0 = p.gw + min(sy, g.nsy - 1) * g.rows;
  const int n = live ? min(g.rows, p.gw + p.ny - r0) : 0;
  const bool out = live && col >= 2 && col < g.lw - 2 && i < p.gw + p.nx;
  const int passes = min(g.rows, p.ny) + 2;
  double best = march2d_wave<RS>(Uin, Uout, p, i, out, r0, n, passes, dt, fold, ring);
  if (fold)
    for (int off = 32; off > 0; off >>= 1) best = fmax(best, __shfl_xor(best, off, 64));
  return best;
}

}  // namespace march2k
}  // namespace PPK_NS
}  // namespace ppk
