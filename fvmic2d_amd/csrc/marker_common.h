// Device bodies of the per-marker passes that both the single-instance
// kernels (ops.hip) and the batched ensemble kernels (ensemble.hip) run:
// advectMarkersRK (with subgridTemperatureChanges pass 2 in front of it) and
// subgridTemperatureChanges passes 1 and 2.  Reference expression order kept;
// compiled without contraction.
#pragma once
#include "fvm_internal.h"

// Quotients by a shared divisor.  n / d is rcp(d) refined by two Newton steps, a
// product and a correction: eleven instructions with the operand scaling and the
// special cases, once for each quotient.  A stage has two quotients for each of
// its four spacings, so the refined reciprocal is formed once per spacing and a
// quotient takes three instructions: the bits are those of the division wherever
// that needs no scaling, and where a quotient is not finite the stage takes the
// divisions themselves.
struct Spacing {
  double d, y;
  __device__ __forceinline__ explicit Spacing(double d_) : d(d_) {
    y = __builtin_amdgcn_rcp(d);
    y = __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
    y = __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
  }
  __device__ __forceinline__ double into(double n) const {
    const double q = n * y;
    return __builtin_fma(__builtin_fma(-d, q, n), y, q);
  }
};

// ---- A6: advectMarkersRK (markers.c:1865-2250) --------------------------------
// PER: x periodic (g.per == 1).  The walk may then leave [0, NX-1] by one cell
// (XCMIN = -1, XCMAX = NX-1, markers.c:1908-1915), the staggered x indices are
// not clamped (:1965-1971), node columns wrap, the left-wall ghost rule is off
// (:2014-2023) and the new X is wrapped into [0, LX] (:2225-2231).  The grid
// coordinates are then read at indices -1 .. NX+1 (set by makePeriodic).
// c0x, c0y, X0, Y0: the marker's stored cell and position (the caller reads them, a
// marker ahead where it can).  tail(m, g, X0, Y0, cellX, cellY, wxy) runs once a marker's
// stages are done, with its old position and cell and its new spin.
template <bool PER, class Tail>
__device__ __forceinline__ void advect_marker(int64_t m, const DGrid &g,
    double *__restrict__ MX,
    double *__restrict__ MY,
    double *__restrict__ MVX,
    double *__restrict__ MVY,
    double *__restrict__ Mwxy,
    const double *__restrict__ vx,
    const double *__restrict__ vy,
    const double *__restrict__ wxy,
    BoundaryValues bv,
    double dt,
    double *__restrict__ MT,
    double *__restrict__ MTdot,
    const double *__restrict__ dTn,
    const double *__restrict__ dTsub,
    double dt_thermal, const Tail &tail, int c0x, int c0y, double X0, double Y0) {
  if (!cell_ok(c0x, c0y, g.ncx(), g.NY)) return;
  const int NX = g.NX, NY = g.NY;
  const int XCMAX = PER ? NX - 1 : NX - 2, XCMIN = PER ? -1 : 0;
  // column offset of node ix + 1 from node ix (wraps past the last column)
  auto right = [&](int ix) -> int { return (PER && ix + 1 >= NX) ? 1 - NX : 1; };
  if (MT) {
    // subgridTemperatureChanges.c:89-103 (pass 2) on the same stored cell,
    // fused here because advectMarkersRK starts from that cell too
    const double dx = g.x[c0x + 1] - g.x[c0x];
    const double dy = g.y[c0y + 1] - g.y[c0y];
    const double mdx = (X0 - g.x[c0x]) / dx;
    const double mdy = (Y0 - g.y[c0y]) / dy;
    // the stored cell is inside the grid: all four corners are owned nodes
    const double *d0 = dTn + (int64_t)c0y * NX + c0x, *d1 = d0 + NX;
    const int r0 = right(c0x);
    const double dtm = (d0[0] * (1.0 - mdy) * (1.0 - mdx) + d1[0] * mdy * (1.0 - mdx) + d0[r0] * (1.0 - mdy) * mdx +
                        d1[r0] * mdy * mdx) +
                       dTsub[m];
    MT[m] = MT[m] + dtm;
    MTdot[m] = dtm / dt_thermal;
  }
  double xcur = X0, ycur = Y0;
  // RK4 weights (k1 + 2 k2 + 2 k3 + k4) / 6 (markers.c:2118-2120), summed in the
  // expression's left-to-right order as the stages complete
  double svx = 0.0, svy = 0.0, swxy = 0.0;
  // the stages stay a loop: unrolled, they held 116-126 VGPRs (four waves per
  // SIMD); rolled and held to 96 (five), the forms with the coordinates in LDS and
  // the periodic one with the rotation spill two (a lane writes 8 bytes once: 5.8 of
  // the 291 MB moved by the case below).  At 1.44 M markers on 201 x 201 nodes a stage
  // takes 8-9 us and the columns about 24: 58 us without a tail, 86 with the rotation
  // behind it, the VALU busy 76 % of that.  Without a tail it took 72 (12 a stage) with
  // eight whole divisions, the walk as loops and the three fields' gathers one after
  // another.
  const bool top0 = bv.mechBCTop.type[0] == 0, top1 = bv.mechBCTop.type[0] == 1;
  const bool left0 = bv.mechBCLeft.type[1] == 0, left1 = bv.mechBCLeft.type[1] == 1;
  const double top2 = 2.0 * bv.mechBCTop.value[0], left2 = 2.0 * bv.mechBCLeft.value[1];
#pragma unroll 1
  for (int irk = 0; irk < 4; irk++) {
    // The walk of both axes from the marker's cell.  It rarely passes more than one
    // cell boundary, so the four coordinates around the cell are read together and
    // decide the first step without a branch; a marker that goes further walks on.
    // (Walked step by step, every lane that moved sent its wavefront through the
    // loops of all four directions, each a chain of reads: more of a stage's time
    // than its arithmetic.)  The cell is made opaque so that the coordinates are
    // read per stage and not held over all of them: registers are what bounds the
    // wavefronts in flight.
    int cellX = c0x, cellY = c0y;
    asm volatile("" : "+v"(cellX), "+v"(cellY));
    double xg0, xg1, yg0, yg1;  // the cell's corners
    {
      const int lx = PER ? cellX - 1 : max(cellX - 1, 0), ly = max(cellY - 1, 0);
      const int hx = PER ? cellX + 2 : min(cellX + 2, NX - 1), hy = min(cellY + 2, NY - 1);
      const double xm1 = g.x[lx], x0 = g.x[cellX], x1 = g.x[cellX + 1], x2 = g.x[hx];
      const double ym1 = g.y[ly], y0 = g.y[cellY], y1 = g.y[cellY + 1], y2 = g.y[hy];
      const bool rx = xcur > x1, ry = ycur > y1, bx = !rx && xcur < x0, by = !ry && ycur < y0;
      const int sx = rx ? (cellX < XCMAX ? 1 : 0) : (bx && cellX > XCMIN ? -1 : 0);
      const int sy = ry ? (cellY < NY - 2 ? 1 : 0) : (by && cellY > 0 ? -1 : 0);
      cellX += sx;
      cellY += sy;
      const bool on = (sx > 0 && xcur > x2) || (sx < 0 && xcur < xm1) || (sy > 0 && ycur > y2) || (sy < 0 && ycur < ym1);
      if (on) {
        if (sx > 0)
          while (xcur > g.x[cellX + 1] && cellX < XCMAX) cellX++;
        if (sx < 0)
          while (xcur < g.x[cellX] && cellX > XCMIN) cellX--;
        if (sy > 0)
          while (ycur > g.y[cellY + 1] && cellY < NY - 2) cellY++;
        if (sy < 0)
          while (ycur < g.y[cellY] && cellY > 0) cellY--;
      }
      if (PER && !on) {  // coordinates in memory: what has been read is not read again
        xg0 = sx > 0 ? x1 : (sx < 0 ? xm1 : x0), xg1 = sx > 0 ? x2 : (sx < 0 ? x0 : x1);
        yg0 = sy > 0 ? y1 : (sy < 0 ? ym1 : y0), yg1 = sy > 0 ? y2 : (sy < 0 ? y0 : y1);
      } else {
        xg0 = g.x[cellX], xg1 = g.x[cellX + 1], yg0 = g.y[cellY], yg1 = g.y[cellY + 1];
      }
    }
    // the half cells: cellY in [0, NY-2], cellX in [0, NX-2] (PER: [-1, NX-1]), so
    // the reference's clamps of vxX, vxY, vyX and vyY change nothing
    const int vxX = cellX, vyY = cellY;
    const double xc0 = g.xc[PER ? max(cellX, 0) : cellX], xc1 = g.xc[cellX + 1], xc2 = g.xc[cellX + 2];
    const double yc0 = g.yc[cellY], yc1 = g.yc[cellY + 1], yc2 = g.yc[cellY + 2];
    const bool up = ycur < yc1, left = (!PER || cellX > -1) && xcur < xc1;
    const int vxY = up ? cellY - 1 : cellY, vyX = left ? cellX - 1 : cellX;
    const double xcl = left ? xc0 : xc1, xch = left ? xc1 : xc2, ycl = up ? yc0 : yc1, ych = up ? yc1 : yc2;

    // the twelve nodes, all loads in flight before the arithmetic of any.
    // vx nodes: rows vxY (-1 is the ghost row) and vxY + 1, columns vxX and vxX + 1
    // (both owned: vxX is in [0, NX-2]; when PER the columns wrap).  Loads are
    // unconditional from a valid address; a ghost value is selected away.
    const bool vrow = vxY >= 0;
    const int vxc = PER && vxX < 0 ? vxX + NX : vxX;
    const int vxr = right(vxc);
    const double *vr1 = vx + (int64_t)(vxY + 1) * NX + vxc;
    const double *vr0 = vrow ? vr1 - NX : vr1;
    double vxll, vxlr, vx0, vx1;
    if (PER) {
      vxll = vr1[0], vxlr = vr1[vxr], vx0 = vr0[0], vx1 = vr0[vxr];
    } else {
      const fvm_pair lo = load_pair(vr1), hi = load_pair(vr0);
      vxll = lo.a, vxlr = lo.b, vx0 = hi.a, vx1 = hi.b;
    }
    // vy nodes: columns vyX (-1 is the ghost column; when PER it is column NX-1)
    // and vyX + 1, rows vyY and vyY + 1 (both owned: vyY is in [0, NY-2])
    const bool vcol = PER || vyX >= 0;
    double vyur, vylr, vy0, vy1;
    if (PER) {
      const int vyc = vyX + 1 >= NX ? vyX + 1 - NX : vyX + 1;  // column of vyX + 1
      const int vyl = vyc == 0 ? NX - 1 : -1;                  // offset of column vyX
      const double *q0 = vy + (int64_t)vyY * NX + vyc, *q1 = q0 + NX;
      vyur = q0[0], vylr = q1[0];
      vy0 = q0[vyl], vy1 = q1[vyl];
    } else {
      // both columns of a row in one load: vyX and vyX + 1, or 0 and 1 at the
      // ghost column (where the left value is selected away)
      const double *q0 = vy + (int64_t)vyY * NX + (vcol ? vyX : 0);
      const fvm_pair a = load_pair(q0), b = load_pair(q0 + NX);
      vyur = vcol ? a.b : a.a, vylr = vcol ? b.b : b.a;
      vy0 = a.a, vy1 = b.a;
    }
    // wxy: cellX in [0, NX-2] ([-1, NX-1] wrapped when PER), cellY in [0, NY-2]:
    // four owned nodes
    const int wc = PER && cellX < 0 ? cellX + NX : cellX;
    const int wr = right(wc);
    const double *w0 = wxy + (int64_t)cellY * NX + wc, *w1 = w0 + NX;
    double w00, w01, w10, w11;
    if (PER) {
      w00 = w0[0], w01 = w0[wr], w10 = w1[0], w11 = w1[wr];
    } else {
      const fvm_pair a = load_pair(w0), b = load_pair(w1);
      w00 = a.a, w01 = a.b, w10 = b.a, w11 = b.b;
    }

    // vxX == cellX and vyY == cellY, so qx and qy are also the mdx and mdy of wxy
    // (markers.c:2089-2090: the same operands)
    const double dxm = xcur - xg0, dym = ycur - ycl, dxv = xcur - xcl, dyv = ycur - yg0;
    const double nxy = vxlr * (dxm * dym), nvv = vylr * (dxv * dyv);
    double qx, qyv, qxy, qxv, qy, qvv;
    {
      const Spacing hx(xg1 - xg0), hyc(ych - ycl), hxc(xch - xcl), hy(yg1 - yg0);
      qx = hx.into(dxm);
      qyv = hyc.into(dym);
      qxy = hyc.into(hx.into(nxy));
      qxv = hxc.into(dxv);
      qy = hy.into(dyv);
      qvv = hy.into(hxc.into(nvv));
      // false for an infinity or a NaN in any of them
      if (!(fabs(qx + qyv + qxy + qxv + qy + qvv) < 1e300)) {
        qx = dxm / hx.d;
        qyv = dym / hyc.d;
        qxy = nxy / hx.d / hyc.d;
        qxv = dxv / hxc.d;
        qy = dyv / hy.d;
        qvv = nvv / hxc.d / hy.d;
      }
    }
    // ghost values by the kind of the wall: 0 a given velocity, 1 free slip, else 0
    double vxul = vrow ? vx0 : (top0 ? top2 - vxll : (top1 ? vxll : 0.0));
    double vxur = vrow ? vx1 : (top0 ? top2 - vxlr : (top1 ? vxlr : 0.0));
    double a = vxul * (1.0 - qx) * (1.0 - qyv);
    a += vxur * (qx) * (1.0 - qyv);
    a += vxll * (1.0 - qx) * (qyv);
    a += qxy;
    double vyul = vcol ? vy0 : (left0 ? left2 - vyur : (left1 ? vyur : 0.0));
    double vyll = vcol ? vy1 : (left0 ? left2 - vylr : (left1 ? vylr : 0.0));
    double b = vyul * (1.0 - qxv) * (1.0 - qy);
    b += vyur * (qxv) * (1.0 - qy);
    b += vyll * (1.0 - qxv) * (qy);
    b += qvv;

    double w = (1.0 - qx) * (1.0 - qy) * w00;
    w += (qx) * (1.0 - qy) * w01;
    w += (1.0 - qx) * (qy) * w10;
    w += (qx) * (qy) * w11;
    if (irk == 0) {
      svx = a;
      svy = b;
      swxy = w;
    } else if (irk < 3) {
      svx = svx + 2 * a;
      svy = svy + 2 * b;
      swxy = swxy + 2 * w;
    } else {
      svx = svx + a;
      svy = svy + b;
      swxy = swxy + w;
    }
    if (irk < 3) {
      if (irk < 2) {
        xcur = X0 + dt / 2 * a;
        ycur = Y0 + dt / 2 * b;
      } else {
        xcur = X0 + dt * a;
        ycur = Y0 + dt * b;
      }
    }
  }
  const double VX = svx / 6;
  const double VY = svy / 6;
  const double wm = swxy / 6.0;
  MVX[m] = VX;
  MVY[m] = VY;
  Mwxy[m] = wm;
  double Xn = X0 + dt * VX;
  if (PER) {
    if (Xn > g.LX) Xn -= g.LX;
    else if (Xn < 0) Xn += g.LX;
  }
  MX[m] = Xn;
  MY[m] = Y0 + dt * VY;
  tail(m, g, X0, Y0, c0x, c0y, wm);
}

// ---- A6, second part: the stress rotation by the marker spin (k1 + 2 k2 + 2 k3 +
// k4) / 6 and the strain invariant update (markers.c:2141-2164, 2223).  Behind the
// stages of each marker: their registers are free by then, and the columns stream
// while other wavefronts compute (as a pass of its own it read the cells and the
// spin again: 4 M tracers 743 us a step, so 729; 1.44 M markers 254 either way).
__device__ __forceinline__ void rotate_stress(double &sxx, double &syy, double &sxy, double wm, double dt,
                                              int jaumann) {
  const double msxx0 = sxx, msyy0 = syy, msxy0 = sxy;
  if (jaumann) {
    const double wxy1 = wm * dt;
    sxx = msxx0 + 2.0 * msxy0 * -wxy1;
    syy = msyy0 + 2.0 * msxy0 * wxy1;
    sxy = msxy0 + (msxx0 - msyy0) * wxy1;
  } else {
    const double thetaz = -wm * dt;
    // one shared range reduction per angle (sincos); the values are those of sin and cos
    double c, s, s2, c2;
    sincos(thetaz, &s, &c);
    sincos(2.0 * thetaz, &s2, &c2);
    // pow(v, 2.0) of markers.c:2162-2163: gcc -O3 (makefile:14) folds it to v*v,
    // which is what the reference binary executes
    sxx = msxx0 * (c * c) + msyy0 * (s * s) - msxy0 * s2;
    syy = msxx0 * (s * s) + msyy0 * (c * c) + msxy0 * s2;
    sxy = 0.5 * (msxx0 - msyy0) * s2 + msxy0 * c2;
  }
}

// The rotation behind a marker's advection.
struct RotateTail {
  double *sxx, *syy, *sxy, *Eii;
  const double *exx, *eyy, *exy;
  double dt;
  int jaumann;
  __device__ __forceinline__ void operator()(int64_t m, const DGrid &, double, double, int, int, double wm) const {
    double s11 = sxx[m], s22 = syy[m], s12 = sxy[m];
    rotate_stress(s11, s22, s12, wm, dt, jaumann);
    sxx[m] = s11;
    syy[m] = s22;
    sxy[m] = s12;
    const double e11 = exx[m], e22 = eyy[m], e12 = exy[m];
    Eii[m] = Eii[m] + dt * sqrt(0.5 * (e11 * e11 + e22 * e22) + e12 * e12);
  }
};

// ---- A9: updateMarkerStress (updateMarkerStress.c:5-163): a marker's increments ----
template <int MODE>
__device__ __forceinline__ void stress_increment(const DGrid &g, double X, double Y, int c0x, int c0y,
                                                 const double *__restrict__ dsxx, const double *__restrict__ dsyy,
                                                 const double *__restrict__ dsxy, double &mdsxx, double &mdsyy,
                                                 double &mdsxy) {
  const int NX = g.NX, NY = g.NY, P = g.per;
  int cellX = c0x, cellY = c0y;
  // periodic: the centre cell may step to NX and is then clamped to NX-1
  // (cellXMax NX, then NX-1); node column NX is column 0
  if (cellX < (P ? NX : NX - 2) && X >= g.xc[cellX + 1]) cellX++;
  if (cellY < NY - 1 && Y >= g.yc[cellY + 1]) cellY++;
  if (cellY < 1) cellY = 1;
  else if (cellY > NY - 2) cellY = NY - 2;
  if (cellX < 1) cellX = 1;
  else if (cellX > (P ? NX - 1 : NX - 2)) cellX = P ? NX - 1 : NX - 2;
  double mdx = (X - g.xc[cellX]) / (g.xc[cellX + 1] - g.xc[cellX]);
  double mdy = (Y - g.yc[cellY]) / (g.yc[cellY + 1] - g.yc[cellY]);
  const Bilinear<MODE> at(g, cellY, cellX, mdx, mdy);
  mdsxx = at(dsxx);
  mdsyy = at(dsyy);
  cellX = c0x;
  cellY = c0y;
  if (cellY < 0) cellY = 0;
  else if (cellY > NY - 2) cellY = NY - 2;
  if (cellX < 0) cellX = 0;
  else if (cellX > (P ? NX - 1 : NX - 2)) cellX = P ? NX - 1 : NX - 2;
  mdx = (X - g.x[cellX]) / (g.x[cellX + 1] - g.x[cellX]);
  mdy = (Y - g.y[cellY]) / (g.y[cellY + 1] - g.y[cellY]);
  mdsxy = Bilinear<MODE>(g, cellY, cellX, mdx, mdy)(dsxy);
}

// The stresses of a whole visco-elasto-plastic step behind a marker's advection:
// subgridStressChanges' own change (dxx, dyy, dxy per marker; null: none),
// updateMarkerStress's increment at the old position, the rotation by the new spin
// and the strain invariant, so that the stresses are read and written once.
template <int MODE>
struct StressTail {
  double *sxx, *syy, *sxy, *Eii;
  const double *exx, *eyy, *exy;           // marker strain rates
  const double *dsxx, *dsyy, *dsxy;        // nodal increments
  const double *dxx, *dyy, *dxy;           // per-marker subgrid changes
  double dt;
  int jaumann;
  __device__ __forceinline__ void operator()(int64_t m, const DGrid &g, double X, double Y, int cx, int cy,
                                             double wm) const {
    double s11 = sxx[m], s22 = syy[m], s12 = sxy[m];
    if (dxx) {
      s11 = s11 + dxx[m];
      s22 = s22 + dyy[m];
      s12 = s12 + dxy[m];
    }
    double i11, i22, i12;
    stress_increment<MODE>(g, X, Y, cx, cy, dsxx, dsyy, dsxy, i11, i22, i12);
    s11 = s11 + i11;
    s22 = s22 + i22;
    s12 = s12 + i12;
    rotate_stress(s11, s22, s12, wm, dt, jaumann);
    sxx[m] = s11;
    syy[m] = s22;
    sxy[m] = s12;
    const double e11 = exx[m], e22 = eyy[m], e12 = exy[m];
    Eii[m] = Eii[m] + dt * sqrt(0.5 * (e11 * e11 + e22 * e22) + e12 * e12);
  }
};

// ---- A7: subgridTemperatureChanges pass 2 (subgridTemperatureChanges.c:89-103) ---
template <bool PER>
__device__ __forceinline__ void subgrid_t2_marker(int64_t m, const DGrid &g,
    const double *__restrict__ MX,
    const double *__restrict__ MY,
    double *__restrict__ MT,
    double *__restrict__ MTdot,
    const int32_t *__restrict__ cX,
    const int32_t *__restrict__ cY,
    const double *__restrict__ dT,
    const double *__restrict__ dTsub,
    double dt) {
  const int cellX = cX[m], cellY = cY[m];
  if (!cell_ok(cellX, cellY, g.ncx(), g.NY)) return;
  const double dx = g.x[cellX + 1] - g.x[cellX];
  const double dy = g.y[cellY + 1] - g.y[cellY];
  const double mdx = (MX[m] - g.x[cellX]) / dx;
  const double mdy = (MY[m] - g.y[cellY]) / dy;
  const Corners q = cell_corners<PER>(dT, g.NX, cellY, cellX);
  const double dtm = (q.f00 * (1.0 - mdy) * (1.0 - mdx) + q.f10 * mdy * (1.0 - mdx) + q.f01 * (1.0 - mdy) * mdx +
                      q.f11 * mdy * mdx) +
                     dTsub[m];
  MT[m] = MT[m] + dtm;
  MTdot[m] = dtm / dt;
}
