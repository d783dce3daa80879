// Preconditioners of the nodal solves' BiCGStab (pressure_guess.hip): y = M b for
// a 5-point system whose rows are divided by their diagonal (unit diagonal,
// couplings e, w, s, n; a row without couplings is solved by its right-hand side).
//
// Jacobi alone needs hundreds to thousands of iterations on the Poisson problem
// of the pressure guess (1304 at 257x257), each five short kernels bound by launch
// and reduction latency.  Two preconditioners replace it:
//
// * a multigrid V-cycle: FV_NU Chebyshev-Jacobi sweeps before and after the coarse
//   correction, cells aggregated in pairs along each axis (along one axis only
//   while its couplings are much the stronger), the coarse couplings rediscretised
//   from the aggregated ones (divided by the grown distance), restriction by sums,
//   prolongation bilinear.  6 iterations at 257x257 (solve 31.7 -> 0.85 ms).
// * where every row is dominated by its diagonal (an energy equation with a
//   moderate time step) the same polynomial at degree FV_POLY on the finest
//   level alone, over the interval the row sums give: 5 iterations instead of 40
//   at 801x401 (assembly and solve 1.67 -> 0.39 ms).
//
// What bounds them is latency, so a kernel does as much as its tile allows: a
// tile and a halo as wide as the number of sweeps are read once, all sweeps run in
// LDS (the halo is swept redundantly: 2.3 times the tile's points), everything
// below FV_COARSE_MAX points is one workgroup's kernel, and around the one-level
// polynomial the whole iteration is three kernels.
#include <new>

#include "bicgstab.h"

namespace {

constexpr int FV_NU = 4;        // sweeps on each side of the coarse correction
constexpr int FV_POLY = 8;      // degree of the one-level preconditioner
constexpr int FV_T = 16;        // tile of the level kernels
constexpr int FV_R = FV_T + 2 * FV_NU;
constexpr int FV_PT = FVM_ONE_TILE;  // tile of the one-level kernels
constexpr int FV_PR = FV_PT + 2 * FV_POLY;
// points of the finest level that the one-workgroup kernel takes: 33 x 33 and the
// levels below cost 22 us, 65 x 65 44 us against 9 for two more level kernels
constexpr int FV_COARSE_MAX = 1100;
constexpr int FV_CT = 512;      // threads of the coarse kernel
constexpr int FV_CLEVELS = 16;
constexpr int FV_LEVELS = 64;
constexpr int FV_LAST = 12;     // sweeps on the last level

struct Coefs {
  const double *e, *w, *s, *n;
};

// Chebyshev steps d = c1 d + c2 r, x += d for the spectrum [a, b].  A row without
// couplings starts at its solution x = b with d = 0: its residual is 0 and the
// steps leave it there without a branch.
struct Cheb {
  double c1[16], c2[16];
};

struct Pt {
  double e, w, s, n;
  __device__ __forceinline__ bool live() const { return (fabs(e) + fabs(w)) + (fabs(s) + fabs(n)) != 0.0; }
};
__device__ __forceinline__ Pt load_pt(const Coefs &c, bool in, int64_t i) {
  Pt p = {0.0, 0.0, 0.0, 0.0};
  if (in) p = Pt{c.e[i], c.w[i], c.s[i], c.n[i]};
  return p;
}

// ---- one level: the polynomial p(A), with the iteration around it --------------------
// 1024 threads sweep a 48x48 region for a 32x32 tile: FV_POLY - 1 sweeps and the
// product with A need a halo of FV_POLY.
struct Region {
  static constexpr int RW = FV_PR + 2, NP = FV_PR * FV_PR, PTS = (NP + 1023) / 1024;
  Pt p[PTS];
  int i[PTS];   // node, or -1 outside the grid
  int at[PTS];  // place in LDS, or -1

  __device__ __forceinline__ bool own(int k) const {  // of the tile
    const int q = threadIdx.x + 1024 * k, ry = q / FV_PR, rx = q - ry * FV_PR;
    return i[k] >= 0 && rx >= FV_POLY && rx < FV_POLY + FV_PT && ry >= FV_POLY && ry < FV_POLY + FV_PT;
  }

  __device__ __forceinline__ void place(int NX, int NY, const Coefs &c) {
#pragma unroll
    for (int k = 0; k < PTS; k++) {
      const int q = threadIdx.x + 1024 * k, ry = q / FV_PR, rx = q - ry * FV_PR;
      const int ix = (int)blockIdx.x * FV_PT - FV_POLY + rx, iy = (int)blockIdx.y * FV_PT - FV_POLY + ry;
      const bool in = q < NP && ix >= 0 && ix < NX && iy >= 0 && iy < NY;
      i[k] = in ? iy * NX + ix : -1;
      at[k] = q < NP ? (ry + 1) * RW + rx + 1 : -1;
      p[k] = load_pt(c, in, i[k]);
    }
  }
  // x = p(A) b, then ax = A x of the tile's points; sh zeroed before
  __device__ __forceinline__ void poly(const Cheb &ch, double (*sh)[RW * RW], const double *b, double *x, double *ax) {
    double d[PTS];
#pragma unroll
    for (int k = 0; k < PTS; k++) {
      const bool live = p[k].live();
      d[k] = live ? b[k] * ch.c2[0] : 0.0;
      x[k] = live ? d[k] : b[k];
      if (at[k] >= 0) sh[0][at[k]] = x[k];
    }
    __syncthreads();
#pragma unroll 1
    for (int t = 1; t < FV_POLY; t++) {
      const double *xs = sh[(t - 1) & 1];
      double *xn = sh[t & 1];
#pragma unroll
      for (int k = 0; k < PTS; k++) {
        if (at[k] < 0) continue;
        const int a = at[k];
        const double r = b[k] - (x[k] + p[k].e * xs[a + 1] + p[k].w * xs[a - 1] + p[k].s * xs[a + RW] + p[k].n * xs[a - RW]);
        d[k] = ch.c1[t] * d[k] + ch.c2[t] * r;
        x[k] += d[k];
        xn[a] = x[k];
      }
      __syncthreads();
    }
    const double *xs = sh[(FV_POLY - 1) & 1];
#pragma unroll
    for (int k = 0; k < PTS; k++) {
      const int a = at[k];
      ax[k] = own(k) ? x[k] + p[k].e * xs[a + 1] + p[k].w * xs[a - 1] + p[k].s * xs[a + RW] + p[k].n * xs[a - RW] : 0.0;
    }
  }
};

// sum over the 1024 threads of a block, the same bits in every thread
__device__ __forceinline__ double total_1024(double v) {
  __shared__ double sh[16];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0.0;
#pragma unroll
  for (int k = 0; k < 16; k++) t += sh[k];
  return t;
}
__device__ __forceinline__ double parts_1024(const double *__restrict__ part, int n) {
  double s = 0.0;
  for (int k = threadIdx.x; k < n; k += 1024) s += part[k];
  return total_1024(s);
}

// p = r + beta (p - omega v), y = p(A) p, v = A y; partials of (rhat, v).  p and v
// are read in the halo too, so the new ones go to other arrays.
// (8 waves per SIMD: two blocks a CU, so that 801 x 401's 338 run at once)
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(8))) k_one_p(int NX, int NY, Coefs c, Cheb ch, FvmBcgOne O) {
  __shared__ double sh[2][Region::RW * Region::RW];
  // an iteration enqueued behind the last one: k_one_x has written no partials since
  if (O.sc[FVM_S_DONE] != 0.0) return;
  const double rho = parts_1024(O.prho, O.n_r), rr = parts_1024(O.prr, O.n_r);
  const bool lead = blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0;
  const double bb = O.first ? rr : O.sc[FVM_S_BB];
  if (fvm_bcg_done(rr, bb, O.rtol)) {
    if (lead) O.sc[FVM_S_DONE] = 1.0, O.sc[FVM_S_RR] = rr, O.sc[FVM_S_BB] = bb;
    return;
  }
  for (int k = threadIdx.x; k < 2 * Region::RW * Region::RW; k += 1024) (&sh[0][0])[k] = 0.0;
  const double omega = O.sc[FVM_S_OMEGA], beta = fvm_bcg_beta(O.first, rho, O.sc);
  Region R;
  R.place(NX, NY, c);
  double b[Region::PTS], y[Region::PTS], v[Region::PTS];
#pragma unroll
  for (int k = 0; k < Region::PTS; k++) {
    const int i = R.i[k];
    b[k] = i >= 0 ? O.r[i] + beta * (O.p[i] - omega * O.v[i]) : 0.0;
  }
  __syncthreads();
  R.poly(ch, sh, b, y, v);
  double d = 0.0;
#pragma unroll
  for (int k = 0; k < Region::PTS; k++)
    if (R.own(k)) {
      const int i = R.i[k];
      O.p_new[i] = b[k];
      O.y[i] = y[k];
      O.v_new[i] = v[k];
      d += O.rh[i] * v[k];
    }
  const double t = total_1024(d);
  if (threadIdx.x == 0) O.prv[blockIdx.y * gridDim.x + blockIdx.x] = t;
  if (lead) {
    O.sc[FVM_S_RHO] = rho, O.sc[FVM_S_BB] = bb, O.sc[FVM_S_RR] = rr, O.sc[FVM_S_DONE] = 0.0;
    O.sc[FVM_S_ITS] = O.first ? 1.0 : O.sc[FVM_S_ITS] + 1.0;
  }
}

// alpha = rho / (rhat, v), x += alpha y, s = r - alpha v, z = p(A) s, t = A z;
// partials of (t, s) and (t, t)
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(8))) k_one_s(int NX, int NY, Coefs c, Cheb ch, FvmBcgOne O) {
  __shared__ double sh[2][Region::RW * Region::RW];
  if (O.sc[FVM_S_DONE] != 0.0) return;
  const double rv = parts_1024(O.prv, gridDim.x * gridDim.y), alpha = rv != 0.0 ? O.sc[FVM_S_RHO] / rv : 0.0;
  for (int k = threadIdx.x; k < 2 * Region::RW * Region::RW; k += 1024) (&sh[0][0])[k] = 0.0;
  Region R;
  R.place(NX, NY, c);
  double b[Region::PTS], z[Region::PTS], t[Region::PTS];
#pragma unroll
  for (int k = 0; k < Region::PTS; k++) {
    const int i = R.i[k];
    b[k] = i >= 0 ? O.r[i] - alpha * O.v_new[i] : 0.0;
  }
  __syncthreads();
  R.poly(ch, sh, b, z, t);
  double ts = 0.0, tt = 0.0;
#pragma unroll
  for (int k = 0; k < Region::PTS; k++)
    if (R.own(k)) {
      const int i = R.i[k];
      O.x[i] += alpha * O.y[i];
      O.s[i] = b[k];
      O.z[i] = z[k];
      O.t[i] = t[k];
      ts += t[k] * b[k];
      tt += t[k] * t[k];
    }
  const double a = total_1024(ts), e = total_1024(tt);
  if (threadIdx.x == 0) {
    O.pts[blockIdx.y * gridDim.x + blockIdx.x] = a;
    O.ptt[blockIdx.y * gridDim.x + blockIdx.x] = e;
  }
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) O.sc[FVM_S_ALPHA] = alpha;
}

// omega = (t, s) / (t, t), x += omega z, r = s - omega t; partials of (rhat, r), (r, r)
__global__ void __launch_bounds__(1024) k_one_x(int64_t n, int n_t, FvmBcgOne O) {
  if (O.sc[FVM_S_DONE] != 0.0) return;
  const double ts = parts_1024(O.pts, n_t), tt = parts_1024(O.ptt, n_t), omega = tt != 0.0 ? ts / tt : 0.0;
  double a = 0.0, b = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * 1024 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 1024) {
    O.x[i] += omega * O.z[i];
    const double r = O.s[i] - omega * O.t[i];
    O.r[i] = r;
    a += O.rh[i] * r;
    b += r * r;
  }
  const double ta = total_1024(a), tb = total_1024(b);
  if (threadIdx.x == 0) O.prho[blockIdx.x] = ta, O.prr[blockIdx.x] = tb;
  if (blockIdx.x == 0 && threadIdx.x == 0) O.sc[FVM_S_OMEGA] = omega, O.sc[FVM_S_RHO_OLD] = O.sc[FVM_S_RHO];
}

// ---- multigrid ------------------------------------------------------------------------
struct Lv {
  int NX, NY;
  int fx, fy;       // aggregation to the next level: 2 pairs (2I-1, 2I), 1 none
  int NXc, NYc;
  Coefs c;
  const double *idc;  // 1 / diagonal of the next level's rows before their scaling
};

__device__ __forceinline__ int agg(int i, int f) { return f == 2 ? (i + 1) >> 1 : i; }
// fine indices in aggregate I of an axis with N indices
__device__ __forceinline__ int agg_count(int I, int f, int N) {
  return f == 2 && I > 0 && 2 * I < N ? 2 : 1;
}

__device__ __forceinline__ double row_residual(const Pt &p, double b, const double *xs, int a, int w) {
  return b - (xs[a] + p.e * xs[a + 1] + p.w * xs[a - 1] + p.s * xs[a + w] + p.n * xs[a - w]);
}

// x = FV_NU sweeps from 0, then the residual summed over the aggregates
__global__ void __launch_bounds__(FV_R *FV_R) k_down(Lv L, Cheb ch, const double *__restrict__ b, double *__restrict__ x,
                                                     double *__restrict__ bc, const double *__restrict__ sc) {
  if (sc[FVM_S_DONE] != 0.0) return;
  constexpr int RW = FV_R + 2;
  __shared__ double sh[2][RW * RW];
  const int t = threadIdx.x, ry = t / FV_R, rx = t - ry * FV_R;
  for (int k = t; k < 2 * RW * RW; k += FV_R * FV_R) (&sh[0][0])[k] = 0.0;
  // tiles start on an aggregate's first index
  const int fx0 = blockIdx.x * FV_T - (L.fx == 2 ? 1 : 0), fy0 = blockIdx.y * FV_T - (L.fy == 2 ? 1 : 0);
  const int ix = fx0 - FV_NU + rx, iy = fy0 - FV_NU + ry;
  const bool in = ix >= 0 && ix < L.NX && iy >= 0 && iy < L.NY;
  const int64_t i = (int64_t)iy * L.NX + ix;
  const Pt p = load_pt(L.c, in, i);
  const double bb = in ? b[i] : 0.0;
  const bool live = p.live();
  double d = live ? bb * ch.c2[0] : 0.0, xv = live ? d : bb;
  const int a = (ry + 1) * RW + rx + 1;
  __syncthreads();
  sh[0][a] = xv;
  __syncthreads();
#pragma unroll
  for (int s = 1; s < FV_NU; s++) {
    const double r = row_residual(p, bb, sh[(s - 1) & 1], a, RW);
    d = ch.c1[s] * d + ch.c2[s] * r;
    xv += d;
    sh[s & 1][a] = xv;
    __syncthreads();
  }
  const double r = row_residual(p, bb, sh[(FV_NU - 1) & 1], a, RW);
  const bool own = in && rx >= FV_NU && rx < FV_NU + FV_T && ry >= FV_NU && ry < FV_NU + FV_T;
  if (own) x[i] = xv;
  sh[FV_NU & 1][a] = own ? r : 0.0;
  __syncthreads();
  const int cw = FV_T / L.fx, chh = FV_T / L.fy;
  if (t < cw * chh) {
    const int cy = t / cw, cx = t - cy * cw;
    const int I = blockIdx.x * cw + cx, J = blockIdx.y * chh + cy;
    if (I < L.NXc && J < L.NYc) {
      const double *rs = sh[FV_NU & 1] + (cy * L.fy + FV_NU + 1) * RW + cx * L.fx + FV_NU + 1;
      double v = rs[0];
      if (L.fx == 2) v += rs[1];
      if (L.fy == 2) v += L.fx == 2 ? rs[RW] + rs[RW + 1] : rs[RW];
      const int64_t k = (int64_t)J * L.NXc + I;
      bc[k] = v * L.idc[k];
    }
  }
}

// value of the coarse correction ec at fine index (ix, iy): bilinear, an axis
// without a coupling towards the neighbouring aggregate takes its own value
template <class Get>
__device__ __forceinline__ double prolong(const Lv &L, const Pt &p, int ix, int iy, Get ec) {
  const int I = agg(ix, L.fx), J = agg(iy, L.fy);
  int In = I, Jn = J;
  double wx = 0.0, wy = 0.0;
  if (L.fx == 2) {
    const bool lo = ix & 1;
    if ((lo ? p.w : p.e) != 0.0) In = lo ? I - 1 : I + 1, wx = 0.25;
    if (In < 0 || In >= L.NXc) In = I;
  }
  if (L.fy == 2) {
    const bool lo = iy & 1;
    if ((lo ? p.n : p.s) != 0.0) Jn = lo ? J - 1 : J + 1, wy = 0.25;
    if (Jn < 0 || Jn >= L.NYc) Jn = J;
  }
  const double top = (1.0 - wx) * ec(I, J) + wx * ec(In, J);
  const double bot = (1.0 - wx) * ec(I, Jn) + wx * ec(In, Jn);
  return (1.0 - wy) * top + wy * bot;
}

// out = FV_NU sweeps from x + P ec
__global__ void __launch_bounds__(FV_R *FV_R) k_up(Lv L, Cheb ch, const double *__restrict__ b, const double *__restrict__ x,
                                                   const double *__restrict__ ec, double *__restrict__ out,
                                                   const double *__restrict__ sc) {
  if (sc[FVM_S_DONE] != 0.0) return;
  constexpr int RW = FV_R + 2;
  __shared__ double sh[2][RW * RW];
  const int t = threadIdx.x, ry = t / FV_R, rx = t - ry * FV_R;
  for (int k = t; k < 2 * RW * RW; k += FV_R * FV_R) (&sh[0][0])[k] = 0.0;
  const int ix = (int)blockIdx.x * FV_T - FV_NU + rx, iy = (int)blockIdx.y * FV_T - FV_NU + ry;
  const bool in = ix >= 0 && ix < L.NX && iy >= 0 && iy < L.NY;
  const int64_t i = (int64_t)iy * L.NX + ix;
  const Pt p = load_pt(L.c, in, i);
  const double bb = in ? b[i] : 0.0;
  const bool live = p.live();
  double xv = in ? x[i] : 0.0, d = 0.0;
  if (live) xv += prolong(L, p, ix, iy, [&](int I, int J) { return ec[(int64_t)J * L.NXc + I]; });
  const int a = (ry + 1) * RW + rx + 1;
  __syncthreads();
  sh[0][a] = xv;
  __syncthreads();
#pragma unroll
  for (int s = 0; s < FV_NU; s++) {
    const double r = row_residual(p, bb, sh[s & 1], a, RW);
    d = ch.c1[s] * d + ch.c2[s] * r;
    xv += d;
    sh[(s + 1) & 1][a] = xv;
    __syncthreads();
  }
  if (in && rx >= FV_NU && rx < FV_NU + FV_T && ry >= FV_NU && ry < FV_NU + FV_T) out[i] = xv;
}

// The levels of at most FV_COARSE_MAX points in one workgroup: their rows, right-hand
// sides and two copies of x (a sweep reads one and writes the other) lie in LDS,
// between zeros wide enough for the stencil's reach (a missing neighbour's
// coefficient is 0).
struct CoarseArgs {
  int n;
  Lv lv[FV_CLEVELS];
  int off[FV_CLEVELS];  // of point 0 in the LDS arrays
  int total;            // doubles per LDS array
};
constexpr int FV_LDS = 2400;  // doubles per array (e, w, s, n, b, x, x, 1/diagonal)

struct CoarseLv {
  int NX, np, off;
};
// STEPS sweeps on level v from x in lds[6], or from 0 (ZERO); the sweeps alternate
// between lds[5] and lds[6] and end in lds[6] (from 0, the first only fills lds[5])
template <int STEPS, bool ZERO>
__device__ __forceinline__ void coarse_sweep(const CoarseLv &v, const Cheb &ch, double (*lds)[FV_LDS]) {
  static_assert(STEPS % 2 == 0, "coarse_sweep ends in lds[6]");
  constexpr int PTS = (FV_COARSE_MAX + FV_CT - 1) / FV_CT;
  Pt p[PTS];
  double d[PTS], xv[PTS], b[PTS];
#pragma unroll
  for (int k = 0; k < PTS; k++) {
    const int q = threadIdx.x + FV_CT * k, a = v.off + q;
    d[k] = 0.0;
    if (q < v.np) {
      p[k] = Pt{lds[0][a], lds[1][a], lds[2][a], lds[3][a]};
      b[k] = lds[4][a];
      if (ZERO) {
        const bool live = p[k].live();
        d[k] = live ? b[k] * ch.c2[0] : 0.0;
        xv[k] = live ? d[k] : b[k];
        lds[5][a] = xv[k];
      } else {
        xv[k] = lds[6][a];
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int s = ZERO ? 1 : 0; s < STEPS; s++) {
    const double *xs = lds[s & 1 ? 5 : 6];
    double *xn = lds[s & 1 ? 6 : 5];
#pragma unroll
    for (int k = 0; k < PTS; k++) {
      const int q = threadIdx.x + FV_CT * k, a = v.off + q;
      if (q < v.np) {
        d[k] = ch.c1[s] * d[k] + ch.c2[s] * row_residual(p[k], b[k], xs, a, v.NX);
        xv[k] += d[k];
        xn[a] = xv[k];
      }
    }
    __syncthreads();
  }
}

__global__ void __launch_bounds__(FV_CT) k_coarse(CoarseArgs A, Cheb ch, Cheb last,
                                                  const double *__restrict__ bin, double *__restrict__ xout,
                                                  const double *__restrict__ sc) {
  if (sc[FVM_S_DONE] != 0.0) return;
  __shared__ double lds[8][FV_LDS];
  // every level's rows, all loads of a thread in flight together
  for (int k = threadIdx.x; k < A.total; k += FV_CT) {
    int l = 0;
    while (l + 1 < A.n && k >= A.off[l + 1] - (A.lv[l + 1].NX + 1)) l++;
    const Lv &L = A.lv[l];
    const int q = k - A.off[l];
    const bool in = q >= 0 && q < L.NX * L.NY;
    const Pt p = load_pt(L.c, in, q);
    lds[0][k] = p.e, lds[1][k] = p.w, lds[2][k] = p.s, lds[3][k] = p.n;
    lds[4][k] = in && l == 0 ? bin[q] : 0.0;
    lds[5][k] = lds[6][k] = 0.0;
    lds[7][k] = in && l ? A.lv[l - 1].idc[q] : 0.0;
  }
  __syncthreads();
#pragma unroll 1
  for (int l = 0; l + 1 < A.n; l++) {
    const Lv &L = A.lv[l];
    const int o = A.off[l], oc = A.off[l + 1];
    coarse_sweep<FV_NU, true>(CoarseLv{L.NX, L.NX * L.NY, o}, ch, lds);
    for (int q = threadIdx.x; q < L.NXc * L.NYc; q += FV_CT) {
      const int J = q / L.NXc, I = q - J * L.NXc;
      const int i0 = L.fx == 2 ? (I ? 2 * I - 1 : 0) : I, j0 = L.fy == 2 ? (J ? 2 * J - 1 : 0) : J;
      const int ni = agg_count(I, L.fx, L.NX), nj = agg_count(J, L.fy, L.NY);
      double v = 0.0;
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int i = 0; i < 2; i++) {
          if (i >= ni || j >= nj) continue;
          const int a = o + (j0 + j) * L.NX + i0 + i;
          const Pt p = {lds[0][a], lds[1][a], lds[2][a], lds[3][a]};
          v += row_residual(p, lds[4][a], lds[6], a, L.NX);
        }
      lds[4][oc + q] = v * lds[7][oc + q];
    }
    __syncthreads();
  }
  {
    const Lv &L = A.lv[A.n - 1];
    coarse_sweep<FV_LAST, true>(CoarseLv{L.NX, L.NX * L.NY, A.off[A.n - 1]}, last, lds);
  }
#pragma unroll 1
  for (int l = A.n - 2; l >= 0; l--) {
    const Lv &L = A.lv[l];
    const int o = A.off[l], oc = A.off[l + 1];
    for (int q = threadIdx.x; q < L.NX * L.NY; q += FV_CT) {
      const int a = o + q, iy = q / L.NX, ix = q - iy * L.NX;
      const Pt p = {lds[0][a], lds[1][a], lds[2][a], lds[3][a]};
      if (p.live()) lds[6][a] += prolong(L, p, ix, iy, [&](int I, int J) { return lds[6][oc + J * L.NXc + I]; });
    }
    __syncthreads();
    coarse_sweep<FV_NU, false>(CoarseLv{L.NX, L.NX * L.NY, o}, ch, lds);
  }
  for (int q = threadIdx.x; q < A.lv[0].NX * A.lv[0].NY; q += FV_CT) xout[q] = lds[6][A.off[0] + q];
}

// The next level's rows.  A coupling between aggregates is the sum of the fine
// ones over the grown distance between their centres (2 fine steps instead of 1
// between two pairs); one to a row without couplings of its own (a boundary value,
// the pinned cell) stays on the diagonal; the row sums (a time derivative) add up.
__global__ void __launch_bounds__(256) k_coarsen(Lv L, double *__restrict__ ce, double *__restrict__ cw,
                                                 double *__restrict__ cs, double *__restrict__ cn,
                                                 double *__restrict__ idc) {
  const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (q >= (int64_t)L.NXc * L.NYc) return;
  const int J = (int)(q / L.NXc), I = (int)(q - (int64_t)J * L.NXc);
  const int i0 = L.fx == 2 ? (I ? 2 * I - 1 : 0) : I, j0 = L.fy == 2 ? (J ? 2 * J - 1 : 0) : J;
  const int ni = agg_count(I, L.fx, L.NX), nj = agg_count(J, L.fy, L.NY);
  // the aggregate's rows and their neighbours', all loads in flight together
  Pt blk[4][4];
#pragma unroll
  for (int j = 0; j < 4; j++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int ix = i0 + i - 1, iy = j0 + j - 1;
      blk[j][i] = load_pt(L.c, ix >= 0 && ix < L.NX && iy >= 0 && iy < L.NY, (int64_t)iy * L.NX + ix);
    }
  double off[4] = {0.0, 0.0, 0.0, 0.0}, rho = 0.0, delta = 0.0;
  int nlive = 0;
#pragma unroll
  for (int j = 0; j < 2; j++)
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const Pt &p = blk[j + 1][i + 1];
      if (i >= ni || j >= nj || !p.live()) continue;
      nlive++;
      rho += 1.0 + p.e + p.w + p.s + p.n;
      const double co[4] = {p.e, p.w, p.s, p.n};
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int di = (k == 0) - (k == 1), dj = (k == 2) - (k == 3);
        const int jx = i0 + i + di, jy = j0 + j + dj;
        if (co[k] == 0.0 || jx < 0 || jx >= L.NX || jy < 0 || jy >= L.NY) continue;
        const bool alongx = k < 2;
        const int f = alongx ? L.fx : L.fy, mine = alongx ? ni : nj;
        if (!blk[j + 1 + dj][i + 1 + di].live()) {
          delta -= co[k] * (f == 2 ? 2.0 / (mine + 1) : 1.0);
        } else if (agg(jx, L.fx) != I || agg(jy, L.fy) != J) {
          const int his = alongx ? agg_count(agg(jx, L.fx), L.fx, L.NX) : agg_count(agg(jy, L.fy), L.fy, L.NY);
          off[k] += co[k] * (f == 2 ? 2.0 / (mine + his) : 1.0);
        }
      }
    }
  const double diag = rho - (((off[0] + off[1]) + off[2]) + off[3]) + delta;
  const double id = nlive ? 1.0 / diag : 0.0;
  ce[q] = off[0] * id;
  cw[q] = off[1] * id;
  cs[q] = off[2] * id;
  cn[q] = off[3] * id;
  idc[q] = id;
}

// sums and least value over a block of 256, in thread 0
__device__ __forceinline__ void rows_block(double &sx, double &sy, double &lo, double &skew, double (*sh)[4]) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    sx += __shfl_xor(sx, o);
    sy += __shfl_xor(sy, o);
    lo = fmin(lo, __shfl_xor(lo, o));
    skew += __shfl_xor(skew, o);
  }
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) sh[0][w] = sx, sh[1][w] = sy, sh[2][w] = lo, sh[3][w] = skew;
  __syncthreads();
  sx = (sh[0][0] + sh[0][1]) + (sh[0][2] + sh[0][3]);
  sy = (sh[1][0] + sh[1][1]) + (sh[1][2] + sh[1][3]);
  lo = fmin(fmin(sh[2][0], sh[2][1]), fmin(sh[2][2], sh[2][3]));
  skew = (sh[3][0] + sh[3][1]) + (sh[3][2] + sh[3][3]);
}

// rows divided by their diagonal, and per block what the choice of a
// preconditioner needs: the sums of |e| + |w| and |s| + |n|, the least row sum, the
// pairs of couplings of opposite signs (a skew part)
__global__ void __launch_bounds__(256) k_rows(int64_t n, int NX, const double *__restrict__ d, Coefs c,
                                              double *__restrict__ e, double *__restrict__ w, double *__restrict__ s,
                                              double *__restrict__ nn, double *__restrict__ part) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  double sx = 0.0, sy = 0.0, lo = 1.0, skew = 0.0;
  if (i < n) {
    const double di = d[i];
    const Pt p = {c.e[i] / di, c.w[i] / di, c.s[i] / di, c.n[i] / di};
    if (e) e[i] = p.e, w[i] = p.w, s[i] = p.s, nn[i] = p.n;
    sx = fabs(p.e) + fabs(p.w);
    sy = fabs(p.s) + fabs(p.n);
    lo = 1.0 - sx - sy;
    if (!(lo == lo)) lo = -1.0;  // NaN rows: no bound
    auto opposite = [&](double to, const double *back, int64_t j) {
      return to != 0.0 && j < n && (to < 0.0) != (back[j] < 0.0 != d[j] < 0.0) && back[j] != 0.0 ? 1.0 : 0.0;
    };
    skew = opposite(p.e, c.w, i + 1) + opposite(p.s, c.n, i + NX);
  }
  __shared__ double sh[4][4];
  rows_block(sx, sy, lo, skew, sh);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = sx;
    part[gridDim.x + blockIdx.x] = sy;
    part[2 * gridDim.x + blockIdx.x] = lo;
    part[3 * gridDim.x + blockIdx.x] = skew;
  }
}
__global__ void __launch_bounds__(256) k_rows_total(int nb, const double *__restrict__ part, double *__restrict__ out) {
  double sx = 0.0, sy = 0.0, lo = 1.0, skew = 0.0;
  for (int k = threadIdx.x; k < nb; k += 256) {
    sx += part[k];
    sy += part[nb + k];
    lo = fmin(lo, part[2 * nb + k]);
    skew += part[3 * nb + k];
  }
  __shared__ double sh[4][4];
  rows_block(sx, sy, lo, skew, sh);
  if (threadIdx.x == 0) out[0] = sx, out[1] = sy, out[2] = lo, out[3] = skew;
}

Cheb cheb(double a, double b, int steps) {
  Cheb c;
  const double th = (b + a) / 2.0, de = (b - a) / 2.0, sg = th / de;
  double ro = 1.0 / sg;
  c.c1[0] = 0.0;
  c.c2[0] = 1.0 / th;
  for (int k = 1; k < steps; k++) {
    const double rn = 1.0 / (2.0 * sg - ro);
    c.c1[k] = rn * ro;
    c.c2[k] = 2.0 * rn / de;
    ro = rn;
  }
  return c;
}

int64_t padded(int64_t n) { return (n + 31) / 32 * 32; }

}  // namespace

// A system's preconditioner; its arrays lie in ctx->mg.
struct fvm_precond {
  double lo = 0.0;             // least row sum
  bool one_level = false;      // the polynomial on the finest level
  int n_lv = 0;                // each halves an axis at least: 2 x 31 of them at most
  Lv lv[FV_LEVELS];            // finest first
  // per level: right-hand side (not the finest's), the sweeps before its
  // correction, the result (not the finest's)
  double *b[FV_LEVELS], *x[FV_LEVELS], *y[FV_LEVELS];
  int first_coarse = 0;        // level at which the one-workgroup kernel takes over
  CoarseArgs coarse;
  Cheb smooth, last, poly;
};
void fvm_precond_free(fvm_precond *m) { delete m; }

int fvm_precond_build(fvm_ctx *ctx, int NX, int NY, const double *d, const double *e, const double *w, const double *s,
                      const double *n, bool scale, fvm_precond **out) {
  // how much stronger an axis' couplings are before it alone is coarsened
  constexpr double SEMI = 2.5;
  // least row sum from which the finest level alone is preconditioned: degree
  // FV_POLY then contracts every component about as well as a V-cycle does
  constexpr double DOMINANT = 0.05;
  // least row sum from which the polynomial damps all of the disc |z - 1| <= 1 - lo by
  // 5 or more: |T8| <= 577 on the unit disc, T8(1 / 0.6) = 3280.  Rows with couplings
  // +-0.1 (sum 0.6): 171 us, Jacobi 430; +-0.17 (0.32): 585 and 428 (300 x 200)
  constexpr double SKEW_DOMINANT = 0.4;
  *out = nullptr;
  const int64_t nn = (int64_t)NX * NY;
  const unsigned nb = fvm_blocks(nn, 256);
  // the finest level's rows and sweeps, the levels below (at most half the
  // points each, and a column and row more)
  const size_t words = (size_t)(5 * padded(nn) + padded(4 * (int64_t)nb) + 64) +
                       8 * (size_t)(nn + 24 * ((int64_t)NX + NY) + 4096);
  // without room for the levels, or with more rows than a grid has blocks for, the
  // solve runs without them
  if (nn > INT32_MAX || fvm_blocks(NY, FV_T) > 65535u) return FVM_OK;
  const int rc = fvm_ws(ctx, ctx->mg, words * sizeof(double));
  if (rc == FVM_ERR_NOMEM) {
    (void)hipGetLastError();
    return FVM_OK;
  }
  FVM_TRY(rc);
  double *p = (double *)ctx->mg.ptr, *end = p + words;
  auto take = [&](int64_t k) {
    double *r = p;
    p += padded(k);
    return r;
  };
  if (!ctx->precond) ctx->precond = new (std::nothrow) fvm_precond();
  fvm_precond *m = ctx->precond;
  if (!m) return fvm_set_err(ctx, FVM_ERR_NOMEM, "preconditioner");
  m->n_lv = m->first_coarse = 0;
  double *part = take(4 * (int64_t)nb), *tot = take(4);
  double *rows[4] = {nullptr, nullptr, nullptr, nullptr};
  Coefs c = {e, w, s, n};
  if (scale)
    for (int k = 0; k < 4; k++) rows[k] = take(nn);
  k_rows<<<nb, 256, 0, ctx->stream>>>(nn, NX, d, c, rows[0], rows[1], rows[2], rows[3], part);
  k_rows_total<<<1, 256, 0, ctx->stream>>>((int)nb, part, tot);
  FVM_LAUNCH_CHECK(ctx);
  double *host = (double *)ctx->pinned.ptr;
  FVM_HIP(ctx, hipMemcpyAsync(host, tot, 4 * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
  FVM_HIP(ctx, hipStreamSynchronize(ctx->stream));
  double sx = host[0], sy = host[1];
  m->lo = host[2];
  // Both kinds are made for a spectrum near the real axis.  On rows with couplings of
  // opposite signs it is not, and they would cost more than they give (an iteration's
  // polynomial can grow what it should damp) unless the row sums keep it small.
  if (host[3] > 0.0 && m->lo < SKEW_DOMINANT) return FVM_OK;
  if (scale) c = Coefs{rows[0], rows[1], rows[2], rows[3]};
  auto push = [&](int nx, int ny, const Coefs &co, double *b, double *x, double *y) {
    Lv L{};
    L.NX = nx, L.NY = ny, L.c = co, L.fx = L.fy = 1;
    m->lv[m->n_lv] = L;
    m->b[m->n_lv] = b, m->x[m->n_lv] = x, m->y[m->n_lv] = y;
    m->n_lv++;
  };
  m->one_level = !scale && m->lo >= DOMINANT;  // its kernels take a unit diagonal
  if (m->one_level) {
    push(NX, NY, c, nullptr, nullptr, nullptr);
    const double lo = m->lo < 0.99 ? m->lo : 0.99;  // rows without couplings: not an empty interval
    m->poly = cheb(lo, 2.0 - lo, FV_POLY);
    *out = m;
    return FVM_OK;
  }
  push(NX, NY, c, nullptr, take(nn), nullptr);
  m->smooth = cheb(0.1, 2.0, FV_NU);
  m->last = cheb(0.1, 2.0, FV_LAST);
  for (;;) {
    Lv &f = m->lv[m->n_lv - 1];
    if (m->n_lv == FV_LEVELS || (int64_t)f.NX * f.NY <= 20 || (f.NX <= 3 && f.NY <= 3)) break;
    f.fx = f.NX > 3 ? 2 : 1, f.fy = f.NY > 3 ? 2 : 1;
    if (f.fx == 2 && f.fy == 2) {
      if (sx > SEMI * sy) f.fy = 1, sx /= 4.0;
      else if (sy > SEMI * sx) f.fx = 1, sy /= 4.0;
    }
    f.NXc = f.fx == 2 ? f.NX / 2 + 1 : f.NX;
    f.NYc = f.fy == 2 ? f.NY / 2 + 1 : f.NY;
    const int64_t nc = (int64_t)f.NXc * f.NYc;
    if (p + 8 * padded(nc) > end) return FVM_OK;  // no preconditioner for such a shape
    double *ce = take(nc), *cw = take(nc), *cs = take(nc), *cn = take(nc), *id = take(nc);
    f.idc = id;
    k_coarsen<<<fvm_blocks(nc, 256), 256, 0, ctx->stream>>>(f, ce, cw, cs, cn, id);
    FVM_LAUNCH_CHECK(ctx);
    double *b = take(nc), *x = take(nc), *y = take(nc);
    push(f.NXc, f.NYc, Coefs{ce, cw, cs, cn}, b, x, y);
  }
  // the one-workgroup kernel takes the levels that fit its LDS and threads
  const int n_lv = m->n_lv;
  for (int l = 0; l < n_lv; l++) {
    if ((int64_t)m->lv[l].NX * m->lv[l].NY > FV_COARSE_MAX || n_lv - l > FV_CLEVELS) continue;
    CoarseArgs &A = m->coarse;
    int at = 0;
    for (int k = l; k < n_lv; k++) {
      const Lv &L = m->lv[k];
      A.lv[k - l] = L;
      A.off[k - l] = at + L.NX + 1;
      at += 2 * (L.NX + 1) + L.NX * L.NY;
    }
    A.n = n_lv - l;
    A.total = at;
    if (at > FV_LDS) continue;
    m->first_coarse = l;
    *out = m;
    return FVM_OK;
  }
  return FVM_OK;  // no level fits: no preconditioner
}

bool fvm_precond_one_level(const fvm_precond *m) { return m->one_level; }

// one iteration with the one-level preconditioner: 3 kernels (O.n_r partials of
// (rhat, r) and (r, r) come in, FVM_ONE_BLOCKS go out)
int fvm_precond_one_iteration(fvm_ctx *ctx, const fvm_precond *m, const FvmBcgOne &O) {
  const Lv &F = m->lv[0];
  const dim3 grid(fvm_blocks(F.NX, FV_PT), fvm_blocks(F.NY, FV_PT));
  k_one_p<<<grid, 1024, 0, ctx->stream>>>(F.NX, F.NY, F.c, m->poly, O);
  k_one_s<<<grid, 1024, 0, ctx->stream>>>(F.NX, F.NY, F.c, m->poly, O);
  k_one_x<<<FVM_ONE_BLOCKS, 1024, 0, ctx->stream>>>((int64_t)F.NX * F.NY, (int)(grid.x * grid.y), O);
  FVM_LAUNCH_CHECK(ctx);
  return FVM_OK;
}

// sc: the iteration's scalars (a finished iteration's kernels return at once)
int fvm_precond_apply(fvm_ctx *ctx, const fvm_precond *m, const double *b, double *x, const double *sc) {
  const int fc = m->first_coarse;
  auto rhs = [&](int l) { return l ? m->b[l] : b; };
  auto res = [&](int l) { return l ? m->y[l] : x; };
  for (int l = 0; l < fc; l++) {
    const Lv &L = m->lv[l];
    k_down<<<dim3(fvm_blocks(L.NXc, FV_T / L.fx), fvm_blocks(L.NYc, FV_T / L.fy)), FV_R * FV_R, 0, ctx->stream>>>(
        L, m->smooth, rhs(l), m->x[l], m->b[l + 1], sc);
  }
  k_coarse<<<1, FV_CT, 0, ctx->stream>>>(m->coarse, m->smooth, m->last, rhs(fc), res(fc), sc);
  for (int l = fc - 1; l >= 0; l--) {
    const Lv &L = m->lv[l];
    k_up<<<dim3(fvm_blocks(L.NX, FV_T), fvm_blocks(L.NY, FV_T)), FV_R * FV_R, 0, ctx->stream>>>(
        L, m->smooth, rhs(l), m->x[l], res(l + 1), res(l), sc);
  }
  FVM_LAUNCH_CHECK(ctx);
  return FVM_OK;
}
