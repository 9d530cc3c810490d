// adjoint.hip -- hand-written adjoint of one time step (FP64, gfx950).
//
// The step maps f^n to f^{n+1} = I4(C4(f^n); feet(E(f^n))) with
//   C4 = (M_vy x M_vx x M_y x M_x) f^n          (computeCoeff_xy + _vxvy,
//                                                 VMO/Spline.hpp:384-469)
//   I4 = the 4^4 B-spline interpolation at the feet (interp_4D,
//        VMO/Advection.hpp:221-296), feet from computeFeet (:166-218),
//   E  = K rho_half, rho_half = dvx dvy sum_v I2(C_xy(f^n)) (advect_2D_xy
//        :299-406, field_rho VMO/Field.cpp:37-53, Poisson :71-137).
// For a cotangent g of f^{n+1} the adjoint is
//   grad = C4^T I4^T g                                   (direct term)
//        + C_xy^T I2^T (dvx dvy (K^T lambda_E))          (through the field)
// with lambda_E the foot term: g times the derivative of I4 along the foot,
// times d foot / d E-bar (dt^2/2 for x, y; -dt for vx, vy unless clamped),
// scattered back through computeFeet's 3x3 Lagrange interpolation of E.
// M_d is the (N_d+4) x N_d spline operator of one line (the same for every
// direction of a given length), K the periodic E-from-rho operator.
#include "advect_common.hpp"

#include <cstdlib>

namespace vlp {

namespace {

// Derivative of the cubic B-spline weights bspline_eta with respect to w.
__device__ __forceinline__ void bspline_deta(double w, double d[4]) {
  const double d3 = 0.5 * w * w;
  const double d0 = 0.5 * (2. * w - 1.) - d3;
  const double d2 = 1. + d0 - 2. * d3;
  d[0] = d0;
  d[1] = -d0 - d2 - d3;
  d[2] = d2;
  d[3] = d3;
}

}  // namespace

// Per cell: the feet of the forward step, then
//  * g * w0 w1 w2 w3 added to lc4 at the 4^4 stencil (lc4 has the C4
//    storage layout, pitches c4_pitch);
//  * the foot term g * dI4/dfoot * dfoot/dEbar, scattered to lE (Ex, Ey
//    interleaved, N1 x N0) with computeFeet's Lagrange weights.
__global__ __launch_bounds__(256) void k_adj_advect4d(const double *__restrict__ c4, const double *__restrict__ ex,
                                                      const double *__restrict__ ey, Geom g, FeetConsts fc, double dt,
                                                      const double *__restrict__ gin, double *__restrict__ lc4,
                                                      double *__restrict__ lE, int field_term) {
  const int N0 = g.n[0], N1 = g.n[1], N2 = g.n[2], N3 = g.n[3];
  const long ncell = (long)N0 * N1 * N2 * N3;
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ncell) return;
  const int ix = (int)(t % N0), iy = (int)((t / N0) % N1), ivx = (int)((t / ((long)N0 * N1)) % N2),
            ivy = (int)(t / ((long)N0 * N1 * N2));
  const double gv = gin[t];
  if (gv == 0.) return;
  const double x = g.minPhy[0] + ix * g.dx[0], y = g.minPhy[1] + iy * g.dx[1];
  const double vx = g.minPhy[2] + ivx * g.dx[2], vy = g.minPhy[3] + ivy * g.dx[3];
  const double xt1 = half_y(g, y, vy, dt);
  const int ip1 = (int)(round(xt1) - 1);
  EGlobal E{ex, ey, N0, N1, ip1};
  double xs[4];
  if (!compute_foot(g, fc, E, xt1, ip1, x, y, vx, vy, dt, xs)) return;  // the forward step reports the error
  int ip[4];
  double w[4][4], dw[4][4];
  for (int j = 0; j < 4; j++) {
    const double fj = g.inv_dx[j] * (xs[j] - g.minPhy[j]);
    ip[j] = (int)floor(fj);
    bspline_eta<double>(fj - ip[j], w[j]);
    bspline_deta(fj - ip[j], dw[j]);
  }
  const C4Pitch cp = c4_pitch(N0, N1, N2);
  const long S1 = cp.s1, S2 = cp.s2, S3 = cp.s3;
  const long base = (ip[0] + 2) + S1 * (ip[1] + 2) + S2 * (ip[2] + 2) + S3 * (long)(ip[3] + 2);
  double dI[4] = {0., 0., 0., 0.};
  for (int k3 = 0; k3 < 4; k3++)
    for (int k2 = 0; k2 < 4; k2++)
      for (int k1 = 0; k1 < 4; k1++)
        for (int k0 = 0; k0 < 4; k0++) {
          const long o = base + k0 + S1 * k1 + S2 * k2 + S3 * k3;
          atomicAdd(lc4 + o, gv * w[0][k0] * w[1][k1] * w[2][k2] * w[3][k3]);
          if (field_term) {
            const double c = c4[o];
            dI[0] += c * dw[0][k0] * w[1][k1] * w[2][k2] * w[3][k3];
            dI[1] += c * w[0][k0] * dw[1][k1] * w[2][k2] * w[3][k3];
            dI[2] += c * w[0][k0] * w[1][k1] * dw[2][k2] * w[3][k3];
            dI[3] += c * w[0][k0] * w[1][k1] * w[2][k2] * dw[3][k3];
          }
        }
  if (!field_term) return;
  // d f^{n+1} / d xs_j = dI_j / dx_j; dxs/dEbar: x, y: dt^2/2; vx, vy: -dt
  // inside the velocity box (the clamp has zero derivative outside)
  const double vhi2 = g.minPhy[2] + fc.rxwidth[2], vhi3 = g.minPhy[3] + fc.rxwidth[3];
  const double ax = gv * (dI[0] * g.inv_dx[0] * 0.5 * dt * dt +
                          ((xs[2] > g.minPhy[2] && xs[2] < vhi2) ? -dt * dI[2] * g.inv_dx[2] : 0.));
  const double ay = gv * (dI[1] * g.inv_dx[1] * 0.5 * dt * dt +
                          ((xs[3] > g.minPhy[3] && xs[3] < vhi3) ? -dt * dI[3] * g.inv_dx[3] : 0.));
  // Ebar = sum_{k0,k1} cx[k0] cy[k1] E(ip0+k0, ip1+k1), VMO/Advection.hpp:174-196
  double xt0 = x - 0.5 * dt * vx;
  xt0 = g.inv_dx[0] * (xt0 - g.minPhy[0]);
  const int ip0 = (int)(round(xt0) - 1);
  const double px = xt0 - ip0, py = xt1 - ip1;
  const double cx[3] = {.5 * (px - 1.) * (px - 2.), -1. * (px) * (px - 2.), .5 * (px) * (px - 1.)};
  const double cy[3] = {.5 * (py - 1.) * (py - 2.), -1. * (py) * (py - 2.), .5 * (py) * (py - 1.)};
  for (int k1 = 0; k1 < 3; k1++)
    for (int k0 = 0; k0 < 3; k0++) {
      const int jx = ((ip0 + k0) % N0 + N0) % N0, jy = ((ip1 + k1) % N1 + N1) % N1;
      const double cc = cx[k0] * cy[k1];
      const long e = 2 * ((long)jy * N0 + jx);
      atomicAdd(lE + e, cc * ax);
      atomicAdd(lE + e + 1, cc * ay);
    }
}

// Fixed-point form of a coefficient-adjoint contribution: x * S rounded to
// the nearest integer (|x S| < 2^51: adding 1.5 * 2^52 leaves the integer in
// the low mantissa bits).  Integer sums do not depend on the order of the
// adds, so the result is the same on every run.
__device__ __forceinline__ unsigned long long to_fixed(double x) {
  const double M = 6755399441055744.0;  // 1.5 * 2^52
  return (unsigned long long)(__double_as_longlong(x + M) - __double_as_longlong(M));
}

// The same scatter by blocks of cells, with reproducible sums.  A workgroup
// takes BX x BV x BV x BV cells and adds their coefficient-adjoint
// contributions, as 64-bit fixed-point integers (scale S = *scl, a power of two
// with |g| S < 2^50), into an LDS copy of the coefficient region they reach
// when every foot lies within one cell below its own (ip_d - c_d in {-1, 0}:
// positions c - 2 .. c + 2 per dimension); a contribution outside it goes
// straight to lc4 (read as 64-bit integers).  The region is then added to lc4,
// one atomic per nonzero entry instead of one per cell and stencil point:
// (BX + 4) (BV + 4)^3 per BX BV^3 cells, 9 per cell for BX = 32, BV = 4
// instead of 256.  With the field term, each cell's pair (ax, ay) -- g times
// the derivative of the interpolation along the foot, times d foot / d E-bar --
// is written to axy, for the E gathers below.
//
// Bound: the 256 LDS atomics per cell at 2 waves per SIMD (LDS and registers).
// BV = 4 flushes 3 times fewer entries than BV = 2 (29 per cell): 48^4 2.02 ->
// 1.30 ms.  The coefficients of the foot term are loaded 16 at a time, one
// (vx, vy) point ahead of the atomics that hide them: 1.30 -> 0.81 ms (they
// took 0.54 ms while each was loaded where it was used; from an LDS copy of
// the region, which needs a second pass over the cells, 1.38 ms).
template <int BV>
__global__ __launch_bounds__(512) void k_adj_advect4d_blk(const double *__restrict__ c4,
                                                          const double *__restrict__ ex,
                                                          const double *__restrict__ ey, Geom g, FeetConsts fc,
                                                          double dt, const double *__restrict__ gin,
                                                          unsigned long long *__restrict__ lc4,
                                                          double *__restrict__ axy, const double *__restrict__ scl,
                                                          int field_term, int BX) {
  constexpr int RY = BV + 4, RV = BV + 4;  // coefficient region along y, vx, vy
  const int RX = BX + 4, NREG = RX * RY * RV * RV, NT = blockDim.x;
  extern __shared__ __align__(16) unsigned char adj_smem[];
  unsigned long long *reg = (unsigned long long *)adj_smem;
  const int N0 = g.n[0], N1 = g.n[1], N2 = g.n[2], N3 = g.n[3];
  const int nbx = (N0 + BX - 1) / BX, nby = (N1 + BV - 1) / BV, nbv = (N2 + BV - 1) / BV;
  long b = blockIdx.x;
  const int bx = (int)(b % nbx);
  b /= nbx;
  const int by = (int)(b % nby);
  b /= nby;
  const int bvx = (int)(b % nbv), bvy = (int)(b / nbv);
  const int x0 = bx * BX, y0 = BV * by, vx0 = BV * bvx, vy0 = BV * bvy;
  const int tid = threadIdx.x;
  const double S = scl[0];
  for (int i = tid; i < NREG; i += NT) reg[i] = 0ull;
  __syncthreads();
  const C4Pitch cp = c4_pitch(N0, N1, N2);
  const long S1 = cp.s1, S2 = cp.s2, S3 = cp.s3;
  for (int cell = tid; cell < BX * BV * BV * BV; cell += NT) {
    const int lx = cell % BX, r = cell / BX;
    const int ix = x0 + lx, iy = y0 + r % BV, ivx = vx0 + r / BV % BV, ivy = vy0 + r / (BV * BV);
    if (ix >= N0 || iy >= N1 || ivx >= N2 || ivy >= N3) continue;
    const long t = ix + (long)N0 * (iy + (long)N1 * (ivx + (long)N2 * ivy));
    const double gv = gin[t];
    const double x = g.minPhy[0] + ix * g.dx[0], y = g.minPhy[1] + iy * g.dx[1];
    const double vx = g.minPhy[2] + ivx * g.dx[2], vy = g.minPhy[3] + ivy * g.dx[3];
    const double xt1 = half_y(g, y, vy, dt);
    const int ip1 = (int)(round(xt1) - 1);
    EGlobal E{ex, ey, N0, N1, ip1};
    double xs[4];
    double ax = 0., ay = 0.;
    // (a zero cotangent or a foot out of the box adds nothing; the forward
    // step reports the latter)
    if (gv != 0. && compute_foot(g, fc, E, xt1, ip1, x, y, vx, vy, dt, xs)) {
      int ip[4];
      double w[4][4], dw[4][4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const double fj = g.inv_dx[j] * (xs[j] - g.minPhy[j]);
        ip[j] = (int)floor(fj);
        bspline_eta<double>(fj - ip[j], w[j]);
        bspline_deta(fj - ip[j], dw[j]);
      }
      // stencil origin in the region (positions x0 - 2 .., y0 - 2 .., ...)
      const int r0 = ip[0] - 1 - (x0 - 2), r1 = ip[1] - 1 - (y0 - 2), r2 = ip[2] - 1 - (vx0 - 2),
                r3 = ip[3] - 1 - (vy0 - 2);
      const bool inreg = r0 >= 0 && r0 + 3 < RX && r1 >= 0 && r1 + 3 < RY && r2 >= 0 && r2 + 3 < RV && r3 >= 0 &&
                         r3 + 3 < RV;
      const long base = (ip[0] + 2) + S1 * (ip[1] + 2) + S2 * (ip[2] + 2) + S3 * (long)(ip[3] + 2);
      // dI_j = sum over the stencil of c * (the weight product with dimension
      // j differentiated), contracted one dimension at a time: x (s, sd),
      // then y (u*), vx (v*), vy (dI)
      double dI[4] = {0., 0., 0., 0.};
      double gw0[4];
#pragma unroll
      for (int k0 = 0; k0 < 4; k0++) gw0[k0] = gv * S * w[0][k0];
      // the 4 x 4 coefficients of the next (vx, vy) point are loaded while this
      // one's 16 contributions go to LDS
      double cv[4][4], cn[4][4];
      auto load = [&](int k2, int k3, double (&c)[4][4]) {
        const double *q = c4 + base + S2 * k2 + S3 * k3;
#pragma unroll
        for (int k1 = 0; k1 < 4; k1++)
#pragma unroll
          for (int k0 = 0; k0 < 4; k0++) c[k1][k0] = q[S1 * k1 + k0];
      };
      if (field_term) load(0, 0, cv);
#pragma unroll
      for (int k3 = 0; k3 < 4; k3++) {
        double v = 0., vd0 = 0., vd1 = 0., vd2 = 0.;
#pragma unroll
        for (int k2 = 0; k2 < 4; k2++) {
          if (field_term && 4 * k3 + k2 < 15) load((k2 + 1) & 3, k3 + (k2 + 1) / 4, cn);
          __builtin_amdgcn_sched_barrier(0);
          const double w23 = w[2][k2] * w[3][k3];
          if (inreg) {
            unsigned long long *lrow = reg + (((r3 + k3) * RV + (r2 + k2)) * RY + r1) * RX + r0;
#pragma unroll
            for (int k1 = 0; k1 < 4; k1++)
#pragma unroll
              for (int k0 = 0; k0 < 4; k0++) atomicAdd(lrow + k1 * RX + k0, to_fixed(gw0[k0] * (w[1][k1] * w23)));
          } else {
            unsigned long long *grow = lc4 + base + S2 * k2 + S3 * k3;
#pragma unroll
            for (int k1 = 0; k1 < 4; k1++)
#pragma unroll
              for (int k0 = 0; k0 < 4; k0++) atomicAdd(grow + S1 * k1 + k0, to_fixed(gw0[k0] * (w[1][k1] * w23)));
          }
          if (!field_term) continue;
          double u = 0., ud0 = 0., ud1 = 0.;
#pragma unroll
          for (int k1 = 0; k1 < 4; k1++) {
            double s0 = 0., sd = 0.;
#pragma unroll
            for (int k0 = 0; k0 < 4; k0++) {
              s0 += w[0][k0] * cv[k1][k0];
              sd += dw[0][k0] * cv[k1][k0];
              cv[k1][k0] = cn[k1][k0];
            }
            u += w[1][k1] * s0;
            ud0 += w[1][k1] * sd;
            ud1 += dw[1][k1] * s0;
          }
          v += w[2][k2] * u;
          vd0 += w[2][k2] * ud0;
          vd1 += w[2][k2] * ud1;
          vd2 += dw[2][k2] * u;
        }
        dI[0] += w[3][k3] * vd0;
        dI[1] += w[3][k3] * vd1;
        dI[2] += w[3][k3] * vd2;
        dI[3] += dw[3][k3] * v;
      }
      if (field_term) {
        const double vhi2 = g.minPhy[2] + fc.rxwidth[2], vhi3 = g.minPhy[3] + fc.rxwidth[3];
        ax = gv * (dI[0] * g.inv_dx[0] * 0.5 * dt * dt +
                   ((xs[2] > g.minPhy[2] && xs[2] < vhi2) ? -dt * dI[2] * g.inv_dx[2] : 0.));
        ay = gv * (dI[1] * g.inv_dx[1] * 0.5 * dt * dt +
                   ((xs[3] > g.minPhy[3] && xs[3] < vhi3) ? -dt * dI[3] * g.inv_dx[3] : 0.));
      }
    }
    if (field_term) {
      axy[2 * t] = ax;
      axy[2 * t + 1] = ay;
    }
  }
  __syncthreads();
  // the region to global memory: region position (r0, r1, r2, r3) is the
  // coefficient at position (x0 - 2 + r0, ...), storage index + 3 per
  // dimension; only entries some cell reached are nonzero.  A wave takes a
  // row at a time.
  const int lane = tid & 63;
  for (int row = tid >> 6; row < RY * RV * RV; row += NT >> 6) {
    const int q1 = row % RY, q2 = row / RY % RV, q3 = row / (RY * RV);
    unsigned long long *dst =
        lc4 + ((x0 + 1) + S1 * (y0 + 1 + q1) + S2 * (vx0 + 1 + q2) + S3 * (long)(vy0 + 1 + q3));
    if (lane < RX) {
      const unsigned long long v = reg[row * RX + lane];
      if (v != 0ull) atomicAdd(dst + lane, v);
    }
  }
}

// Scale of the fixed-point coefficient adjoint: the largest |g| (as the bit
// pattern of a non-negative double, whose order is the numeric order), then
// S = 2^(50 - e) with max|g| < 2^e, and 1/S.
__global__ __launch_bounds__(256) void k_absmax_bits(const double *__restrict__ gin, long n,
                                                     unsigned long long *__restrict__ mx) {
  __shared__ unsigned long long sh[4];
  unsigned long long m = 0ull;
#pragma unroll 4
  for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (long)gridDim.x * blockDim.x) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(fabs(gin[t]));
    m = b > m ? b : m;
  }
  for (int off = 32; off > 0; off >>= 1) {
    const unsigned long long o = __shfl_down(m, off, 64);
    m = o > m ? o : m;
  }
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {  // one atomic per workgroup: they all meet at one address
    for (int w = 1; w < 4; w++) m = sh[w] > m ? sh[w] : m;
    atomicMax(mx, m);
  }
}
__global__ void k_fixed_zero(unsigned long long *__restrict__ mx) {
  if (threadIdx.x == 0) *mx = 0ull;
}
__global__ void k_fixed_scale(const unsigned long long *__restrict__ mx, double *__restrict__ scl) {
  if (threadIdx.x != 0) return;
  const double m = __longlong_as_double((long long)*mx);
  double S = 1.;
  if (m > 0. && m <= 1.7976931348623157e308) {
    int e = 0;
    (void)frexp(m, &e);  // m < 2^e
    S = ldexp(1., 50 - e);
  }
  scl[0] = S;
  scl[1] = 1. / S;
}

// E adjoint by gathers, in a fixed order.  computeFeet takes E-bar from the
// 3 x 3 nodes (ip0 + k0, ip1 + k1) (mod N0, N1) with weights cx[k0] cy[k1],
// ip0 and cx depending on (x, vx) and ip1 and cy on (y, vy).  First, for
// every (jx, y, vy): the sum over vx and over the cells x whose node
// ip0 + k0 is jx of cx[k0] (ax, ay)(x, y, vx, vy) -- ip0 = x + round(d) - 1
// with d = -dt vx / (2 dx) up to rounding, so x is one of five candidates,
// each checked exactly; then for every node (jx, jy) the same over (y, vy)
// with cy.
//
// Bound: latency and the candidates' arithmetic.  Shifts are reduced modulo
// the axis once per velocity (uniform), not per candidate, and the velocity
// sums are split over ADJE_PARTS waves of a workgroup and added in order:
// 48^4 k_adjE_x 48 us (113 us), k_adjE_y 15 us (93 us; one wave per 64 nodes).
constexpr int ADJE_PARTS = 8;

// Quadratic weight of node ip + k at p = x - ip.
__device__ __forceinline__ double node_weight(double p, int k) {
  return k == 0 ? .5 * (p - 1.) * (p - 2.) : k == 1 ? -1. * (p) * (p - 2.) : .5 * (p) * (p - 1.);
}
// r in [0, N) for q within one N of it
__device__ __forceinline__ int wrap1(int q, int N) { return q < 0 ? q + N : q >= N ? q - N : q; }

// Lane (64 per workgroup and part) per (jx, y, vy); node j and axis length N of
// the gather along it; foot(i, v) the displaced position of point i in cells,
// visit(i, v, weight) in ascending candidate order for every velocity v of the
// part.  base: round(-dt v / (2 dx)) - 1.
template <typename B, typename F, typename V>
__device__ __forceinline__ void gather_nodes(int j, int N, int nv, int part, B base, F foot, V visit) {
  for (int v = part * nv / ADJE_PARTS; v < (part + 1) * nv / ADJE_PARTS; v++) {
    const int sh = base(v);
    int red = sh % N;  // (uniform)
    if (red < 0) red += N;
    const int turns = sh - red;  // a multiple of N
#pragma unroll
    for (int q = -3; q <= 1; q++) {
      const int i = wrap1(wrap1(j - red + q, N), N);
      const double xt = foot(i, v);
      const int ip = (int)(round(xt) - 1);
      // (j - ip) mod N: ip + 3 N > j > ip - 3 N after the turns are taken out
      const int k = wrap1(wrap1(wrap1(j - (ip - turns), N), N), N);
      if ((unsigned)k <= 2u) visit(i, v, node_weight(xt - ip, k));
    }
  }
}

__global__ __launch_bounds__(64 * ADJE_PARTS) void k_adjE_x(const double *__restrict__ axy, Geom g, double dt,
                                                            double *__restrict__ part) {
  __shared__ double2 sh[ADJE_PARTS][64];
  const int N0 = g.n[0], N1 = g.n[1], N2 = g.n[2], N3 = g.n[3];
  const long n = (long)N0 * N1 * N3;
  const int lane = threadIdx.x & 63, pt = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long t = (long)blockIdx.x * 64 + lane, tc = t < n ? t : n - 1;
  const int jx = (int)(tc % N0), iy = (int)((tc / N0) % N1), ivy = (int)(tc / ((long)N0 * N1));
  const double2 *src = (const double2 *)axy + (long)N0 * (iy + (long)N1 * N2 * ivy);
  double sx = 0., sy = 0.;
  gather_nodes(
      jx, N0, N2, pt,
      [&](int v) { return (int)round(-0.5 * dt * (g.minPhy[2] + v * g.dx[2]) * g.inv_dx[0]) - 1; },
      [&](int i, int v) {
        const double xt0 = (g.minPhy[0] + i * g.dx[0]) - 0.5 * dt * (g.minPhy[2] + v * g.dx[2]);
        return g.inv_dx[0] * (xt0 - g.minPhy[0]);
      },
      [&](int i, int v, double w) {
        const double2 a = src[i + (long)N0 * N1 * v];
        sx += w * a.x;
        sy += w * a.y;
      });
  sh[pt][lane] = make_double2(sx, sy);
  __syncthreads();
  if (pt == 0 && t < n) {
    for (int p = 1; p < ADJE_PARTS; p++) {
      sx += sh[p][lane].x;
      sy += sh[p][lane].y;
    }
    part[2 * t] = sx;
    part[2 * t + 1] = sy;
  }
}
__global__ __launch_bounds__(64 * ADJE_PARTS) void k_adjE_y(const double *__restrict__ part, Geom g, double dt,
                                                            double *__restrict__ lE) {
  __shared__ double2 sh[ADJE_PARTS][64];
  const int N0 = g.n[0], N1 = g.n[1], N3 = g.n[3];
  const long n = (long)N0 * N1;
  const int lane = threadIdx.x & 63, pt = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long t = (long)blockIdx.x * 64 + lane, tc = t < n ? t : n - 1;
  const int jx = (int)(tc % N0), jy = (int)(tc / N0);
  const double2 *src = (const double2 *)part + jx;
  double sx = 0., sy = 0.;
  gather_nodes(
      jy, N1, N3, pt,
      [&](int v) { return (int)round(-0.5 * dt * (g.minPhy[3] + v * g.dx[3]) * g.inv_dx[1]) - 1; },
      [&](int i, int v) { return half_y(g, g.minPhy[1] + i * g.dx[1], g.minPhy[3] + v * g.dx[3], dt); },
      [&](int i, int v, double w) {
        const double2 a = src[(long)N0 * (i + (long)N1 * v)];
        sx += w * a.x;
        sy += w * a.y;
      });
  sh[pt][lane] = make_double2(sx, sy);
  __syncthreads();
  if (pt == 0 && t < n) {
    for (int p = 1; p < ADJE_PARTS; p++) {
      sx += sh[p][lane].x;
      sy += sh[p][lane].y;
    }
    lE[2 * t] = sx;
    lE[2 * t + 1] = sy;
  }
}

// out[o][n][i] (+)= sum_m Mt[n][m] in[o][m][i]: a line operator's transpose
// applied along one axis (Mt is M^T, Nout x Min, row-major).
__global__ __launch_bounds__(256) void k_axis_contract(const double *__restrict__ Mt, int Min, int Nout,
                                                       const double *__restrict__ in, double *__restrict__ out, long O,
                                                       long I, int accumulate) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= O * Nout * I) return;
  const long i = t % I, n = (t / I) % Nout, o = t / (I * Nout);
  const double *src = in + o * Min * I + i;
  const double *a = Mt + (long)n * Min;
  double s = 0.;
  for (int m = 0; m < Min; m++) s += a[m] * src[(long)m * I];
  if (accumulate) out[t] += s;
  else out[t] = s;
}

// The same contraction by tiles: a workgroup stages in[o][0..Min-1][64
// columns] in LDS once (columns: 64 consecutive i of one o, or, when I = 1,
// 64 consecutive o) and each wave forms 16 outputs n per pass from it, the
// operator entries M[m][n] (M = Mt^T, Min x Nout row-major) arriving as
// wave-uniform scalar loads.  Same sums in the same order as k_axis_contract.
//
// Bound: HBM for I > 1 (48^4 36 us a pass).  For I = 1 the axis is the fastest
// index: the tile is transposed through an odd LDS pitch and a wave's outputs
// go through LDS eight at a time, so that both sides of the pass are coalesced
// (48^4 46 us; 74 us with a lane's outputs stored down its own row, and
// staging stores that all met in one bank).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
template <bool COLO>
__global__ __launch_bounds__(256) void k_axis_contract_t(const double *__restrict__ M, int Min, int Nout,
                                                         const double *__restrict__ in, double *__restrict__ out,
                                                         long O, long I, int accumulate) {
  constexpr int CP = COLO ? 65 : 64;
  extern __shared__ __align__(16) double ctile[];  // [Min][CP], then for COLO 8 x CP per wave
  const int tid = threadIdx.x, c = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  long o0, i0;
  int ncol;
  if (COLO) {
    o0 = (long)blockIdx.x * 64;
    i0 = 0;
    ncol = (int)(O - o0 < 64 ? O - o0 : 64);
  } else {
    const long nt = (I + 63) / 64;
    o0 = blockIdx.x / nt;
    i0 = (blockIdx.x % nt) * 64;
    ncol = (int)(I - i0 < 64 ? I - i0 : 64);
  }
  if (COLO) {
    for (int e = tid; e < 64 * Min; e += 256) {
      const int cc = e / Min, m = e - cc * Min;
      ctile[m * CP + cc] = cc < ncol ? in[o0 * Min + e] : 0.;
    }
  } else {
    const double *src = in + o0 * Min * I + i0;
    for (int e = tid; e < 64 * Min; e += 256) {
      const int m = e >> 6, cc = e & 63;
      ctile[e] = cc < ncol ? src[(long)m * I + cc] : 0.;
    }
  }
  __syncthreads();
  for (int n0 = 16 * wv; n0 < Nout; n0 += 64) {
    const int jmax = Nout - n0 < 16 ? Nout - n0 : 16;
    double acc[16];
#pragma unroll
    for (int j = 0; j < 16; j++) acc[j] = 0.;
    if (jmax == 16) {  // whole chunk: 16 consecutive entries per m, loaded together
      for (int m = 0; m < Min; m++) {
        const double x = ctile[m * CP + c];
        const double *mr = M + (long)m * Nout + n0;
#pragma unroll
        for (int j = 0; j < 16; j++) acc[j] += mr[j] * x;
      }
    } else {
      for (int m = 0; m < Min; m++) {
        const double x = ctile[m * CP + c];
        const double *mr = M + (long)m * Nout + n0;
#pragma unroll
        for (int j = 0; j < 16; j++)
          if (j < jmax) acc[j] += mr[j] * x;
      }
    }
    if (COLO) {
      double *ot = ctile + Min * CP + wv * 8 * CP;
#pragma unroll
      for (int h = 0; h < 16; h += 8) {
        wave_lds_fence();  // (the previous eight are read)
#pragma unroll
        for (int j = 0; j < 8; j++) ot[j * CP + c] = acc[h + j];
        wave_lds_fence();
        // eight lanes a row of eight outputs
        const int j = c & 7;
        if (h + j < jmax)
          for (int cc = c >> 3; cc < ncol; cc += 8) {
            const long idx = (o0 + cc) * Nout + n0 + h + j;
            const double v = ot[j * CP + cc];
            out[idx] = accumulate ? out[idx] + v : v;
          }
      }
    } else if (c < ncol) {
#pragma unroll
      for (int j = 0; j < 16; j++)
        if (j < jmax) {
          const long idx = (o0 * Nout + n0 + j) * I + i0 + c;
          out[idx] = accumulate ? out[idx] + acc[j] : acc[j];
        }
    }
  }
}

// Contiguous copy of the coefficient block (positions -2..N+1 per dimension)
// out of the C4 storage layout (positions -3..N+2); with scl, the storage
// holds 64-bit fixed-point sums, converted with the factor scl[1] = 1/S.
__global__ __launch_bounds__(256) void k_c4_block(const double *__restrict__ c4s, double *__restrict__ blk, Geom g,
                                                  const double *__restrict__ scl) {
  const long E0 = g.n[0] + 4, E1 = g.n[1] + 4, E2 = g.n[2] + 4, E3 = g.n[3] + 4;
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= E0 * E1 * E2 * E3) return;
  const long a = t % E0, b = (t / E0) % E1, c = (t / (E0 * E1)) % E2, d = t / (E0 * E1 * E2);
  const C4Pitch cp = c4_pitch(g.n[0], g.n[1], g.n[2]);
  const long o = (a + 1) + cp.s1 * (b + 1) + cp.s2 * (c + 1) + cp.s3 * (d + 1);
  if (scl) blk[t] = (double)((const long long *)c4s)[o] * scl[1];
  else blk[t] = c4s[o];
}

// lambda_rho(j) = sum_i lE_x(i) kx(i - j) + lE_y(i) ky(i - j): the transpose
// of the periodic E-from-rho convolution, kx/ky its response to a unit
// density at the origin (indices mod N0, N1).
__global__ __launch_bounds__(256) void k_poisson_T(const double *__restrict__ lE, const double *__restrict__ kx,
                                                   const double *__restrict__ ky, double *__restrict__ lrho, int N0,
                                                   int N1) {
  // 16 outputs per workgroup, each summed over 16 slices of the source rows
  // by 16 lanes, then the slices added in a fixed order
  __shared__ double part[16][16];
  const int o = threadIdx.x & 15, p = threadIdx.x >> 4;
  const long t = (long)blockIdx.x * 16 + o;
  double s = 0.;
  if (t < (long)N0 * N1) {
    const int jx = (int)(t % N0), jy = (int)(t / N0);
    const int y0 = (int)((long)p * N1 / 16), y1 = (int)((long)(p + 1) * N1 / 16);
    for (int iy = y0; iy < y1; iy++) {
      const int dy = iy >= jy ? iy - jy : iy - jy + N1;
      const double *e = lE + 2 * (long)iy * N0;
      const double *kxr = kx + (long)dy * N0, *kyr = ky + (long)dy * N0;
      // ix = 0 .. N0-1 with dx = (ix - jx) mod N0, without a division per term
      for (int ix = 0; ix < jx; ix++) s += e[2 * ix] * kxr[ix - jx + N0] + e[2 * ix + 1] * kyr[ix - jx + N0];
      for (int ix = jx; ix < N0; ix++) s += e[2 * ix] * kxr[ix - jx] + e[2 * ix + 1] * kyr[ix - jx];
    }
  }
  part[p][o] = s;
  __syncthreads();
  if (p == 0 && t < (long)N0 * N1) {
    double r = 0.;
    for (int q = 0; q < 16; q++) r += part[q][o];
    lrho[t] = r;
  }
}

// Through the half step: f_half(x, y, v) = I2(C_xy) at (x - dt/2 vx,
// y - dt/2 vy) and rho_half = dvx dvy sum_v f_half, so lambda_{f_half} =
// dvx dvy lambda_rho(x, y), scattered by the 4x4 B-spline weights of the
// half-step foot into lcxy (the C_xy layout: positions -2..N+1 in x and y,
// then vx, vy).
__global__ __launch_bounds__(256) void k_adj_advect2d(const double *__restrict__ lrho, Geom g, double dth,
                                                      double *__restrict__ lcxy) {
  const int N0 = g.n[0], N1 = g.n[1], N2 = g.n[2], N3 = g.n[3];
  const long ncell = (long)N0 * N1 * N2 * N3;
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ncell) return;
  const int ix = (int)(t % N0), iy = (int)((t / N0) % N1), ivx = (int)((t / ((long)N0 * N1)) % N2),
            ivy = (int)(t / ((long)N0 * N1 * N2));
  const double lv = lrho[(long)iy * N0 + ix] * g.dx[2] * g.dx[3];
  if (lv == 0.) return;
  const double x = g.minPhy[0] + ix * g.dx[0], y = g.minPhy[1] + iy * g.dx[1];
  const double vx = g.minPhy[2] + ivx * g.dx[2], vy = g.minPhy[3] + ivy * g.dx[3];
  const double fx = ((x - dth * vx) - g.minPhy[0]) * g.inv_dx[0];
  const double fy = ((y - dth * vy) - g.minPhy[1]) * g.inv_dx[1];
  const int jx0 = (int)floor(fx), jy0 = (int)floor(fy);
  if (jx0 < -1 || jx0 > N0 - 1 || jy0 < -1 || jy0 > N1 - 1) return;  // interp_2D leaves 0 there
  double ex[4], ey[4];
  bspline_eta<double>(fx - jx0, ex);
  bspline_eta<double>(fy - jy0, ey);
  const long E0 = N0 + 4, E1 = N1 + 4;
  double *pl = lcxy + ((long)ivx + (long)N2 * ivy) * E0 * E1;
  // stencil position jx0-1+k at column (position + 2)
  for (int ky = 0; ky < 4; ky++)
    for (int kx = 0; kx < 4; kx++) atomicAdd(pl + (long)(jy0 + 1 + ky) * E0 + (jx0 + 1 + kx), lv * ex[kx] * ey[ky]);
}

// The same adjoint as a gather, one lane per C_xy entry (X, Y) of a plane
// (positions -2..N+1 as columns 0..N+3): the cells whose half-step stencil
// covers X have jx0 = X - 1 - kx, kx in 0..3, and jx0(ix) = floor(ix + d)
// up to rounding, d = -dth vx / dx, so ix lies in
// [X - 5 - floor(d), X - floor(d)]; each candidate's jx0 and weights are
// recomputed exactly as the scatter (and the forward) computes them, and
// likewise in y.  No atomics: the result does not depend on scheduling.
//
// The y sums depend on (ix, Y, vy) only and the x weights on (X, vx): a
// workgroup takes ADJ2_Y rows of one vy, forms their y sums in LDS and runs
// through its part of the vx, a lane with one column and all the rows.
// Bound: the writes of lcxy and the weights' arithmetic; 48^4 24 us (104 us
// with a lane per entry that formed both).
constexpr int ADJ2_Y = 8;

// Candidate point c of column (or row) X of an axis: true if its half-step
// stencil covers X, with the weight there.
__device__ __forceinline__ bool half_weight(const Geom &g, int d, double dth, double v, int c, int X, double &w) {
  if (c < 0 || c >= g.n[d]) return false;
  const double x = g.minPhy[d] + c * g.dx[d];
  const double f = ((x - dth * v) - g.minPhy[d]) * g.inv_dx[d];
  const int j0 = (int)floor(f), k = X - 1 - j0;
  if (j0 < -1 || j0 > g.n[d] - 1 || k < 0 || k > 3) return false;
  double e[4];
  bspline_eta<double>(f - j0, e);
  w = k == 0 ? e[0] : k == 1 ? e[1] : k == 2 ? e[2] : e[3];
  return true;
}

__global__ __launch_bounds__(256) void k_adj_advect2d_g(const double *__restrict__ lrho, Geom g, double dth,
                                                        double *__restrict__ lcxy, int nyt, int nvp) {
  extern __shared__ __align__(16) double ysum[];  // [ADJ2_Y][N0]
  const int N0 = g.n[0], N1 = g.n[1], N2 = g.n[2], E0 = N0 + 4, E1 = N1 + 4;
  unsigned b = blockIdx.x;
  const int vp = b % nvp;
  b /= nvp;
  const int Y0 = (int)(b % nyt) * ADJ2_Y, ivy = b / nyt, ny = min(ADJ2_Y, E1 - Y0);
  const double vy = g.minPhy[3] + ivy * g.dx[3];
  const int fdy = (int)floor(-dth * vy * g.inv_dx[1]);
  for (int e = threadIdx.x; e < ny * N0; e += 256) {
    const int r = e / N0, ix = e - r * N0, Y = Y0 + r;
    double sy = 0.;
#pragma unroll
    for (int q = 0; q < 6; q++) {
      const int iy = Y - 5 - fdy + q;
      double w;
      if (half_weight(g, 1, dth, vy, iy, Y, w) && w != 0.) sy += w * lrho[(long)iy * N0 + ix];
    }
    ysum[r * N0 + ix] = sy;
  }
  __syncthreads();
  // lanes: columns, several vx at a time where a row is short
  const int nx = 256 / E0 > 0 ? 256 / E0 : 1, sub = threadIdx.x / E0, X = threadIdx.x - sub * E0;
  if (sub >= nx) return;
  const int v1 = (int)((long)(vp + 1) * N2 / nvp);
  for (int ivx = (int)((long)vp * N2 / nvp) + sub; ivx < v1; ivx += nx) {
    const double vx = g.minPhy[2] + ivx * g.dx[2];
    const int ix0 = X - 5 - (int)floor(-dth * vx * g.inv_dx[0]);
    double w[6];
    bool in[6];
#pragma unroll
    for (int p = 0; p < 6; p++) in[p] = half_weight(g, 0, dth, vx, ix0 + p, X, w[p]);
    double *dst = lcxy + ((long)ivx + (long)N2 * ivy) * E0 * E1 + (long)Y0 * E0 + X;
    for (int r = 0; r < ny; r++) {
      double acc = 0.;
#pragma unroll
      for (int p = 0; p < 6; p++)
        if (in[p]) acc += w[p] * ysum[r * N0 + ix0 + p];
      dst[(long)r * E0] = acc * g.dx[2] * g.dx[3];
    }
  }
}

// Field-energy source: W(f) = dx dy sum (Ex^2 + Ey^2) of the field solved
// from f, so dW/dE = 2 dx dy E.  lE = scale * (Ex, Ey) pairs.
__global__ __launch_bounds__(256) void k_scale_pairs(const double *__restrict__ exy, double scale, long n,
                                                     double *__restrict__ lE) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) lE[t] = scale * exy[t];
}

// g(x, y, v) += scale * lrho(x, y) for every (vx, vy): the density's adjoint
// (rho = dvx dvy sum_v f).
__global__ __launch_bounds__(256) void k_add_density_adj(const double *__restrict__ lrho, double scale, long nxy,
                                                         long ncell, double *__restrict__ gbuf) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < ncell) gbuf[t] += scale * lrho[t % nxy];
}

// out(x, y) = sum_{vx, vy} w(vx, vy) in(x, y, vx, vy), summed in a fixed order.
__global__ __launch_bounds__(1024) void k_vmoment(const double *__restrict__ in, const double *__restrict__ w, long nxy,
                                                  long nv, double *__restrict__ out) {
  // 64 points by 16 parts of the velocities (one lane per point ran 0.55 ms at
  // 48^4, bound by the latency of its nv loads)
  __shared__ double sh[16][64];
  const int lane = threadIdx.x & 63, part = threadIdx.x >> 6;
  const long t = (long)blockIdx.x * 64 + lane;
  double s = 0.;
  if (t < nxy)
#pragma unroll 8
    for (long v = part; v < nv; v += 16) s += w[v] * in[t + nxy * v];
  sh[part][lane] = s;
  __syncthreads();
  if (part == 0 && t < nxy) {
    for (int p = 1; p < 16; p++) s += sh[p][lane];
    out[t] = s;
  }
}

void launch_scale_pairs(const double *exy, double scale, long n, double *lE, hipStream_t s) {
  hipLaunchKernelGGL(k_scale_pairs, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, exy, scale, n, lE);
}

void launch_add_density_adj(const double *lrho, double scale, long nxy, long ncell, double *g, hipStream_t s) {
  hipLaunchKernelGGL(k_add_density_adj, dim3((unsigned)((ncell + 255) / 256)), dim3(256), 0, s, lrho, scale, nxy,
                     ncell, g);
}

void launch_vmoment(const double *in, const double *w, long nxy, long nv, double *out, hipStream_t s) {
  hipLaunchKernelGGL(k_vmoment, dim3((unsigned)((nxy + 63) / 64)), dim3(1024), 0, s, in, w, nxy, nv, out);
}

template <int BV>
static void launch_adj_blk(const Geom &g, const double *c4, const double *ex, const double *ey, double dt,
                           const double *gin, double *lc4, double *axy, const double *scl, bool field_term,
                           hipStream_t s) {
  // x extents of up to 32, equal ones where N0 is not a multiple
  const int nbx = (g.n[0] + 31) / 32, BX = (g.n[0] + nbx - 1) / nbx;
  const size_t lds = (size_t)(BX + 4) * (BV + 4) * (BV + 4) * (BV + 4) * sizeof(unsigned long long);
  const void *fn = (const void *)k_adj_advect4d_blk<BV>;
  if (lds > 64 * 1024) (void)hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  const long nb = (long)nbx * ((g.n[1] + BV - 1) / BV) * ((g.n[2] + BV - 1) / BV) * ((g.n[3] + BV - 1) / BV);
  hipLaunchKernelGGL(k_adj_advect4d_blk<BV>, dim3((unsigned)nb), dim3(BV == 4 ? 512 : 256), lds, s, c4, ex, ey, g,
                     feet_consts(g), dt, gin, (unsigned long long *)lc4, axy, scl, field_term ? 1 : 0, BX);
}

bool adj_blocked() {
  // VLP4D_ADJ_BLOCK=0: the per-cell scatter (floating-point atomics: one per
  // stencil point and E node) and the half-step scatter
  if (const char *e = getenv("VLP4D_ADJ_BLOCK")) return atoi(e) != 0;
  return true;
}

void launch_adj_advect4d(const Geom &g, const double *c4, const double *ex, const double *ey, double dt,
                         const double *gin, double *lc4, double *lE, bool field_term, hipStream_t s,
                         const AdjWork *wk) {
  if (wk) {
    // reproducible form: fixed-point scale from max|g|, blocked scatter,
    // then the two E gathers
    const long n = (long)g.n[0] * g.n[1] * g.n[2] * g.n[3];
    unsigned long long *mx = (unsigned long long *)(wk->scl + 2);
    hipLaunchKernelGGL(k_fixed_zero, dim3(1), dim3(64), 0, s, mx);
    hipLaunchKernelGGL(k_absmax_bits, dim3(1024), dim3(256), 0, s, gin, n, mx);
    hipLaunchKernelGGL(k_fixed_scale, dim3(1), dim3(64), 0, s, (const unsigned long long *)mx, wk->scl);
    // 4^3 blocks when they give every CU two workgroups to run in turn (one
    // fits at a time), else 2^3
    const long big = (long)((g.n[0] + 31) / 32) * (g.n[1] / 4) * (g.n[2] / 4) * (g.n[3] / 4);
    if (big >= 512) launch_adj_blk<4>(g, c4, ex, ey, dt, gin, lc4, wk->axy, wk->scl, field_term, s);
    else launch_adj_blk<2>(g, c4, ex, ey, dt, gin, lc4, wk->axy, wk->scl, field_term, s);
    if (field_term) {
      const long np = (long)g.n[0] * g.n[1] * g.n[3], ne = (long)g.n[0] * g.n[1];
      hipLaunchKernelGGL(k_adjE_x, dim3((unsigned)((np + 63) / 64)), dim3(64 * ADJE_PARTS), 0, s, wk->axy, g, dt,
                         wk->part);
      hipLaunchKernelGGL(k_adjE_y, dim3((unsigned)((ne + 63) / 64)), dim3(64 * ADJE_PARTS), 0, s, wk->part, g, dt,
                         lE);
    }
    return;
  }
  const long n = (long)g.n[0] * g.n[1] * g.n[2] * g.n[3];
  hipLaunchKernelGGL(k_adj_advect4d, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, c4, ex, ey, g,
                     feet_consts(g), dt, gin, lc4, lE, field_term ? 1 : 0);
}

void launch_axis_contract(const double *Mt, int Min, int Nout, const double *in, double *out, long O, long I,
                          bool accumulate, hipStream_t s, const double *M) {
  if (M) {  // tiled form (M = Mt^T)
    const size_t lds = (size_t)Min * 64 * sizeof(double);
    if (I == 1) {
      const size_t lds = (size_t)(Min + 32) * 65 * sizeof(double);
      (void)hipFuncSetAttribute((const void *)k_axis_contract_t<true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds);
      hipLaunchKernelGGL(k_axis_contract_t<true>, dim3((unsigned)((O + 63) / 64)), dim3(256), lds, s, M, Min, Nout,
                         in, out, O, I, accumulate ? 1 : 0);
    } else {
      (void)hipFuncSetAttribute((const void *)k_axis_contract_t<false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds);
      hipLaunchKernelGGL(k_axis_contract_t<false>, dim3((unsigned)(O * ((I + 63) / 64))), dim3(256), lds, s, M, Min,
                         Nout, in, out, O, I, accumulate ? 1 : 0);
    }
    return;
  }
  const long n = O * Nout * I;
  hipLaunchKernelGGL(k_axis_contract, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, Mt, Min, Nout, in, out, O,
                     I, accumulate ? 1 : 0);
}

void launch_c4_block(const Geom &g, const double *c4s, double *blk, hipStream_t s, const double *scl) {
  const long n = (long)(g.n[0] + 4) * (g.n[1] + 4) * (g.n[2] + 4) * (g.n[3] + 4);
  hipLaunchKernelGGL(k_c4_block, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, c4s, blk, g, scl);
}

void launch_poisson_T(const double *lE, const double *kx, const double *ky, double *lrho, int N0, int N1,
                      hipStream_t s) {
  hipLaunchKernelGGL(k_poisson_T, dim3((unsigned)((N0 * N1 + 15) / 16)), dim3(256), 0, s, lE, kx, ky, lrho, N0, N1);
}

void launch_adj_advect2d(const double *lrho, const Geom &g, double dth, double *lcxy, hipStream_t s) {
  const long n = (long)g.n[0] * g.n[1] * g.n[2] * g.n[3];
  // VLP4D_ADJ_BLOCK=0 also selects the scatter form here (lcxy zeroed by the caller)
  if (adj_blocked()) {
    // vx in parts until there are four workgroups per CU
    const int nyt = (g.n[1] + 4 + ADJ2_Y - 1) / ADJ2_Y;
    int nvp = 1;
    while (nvp < 8 && nyt * g.n[3] * nvp < 1024) nvp *= 2;
    hipLaunchKernelGGL(k_adj_advect2d_g, dim3((unsigned)(nyt * g.n[3] * nvp)), dim3(256),
                       sizeof(double) * ADJ2_Y * g.n[0], s, lrho, g, dth, lcxy, nyt, nvp);
    return;
  }
  hipLaunchKernelGGL(k_adj_advect2d, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, lrho, g, dth, lcxy);
}

}  // namespace vlp
