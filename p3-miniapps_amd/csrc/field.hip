// field.hip -- field solve and diagnostics kernels (FP64, gfx950).
#include <algorithm>

#include "device_common.hpp"

namespace vlp {

// ---------------------------------------------------------------------------
// Field solve, FP64.  rho = dvx*dvy*sum rho_part over its outer planes
// (vy, and the vx groups of the fused xy kernel; VMO/Field.cpp:37-53),
// rho -= 1 for idcase 10/20 (VMO/Field.cpp:110-126), then solve_poisson_fftw
// (VMO/Efield.cpp:54-106) with the FFT conventions of lib/OpenMP_FFT.hpp:
// unnormalised r2c along x, c2c along y, normalisation in k-space, inverse
// c2c along y, c2r along x (imaginary parts of DC/Nyquist ignored).
//
// A transform of N = A B points (A the largest divisor up to sqrt(N)) goes in
// two stages with one exactly reduced twiddle table,
//   Y[k1][n2] = sum_{n1 < A} x[B n1 + n2] w^(B n1 k1),
//   X[k] = sum_{n2 < B} Y[k mod A][n2] w^(n2 k),
// A + B terms per output instead of N; a prime N is the direct sum.  (The c2r
// transform, half as many real terms, stays a direct sum: 8.6 us against 9.5.)
//
// Bound: LDS reads and latency of the few workgroups (one per row or column).
// The direct sums read 6 N^2 complex values per column: the transform of 128
// points along y took 17.9 us, now 8.6; of 128 along x 7.4, now 5.2 and 14.3 with
// the sum of 512 density planes (11 us in a launch of its own before).  The data
// of a sum are broadcasts or runs from LDS; the twiddles, one per lane at strides
// that meet in the banks, stay in global memory (copied to LDS too: 128 points
// along y 10.5 us, 251 45.3 against 33.8, where direct sums without a second
// lane per output took 36.7).
// ---------------------------------------------------------------------------
constexpr int FIELD_NT = 1024;

// Lanes per output of a sum: a power of two <= 64 with `nout` outputs on nt
// threads.
__device__ __forceinline__ int dft_lanes(int nout, int nt) {
  int lp = 1;
  while (lp < 64 && 2 * lp * nout <= nt) lp *= 2;
  return lp;
}
__device__ __forceinline__ double lanes_sum(double v, int lp) {
  for (int d = lp >> 1; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}

// Transforms of nf fields of N complex values x (LDS, one after another; y: as
// much room for stage 1, unused when A = 1): out(f, k, re, im) for k < nout.
// sgn: 1 forward, -1 inverse (tw holds w = exp(-2 pi i / N)).  The whole
// workgroup calls it; x is complete before, and is free after a barrier.
template <typename F>
__device__ __forceinline__ void dft(const double *x, double *y, const double *tw, int nf, int N, int A, int nout,
                                    double sgn, F out) {
  const int nt = blockDim.x, tid = threadIdx.x;
  const int B = N / A;
  if (A > 1) {
    for (int t = tid; t < nf * N; t += nt) {
      const int f = t / N, r = t - f * N, k1 = r / B, n2 = r - k1 * B;
      const double *xf = x + 2 * (f * N + n2);
      double sr = 0., si = 0.;
      int m = 0;
      const int dm = B * k1;  // < N
#pragma unroll 4
      for (int n1 = 0; n1 < A; n1++) {
        const double wr = tw[2 * m], wi = sgn * tw[2 * m + 1];
        const double xr = xf[2 * B * n1], xi = xf[2 * B * n1 + 1];
        sr += xr * wr - xi * wi;
        si += xr * wi + xi * wr;
        m += dm;
        if (m >= N) m -= N;
      }
      y[2 * t] = sr;
      y[2 * t + 1] = si;
    }
    __syncthreads();
    x = y;
  }
  const int no = nf * nout, lp = dft_lanes(no, nt), sub = tid & (lp - 1), np = nt / lp;
  for (int t0 = 0; t0 < no; t0 += np) {
    const int t = min(t0 + tid / lp, no - 1);  // (lanes past the end repeat the last output)
    const int f = t / nout, k = t - f * nout;
    const double *xf = x + 2 * (f * N + k % A * B);
    double sr = 0., si = 0.;
    int m = (sub * k) % N;
    const int dm = (lp * k) % N;
#pragma unroll 4
    for (int n2 = sub; n2 < B; n2 += lp) {
      const double wr = tw[2 * m], wi = sgn * tw[2 * m + 1];
      const double xr = xf[2 * n2], xi = xf[2 * n2 + 1];
      sr += xr * wr - xi * wi;
      si += xr * wi + xi * wr;
      m += dm;
      if (m >= N) m -= N;
    }
    sr = lanes_sum(sr, lp);
    si = lanes_sum(si, lp);
    if (sub == 0) out(f, k, sr, si);
  }
}

// rho partials summed over their planes (planes o = part, part + parts, ...
// by the threads of a part), then the r2c transform of row iy.
__global__ __launch_bounds__(FIELD_NT) void k_rho_rfftx(const double *__restrict__ rho_part, long rho_outer, Geom g,
                                                        FieldBufs b, int sub1, int A) {
  extern __shared__ double sh[];  // row, stage 1 ([N0][2] each); part sums [parts][XL]
  const int N0 = g.n[0], N1 = g.n[1], nt = blockDim.x, tid = threadIdx.x;
  const int iy = blockIdx.x;
  const int nxh = N0 / 2 + 1;
  double *row = sh, *y = row + 2 * N0, *ps = y + 2 * N0;
  const int XL = (N0 + 63) & ~63, parts = nt / XL, x = tid % XL, part = tid / XL;
  if (x < N0 && part < parts) {
    const double *src = rho_part + x + (long)N0 * iy;
    const long plane = (long)N0 * N1;
    double s = 0.;
#pragma unroll 8
    for (long o = part; o < rho_outer; o += parts) s += src[plane * o];
    ps[part * XL + x] = s;
  }
  __syncthreads();
  if (tid < N0) {
    double s = 0.;
    for (int q = 0; q < parts; q++) s += ps[q * XL + tid];
    double r = s * g.dx[2] * g.dx[3];
    if (sub1) r -= 1.;
    row[2 * tid] = r;
    row[2 * tid + 1] = 0.;
  }
  __syncthreads();
  dft(row, y, b.twx, 1, N0, A, nxh, 1., [&](int, int k, double re, double im) {
    *(double2 *)(b.spec1 + 2 * (k + (long)nxh * iy)) = make_double2(re, im);
  });
}

__global__ __launch_bounds__(FIELD_NT) void k_poisson_y(Geom g, FieldBufs b, int A) {
  extern __shared__ double sh[];
  const int N0 = g.n[0], N1 = g.n[1], nt = blockDim.x, tid = threadIdx.x;
  const int nxh = N0 / 2 + 1, nyh = N1 / 2 + 1;
  const int kcol = blockIdx.x;
  const double *tw = b.twy;
  double *hat = sh;              // 3 * N1 complex: phi, ex, ey
  double *y = sh + 6 * N1;       // 3 * N1 complex: stage 1
  double *col = hat + 4 * N1;    // N1 complex, in ey's place until stage 2 of the forward transform
  for (int i = tid; i < 2 * N1; i += nt) col[i] = b.spec1[2 * (kcol + (long)nxh * (i >> 1)) + (i & 1)];
  __syncthreads();
  if (A == 1) {  // stage 2 reads the column itself: move it out of the result's way
    for (int i = tid; i < 2 * N1; i += nt) y[i] = col[i];
    col = y;
    __syncthreads();
  }
  const double kx0 = 2 * M_PI / g.maxPhy[0];
  const double ky0 = 2 * M_PI / g.maxPhy[1];
  const double normcoeff = 1.0 / (double)(N0 * N1);
  const double kx = kcol * kx0;
  dft(col, y, tw, 1, N1, A, N1, 1., [&](int, int q, double cr, double ci) {
    double pr, pi, er, ei, fr, fi;
    if (q == 0) {  // VMO/Efield.cpp:76-81, filter of :38-43
      const double kxf = kcol * (2 * M_PI / g.maxPhy[0]);
      const double filter = (kcol == 0) ? 0. : 1. / (kxf * kxf);
      er = ((kx * ci) * filter) * normcoeff;
      ei = ((-kx * cr) * filter) * normcoeff;
      fr = 0.;
      fi = 0.;
      pr = (cr * filter) * normcoeff;
      pi = (ci * filter) * normcoeff;
    } else {  // VMO/Efield.cpp:83-100
      const double ky = (q < nyh) ? q * ky0 : (q - N1) * ky0;
      const double k2 = kx * kx + ky * ky;
      const double sx = kx / k2, sy = ky / k2;
      er = (sx * ci) * normcoeff;
      ei = (-sx * cr) * normcoeff;
      fr = (sy * ci) * normcoeff;
      fi = (-sy * cr) * normcoeff;
      pr = (cr / k2) * normcoeff;
      pi = (ci / k2) * normcoeff;
    }
    hat[2 * q] = pr;
    hat[2 * q + 1] = pi;
    hat[2 * (N1 + q)] = er;
    hat[2 * (N1 + q) + 1] = ei;
    hat[2 * (2 * N1 + q)] = fr;
    hat[2 * (2 * N1 + q) + 1] = fi;
  });
  __syncthreads();
  if (A > 1) {
    dft(hat, y, tw, 3, N1, A, N1, -1., [&](int f, int iy, double re, double im) {
      *(double2 *)(b.spec2 + 2 * ((long)nxh * N1 * f + kcol + (long)nxh * iy)) = make_double2(re, im);
    });
    return;
  }
  // direct sums, the three fields side by side: one twiddle per term
  const int lp = dft_lanes(N1, nt), sub = tid & (lp - 1), np = nt / lp;
  for (int y0 = 0; y0 < N1; y0 += np) {
    const int iy = min(y0 + tid / lp, N1 - 1);
    double sr[3] = {0., 0., 0.}, si[3] = {0., 0., 0.};
    int m = (sub * iy) % N1;
    const int dm = (lp * iy) % N1;
#pragma unroll 4
    for (int q = sub; q < N1; q += lp) {
      const double wr = tw[2 * m], wi = -tw[2 * m + 1];  // exp(+2 pi i m/N)
#pragma unroll
      for (int fld = 0; fld < 3; fld++) {
        const double *h = hat + 2 * N1 * fld;
        sr[fld] += h[2 * q] * wr - h[2 * q + 1] * wi;
        si[fld] += h[2 * q] * wi + h[2 * q + 1] * wr;
      }
      m += dm;
      if (m >= N1) m -= N1;
    }
#pragma unroll
    for (int fld = 0; fld < 3; fld++) {
      sr[fld] = lanes_sum(sr[fld], lp);
      si[fld] = lanes_sum(si[fld], lp);
      if (sub == 0)
        *(double2 *)(b.spec2 + 2 * ((long)nxh * N1 * fld + kcol + (long)nxh * iy)) = make_double2(sr[fld], si[fld]);
    }
  }
}

__global__ __launch_bounds__(256) void k_c2rx_diag(Geom g, FieldBufs b) {
  extern __shared__ double sh[];
  const int N0 = g.n[0], N1 = g.n[1];
  const int nxh = N0 / 2 + 1;
  const int iy = blockIdx.x;
  double *rows = sh;             // 3 * nxh complex
  double *red = sh + 6 * nxh;    // 8 doubles for reductions
  for (int i = threadIdx.x; i < 3 * nxh; i += blockDim.x) {
    const int fld = i / nxh, k = i - fld * nxh;
    const double *src = b.spec2 + 2 * ((long)nxh * N1 * fld + k + (long)nxh * iy);
    rows[2 * i] = src[0];
    rows[2 * i + 1] = src[1];
  }
  __syncthreads();
  double pm = 0., pe = 0., pex = 0., pey = 0.;
  for (int ix = threadIdx.x; ix < N0; ix += blockDim.x) {
    // the three fields side by side (one twiddle load per term, each sum in
    // the same order as alone)
    double out[3];
#pragma unroll
    for (int fld = 0; fld < 3; fld++) out[fld] = rows[2 * nxh * fld];
    int m = ix;
#pragma unroll 8
    for (int k = 1; k < (N0 + 1) / 2; k++) {
      const double wr = b.twx[2 * m], wi = -b.twx[2 * m + 1];
#pragma unroll
      for (int fld = 0; fld < 3; fld++) {
        const double *X = rows + 2 * nxh * fld;
        out[fld] += 2.0 * (X[2 * k] * wr - X[2 * k + 1] * wi);
      }
      m += ix;
      if (m >= N0) m -= N0;
    }
    if ((N0 & 1) == 0)
#pragma unroll
      for (int fld = 0; fld < 3; fld++) out[fld] += rows[2 * nxh * fld + 2 * (N0 / 2)] * ((ix & 1) ? -1.0 : 1.0);
    const long id = ix + (long)N0 * iy;
    b.rho[id] = out[0];
    b.ex[id] = out[1];
    b.ey[id] = out[2];
    b.exy[2 * id] = out[1];
    b.exy[2 * id + 1] = out[2];
    pm += out[0];
    pe += out[1] * out[1] + out[2] * out[2];
    pex += out[1] * out[1];
    pey += out[2] * out[2];
  }
  const double s0 = block_sum(pm, red);
  const double s1 = block_sum(pe, red);
  const double s2 = block_sum(pex, red);
  const double s3 = block_sum(pey, red);
  if (threadIdx.x == 0) {
    b.diag_part[4 * iy + 0] = s0;
    b.diag_part[4 * iy + 1] = s1;
    b.diag_part[4 * iy + 2] = s2;
    b.diag_part[4 * iy + 3] = s3;
  }
}

// Slice s of the density partials: tmp[s][i] = sum of planes o = s, s + S, ...
__global__ __launch_bounds__(256) void k_rho_slices(const double *__restrict__ rho_part, long rho_outer, long npt,
                                                    double *__restrict__ tmp) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int s = blockIdx.y, S = gridDim.y;
  if (i >= npt) return;
  double acc = 0.;
  for (long o = s; o < rho_outer; o += S) acc += rho_part[i + npt * o];
  tmp[i + npt * s] = acc;
}

// Analytic fields of idcase 2 and 6 (VMO/Field.cpp:81-108); rho is kept.
__global__ __launch_bounds__(256) void k_analytic_field(const double *__restrict__ rho_part, long rho_outer, Geom g,
                                                        FieldBufs b) {
  __shared__ double red[8];
  const int N0 = g.n[0], N1 = g.n[1];
  const int iy = blockIdx.x;
  double pm = 0., pe = 0., pex = 0., pey = 0.;
  for (int ix = threadIdx.x; ix < N0; ix += blockDim.x) {
    double s = 0.;
#pragma unroll 8
    for (long o = 0; o < rho_outer; o++) s += rho_part[ix + (long)N0 * (iy + (long)N1 * o)];
    const double r = s * g.dx[2] * g.dx[3];
    const double e = (g.idcase == 2) ? -(g.minPhy[0] + ix * g.dx[0]) : -(g.minPhy[1] + iy * g.dx[1]);
    const long id = ix + (long)N0 * iy;
    b.rho[id] = r;
    b.ex[id] = e;
    b.ey[id] = 0.;
    b.exy[2 * id] = e;
    b.exy[2 * id + 1] = 0.;
    pm += r;
    pe += e * e;
    pex += e * e;
  }
  const double s0 = block_sum(pm, red);
  const double s1 = block_sum(pe, red);
  const double s2 = block_sum(pex, red);
  const double s3 = block_sum(pey, red);
  if (threadIdx.x == 0) {
    b.diag_part[4 * iy + 0] = s0;
    b.diag_part[4 * iy + 1] = s1;
    b.diag_part[4 * iy + 2] = s2;
    b.diag_part[4 * iy + 3] = s3;
  }
}

// Diags::compute and computeL2norm, VMO/Diags.cpp:16-76.
// The record index is iter, or -- iter_dev non-null, for launches replayed
// from a captured graph -- *iter_dev + 1, which is then stored back.
__global__ __launch_bounds__(256) void k_diag_final(Geom g, FieldBufs b, const double *__restrict__ l2_part, long n_l2,
                                                    int iter, int with_l2, int *__restrict__ iter_dev) {
  __shared__ double red[8];
  const int N1 = g.n[1];
  double s[4];
  for (int c = 0; c < 4; c++) {
    double v = 0.;
    for (int iy = threadIdx.x; iy < N1; iy += blockDim.x) v += b.diag_part[4 * iy + c];
    s[c] = block_sum(v, red);
  }
  double l2 = 0.;
  if (with_l2) {
    double v = 0.;
    // unrolled so that the independent loads are in flight together (the
    // additions keep their order)
#pragma unroll 8
    for (long i = threadIdx.x; i < n_l2; i += blockDim.x) v += l2_part[i];
    l2 = block_sum(v, red);
  }
  if (threadIdx.x == 0) {
    if (iter_dev) {
      iter = *iter_dev + 1;
      *iter_dev = iter;
    }
    const int nb = b.nbiter + 1;
    if (iter < 0 || iter >= nb) return;
    double it_nrj = sqrt(s[1] * g.dx[0] * g.dx[1]);
    it_nrj = it_nrj > 1.e-30 ? log(it_nrj) : -1.e9;
    b.diag[0 * nb + iter] = it_nrj;
    b.diag[1 * nb + iter] = sqrt(0.5 * s[2] * g.dx[0] * g.dx[1]);
    b.diag[2 * nb + iter] = sqrt(0.5 * s[3] * g.dx[0] * g.dx[1]);
    b.diag[3 * nb + iter] = s[0] * g.dx[0] * g.dx[1];
    if (with_l2) b.diag[4 * nb + iter] = sqrt(l2 * g.dx[0] * g.dx[1] * g.dx[2] * g.dx[3]);
  }
}

// Largest divisor of n up to its square root.
static int dft_factor(int n) {
  int a = 1;
  for (int d = 2; d * d <= n; d++)
    if (n % d == 0) a = d;
  return a;
}

void launch_field(const Geom &g, const FieldBufs &b, const double *rho_part, long rho_outer, const double *l2_part,
                  long n_l2, int iter, bool record_diag, hipStream_t s, int *iter_dev) {
  const int N0 = g.n[0], N1 = g.n[1];
  const int nxh = N0 / 2 + 1;
  if (g.idcase == 2 || g.idcase == 6) {
    if (rho_outer > 64 && b.rho_tmp) {
      const long npt = (long)N0 * N1;
      hipLaunchKernelGGL(k_rho_slices, dim3((unsigned)((npt + 255) / 256), RHO_SLICES), dim3(256), 0, s, rho_part,
                         rho_outer, npt, b.rho_tmp);
      rho_part = b.rho_tmp;
      rho_outer = RHO_SLICES;
    }
    hipLaunchKernelGGL(k_analytic_field, dim3(N1), dim3(256), 0, s, rho_part, rho_outer, g, b);
  } else {
    const int sub1 = (g.idcase == 10 || g.idcase == 20);
    // along x a thread per eight planes and point of the density sum, 256 to
    // 1024 (a solve of 48 x 48 x 32 x 48: 58 us with 1024 and a launch more for
    // the twiddles, 54.7); along y a thread per output of the inverse
    // transforms, or two or more lanes per output of a direct sum
    const int Ax = dft_factor(N0), Ay = dft_factor(N1);
    const int ty = Ay == 1 ? (N1 > 128 ? 512 : 256) : std::min(FIELD_NT, (3 * N1 + 63) / 64 * 64);
    const int XL = (N0 + 63) & ~63;
    const int tx = std::min((long)FIELD_NT, std::max(256l, XL * ((rho_outer + 7) / 8)));
    hipLaunchKernelGGL(k_rho_rfftx, dim3(N1), dim3(tx), sizeof(double) * (4 * N0 + tx / XL * XL), s,
                       rho_part, rho_outer, g, b, sub1, Ax);
    hipLaunchKernelGGL(k_poisson_y, dim3(nxh), dim3(ty), sizeof(double) * 12 * N1, s, g, b, Ay);
    hipLaunchKernelGGL(k_c2rx_diag, dim3(N1), dim3(256), sizeof(double) * (6 * nxh + 8), s, g, b);
  }
  if (record_diag)
    hipLaunchKernelGGL(k_diag_final, dim3(1), dim3(256), 0, s, g, b, l2_part, n_l2, iter, l2_part != nullptr ? 1 : 0,
                       iter_dev);
}

}  // namespace vlp
