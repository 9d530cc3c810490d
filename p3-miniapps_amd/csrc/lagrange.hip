// lagrange.hip -- the Lagrange split-step vlp4d (miniapps/vlp4d/openmp, "VO/").
//
// One step is the Strang split of VO/timestep.hpp:11-55: 1-D advections along
// x and y by dt/2 (displacement dt*v of the cell's own velocity), the density
// of the result and the FFT Poisson solve (field.hip, shared with the spline
// path), 1-D advections along vx and vy by dt (displacement dt*E(x, y)), and x,
// y by dt/2 again.  Every advection is the 6-point order-5 interpolation of
// VO/advect.hpp:72-86 on a periodic axis (velocity too).  The x and
// y passes go through an LDS-resident (x, y) plane, the velocity passes through
// LDS rows of vx and register windows of vy, so a step in a run of steps
// streams f twice (8 B read + 8 B write per cell each).
#include <cstdlib>

#include "device_common.hpp"
#include "vlp4d_internal.hpp"

namespace vlp {

namespace {

// The order-5 basis of VO/advect.hpp:72-86, px in [2, 3).
__device__ __forceinline__ void lag5_basis(double px, double c[6]) {
  const double pxm2 = px - 2.;
  const double sq = pxm2 * pxm2;
  const double p01 = pxm2 * (pxm2 - 1.);
  c[0] = (-1. / 24) * p01 * (pxm2 + 1.) * (pxm2 - 2.) * (pxm2 - 1.);
  c[1] = (1. / 24.) * p01 * (pxm2 - 2.) * (5 * sq + pxm2 - 8.);
  c[2] = (-1. / 12.) * (pxm2 - 1.) * (pxm2 - 2.) * (pxm2 + 1.) * (5 * sq - 3 * pxm2 - 6.);
  c[3] = (1. / 12.) * pxm2 * (pxm2 + 1.) * (pxm2 - 2.) * (5 * sq - 7 * pxm2 - 4.);
  c[4] = (-1. / 24.) * p01 * (pxm2 + 1.) * (5 * sq - 11 * pxm2 - 2.);
  c[5] = (1. / 24.) * p01 * pxm2 * (pxm2 + 1.) * (pxm2 - 2.);
}

// Foot of a 1-D advection by `dep` on the periodic axis d (VO/advect.hpp:
// 137-154): the six stencil indices, already wrapped into [0, N), and weights.
__device__ __forceinline__ void lag_stencil(const Geom &g, int d, double h, double dep, int j[6], double c[6]) {
  const double hmin = g.minPhy[d], hwidth = g.maxPhy[d] - g.minPhy[d], dh = g.dx[d];
  const double idh = 1. / dh;
  const int N = g.n[d];
  const double hstar = hmin + fmod(hwidth + h - dep - hmin, hwidth);
  const int ip = (int)floor((hstar - hmin) * idh);
  lag5_basis(2. + idh * (hstar - (hmin + ip * dh)), c);
  // the reference wraps with (N + ip - 2 + k) % N; a full modulo keeps any
  // foot (even beyond one box width) in range
  int b = (ip - 2) % N;
  if (b < 0) b += N;
#pragma unroll
  for (int k = 0; k < 6; k++) {
    const int q = b + k;
    j[k] = q >= N ? q - N : q;
  }
}

}  // namespace

// Logical block of hardware block b: block b runs on XCD b % 8, so with the
// grid a multiple of 8 each XCD takes one contiguous range of logical blocks
// and the stencil neighbours of a block (the next rows, planes or lines) sit
// in the same L2.
__device__ __forceinline__ unsigned xcd_block(unsigned b, unsigned grid) {
  return (grid & 7u) ? b : (b & 7u) * (grid >> 3) + (b >> 3);
}

// advect_1D_x (VO/advect.hpp:112-158).  Lane per (x, vx, vy), x fastest; the
// weights depend on x and vx only, so each lane computes them once and runs
// down the y rows of its (vx, vy) plane.
__global__ __launch_bounds__(256) void k_lag_x(const double *__restrict__ in, double *__restrict__ out, Geom g,
                                               double dt) {
  const int N0 = g.n[0], N1 = g.n[1], N2 = g.n[2], N3 = g.n[3];
  const unsigned t = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (t >= (unsigned)N0 * N2 * N3) return;
  const int ix = (int)(t % (unsigned)N0);
  const unsigned r = t / (unsigned)N0;  // ivx + N2 * ivy
  const int ivx = (int)(r % (unsigned)N2);
  const double vx = g.minPhy[2] + ivx * g.dx[2];
  int j[6];
  double c[6];
  lag_stencil(g, 0, g.minPhy[0] + ix * g.dx[0], dt * vx, j, c);
  const double *src = in + (size_t)r * N1 * N0;
  double *dst = out + (size_t)r * N1 * N0 + ix;
#pragma unroll 2
  for (int iy = 0; iy < N1; iy++) {
    const double *row = src + (size_t)iy * N0;
    double s = 0.;
#pragma unroll
    for (int k = 0; k < 6; k++) s += c[k] * row[j[k]];
    dst[(size_t)iy * N0] = s;
  }
}

// advect_1D_y (VO/advect.hpp:160-204): lane per (x, y, vy), looping over vx
// (the weights depend on y and vy only).  With rho_part, also the velocity
// sum of the result over vx: rho_part[vy][y][x] (field_rho, VO/field.cpp:5-29).
__global__ __launch_bounds__(256) void k_lag_y(const double *__restrict__ in, double *__restrict__ out, Geom g,
                                               double dt, double *__restrict__ rho_part) {
  const int N0 = g.n[0], N1 = g.n[1], N2 = g.n[2], N3 = g.n[3];
  const unsigned t = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  const unsigned plane = (unsigned)N0 * N1;
  if (t >= plane * N3) return;
  const unsigned pxy = t % plane;
  const int ix = (int)(pxy % (unsigned)N0);
  const int iy = (int)(pxy / (unsigned)N0);
  const int ivy = (int)(t / plane);
  const double vy = g.minPhy[3] + ivy * g.dx[3];
  int j[6];
  double c[6];
  lag_stencil(g, 1, g.minPhy[1] + iy * g.dx[1], dt * vy, j, c);
  const double *src = in + (size_t)ivy * N2 * plane + ix;
  double *dst = out + (size_t)ivy * N2 * plane + pxy;
  double sum = 0.;
#pragma unroll 2
  for (int ivx = 0; ivx < N2; ivx++) {
    const double *p = src + (size_t)ivx * plane;
    double s = 0.;
#pragma unroll
    for (int k = 0; k < 6; k++) s += c[k] * p[j[k] * N0];
    dst[(size_t)ivx * plane] = s;
    sum += s;
  }
  if (rho_part) rho_part[t] = sum;
}

// advect_1D_vx then advect_1D_vy (VO/advect.hpp:206-301), displacements
// dt*E(x, y) along the velocity axes, in one pass over f.  A shift is the same
// for a whole line, so the foot of point iv is that of point 0 moved by iv
// cells: one set of weights per (x, y) point and axis, and a window of six
// values that slides by one per output (the reference recomputes the foot per
// point; the two agree to rounding, and where rounding moves a foot across a
// node the interpolant, continuous there, gives the same value).
//
// A workgroup takes WP points of the (x, y) plane, all of vx and a segment of
// len rows of vy; a lane one point, S consecutive vx and the segment's rows in
// turn.  A row's values go through LDS (two buffers, one barrier a row) for the
// vx pass, whose results enter the lane's windows of six rows for the vy pass,
// while the next row's values are in flight.  The rows that a wave reads may
// differ from lane to lane, as the shifts do.
//
// Bound: HBM (16 bytes per cell and 5 rows' halo per segment; 0.91 ms at 128^4
// at the 4.7 TB/s of a large copy).  WP = 16 points are one 128-byte line of
// every (vx, vy) row, S = 4 keeps the windows within 4 waves per SIMD.  128^4
// 0.87 ms, 1.69 ms as a pass per axis; 48^4 23 us (34), 100 x 91 x 77 x 64
// 0.24 ms (0.33).
constexpr int VV_WP = 16, VV_S = 4;

template <int WP, int S>
__global__ __launch_bounds__(1024) void k_lag_vv(const double *__restrict__ in, double *__restrict__ out, Geom g,
                                                const double *__restrict__ ex, const double *__restrict__ ey,
                                                double dt, int len, int nseg) {
  extern __shared__ double rows[];  // two rows of N2 x WP
  const int N2 = g.n[2], N3 = g.n[3];
  const unsigned P = (unsigned)g.n[0] * g.n[1];
  const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
  const int k0 = (int)(blk % nseg) * len, k1 = min(N3, k0 + len);
  const int l = threadIdx.x % WP;
  const unsigned at = (blk / nseg) * WP + l, pxy = min(at, P - 1);
  const int vx0 = (threadIdx.x / WP) * S;  // (lanes past the plane or the vx axis repeat its last point)
  const int nv = at < P ? min(S, max(0, N2 - vx0)) : 0;  // results to store
  double c2[6], c3[6];
  int j[6];
  lag_stencil(g, 2, g.minPhy[2], dt * ex[pxy], j, c2);
  int q0 = j[0] + min(vx0, N2 - 1);
  q0 = q0 >= N2 ? q0 - N2 : q0;
  lag_stencil(g, 3, g.minPhy[3], dt * ey[pxy], j, c3);
  int r = (j[0] + k0) % N3;  // the row to load next
  unsigned o[S];
#pragma unroll
  for (int i = 0; i < S; i++) o[i] = pxy + (unsigned)min(vx0 + i, N2 - 1) * P;
  const size_t sR = (size_t)P * N2;
  double v[S], w[S][6];
  auto load = [&] {
    const double *src = in + (size_t)r * sR;
#pragma unroll
    for (int i = 0; i < S; i++) v[i] = src[o[i]];
    r = r + 1 == N3 ? 0 : r + 1;
  };
#pragma unroll
  for (int i = 0; i < S; i++)
#pragma unroll
    for (int m = 0; m < 6; m++) w[i][m] = 0.;
  load();
  double *dst = out + (size_t)k0 * sR;
  for (int k = k0 - 5; k < k1; k++) {
    double *buf = rows + ((k - k0) & 1) * N2 * WP;
#pragma unroll
    for (int i = 0; i < S; i++)
      if (vx0 + i < N2) buf[(vx0 + i) * WP + l] = v[i];
    __syncthreads();
    if (k + 1 < k1) load();
    {
      int q = q0;
      double u[6];
#pragma unroll
      for (int m = 0; m < 5; m++) {
        u[m] = buf[q * WP + l];
        q = q + 1 == N2 ? 0 : q + 1;
      }
#pragma unroll
      for (int i = 0; i < S; i++) {
        u[(5 + i) % 6] = buf[q * WP + l];
        q = q + 1 == N2 ? 0 : q + 1;
        double s = c2[0] * u[i % 6];
#pragma unroll
        for (int m = 1; m < 6; m++) s += c2[m] * u[(i + m) % 6];
#pragma unroll
        for (int m = 0; m < 5; m++) w[i][m] = w[i][m + 1];
        w[i][5] = s;
      }
    }
    if (k >= k0) {
#pragma unroll
      for (int i = 0; i < S; i++) {
        double s = c3[0] * w[i][0];
#pragma unroll
        for (int m = 1; m < 6; m++) s += c3[m] * w[i][m];
        if (i < nv) dst[o[i]] = s;
      }
      dst += sR;
    }
  }
}

// x/2 then y/2 through one LDS-resident (x, y) plane (the first or last pair of
// VO/timestep.hpp:11-55 in one pass over f), or, TWICE, the last pair of a step
// and the first pair of the next; RHO also sums the result over the
// workgroup's vx planes (field_rho).  Workgroup per (vy, run of G vx planes).
// A plane goes from registers (loaded during the previous plane's passes)
// to LDS; each pass gives a wave 64 lines across the lanes and S consecutive
// points along them (FLAT: the lanes take the lines' segments one after another,
// so that no lane idles where a plane has few lines).  The displacement is that
// of the line's velocity, the same
// for all its points, so a lane has one set of weights and slides a six-value
// window along its points: (S + 5) / S LDS reads per point, at addresses
// uniform in the wave up to the lane's line (and, FLAT, its segment).  A pass in place reads, waits for
// the workgroup and writes; the last y pass goes from LDS to HBM, and its
// points are the same in every plane, so their density sums stay in
// registers.  The LDS row pitch is odd, so neither direction has bank conflicts.
//
// Bound: HBM (16 bytes per cell; 0.91 ms per pass at 128^4 at the 4.7 TB/s of a
// large copy), with one 132 KB plane per CU there: a TWICE pass takes 1.17 ms.
// With RHO it moves 5.33 GB, not 4.29, since 60 registers of the density sums of
// 32 points go through scratch memory; its LDS work (about 0.35 ms) and barriers
// are not all hidden behind the loads.  128^4 step in a run of steps 4.14 -> 2.97 ms: before, the pair read
// six stencil values per point and pass from LDS (1.01 ms), the density was a
// pass of its own (0.41 ms) and neighbouring steps each had their pair.
struct LagTab {  // stencil of a line: six weights and the wrapped first index of point 0
  double w[6];
  int b;
};

// The stencils of the x/2 and y/2 passes, fixed for a context: x lines for
// every vx, then y lines for every vy.
__global__ __launch_bounds__(256) void k_lag_tables(LagTab *__restrict__ tab, Geom g, double dt) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= g.n[2] + g.n[3]) return;
  const int d = i < g.n[2] ? 0 : 1, iv = d ? i - g.n[2] : i;
  int j[6];
  lag_stencil(g, d, g.minPhy[d], dt * (g.minPhy[2 + d] + iv * g.dx[2 + d]), j, tab[i].w);
  tab[i].b = j[0];
}

// A copy of v that the compiler takes for a new value: uniform in the wave, or
// (VEC) one per lane.
template <bool VEC> __device__ __forceinline__ void opaque(int &v) {
  if constexpr (VEC) asm volatile("" : "+v"(v));
  else asm volatile("" : "+s"(v));
}

// Results of the line at `line` (LDS, stride st between its N points) at the S
// points from p0 on (periodic), each handed to out(i, value).  Everything but
// `line` and (FLAT) p0 is uniform in the wave.  (The opaque copy keeps the
// positions from being hoisted out of the loop over planes, where they would be
// spilled.)
template <int S, bool FLAT, typename F>
__device__ __forceinline__ void lag_slide(const double *line, int st, int N, int p0, const LagTab &t, F out) {
  int q = t.b + p0;
  q = q >= N ? q - N : q;
  opaque<FLAT>(q);
  const double *p = line + q * st;
  const int wrap = st - N * st;
  double w[6];
#pragma unroll
  for (int k = 0; k < 5; k++) {
    w[k] = *p;
    q++;
    p += q == N ? wrap : st;
    q = q == N ? 0 : q;
  }
#pragma unroll
  for (int i = 0; i < S; i++) {
    w[(5 + i) % 6] = *p;
    q++;
    p += q == N ? wrap : st;
    q = q == N ? 0 : q;
    double s = 0.;
#pragma unroll
    for (int k = 0; k < 6; k++) s += t.w[k] * w[(i + k) % 6];
    out(i, s);
    // at most four points' reads in flight (registers)
    if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
  }
}

template <int S, int NT, bool TWICE, bool RHO, bool FLAT>
__global__ __launch_bounds__(NT) void k_lag_plane(const double *__restrict__ in, double *__restrict__ out, Geom g,
                                                    const LagTab *__restrict__ tab, int G, int nchunk,
                                                    double *__restrict__ rho_part) {
  extern __shared__ double pl[];  // the (x, y) plane, rows of `pitch`
  const int N0 = g.n[0], N1 = g.n[1], N2 = g.n[2], N3 = g.n[3];
  const int P = N0 * N1, pitch = N0 | 1;
  const int ivy = blockIdx.x / nchunk, chunk = blockIdx.x % nchunk;
  const int v0 = chunk * G, v1 = min(N2, v0 + G);
  const int l = threadIdx.x, nl = blockDim.x, lane = l & 63;
  const int wave = __builtin_amdgcn_readfirstlane(l >> 6);
  const LagTab &ty = tab[N2 + ivy];
  // x pass: rows 64 rg + lane, points xs .. xs + xn - 1
  const int nsx = (N0 + S - 1) / S, nsy = (N1 + S - 1) / S;
  const int xrow = FLAT ? l % N1 : 64 * (wave / nsx) + lane, xs = S * (FLAT ? l / N1 : wave % nsx);
  const int xn = min(S, N0 - xs);
  const bool xact = FLAT ? xn > 0 : xrow < N1;
  double *const xl = pl + (xact ? xrow : 0) * pitch;
  // y pass: columns 64 cg + lane, points ys .. ys + yn - 1
  const int ycol = FLAT ? l % N0 : 64 * (wave / nsy) + lane, ys = S * (FLAT ? l / N0 : wave % nsy);
  const int yn = min(S, N1 - ys);
  const bool yact = FLAT ? yn > 0 : ycol < N0;
  double *const yl = pl + (yact ? ycol : 0);
  // this lane's plane points l, l + nl, ..., at most S of them
  const int dcol = nl % N0, drow = nl / N0, col0 = l % N0, row0 = l / N0;
  constexpr bool AHEAD = NT <= 512;  // a plane's loads go out a pass ahead of its use (registers permitting)
  double r[AHEAD ? S : 1], o[S], rho[RHO ? S : 1];
  if constexpr (RHO)
#pragma unroll
    for (int i = 0; i < S; i++) rho[i] = 0.;
  // (opaque copies of the lane index keep the addresses and conditions of the
  // plane's points from being held across the loop over planes)
  auto load = [&](const double *src) {
    int p = l;
    asm volatile("" : "+v"(p));
#pragma unroll
    for (int m = 0; m < S; m++) {
      // (lanes past the plane repeat its last point; a 32-bit byte offset)
      r[m] = *(const double *)((const char *)src + 8u * (unsigned)min(p, P - 1));
      p += nl;
      if (m % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto keep = [&](int i, double v) { o[i] = v; };
  if constexpr (AHEAD) load(in + ((size_t)ivy * N2 + v0) * P);
  for (int ivx = v0; ivx < v1; ivx++) {
    const size_t off = ((size_t)ivy * N2 + ivx) * P;
    const LagTab &tx = tab[ivx];
    __syncthreads();  // the previous plane's last pass has read pl
    {
      int p = l, col = col0, o = row0 * pitch + col0;
      asm volatile("" : "+v"(p), "+v"(col), "+v"(o));
#pragma unroll
      for (int m = 0; m < S; m++) {
        // (lanes past the plane write to a slot behind it)
        const int at = p < P ? o : pitch * N1;
        if constexpr (AHEAD) pl[at] = r[m];
        else pl[at] = *(const double *)((const char *)(in + off) + 8u * (unsigned)min(p, P - 1));
        p += nl;
        col += dcol;
        o += drow * pitch + dcol;
        if (col >= N0) {
          col -= N0;
          o += pitch - N0;
        }
      }
    }
    __syncthreads();
    if constexpr (AHEAD)
      if (ivx + 1 < v1) load(in + off + P);  // in flight during the passes
#pragma unroll
    for (int half = 0; half < (TWICE ? 2 : 1); half++) {
      if (xact) lag_slide<S, FLAT>(xl, 1, N0, xs, tx, keep);
      __syncthreads();
      if (xact) {
        int n = xn;
        opaque<FLAT>(n);
#pragma unroll
        for (int i = 0; i < S; i++)
          if (i < n) xl[xs + i] = o[i];
      }
      __syncthreads();
      if (TWICE && half == 0) {
        if (yact) lag_slide<S, FLAT>(yl, pitch, N1, ys, ty, keep);
        __syncthreads();
        if (yact) {
          int n = yn, row = pitch;
          opaque<FLAT>(n);
          opaque<false>(row);
#pragma unroll
          for (int i = 0; i < S; i++)
            if (i < n) yl[(ys + i) * row] = o[i];
        }
        __syncthreads();
      }
    }
    if (yact) {
      // a scalar row address and the lane's offset: its column and (FLAT) first row
      char *dst = (char *)(out + off + (FLAT ? 0 : (size_t)ys * N0));
      int at = 8 * (ycol + (FLAT ? ys * N0 : 0)), n = yn, row = 8 * N0;
      opaque<true>(at);
      opaque<FLAT>(n);
      opaque<false>(row);
      if (!FLAT && n == S) {  // (no branch between the points)
        lag_slide<S, FLAT>(yl, pitch, N1, ys, ty, [&](int i, double v) {
          *(double *)(dst + (unsigned)at) = v;
          dst += row;
          if constexpr (RHO) rho[i] += v;
        });
      } else {
        lag_slide<S, FLAT>(yl, pitch, N1, ys, ty, [&](int i, double v) {
          if (i < n) *(double *)(dst + (unsigned)at) = v;
          dst += row;
          if constexpr (RHO) rho[i] += v;
        });
      }
    }
  }
  if constexpr (RHO)
    if (yact) {
      double *dst = rho_part + ((size_t)chunk * N3 + ivy) * P + (size_t)ys * N0 + ycol;
#pragma unroll
      for (int i = 0; i < S; i++)
        if (i < yn) dst[(size_t)i * N0] = rho[i];
    }
}

// Waves of a workgroup for S points per lane and pass: every pass has a wave
// for each of its 64-line groups and S-point segments, or (flat) a lane for
// each line and segment.
static int lag_waves(const Geom &g, int S, bool flat) {
  const int N0 = g.n[0], N1 = g.n[1], nsx = (N0 + S - 1) / S, nsy = (N1 + S - 1) / S;
  const int x = flat ? (N1 * nsx + 63) / 64 : (N1 + 63) / 64 * nsx;
  const int y = flat ? (N0 * nsy + 63) / 64 : (N0 + 63) / 64 * nsy;
  return x > y ? x : y;
}

static size_t lag_xy_lds(const Geom &g) { return ((size_t)(g.n[0] | 1) * g.n[1] + 1) * sizeof(double); }

// vx runs per vy for workgroups of `waves`: the fewest rounds of
// workgroups over the CUs, counting one plane time for a run's start, with
// runs of at least four planes (their density sums are stored per run) unless
// there are at most three workgroups per CU, whose planes one after another are
// latency: one step a call of 10^4 85 -> 70 us, 24^4 89 -> 80, 100 x 91 x 12 x 12
// 134 -> 102; 16 x 16 x 64 x 64 with runs of two 103 us, with four 100.  (Counting
// 32 waves per CU, not those whose registers fit, 72 x 60 x 60 x 60 took one
// workgroup per CU more than there is room for: four steps a call 250 -> 197 us
// per step.)
static int lag_chunks(const Geom &g, int waves, int points) {
  int per_cu = (int)(160 * 1024 / lag_xy_lds(g));
  // the waves whose registers fit a CU
  const int fit = points == 16 ? 12 : waves <= 8 ? 8 : 16;
  if (per_cu > fit / waves) per_cu = fit / waves;
  if (per_cu > 8) per_cu = 8;
  const long cap = 256L * (per_cu < 1 ? 1 : per_cu);
  int best = 1;
  long cost = -1;
  for (int n = 1; n <= g.n[2]; n++) {
    const int G = (g.n[2] + n - 1) / n;
    if (n > 1 && G < 4 && (long)g.n[3] * n > 3 * 256) break;
    if ((g.n[2] + G - 1) / G != n) continue;  // the same runs in fewer workgroups
    const long c = ((long)g.n[3] * n + cap - 1) / cap * (G + 1);
    if (cost < 0 || c < cost) {
      cost = c;
      best = n;
    }
  }
  return best;
}

// 16 points per lane where that takes at most 8 waves, or 32 (the plane's loads
// run a pass ahead and the density is summed along), else 32 and up to 16 waves
// (longest planes: neither, registers).  The 16-point form goes flat where only
// that fits 8 waves (against 32 points in 64-line groups, one step a call: 68 x
// 68 x 24 x 24 144 -> 116 us, 10 x 251 x 60 x 60 405 -> 218, 160 x 10 x 60 x 60
// 329 -> 153) or takes half the waves (100 x 10 x 60 x 60 183 -> 127; 31 x 64 x 40 x
// 40, 3 instead of 4, 84 -> 87).
// With 32 points a lane's density sums do not fit the registers (54 spills, one
// workgroup per CU): a pass of one pair takes 16 points, up to 16 waves and no
// sums as long as the density pass finds f in the 256 MB last-level cache: one
// step a call of 90 x 90 x 24 x 24 162 -> 145 us, 100 x 91 x 60 x 60 (262 MB) 628
// -> 585; but 90 x 128 x 60 x 60 (332 MB) 597 -> 613.
LagPlan lag_xy_plan(const Geom &g) {
  LagPlan p;
  if (const char *e = getenv("VLP4D_LAG_FUSED"))
    if (atoi(e) == 0) return p;
  if (lag_xy_lds(g) > 160 * 1024) return p;
  const struct { int points; bool flat; int waves; } forms[] = {{16, false, 8}, {16, true, 8}, {32, false, 16}};
  for (const auto &f : forms) {
    const int w = lag_waves(g, f.points, f.flat);
    if (w > f.waves || (f.points == 16 && !f.flat && 2 * lag_waves(g, 16, true) <= w)) continue;
    p.points = f.points;
    p.flat = f.flat;
    p.waves = w;
    p.chunks = lag_chunks(g, w, f.points);
    p.sums = w <= 8;
    break;
  }
  const int w16 = lag_waves(g, 16, false);
  const double mib = 8. * g.n[0] * g.n[1] * g.n[2] * g.n[3] / (1 << 20);
  if (p.points == 32 && p.sums && w16 <= 16 && mib <= 256.) p.waves1 = w16;
  return p;
}

// Initial conditions of VO/init.cpp:144-285 (TSI20 differs from the spline
// miniapp's).
__global__ __launch_bounds__(256) void k_lag_init(double *__restrict__ f, Geom g) {
  const int N0 = g.n[0], N1 = g.n[1], N2 = g.n[2];
  const long ncell = (long)N0 * N1 * N2 * g.n[3];
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ncell) return;
  const int ix = (int)(t % N0), iy = (int)((t / N0) % N1), ivx = (int)((t / ((long)N0 * N1)) % N2),
            ivy = (int)(t / ((long)N0 * N1 * N2));
  const double x = g.minPhy[0] + ix * g.dx[0], y = g.minPhy[1] + iy * g.dx[1];
  const double vx = g.minPhy[2] + ivx * g.dx[2], vy = g.minPhy[3] + ivy * g.dx[3];
  double v = 0.;
  if (g.idcase == 2 || g.idcase == 5) {  // CYL02 (x, vx) / CYL05 (y, vy)
    const double PERIOD = 0.5 * M_PI, AMPLI = 4, cc = 0.50 * (6. / 16.), rc = 0.50 * (4. / 16.);
    const double xx = g.idcase == 2 ? x : y, vv = g.idcase == 2 ? vx : vy;
    double hv = 0.0, hx = 0.0;
    if ((vv <= cc + rc) && (vv >= cc - rc)) hv = cos(PERIOD * ((vv - cc) / rc));
    else if ((vv <= -cc + rc) && (vv >= -cc - rc)) hv = -cos(PERIOD * ((vv + cc) / rc));
    if ((xx <= cc + rc) && (xx >= cc - rc)) hx = cos(PERIOD * ((xx - cc) / rc));
    else if ((xx <= -cc + rc) && (xx >= -cc - rc)) hx = -cos(PERIOD * ((xx + cc) / rc));
    v = AMPLI * hx * hv;
  } else if (g.idcase == 10) {  // SLD10
    const double sum = vx * vx + vy * vy;
    v = (1. / (2 * M_PI)) * exp(-0.5 * (sum)) * (1 + 0.05 * (cos(0.5 * x) * cos(0.5 * y)));
  } else {  // TSI20
    const double xi = 0.90, alpha = 0.05;
    const double sum = vx * vx + vy * vy;
    v = (1 + alpha * (cos(0.5 * x))) * 1 / (2 * M_PI) * ((2 - 2 * xi) / (3 - 2 * xi)) * (1 + .5 * vx * vx / (1 - xi)) *
        exp(-.5 * sum);
  }
  f[t] = v;
}

static unsigned blocks(long n) { return (unsigned)((n + 255) / 256); }

void launch_lag_init(const Geom &g, double *f, hipStream_t s) {
  const long n = (long)g.n[0] * g.n[1] * g.n[2] * g.n[3];
  hipLaunchKernelGGL(k_lag_init, dim3(blocks(n)), dim3(256), 0, s, f, g);
}

void launch_lag_x(const Geom &g, const double *in, double *out, double dt, hipStream_t s) {
  const long n = (long)g.n[0] * g.n[2] * g.n[3];
  hipLaunchKernelGGL(k_lag_x, dim3(blocks(n)), dim3(256), 0, s, in, out, g, dt);
}

size_t lag_tables_bytes(const Geom &g) { return (size_t)(g.n[2] + g.n[3]) * sizeof(LagTab); }

void launch_lag_tables(const Geom &g, void *tab, double dt, hipStream_t s) {
  hipLaunchKernelGGL(k_lag_tables, dim3(blocks(g.n[2] + g.n[3])), dim3(256), 0, s, (LagTab *)tab, g, dt);
}

template <int S, int NT, bool TWICE, bool RHO, bool FLAT = false>
static void launch_plane(const Geom &g, const LagPlan &p, const double *in, double *out, const void *tab,
                         double *rho_part, hipStream_t s) {
  const int G = (g.n[2] + p.chunks - 1) / p.chunks;
  const void *fn = (const void *)k_lag_plane<S, NT, TWICE, RHO, FLAT>;
  if (lag_xy_lds(g) > 64 * 1024)
    (void)hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lag_xy_lds(g));
  hipLaunchKernelGGL((k_lag_plane<S, NT, TWICE, RHO, FLAT>), dim3((unsigned)(g.n[3] * p.chunks)), dim3(64 * p.waves),
                     lag_xy_lds(g), s, in, out, g, (const LagTab *)tab, G, p.chunks, rho_part);
}

template <int S, bool FLAT>
static void launch_plane_sums(const Geom &g, const LagPlan &p, const double *in, double *out, const void *tab,
                              bool twice, double *rho_part, hipStream_t s) {
  if (twice) launch_plane<S, 512, true, true, FLAT>(g, p, in, out, tab, rho_part, s);
  else if (rho_part) launch_plane<S, 512, false, true, FLAT>(g, p, in, out, tab, rho_part, s);
  else launch_plane<S, 512, false, false, FLAT>(g, p, in, out, tab, nullptr, s);
}

void launch_lag_xy(const Geom &g, const LagPlan &p, const double *in, double *out, const void *tab, bool twice,
                   double *rho_part, hipStream_t s) {
  if (!twice && p.waves1) {
    LagPlan q = p;
    q.waves = p.waves1;
    launch_plane<16, 1024, false, false>(g, q, in, out, tab, nullptr, s);
  } else if (!p.sums) {
    if (twice) launch_plane<32, 1024, true, false>(g, p, in, out, tab, nullptr, s);
    else launch_plane<32, 1024, false, false>(g, p, in, out, tab, nullptr, s);
  } else if (p.points == 16) {
    if (p.flat) launch_plane_sums<16, true>(g, p, in, out, tab, twice, rho_part, s);
    else launch_plane_sums<16, false>(g, p, in, out, tab, twice, rho_part, s);
  } else {
    launch_plane_sums<32, false>(g, p, in, out, tab, twice, rho_part, s);
  }
}

void launch_lag_y(const Geom &g, const double *in, double *out, double dt, double *rho_part, hipStream_t s) {
  const long n = (long)g.n[0] * g.n[1] * g.n[3];
  hipLaunchKernelGGL(k_lag_y, dim3(blocks(n)), dim3(256), 0, s, in, out, g, dt, rho_part);
}

void launch_lag_vv(const Geom &g, const double *in, double *out, const double *ex, const double *ey, double dt,
                   hipStream_t s) {
  // (an axis has at most 251 points: nt <= 1024, 32-bit offsets in a row)
  const long P = (long)g.n[0] * g.n[1], nchunk = (P + VV_WP - 1) / VV_WP;
  const int nt = (VV_WP * ((g.n[2] + VV_S - 1) / VV_S) + 63) / 64 * 64;
  // 16 rows a segment: a segment loads five rows more than it has, but
  // workgroups on far-apart rows read HBM better than all on one row after the
  // other (128^4: one segment 1.02 ms, 8 rows 0.91, 16 rows 0.87, 32 rows
  // 0.96).  Fewer where the launch would have under two waves per SIMD (32^4:
  // 16 rows 19 us, 2 rows 13 us; 16 x 16 x 200 x 200, enough waves with 16
  // rows: 43 us, 8 rows 49 us).
  int len = 16;
  while (len > 2 && nchunk * ((g.n[3] + len - 1) / len) * (nt / 64) < 2048) len /= 2;
  const int nseg = (g.n[3] + len - 1) / len;
  hipLaunchKernelGGL((k_lag_vv<VV_WP, VV_S>), dim3((unsigned)(nchunk * nseg)), dim3(nt),
                     2 * sizeof(double) * VV_WP * g.n[2], s, in, out, g, ex, ey, dt, len, nseg);
}

}  // namespace vlp
