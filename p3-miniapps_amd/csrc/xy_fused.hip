// xy_fused.hip -- spline prefilter along x and y, 2-D half-step advection and
// density, fused per (vx, vy) plane (gfx950).
//
// Reference steps (one rank): exchangeHalo + Spline::computeCoeff_xy
// (VMO/Communication.cpp:541-570, VMO/Spline.hpp:384-426 -> :114-199), then
// advect_2D_xy (VMO/Advection.hpp:299-406, spline interp_2D :126-163) and
// field_rho (VMO/Field.cpp:37-53).  For one (vx, vy) plane all of these touch
// only that plane, so a workgroup keeps the plane's coefficients in LDS:
//   1. x recursions: f rows straight from global memory (each lane a chunk of
//      C values, the chunked scan of spline.hip), coefficients into LDS rows;
//   2. y recursions on the LDS columns, in place;
//   3. the CXY plane (positions -2..N+1 in x and y) leaves LDS as 16-byte
//      non-temporal stores;
//   4. the 2-D advection of every (x, y) of the plane reads the stencil from
//      LDS; f at the half step is never stored, it is summed over the
//      workgroup's vx planes into density partials.
// The workgroup owns one vy and a group of N2/G consecutive vx planes; the
// density partials rho_part[grp][vy][y][x] are summed over (grp, vy) by the
// field solve.
#include "spline_scan.hpp"

#include <algorithm>
#include <cstdlib>

namespace vlp {

namespace {

template <typename A> __device__ __forceinline__ void eta4(A w, A e[4]) { bspline_eta<A>(w, e); }

}  // namespace

// Block of NT lanes.  x pass: line y = r0 + tid / Px, lane p = tid % Px;
// y pass: column xc = c0 + tid / Py, lane p = tid % Py; advection: column
// x = tid % N0, rows y0 .. y0+ylen-1 (ylen <= NPT) of segment tid / N0, the
// density sums of those points in registers across the vx planes.
//
// Bound: HBM (16 bytes per cell in double; 0.94 ms at 128^4 at the 4.7 TB/s of a
// large copy, 1.45 ms taken) and, as a plane goes through its phases between
// barriers, the waves that hide one another's latency.  A lane with 32
// points' sums leaves room for two waves per SIMD; with 8 (512 lanes, planes up
// to about 64 x 64) or 16 points (1024 lanes) and no addresses held across the
// planes there is room for four, as two workgroups or one:
//   64^4 double 133 -> 90 us, 48^4 float 55 -> 36, 32^4 double 31 -> 17;
//   96^4 float storage 0.41 -> 0.34 ms, 128^4 float 0.92 -> 0.82, 90 x 77 x 84 x
//   75 float 0.36 -> 0.32.
// The RAG form with C = 16 and over 8 points does not fit in those registers
// (113 x 118 x 60 x 62 float 0.31 ms, with two waves per SIMD 0.28) and keeps 32.
constexpr int XY_NT = 512, XY_NPT = 32;

// RAG: lines of any length (the RAG form of the recursion, Px and Py lanes).
// Such planes used to run the single-lane x kernel, a strided y kernel and
// k_advect2d_rho, three passes over the plane with one lane per line: xy
// phases of 113 x 118 x 101 x 126 in float 2.32 -> 0.92 ms, 90 x 77 x 84 x 75
// in double 1.17 -> 0.41, 33 x 33 x 39 x 37 0.095 -> 0.061.
template <typename T, typename A, int C, bool RAG, int NT, int NPT>
__global__ __launch_bounds__(NT, NPT > 16 ? 2 : 4) void k_xy_adv2d(const T *__restrict__ f, T *__restrict__ cxy, Geom g, double dth,
                                                   int G, double *__restrict__ rho_part, int *__restrict__ err,
                                                   SplineConsts sc, double aC, double aN3x, double aN3y, int Px_,
                                                   int Py_) {
  extern __shared__ __align__(16) unsigned char xy_smem[];
  T *pl = (T *)xy_smem;
  const int N0 = g.n[0], N1 = g.n[1], N2 = g.n[2], N3 = g.n[3];
  const int E0 = N0 + 4, E1 = N1 + 4, R = E0 | 1;
  // y weights of the half-step foot per row (they depend on y and vy only):
  // ety[y][4], and the stencil base row jy0 in jty[y]
  A *ety = (A *)(xy_smem + (((size_t)E1 * R * sizeof(T) + 15) & ~(size_t)15));
  int *jty = (int *)(ety + 4 * N1);
  const int Px = RAG ? Px_ : N0 / C, Py = RAG ? Py_ : N1 / C;
  const int nlx = RAG ? (N0 + C - 1) / C : Px, nly = RAG ? (N1 + C - 1) / C : Py;
  const int skx = RAG ? nlx * C - N0 : 0, sky = RAG ? nly * C - N1 : 0;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int grp = blockIdx.x % G, ivy = blockIdx.x / G;
  const int VG = (N2 + G - 1) / G, v0 = min(N2, grp * VG), v1 = min(N2, v0 + VG);
  // advection lanes
  const int nseg = NT / N0, seg = tid / N0, xi = tid - seg * N0;
  const int ylen = (N1 + nseg - 1) / nseg, y0 = seg * ylen;
  const bool aact = seg < nseg;
  double rho[NPT];
#pragma unroll
  for (int k = 0; k < NPT; k++) rho[k] = 0.;
  int bad = 0;
  const double vy = g.minPhy[3] + ivy * g.dx[3];
  const double xx = g.minPhy[0] + xi * g.dx[0];
  for (int y = tid; y < N1; y += NT) {
    const double yy = g.minPhy[1] + y * g.dx[1];
    const double fy = ((yy - dth * vy) - g.minPhy[1]) * g.inv_dx[1];
    const int jy0 = (int)floor(fy);
    eta4<A>((A)(fy - (double)jy0), ety + 4 * y);
    jty[y] = jy0;
  }
  // (the first plane's barriers order these writes before their reads)
  // x pass lane: first plane's chunk in registers
  const int px = tid & (Px - 1), xl = tid / Px;
  for (int ivx = v0; ivx < v1; ivx++) {
    // 1. x recursions, rows 2..N1+1 of the plane
    for (int r0 = 0; r0 < N1; r0 += NT / Px) {
      const int y = r0 + xl;
      double v[C];
      const int x0 = RAG ? min(px * C, N0 - C) : px * C;  // first point of the lane's chunk
      const T *src = f + ((long)ivx + (long)N2 * ivy) * N0 * N1 + (long)(y < N1 ? y : 0) * N0 + x0;
#pragma unroll
      for (int i = 0; i < C; i++) v[i] = (double)src[i];
      double cm2, cm1, cN, cN1;
      scan_recursion<C, RAG>(v, px, Px, sc, aC, aN3x, cm2, cm1, cN, cN1, nlx, skx);
      if (y < N1 && (!RAG || px < nlx)) {
        T *row = pl + (y + 2) * R;
#pragma unroll
        for (int i = 0; i < C; i++)
          if (!RAG || i >= skx || px < nlx - 1) row[2 + x0 + i] = (T)v[i];
        if (px == 0) {
          row[0] = (T)cm2;
          row[1] = (T)cm1;
        }
        if (px == nlx - 1) {
          row[N0 + 2] = (T)cN;
          row[N0 + 3] = (T)cN1;
        }
      }
    }
    __syncthreads();
    // 2. y recursions on columns 0..E0-1 (a wave stops when its first
    // column is past the plane: its lines are whole within the wave)
    {
      int R_ = R;
      asm volatile("" : "+s"(R_));
      const int R = R_;
      const int py = tid & (Py - 1), yl = tid / Py, yl0 = (wave * 64) / Py;
      for (int c0 = 0; c0 + yl0 < E0; c0 += NT / Py) {
        const int xc = c0 + yl;
        const bool act = xc < E0 && (!RAG || py < nly);
        double w[C];
        const int r0 = RAG ? min(py * C, N1 - C) : py * C;  // first row of the lane's chunk
        const T *col = pl + (xc < E0 ? xc : 0) + (2 + r0) * R;
#pragma unroll
        for (int i = 0; i < C; i++) w[i] = (double)col[i * R];
        double cm2, cm1, cN, cN1;
        scan_recursion<C, RAG>(w, py, Py, sc, aC, aN3y, cm2, cm1, cN, cN1, nly, sky);
        if (act) {
          T *cw = pl + xc;
#pragma unroll
          for (int i = 0; i < C; i++)
            if (!RAG || i >= sky || py < nly - 1) cw[(2 + r0 + i) * R] = (T)w[i];
          if (py == 0) {
            cw[0] = (T)cm2;
            cw[R] = (T)cm1;
          }
          if (py == nly - 1) {
            cw[(N1 + 2) * R] = (T)cN;
            cw[(N1 + 3) * R] = (T)cN1;
          }
        }
      }
    }
    __syncthreads();
    // 3. store the CXY plane (positions -2..N+1 in x and y).  The plane is
    // contiguous in global memory, so it leaves as 16-byte chunks, lane after
    // lane (row and column of a chunk tracked incrementally), as
    // non-temporal stores (the plane is read again only by the vx spline
    // pass, after the whole kernel).  A chunk may straddle two rows when they
    // do not split into whole chunks; the last one ends in the plane's padding.
    {
      T *dst = cxy + ((long)ivx + (long)N2 * ivy) * xy_plane(N0, N1);
      constexpr int VPC = 16 / (int)sizeof(T);
      if (E0 % VPC == 0) {
        const int cpr = E0 / VPC, nch = cpr * E1;
        const int drow = NT / cpr, dcol = NT - drow * cpr;
        int row = tid / cpr, col = tid - row * cpr;
        for (int k = tid; k < nch; k += NT) {
          const T *s = pl + row * R + VPC * col;
          typedef T chunk_t __attribute__((ext_vector_type(VPC)));
          chunk_t v;
#pragma unroll
          for (int e = 0; e < VPC; e++) v[e] = s[e];
          __builtin_nontemporal_store(v, (chunk_t *)(dst + (long)VPC * k));
          row += drow;
          col += dcol;
          if (col >= cpr) {
            col -= cpr;
            row++;
          }
        }
      } else {
        const int nch = (E0 * E1 + VPC - 1) / VPC;
        const int drow = VPC * NT / E0, dcol = VPC * NT - drow * E0;
        int row = VPC * tid / E0, col = VPC * tid - row * E0;
        for (int k = tid; k < nch; k += NT) {
          const T *s = pl + row * R + col;
          typedef T chunk_t __attribute__((ext_vector_type(VPC)));
          chunk_t v;
#pragma unroll
          for (int e = 0; e < VPC; e++) v[e] = s[col + e < E0 ? e : e + R - E0];
          __builtin_nontemporal_store(v, (chunk_t *)(dst + (long)VPC * k));
          row += drow;
          col += dcol;
          if (col >= E0) {
            col -= E0;
            row++;
          }
        }
      }
    }
    // 4. 2-D advection at (x - dt/2 vx, y - dt/2 vy), interp_2D's spline branch
    if (aact) {
      const double vx = g.minPhy[2] + ivx * g.dx[2];
      const double fx = ((xx - dth * vx) - g.minPhy[0]) * g.inv_dx[0];
      const int jx0 = (int)floor(fx);
      A etax[4];
      eta4<A>((A)(fx - (double)jx0), etax);
      const bool xbad = (jx0 < -1 || jx0 > N0 - 1);
      const T *pc = pl + (xbad ? 0 : jx0 + 1);  // stencil column jx0-1 at LDS column jx0+1
      A gw[4];  // x-interpolated rows jw .. jw+3 (LDS rows)
      int jw = -1000;
      // (an opaque copy: the points' table addresses and conditions are not to be
      // held in registers across the planes)
      int y0v = y0;
      asm volatile("" : "+v"(y0v));
      constexpr int GP = sizeof(A) == sizeof(float) ? 4 : 2;
      static_assert(NPT % GP == 0, "groups tile the point range");
      // Points go in groups of GP consecutive y (four for float arithmetic,
      // two for double, whose tables take twice the registers).  The
      // segment's lanes share y, so jy0 and the group's path are uniform in a
      // wave when N0 is a multiple of 64.  When the GP stencils each move down
      // by one row from the previous point's (the usual case), the group's
      // tables and its GP new rows are all read before the arithmetic (one
      // LDS round trip per group instead of several per point); otherwise the
      // points go one at a time.
#pragma unroll
      for (int k0 = 0; k0 < NPT; k0 += GP) {
        const int yg = y0v + k0;
        if (k0 < ylen && yg < N1) {
          int jr[GP];
          A ey[GP][4];
#pragma unroll
          for (int j = 0; j < GP; j++) {
            const int y = min(yg + j, N1 - 1);
            jr[j] = jty[y] + 1;  // stencil row jy0-1 at LDS row jy0+1
#pragma unroll
            for (int jy = 0; jy < 4; jy++) ey[j][jy] = ety[4 * y + jy];
          }
          const bool full = k0 + GP - 1 < ylen && yg + GP - 1 < N1;
          bool slide = full && !xbad && jr[0] == jw + 1;
#pragma unroll
          for (int j = 0; j < GP; j++) slide = slide && jr[j] >= 0 && jr[j] <= N1 && jr[j] == jr[0] + j;
          if (slide) {
            T nr[GP][4];  // rows jw+4 .. jw+3+GP
#pragma unroll
            for (int j = 0; j < GP; j++) {
              const T *p = pc + (jw + 4 + j) * R;
#pragma unroll
              for (int jx = 0; jx < 4; jx++) nr[j][jx] = p[jx];
            }
#pragma unroll
            for (int j = 0; j < GP; j++) {
              gw[0] = gw[1];
              gw[1] = gw[2];
              gw[2] = gw[3];
              A s = 0;
#pragma unroll
              for (int jx = 0; jx < 4; jx++) s += etax[jx] * (A)nr[j][jx];
              gw[3] = s;
              A val = 0;
#pragma unroll
              for (int jy = 0; jy < 4; jy++) val += ey[j][jy] * gw[jy];
              rho[k0 + j] += (double)val;
            }
            jw = jr[GP - 1];
          } else {
#pragma unroll
            for (int j = 0; j < GP; j++) {
              const int k = k0 + j, y = yg + j;
              if (k < ylen && y < N1) {
                const int jy0 = jr[j] - 1;
                A val = 0;
                if (xbad || jy0 < -1 || jy0 > N1 - 1) {
                  bad = 1;  // interp_2D returns 1 and leaves 0 (VMO/Advection.hpp:148-151)
                } else {
                  const int r = jr[j];
                  if (r == jw + 1) {
                    gw[0] = gw[1];
                    gw[1] = gw[2];
                    gw[2] = gw[3];
                    const T *p = pc + (r + 3) * R;
                    A s = 0;
#pragma unroll
                    for (int jx = 0; jx < 4; jx++) s += etax[jx] * (A)p[jx];
                    gw[3] = s;
                  } else if (r != jw) {
#pragma unroll
                    for (int jy = 0; jy < 4; jy++) {
                      const T *p = pc + (r + jy) * R;
                      A s = 0;
#pragma unroll
                      for (int jx = 0; jx < 4; jx++) s += etax[jx] * (A)p[jx];
                      gw[jy] = s;
                    }
                  }
                  jw = r;
#pragma unroll
                  for (int jy = 0; jy < 4; jy++) val += ey[j][jy] * gw[jy];
                }
                rho[k] += (double)val;
              }
            }
          }
        }
        __builtin_amdgcn_sched_barrier(0);  // one group at a time (register pressure)
      }
    }
    __syncthreads();
  }
  if (aact) {
    double *rp = rho_part + ((long)grp * N3 + ivy) * N0 * N1;
#pragma unroll
    for (int k = 0; k < NPT; k++) {
      const int y = y0 + k;
      if (k < ylen && y < N1) rp[(long)y * N0 + xi] = rho[k];
    }
  }
  if (bad) atomicOr(err, 1);
}

namespace {

// LDS bytes: the plane, then the y-weight and y-row tables.
size_t xy_lds(const Geom &g, size_t tsz) {
  const size_t plane = (((size_t)(g.n[1] + 4) * ((g.n[0] + 4) | 1) * tsz) + 15) & ~(size_t)15;
  return plane + (size_t)g.n[1] * (4 * sizeof(double) + sizeof(int));
}

// Chunk and lanes of the fused kernel for a geometry (C = 0: not eligible): the
// plane fits in LDS, every lane of XY_NT owns at most XY_NPT advection points
// (then one of 2 XY_NT at most half as many), and N0 =
// Px C and N1 = Py C with Px, Py powers of two, or (rag) Px C and Py C cover
// N0 and N1 with the fewest lanes.
struct XyPlan {
  int C = 0, Px = 0, Py = 0;
  bool rag = false;
};
XyPlan xy_plan(const Geom &g, size_t tsz) {
  XyPlan p;
  const int N0 = g.n[0], N1 = g.n[1];
  if (N0 > XY_NT || xy_lds(g, tsz) > 160 * 1024) return p;
  const int nseg = XY_NT / N0, ylen = (N1 + nseg - 1) / nseg;
  if (ylen > XY_NPT) return p;
  for (int C : {16, 12}) {
    if (N0 % C || N1 % C) continue;
    const int Px = N0 / C, Py = N1 / C;
    if ((Px & (Px - 1)) || (Py & (Py - 1)) || Px > 16 || Py > 16) continue;
    p.C = C;
    p.Px = Px;
    p.Py = Py;
    return p;
  }
  for (int C : {10, 12, 16}) {
    if (C > N0 || C > N1) continue;
    int Px = 1, Py = 1;
    while (Px * C < N0) Px *= 2;
    while (Py * C < N1) Py *= 2;
    if (Px > 16 || Py > 16 || (p.C && Px + Py >= p.Px + p.Py)) continue;
    p.C = C;
    p.Px = Px;
    p.Py = Py;
    p.rag = true;
  }
  return p;
}

// Advection points per lane of nt.
int xy_points(const Geom &g, int nt) {
  const int nseg = nt / g.n[0];
  return nseg ? (g.n[1] + nseg - 1) / nseg : XY_NPT + 1;
}

// Lanes of a workgroup.  XY_NT with up to 8 points each, else twice as many (or
// XY_NT with up to 32 points: launch_xy_t); rag planes whose lines take fewer
// lanes go in workgroups of those, so that more of them share a CU: most lanes
// of 512 idled through the recursions, and the phases of 25 x 23 x 100 x 100 in
// float took 157 us, 94 in the separate kernels, now 57 (30 x 30 x 130 x 130 328,
// 155 and 111; 40 x 40 x 77 x 77 110, 86 and 63).
int xy_lanes(const Geom &g, const XyPlan &p) {
  if (p.rag)
    for (int nt : {128, 256})
      if (xy_points(g, nt) <= 8 && std::max(g.n[1] * p.Px, (g.n[0] + 4) * p.Py) <= nt) return nt;
  return xy_points(g, XY_NT) <= 8 ? XY_NT : 2 * XY_NT;
}

}  // namespace

// Groups of vx planes per vy: the least time of a CU that runs its k workgroups
// of VG planes (and a plane's time for the start) up to per_cu at once, each
// plane costing latency once per round and throughput once per workgroup, in
// equal shares where 512 lanes or more go through a plane and two to one where
// fewer do.  (Powers of two until the chip was full twice left 130 x 4 = 520
// workgroups for 512 places, a whole round for the last eight: with 512 lanes, 25
// x 23 x 130 x 130 in double 344 us, now 238, 90 x 77 x 66 x 66 312 and 222; 96^4
// 534 and 429.  64 x 64 x 96 x 96 took 236, now 245.  By rounds alone 64 x 64 x
// 128 x 128 in float was 9 % slower.)
int xy_fused_groups(const Geom &g, size_t tsz) {
  if (const char *e = getenv("VLP4D_XY_FUSED"))
    if (atoi(e) == 0) return 0;
  const XyPlan p = xy_plan(g, tsz);
  if (!p.C) return 0;
  const int N2 = g.n[2], nt = xy_lanes(g, p);
  const long per_cu = std::max(1L, std::min((long)(2 * XY_NT / nt), (long)(160 * 1024 / xy_lds(g, tsz))));
  int best = 1;
  long cost = -1;
  for (int n = 1; n <= N2; n++) {
    const int VG = (N2 + n - 1) / n;
    if ((N2 + VG - 1) / VG != n) continue;  // the same groups in fewer workgroups
    const long k = ((long)n * g.n[3] + 255) / 256;
    const long c = (VG + 1) * (2 * ((k + per_cu - 1) / per_cu) + (nt >= XY_NT ? 2 : 1) * k);
    if (cost < 0 || c < cost) {
      cost = c;
      best = n;
    }
  }
  return best;
}

template <typename T, typename A, int C, bool RAG, int NT, int NPT>
static void launch_xy_n(const Geom &g, const T *f, T *cxy, double dth, int G, double *rho_part, int *err,
                        const XyPlan &p, hipStream_t s) {
  const SplineConsts sc = spline_consts();
  double aC = 1.0, aN3x = 1.0, aN3y = 1.0;
  for (int i = 0; i < C; i++) aC *= sc.alpha;
  for (int i = 0; i < g.n[0] + 3; i++) aN3x *= sc.alpha;
  for (int i = 0; i < g.n[1] + 3; i++) aN3y *= sc.alpha;
  const size_t lds = xy_lds(g, sizeof(T));
  const void *fn = (const void *)k_xy_adv2d<T, A, C, RAG, NT, NPT>;
  if (lds > 64 * 1024) (void)hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  hipLaunchKernelGGL((k_xy_adv2d<T, A, C, RAG, NT, NPT>), dim3((unsigned)(G * g.n[3])), dim3(NT), lds, s, f, cxy, g,
                     dth, G, rho_part, err, sc, aC, aN3x, aN3y, p.Px, p.Py);
}

template <typename T, typename A, int C, bool RAG>
static void launch_xy_t(const Geom &g, const T *f, T *cxy, double dth, int G, double *rho_part, int *err,
                        const XyPlan &p, hipStream_t s) {
  if constexpr (RAG) {
    const int nt = xy_lanes(g, p);
    if (nt == 128) return launch_xy_n<T, A, C, RAG, 128, 8>(g, f, cxy, dth, G, rho_part, err, p, s);
    if (nt == 256) return launch_xy_n<T, A, C, RAG, 256, 8>(g, f, cxy, dth, G, rho_part, err, p, s);
  }
  if (xy_points(g, XY_NT) <= 8) launch_xy_n<T, A, C, RAG, XY_NT, 8>(g, f, cxy, dth, G, rho_part, err, p, s);
  else if constexpr (RAG && C == 16) launch_xy_n<T, A, C, RAG, XY_NT, XY_NPT>(g, f, cxy, dth, G, rho_part, err, p, s);
  else launch_xy_n<T, A, C, RAG, 2 * XY_NT, XY_NPT / 2>(g, f, cxy, dth, G, rho_part, err, p, s);
}

template <typename T, typename A>
bool launch_xy_adv2d(const Geom &g, const T *f, T *cxy, double dt_half, double *rho_part, int *err, hipStream_t s) {
  const int G = xy_fused_groups(g, sizeof(T));
  if (!G) return false;
  const XyPlan p = xy_plan(g, sizeof(T));
  if (p.rag) switch (p.C) {
    case 16: launch_xy_t<T, A, 16, true>(g, f, cxy, dt_half, G, rho_part, err, p, s); return true;
    case 12: launch_xy_t<T, A, 12, true>(g, f, cxy, dt_half, G, rho_part, err, p, s); return true;
    case 10: launch_xy_t<T, A, 10, true>(g, f, cxy, dt_half, G, rho_part, err, p, s); return true;
    default: return false;
  }
  switch (p.C) {
    case 16: launch_xy_t<T, A, 16, false>(g, f, cxy, dt_half, G, rho_part, err, p, s); return true;
    case 12: launch_xy_t<T, A, 12, false>(g, f, cxy, dt_half, G, rho_part, err, p, s); return true;
    default: return false;
  }
}

template bool launch_xy_adv2d<double, double>(const Geom &, const double *, double *, double, double *, int *,
                                              hipStream_t);
template bool launch_xy_adv2d<float, double>(const Geom &, const float *, float *, double, double *, int *,
                                             hipStream_t);
template bool launch_xy_adv2d<float, float>(const Geom &, const float *, float *, double, double *, int *,
                                            hipStream_t);

}  // namespace vlp
