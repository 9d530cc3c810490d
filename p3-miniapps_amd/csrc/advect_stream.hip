// advect_stream.hip -- y-streaming 4-D advection (gfx950).
//
// Same arithmetic as advect_4D of the reference (computeFeet
// VMO/Advection.hpp:166-218, interp_4D :221-296, the loop of :409-498); the
// work is organised so that every C4 coefficient a workgroup needs crosses
// from L2 into the CU once, through LDS.
//
// Workgroup = (all x) x (TVX consecutive vx) at one vy.  It walks y (all of it, or
// a segment when there are few workgroups): at step q
// it holds one y-plane of C4 in LDS -- positions x -2..N0+1, vx tile-2 ..
// tile+TVX+1, vy ivy-2..ivy+2 (a slab) -- with the next two in flight.
// Lane (x, vx) keeps the four cells (x, y, vx, vy) whose y-stencil contains
// the current plane "open": their B-spline weights along x, y, vx, vy and an
// accumulator.  For vy > 0 every regular foot has floor(y*) = y-1 (for vy <= 0,
// y), so cell y reads planes y+oy-1 .. y+oy+2 with oy fixed per workgroup, is
// opened when its first plane arrives and written after its fourth.  Each 4-wide
// x row read from LDS then feeds all four open cells: 16 rows x 4 values per
// step and per lane, 340 FMAs per cell, no re-reads from L2.
//
// A lane reads one set of rows for its four cells when they agree on their x,
// vx and vy stencil offsets (each in {-1, 0} relative to the cell), else one
// set per distinct offset pattern.  A foot outside this pattern (displacement
// beyond one cell, or y offset different from the workgroup's) is interpolated
// by the direct 4^4 gather from C4 in global memory at the step it is opened
// and takes no streamed contribution.
//
// The vy = 0 slab has feet of both y offsets (they follow the sign of Ey), so
// it is streamed by two workgroups per vx tile, one for each offset; each
// writes its own feet.  With one workgroup, half of the slab took the gather,
// whose 64 dependent row loads per step made these few workgroups the tail of
// the launch: 140 us of a 16^4 advection, 1.01 ms at 64^4 (FP64).
#include "advect_common.hpp"

#include <algorithm>
#include <cstdlib>

namespace vlp {

namespace {

// One open cell: B-spline weights along x, y, vx, vy ([dim][k]), running
// sum, and the LDS element of its first stencil row in a plane's slab.  A
// cell without a streamed contribution has zero x-weights and the row of the
// cell opened before it.  (Keeping the four y weights rather than
// re-evaluating the one a plane needs from the fractional y position measured
// 1 % faster with double arithmetic.)
template <typename A> struct OpenCell {
  A w[4][4];
  A acc;
  int row;
};

typedef __attribute__((address_space(3))) void lds_void;


// Per-workgroup constants and per-lane state of the streaming loop.  The slab
// is kept in the storage type T (moved by LDS-DMA, 16 bytes per lane) and
// converted to the arithmetic type A as it is read.  Its rows are contiguous
// in LDS, so the slab is moved as one run of 16-byte chunks: DMA instruction j
// fills LDS bytes [1024 j, 1024 j + 1024) of the buffer, lane l taking chunk
// 64 j + l wherever it sits in C4; instructions are dealt to the waves in
// turn, and each lane keeps the C4 byte offset (from the plane's first row)
// of its chunk in every instruction of its wave.  When the C4 rows are not
// whole 16-byte chunks (N0 + 4 odd, or for float not a multiple of 4), a
// plane's rows start shift(q) elements past a chunk boundary, the same for all
// rows of the plane (the pitches past y are multiples of 16 elements): the
// chunks are taken from the boundary and the slab pitch RX holds the
// remainder.  E rows sit in LDS as
// (Ex, Ey) pairs: [buffer][row k1 = 0..2][EPR], moved 64 points per instruction.
//
// computeFeet's 3x3 Lagrange interpolation of E at the half-step position
// (x - dt/2 vx, y - dt/2 vy) separates: the x part (base column ip0 and
// weights cx) depends on the lane's (x, vx) only, the y part (row ip1 and
// weights cy) on (y, vy), which is uniform in the workgroup at a step.  As ip1
// advances by one per step, a lane reads one new row per step,
// g = sum_k0 cx[k0] E(ip0+k0, ip1+2), and adds it to the sums of the three
// cells it belongs to: it completes cell q's, is the second term of cell
// q+1's and the first of cell q+2's.
template <typename T, typename A, int TVX, int NB, int RXC> struct YStream {
  static constexpr int VPL = 16 / (int)sizeof(T);  // slab values per lane load
  static constexpr int MS = 8;  // slab DMA instructions per wave per plane, at most
  const T *__restrict__ c4;
  const double *__restrict__ exy;  // (Ex, Ey) pairs, [N1][N0]
  T *__restrict__ fout;
  T *slab;         // NB buffers of slab_bytes
  double *eb;      // [NB][3][EPR][2]
  double *kconst;  // LDS: domain constants of the foot computation (KC_* layout)
  // LDS: per y-step values uniform in the workgroup, rows q = -2 .. N1-1 of
  // QT: computeFeet's E row ip1 of cell q (as a double), and the y Lagrange
  // weights of the row that is new at step q: cy[2] of cell q, cy[1] of cell
  // q+1, cy[0] of cell q+2
  double *qtab;
  static constexpr int QT = 4;
  T *fbase;  // f^{n+1} at (x, y = 0, vx, vy) of this lane
  static constexpr int KC_MIN = 0, KC_INV = 4, KC_LMIN = 8, KC_LMAX = 12, KC_VHI = 16, KC_DX = 18, KC_DT = 22, KC_N = 24;
  int slab_bytes;  // whole 1 KB blocks
  int EPR, cpr;    // E points per LDS row (whole 64-point chunks), chunks per row
  unsigned voff[MS];  // C4 byte offset of this lane's chunk in the wave's k-th slab DMA
  int nslot;       // slab DMA instructions of this wave (wave-uniform)
  int N0, N1, N2, N3, RX, oyw;
  int y0, y1;  // the cells y0 <= y < y1 of this workgroup: steps y0 .. y1 + 2
  int ix, tv, ivx, ivy;
  int row0;  // LDS element of the stencil row of a foot with offset 0 along x, vx, vy
  bool active;
  bool wave_has_cells;  // some lane of this wave owns cells (wave-uniform)
  long S1, S2, S3;
  int F0;
  int wave, nwave, lane;
  // this slab is shared by two workgroups, one per y offset: 0 no, 1 this one
  // has offset 0 and also the feet outside both patterns, 2 offset -1
  int pair;
  int keep;  // pair: bit c set when this workgroup writes the cell in slot c
  int force;  // bit 0: every lane reads rows per cell; bit 1: every foot by direct gather
  int cbase;  // C4 element of (x -2, y -3, vx tile-2, vy ivy-2)
  double cx[3];          // x Lagrange weights of the half-step foot
  int jx[3];             // wrapped E columns ip0 .. ip0+2
  double s1x, s1y, s2x, s2y;  // partial E of cells q+1 (two rows) and q+2 (one row)
  // The foot in cells from the node: d = -dt (v - dt/2 E) / dx along x and y,
  // -dt E / dv along vx and vy.  ax, ay1: its part without E (along y less
  // the workgroup's offset, so that a streamed foot has 0 <= w < 1, except in
  // a shared slab)
  double ax, ay1;
  double bex, bey, bvx, bvy;  // factors of E in the four directions
  double lo2, lo3;            // lower bounds of the vx and vy displacement (the clamp at v_min)
  int ip1p;              // ip1 of the previous step (wave-uniform)
  OpenCell<A> cell[4];
  int bad;

  // E row ip1 of the cell y (computeFeet: round of the half-step y) - 1;
  // uniform in the workgroup.
  __device__ __forceinline__ int erow0(int y) const {
    return __builtin_amdgcn_readfirstlane((int)qtab[QT * y]);
  }

  // Elements by which plane q's rows sit past a 16-byte boundary (C4's base
  // puts the rows of y = -2 on one).
  __device__ __forceinline__ int shift(int q) const { return RXC ? 0 : (F0 * (q + oyw + 1)) & (VPL - 1); }

  // Start moving step q's slab and E rows into LDS buffer b by LDS-DMA.
  // Returns the number of DMA instructions this wave issued (wave-uniform).
  __device__ __forceinline__ int fetch(int q, int b) {
    const int p = q + oyw - 1;  // y-position of the plane
    const char *src = (const char *)c4 + ((long)cbase + (long)F0 * (p + 3) - shift(q)) * (long)sizeof(T);
    // the slot bookkeeping is recomputed each step from these (a few scalar
    // operations) rather than kept live across the loop, where it would be
    // spilled from the scalar registers
    int ns = nslot, lb = b * slab_bytes + 1024 * wave, ls = 1024 * nwave;
    asm volatile("" : "+s"(ns), "+s"(lb), "+s"(ls));
    char *sb = (char *)slab + lb;
    int n = 0;
#pragma unroll
    for (int k = 0; k < MS; k++)
      if (k < ns) {
        // a fresh 32-bit offset per load keeps the address in the form
        // (scalar base + 32-bit lane offset) the load encodes directly,
        // instead of a 64-bit vector add per load
        unsigned o = voff[k];
        asm volatile("" : "+v"(o));
        __builtin_amdgcn_global_load_lds((const void *)(src + o), (lds_void *)(sb + k * ls), 16, 0, 0);
        n++;
      }
    if (q < y1) {
      const int ip1 = erow0(q);
      char *el = (char *)(eb + b * 6 * EPR);
      for (int e = wave; e < 3 * cpr; e += nwave, n++) {
        const int k1 = (e >= cpr) + (e >= 2 * cpr), c = e - k1 * cpr;
        int row = ip1 + k1;
        // periodic wrap (row is wave-uniform; a scalar loop, no division
        // constants kept live across the y loop)
        while (row < 0) row += N1;
        while (row >= N1) row -= N1;
        // points beyond N0 (last chunk) repeat the row's last point into the padding
        const int pt = min(64 * c + lane, N0 - 1);
        __builtin_amdgcn_global_load_lds((const void *)(exy + 2 * ((long)row * N0 + pt)),
                                         (lds_void *)(el + 16 * (k1 * EPR + 64 * c)), 16, 0, 0);
      }
    }
    return n;
  }

  // E at the half-step foot of cell q (computeFeet, VMO/Advection.hpp:
  // 174-206) from the E rows in buffer b.
  __device__ __forceinline__ void field_at(int q, int b, double &efx, double &efy) {
    const double *t = qtab + QT * q;
    const int ip1 = __builtin_amdgcn_readfirstlane((int)t[0]);
    const double2 *er = (const double2 *)(eb + b * 6 * EPR);
    if (ip1 != ip1p + 1) {  // the first cell (or a rounding tie of the row): its rows 0 and 1
      const double c0 = t[3 - 2 * QT], c1 = t[2 - QT], d0 = t[3 - QT];
      double gx[2], gy[2];
#pragma unroll
      for (int k1 = 0; k1 < 2; k1++) {
        const double2 e0 = er[k1 * EPR + jx[0]], e1 = er[k1 * EPR + jx[1]], e2 = er[k1 * EPR + jx[2]];
        gx[k1] = cx[0] * e0.x + cx[1] * e1.x + cx[2] * e2.x;
        gy[k1] = cx[0] * e0.y + cx[1] * e1.y + cx[2] * e2.y;
      }
      s1x = c0 * gx[0] + c1 * gx[1];
      s1y = c0 * gy[0] + c1 * gy[1];
      s2x = d0 * gx[1];
      s2y = d0 * gy[1];
    }
    ip1p = ip1;
    const double2 e0 = er[2 * EPR + jx[0]], e1 = er[2 * EPR + jx[1]], e2 = er[2 * EPR + jx[2]];
    const double gx = cx[0] * e0.x + cx[1] * e1.x + cx[2] * e2.x;
    const double gy = cx[0] * e0.y + cx[1] * e1.y + cx[2] * e2.y;
    efx = s1x + t[1] * gx;
    efy = s1y + t[1] * gy;
    s1x = s2x + t[2] * gx;
    s1y = s2y + t[2] * gy;
    s2x = t[3] * gx;
    s2y = t[3] * gy;
  }

  // Open cell y = q in slot R with the field at its half-step foot: the
  // displacement, B-spline weights and stencil row.  The displacement is
  // formed in cells from the node, which needs no position, division or
  // floor: the fraction is that of the displacement and the stencil offset its
  // sign, for |displacement| < 1 (other feet take open_direct, the reference's
  // sequence).
  template <int R> __device__ __forceinline__ void open(int q, double efx, double efy) {
    OpenCell<A> &c = cell[R];
    c.acc = 0;
    c.row = cell[(R + 3) & 3].row;
    if (pair) keep &= ~(1 << R);
    if (q >= y1) {
      // no cell: zero x-weights make its share of a common pass zero
#pragma unroll
      for (int k = 0; k < 4; k++) c.w[0][k] = 0;
      return;
    }
    const double d0 = ax + bex * efx;
    double w1 = ay1 + bey * efy;
    // the velocity clamp at v_min binds for the first plane only (a foot
    // beyond v_max is one cell or more away and not taken here)
    const double d2 = fmax(bvx * efx, lo2), d3 = fmax(bvy * efy, lo3);
    // all comparisons fail for a NaN (of Ex in d0, of Ey in w1)
    const bool near = (fabs(d0) < 1.) & (fabs(d2) < 1.) & (fabs(d3) < 1.) & !(force & 2);
    bool in = (w1 >= 0.) & (w1 < 1.);
    bool other = false;  // in a shared slab: the other workgroup's foot
    if (pair) {          // there w1 is the displacement itself, so that the two workgroups split the feet exactly
      const bool neg = (w1 >= -1.) & (w1 < 0.);
      if (pair == 2) {
        in = neg;
        w1 += 1.;
        other = true;
      } else {
        other = near & neg;
      }
    }
    const bool fast = near & in;
    bspline_eta<A>((A)__builtin_amdgcn_fract(d0), c.w[0]);
    bspline_eta<A>((A)w1, c.w[1]);
    bspline_eta<A>((A)__builtin_amdgcn_fract(d2), c.w[2]);
    bspline_eta<A>((A)__builtin_amdgcn_fract(d3), c.w[3]);
    const int rx = RXC ? RXC : RX;
    const int row = row0 + (d0 < 0. ? -1 : 0) + (d2 < 0. ? -rx : 0) + (d3 < 0. ? -(TVX + 4) * rx : 0);
    if (pair) keep |= fast ? 1 << R : 0;
    if (__builtin_amdgcn_ballot_w64(!fast) == 0) {
      c.row = row;
    } else {
      if (fast) {
        c.row = row;
      } else {
        if (!other) open_direct(q, efx, efy, c);
        if (pair) keep |= other ? 0 : 1 << R;
#pragma unroll
        for (int k = 0; k < 4; k++) c.w[0][k] = 0;  // no share of a common pass
      }
    }
    if (q == y0) {  // the slots still empty agree with the first cell
#pragma unroll
      for (int k = 1; k < 4; k++) cell[(R + k) & 3].row = c.row;
    }
  }

  // A foot outside the streamed pattern: computeFeet's own sequence
  // (VMO/Advection.hpp:208-217), the bound check and the direct 4^4 gather.
  // Its constants come from LDS and the C4 strides are rebuilt here, so that
  // this rare path keeps nothing in scalar registers across the loop.
  __device__ __forceinline__ void open_direct(int q, double ftmp1, double ftmp2, OpenCell<A> &c) {
    const double *kc = kconst;
    asm volatile("" : "+s"(kc));
    const double x = kc[KC_MIN] + ix * kc[KC_DX], yq = kc[KC_MIN + 1] + q * kc[KC_DX + 1];
    const double vx = kc[KC_MIN + 2] + ivx * kc[KC_DX + 2], vy = kc[KC_MIN + 3] + ivy * kc[KC_DX + 3];
    const double dtl = kc[KC_DT];
    const double xt2 = vx - 0.5 * dtl * ftmp1;
    const double xt3 = vy - 0.5 * dtl * ftmp2;
    double xs[4];
    xs[0] = x - dtl * xt2;
    xs[1] = yq - dtl * xt3;
    // the velocity clamp max(min(v*, vmax), vmin) as v_min / v_max: they
    // differ from the comparisons only for a NaN v*, which makes x* NaN
    // too, so the bound check below still fails
    xs[2] = fmax(fmin(vx - dtl * ftmp1, kc[KC_VHI]), kc[KC_MIN + 2]);
    xs[3] = fmax(fmin(vy - dtl * ftmp2, kc[KC_VHI + 1]), kc[KC_MIN + 3]);
    // all eight comparisons, no short cut (NaN fails them)
    bool ok = true;
#pragma unroll
    for (int j = 0; j < 4; j++) ok = ok & (xs[j] >= kc[KC_LMIN + j]) & (xs[j] <= kc[KC_LMAX + j]);
    // out of domain: the reference stops with "Time step is too large"
    bad |= !ok;
    if (!ok) return;
    int ip[4];
    // (the weights go to the cell's registers: other lanes of the wave keep
    // theirs there, so this path adds none)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const double fj = kc[KC_INV + j] * (xs[j] - kc[KC_MIN + j]);
      const double fl = floor(fj);
      ip[j] = (int)fl;
      bspline_eta<A>((A)(fj - fl), c.w[j]);
    }
    int n0 = N0, n1 = N1, n2 = N2;
    asm volatile("" : "+s"(n0), "+s"(n1), "+s"(n2));
    const C4Pitch cp = c4_pitch(n0, n1, n2);
    c.acc = gather4d<T, A>(c4, cp.s1, cp.s2, cp.s3, ip, c.w);
  }

  // The plane's contribution t[c] to each of the four open cells from the 16
  // rows at LDS element sp (one stencil key): rows (kvx, kvy) in order, the
  // next row's LDS reads issued before the current row's FMAs (one row of
  // look-ahead hides the LDS latency).  With the slab row pitch known at
  // compile time (RXC = N0 + 4), rows kvx = 0, 1 and 2, 3 of a vy row are
  // read from one base address each, the second row through the immediate
  // offsets of the paired LDS reads (an empty asm keeps the compiler from
  // rebuilding a base per row): 8 address additions per pass instead of 16.
  __device__ __forceinline__ void pass_rows(const T *sp, A t[4]) const {
    const int VS = (TVX + 4) * (RXC ? RXC : RX);  // vy row stride
    typedef const __attribute__((address_space(3))) T lds_t;
    lds_t *pb = (lds_t *)sp;
    if constexpr (RXC != 0) asm volatile("" : "+v"(pb));
    A u[4];
#pragma unroll
    for (int c = 0; c < 4; c++) t[c] = u[c] = 0;
    T r[2][4];
#pragma unroll
    for (int k = 0; k < 4; k++) r[0][k] = RXC ? pb[k] : sp[k];
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int kvx = i & 3, kvy = i >> 2;
      // row i complete (only LDS reads are waited on; the slab DMA stays in
      // flight), then row i+1's reads go out ahead of row i's FMAs
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
      if (i + 1 < 16) {
        const int n = i + 1;
        if constexpr (RXC != 0) {
          if ((n & 1) == 0) {  // first row of a pair: a new base
            pb = (lds_t *)(sp + (n >> 2) * VS + (n & 2) * RXC);
            asm volatile("" : "+v"(pb));
          }
          const int o = (n & 1) * RXC;
#pragma unroll
          for (int k = 0; k < 4; k++) r[n & 1][k] = pb[o + k];
        } else {
          const T *rn = sp + (n >> 2) * VS + (n & 3) * RX;
#pragma unroll
          for (int k = 0; k < 4; k++) r[n & 1][k] = rn[k];
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      const A r0 = (A)r[i & 1][0], r1 = (A)r[i & 1][1], r2 = (A)r[i & 1][2], r3 = (A)r[i & 1][3];
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const A *w0 = cell[c].w[0];
        const A d = w0[0] * r0 + w0[1] * r1 + w0[2] * r2 + w0[3] * r3;
        u[c] += cell[c].w[2][kvx] * d;
      }
      if (kvx == 3) {
#pragma unroll
        for (int c = 0; c < 4; c++) {
          t[c] += cell[c].w[3][kvy] * u[c];
          u[c] = 0;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // Add plane q (LDS buffer b) to the four open cells; the cell opened at
  // step q - j sits in slot (R - j) & 3 and takes y-weight j.  When every
  // lane's cells agree on their first stencil row (the usual case), one pass
  // over the 16 rows serves all four cells; cells without a streamed
  // contribution have zero x-weights, so their share is zero.  Otherwise one
  // pass reads the rows of one cell per lane (the first still to do) and adds
  // to the cells with the same rows; the wave repeats until no lane has cells
  // left.  force & 1 takes the second
  // form with one cell per pass.
  template <int R> __device__ __forceinline__ void accumulate(int q, int b) {
    const T *s = (const T *)((const char *)slab + b * slab_bytes) + shift(q);
    const int r0 = cell[0].row;
    const bool same = (r0 == cell[1].row) & (r0 == cell[2].row) & (r0 == cell[3].row) & !(force & 1);
    A t[4];
    if (__builtin_amdgcn_ballot_w64(!same) == 0) {
      pass_rows(s + r0, t);
      close_plane<R, 0>(t, 15u);
      close_plane<R, 1>(t, 15u);
      close_plane<R, 2>(t, 15u);
      close_plane<R, 3>(t, 15u);
      return;
    }
    unsigned todo = 15u;
    while (__builtin_amdgcn_ballot_w64(todo != 0)) {
      int rp = r0;
#pragma unroll
      for (int c = 3; c >= 0; c--)
        if ((todo >> c) & 1) rp = cell[c].row;
      unsigned sel = 0;
#pragma unroll
      for (int c = 0; c < 4; c++)
        if (((todo >> c) & 1) && cell[c].row == rp && !((force & 1) && sel)) sel |= 1u << c;
      todo &= ~sel;
      pass_rows(s + rp, t);
      close_plane<R, 0>(t, sel);
      close_plane<R, 1>(t, sel);
      close_plane<R, 2>(t, sel);
      close_plane<R, 3>(t, sel);
    }
  }

  // The cell opened J steps ago takes the plane's contribution with its y
  // weight J, when sel has its bit.
  template <int R, int J> __device__ __forceinline__ void close_plane(const A t[4], unsigned sel) {
    constexpr int c = (R - J) & 3;
    OpenCell<A> &oc = cell[c];
    const A add = oc.w[1][J] * t[c];
    if (sel == 15u) oc.acc += add;
    else oc.acc += ((sel >> c) & 1) ? add : (A)0;
  }

  // Write cell y = q - 3 (slot (R + 1) & 3).
  template <int R> __device__ __forceinline__ void close(int q) {
    const int y = q - 3;
    if (y < y0 || y >= y1) return;
    const A v = cell[(R + 1) & 3].acc;
    if (pair && !((keep >> ((R + 1) & 3)) & 1)) return;
    fbase[(long)N0 * y] = (T)v;
  }

  // Step q: plane q sits in LDS buffer b = q mod NB; vector memory operations
  // of a wave retire in issue order, so a vmcnt wait on all but the newest
  // operations completes every older load.
  //  NB = 3: the loads of plane q+2 are issued last; the wait before the
  //   barrier leaves exactly those in flight, so plane q+1 is complete in LDS
  //   for every wave after the barrier.
  //  NB = 2: the loads of plane q+1 are issued first and overlap the step;
  //   the wait leaves only this step's store of f in flight.
  template <int R> __device__ __forceinline__ void step(int q, int b) {
    if (NB == 2 && q + 1 < y1 + 3) fetch(q + 1, b ^ 1);
    if (active) {
      double efx = 0., efy = 0.;
      if (q < y1) field_at(q, b, efx, efy);  // no cell opens beyond the last y
      open<R>(q, efx, efy);
      accumulate<R>(q, b);
      close<R>(q);
    }
    int n = 0;
    if (NB == 3) {
      if (q + 2 < y1 + 3) n = fetch(q + 2, b == 0 ? 2 : b - 1);
    } else {
      // (a shared slab's store may have been skipped: wait for everything)
      n = (wave_has_cells && !pair && q >= y0 + 3 && q - 3 < y1) ? 1 : 0;
    }
    wait_vm(n);
    __builtin_amdgcn_s_barrier();
  }
};

// 16-byte chunks of a slab row: the row's N0 + 4 values and, when they are not
// whole chunks, the up to vpl - 1 values before them (see YStream).
__host__ __device__ inline int ys_row_chunks(int N0, int vpl) {
  const int n = N0 + 4;
  return n % vpl ? (n + vpl - 1 + vpl - 1) / vpl : n / vpl;
}

// Workgroup -> (vx tile, vy).  Workgroups go to the 8 XCDs (each with its
// own L2) round-robin: block b runs on XCD b mod 8, as the (b / 8)-th of
// that XCD.  The workgroups that stage the same C4 rows are those of the 5
// neighbouring vy and the neighbouring vx tiles; with remap, XCD x takes the
// vx tiles [x ntile/8, (x+1) ntile/8) for every vy, vy slower and tile
// faster, so that the workgroups resident on one XCD at a time cover a
// compact block of (tile, vy) and share their rows through its L2, while
// every XCD gets its share of each vy.  Without remap (or when the tiles do
// not split over the XCDs) block b is (b mod ntile, b / ntile).
__device__ __forceinline__ void ys_block_tile(int b, int ntile, int remap, int &tile, int &ivy) {
  constexpr int NX = 8;
  if (remap && ntile % NX == 0) {
    const int x = b % NX, k = b / NX;
    const int tx = ntile / NX;  // tiles per XCD
    ivy = k / tx;
    tile = x * tx + k % tx;
  } else {
    tile = b % ntile;
    ivy = b / ntile;
  }
}

}  // namespace

template <typename T, typename A, int TVX, int NB, int RXC>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(sizeof(A) == 4 ? 3 : 1)))
void k_advect4d_ys(const T *__restrict__ c4, const double *__restrict__ exy, Geom g,
                                                     FeetConsts fc, double dt, T *__restrict__ fout,
                                                     int *__restrict__ err, int force, int remap, int iv0, int nslab, int ylen) {
  extern __shared__ __align__(16) unsigned char ys_smem[];
  YStream<T, A, TVX, NB, RXC> s;
  s.force = force;
  s.c4 = c4;
  s.exy = exy;
  s.fout = fout;
  s.N0 = g.n[0];
  s.N1 = g.n[1];
  s.N2 = g.n[2];
  s.N3 = g.n[3];
  const int per_row = ys_row_chunks(s.N0, s.VPL);  // 16-byte chunks per slab row
  s.RX = per_row * s.VPL;
  const int nchunk = 5 * (TVX + 4) * per_row;
  const int ninstr = (nchunk + 63) >> 6;
  s.slab_bytes = ninstr * 1024;
  s.cpr = (s.N0 + 63) >> 6;
  s.EPR = 64 * s.cpr;
  s.slab = (T *)ys_smem;
  s.eb = (double *)(ys_smem + NB * (size_t)s.slab_bytes);
  s.kconst = s.eb + NB * 6 * s.EPR;
  s.qtab = s.kconst + s.KC_N + 2 * s.QT;
  if (threadIdx.x == 0) {
    double *k = s.kconst;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      k[s.KC_MIN + j] = g.minPhy[j];
      k[s.KC_INV + j] = g.inv_dx[j];
      k[s.KC_LMIN + j] = fc.locmin[j];
      k[s.KC_LMAX + j] = fc.locmax[j];
      k[s.KC_DX + j] = g.dx[j];
    }
    k[s.KC_DT] = dt;
    k[s.KC_VHI] = g.minPhy[2] + fc.rxwidth[2];
    k[s.KC_VHI + 1] = g.minPhy[3] + fc.rxwidth[3];
  }
  const int ntile = (s.N2 + TVX - 1) / TVX;
  int tile, ivy;
  // y segments of the whole (tile, slab) grid one after another
  const int seg = blockIdx.x / (ntile * nslab);
  s.y0 = seg * ylen;
  s.y1 = min(s.N1, s.y0 + ylen);
  ys_block_tile(blockIdx.x - seg * ntile * nslab, ntile, remap, tile, ivy);
  // slab N3 (launched when iv0 >= 0): the second workgroups of slab iv0
  s.pair = 0;
  if (iv0 >= 0) {
    if (ivy == s.N3) {
      ivy = iv0;
      s.pair = 2;
    } else if (ivy == iv0) {
      s.pair = 1;
    }
  }
  s.keep = 0;
  s.ivy = ivy;
  {  // the y part of computeFeet for every cell y of this vy (VMO/Advection.hpp:174-196)
    const double vyw = g.minPhy[3] + ivy * g.dx[3];
    for (int q = threadIdx.x; q < s.N1; q += blockDim.x) {
      const double yq = g.minPhy[1] + q * g.dx[1];
      const double xt1 = half_y(g, yq, vyw, dt);
      const int ip1 = (int)(round(xt1) - 1);
      const double py = xt1 - ip1;
      double *t = s.qtab + s.QT * q;
      t[0] = (double)ip1;
      t[1] = .5 * (py) * (py - 1.);
      t[2 - s.QT] = -1. * (py) * (py - 2.);
      t[3 - 2 * s.QT] = .5 * (py - 1.) * (py - 2.);
    }
    // past the last cell: weights of cells that do not exist
    if (threadIdx.x == 0) {
      double *t = s.qtab + s.QT * s.N1;
      t[2 - s.QT] = t[3 - s.QT] = t[3 - 2 * s.QT] = 0.;
    }
  }
  __syncthreads();  // both tables are written before the first fetch reads them
  const int tid = threadIdx.x;
  // (the last tile may reach past N2)
  s.active = tid < s.N0 * TVX && tile * TVX + tid / s.N0 < s.N2;
  s.ix = s.active ? tid % s.N0 : 0;
  s.tv = s.active ? tid / s.N0 : 0;
  s.ivx = tile * TVX + s.tv;
  const double x = g.minPhy[0] + s.ix * g.dx[0];
  const double vx = g.minPhy[2] + s.ivx * g.dx[2];
  const double vy = g.minPhy[3] + s.ivy * g.dx[3];
  s.oyw = s.pair ? s.pair == 2 ? -1 : 0 : vy > 0. ? -1 : 0;
  s.ax = -(dt * vx) * g.inv_dx[0];
  s.ay1 = -(dt * vy) * g.inv_dx[1] - (s.pair ? 0 : s.oyw);
  s.bex = 0.5 * dt * dt * g.inv_dx[0];
  s.bey = 0.5 * dt * dt * g.inv_dx[1];
  s.bvx = -dt * g.inv_dx[2];
  s.bvy = -dt * g.inv_dx[3];
  s.lo2 = s.ivx == 0 ? 0. : -2.;
  s.lo3 = s.ivy == 0 ? 0. : -2.;
  s.row0 = s.ix + 1 + (RXC ? RXC : s.RX) * (s.tv + 1 + (TVX + 4));
  s.fbase = fout + s.ix + (long)s.N0 * s.N1 * (s.ivx + (long)s.N2 * s.ivy);
  {
    const C4Pitch cp = c4_pitch(s.N0, s.N1, s.N2);
    s.F0 = (int)cp.s1;
    s.S1 = cp.s1;
    s.S2 = cp.s2;
    s.S3 = cp.s3;
  }
  s.wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  s.lane = tid & 63;
  s.nwave = (int)(blockDim.x >> 6);
  s.nslot = s.wave < ninstr ? (ninstr - 1 - s.wave) / s.nwave + 1 : 0;
  {
#pragma unroll
    for (int k = 0; k < s.MS; k++) {
      // chunks past the slab repeat its last chunk into the buffer's padding
      const int c = min(64 * (s.wave + k * s.nwave) + s.lane, nchunk - 1);
      const int row = c / per_row, col = c - row * per_row;
      // (rows past the last plane of C4 belong to no cell: repeat it)
      const int kvx = min(row % (TVX + 4), s.N2 + 4 - tile * TVX), kvy = row / (TVX + 4);
      s.voff[k] = (unsigned)((s.S2 * kvx + s.S3 * kvy + (long)s.VPL * col) * (long)sizeof(T));
    }
  }
  {  // x part of computeFeet's E interpolation (VMO/Advection.hpp:174-196)
    double xt0 = x - 0.5 * dt * vx;
    xt0 = g.inv_dx[0] * (xt0 - g.minPhy[0]);
    const int ip0 = (int)(round(xt0) - 1);
    const double px = xt0 - ip0;
    s.cx[0] = .5 * (px - 1.) * (px - 2.);
    s.cx[1] = -1. * (px) * (px - 2.);
    s.cx[2] = .5 * (px) * (px - 1.);
#pragma unroll
    for (int k0 = 0; k0 < 3; k0++) s.jx[k0] = ((ip0 + k0) % s.N0 + s.N0) % s.N0;
  }
  s.ip1p = -(1 << 30);
  // position (x -2, y -3, vx tile-2, vy ivy-2) sits at storage (1, 0, tile+1, ivy+1)
  s.cbase = (int)(1 + s.S2 * (tile * TVX + 1) + s.S3 * (s.ivy + 1));
#pragma unroll
  for (int c = 0; c < 4; c++) {
    s.cell[c].row = s.row0;
    s.cell[c].acc = 0;
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int k = 0; k < 4; k++) s.cell[c].w[j][k] = 0;
  }
  s.bad = 0;
  s.wave_has_cells = __builtin_amdgcn_ballot_w64(s.active) != 0;
  if (NB == 3) {  // planes 0 and 1 in flight; wait for plane 0
    s.fetch(s.y0, 0);
    wait_vm(s.fetch(s.y0 + 1, 1));
  } else {
    s.fetch(s.y0, 0);
    wait_vm(0);
  }
  __builtin_amdgcn_s_barrier();
  int b = 0;  // (q - y0) mod NB
  for (int q0 = s.y0; q0 < s.y1 + 3; q0 += 4) {
    s.template step<0>(q0, b);
    b = b == NB - 1 ? 0 : b + 1;
    if (q0 + 1 < s.y1 + 3) s.template step<1>(q0 + 1, b);
    b = b == NB - 1 ? 0 : b + 1;
    if (q0 + 2 < s.y1 + 3) s.template step<2>(q0 + 2, b);
    b = b == NB - 1 ? 0 : b + 1;
    if (q0 + 3 < s.y1 + 3) s.template step<3>(q0 + 3, b);
    b = b == NB - 1 ? 0 : b + 1;
  }
  if (s.bad) atomicOr(err, 2);
}

namespace {

struct YsPlan {
  int tvx = 0;  // 0: not eligible
  int nb = 3;   // LDS plane buffers
  int block = 0;
  size_t lds = 0;
};

// Slab DMA instructions per plane and E points per LDS row of the streaming
// kernel (the same arithmetic as its set-up).
long ys_slab_instr(long N0, long tvx, size_t tsz) {
  return (5 * (tvx + 4) * ys_row_chunks((int)N0, 16 / (int)tsz) + 63) / 64;
}
long ys_epr(long N0) { return (N0 + 63) / 64 * 64; }

// want_tvx / want_nb: a chosen vx tile and buffer count (0: free); the
// environment (VLP4D_YS_TVX, VLP4D_YS_NBUF) overrides them.
YsPlan ys_plan(const Geom &g, size_t tsz, int want_tvx = 0, int want_nb = 0) {
  YsPlan p;
  const long N0 = g.n[0], N1 = g.n[1], N2 = g.n[2], N3 = g.n[3];
  const long c4n = c4_elems(N0, N1, N2, N3);
  if (c4n >= (1L << 31)) return p;
  int force = want_tvx, force_nb = want_nb;
  if (const char *e = getenv("VLP4D_YS_TVX")) force = atoi(e);
  if (const char *e = getenv("VLP4D_YS_NBUF")) force_nb = atoi(e);
  // Preference order measured at 128^4: two or more small workgroups per CU
  // (vx tile 2, two buffers), whose barriers are independent, run best for
  // both slab types (double: 8.0 ms against 8.7 at tile 4; float storage 7.5
  // against 8.1; float arithmetic, three waves per SIMD, 5.2 against 6.2).
  // Tiles of 2 in rows of 33 to 64 points make workgroups of two waves; tile 4,
  // as the same three or four waves as tile 2 in longer rows, is taken first
  // there: it stages 8 slab rows for 4 of vx instead of 12 (64 x 48 x 100 x 100
  // 1.17 -> 0.78 ms in double, 0.70 -> 0.48 in float; 48^4 0.226 -> 0.200, 56^4
  // 0.333 -> 0.311; 96^4 stays with tile 2, 2.6 ms against 3.0).
  // A tile is passed over when another has over 1/0.9 times as many lanes with
  // cells on a CU: lanes past N0 TVX (to whole waves) and past N2 (last tile)
  // do nothing, and the workgroups of a CU are bounded by LDS and waves, counted
  // as three per SIMD for float storage, else two.  (By the share of such lanes
  // alone, 80 x 96 x 96 x 80 in float took tile 4: 1.76 ms, tile 2 takes 1.09.)
  // Float storage with double arithmetic has the registers for two waves only,
  // but counted so it fares no better: over 90 ragged grids, rows of 17 to 24
  // points would take tile 2 instead of 8, 4 % slower (31 of 35 slower, by up to 8
  // %), the others even (tile 8 to 4 0.99, 4 to 2 0.99 of the time, 0.77 to 1.32).
  // Any extents are taken; the vx-blocked kernel, which ragged grids used to
  // run, is bound by L1 latency: 90 x 77 x 84 x 75 4.23 -> 1.51 ms (double) and
  // 2.95 -> 0.78 (float), 61 x 50 x 45 x 58 0.78 -> 0.33, 20 x 21 x 22 x 23
  // 0.30 -> 0.07.  It keeps the grids whose C4 has 2^31 elements or whose
  // slab does not fit LDS.
  static const int pref_f[][2] = {{2, 2}, {4, 2}, {8, 2}, {4, 3}, {2, 3}, {8, 3}};
  static const int pref_d[][2] = {{2, 2}, {4, 2}, {8, 2}, {4, 3}, {8, 3}, {2, 3}};
  static const int pref_4[][2] = {{4, 2}, {2, 2}, {8, 2}, {4, 3}, {8, 3}, {2, 3}};
  const auto &pref = N0 > 32 && N0 <= 64 ? pref_4 : tsz == sizeof(float) ? pref_f : pref_d;
  double best = 0.;
  for (int pass = 0; pass < 2; pass++)
    for (const auto &c : pref) {
      const int tvx = c[0], nb = c[1];
      if (force && tvx != force) continue;
      if (force_nb && nb != force_nb) continue;
      const long lanes = N0 * tvx;
      if (lanes > 512) continue;
      const int block = (int)((lanes + 63) / 64 * 64);
      const long ninstr = ys_slab_instr(N0, tvx, tsz);
      if ((ninstr + block / 64 - 1) / (block / 64) > 8) continue;  // DMA slots per wave
      const size_t lds = nb * (size_t)ninstr * 1024 + nb * 3 * (size_t)ys_epr(N0) * 2 * sizeof(double) +
                         (24 + 4 * (size_t)(N1 + 2)) * sizeof(double);  // domain constants, per-step table
      if (lds > 160 * 1024) continue;
      const long per_cu = std::max(1L, std::min((long)(160 * 1024 / lds),
                                                4L * (tsz == sizeof(float) ? 3 : 2) / (block / 64)));
      const double busy = (double)per_cu * N0 * N2 / ((N2 + tvx - 1) / tvx);
      if (pass == 0) {
        if (busy > best) best = busy;
        continue;
      }
      if (busy < 0.9 * best) continue;
      p.tvx = tvx;
      p.nb = nb;
      p.block = block;
      p.lds = lds;
      return p;
    }
  return p;
}

template <typename T, typename A, int TVX, int NB, int RXC>
void launch_ys_t(const Geom &g, const YsPlan &p, const T *c4, const double *exy, double dt, T *fout, int *err,
                 hipStream_t s) {
  const void *fn = (const void *)k_advect4d_ys<T, A, TVX, NB, RXC>;
  if (p.lds > 64 * 1024) (void)hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.lds);
  // the slab whose velocity vanishes (to rounding), if there is one: its
  // drift dt vy / dy is below that of any field.  It is shared by two sets
  // of workgroups as long as the launch is short enough for its tail to show:
  // 48^4 gradient 29.2 -> 26.3 ms, 64^4 two-stream 30.8 -> 27.4 ms for 20
  // steps, but 96^4 float storage (4608 workgroups) 187.8 -> 191.0 ms and
  // 128^4 (8192) 215.1 -> 216.6 ms, the gathering workgroups being hidden
  // there by the others.
  int iv0 = -1;
  const int ntile = (g.n[2] + TVX - 1) / TVX;
  if ((long)ntile * g.n[3] < 4096) {
    const double r = -g.minPhy[3] * g.inv_dx[3];
    if (r > -0.5 && r < g.n[3] - 0.5 && std::fabs(r - std::nearbyint(r)) < 1e-6) iv0 = (int)std::nearbyint(r);
  }
  const int nslab = g.n[3] + (iv0 >= 0);
  // y segments, when the workgroups would not fill the chip: the fewest
  // rounds of workgroups times steps (three beyond the cells, two steps' time
  // for the set-up).  Workgroups per CU by LDS and by the waves per SIMD that
  // registers allow (two with double arithmetic, three with float).  Advection of 16^4 FP64 58 ->
  // 23 us, 32^4 float 97 -> 43, 48^4 FP64 355 -> 195; from four rounds on one
  // segment is taken.
  int ylen = g.n[1];
  {
    const int waves = p.block / 64, per_simd = sizeof(A) == 4 ? 3 : 2;
    const long per_cu = std::max(1L, std::min((long)(160 * 1024 / p.lds), 4L * per_simd / waves));
    const long cap = 256 * per_cu, w = (long)ntile * nslab;
    long best = -1;
    for (int n = 1; n <= (w < 4 * cap ? g.n[1] / 4 : 1); n++) {
      const int len = (g.n[1] + n - 1) / n;
      const long cost = (w * n + cap - 1) / cap * (len + 5);
      if (best < 0 || cost < best) {
        best = cost;
        ylen = len;
      }
    }
  }
  const int nseg = (g.n[1] + ylen - 1) / ylen;
  const unsigned grid = (unsigned)(ntile * nslab * nseg);
  int force = 0;  // test switch: VLP4D_YS_FORCE=1 rows per cell, 2 direct gather, 3 both
  if (const char *e = getenv("VLP4D_YS_FORCE")) force = atoi(e) & 3;
  int remap = 1;  // VLP4D_YS_REMAP=0: block b -> (b mod ntile, b / ntile)
  if (const char *e = getenv("VLP4D_YS_REMAP")) remap = atoi(e) != 0;
  hipLaunchKernelGGL((k_advect4d_ys<T, A, TVX, NB, RXC>), dim3(grid), dim3(p.block), p.lds, s, c4, exy, g,
                     feet_consts(g), dt, fout, err, force, remap, iv0, nslab, ylen);
}

template <typename T, typename A, int TVX>
void launch_ys_nb(const Geom &g, const YsPlan &p, const T *c4, const double *exy, double dt, T *fout, int *err,
                  hipStream_t s) {
  // N0 = 128 with the vx tile of 2 (the tile chosen at 128^4) takes the
  // kernel with the slab row pitch 132 built in
  if constexpr (TVX == 2) {
    if (g.n[0] == 128) {
      if (p.nb == 2) launch_ys_t<T, A, TVX, 2, 132>(g, p, c4, exy, dt, fout, err, s);
      else launch_ys_t<T, A, TVX, 3, 132>(g, p, c4, exy, dt, fout, err, s);
      return;
    }
  }
  if (p.nb == 2) launch_ys_t<T, A, TVX, 2, 0>(g, p, c4, exy, dt, fout, err, s);
  else launch_ys_t<T, A, TVX, 3, 0>(g, p, c4, exy, dt, fout, err, s);
}

}  // namespace

// Returns false (nothing launched) when the geometry does not fit the
// streaming kernel.
template <typename T, typename A>
bool launch_advect4d_ystream(const Geom &g, const T *c4, const double *exy, double dt, T *fout, int *err,
                             hipStream_t s, int ys_tvx, int ys_nb) {
  if (const char *e = getenv("VLP4D_YSTREAM"))
    if (atoi(e) == 0) return false;
  YsPlan p = ys_plan(g, sizeof(T), ys_tvx, ys_nb);
  if (!p.tvx && (ys_tvx || ys_nb)) p = ys_plan(g, sizeof(T));  // a choice this geometry cannot take
  switch (p.tvx) {
    case 8: launch_ys_nb<T, A, 8>(g, p, c4, exy, dt, fout, err, s); return true;
    case 4: launch_ys_nb<T, A, 4>(g, p, c4, exy, dt, fout, err, s); return true;
    case 2: launch_ys_nb<T, A, 2>(g, p, c4, exy, dt, fout, err, s); return true;
    default: return false;
  }
}

bool ystream_eligible(const Geom &g, size_t tsz, int tvx, int nb) {
  const YsPlan p = ys_plan(g, tsz, tvx, nb);
  return p.tvx == tvx && p.nb == nb;
}

bool ystream_preferred(const Geom &g, size_t tsz, int tvx, int nb) {
  const YsPlan p = ys_plan(g, tsz);
  return p.tvx == tvx && p.nb == nb;
}

int ystream_tvx(const Geom &g, bool fp32_storage) {
  if (const char *e = getenv("VLP4D_YSTREAM"))
    if (atoi(e) == 0) return 0;
  return ys_plan(g, fp32_storage ? sizeof(float) : sizeof(double)).tvx;
}

template bool launch_advect4d_ystream<double, double>(const Geom &, const double *, const double *, double, double *,
                                                      int *, hipStream_t, int, int);
template bool launch_advect4d_ystream<float, double>(const Geom &, const float *, const double *, double, float *,
                                                     int *, hipStream_t, int, int);
template bool launch_advect4d_ystream<float, float>(const Geom &, const float *, const double *, double, float *, int *,
                                                    hipStream_t, int, int);

}  // namespace vlp
