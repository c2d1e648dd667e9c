// The binary64 three-centre kernels of s/p species with canonical tables:
// bcna (neutral, and with charged shells) and the McWEDA densities (orbital
// and shell blocks).  A workgroup owns a tile of whole target segments (at
// most 64 triplets unless one segment is longer) and has one wavefront per
// term: the neutral bcna term and each charged shell of the third atom
// (M_assemble_3c_DOGS.f90:298-318), or each of its shells
// (M_assemble_rho_McWEDA_DOGS.f90:470-500).  A wavefront works alone up to the
// sum, in four phases:
//   A  one lane per triplet: geometry and frame, grid cell, method of the cell
//      (the reference's gradient test, precomputed per cell), Legendre values;
//      the triplets are listed by matrix-element count and method;
//   B  the theta sums (M_Fdata_3c.f90:383-489): a lane takes one element of a
//      3-point cell; four lanes take one of a 16-point cell, a column each;
//   C  one lane per triplet: rotation (or the shell-block order) and the
//      term's factors, into the triplet's LDS row;
//   D  one lane per (segment, block element): the rows added in triplet order,
//      term by term.
// Every operation and its order is that of the one-lane-per-triplet form, so
// the blocks are the reference's bits; the phases only change which lane does
// what.
//
// What bounds it: a lane's chain of table gathers and LDS round trips, so the
// layout is chosen for wavefronts that do not wait for each other before the
// sum and for many loads per wait: the five theta values of an element are
// contiguous in the slab (two 16-byte loads and one of 8), all loads of a
// 3-point sum or of a column are issued before the first is used, and lanes of
// one list share element count and method, so no lane of a C/H/N/O tile idles
// for elements that its pair does not have.  A wavefront's LDS is 10 KB;
// registers for three wavefronts per SIMD (at four, 14 values spill: equal or
// up to 8 % slower, 43 % with charged shells).
//
// Measured, one lane per element with a loop over theta -> this form:
// C/H/N/O, 3000 atoms, 2.81 M triplets: bcna 621 -> 217 us; Si, 4096 atoms,
// 2.00 M: 316 -> 185 us; C/H/N/O, 1001 atoms with charged shells 1188 -> 350
// us; densities, Si of 1728 atoms, 0.85 M: 498 -> 192 us, shell blocks 173 ->
// 85 us.
#pragma once

#include "fb_device.h"
#include "fb_3c_dev.h"
#include "fb_sp.h"

enum { W3_BCNA = 0, W3_BCNA_Q = 1, W3_RHO = 2, W3_RHOS = 3 };

// wavefronts (terms) per workgroup
__host__ __device__ constexpr int w3_terms(int mode) { return mode == W3_BCNA ? 1 : (mode == W3_BCNA_Q ? 3 : 2); }

#define W3_T 64            // triplets per pass
#define W3_F 11            // LDS row of one triplet's elements (10, odd stride)
#define W3_ROW 17          // contribution row: 16 block elements and whether the triplet has the term

struct W3Par {
  double px, py, sint, p[4];   // p1..p4 (p0 = 1)
  int64_t base;                // FP64 slab index of (theta 0, ix, iy, ME 0)
  int rs, pad;                 // slab values per iy row
};

struct W3Lds {
  W3Par q[W3_T];
  double F[W3_T][W3_F];
};
static_assert(sizeof(W3Lds) >= sizeof(double) * W3_T * W3_ROW, "the rows take the place of the parameters");

__device__ __forceinline__ void w3_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// value of lane K of the quad
template <int K>
__device__ __forceinline__ double quad_lane(double x) {
  const int2 v = __builtin_bit_cast(int2, x);
  int2 r;
  r.x = __builtin_amdgcn_mov_dpp(v.x, K * 0x55, 0xf, 0xf, true);
  r.y = __builtin_amdgcn_mov_dpp(v.y, K * 0x55, 0xf, 0xf, true);
  return __builtin_bit_cast(double, r);
}

// elements of a list of n triplets with NME elements each, 3-point cells
template <int NME, int NM0>
__device__ __forceinline__ void w3_three(const double *tab, W3Lds &S, const unsigned char *ord, int n, int lane) {
  for (int it = lane; it < n * NME; it += 64) {
    const int k = it / NME, m = it - k * NME, t = ord[k];
    const W3Par &q = S.q[t];
    const double *e = tab + q.base + m * FB_NTHETA;
    double a[FB_NTHETA], b[FB_NTHETA], c[FB_NTHETA];
    load_theta(e, a);
    load_theta(e + NME * FB_NTHETA, b);
    load_theta(e + q.rs, c);
    const double px = q.px, py = q.py, p[5] = {1.0, q.p[0], q.p[1], q.p[2], q.p[3]};
    double F = 0.0;
#pragma unroll
    for (int th = 0; th < FB_NTHETA; th++) {
      const double interim = ((1.0 - px - py) * a[th] + px * b[th]) + py * c[th];
      F = F + p[th] * interim;
    }
    S.F[t][m] = m >= NM0 ? F * q.sint : F;
  }
}

// the same for 16-point cells: lane c of a quad interpolates column ix + c - 1
// along y, every lane of the quad then the four columns along x
template <int NME, int NM0>
__device__ __forceinline__ void w3_sixteen(const double *tab, W3Lds &S, const unsigned char *ord, int n, int lane) {
  const int c = lane & 3;
  for (int it = lane >> 2; it < n * NME; it += 16) {
    const int k = it / NME, m = it - k * NME, t = ord[k];
    const W3Par &q = S.q[t];
    const double *e = tab + q.base + m * FB_NTHETA + (c - 1) * (NME * FB_NTHETA);
    double y0[FB_NTHETA], y1[FB_NTHETA], y2[FB_NTHETA], y3[FB_NTHETA];
    load_theta(e - q.rs, y0);
    load_theta(e, y1);
    load_theta(e + q.rs, y2);
    load_theta(e + 2 * q.rs, y3);
    const double px = q.px, py = q.py, p[5] = {1.0, q.p[0], q.p[1], q.p[2], q.p[3]};
    double F = 0.0;
#pragma unroll
    for (int th = 0; th < FB_NTHETA; th++) {
      auto cubic = [](double v0, double v1, double v2, double v3, double x) {
        double f1m1 = v0;
        double f1m2 = 2.0 * f1m1, f1m3 = 3.0 * f1m1;
        double f0p3 = 3.0 * v1, f0p6 = 2.0 * f0p3;
        double f1p3 = 3.0 * v2, f1p6 = 2.0 * f1p3;
        double f2p1 = v3;
        double bb3 = -f1m1 + f0p3 - f1p3 + f2p1;
        double bb2 = f1m3 - f0p6 + f1p3;
        double bb1 = -f1m2 - f0p3 + f1p6 - f2p1;
        double bb0 = f0p6;
        return ((bb3 * x + bb2) * x + bb1) * x + bb0;
      };
      const double g = cubic(y0[th], y1[th], y2[th], y3[th], py);
      const double interim = cubic(quad_lane<0>(g), quad_lane<1>(g), quad_lane<2>(g), quad_lane<3>(g), px) / 36.0;
      F = F + p[th] * interim;
    }
    if (c == 0) S.F[t][m] = m >= NM0 ? F * q.sint : F;
  }
}

// shell blocks (rhoS, issh major in the table, column-major in the block) of
// NSI x NSJ shells
template <int MODE>
__device__ __forceinline__ void w3_block(int cls, const double *pm, const double *F, double *X) {
  if (MODE == W3_RHOS) {
    const int nsi = (cls & 2) ? 2 : 1, nsj = (cls & 1) ? 2 : 1;
    X[0] = F[0];
    X[1] = nsi == 2 ? (nsj == 2 ? F[2] : F[1]) : F[1];
    X[2] = F[1];
    X[3] = F[3];
    return;
  }
  switch (cls) {
    case 3: rot3c_sp<double>(3, pm, F, X); break;
    case 2: rot3c_sp<double>(2, pm, F, X); break;
    case 1: rot3c_sp<double>(1, pm, F, X); break;
    default: rot3c_sp<double>(0, pm, F, X); break;
  }
}

template <int MODE>
__global__ __launch_bounds__(64 * w3_terms(MODE), 3) void k_3c_wave(DView v) {
  constexpr int NT = w3_terms(MODE);
  constexpr bool ORB = MODE != W3_RHOS, RHO = MODE >= W3_RHO;
  constexpr int NB = ORB ? 16 : 4;                      // block elements, at most
  constexpr int N3 = ORB ? 10 : 4, N2 = ORB ? 3 : 2;    // elements of an sp-sp and an s-sp or sp-s pair
  __shared__ W3Lds sm[NT];
  __shared__ int sSeg[W3_T + 1];
  __shared__ int64_t sBo[W3_T];
  __shared__ unsigned char sNb[W3_T], sOrd[NT][W3_T];
  __shared__ double sQ[MODE == W3_BCNA_Q ? 2 : 1][4][MODE == W3_BCNA_Q ? W3_T : 1];   // geometry of the charged terms
  const int tid = threadIdx.x, lane = tid & 63, term = NT == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 6);
  W3Lds &S = sm[term];
  double(*const sC)[W3_ROW] = reinterpret_cast<double(*)[W3_ROW]>(&S);
  unsigned char *const ord = sOrd[term];
  const int4 td = v.tiles[0][xcd_tile(blockIdx.x, gridDim.x)];
  const int first = td.x, nown = td.y - td.x + 1, r0 = td.z, r1 = td.w;
  if (nown <= 0) return;
  const int64_t *const off = MODE == W3_RHOS ? v.wboff : v.boff;
  double *const out = v.mat[MODE == W3_RHO ? FB_MAT_RHO_IN : (MODE == W3_RHOS ? FB_MAT_RHOW_IN : FB_MAT_VNA)];
  for (int k = tid; k <= nown; k += 64 * NT) sSeg[k] = (int)v.seg_off[first + k];
  for (int k = tid; k < nown; k += 64 * NT) {
    const int p = v.seg_pair[first + k];
    const int64_t b0 = off[p];
    sBo[k] = b0;
    sNb[k] = (unsigned char)(off[p + 1] - b0);
  }
  int status = 0;
  for (int c0 = r0; c0 < r1; c0 += W3_T) {
    const int nt = min(W3_T, r1 - c0);
    // ---------------- phase A
    bool have = false, m1 = false;
    int cls = 0;
    double pm[9], factor = FB_P_EQ2;
    if (lane < nt) {
      const int4 tr = v.trip[c0 + lane];
      const int aux = v.trip_aux[c0 + lane];
      Geo3 G;
      d_geo3(v, tr, aux, G);
      cls = (G.nmu == 4 ? 2 : 0) + (G.nnu == 4 ? 1 : 0);
      int gid = -1;
      if (MODE == W3_BCNA || (MODE == W3_BCNA_Q && term == 0)) {
        have = true;
        gid = (aux & 0xffff) == 0xffff ? -1 : (aux & 0xffff);
      } else if (v.sp.nssh[G.indna - 1] >= (RHO ? term + 1 : term)) {
        const int sh = RHO ? term : term - 1;   // shell of the third atom, 0-based
        factor = RHO ? v.qin[tr.x * FB_MAXSH + sh] : v.dQ[tr.x * FB_MAXSH + sh];
        have = RHO || factor != 0.0;            // the reference adds an exact zero for dQ = 0
        const int k = ((G.in1 - 1) * v.sp.ns + (G.in2 - 1)) * v.sp.ns + (G.indna - 1);
        if (have) gid = RHO ? v.idx3r[(k * 2 + (ORB ? 0 : 1)) * FB_MAXSUB3 + sh + 1] : v.idx3c[k * FB_MAXSUB3 + sh + 1];
      }
      if (have && gid < 0) {
        status |= ST_NO_TABLE;
        have = false;
      }
      if (have) {
        W3Par &q = S.q[lane];
        double p[5], sint;
        d_legendre(G.cost, p, &sint);
        q.sint = sint;
#pragma unroll
        for (int k = 0; k < 4; k++) q.p[k] = p[k + 1];
        const DGroup3c g = group3c_scalar(v, gid);
        const int nx = g.nx, ny = g.ny;
        const double dx = g.xmax / (nx - 1.0), dy = g.ymax / (ny - 1.0);
        int ix = (int)(G.x / dx) + 1, iy = (int)(G.z / dy) + 1;
        if (ix < 2) ix = 2;
        if (iy < 2) iy = 2;
        if (ix > nx - 2) ix = nx - 2;
        if (iy > ny - 2) iy = ny - 2;
        q.px = G.x / dx - ix + 1.0;
        q.py = G.z / dy - iy + 1.0;
        q.rs = nx * g.nME * FB_NTHETA;
        q.base = g.off + FB_T64(0, ix, iy, 0, nx, g.nME);
        m1 = v.meth3c[g.moff + (int64_t)(iy - 1) * nx + (ix - 1)] != 0;
      }
      if (ORB) d_pmat<double>(G.eps, pm);
      if (MODE == W3_BCNA_Q && term > 0) {
        sQ[term - 1][0][lane] = G.z;
        sQ[term - 1][1][lane] = G.d13;
        sQ[term - 1][2][lane] = G.d23;
        sQ[term - 1][3][lane] = G.stinky;
      }
    }
    // lists: three element counts, each with its 3-point cells first
    int n[6], at = 0;
    {
      const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
      for (int c = 0; c < 3; c++) {
        const bool mine = have && (c == 0 ? cls == 3 : (c == 1 ? cls == 1 || cls == 2 : cls == 0));
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const unsigned long long b = __ballot(mine && m1 == (h == 0));
          if (mine && m1 == (h == 0)) ord[at + __popcll(b & below)] = (unsigned char)lane;
          n[2 * c + h] = __popcll(b);
          at += __popcll(b);
        }
      }
    }
    w3_fence();
    // ---------------- phase B
    {
      const double *tab = v.tab3c;
      const unsigned char *o = ord;
      constexpr int A3 = ORB ? 6 : 4, A2 = 2;   // leading elements without sin(theta)
      w3_three<N3, A3>(tab, S, o, n[0], lane);
      o += n[0];
      w3_sixteen<N3, A3>(tab, S, o, n[1], lane);
      o += n[1];
      w3_three<N2, A2>(tab, S, o, n[2], lane);
      o += n[2];
      w3_sixteen<N2, A2>(tab, S, o, n[3], lane);
      o += n[3];
      w3_three<1, 1>(tab, S, o, n[4], lane);
      o += n[4];
      w3_sixteen<1, 1>(tab, S, o, n[5], lane);
    }
    w3_fence();
    // ---------------- phase C
    double X[NB];
    if (have) {
      double F[N3];
#pragma unroll
      for (int m = 0; m < N3; m++) F[m] = S.F[lane][m];
      // xp = yp x zp of epsilon.f90 in the (y, z, x) order: the third column
      // need not be kept through phase B
      pm[6] = pm[1] * pm[5] - pm[2] * pm[4];
      pm[7] = pm[2] * pm[3] - pm[0] * pm[5];
      pm[8] = pm[0] * pm[4] - pm[1] * pm[3];
      w3_block<MODE>(cls, pm, F, X);
    }
    w3_fence();   // the rows overwrite parameters and elements
    if (lane < nt) {
      double *row = sC[lane];
      row[16] = have ? 1.0 : 0.0;
      if (have) {
        const int nbl = ORB ? (cls & 2 ? 4 : 1) * (cls & 1 ? 4 : 1) : (cls & 2 ? 2 : 1) * (cls & 1 ? 2 : 1);
        if (MODE == W3_BCNA_Q && term > 0) {
          const int64_t bo = v.boff[v.trip_pair[c0 + lane]];
          const double *sb = v.mat[FB_MAT_S] + bo, *db = v.mat[FB_MAT_DIP] + bo;
          const double z = sQ[term - 1][0][lane], d13 = sQ[term - 1][1][lane], d23 = sQ[term - 1][2][lane];
          const double stinky = sQ[term - 1][3][lane];
#pragma unroll
          for (int i = 0; i < NB; i++) {
            if (i >= nbl) break;
            double sterm = sb[i] / 2.0, dterm = db[i] / z;
            double emnpl = (sterm - dterm) / d13 + (sterm + dterm) / d23;
            row[i] = factor * (stinky * X[i] + (1.0 - stinky) * emnpl) * FB_P_EQ2;
          }
        } else {
#pragma unroll
          for (int i = 0; i < NB; i++)
            if (i < nbl) row[i] = X[i] * factor;
        }
      }
    }
    if (NT > 1) __syncthreads();
    else w3_fence();
    // ---------------- phase D: bcna sums start from zero in the segment's
    // first pass and continue from the block; densities add onto the block
    for (int sl = tid; sl < nown * NB; sl += 64 * NT) {
      const int sg = sl / NB, e = sl - sg * NB;
      const int s0 = sSeg[sg] - c0, s1 = sSeg[sg + 1] - c0;
      const int k0 = max(s0, 0), k1 = min(s1, nt);
      if (k0 < k1 && e < sNb[sg]) {
        double *const o = out + sBo[sg] + e;
        double a = (RHO || s0 < 0) ? *o : 0.0;
        const double *row = reinterpret_cast<const double *>(&sm[0]) + k0 * W3_ROW;
        constexpr int TS = sizeof(W3Lds) / sizeof(double);   // rows of the next term
        int k = k0;
        for (; k + 4 <= k1; k += 4, row += 4 * W3_ROW) {
          double x[4][NT], h[4][NT];
#pragma unroll
          for (int u = 0; u < 4; u++)
#pragma unroll
            for (int j = 0; j < NT; j++) {
              x[u][j] = row[u * W3_ROW + j * TS + e];
              h[u][j] = NT > 1 ? row[u * W3_ROW + j * TS + 16] : 1.0;
            }
#pragma unroll
          for (int u = 0; u < 4; u++)
#pragma unroll
            for (int j = 0; j < NT; j++)
              if (h[u][j] != 0.0) a = a + x[u][j];
        }
        for (; k < k1; k++, row += W3_ROW)
#pragma unroll
          for (int j = 0; j < NT; j++)
            if (NT == 1 || row[j * TS + 16] != 0.0) a = a + row[j * TS + e];
        *o = a;
      }
    }
    if (NT > 1) __syncthreads();
    else w3_fence();
  }
  if (status) atomicOr(v.status, status);
}
