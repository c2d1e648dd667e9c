// Binary64 three-centre interpolation shared by the 3c assemblers:
// getMEs_Fdata_3c (e.FDATA/M_Fdata_3c.f90:293-517) evaluated literally, and the
// segment ownership of a workgroup over triplets sorted by target block.
#pragma once

#include "fb_device.h"

// Legendre P0..P4 and sin(theta) (M_Fdata_3c.f90:347-354)
__device__ __forceinline__ void d_legendre(double cost, double *p, double *sint) {
  double cost2 = cost * cost;
  *sint = sqrt(fmax(1.0e-5, 1.0 - cost2));
  p[0] = 1.0;
  p[1] = cost;
  p[2] = 0.5 * (3.0 * cost2 - 1.0);
  p[3] = 0.5 * cost * (5.0 * cost2 - 3.0);
  p[4] = 0.125 * (3.0 - cost2 * (30.0 - 35.0 * cost2));
}

// getMEs_Fdata_3c in binary64 with the reference's method selection and
// evaluation order; writes the recovered molecular-frame block hm (nmu x nnu).
template <int NMAX>
__device__ inline int d_getMEs_3c(const DView &v, int gid, double x, double y, double cost, int nmu, int nnu,
                                  double *hm) {
  if (gid < 0) return ST_NO_TABLE;
  const DGroup3c g = v.grp3c[gid];
  const int nME = g.nME, nx = g.nx, ny = g.ny;
  if (nME > NMAX) return ST_CAPACITY;
  double p[5], sint;
  d_legendre(cost, p, &sint);
  const double dx = g.xmax / (nx - 1.0), dy = g.ymax / (ny - 1.0);
  int ix = (int)(x / dx) + 1, iy = (int)(y / dy) + 1;
  if (ix < 2) ix = 2;
  if (iy < 2) iy = 2;
  if (ix > nx - 2) ix = nx - 2;
  if (iy > ny - 2) iy = ny - 2;
  const double px = x / dx - ix + 1.0, py = y / dy - iy + 1.0;
  const double *tab = v.tab3c + g.off;
#define T3D(th, i, j, m) tab[FB_T64(th, i, j, m, nx, nME)]
  const double gx = (T3D(0, ix + 1, iy, 0) - T3D(0, ix, iy, 0)) / dx;
  const double gy = (T3D(0, ix, iy + 1, 0) - T3D(0, ix, iy, 0)) / dy;
  const double gg = gx * gx + gy * gy;
  double F[NMAX];
  for (int m = 0; m < nME; m++) F[m] = 0.0;
  for (int th = 0; th < FB_NTHETA; th++) {
    for (int m = 0; m < nME; m++) {
      double interim;
      if (gg < 1.0e-6) {
        interim = ((1.0 - px - py) * T3D(th, ix, iy, m) + px * T3D(th, ix + 1, iy, m)) + py * T3D(th, ix, iy + 1, m);
      } else {
        double gk[4];
        for (int k = -1; k <= 2; k++) {
          double f1m1 = T3D(th, ix + k, iy - 1, m);
          double f1m2 = 2.0 * f1m1, f1m3 = 3.0 * f1m1;
          double f0p3 = 3.0 * T3D(th, ix + k, iy, m), f0p6 = 2.0 * f0p3;
          double f1p3 = 3.0 * T3D(th, ix + k, iy + 1, m), f1p6 = 2.0 * f1p3;
          double f2p1 = T3D(th, ix + k, iy + 2, m);
          double bb3 = -f1m1 + f0p3 - f1p3 + f2p1;
          double bb2 = f1m3 - f0p6 + f1p3;
          double bb1 = -f1m2 - f0p3 + f1p6 - f2p1;
          double bb0 = f0p6;
          gk[k + 1] = ((bb3 * py + bb2) * py + bb1) * py + bb0;
        }
        double f1m1 = gk[0], f1m2 = 2.0 * f1m1, f1m3 = 3.0 * f1m1;
        double f0p3 = 3.0 * gk[1], f0p6 = 2.0 * f0p3;
        double f1p3 = 3.0 * gk[2], f1p6 = 2.0 * f1p3;
        double f2p1 = gk[3];
        double bb3 = -f1m1 + f0p3 - f1p3 + f2p1;
        double bb2 = f1m3 - f0p6 + f1p3;
        double bb1 = -f1m2 - f0p3 + f1p6 - f2p1;
        double bb0 = f0p6;
        interim = (((bb3 * px + bb2) * px + bb1) * px + bb0) / 36.0;
      }
      F[m] = F[m] + p[th] * interim;
    }
  }
#undef T3D
  for (int i = 0; i < nmu * nnu; i++) hm[i] = 0.0;
  for (int k = 0; k < nME; k++) {
    double val = (v.mv[g.munu + k] != 1) ? F[k] : F[k] * sint;
    hm[(v.nu[g.munu + k] - 1) * nmu + (v.mu[g.munu + k] - 1)] = val;
  }
  return 0;
}

// triplet geometry, M_assemble_3c_DOGS.f90:175-271
struct Geo3 {
  double x, z, cost, d13, d23, stinky;
  double eps[9];
  int in1, in2, indna, nmu, nnu;
};

// aux: the triplet's trip_aux word (neutral group | structure << 16)
__device__ inline void d_geo3(const DView &v, int4 tr, int aux, Geo3 &G) {
  const int ial = tr.x, gia = tr.y, gja = tr.z;
  const int ib = tr.w & 0xffff, jb = (tr.w >> 16) & 0xffff;
  const int s = aux >> 16;
  const double *xls = v.xl + (int64_t)s * FB_NIMG * 3;
  double r1[3], r2[3], rna[3], r21[3], sighat[3], rnabc[3], rhat[3];
  for (int k = 0; k < 3; k++) {
    r1[k] = v.ratom[3 * gia + k] + xls[3 * ib + k];
    r2[k] = v.ratom[3 * gja + k] + xls[3 * jb + k];
    rna[k] = v.ratom[3 * ial + k];
    r21[k] = r2[k] - r1[k];
  }
  G.in1 = v.imass[gia];
  G.in2 = v.imass[gja];
  G.indna = v.imass[ial];
  G.nmu = v.sp.norb[G.in1 - 1];
  G.nnu = v.sp.norb[G.in2 - 1];
  G.z = d_distance(r1, r2);
  if (G.z < 1.0e-5) { sighat[0] = 0.0; sighat[1] = 0.0; sighat[2] = 1.0; }
  else for (int k = 0; k < 3; k++) sighat[k] = r21[k] / G.z;
  for (int k = 0; k < 3; k++) rnabc[k] = rna[k] - (r1[k] + r21[k] / 2.0);
  G.x = sqrt(rnabc[0] * rnabc[0] + rnabc[1] * rnabc[1] + rnabc[2] * rnabc[2]);
  G.d13 = d_distance(rna, r1);
  G.d23 = d_distance(rna, r2);
  if (G.x < 1.0e-5) { rhat[0] = 0.0; rhat[1] = 0.0; rhat[2] = 0.0; }
  else for (int k = 0; k < 3; k++) rhat[k] = rnabc[k] / G.x;
  G.cost = sighat[0] * rhat[0] + sighat[1] * rhat[1] + sighat[2] * rhat[2];
  d_epsilon(rhat, sighat, G.eps);
  double rc1 = v.sp.rcmin[G.in1 - 1], rc2 = v.sp.rcmin[G.in2 - 1], rc3 = v.sp.rcmin[G.indna - 1];
  G.stinky = d_smoother(G.d13, rc1 + rc3, 0.8);
  G.stinky = G.stinky * d_smoother(G.d23, rc2 + rc3, 0.8);
}

// the five theta values of one (point, ME)
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));
__device__ __forceinline__ void load_theta(const double *p, double *t) {
  const d2u a = *reinterpret_cast<const d2u *>(p), b = *reinterpret_cast<const d2u *>(p + 2);
  t[0] = a[0];
  t[1] = a[1];
  t[2] = b[0];
  t[3] = b[1];
  t[4] = p[4];
}

// segment range owned by the workgroup of tile [ts, te)
__device__ __forceinline__ bool tile_segments(const DView &v, int64_t ts, int64_t te, int64_t &first, int64_t &last,
                                              int64_t &r0, int64_t &r1) {
  int64_t sgs = v.trip_seg[ts];
  first = (v.seg_off[sgs] == ts) ? sgs : sgs + 1;
  last = v.trip_seg[te - 1];
  if (first > last) return false;
  r0 = v.seg_off[first];
  r1 = v.seg_off[last + 1];
  return true;
}
