// Three-centre Vna forces (Dassemble_vna_3c, k.DASSEMBLERS/
// M_Dassemble_3c_DOGS.f90:136-793) of s/p species with canonical tables.
//
// The reference rotates the derivative of every block element and contracts
// the three derivative blocks with the density block.  The force is a gradient
// of one number per triplet, E = sum rho_ij V_ij, so it is formed the other
// way round: the density block is rotated into the molecular frame once (D),
// E becomes a sum over the table's matrix elements, and the chain rule needs
//   dE/dx, dE/dz, dE/dcos   sums of D times the interpolated derivatives,
//   the torque on the frame  tau = sum eps (D M^T + D^T M), three numbers,
// from which the gradients with respect to the third atom and to the bond
// follow in closed form.  That is some 400 operations per triplet after the
// interpolation, where the derivative blocks take 8,260.  The results agree
// with the reference's to rounding (1e-14 of the largest force).
//
// A wavefront owns a tile of whole target segments: A lane per triplet, B the
// interpolation with a lane per element (four per element of a 16-point cell,
// a column each), C lane per triplet, D the segment sums.  Each triplet leaves
// its force on the third atom (f3a, target order); the forces on iatom and on
// jatom are summed per segment (fseg).  k_d3c_atom then sums f3a per (iatom,
// third atom) pair and fseg over iatom's targets, k_d3c_back the pair sums
// over each atom's neighbours: fixed orders, no atomics, 24 bytes written and
// read per triplet where three sorted record arrays took 72.
//
// Registers for two wavefronts per SIMD (three spill 13 to 133 of them), LDS
// 16 KB.  Bound by the latency of A's and C's dependent binary64 work and of
// the table gathers.  Measured (derivative blocks -> this form, triplets +
// sums): Si of 1728 atoms, 0.85 M triplets, mixed 307 + 18 -> 91 + 34 us;
// charged binary64 droplet of 151 atoms, 67,656 triplets, 317 + 22 -> 68 +
// 23 us.  Error against 80-bit arithmetic (charged C/H/N/O, 60 atoms)
// 4.1e-13 -> 6.7e-15, mixed against binary64 7.3e-8 -> 4.5e-8 eV/A.
#pragma once

#include "fb_3c_wave.h"
#include "fb_forces.h"
#include "fb_lists_dev.h"

#define D3_T 64                 // triplets per pass
#define D3_ROW 41               // LDS row: 10 values, cos, x and y derivatives, odd stride

struct D3Par {
  double px, py, p[4], dp[3];   // P1..P4 and dP2..dP4 (P0 = 1, dP0 = 0, dP1 = 1)
  int64_t base;                 // slab index of (theta 0, ix, iy, ME 0)
  int rs, pad;                  // slab values per iy row
};

union D3Rows {                  // FP32 rows of a whole pass, or binary64 rows of half of it
  float f[D3_T][D3_ROW];
  double d[D3_T / 2][D3_ROW];
};

template <typename T> struct D3Type;
template <> struct D3Type<double> {
  static constexpr int PASS = D3_T / 2;
  static __device__ __forceinline__ double (*rows(D3Rows &r))[D3_ROW] { return r.d; }
};
template <> struct D3Type<float> {
  static constexpr int PASS = D3_T;
  static __device__ __forceinline__ float (*rows(D3Rows &r))[D3_ROW] { return r.f; }
};

__device__ __forceinline__ void load_theta(const float *p, float *t) {
  typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
  const f4u a = *reinterpret_cast<const f4u *>(p);
  t[0] = a[0];
  t[1] = a[1];
  t[2] = a[2];
  t[3] = a[3];
  t[4] = p[4];
}

__device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

template <int CTRL>
__device__ __forceinline__ float dpp_(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp_(double x) {
  int2 v = __builtin_bit_cast(int2, x);
  v.x = __builtin_amdgcn_mov_dpp(v.x, CTRL, 0xf, 0xf, true);
  v.y = __builtin_amdgcn_mov_dpp(v.y, CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(double, v);
}
// sum over the four lanes of a quad, in all of them
template <typename T>
__device__ __forceinline__ T quad_sum(T x) {
  x = x + dpp_<0xb1>(x);        // quad_perm 1 0 3 2
  return x + dpp_<0x4e>(x);     // quad_perm 2 3 0 1
}

// sum_theta P t and sum_theta dP t.  Here and in the weights below the largest
// term is added last and the others as differences to it: in FP32 one rounding
// of the value's size instead of one per term, in the slopes none.
template <typename T>
__device__ __forceinline__ void d3_fold(const T *t, const T *p, const T *dp, T &v, T &d) {
  v = t[0] + fma_(p[0], t[1], fma_(p[1], t[2], fma_(p[2], t[3], p[3] * t[4])));
  d = fma_(dp[2], t[4], fma_(dp[1], t[3], fma_(dp[0], t[2], t[1])));
}

// values and cos derivatives of a list of 3-point cells (their x and y slopes
// are the cell's, phase C)
template <typename T, int NME>
__device__ __forceinline__ void d3_three(const T *tab, const D3Par *par, T (*rows)[D3_ROW], int t0,
                                         const unsigned char *ord, int n, int lane) {
  for (int it = lane; it < n * NME; it += 64) {
    const int k = it / NME, m = it - k * NME, t = ord[k];
    const D3Par &q = par[t];
    const T *e = tab + q.base + m * FB_NTHETA;
    T a[FB_NTHETA], b[FB_NTHETA], c[FB_NTHETA];
    load_theta(e, a);
    load_theta(e + NME * FB_NTHETA, b);
    load_theta(e + q.rs, c);
    const T px = (T)q.px, py = (T)q.py;
    const T p[4] = {(T)q.p[0], (T)q.p[1], (T)q.p[2], (T)q.p[3]}, dp[3] = {(T)q.dp[0], (T)q.dp[1], (T)q.dp[2]};
    T va, vb, vc, da, db, dc;
    d3_fold(a, p, dp, va, da);
    d3_fold(b, p, dp, vb, db);
    d3_fold(c, p, dp, vc, dc);
    rows[t - t0][m] = va + fma_(py, vc - va, px * (vb - va));
    rows[t - t0][10 + m] = da + fma_(py, dc - da, px * (db - da));
  }
}

// 16-point cells: the 4-point cubic (nodes -1, 0, 1, 2) in both directions;
// lane c of a quad folds column ix + c - 1
template <typename T, int NME>
__device__ __forceinline__ void d3_sixteen(const T *tab, const D3Par *par, T (*rows)[D3_ROW], int t0,
                                           const unsigned char *ord, int n, int lane) {
  const int c = lane & 3;
  for (int it = lane >> 2; it < n * NME; it += 16) {
    const int k = it / NME, m = it - k * NME, t = ord[k];
    const D3Par &q = par[t];
    const T *e = tab + q.base + m * FB_NTHETA + (c - 1) * (NME * FB_NTHETA) - q.rs;
    T y[4][FB_NTHETA];
#pragma unroll
    for (int l = 0; l < 4; l++) load_theta(e + l * q.rs, y[l]);
    const T p[4] = {(T)q.p[0], (T)q.p[1], (T)q.p[2], (T)q.p[3]}, dp[3] = {(T)q.dp[0], (T)q.dp[1], (T)q.dp[2]};
    const T s6 = (T)(1.0 / 6.0), h = (T)0.5;
    // of nodes -1, 1 and 2: the weights of the values sum to 1, those of the slopes to 0
    auto weights = [&](T x, T *w, T *d) {
      const T a = x + 1, b = x - 1, z = x - 2, x2 = x * x;
      w[0] = -x * b * z * s6;
      w[1] = -a * x * z * h;
      w[2] = a * x * b * s6;
      d[0] = -(3 * x2 - 6 * x + 2) * s6;
      d[1] = -(3 * x2 - 2 * x - 2) * h;
      d[2] = (3 * x2 - 1) * s6;
    };
    T wx[3], dx[3], wy[3], dy[3];
    weights((T)q.px, wx, dx);
    weights((T)q.py, wy, dy);
    const T w = c == 0 ? wx[0] : (c == 2 ? wx[1] : wx[2]), d = c == 0 ? dx[0] : (c == 2 ? dx[1] : dx[2]);
    T t1, p1, gv = 0, gp = 0, gd = 0;
    d3_fold(y[1], p, dp, t1, p1);
#pragma unroll
    for (int l = 0; l < 3; l++) {
      T tv, tp;
      d3_fold(y[l == 0 ? 0 : l + 1], p, dp, tv, tp);
      gv = fma_(wy[l], tv - t1, gv);
      gp = fma_(wy[l], tp - p1, gp);
      gd = fma_(dy[l], tv - t1, gd);
    }
    gv += t1;
    gp += p1;
    // node 0's column is lane 1's, whose differences are zero
    const T cv = dpp_<0x55>(gv), cp = dpp_<0x55>(gp), cd = dpp_<0x55>(gd), dv = gv - cv;
    const T o0 = cv + quad_sum(w * dv), o1 = cp + quad_sum(w * (gp - cp)), o2 = quad_sum(d * dv),
            o3 = cd + quad_sum(w * (gd - cd));
    rows[t - t0][10 * c + m] = c == 0 ? o0 : (c == 1 ? o1 : (c == 2 ? o2 : o3));
  }
}

// Density block in the molecular frame, R^T rho R (orbitals s, y, z, x; axes
// y', z', x'); rows and columns of absent p shells are zero.
__device__ __forceinline__ void d3_density(const double *rho, int cls, const double *yp, const double *zp,
                                           const double *xp, double D[4][4]) {
  const bool p1 = cls & 2, p2 = cls & 1;
  const int nmu = p1 ? 4 : 1;
#pragma unroll
  for (int k2 = 0; k2 < 4; k2++)
#pragma unroll
    for (int k1 = 0; k1 < 4; k1++) D[k1][k2] = ((p1 || k1 == 0) && (p2 || k2 == 0)) ? rho[k2 * nmu + k1] : 0.0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const double a = D[k][1], b = D[k][2], c = D[k][3];
    D[k][1] = fma_(c, yp[0], fma_(b, yp[2], a * yp[1]));
    D[k][2] = fma_(c, zp[0], fma_(b, zp[2], a * zp[1]));
    D[k][3] = fma_(c, xp[0], fma_(b, xp[2], a * xp[1]));
  }
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const double a = D[1][k], b = D[2][k], c = D[3][k];
    D[1][k] = fma_(c, yp[0], fma_(b, yp[2], a * yp[1]));
    D[2][k] = fma_(c, zp[0], fma_(b, zp[2], a * zp[1]));
    D[3][k] = fma_(c, xp[0], fma_(b, xp[2], a * xp[1]));
  }
}

// the seven numbers of one term of a triplet
struct D3Sums {
  double E, Ex, Ey, Ec, tx, ty, tz;
};

// element m of the sp-sp order from the row of a pair of class cls (0 where
// the pair has none)
template <typename T>
__device__ __forceinline__ double d3_el(const T *row, int cls, int m) {
  if (cls == 3) return row[m];
  const int k = cls == 1 ? (m == 1 ? 1 : (m == 6 ? 2 : 0)) : (cls == 2 ? (m == 2 ? 1 : (m == 7 ? 2 : 0)) : 0);
  return (m == 0 || k > 0) ? (double)row[k] : 0.0;
}

// D: molecular-frame density (0 s, 1 y', 2 z', 3 x'); gx, gy: a 3-point
// cell's slopes times sum P, else the reciprocal grid steps
template <typename T>
__device__ __forceinline__ D3Sums d3_contract(const T *row, int cls, bool m1, const double D[4][4], double cost,
                                              double sint, double gx, double gy, double *M) {
  const double d[10] = {D[0][0], D[0][2], D[2][0], D[1][1], D[2][2], D[3][3], D[0][3], D[3][0], D[3][2], D[2][3]};
  D3Sums r;
  double e0 = 0.0, e1 = 0.0, c0 = 0.0, c1 = 0.0, x0 = 0.0, x1 = 0.0, y0 = 0.0, y1 = 0.0;
#pragma unroll
  for (int m = 0; m < 10; m++) {
    const double F = d3_el(row, cls, m), P = d3_el(row + 10, cls, m);
    M[m] = m < 6 ? F : F * sint;
    (m < 6 ? e0 : e1) = fma_(d[m], F, m < 6 ? e0 : e1);
    (m < 6 ? c0 : c1) = fma_(d[m], P, m < 6 ? c0 : c1);
  }
  if (m1) {
    x0 = ((((d[0] + d[1]) + d[2]) + d[3]) + d[4]) + d[5];
    x1 = ((d[6] + d[7]) + d[8]) + d[9];
    y0 = x0;
    y1 = x1;
  } else {
#pragma unroll
    for (int m = 0; m < 10; m++) {
      const double X = d3_el(row + 20, cls, m), Y = d3_el(row + 30, cls, m);
      (m < 6 ? x0 : x1) = fma_(d[m], X, m < 6 ? x0 : x1);
      (m < 6 ? y0 : y1) = fma_(d[m], Y, m < 6 ? y0 : y1);
    }
  }
  r.E = fma_(sint, e1, e0);
  r.Ex = fma_(sint, x1, x0) * gx;
  r.Ey = fma_(sint, y1, y0) * gy;
  r.Ec = fma_(sint, c1, c0) - cost * e1 / sint;
  // tau_a = sum_nm e_n . (e_a x e_m) W_nm, W = D M^T + D^T M
  r.tx = (D[2][1] + D[1][2]) * (M[3] - M[4]) - D[1][0] * M[2] - D[0][1] * M[1] - D[1][3] * M[9] - D[3][1] * M[8];
  r.ty = (D[3][2] + D[2][3]) * (M[4] - M[5]) + D[3][0] * M[2] + D[0][3] * M[1] - D[2][0] * M[7] - D[0][2] * M[6] +
         (D[3][3] - D[2][2]) * (M[9] + M[8]);
  r.tz = D[1][0] * M[7] + D[0][1] * M[6] + D[1][2] * M[8] + D[2][1] * M[9] + (D[1][3] + D[3][1]) * (M[5] - M[3]);
  return r;
}

// MX: FP32 interpolation of the neutral term (charged shells stay binary64)
template <bool MX, bool CHG>
__global__ __launch_bounds__(64, 2) void k_d3c_wave(DView v, DForce Fo) {
  __shared__ D3Par par[D3_T];
  __shared__ D3Rows rw;
  __shared__ unsigned char ord[D3_T];
  __shared__ int sSeg[D3_T + 1];
  double(*const sOut)[7] = reinterpret_cast<double(*)[7]>(par);   // forces of the pass, once phase B is over
  static_assert(sizeof(par) >= sizeof(double) * 7 * D3_T, "the forces take the place of the parameters");
  const int lane = threadIdx.x;
  const int4 td = v.tiles[0][xcd_tile(blockIdx.x, gridDim.x)];
  const int first = td.x, nown = td.y - td.x + 1, r0 = td.z, r1 = td.w;
  if (nown <= 0) return;
  for (int k = lane; k <= nown; k += 64) sSeg[k] = (int)v.seg_off[first + k];
  int status = 0;
  for (int c0 = r0; c0 < r1; c0 += D3_T) {
    const int nt = min(D3_T, r1 - c0);
    const bool on = lane < nt;
    // ---------------- phase A
    int cls = 0, gid0 = -1, in12 = 0, in3 = 0, ial = 0, cell = 0, pair = 0;
    bool zero = true, fb = false;
    double s[3], h[3], yp[3], z = 1.0, x = 0.0, cost = 0.0, cm = 1.0;   // what phase C needs of the frame
    if (on) {
      const int4 tr = v.trip[c0 + lane];
      const int aux = v.trip_aux[c0 + lane];
      pair = v.trip_pair[c0 + lane];
      gid0 = (aux & 0xffff) == 0xffff ? -1 : (aux & 0xffff);
      ial = tr.x;
      const int in1 = v.imass[tr.y], in2 = v.imass[tr.z];
      in3 = v.imass[tr.x];
      in12 = (in1 - 1) * v.sp.ns + (in2 - 1);
      const bool p1 = v.sp.norb[in1 - 1] == 4, p2 = v.sp.norb[in2 - 1] == 4;
      cls = (p1 ? 2 : 0) + (p2 ? 1 : 0);
      const double *xls = v.xl + (int64_t)(aux >> 16) * FB_NIMG * 3;
      const int ib = tr.w & 0xffff, jb = (tr.w >> 16) & 0xffff;
      double ra[3], a1[3], a2[3], d[3], c[3];
#pragma unroll
      for (int k = 0; k < 3; k++) {
        a1[k] = v.ratom[3 * tr.y + k] + xls[3 * ib + k];
        a2[k] = v.ratom[3 * tr.z + k] + xls[3 * jb + k];
        ra[k] = v.ratom[3 * tr.x + k];
        d[k] = a2[k] - a1[k];
        c[k] = ra[k] - (a1[k] + d[k] / 2.0);
      }
      z = d_distance(a1, a2);
      x = sqrt(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]);
      const double iz = 1.0 / z, ixv = x < 1.0e-5 ? 0.0 : 1.0 / x;
      double cr[3];
      d_cross(d, c, cr);
      cm = d_mag(cr);
      zero = cm < 1.0e-3;
#pragma unroll
      for (int k = 0; k < 3; k++) {
        s[k] = d[k] * iz;
        h[k] = c[k] * ixv;
      }
      cost = s[0] * h[0] + s[1] * h[1] + s[2] * h[2];
      fb = cm * iz * ixv < 1.0e-4;
      if (fb && !zero) Fo.afix[tr.y] = 1;   // k_d3c_fix adds what such a frame contributes
      double ym;
      if (fb) {   // epsilon.f90:148-168
        if (fabs(s[0]) > 1.0e-4) { cr[0] = -(s[1] + s[2]) / s[0]; cr[1] = 1.0; cr[2] = 1.0; }
        else if (fabs(s[1]) > 1.0e-4) { cr[0] = 1.0; cr[1] = -(s[0] + s[2]) / s[1]; cr[2] = 1.0; }
        else { cr[0] = 1.0; cr[1] = 1.0; cr[2] = -(s[0] + s[1]) / s[2]; }
        ym = 1.0 / d_mag(cr);
      } else {
        ym = 1.0 / cm;
      }
#pragma unroll
      for (int k = 0; k < 3; k++) yp[k] = cr[k] * ym;
      if (gid0 < 0) {
        status |= ST_NO_TABLE;
      } else {
        const DGroup3c g = group3c_scalar(v, gid0);
        const int nx = g.nx, ny = g.ny;
        const double dx = g.xmax / (nx - 1.0), dy = g.ymax / (ny - 1.0);
        int ix = (int)(x / dx) + 1, iy = (int)(z / dy) + 1;
        if (ix < 2) ix = 2;
        if (iy < 2) iy = 2;
        if (ix > nx - 2) ix = nx - 2;
        if (iy > ny - 2) iy = ny - 2;
        D3Par &q = par[lane];
        q.px = x / dx - ix + 1.0;
        q.py = z / dy - iy + 1.0;
        const double c2 = cost * cost;
        double p[5], sint;
        d_legendre(cost, p, &sint);
#pragma unroll
        for (int k = 0; k < 4; k++) q.p[k] = p[k + 1];
        q.dp[0] = 3.0 * cost;
        q.dp[1] = (15.0 * c2 - 3.0) / 2.0;
        q.dp[2] = 0.5 * cost * (35.0 * c2 - 15.0);
        q.rs = nx * g.nME * FB_NTHETA;
        cell = (iy - 1) * nx + (ix - 1);
      }
    }
    D3Sums S = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    double Eq = 0.0, Q = 0.0, stinky = 0.0;
    bool charged = false;   // any shell of ialpha: of charges that cancel, E still follows the smoothing
    // ialpha - iatom and ialpha - jatom, and the smoothing of each
    auto arms = [&](double *a, double *b, double &d13, double &d23, double &e1, double &e2) {
#pragma unroll
      for (int k = 0; k < 3; k++) {
        a[k] = fma_(x, h[k], 0.5 * z * s[k]);
        b[k] = fma_(x, h[k], -0.5 * z * s[k]);
      }
      d13 = d_mag(a);
      d23 = d_mag(b);
      const double rc3 = v.sp.rcmin[in3 - 1];
      e1 = v.sp.rcmin[in12 / v.sp.ns] + rc3;
      e2 = v.sp.rcmin[in12 % v.sp.ns] + rc3;
    };
    if (CHG && on) {
      double a[3], b[3], d13, d23, e1, e2;
      arms(a, b, d13, d23, e1, e2);
      stinky = d_smoother(d13, e1, 0.8) * d_smoother(d23, e2, 0.8);
    }
    // ---------------- the terms: neutral, then the charged shells of ialpha
    auto one_term = [&](auto zeroT, int gid, double coef, double dQ) {
      typedef decltype(zeroT) T;
      const bool have = gid >= 0;
      bool m1 = false;
      double gx = 0.0, gy = 0.0;
      if (have) {
        const DGroup3c g = group3c_scalar(v, gid);
        const int nM = g.nME * FB_NTHETA;
        par[lane].base = (sizeof(T) == 4 ? g.off32 : g.off) + (int64_t)cell * nM;
        m1 = v.meth3c[g.moff + cell] != 0;
        if (m1) {
          // the 3-point rule takes the slopes of ME 1 of theta cell 1 (binary64 table) for every element
          const double *t = v.tab3c + g.off + (int64_t)cell * nM;
          const double f = t[0], *p = par[lane].p, ps = (((1.0 + p[0]) + p[1]) + p[2]) + p[3];
          gx = (t[nM] - f) / g.dx * ps;
          gy = (t[g.nx * nM] - f) / g.dy * ps;
        } else {
          gx = 1.0 / g.dx;
          gy = 1.0 / g.dy;
        }
      }
      constexpr int PASS = D3Type<T>::PASS;
      for (int t0 = 0; t0 < nt; t0 += PASS) {
        const bool mine = have && (PASS == D3_T || (lane >= t0 && lane < t0 + PASS));
        int n[6], at = 0;
        const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
        for (int c = 0; c < 3; c++) {
          const bool in = mine && (c == 0 ? cls == 3 : (c == 1 ? cls == 1 || cls == 2 : cls == 0));
#pragma unroll
          for (int hf = 0; hf < 2; hf++) {
            const unsigned long long bl = __ballot(in && m1 == (hf == 0));
            if (in && m1 == (hf == 0)) ord[at + __popcll(bl & below)] = (unsigned char)lane;
            n[2 * c + hf] = __popcll(bl);
            at += __popcll(bl);
          }
        }
        w3_fence();
        T(*const rows)[D3_ROW] = D3Type<T>::rows(rw);
        const T *tab;
        if constexpr (sizeof(T) == 4) tab = v.tab3c32;
        else tab = v.tab3c;
        const unsigned char *o = ord;
        d3_three<T, 10>(tab, par, rows, t0, o, n[0], lane);
        o += n[0];
        d3_sixteen<T, 10>(tab, par, rows, t0, o, n[1], lane);
        o += n[1];
        d3_three<T, 3>(tab, par, rows, t0, o, n[2], lane);
        o += n[2];
        d3_sixteen<T, 3>(tab, par, rows, t0, o, n[3], lane);
        o += n[3];
        d3_three<T, 1>(tab, par, rows, t0, o, n[4], lane);
        o += n[4];
        d3_sixteen<T, 1>(tab, par, rows, t0, o, n[5], lane);
        w3_fence();
        // ---------------- phase C
        if (mine) {
          double M[10], D[4][4], xp[3];
          d_cross(yp, s, xp);
          d3_density(Fo.rho + v.boff[pair], cls, yp, s, xp, D);
          const double sint = sqrt(fmax(1.0e-5, 1.0 - cost * cost));
          const D3Sums r = d3_contract(rows[lane - t0], cls, m1, D, cost, sint, gx, gy, M);
          S.Ex = fma_(coef, r.Ex, S.Ex);
          S.Ey = fma_(coef, r.Ey, S.Ey);
          S.Ec = fma_(coef, r.Ec, S.Ec);
          if (CHG) Eq = fma_(dQ, r.E, Eq);
          if (!zero && !fb) {
            S.tx = fma_(coef, r.tx, S.tx);
            S.ty = fma_(coef, r.ty, S.ty);
            S.tz = fma_(coef, r.tz, S.tz);
          }
        }
        w3_fence();
      }
    };
    if constexpr (MX) one_term(0.0f, on ? gid0 : -1, 1.0, 0.0);
    else one_term(0.0, on ? gid0 : -1, 1.0, 0.0);
    if (CHG) {
      for (int sh = 0; sh < 2; sh++) {
        int gid = -1;
        double dQ = 0.0;
        if (on && sh < v.sp.nssh[in3 - 1]) {
          dQ = v.dQ[ial * FB_MAXSH + sh];
          if (dQ != 0.0) {
            gid = v.idx3c[(in12 * v.sp.ns + (in3 - 1)) * FB_MAXSUB3 + sh + 1];
            if (gid < 0) {
              status |= ST_NO_TABLE;
            } else {
              Q += dQ;
              charged = true;
            }
          }
        }
        if (__ballot(gid >= 0)) one_term(0.0, gid, stinky * dQ, dQ);
      }
    }
    // ---------------- gradients of the triplet
    if (on) {
      double fa[3], fbv[3], xp[3];
      d_cross(yp, s, xp);
      const double iz = 1.0 / z, ixv = x < 1.0e-5 ? 0.0 : 1.0 / x;
      const double ct = zero ? 0.0 : cost * x * z / cm, t3 = zero ? 0.0 : S.tz * z / cm;
      const double t1 = fma_(S.tz, ct, S.tx);
      double dA[3] = {0.0, 0.0, 0.0}, dB[3] = {0.0, 0.0, 0.0}, wA[3] = {0.0, 0.0, 0.0}, wB[3] = {0.0, 0.0, 0.0};
      double dE = 0.0;
      if (CHG && charged) {
        // smoothed monopole: the density contracted with S, dipole_z and their Dblocks per target pair
        double a[3], b[3], d13, d23, e1, e2;
        arms(a, b, d13, d23, e1, e2);
        const double i13 = 1.0 / d13, i23 = 1.0 / d23;
        const double st13 = d_smoother(d13, e1, 0.8), st23 = d_smoother(d23, e2, 0.8);
        const double dst13 = d_Dsmoother(d13, e1, 0.8), dst23 = d_Dsmoother(d23, e2, 0.8);
        const double *pq = Fo.pq + 8 * (int64_t)pair;
        const double st = pq[0] / 2.0, dt = pq[1] * iz, m = st - dt, p = st + dt;
        dE = Eq - Q * (m * i13 + p * i23);
#pragma unroll
        for (int k = 0; k < 3; k++) {
          const double u1 = a[k] * i13, u2 = b[k] * i23, sp = pq[2 + k] / 2.0, dp = fma_(dt, s[k], pq[5 + k]) * iz;
          const double r1_ = m * u1 * i13 * i13;
          dA[k] = -r1_ - p * u2 * i23 * i23;
          dB[k] = r1_ + (sp - dp) * i13 + (sp + dp) * i23;
          wB[k] = -dst13 * st23 * u1;
          wA[k] = fma_(st13 * dst23, u2, -wB[k]);
        }
      }
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const double g_a = fma_(S.Ex, h[k], fma_(S.Ec * ixv, fma_(-cost, h[k], s[k]), t3 * yp[k]));
        const double g_d =
            fma_(S.Ey, s[k], iz * (fma_(S.Ec, fma_(-cost, s[k], h[k]), fma_(S.ty, xp[k], -t1 * yp[k]))));
        // iatom: minus the bond gradient, minus half of the third atom's (the bond centre moves along)
        double g_b = -g_d - 0.5 * g_a;
        double gt = g_a;
        if (CHG) {
          gt = fma_(dE, wA[k], fma_((1.0 - stinky) * Q, dA[k], gt));
          g_b = fma_(dE, wB[k], fma_((1.0 - stinky) * Q, dB[k], g_b));
        }
        fa[k] = -FB_P_EQ2 * gt;
        fbv[k] = -FB_P_EQ2 * g_b;
      }
#pragma unroll
      for (int k = 0; k < 3; k++) {
        Fo.f3a[3 * (int64_t)(c0 + lane) + k] = fa[k];
        sOut[lane][k] = fa[k];
        sOut[lane][3 + k] = fbv[k];
      }
    }
    w3_fence();
    // ---------------- phase D: segment sums; jatom's force by Newton's third law
    for (int sl = lane; sl < nown * 3; sl += 64) {
      const int sg = sl / 3, k3 = sl - 3 * sg;
      const int s0 = sSeg[sg] - c0, k0 = max(s0, 0), k1 = min(sSeg[sg + 1] - c0, nt);
      if (k0 < k1) {
        double *const o = Fo.fseg + 6 * (int64_t)v.seg_pair[first + sg] + k3;
        double A = 0.0, B = 0.0;
#pragma unroll 4
        for (int k = k0; k < k1; k++) {
          A += sOut[k][k3];
          B += sOut[k][3 + k3];
        }
        o[0] = s0 < 0 ? o[0] + B : B;
        o[3] = s0 < 0 ? o[3] - (A + B) : -(A + B);
      }
    }
    w3_fence();
  }
  if (status) atomicOr(v.status, status);
}

// per target pair, the density contracted with S, dipole_z and their Dblocks
// (the monopole part of the charged terms is linear in them)
__global__ __launch_bounds__(256) void k_d3c_pair(DView v, DForce Fo) {
  const int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (p >= v.npairs || !v.pair_tgt[p]) return;
  const int64_t b0 = v.boff[p];
  const int n = (int)(v.boff[p + 1] - b0);
  double r[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  for (int i = 0; i < n; i++) {
    const double rho = Fo.rho[b0 + i];
    r[0] = fma_(rho, v.mat[FB_MAT_S][b0 + i], r[0]);
    r[1] = fma_(rho, v.mat[FB_MAT_DIP][b0 + i], r[1]);
#pragma unroll
    for (int k = 0; k < 3; k++) {
      r[2 + k] = fma_(rho, Fo.dmat[0][3 * (b0 + i) + k], r[2 + k]);
      r[5 + k] = fma_(rho, Fo.dmat[2][3 * (b0 + i) + k], r[5 + k]);
    }
  }
#pragma unroll
  for (int k = 0; k < 8; k++) Fo.pq[8 * p + k] = r[k];
}

// pair (iatom -> ialpha) of every triplet: ialpha at the negated image in iatom's list
__global__ void k_trip_nb(DView v, int *nb) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= v.ntrip) return;
  const int4 tr = v.trip[t];
  int c[3];
  image_coords(tr.w & 0xffff, c);
  const int b = image_of(-c[0], -c[1], -c[2]), j = tr.x - v.st[v.trip_aux[t] >> 16].atom_off + 1;
  int64_t lo = v.noff[tr.y], hi = v.noff[tr.y + 1];
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    const int bm = v.neigh_b[mid];
    if (bm < b || (bm == b && v.neigh_j[mid] < j)) lo = mid + 1;
    else hi = mid;
  }
  nb[t] = (int)lo;
}

// first segment of every atom's targets
__global__ void k_atom_seg(DView v, int *aseg) {
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a > v.natoms) return;
  const int64_t key = v.noff[a];
  int64_t lo = 0, hi = v.nseg;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (v.seg_pair[mid] < key) lo = mid + 1;
    else hi = mid;
  }
  aseg[a] = (int)lo;
}

// Near-collinear triplets whose frame is epsilon's fallback one and to which
// Depsilon_3c still applies (sin < 1e-4 but crossmag >= 1e-3: the atoms are far
// apart): the frame then does not follow the plane of the three atoms, and the
// reference's deps of it (b.FUNCTIONS/Depsilon_3c.f90) are contracted as they
// are with U_axis = sum_n axis_n W_n,axis.  k_d3c_wave leaves these triplets
// without their rotational part and marks their iatom; here it is added to
// f3a and fseg, in triplet order.
__device__ __forceinline__ void d3_fix_triplets(const DView &v, const DForce &Fo, int64_t tl, int64_t tend) {
  const bool own = tl < tend;
  const int64_t t = own ? tl : tend - 1;
  const int4 tr = v.trip[t];
  const int aux = v.trip_aux[t], in1 = v.imass[tr.y], in2 = v.imass[tr.z], in3 = v.imass[tr.x];
  const double *xls = v.xl + (int64_t)(aux >> 16) * FB_NIMG * 3;
  double d[3], a[3], c[3], zp[3], h[3], yp[3], xp[3], cr[3], a1[3], a2[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    a1[k] = v.ratom[3 * tr.y + k] + xls[3 * (tr.w & 0xffff) + k];
    a2[k] = v.ratom[3 * tr.z + k] + xls[3 * ((tr.w >> 16) & 0xffff) + k];
    d[k] = a2[k] - a1[k];
    a[k] = v.ratom[3 * tr.x + k] - a1[k];
    c[k] = v.ratom[3 * tr.x + k] - (a1[k] + d[k] / 2.0);
  }
  const double z = d_distance(a1, a2), x = sqrt(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]);
  const double iz = 1.0 / z, ixv = x < 1.0e-5 ? 0.0 : 1.0 / x;
  d_cross(d, c, cr);
  const double cm = d_mag(cr);
  const bool hit = own && !(cm < 1.0e-3) && cm * iz * ixv < 1.0e-4;
  for (unsigned long long hits = __ballot(hit); hits; hits &= hits - 1) {
    if ((int)(threadIdx.x & 63) != __ffsll((long long)hits) - 1) continue;
    double cost = 0.0, eps[9];
#pragma unroll
    for (int k = 0; k < 3; k++) {
      zp[k] = d[k] * iz;
      h[k] = c[k] * ixv;
    }
#pragma unroll
    for (int k = 0; k < 3; k++) cost += zp[k] * h[k];
    d_epsilon(h, zp, eps);
#pragma unroll
    for (int k = 0; k < 3; k++) {
      xp[k] = eps[k];
      yp[k] = eps[3 + k];
    }
    const int cls = (v.sp.norb[in1 - 1] == 4 ? 2 : 0) + (v.sp.norb[in2 - 1] == 4 ? 1 : 0);
    double D[4][4], F[10], M[10], b[3], p[5], sint;
    d3_density(Fo.rho + v.boff[v.trip_pair[t]], cls, yp, zp, xp, D);
    d_legendre(cost, p, &sint);
#pragma unroll
    for (int k = 0; k < 3; k++) b[k] = a[k] - d[k];
    const double rc3 = v.sp.rcmin[in3 - 1];
    const double stinky =
        d_smoother(d_mag(a), v.sp.rcmin[in1 - 1] + rc3, 0.8) * d_smoother(d_mag(b), v.sp.rcmin[in2 - 1] + rc3, 0.8);
#pragma unroll
    for (int m = 0; m < 10; m++) F[m] = 0.0;
    for (int sh = 0; sh <= v.sp.nssh[in3 - 1]; sh++) {
      const double coef = sh == 0 ? 1.0 : stinky * v.dQ[tr.x * FB_MAXSH + sh - 1];
      const int gid = v.idx3c[(((in1 - 1) * v.sp.ns + (in2 - 1)) * v.sp.ns + (in3 - 1)) * FB_MAXSUB3 + sh];
      if (coef == 0.0 || gid < 0) continue;
      const DGroup3c g = v.grp3c[gid];
      const double dx = g.xmax / (g.nx - 1.0), dy = g.ymax / (g.ny - 1.0);
      const int ix = min(max((int)(x / dx) + 1, 2), g.nx - 2), iy = min(max((int)(z / dy) + 1, 2), g.ny - 2);
      const double px = x / dx - ix + 1.0, py = z / dy - iy + 1.0;
      const bool m1 = v.meth3c[g.moff + (int64_t)(iy - 1) * g.nx + (ix - 1)] != 0;
      auto w4 = [](double q, int k) {
        return k == 0 ? -q * (q - 1) * (q - 2) / 6 : (k == 1 ? (q + 1) * (q - 1) * (q - 2) / 2
               : (k == 2 ? -(q + 1) * q * (q - 2) / 2 : (q + 1) * q * (q - 1) / 6));
      };
#pragma unroll
      for (int m = 0; m < 10; m++) {
        if (m >= g.nME) break;
        for (int e = 0; e < 16; e++) {
          const int i = e & 3, j = e >> 2;
          const double w = m1 ? (i == 1 && j == 1 ? 1.0 - px - py : (i == 2 && j == 1 ? px : (i == 1 && j == 2 ? py : 0.0)))
                              : w4(px, i) * w4(py, j);
          if (w == 0.0) continue;
          double f = 0.0;
#pragma unroll
          for (int th = 0; th < FB_NTHETA; th++) f += p[th] * v.tab3c[g.off + FB_T64(th, ix + i - 1, iy + j - 1, m, g.nx, g.nME)];
          F[m] += coef * w * f;
        }
      }
    }
#pragma unroll
    for (int m = 0; m < 10; m++) M[m] = d3_el(F, cls, m) * (m < 6 ? 1.0 : sint);
    const double m4[4][4] = {{M[0], 0.0, M[1], M[6]}, {0.0, M[3], 0.0, 0.0}, {M[2], 0.0, M[4], M[9]}, {M[7], 0.0, M[8], M[5]}};
    double U[3][3];   // [axis y', z', x'][component]
#pragma unroll
    for (int ax = 0; ax < 3; ax++) {
      double W[3];
#pragma unroll
      for (int n = 0; n < 3; n++) {
        W[n] = 0.0;
#pragma unroll
        for (int j = 0; j < 4; j++) W[n] += D[n + 1][j] * m4[ax + 1][j] + D[j][n + 1] * m4[j][ax + 1];
      }
#pragma unroll
      for (int k = 0; k < 3; k++) U[ax][k] = yp[k] * W[0] + zp[k] * W[1] + xp[k] * W[2];
    }
    const double ad = a[0] * d[0] + a[1] * d[1] + a[2] * d[2], bd = b[0] * d[0] + b[1] * d[1] + b[2] * d[2];
    const double bb = b[0] * b[0] + b[1] * b[1] + b[2] * b[2];
    auto levi = [](int i, int j, int k) { return (double)((i - j) * (j - k) * (k - i)) / 2.0; };
#pragma unroll
    for (int ix = 0; ix < 3; ix++) {
      // gradients of crossmag^2 / 2 with respect to ialpha and to iatom
      const double Va = z * z * a[ix] - ad * d[ix], Vb = bd * b[ix] - bb * d[ix];
      double ya[3], yb[3], zb[3], ga = 0.0, gb = 0.0;
#pragma unroll
      for (int mu = 0; mu < 3; mu++) {
        double sa = 0.0, sb = 0.0;
#pragma unroll
        for (int l = 0; l < 3; l++) {
          sa += levi(ix, mu, l) * d[l];
          sb += levi(ix, mu, l) * b[l];
        }
        ya[mu] = (sa - yp[mu] / cm * Va) / cm;
        yb[mu] = (sb - yp[mu] / cm * Vb) / cm;
        zb[mu] = (zp[mu] * zp[ix] - (mu == ix ? 1.0 : 0.0)) * iz;
      }
#pragma unroll
      for (int mu = 0; mu < 3; mu++) {
        const int u = (mu + 1) % 3, w = (mu + 2) % 3;
        const double xa = ya[u] * zp[w] - ya[w] * zp[u];
        const double xb = yb[u] * zp[w] - yb[w] * zp[u] + yp[u] * zb[w] - yp[w] * zb[u];
        ga += ya[mu] * U[0][mu] + xa * U[2][mu];
        gb += yb[mu] * U[0][mu] + zb[mu] * U[1][mu] + xb * U[2][mu];
      }
      double *fs = Fo.fseg + 6 * (int64_t)v.trip_pair[t] + ix;
      Fo.f3a[3 * (int64_t)t + ix] -= FB_P_EQ2 * ga;
      fs[0] -= FB_P_EQ2 * gb;
      fs[3] += FB_P_EQ2 * (ga + gb);
    }
    __threadfence_block();   // the next one's lane may add to the same segment
  }
}

// A wavefront looks at 64 atoms' marks: nearly always there is nothing to do.
// (Loops unrolled: with its arrays in scratch memory the launch alone took
// 19 us of the sums' time; this one takes under 2 us.)
__global__ __launch_bounds__(64) void k_d3c_fix(DView v, DForce Fo) {
  const int lane = threadIdx.x, a64 = blockIdx.x * 64;
  const bool mark = a64 + lane < v.natoms && Fo.afix[a64 + lane] != 0;
  if (mark) Fo.afix[a64 + lane] = 0;
  for (unsigned long long atoms = __ballot(mark); atoms; atoms &= atoms - 1) {
    const int at = a64 + __ffsll((long long)atoms) - 1;
    const int64_t tend = v.seg_off[Fo.aseg[at + 1]];
    for (int64_t t0 = v.seg_off[Fo.aseg[at]]; t0 < tend; t0 += 64) d3_fix_triplets(v, Fo, t0 + lane, tend);
  }
}


// Per iatom: f3a summed over its targets for every neighbour (fpair), and
// fseg's iatom part over its targets (f3nab).  Wavefronts take the segments in
// turn; within one a neighbour occurs once, so the LDS sums do not collide.
#define D3_NC 128   // neighbours per pass
__global__ __launch_bounds__(256) void k_d3c_atom(DView v, DForce Fo) {
  __shared__ double acc[4][D3_NC][3];
  const int a = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t o = v.noff[a];
  const int n = (int)(v.noff[a + 1] - o);
  const int s0 = Fo.aseg[a], s1 = Fo.aseg[a + 1];
  for (int kc = 0; kc < n; kc += D3_NC) {
    for (int e = tid; e < 4 * D3_NC * 3; e += 256) (&acc[0][0][0])[e] = 0.0;
    __syncthreads();
    // four segments of the wavefront at a time, their loads in flight together
    for (int s = s0 + w; s < s1; s += 16) {
      int64_t t0[4], t1[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const bool in = s + 4 * i < s1;
        t0[i] = in ? v.seg_off[s + 4 * i] + lane : 0;
        t1[i] = in ? v.seg_off[s + 4 * i + 1] : 0;
      }
      while (__ballot(t0[0] < t1[0] || t0[1] < t1[1] || t0[2] < t1[2] || t0[3] < t1[3])) {
        int k[4];
        double f[4][3];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          k[i] = -1;
          if (t0[i] < t1[i]) {
            k[i] = Fo.trip_nb[t0[i]] - (int)o - kc;
#pragma unroll
            for (int q = 0; q < 3; q++) f[i][q] = Fo.f3a[3 * t0[i] + q];
          }
          t0[i] += 64;
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
          if (k[i] >= 0 && k[i] < D3_NC) {
#pragma unroll
            for (int q = 0; q < 3; q++) acc[w][k[i]][q] += f[i][q];
          }
          w3_fence();
        }
      }
    }
    __syncthreads();
    const int m = min(n - kc, D3_NC);
    for (int e = tid; e < m * 3; e += 256) {
      const int k = e / 3, q = e - 3 * k;
      Fo.fpair[3 * (o + kc) + e] = ((acc[0][k][q] + acc[1][k][q]) + acc[2][k][q]) + acc[3][k][q];
    }
    __syncthreads();
  }
  if (w == 0) {
    double f[3] = {0.0, 0.0, 0.0};
    for (int s = s0 + lane; s < s1; s += 64) {
      const double *p = Fo.fseg + 6 * (int64_t)v.seg_pair[s];
#pragma unroll
      for (int q = 0; q < 3; q++) f[q] += p[q];
    }
#pragma unroll
    for (int q = 0; q < 3; q++) {
      const double r = wave_sum(f[q]);
      if (lane == 0) Fo.f3[9 * (int64_t)a + 3 + q] = r;
    }
  }
}

// Per atom, over the pairs that point at it: f3naa from fpair, f3nac from fseg
__global__ __launch_bounds__(64) void k_d3c_back(DView v, DForce Fo) {
  const int a = blockIdx.x, lane = threadIdx.x;
  const int off = v.st[v.atom_struct[a]].atom_off;
  double f[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  for (int64_t p = v.noff[a] + lane; p < v.noff[a + 1]; p += 64) {
    const int64_t b = v.noff[off + v.neigh_j[p] - 1] + v.neigh_back[p] - 1;
    const bool tgt = v.pair_tgt[b] != 0;
#pragma unroll
    for (int q = 0; q < 3; q++) {
      f[q] += Fo.fpair[3 * b + q];
      if (tgt) f[3 + q] += Fo.fseg[6 * b + 3 + q];
    }
  }
#pragma unroll
  for (int q = 0; q < 6; q++) {
    const double r = wave_sum(f[q]);
    if (lane == 0) Fo.f3[9 * (int64_t)a + (q < 3 ? q : 3 + q)] = r;
  }
}
