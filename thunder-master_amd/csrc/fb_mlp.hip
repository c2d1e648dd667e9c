// Learned three-centre surrogate: training data, FP32 training kernels,
// calibration and standalone inference (the in-assembly inference is part of
// the mixed 3c kernel).  No counterpart in the reference.
//
// Training data are generated by the binary64 table path itself: the theta
// cells of getMEs_Fdata_3c (e.FDATA/M_Fdata_3c.f90:356-489) at random (x, y),
// with the reference's method choice (3-point rule where the gradient of ME 1
// of theta cell 1 is below 1e-6, bicubic otherwise).
#include "fb_mlp.h"

#include <algorithm>

// ---------------------------------------------------------------- samples
__device__ inline unsigned long long mlp_mix(unsigned long long z) {
  z += 0x9e3779b97f4a7c15ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

__device__ inline double mlp_u01(unsigned long long seed, long long i, int k) {
  return (double)(mlp_mix(seed ^ mlp_mix((unsigned long long)i * 4ull + (unsigned long long)k)) >> 11) *
         (1.0 / 9007199254740992.0);
}

// theta cells of one group at (x, y), binary64 with the reference's method
// choice and evaluation order (same arithmetic as the binary64 3c kernel)
__device__ inline void mlp_interim(const DView &v, const DGroup3c &g, double x, double y, double out[FB_NTHETA][12],
                                   int *pix, int *piy) {
  const int nME = g.nME, nx = g.nx, ny = g.ny;
  const double dx = g.xmax / (nx - 1.0), dy = g.ymax / (ny - 1.0);
  int ix = (int)(x / dx) + 1, iy = (int)(y / dy) + 1;
  if (ix < 2) ix = 2;
  if (iy < 2) iy = 2;
  if (ix > nx - 2) ix = nx - 2;
  if (iy > ny - 2) iy = ny - 2;
  *pix = ix;
  *piy = iy;
  const double px = x / dx - ix + 1.0, py = y / dy - iy + 1.0;
  const double *tab = v.tab3c + g.off;
#define T3D(th, i, j, m) tab[FB_T64(th, i, j, m, nx, nME)]
  const double gx = (T3D(0, ix + 1, iy, 0) - T3D(0, ix, iy, 0)) / dx;
  const double gy = (T3D(0, ix, iy + 1, 0) - T3D(0, ix, iy, 0)) / dy;
  const double gg = gx * gx + gy * gy;
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
      out[th][m] = interim;
    }
  }
#undef T3D
}

// n samples of group gid: X [n][3] normalised inputs, T [n][64] slot targets
__global__ __launch_bounds__(256) void k_mlp_samples(DView v, int gid, int64_t n, unsigned long long seed, float *X,
                                                     float *T) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const DGroup3c g = v.grp3c[gid];
  const double x = mlp_u01(seed, i, 0) * g.xmax, y = mlp_u01(seed, i, 1) * g.ymax;
  const double cost = 2.0 * mlp_u01(seed, i, 2) - 1.0;
  double it[FB_NTHETA][12];
  int ix, iy;
  mlp_interim(v, g, x, y, it, &ix, &iy);
  X[i * 3 + 0] = (float)(2.0 * x / g.xmax - 1.0);
  X[i * 3 + 1] = (float)(2.0 * y / g.ymax - 1.0);
  X[i * 3 + 2] = (float)cost;
  for (int o = 0; o < MLP_O; o++) {
    int th, m;
    T[i * MLP_O + o] = mlp_slot(o, g.nME, &th, &m) ? (float)it[th][m] : 0.0f;
  }
}

// M[i] = max over valid slots |T[i][o]| (envelope fit data)
__global__ __launch_bounds__(256) void k_mlp_rowmax(int64_t n, const float *T, float *M) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  float m = 0.f;
  for (int o = 0; o < MLP_O; o++) m = fmaxf(m, fabsf(T[i * MLP_O + o]));
  M[i] = m;
}

// T[i][:] /= exp(c - kx x_i - ky y_i), x_i and y_i recovered from the inputs
__global__ __launch_bounds__(256) void k_mlp_unenvelope(int64_t n, const float *X, float *T, float c, float kx,
                                                        float ky, float xh, float yh) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float x = (X[i * 3] + 1.0f) * xh, y = (X[i * 3 + 1] + 1.0f) * yh;
  const float inv = 1.0f / __expf(c - kx * x - ky * y);
  for (int o = 0; o < MLP_O; o++) T[i * MLP_O + o] *= inv;
}

// per-column max |a| over n rows (one workgroup per column, deterministic)
__global__ __launch_bounds__(256) void k_colmaxabs(int64_t n, int ncol, const float *A, float *out) {
  __shared__ float s[256];
  const int c = blockIdx.x;
  float m = 0.f;
  for (int64_t i = threadIdx.x; i < n; i += 256) m = fmaxf(m, fabsf(A[i * ncol + c]));
  s[threadIdx.x] = m;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) s[threadIdx.x] = fmaxf(s[threadIdx.x], s[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) out[c] = s[0];
}

__global__ __launch_bounds__(256) void k_scale_cols(int64_t n, int ncol, float *A, const float *inv) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n * ncol; e += (int64_t)gridDim.x * blockDim.x)
    A[e] *= inv[e % ncol];
}

// ---------------------------------------------------------------- FP32 training pass
// Forward and backward of one batch.  A workgroup takes tiles of 16 rows
// through the whole network: both 64 x 64 weight matrices and the rows'
// activations stay in LDS, every product runs on v_mfma_f32_16x16x4_f32
// (FP32 operands and sums), and the weight gradients of its tiles add up in
// accumulator registers.  It writes one partial gradient; k_mlp_sum adds the
// partials in workgroup order, so the result is the same run to run.
//
// The work is 105 MFLOP for 2048 rows: the bound is the chain of launches and,
// within them, of LDS round trips.  As 24 launches (one per product, bias,
// activation and split sum) the pass took 82 us with passes in flight and
// 241 us alone; as these two it takes 7.4 us and 25 us.  Tiles of 16 rows, the
// smallest of the instruction, give 2048 rows 128 workgroups.
//
// Lane layout (l = lane, r = l % 16, g = l / 16, wave w): a wavefront owns
// units 16w .. 16w + 15 of every layer.  An accumulator holds rows 4g + j of
// unit 16w + r; as the A operand of a weight gradient the same registers are
// (unit r, row index g), so the row gradients feed it in place.  A contraction
// index is free, so step j of a group of four takes k = 4g + j of 16: one
// 16-byte LDS read feeds four instructions.
#define MLP_ROWS 16
#define MLP_LD 68   // LDS row of 64 units: 16-byte reads stay aligned, columns do not share banks

typedef float mlp_v4 __attribute__((ext_vector_type(4)));

// c += A[16 rows][64] (rows of s) times the 64 x 16 operand whose element
// (k, unit r) is b(k)
template <typename B>
__device__ __forceinline__ mlp_v4 mlp_rows64(const float (*s)[MLP_LD], int r, int g, B b) {
  mlp_v4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const mlp_v4 a = *reinterpret_cast<const mlp_v4 *>(&s[r][16 * q + 4 * g]);
    const mlp_v4 x = b(16 * q + 4 * g);
#pragma unroll
    for (int j = 0; j < 4; j++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], x[j], c, 0, 0, 0);
  }
  return c;
}

__global__ __launch_bounds__(256) void k_mlp_pass(int64_t n, int nme, const float *P, const float *X, const float *T,
                                                  float inv_count, float *part, float *rowloss) {
  __shared__ __align__(16) float sW2[MLP_H][MLP_LD], sW3[MLP_O][MLP_LD];
  __shared__ __align__(16) float sA1[MLP_ROWS][MLP_LD], sA2[MLP_ROWS][MLP_LD], sD[MLP_ROWS][MLP_LD];
  __shared__ float sX[MLP_ROWS][4], sL[4][MLP_ROWS];
  const int tid = threadIdx.x, l = tid & 63, w = tid >> 6, r = l & 15, g = l >> 4;
  const int u = 16 * w + r;   // this lane's unit
  for (int e = tid; e < MLP_H * MLP_H; e += 256) {
    sW2[e >> 6][e & 63] = P[MLP_P_W2 + e];
    sW3[e >> 6][e & 63] = P[MLP_P_W3 + e];
  }
  const float w1[3] = {P[MLP_P_W1 + 3 * u], P[MLP_P_W1 + 3 * u + 1], P[MLP_P_W1 + 3 * u + 2]};
  const float b1 = P[MLP_P_B1 + u], b2 = P[MLP_P_B2 + u], b3 = P[MLP_P_B3 + u];
  int th, me;
  const bool valid = mlp_slot(u, nme, &th, &me);
  mlp_v4 g3[4] = {}, g2[4] = {};
  float gb1 = 0.f, gb2 = 0.f, gb3 = 0.f, g1[3] = {0.f, 0.f, 0.f};
  const int64_t ntile = (n + MLP_ROWS - 1) / MLP_ROWS;
  for (int64_t tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
    const int64_t row0 = tile * MLP_ROWS;
    __syncthreads();   // the previous tile's reads
    if (tid < 3 * MLP_ROWS) sX[tid / 3][tid % 3] = row0 + tid / 3 < n ? X[row0 * MLP_IN + tid] : 0.f;
    float t[4];
#pragma unroll
    for (int j = 0; j < 4; j++) t[j] = row0 + 4 * g + j < n ? T[(row0 + 4 * g + j) * MLP_O + u] : 0.f;
    __syncthreads();
    mlp_v4 z1, z2, d, c;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const float *x = sX[4 * g + j];
      z1[j] = __builtin_fmaf(x[2], w1[2], __builtin_fmaf(x[1], w1[1], x[0] * w1[0])) + b1;
      sA1[4 * g + j][u] = mlp_act(z1[j]);
    }
    __syncthreads();
    z2 = mlp_rows64(sA1, r, g, [&](int k) { return *reinterpret_cast<const mlp_v4 *>(&sW2[u][k]); });
#pragma unroll
    for (int j = 0; j < 4; j++) {
      z2[j] += b2;
      sA2[4 * g + j][u] = mlp_act(z2[j]);
    }
    __syncthreads();
    c = mlp_rows64(sA2, r, g, [&](int k) { return *reinterpret_cast<const mlp_v4 *>(&sW3[u][k]); });
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const float e = (valid && row0 + 4 * g + j < n) ? c[j] + b3 - t[j] : 0.f;
      d[j] = 2.0f * e * inv_count;
      sD[4 * g + j][u] = d[j];
      float s = e * e;
#pragma unroll
      for (int x = 1; x < 16; x <<= 1) s += __shfl_xor(s, x);
      if (r == 0) sL[w][4 * g + j] = s;
    }
    __syncthreads();
    if (tid < MLP_ROWS && row0 + tid < n) rowloss[row0 + tid] = ((sL[0][tid] + sL[1][tid]) + sL[2][tid]) + sL[3][tid];
    // output layer
#pragma unroll
    for (int j = 0; j < 4; j++) {
      gb3 += d[j];
#pragma unroll
      for (int q = 0; q < 4; q++)
        g3[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(d[j], sA2[4 * g + j][16 * q + r], g3[q], 0, 0, 0);
    }
    c = mlp_rows64(sD, r, g, [&](int k) { return mlp_v4{sW3[k][u], sW3[k + 1][u], sW3[k + 2][u], sW3[k + 3][u]}; });
#pragma unroll
    for (int j = 0; j < 4; j++) d[j] = c[j] * mlp_dact(z2[j]);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; j++) sD[4 * g + j][u] = d[j];
    __syncthreads();
    // second layer
#pragma unroll
    for (int j = 0; j < 4; j++) {
      gb2 += d[j];
#pragma unroll
      for (int q = 0; q < 4; q++)
        g2[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(d[j], sA1[4 * g + j][16 * q + r], g2[q], 0, 0, 0);
    }
    c = mlp_rows64(sD, r, g, [&](int k) { return mlp_v4{sW2[k][u], sW2[k + 1][u], sW2[k + 2][u], sW2[k + 3][u]}; });
    // first layer
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const float e = c[j] * mlp_dact(z1[j]);
      gb1 += e;
#pragma unroll
      for (int k = 0; k < 3; k++) g1[k] = __builtin_fmaf(e, sX[4 * g + j][k], g1[k]);
    }
  }
  float *out = part + (int64_t)blockIdx.x * MLP_NP;
#pragma unroll
  for (int q = 0; q < 4; q++)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      out[MLP_P_W3 + (16 * w + 4 * g + j) * MLP_H + 16 * q + r] = g3[q][j];
      out[MLP_P_W2 + (16 * w + 4 * g + j) * MLP_H + 16 * q + r] = g2[q][j];
    }
  // the row groups g of a unit
  auto rows = [&](float x) {
    x += __shfl_xor(x, 16);
    return x + __shfl_xor(x, 32);
  };
  gb1 = rows(gb1);
  gb2 = rows(gb2);
  gb3 = rows(gb3);
#pragma unroll
  for (int k = 0; k < 3; k++) g1[k] = rows(g1[k]);
  if (g == 0) {
    out[MLP_P_B1 + u] = gb1;
    out[MLP_P_B2 + u] = gb2;
    out[MLP_P_B3 + u] = gb3;
#pragma unroll
    for (int k = 0; k < 3; k++) out[MLP_P_W1 + 3 * u + k] = g1[k];
  }
}

// grads[e] = sum over the partial gradients (four ranges of them side by
// side, added in order); the last workgroup, when asked, the mean batch loss
// from the row losses (lane-strided sums, then a fixed tree)
__global__ __launch_bounds__(256) void k_mlp_sum(int npart, const float *part, float *grads, int64_t n,
                                                 const float *rowloss, float scale, float *loss) {
  __shared__ float s[256];
  const int tid = threadIdx.x;
  if (blockIdx.x == MLP_NP / 64) {
    float a = 0.f;
    for (int64_t i = tid; i < n; i += 256) a += rowloss[i];
    s[tid] = a;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
      if (tid < h) s[tid] += s[tid + h];
      __syncthreads();
    }
    if (tid == 0) loss[0] = s[0] * scale;
    return;
  }
  const int e = blockIdx.x * 64 + (tid & 63), q = tid >> 6, per = (npart + 3) / 4;
  const int z1 = min(npart, (q + 1) * per);
  float a = 0.f;
#pragma unroll 8
  for (int z = q * per; z < z1; z++) a += part[(int64_t)z * MLP_NP + e];
  s[tid] = a;
  __syncthreads();
  if (q == 0) grads[e] = ((s[tid] + s[64 + tid]) + s[128 + tid]) + s[192 + tid];
}
static_assert(MLP_NP % 64 == 0, "k_mlp_sum covers the gradient in whole workgroups");

// ---------------------------------------------------------------- elementwise
// Adam (bias-corrected), lr given per step by the host schedule
__global__ __launch_bounds__(256) void k_mlp_adam(int np, float *p, const float *g, float *m, float *v, float lr,
                                                  float b1, float b2, float c1, float c2, float eps) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= np) return;
  const float gi = g[e];
  const float mi = b1 * m[e] + (1.0f - b1) * gi;
  const float vi = b2 * v[e] + (1.0f - b2) * gi * gi;
  m[e] = mi;
  v[e] = vi;
  p[e] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
}

// ---------------------------------------------------------------- inference
// Standalone BF16/MFMA evaluation of a network on n normalised inputs (the
// arithmetic of the 3c kernel's network phase): Y [n][64] = outputs x envelope
// (the slot scale is folded into the last layer).  One wavefront per 16
// samples.
__global__ __launch_bounds__(256) void k_mlp_infer(const DMlp *w, int64_t n, const float *X, float *Y) {
  const int64_t wave = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6;
  const int l = threadIdx.x & 63, q = l >> 4;
  const int64_t i = wave * 16 + (l & 15);
  const bool ok = i < n;
  float out[16];
  mlp_eval16(&w->w, ok ? X[i * 3] : 0.f, ok ? X[i * 3 + 1] : 0.f, ok ? X[i * 3 + 2] : 0.f, out);
  if (!ok) return;
  const float env = mlp_envelope(w, (X[i * 3] + 1.0f) * 0.5f * w->xmax, (X[i * 3 + 1] + 1.0f) * 0.5f * w->ymax);
#pragma unroll
  for (int r = 0; r < 16; r++) {
    const int o = 16 * (r >> 2) + 4 * q + (r & 3);
    Y[i * MLP_O + o] = out[r] * env;
  }
}

// Calibration: for each sub-cell of the calibration grid (MLP_CSUB x MLP_CSUB
// per table cell), the largest Frobenius norm of the molecular-frame block
// error |M_network - M_table|_F (theta cells folded with P(cos), sin(theta)
// on mvalue = 1 elements) over n uniform samples (x, y, cos).  Orthogonal
// rotations keep the Frobenius norm, which bounds every element of the
// rotated block.  err holds float bits (non-negative, so integer max is float
// max).
__global__ __launch_bounds__(256) void k_mlp_calib(DView v, int gid, const DMlp *w, int64_t n,
                                                   unsigned long long seed, unsigned *err) {
  const int64_t wave = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6;
  const int l = threadIdx.x & 63, q = l >> 4;
  const int64_t i = wave * 16 + (l & 15);
  const bool ok = i < n;
  const DGroup3c g = v.grp3c[gid];
  const double x = mlp_u01(seed, i, 0) * g.xmax, y = mlp_u01(seed, i, 1) * g.ymax;
  const double cost = 2.0 * mlp_u01(seed, i, 2) - 1.0;
  float out[16];
  mlp_eval16(&w->w, (float)(2.0 * x / g.xmax - 1.0), (float)(2.0 * y / g.ymax - 1.0), (float)cost, out);
  double it[FB_NTHETA][12];
  int ix = 2, iy = 2;
  double e2 = 0.0;
  if (ok) {
    mlp_interim(v, g, x, y, it, &ix, &iy);
    const float env = mlp_envelope(w, (float)x, (float)y);
    const double c2 = cost * cost;
    const double P[5] = {1.0, cost, 0.5 * (3.0 * c2 - 1.0), 0.5 * cost * (5.0 * c2 - 3.0),
                         0.125 * (3.0 - c2 * (30.0 - 35.0 * c2))};
    const double sint = sqrt(fmax(1.0e-5, 1.0 - c2));
    for (int ml = 0; ml < 3; ml++) {
      const int m = q + 4 * ml;
      if (m >= g.nME) break;
      double d = 0.0;
      for (int th = 0; th < 5; th++) d += P[th] * ((double)(out[ml * 5 + th] * env) - it[th][m]);
      if (v.mv[g.munu + m] == 1) d *= sint;
      e2 += d * d;
    }
  }
  // the four lane groups of one sample hold disjoint matrix elements
  e2 += __shfl_xor(e2, 16);
  e2 += __shfl_xor(e2, 32);
  if (!ok || q != 0) return;
  atomicMax(&err[mlp_subcell(x, y, g.xmax, g.ymax, g.nx, g.ny)], __float_as_uint((float)sqrt(e2)));
}

// ---------------------------------------------------------------- launchers
extern "C" {

// gradients of one batch into grads (part: MLP_PARTS partial gradients), the
// rows' squared errors into rowloss and, unless null, their mean into loss
int fbk_mlp_pass(int64_t n, int nme, float inv_count, const float *P, const float *X, const float *T, float *part,
                 float *rowloss, float *grads, float loss_scale, float *loss, hipStream_t st) {
  const int npart = (int)std::min<int64_t>((n + MLP_ROWS - 1) / MLP_ROWS, MLP_PARTS);
  hipLaunchKernelGGL(k_mlp_pass, dim3(npart), dim3(256), 0, st, n, nme, P, X, T, inv_count, part, rowloss);
  hipLaunchKernelGGL(k_mlp_sum, dim3(MLP_NP / 64 + (loss ? 1 : 0)), dim3(256), 0, st, npart, part, grads, n, rowloss,
                     loss_scale, loss);
  return (int)hipGetLastError();
}

int fbk_mlp_samples(const DView &v, int gid, int64_t n, unsigned long long seed, float *X, float *T, hipStream_t st) {
  hipLaunchKernelGGL(k_mlp_samples, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, v, gid, n, seed, X, T);
  return (int)hipGetLastError();
}

int fbk_mlp_rowmax(int64_t n, const float *T, float *M, hipStream_t st) {
  hipLaunchKernelGGL(k_mlp_rowmax, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, T, M);
  return (int)hipGetLastError();
}

int fbk_mlp_unenvelope(int64_t n, const float *X, float *T, float c, float kx, float ky, float xh, float yh,
                       hipStream_t st) {
  hipLaunchKernelGGL(k_mlp_unenvelope, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, X, T, c, kx, ky, xh,
                     yh);
  return (int)hipGetLastError();
}

int fbk_mlp_colmaxabs(int64_t n, int ncol, const float *A, float *out, hipStream_t st) {
  hipLaunchKernelGGL(k_colmaxabs, dim3(ncol), dim3(256), 0, st, n, ncol, A, out);
  return (int)hipGetLastError();
}

int fbk_mlp_scale_cols(int64_t n, int ncol, float *A, const float *inv, hipStream_t st) {
  hipLaunchKernelGGL(k_scale_cols, dim3(4096), dim3(256), 0, st, n, ncol, A, inv);
  return (int)hipGetLastError();
}

int fbk_mlp_adam(int np, float *p, const float *g, float *m, float *v, float lr, float b1, float b2, float c1,
                 float c2, float eps, hipStream_t st) {
  hipLaunchKernelGGL(k_mlp_adam, dim3((unsigned)((np + 255) / 256)), dim3(256), 0, st, np, p, g, m, v, lr, b1, b2,
                     c1, c2, eps);
  return (int)hipGetLastError();
}

int fbk_mlp_infer(const DMlp *w, int64_t n, const float *X, float *Y, hipStream_t st) {
  const int64_t waves = (n + 15) / 16;
  hipLaunchKernelGGL(k_mlp_infer, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, st, w, n, X, Y);
  return (int)hipGetLastError();
}

int fbk_mlp_calib(const DView &v, int gid, const DMlp *w, int64_t n, unsigned long long seed, unsigned *err,
                  hipStream_t st) {
  const int64_t waves = (n + 15) / 16;
  hipLaunchKernelGGL(k_mlp_calib, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, st, v, gid, w, n, seed, err);
  return (int)hipGetLastError();
}

}  // extern "C"
