// Three-centre neutral-atom (bcna) assembly, j.ASSEMBLERS/M_assemble_3c_DOGS.f90:86-340.
//
// Triplets arrive sorted by their target block (iatom, mneigh), stably, so a
// segment of consecutive triplets holds every contribution to one block in the
// reference's accumulation order (ialpha ascending, then the common-pair
// order).  A workgroup owns the segments that start inside its tile of
// consecutive triplets: it computes the contributions of their triplets in
// chunks, and one thread per segment adds them in order and stores the block
// once.  No atomics; results are deterministic.  A triplet contributes one
// term (neutral) or, with shell charges on its third atom, one more term per
// charged shell; the reference adds each term to the block on its own
// (M_assemble_3c_DOGS.f90:298-318), so the terms are kept apart and the
// segment owner adds them one by one in that order.
//
// k_3c_fp64 is the plain binary64 kernel: one thread per triplet evaluates the
// reference's interpolation (e.FDATA/M_Fdata_3c.f90:293-517) literally.
#include "fb_device.h"
#include "fb_3c_dev.h"

__device__ __forceinline__ int group3c_id(const DView &v, int in1, int in2, int in3, int isub) {
  return v.idx3c[(((in1 - 1) * v.sp.ns + (in2 - 1)) * v.sp.ns + (in3 - 1)) * FB_MAXSUB3 + isub];
}

// terms per triplet: the neutral one plus one per charged shell of the third atom
#define KT_GEN (1 + FB_MAXSH)

// the generic kernel's sizes: s/p species (MO 4), or with d shells (MO 9)
template <int MO> struct Gen3c;
template <> struct Gen3c<FB_MO> {
  static constexpr int T = 64;     // triplets per tile (the LDS holds KT_GEN terms of each)
  static constexpr int NME = 10;   // non-zero bcna matrix elements
};
template <> struct Gen3c<FB_MOD> {
  static constexpr int T = 16;
  static constexpr int NME = FB_NME3_WIDE;
};

template <int MO>
__global__ __launch_bounds__(Gen3c<MO>::T) void k_3c_fp64(DView v) {
  constexpr int T3G = Gen3c<MO>::T, NBG = MO * MO;
  __shared__ double s_c[T3G][KT_GEN][NBG + 1];
  __shared__ int s_n[T3G];
  const int64_t ts = xcd_tile(blockIdx.x, gridDim.x) * T3G;
  const int64_t te = min(ts + T3G, v.ntrip);
  int64_t first, last, r0, r1;
  if (!tile_segments(v, ts, te, first, last, r0, r1)) return;
  const int64_t my = first + threadIdx.x;
  const bool own = my <= last;
  int64_t a = 0, b = 0;
  if (own) { a = v.seg_off[my]; b = v.seg_off[my + 1]; }
  double acc[NBG];
  for (int i = 0; i < NBG; i++) acc[i] = 0.0;
  int status = 0;
  for (int64_t c0 = r0; c0 < r1; c0 += T3G) {
    const int64_t t = c0 + threadIdx.x;
    int nt = 0;
    if (t < r1) {
      const int4 tr = v.trip[t];
      Geo3 G;
      d_geo3(v, tr, v.trip_aux[t], G);
      double pm[9], dm[MO == FB_MOD ? 25 : 1], hm[NBG], bx[NBG];
      d_pmat<double>(G.eps, pm);
      if (MO == FB_MOD) d_dmat(G.eps, dm);
      const int nb = G.nmu * G.nnu;
      int gid = group3c_id(v, G.in1, G.in2, G.indna, 0);
      status |= d_getMEs_3c<Gen3c<MO>::NME>(v, gid, G.x, G.z, G.cost, G.nmu, G.nnu, hm);
      d_rotate<double>(v.sp, G.in1, G.in2, pm, hm, G.nmu, bx, dm);
      for (int i = 0; i < nb; i++) s_c[threadIdx.x][0][i] = bx[i] * FB_P_EQ2;
      nt = 1;
      bool charged = false;
      for (int isorp = 1; isorp <= v.sp.nssh[G.indna - 1]; isorp++)
        charged |= (v.dQ[tr.x * FB_MAXSH + isorp - 1] != 0.0);
      if (charged) {
        const int p = v.trip_pair[t];
        const double *sb = v.mat[FB_MAT_S] + v.boff[p];
        const double *db = v.mat[FB_MAT_DIP] + v.boff[p];
        for (int isorp = 1; isorp <= v.sp.nssh[G.indna - 1]; isorp++) {
          double dQ = v.dQ[tr.x * FB_MAXSH + isorp - 1];
          if (dQ == 0.0) continue;   // the reference adds an exact zero here
          gid = group3c_id(v, G.in1, G.in2, G.indna, isorp);
          status |= d_getMEs_3c<Gen3c<MO>::NME>(v, gid, G.x, G.z, G.cost, G.nmu, G.nnu, hm);
          d_rotate<double>(v.sp, G.in1, G.in2, pm, hm, G.nmu, bx, dm);
          for (int i = 0; i < nb; i++) {
            double sterm = sb[i] / 2.0, dterm = db[i] / G.z;
            double emnpl = (sterm - dterm) / G.d13 + (sterm + dterm) / G.d23;
            s_c[threadIdx.x][nt][i] = dQ * (G.stinky * bx[i] + (1.0 - G.stinky) * emnpl) * FB_P_EQ2;
          }
          nt++;
        }
      }
    }
    s_n[threadIdx.x] = nt;
    __syncthreads();
    if (own) {
      int64_t k0 = max(a, c0), k1 = min(b, c0 + T3G);
      for (int64_t k = k0; k < k1; k++)
        for (int j = 0; j < s_n[k - c0]; j++)
          for (int i = 0; i < NBG; i++) acc[i] = acc[i] + s_c[k - c0][j][i];
    }
    __syncthreads();
  }
  if (own) {
    const int p = v.seg_pair[my];
    const int ia = v.pair_atom[p];
    const int s = v.atom_struct[ia];
    const int ja = v.st[s].atom_off + v.neigh_j[p] - 1;
    const int nb = v.sp.norb[v.imass[ia] - 1] * v.sp.norb[v.imass[ja] - 1];
    double *dst = v.mat[FB_MAT_VNA] + v.boff[p];
    for (int i = 0; i < nb; i++) dst[i] = acc[i];
  }
  if (status) atomicOr(v.status, status);
}

extern "C" int fbk_3c_fp64(const DView &v, hipStream_t st) {
  if (v.ntrip == 0) return 0;
  if (fb_wide_species(v.sp)) {
    constexpr int T = Gen3c<FB_MOD>::T;
    hipLaunchKernelGGL(k_3c_fp64<FB_MOD>, dim3((unsigned)((v.ntrip + T - 1) / T)), dim3(T), 0, st, v);
  } else {
    constexpr int T = Gen3c<FB_MO>::T;
    hipLaunchKernelGGL(k_3c_fp64<FB_MO>, dim3((unsigned)((v.ntrip + T - 1) / T)), dim3(T), 0, st, v);
  }
  return (int)hipGetLastError();
}

// s/p species with canonical tables
#include "fb_3c_wave.h"

extern "C" int fbk_3c_fp64_ph(const DView &v, int charged, hipStream_t st) {
  if (v.ntiles[0] == 0) return 0;
  const dim3 grid((unsigned)v.ntiles[0]);
  if (charged)
    hipLaunchKernelGGL(k_3c_wave<W3_BCNA_Q>, grid, dim3(64 * w3_terms(W3_BCNA_Q)), 0, st, v);
  else
    hipLaunchKernelGGL(k_3c_wave<W3_BCNA>, grid, dim3(64 * w3_terms(W3_BCNA)), 0, st, v);
  return (int)hipGetLastError();
}
