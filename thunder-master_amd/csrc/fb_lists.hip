// Neighbour and common-neighbour (triplet) lists on the GPU, bit-identical to
// c.SYSTEM/M_neighbors.f90 (find_neighbors :356-519, find_common_neighbors
// :681-812).
//
// The general kernels, one workgroup per central atom, walk the candidates in
// the reference's order (image mbeta outer, atom jatom inner; or ineigh outer,
// jneigh inner for the triplets) in chunks of the workgroup size; an ordered compaction (wave
// ballot + cross-wave prefix in LDS) appends the accepted candidates, so no
// sort is needed and the list order is the reference's.  Distances use the
// reference's expression with contraction off.  Images whose bounding box lies
// farther than the cutoff (plus a 1e-6 A margin) from the central atom are
// skipped: they cannot contain a neighbour.
#include "fb_device.h"

#define LWG 256
#include "fb_lists_dev.h"

// Atoms up to which the list kernels of one workgroup per atom take 1024
// threads instead of 256: two such workgroups fit a compute unit, so all run at
// once.  Measured (targets counted / filled): 96 atoms 39 / 30 -> 30 / 23 us;
// 1000 atoms, 256 threads 61 / 49, 1024 threads 57 / 60 us.
#define LIST_WIDE 512

// n16 16-byte words from page-locked host memory
__global__ void k_copy_in(const int4 *src, int4 *dst, int64_t n16) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n16; i += (int64_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}

// atoms binned by cell (counting sort of the neighbour search)
__global__ void k_cell_count(DView v, int *cnt, int *atom_cell) {
  const int ia = blockIdx.x * blockDim.x + threadIdx.x;
  if (ia >= v.natoms) return;
  const DStruct S = v.st[v.atom_struct[ia]];
  const double r[3] = {v.ratom[3 * ia], v.ratom[3 * ia + 1], v.ratom[3 * ia + 2]};
  const int c = S.cell_off + cell_of(S, r);
  atom_cell[ia] = c;
  atomicAdd(&cnt[c], 1);
}

__device__ __forceinline__ CellAtom cell_record(const DView &v, int ia) {
  return CellAtom{{v.ratom[3 * ia], v.ratom[3 * ia + 1], v.ratom[3 * ia + 2]}, v.sp.rcmax[v.imass[ia] - 1]};
}

__global__ void k_cell_fill(DView v, const int *atom_cell, int *cursor, int *cell_atoms, CellAtom *cell_rec) {
  const int ia = blockIdx.x * blockDim.x + threadIdx.x;
  if (ia >= v.natoms) return;
  const int c = atom_cell[ia];
  const int k = atomicAdd(&cursor[c], 1);
  cell_atoms[v.cell_start[c] + k] = ia - v.st[v.atom_struct[ia]].atom_off;
  cell_rec[v.cell_start[c] + k] = cell_record(v, ia);
}

// The same in one launch of one workgroup, for few cells and atoms: clearing,
// counting, scan and fill are six launches, 36 us at 96 atoms and at 2048
// where this one takes 7 and 14 us.
__global__ __launch_bounds__(1024) void k_cells(DView v, int ncells, int64_t *cell_start, int *cell_atoms,
                                                CellAtom *cell_rec) {
  __shared__ int s_cnt[FB_CELLS_ONE];
  __shared__ int s_wave[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int c = tid; c < FB_CELLS_ONE; c += 1024) s_cnt[c] = 0;
  __syncthreads();
  auto cell = [&](int ia) {
    const DStruct &S = v.st[v.atom_struct[ia]];
    const double r[3] = {v.ratom[3 * ia], v.ratom[3 * ia + 1], v.ratom[3 * ia + 2]};
    return S.cell_off + cell_of(S, r);
  };
  for (int ia = tid; ia < v.natoms; ia += 1024) atomicAdd(&s_cnt[cell(ia)], 1);
  __syncthreads();
  int own[FB_CELLS_ONE / 1024], sum = 0;
#pragma unroll
  for (int u = 0; u < FB_CELLS_ONE / 1024; u++) {
    own[u] = s_cnt[tid * (FB_CELLS_ONE / 1024) + u];
    sum += own[u];
  }
  int inc = sum;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int y = __shfl_up(inc, d);
    if (lane >= d) inc += y;
  }
  if (lane == 63) s_wave[wave] = inc;
  __syncthreads();
  int at = inc - sum;
  for (int w = 0; w < wave; w++) at += s_wave[w];
#pragma unroll
  for (int u = 0; u < FB_CELLS_ONE / 1024; u++) {
    const int c = tid * (FB_CELLS_ONE / 1024) + u;
    s_cnt[c] = at;
    if (c <= ncells) cell_start[c] = at;
    at += own[u];
  }
  if (tid == 0 && ncells == FB_CELLS_ONE) cell_start[ncells] = v.natoms;
  __syncthreads();
  for (int ia = tid; ia < v.natoms; ia += 1024) {
    const int k = atomicAdd(&s_cnt[cell(ia)], 1);
    cell_atoms[k] = ia - v.st[v.atom_struct[ia]].atom_off;
    cell_rec[k] = cell_record(v, ia);
  }
}

// FILL = false: count neighbours (find_neigh_max); FILL = true: write them.
// With a cell list (v.cell_bits > 0) the candidates of each image are the
// atoms of the cells around r1 - xl(mbeta); the accepted ones are marked in a
// bitmap over jatom and written in jatom order, so the list order is the
// reference's either way.  Dynamic LDS: v.cell_bits words.
template <bool FILL>
__global__ __launch_bounds__(LWG) void k_neighbors(DView v, int *neighn_out, const int64_t *noff,
                                                   int *neigh_j, int *neigh_b, int *neigh_self,
                                                   int *pair_atom, int *status) {
  extern __shared__ unsigned s_bits[];
  __shared__ int64_t s_cs[27];
  __shared__ int s_pre[28];
  __shared__ int s_wave[LWG / 64];
  __shared__ int s_img[FB_NIMG];
  const int ia = blockIdx.x;  // global atom
  const int s = v.atom_struct[ia];
  const DStruct S = v.st[s];
  const int li = ia - S.atom_off;  // local 0-based
  const int in1 = v.imass[ia];
  double r1[3] = {v.ratom[3 * ia], v.ratom[3 * ia + 1], v.ratom[3 * ia + 2]};
  const double rci = v.sp.rcmax[in1 - 1];
  const double reach = rci + S.rcmax_all + 1.0e-6;
  const double *xls = v.xl + (int64_t)s * FB_NIMG * 3;
  int count = 0;
  int64_t base = FILL ? noff[ia] : 0;
  if (v.cell_bits > 0) {
    const int nw = (S.natoms + 31) >> 5;
    const int nimg = hit_images(S, xls, r1, reach, s_img, s_wave);
    for (int ki = 0; ki < nimg; ki++) {
      const int mb = s_img[ki];
      const double *xlb = xls + 3 * mb;
      const double q[3] = {r1[0] - xlb[0], r1[1] - xlb[1], r1[2] - xlb[2]};
      const int nc = query_cells(v, S, q, s_cs, s_pre);
      if (nc == 0) continue;
      for (int w = threadIdx.x; w < nw; w += LWG) s_bits[w] = 0u;
      __syncthreads();
      for (int t = threadIdx.x; t < s_pre[nc]; t += LWG) {
        const int lj = cell_candidate(v, s_cs, s_pre, nc, t);
        const int ja = S.atom_off + lj;
        double r2[3];
#pragma unroll
        for (int k = 0; k < 3; k++) r2[k] = v.ratom[3 * ja + k] + xlb[k];
        const double z = d_distance(r1, r2);
        const double range_max = rci + v.sp.rcmax[v.imass[ja] - 1] - 0.01;
        if (lj != li && z < 0.5) atomicOr(status, ST_TOO_CLOSE);
        if (z < range_max) atomicOr(&s_bits[lj >> 5], 1u << (lj & 31));
      }
      __syncthreads();
      for (int w0 = 0; w0 < nw; w0 += LWG) {
        const int w = w0 + threadIdx.x;
        const unsigned bits = (w < nw) ? s_bits[w] : 0u;
        int tot;
        const int pos = block_scan_count(__popc(bits), s_wave, &tot);
        if (FILL) {
          unsigned b = bits;
          int r = 0;
          while (b) {
            const int lj = w * 32 + __ffs(b) - 1;
            b &= b - 1u;
            const int64_t p = base + count + pos + r;
            neigh_j[p] = lj + 1;
            neigh_b[p] = mb;
            pair_atom[p] = ia;
            if (lj == li && mb == 0) neigh_self[ia] = count + pos + r + 1;
            r++;
          }
        }
        count += tot;
      }
    }
    if (!FILL && threadIdx.x == 0) neighn_out[ia] = count;
    return;
  }
  const int nimg = hit_images(S, xls, r1, reach, s_img, s_wave);
  for (int ki = 0; ki < nimg; ki++) {
    const int mb = s_img[ki];
    const double *xlb = xls + 3 * mb;
    for (int j0 = 0; j0 < S.natoms; j0 += LWG) {
      int lj = j0 + threadIdx.x;
      bool pass = false;
      if (lj < S.natoms) {
        int ja = S.atom_off + lj;
        double r2[3];
#pragma unroll
        for (int k = 0; k < 3; k++) r2[k] = v.ratom[3 * ja + k] + xlb[k];
        double z = d_distance(r1, r2);
        double range_max = rci + v.sp.rcmax[v.imass[ja] - 1] - 0.01;
        if (lj != li && z < 0.5) atomicOr(status, ST_TOO_CLOSE);
        pass = z < range_max;
      }
      int tot;
      int pos = block_rank(pass, s_wave, &tot);
      if (FILL && pass) {
        int64_t p = base + count + pos;
        neigh_j[p] = lj + 1;
        neigh_b[p] = mb;
        pair_atom[p] = ia;
        if (lj == li && mb == 0) neigh_self[ia] = count + pos + 1;
      }
      count += tot;
    }
  }
  if (!FILL && threadIdx.x == 0) neighn_out[ia] = count;
}

// ------------------------------------------------ neighbours in one search
// The search once instead of twice (count, then fill): a workgroup per atom
// tests the atoms of all cells of all images that may reach it, a wavefront
// per cell, keeps the hits in LDS as image << 18 | jatom, and sorts them by
// rank.  That key order is the reference's list order (mbeta outer, jatom
// inner).  The sorted keys go to the atom's FB_NB_CAP entries of a scratch
// array; k_list_scan turns counts into offsets, and k_nb_place writes the
// lists with all that follows from a pair (displacement, block offset, record)
// and finds neigh_back by binary search among the partner's keys.
// k_neighbors and the kernels below serve what this form does not: atoms with
// more neighbours than FB_NB_CAP, lattices with images within the reference's
// tolerances of each other, structures without a cell list.
// Latency-bound: 1024 threads per atom where there are fewer atoms than fill
// the chip.  Measured with the scans and launches they replace, C/H/N/O of 96
// atoms / carbon of 2048: 131 / 180 -> 25 / 59 us.
#define NB_SHIFT 18       // jatom's bits in a key (cell lists are used up to 262,144 atoms)

template <int W>
__global__ __launch_bounds__(W) void k_nb_find(DView v, const CellAtom *cell_rec, int *neighn, int *nblk,
                                               unsigned *keys, int *neigh_self, int *status) {
  constexpr int NI = 64;   // images per round
  __shared__ int s_img[FB_NIMG];
  __shared__ int s_cell[NI * 27];
  __shared__ short s_cimg[NI * 27];
  __shared__ unsigned s_key[FB_NB_CAP];
  __shared__ int s_nimg, s_ne, s_n, s_b;
  const int ia = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int s = v.atom_struct[ia];
  const DStruct &S = v.st[s];
  const int li = ia - S.atom_off, in1 = v.imass[ia], norb1 = v.sp.norb[in1 - 1];
  const double r1[3] = {v.ratom[3 * ia], v.ratom[3 * ia + 1], v.ratom[3 * ia + 2]};
  const double rci = v.sp.rcmax[in1 - 1], reach = rci + S.rcmax_all + 1.0e-6;
  const double *xls = v.xl + (int64_t)s * FB_NIMG * 3;
  if (tid == 0) {
    s_nimg = 0;
    s_n = 0;
    s_b = 0;
  }
  __syncthreads();
  for (int mb = tid; mb <= S.mbeta_max; mb += W)
    if (image_may_hit(S, xls + 3 * mb, r1, reach)) s_img[atomicAdd(&s_nimg, 1)] = mb;
  __syncthreads();
  const int nimg = s_nimg;
  int blk = 0;
  bool close = false;
  for (int i0 = 0; i0 < nimg; i0 += NI) {
    if (tid == 0) s_ne = 0;
    __syncthreads();
    if (tid < NI && i0 + tid < nimg) {
      // the cells that overlap the box +- crange around r1 in this image (query_cells)
      const int mb = s_img[i0 + tid];
      int lo[3], n[3];
      bool any = true;
#pragma unroll
      for (int a = 0; a < 3; a++) {
        const double q = r1[a] - xls[3 * mb + a];
        const double fl = floor((q - S.crange - S.clo[a]) / S.cw[a]);
        const double fh = floor((q + S.crange - S.clo[a]) / S.cw[a]);
        any = any && !(fh < 0.0 || fl > (double)(S.cn[a] - 1));
        lo[a] = (int)fmin(fmax(fl, 0.0), (double)(S.cn[a] - 1));
        n[a] = max(min((int)fmin(fh, (double)(S.cn[a] - 1)) - lo[a] + 1, 3), 0);
      }
      const int nc = any ? n[0] * n[1] * n[2] : 0;
      const int at = atomicAdd(&s_ne, nc);
      for (int t = 0; t < nc; t++) {
        const int cx = lo[0] + t % n[0], cy = lo[1] + (t / n[0]) % n[1], cz = lo[2] + t / (n[0] * n[1]);
        s_cell[at + t] = S.cell_off + (cz * S.cn[1] + cy) * S.cn[0] + cx;
        s_cimg[at + t] = (short)mb;
      }
    }
    __syncthreads();
    const int ne = s_ne;
    for (int e = wave; e < ne; e += W / 64) {
      const int c = s_cell[e], mb = s_cimg[e];
      const double x0 = xls[3 * mb], x1 = xls[3 * mb + 1], x2 = xls[3 * mb + 2];
      const int64_t k1 = v.cell_start[c + 1];
      for (int64_t k0 = v.cell_start[c]; k0 < k1; k0 += 64) {
        const int64_t k = k0 + lane;
        int lj = 0;
        bool hit = false;
        if (k < k1) {
          lj = v.cell_atoms[k];
          const CellAtom a = cell_rec[k];
          const double r2[3] = {a.r[0] + x0, a.r[1] + x1, a.r[2] + x2};
          const double z = d_distance(r1, r2);
          close |= lj != li && z < 0.5;
          hit = z < rci + a.rc - 0.01;
          if (hit) blk += norb1 * v.sp.norb[v.imass[S.atom_off + lj] - 1];
        }
        const unsigned long long m = __ballot(hit);
        if (m == 0) continue;
        int at = 0;
        if (lane == 0) at = atomicAdd(&s_n, __popcll(m));
        at = __builtin_amdgcn_readfirstlane(at) + __popcll(m & ((1ull << lane) - 1ull));
        if (hit && at < FB_NB_CAP) s_key[at] = ((unsigned)mb << NB_SHIFT) | (unsigned)lj;
      }
    }
    __syncthreads();
  }
  if (close) atomicOr(status, ST_TOO_CLOSE);
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) blk += __shfl_xor(blk, d);
  if (lane == 0 && blk) atomicAdd(&s_b, blk);
  __syncthreads();
  const int n = s_n;
  if (tid == 0) {
    neighn[ia] = n;
    nblk[ia] = s_b;
  }
  if (n > FB_NB_CAP) return;   // the general kernels take the whole build
  bool self = false;
  for (int i = tid; i < n; i += W) {
    const unsigned key = s_key[i];
    int rank = 0;
    for (int j = 0; j < n; j++) rank += s_key[j] < key ? 1 : 0;
    keys[(int64_t)ia * FB_NB_CAP + rank] = key;
    if (key == (unsigned)li) {
      neigh_self[ia] = rank + 1;
      self = true;
    }
  }
  if (!__syncthreads_or(self) && tid == 0) {
    neigh_self[ia] = -999;
    atomicOr(status, ST_SELF);
  }
}

// offsets of every atom's neighbours and block elements, on the device and in
// page-locked host memory (h_off: [natoms+1] pairs, [natoms+1] elements), and
// the status word
__global__ __launch_bounds__(1024) void k_list_scan(int natoms, const int *neighn, const int *nblk, int64_t *noff,
                                                    int64_t *aboff, int64_t *h_off, const int *status,
                                                    int *h_status) {
  __shared__ int64_t s_w[16][2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int64_t run[2] = {0, 0};
  for (int a0 = 0; a0 < natoms; a0 += 4096) {
    const int a = a0 + 4 * tid;
    int64_t e[4][2], mine[2] = {0, 0}, inc[2];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      e[u][0] = a + u < natoms ? neighn[a + u] : 0;
      e[u][1] = a + u < natoms ? nblk[a + u] : 0;
      mine[0] += e[u][0];
      mine[1] += e[u][1];
    }
    inc[0] = mine[0];
    inc[1] = mine[1];
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int64_t y0 = __shfl_up(inc[0], d), y1 = __shfl_up(inc[1], d);
      if (lane >= d) {
        inc[0] += y0;
        inc[1] += y1;
      }
    }
    if (lane == 63) {
      s_w[wave][0] = inc[0];
      s_w[wave][1] = inc[1];
    }
    __syncthreads();
    int64_t off[2] = {run[0] + inc[0] - mine[0], run[1] + inc[1] - mine[1]};
    for (int w = 0; w < 16; w++)
#pragma unroll
      for (int q = 0; q < 2; q++) {
        if (w < wave) off[q] += s_w[w][q];
        run[q] += s_w[w][q];
      }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (a + u < natoms) {
        noff[a + u] = off[0];
        aboff[a + u] = off[1];
        h_off[a + u] = off[0];
        h_off[natoms + 1 + a + u] = off[1];
        off[0] += e[u][0];
        off[1] += e[u][1];
      }
  }
  if (tid == 0) {
    noff[natoms] = run[0];
    aboff[natoms] = run[1];
    h_off[natoms] = run[0];
    h_off[2 * natoms + 1] = run[1];
    *h_status = *status;
  }
}

// a wavefront per atom
__global__ __launch_bounds__(256) void k_nb_place(DView v, const unsigned *keys, const int64_t *aboff, NbOut o,
                                                  int *status) {
  const int ia = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (ia >= v.natoms) return;
  const int s = v.atom_struct[ia], off = v.st[s].atom_off, li = ia - off;
  const int n = v.neighn[ia], in1 = v.imass[ia], norb1 = v.sp.norb[in1 - 1];
  const int64_t p0 = v.noff[ia];
  int64_t b = aboff[ia];
  const double *xls = v.xl + (int64_t)s * FB_NIMG * 3;
  for (int k0 = 0; k0 < n; k0 += 64) {
    const int k = k0 + lane;
    const bool on = k < n;
    const unsigned key = on ? keys[(int64_t)ia * FB_NB_CAP + k] : 0u;
    const int lj = (int)(key & ((1u << NB_SHIFT) - 1u)), mb = (int)(key >> NB_SHIFT), ja = off + lj;
    const int in2 = v.imass[ja], size = on ? norb1 * v.sp.norb[in2 - 1] : 0;
    int inc = size;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int y = __shfl_up(inc, d);
      if (lane >= d) inc += y;
    }
    if (on) {
      const int64_t p = p0 + k;
      o.neigh_j[p] = lj + 1;
      o.neigh_b[p] = mb;
      o.pair_atom[p] = ia;
      o.rec[p] = make_int4(ia, ja, s * FB_NIMG + mb, in1 | (in2 << 16));
      o.boff[p] = b + inc - size;
#pragma unroll
      for (int q = 0; q < 3; q++) o.disp[3 * p + q] = xls[3 * mb + q] + v.ratom[3 * ja + q] - v.ratom[3 * ia + q];
      int c[3];
      image_coords(mb, c);
      const unsigned want = ((unsigned)image_of(-c[0], -c[1], -c[2]) << NB_SHIFT) | (unsigned)li;
      const unsigned *kj = keys + (int64_t)ja * FB_NB_CAP;
      const int nj = v.neighn[ja];
      int lo = 0, hi = nj;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (kj[mid] < want) lo = mid + 1;
        else hi = mid;
      }
      const bool found = lo < nj && kj[lo] == want;
      if (!found) atomicOr(status, ST_BACK);
      o.neigh_back[p] = found ? lo + 1 : -999;
    }
    b += __shfl(inc, 63);
  }
  if (ia == v.natoms - 1 && lane == 0) o.boff[p0 + n] = b;
}

// displacement of every neighbour pair, xl(jbeta) + r_j - r_i with the
// reference's evaluation order (M_neighbors.f90:766-769 compares it with r2 - r1)
__global__ void k_pair_disp(DView v, double *disp) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= v.npairs) return;
  const int ia = v.pair_atom[p];
  const int s = v.atom_struct[ia];
  const int ja = v.st[s].atom_off + v.neigh_j[p] - 1;
  const double *xlb = v.xl + (int64_t)s * FB_NIMG * 3 + 3 * v.neigh_b[p];
#pragma unroll
  for (int k = 0; k < 3; k++) disp[3 * p + k] = xlb[k] + v.ratom[3 * ja + k] - v.ratom[3 * ia + k];
}

// neigh_back, c.SYSTEM/M_neighbors.f90:469-486: the jneigh of jatom that
// points back at (iatom, -xl(mbeta)) within 1e-3 A per component.
__global__ void k_neigh_back(DView v, int *neigh_back, int *status) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= v.npairs) return;
  int ia = v.pair_atom[p];
  int s = v.atom_struct[ia];
  const DStruct S = v.st[s];
  int li1 = ia - S.atom_off + 1;
  int ja = S.atom_off + v.neigh_j[p] - 1;
  const double *xls = v.xl + (int64_t)s * FB_NIMG * 3;
  const double *xm = xls + 3 * v.neigh_b[p];
  int found = -999;
  int64_t jo = v.noff[ja];
  int nj = v.neighn[ja];
  for (int jn = 0; jn < nj; jn++) {
    int ka = v.neigh_j[jo + jn];
    const double *xj = xls + 3 * v.neigh_b[jo + jn];
    if (li1 != ka || fabs(xm[0] + xj[0]) > 1.0e-3 || fabs(xm[1] + xj[1]) > 1.0e-3 ||
        fabs(xm[2] + xj[2]) > 1.0e-3) {
    } else {
      if (found != -999) atomicOr(status, ST_BACK);
      found = jn + 1;
    }
  }
  if (found == -999) atomicOr(status, ST_BACK);
  neigh_back[p] = found;
}

// ------------------------------------------------ triplets in target order
// Every assembler sums triplets per target block, in the reference's order
// (ialpha ascending, then the common-pair order).  A target pair (iatom,
// jatom at image mbeta) receives a triplet from every other neighbour of
// iatom, an atom ialpha at image b, that has jatom among its own neighbours;
// seen from ialpha, iatom lies at image ib = -b and jatom at jb = ib + mbeta.
// So the neighbours of iatom, sorted by (ialpha, ib), give the segment of a
// target directly and in order: no list-order pass, no search for mneigh (the
// target is the pair at hand) and no sort.  The conditions are those of
// find_common_neighbors (M_neighbors.f90:681-812) in ialpha's frame, with the
// same binary64 expressions: jatom in ialpha's list, |r2 - r1| below the
// range, and the pair's displacement within 1e-4 of r2 - r1.
//
// One workgroup per atom, one wavefront per target, lanes over the sorted
// neighbours.  k_targets<false> tests the candidates and keeps the ballot
// masks (one word per target and 64 neighbours), the targets' counts and the
// atom's totals, with its tiles of whole segments (greedy, at most 64, 128 or
// 256 triplets); k_targets<true> writes triplets, segments and tiles at the
// scanned offsets from the masks alone.
// LDS per neighbour: home position, iatom at image ib and cutoff (tests only),
// atom, image, ib, count, prefix, segment, order
#define TGT_LDS(FILL) (((FILL) ? 0 : 56) + 20 + 4)
#define TGT_NMAX 768      // neighbours per atom: 61 KB

template <bool FILL, int W>
__global__ __launch_bounds__(W) void k_targets(DView v, TgtSum *sum, unsigned long long *mask, int nword, int *pcnt,
                                                 TgtOut out) {
  extern __shared__ __align__(16) unsigned char s_mem[];
  __shared__ int s_wave[W / 64];
  const int ia = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int s = v.atom_struct[ia];
  const DStruct S = v.st[s];
  const double *xls = v.xl + (int64_t)s * FB_NIMG * 3;
  const int64_t o = v.noff[ia];
  const int n = (int)(v.noff[ia + 1] - o);
  double *sRa = reinterpret_cast<double *>(s_mem), *sR1 = sRa + 3 * n, *sRc = sR1 + 3 * n;
  int *sAt = reinterpret_cast<int *>(s_mem + (FILL ? 0 : 56 * (size_t)n));
  int *sImg = sAt + n, *sIb = sImg + n, *sCnt = sIb + n, *sPre = sCnt + n;
  unsigned short *sSeg = reinterpret_cast<unsigned short *>(sPre + n), *sOrd = sSeg + n;
  const int in1 = v.imass[ia];
  const double rc1 = v.sp.rcmax[in1 - 1];
  for (int k = tid; k < n; k += W) {
    const int at = S.atom_off + v.neigh_j[o + k] - 1, b = v.neigh_b[o + k];
    int c[3];
    image_coords(b, c);
    const int ib = image_of(-c[0], -c[1], -c[2]);
    sAt[k] = at;
    sImg[k] = (c[0] + 4) | (c[1] + 4) << 4 | (c[2] + 4) << 8;
    sIb[k] = ib;
    if (FILL) {
      sCnt[k] = pcnt[o + k];
    } else {
      sRc[k] = v.sp.rcmax[v.imass[at] - 1];
#pragma unroll
      for (int q = 0; q < 3; q++) {
        sRa[3 * k + q] = v.ratom[3 * at + q];
        sR1[3 * k + q] = v.ratom[3 * ia + q] + xls[3 * ib + q];
      }
    }
  }
  __syncthreads();
  // order of the neighbours by (ialpha, ib); the entries are distinct
  for (int k = tid; k < n; k += W) {
    const int at = sAt[k], ib = sIb[k];
    int rank = 0;
    for (int j = 0; j < n; j++) rank += (sAt[j] < at || (sAt[j] == at && sIb[j] < ib)) ? 1 : 0;
    sOrd[rank] = (unsigned short)k;
  }
  TgtSum base = {0, 0, {0, 0, 0}};
  if (FILL) {
    base = sum[ia];
    // first triplet and segment of every target
    int run = 0, srun = 0;
    for (int k0 = 0; k0 < n; k0 += W) {
      const int k = k0 + tid, c = k < n ? sCnt[k] : 0;
      int tot, stot;
      const int pos = run + block_scan_count<W>(c, s_wave, &tot);
      const int sg = srun + block_rank<W>(c > 0, s_wave, &stot);
      if (k < n) {
        sPre[k] = pos;
        sSeg[k] = (unsigned short)sg;
        out.pair_tgt[o + k] = c > 0;
        if (c > 0) {
          out.seg_off[base.seg + sg] = base.trip + pos;
          out.seg_pair[base.seg + sg] = (int)(o + k);
        }
      }
      run += tot;
      srun += stot;
    }
    if (ia == v.natoms - 1 && tid == 0) out.seg_off[base.seg + srun] = base.trip + run;
  }
  __syncthreads();
  for (int p = wave; p < n; p += W / 64) {
    const int ja = sAt[p], cp = sImg[p];
    const int px = (cp & 15) - 4, py = (cp >> 4 & 15) - 4, pz = (cp >> 8 & 15) - 4;
    const bool target = !(ja == ia && px == 0 && py == 0 && pz == 0);   // not the self entry
    if (FILL && sCnt[p] == 0) continue;
    double rj[3] = {0.0, 0.0, 0.0}, dp[3] = {0.0, 0.0, 0.0}, rc2 = 0.0, range = 0.0;
    if (!FILL) {
      rc2 = sRc[p];
      range = rc1 + rc2 - 0.01;
#pragma unroll
      for (int q = 0; q < 3; q++) {
        rj[q] = sRa[3 * p + q];
        dp[q] = v.pair_disp[3 * (o + p) + q];
      }
    }
    int count = 0;
    for (int k0 = 0; k0 < n; k0 += 64) {
      unsigned long long m = FILL ? mask[(o + p) * nword + (k0 >> 6)] : 0ull;
      int ial = 0, ib = 0, jb = 0;
      bool pass = FILL ? (m >> lane & 1ull) : (target && k0 + lane < n);
      if (pass) {
        const int k = sOrd[k0 + lane], ck = sImg[k];
        ial = sAt[k];
        ib = sIb[k];
        const int x = px - (ck & 15) + 4, y = py - (ck >> 4 & 15) + 4, z = pz - (ck >> 8 & 15) + 4;
        if (FILL) {
          jb = image_of(x, y, z);
        } else {
          pass = abs(x) <= 4 && abs(y) <= 4 && abs(z) <= 4 && !(ial == ia && ib == 0);
          if (pass) {
            jb = image_of(x, y, z);
            double r1[3], r2[3], ra[3];
#pragma unroll
            for (int q = 0; q < 3; q++) {
              r1[q] = sR1[3 * k + q];
              r2[q] = rj[q] + xls[3 * jb + q];
              ra[q] = sRa[3 * k + q];
            }
            pass = !(ja == ial && jb == 0) && d_distance(ra, r2) < sRc[k] + rc2 - 0.01 &&
                   d_distance(r1, r2) < range && fabs(dp[0] - r2[0] + r1[0]) < 1.0e-4 &&
                   fabs(dp[1] - r2[1] + r1[1]) < 1.0e-4 && fabs(dp[2] - r2[2] + r1[2]) < 1.0e-4;
          }
        }
      }
      if (!FILL) {
        m = __ballot(pass);
        if (lane == 0) mask[(o + p) * nword + (k0 >> 6)] = m;
      } else if (pass) {
        const int64_t t = base.trip + sPre[p] + count + __popcll(m & ((1ull << lane) - 1ull));
        out.trip[t] = make_int4(ial, ia, ja, (ib & 0xffff) | (jb << 16));
        out.trip_pair[t] = (int)(o + p);
        out.trip_seg[t] = base.seg + sSeg[p];
        const int gid = v.idx3c[(((in1 - 1) * v.sp.ns + (v.imass[ja] - 1)) * v.sp.ns + (v.imass[ial] - 1)) *
                                FB_MAXSUB3];
        out.trip_aux[t] = (gid < 0 ? 0xffff : gid) | (s << 16);
      }
      count += __popcll(m);
    }
    if (!FILL && lane == 0) {
      pcnt[o + p] = count;
      sCnt[p] = count;
    }
  }
  __syncthreads();
  // tiles of whole segments: thread c packs greedily for 64 << c triplets (a
  // longer segment alone), the rule of k_tiles_atom
  if (tid < 3) {
    const int ch = 64 << tid;
    int4 *tl = out.tiles[tid];
    int cur = 0, nt = 0, seg = 0, t = 0, s0 = 0, f0 = 0;
    for (int k = 0; k < n; k++) {
      const int c = sCnt[k];
      if (c == 0) continue;
      if (cur > 0 && cur + c > ch) {
        if (FILL)
          tl[base.tile[tid] + nt] =
              make_int4(base.seg + s0, base.seg + seg - 1, (int)base.trip + f0, (int)base.trip + t);
        nt++;
        cur = 0;
        s0 = seg;
        f0 = t;
      }
      cur += c;
      t += c;
      seg++;
    }
    if (cur > 0) {
      if (FILL)
        tl[base.tile[tid] + nt] = make_int4(base.seg + s0, base.seg + seg - 1, (int)base.trip + f0, (int)base.trip + t);
      nt++;
    }
    if (!FILL) {
      sum[ia].tile[tid] = nt;
      if (tid == 0) {
        sum[ia].trip = t;
        sum[ia].seg = seg;
      }
    }
  }
}

// exclusive prefix of the atoms' totals in place (entry natoms: the totals);
// one workgroup, four atoms per thread and pass
__global__ __launch_bounds__(1024) void k_target_scan(int natoms, TgtSum *sum, int64_t *h_toff, TgtSum *h_tot,
                                                      const int *status, int *h_status) {
  __shared__ int64_t s_t[16];
  __shared__ int s_i[16][4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  TgtSum run = {0, 0, {0, 0, 0}};
  for (int a0 = 0; a0 < natoms; a0 += 4096) {
    const int a = a0 + 4 * tid;
    TgtSum e[4], mine = {0, 0, {0, 0, 0}};
    for (int u = 0; u < 4; u++) {
      e[u] = (a + u < natoms) ? sum[a + u] : TgtSum{0, 0, {0, 0, 0}};
      mine.trip += e[u].trip;
      mine.seg += e[u].seg;
      for (int c = 0; c < 3; c++) mine.tile[c] += e[u].tile[c];
    }
    TgtSum inc = mine;
    for (int d = 1; d < 64; d <<= 1) {
      const int64_t yt = __shfl_up(inc.trip, d);
      const int ys = __shfl_up(inc.seg, d);
      int yc[3];
      for (int c = 0; c < 3; c++) yc[c] = __shfl_up(inc.tile[c], d);
      if (lane >= d) {
        inc.trip += yt;
        inc.seg += ys;
        for (int c = 0; c < 3; c++) inc.tile[c] += yc[c];
      }
    }
    if (lane == 63) {
      s_t[wave] = inc.trip;
      s_i[wave][0] = inc.seg;
      for (int c = 0; c < 3; c++) s_i[wave][1 + c] = inc.tile[c];
    }
    __syncthreads();
    TgtSum off = run;
    for (int w = 0; w < 16; w++) {
      if (w < wave) {
        off.trip += s_t[w];
        off.seg += s_i[w][0];
        for (int c = 0; c < 3; c++) off.tile[c] += s_i[w][1 + c];
      }
      run.trip += s_t[w];
      run.seg += s_i[w][0];
      for (int c = 0; c < 3; c++) run.tile[c] += s_i[w][1 + c];
    }
    __syncthreads();
    off.trip += inc.trip - mine.trip;
    off.seg += inc.seg - mine.seg;
    for (int c = 0; c < 3; c++) off.tile[c] += inc.tile[c] - mine.tile[c];
    for (int u = 0; u < 4; u++) {
      if (a + u < natoms) {
        sum[a + u] = off;
        h_toff[a + u] = off.trip;
      }
      off.trip += e[u].trip;
      off.seg += e[u].seg;
      for (int c = 0; c < 3; c++) off.tile[c] += e[u].tile[c];
    }
  }
  if (tid == 0) {
    sum[natoms] = run;
    h_toff[natoms] = run.trip;
    *h_tot = run;
    *h_status = *status;
  }
}

// common neighbours of ialpha in the reference's list order (fb_get_common,
// the force assemblers).  FILL = false counts (find_common_max plus the drop
// rule of find_common_neighbors, so the counts are exact); FILL = true writes
// the triplet and its target pair.  mneigh is the first entry of iatom whose
// displacement matches r2 - r1 within 1e-4.  A list is sorted by (mbeta,
// jatom) and names (jatom, jbeta - ibeta) at most once, so a binary search
// finds it; SCAN tests the entries in order instead, for lattices in which
// two images coincide and the difference may go by another image's number.
template <bool FILL, bool SCAN>
__global__ __launch_bounds__(LWG) void k_common(DView v, int *ncommon_out, const int64_t *toff,
                                                int4 *trip, int *trip_pair) {
  __shared__ int s_wave[LWG / 64];
  const int ial = blockIdx.x;
  const int s = v.atom_struct[ial];
  const DStruct S = v.st[s];
  const int lal = ial - S.atom_off + 1;  // 1-based local
  const double *xls = v.xl + (int64_t)s * FB_NIMG * 3;
  const int64_t o = v.noff[ial];
  const int n = v.neighn[ial];
  const int64_t ncand = (int64_t)n * n;
  int count = 0;
  int64_t base = FILL ? toff[ial] : 0;
  for (int64_t c0 = 0; c0 < ncand; c0 += LWG) {
    int64_t c = c0 + threadIdx.x;
    bool pass = false;
    int ia = 0, ib = 0, ja = 0, jb = 0, m = -9999;
    if (c < ncand) {
      int in = (int)(c / n), jn = (int)(c % n);
      ia = v.neigh_j[o + in];
      ib = v.neigh_b[o + in];
      ja = v.neigh_j[o + jn];
      jb = v.neigh_b[o + jn];
      if (!(ia == lal && ib == 0) && !(ja == lal && jb == 0) && in != jn) {
        int gia = S.atom_off + ia - 1, gja = S.atom_off + ja - 1;
        double r1[3], r2[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
          r1[k] = v.ratom[3 * gia + k] + xls[3 * ib + k];
          r2[k] = v.ratom[3 * gja + k] + xls[3 * jb + k];
        }
        double z = d_distance(r1, r2);
        double range_max = v.sp.rcmax[v.imass[gia] - 1] + v.sp.rcmax[v.imass[gja] - 1] - 0.01;
        if (z < range_max) {
          const double *dp = v.pair_disp + 3 * v.noff[gia];
          auto match = [&](int k) {
            return fabs(dp[3 * k] - r2[0] + r1[0]) < 1.0e-4 && fabs(dp[3 * k + 1] - r2[1] + r1[1]) < 1.0e-4 &&
                   fabs(dp[3 * k + 2] - r2[2] + r1[2]) < 1.0e-4;
          };
          const int ni = v.neighn[gia];
          if (SCAN) {
            for (int k = 0; k < ni && m == -9999; k++)
              if (match(k)) m = k + 1;
          } else {
            int ci[3], cj[3];
            image_coords(ib, ci);
            image_coords(jb, cj);
            const int x = cj[0] - ci[0], y = cj[1] - ci[1], w = cj[2] - ci[2];
            if (abs(x) <= 4 && abs(y) <= 4 && abs(w) <= 4) {
              const int kb = image_of(x, y, w);
              const int *lj = v.neigh_j + v.noff[gia], *lb = v.neigh_b + v.noff[gia];
              int lo = 0, hi = ni;
              while (lo < hi) {
                const int mid = (lo + hi) >> 1, b = lb[mid];
                if (b < kb || (b == kb && lj[mid] < ja)) lo = mid + 1;
                else hi = mid;
              }
              if (lo < ni && lb[lo] == kb && lj[lo] == ja && match(lo)) m = lo + 1;
            }
          }
          pass = (m != -9999);
        }
      }
    }
    int tot;
    int pos = block_rank(pass, s_wave, &tot);
    if (FILL && pass) {
      int64_t t = base + count + pos;
      int gia = S.atom_off + ia - 1, gja = S.atom_off + ja - 1;
      trip[t] = make_int4(ial, gia, gja, (ib & 0xffff) | (jb << 16));
      trip_pair[t] = (int)(v.noff[gia] + m - 1);
      // mneigh is recovered from the target pair: m = trip_pair - noff[iatom] + 1
    }
    count += tot;
  }
  if (!FILL && threadIdx.x == 0) ncommon_out[ial] = count;
}

// segment bookkeeping after the stable sort of triplets by target pair
__global__ void k_seg_mark(int64_t ntrip, const int *sorted_pair, int *flag) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntrip) return;
  flag[t] = (t == 0 || sorted_pair[t] != sorted_pair[t - 1]) ? 1 : 0;
}

__global__ void k_seg_fill(int64_t ntrip, const int *sorted_pair, const int *segid_incl, int64_t *seg_off,
                           int *seg_pair, int *trip_seg, int *pair_tgt) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntrip) return;
  int sid = segid_incl[t] - 1;
  trip_seg[t] = sid;
  if (t == 0 || sorted_pair[t] != sorted_pair[t - 1]) {
    seg_off[sid] = t;
    seg_pair[sid] = sorted_pair[t];
    pair_tgt[sorted_pair[t]] = 1;
  }
  if (t == ntrip - 1) seg_off[sid + 1] = ntrip;
}

__global__ void k_gather_trip(int64_t ntrip, const int *perm, const int4 *trip_in, int4 *trip_out) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntrip) return;
  trip_out[t] = trip_in[perm[t]];
}

__global__ void k_iota(int64_t n, int *a) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) a[t] = (int)t;
}

// block offsets: boff[p] = sum of norb_i * norb_j over earlier pairs; and
// the pair's record (the atoms, the image and the species in one int4)
__global__ void k_block_sizes(DView v, int64_t *sz, int4 *rec) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= v.npairs) return;
  int ia = v.pair_atom[p];
  int s = v.atom_struct[ia];
  int ja = v.st[s].atom_off + v.neigh_j[p] - 1;
  const int in1 = v.imass[ia], in2 = v.imass[ja];
  sz[p] = (int64_t)v.sp.norb[in1 - 1] * v.sp.norb[in2 - 1];
  rec[p] = make_int4(ia, ja, s * FB_NIMG + v.neigh_b[p], in1 | (in2 << 16));
}

// Tiles of whole target segments for the segment-owning kernels, packed per
// atom (a segment's target pair belongs to one atom, so a tile never needs to
// span atoms): greedily at most ch triplets per tile, a longer segment alone.
// A wavefront per atom over its segments, found by binary search of its pair
// range in the sorted segment pairs: it holds the offsets of 64 segments and
// finds a tile's end with one ballot, where a thread per atom waited for a
// load per segment (PP lists of 1000 atoms: counted and filled in 105 + 63 ->
// 11 + 11 us).  FILL = false counts, FILL = true writes (first, last segment,
// first, end triplet).  Any partition into whole segments gives the kernels
// the same per-segment order, hence the same bits.
template <bool FILL>
__global__ __launch_bounds__(256) void k_tiles_atom(int natoms, const int64_t *pair_off, const int64_t *seg_off,
                                                    const int *seg_pair, int64_t nseg, int ch, int *cnt,
                                                    const int64_t *tile_off, int4 *tiles) {
  const int ia = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (ia >= natoms) return;
  // the first segments of this atom and of the next one, by two lanes
  const int64_t key = pair_off[ia + (lane & 1)];
  int64_t lo = 0, hi = nseg;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if ((int64_t)seg_pair[mid] < key) lo = mid + 1;
    else hi = mid;
  }
  int64_t s = __shfl(lo, 0);
  const int64_t s1 = __shfl(lo, 1), t0 = FILL ? tile_off[ia] : 0;
  int count = 0;
  while (s < s1) {   // the window of 64 segments from s
    const bool in = s + lane < s1;
    const int64_t o0 = in ? seg_off[s + lane] : 0, o1 = in ? seg_off[s + lane + 1] : 0;
    const bool last = s + 64 >= s1;
    int i = 0;
    for (;;) {
      const int64_t first = __shfl(o0, i);
      const unsigned long long m = __ballot(in && lane >= i && (lane == i || o1 - first <= ch));
      int64_t e = i + __popcll(m);   // one past the tile's last segment, in the window
      if (e == 64 && !last) {
        if (i > 0) break;            // it may go on: again from its first segment
        while (s + e < s1 && seg_off[s + e + 1] - first <= ch) e++;
      }
      if (FILL && lane == 0)
        tiles[t0 + count] = make_int4((int)s + i, (int)(s + e) - 1, (int)first, (int)seg_off[s + e]);
      count++;
      i = (int)e;
      if (i >= 64 || s + i >= s1) break;
    }
    s += i;
  }
  if (!FILL && lane == 0) cnt[ia] = count;
}

__global__ void k_gather_i64(int n, const int64_t *src, const int64_t *idx, int64_t *dst) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) dst[k] = src[idx[k]];
}

// ----------------------------------------------------------------- launchers
#include <hipcub/hipcub.hpp>

extern "C" {

int fbk_tiles_atom(int natoms, const int64_t *pair_off, const int64_t *seg_off, const int *seg_pair, int64_t nseg,
                   int ch, int fill, int *cnt, const int64_t *tile_off, int4 *tiles, hipStream_t st) {
  if (natoms == 0) return 0;
  const dim3 g((unsigned)((natoms + 3) / 4));
  if (fill)
    hipLaunchKernelGGL(k_tiles_atom<true>, g, dim3(256), 0, st, natoms, pair_off, seg_off, seg_pair, nseg, ch, cnt,
                       tile_off, tiles);
  else
    hipLaunchKernelGGL(k_tiles_atom<false>, g, dim3(256), 0, st, natoms, pair_off, seg_off, seg_pair, nseg, ch, cnt,
                       tile_off, tiles);
  return (int)hipGetLastError();
}

int fbk_gather_i64(int n, const int64_t *src, const int64_t *idx, int64_t *dst, hipStream_t st) {
  if (n == 0) return 0;
  hipLaunchKernelGGL(k_gather_i64, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, src, idx, dst);
  return (int)hipGetLastError();
}

int fbk_cell_count(const DView &v, int *cnt, int *atom_cell, hipStream_t st) {
  if (v.natoms == 0) return 0;
  hipLaunchKernelGGL(k_cell_count, dim3((unsigned)((v.natoms + 255) / 256)), dim3(256), 0, st, v, cnt, atom_cell);
  return (int)hipGetLastError();
}

int fbk_copy_in(const void *src, void *dst, int64_t n16, hipStream_t st) {
  if (n16 == 0) return 0;
  hipLaunchKernelGGL(k_copy_in, dim3((unsigned)std::min<int64_t>((n16 + 255) / 256, 256)), dim3(256), 0, st,
                     (const int4 *)src, (int4 *)dst, n16);
  return (int)hipGetLastError();
}
int fbk_cell_fill(const DView &v, const int *atom_cell, int *cursor, int *cell_atoms, CellAtom *cell_rec,
                  hipStream_t st) {
  if (v.natoms == 0) return 0;
  hipLaunchKernelGGL(k_cell_fill, dim3((unsigned)((v.natoms + 255) / 256)), dim3(256), 0, st, v, atom_cell, cursor,
                     cell_atoms, cell_rec);
  return (int)hipGetLastError();
}
int fbk_cells(const DView &v, int ncells, int64_t *cell_start, int *cell_atoms, CellAtom *cell_rec, hipStream_t st) {
  if (ncells > FB_CELLS_ONE) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(k_cells, dim3(1), dim3(1024), 0, st, v, ncells, cell_start, cell_atoms, cell_rec);
  return (int)hipGetLastError();
}
int fbk_nb_find(const DView &v, const CellAtom *cell_rec, int *neighn, int *nblk, unsigned *keys, int *neigh_self,
                int64_t *noff, int64_t *aboff, int64_t *h_off, int *h_status, hipStream_t st) {
  if (v.natoms == 0) return (int)hipErrorInvalidValue;
  if (v.natoms <= LIST_WIDE)
    hipLaunchKernelGGL(k_nb_find<1024>, dim3((unsigned)v.natoms), dim3(1024), 0, st, v, cell_rec, neighn, nblk, keys,
                       neigh_self, v.status);
  else
    hipLaunchKernelGGL(k_nb_find<256>, dim3((unsigned)v.natoms), dim3(256), 0, st, v, cell_rec, neighn, nblk, keys,
                       neigh_self, v.status);
  hipLaunchKernelGGL(k_list_scan, dim3(1), dim3(1024), 0, st, v.natoms, neighn, nblk, noff, aboff, h_off, v.status,
                     h_status);
  return (int)hipGetLastError();
}
int fbk_nb_place(const DView &v, const unsigned *keys, const int64_t *aboff, const NbOut &o, hipStream_t st) {
  hipLaunchKernelGGL(k_nb_place, dim3((unsigned)((v.natoms + 3) / 4)), dim3(256), 0, st, v, keys, aboff, o, v.status);
  return (int)hipGetLastError();
}

int fbk_neighbors_count(const DView &v, int *neighn, int *status, hipStream_t st) {
  const size_t lds = sizeof(unsigned) * (size_t)v.cell_bits;
  hipLaunchKernelGGL(k_neighbors<false>, dim3(v.natoms), dim3(LWG), lds, st, v, neighn, (const int64_t *)nullptr,
                     (int *)nullptr, (int *)nullptr, (int *)nullptr, (int *)nullptr, status);
  return (int)hipGetLastError();
}

int fbk_neighbors_fill(const DView &v, const int64_t *noff, int *neigh_j, int *neigh_b, int *neigh_self,
                       int *pair_atom, int *status, hipStream_t st) {
  const size_t lds = sizeof(unsigned) * (size_t)v.cell_bits;
  hipLaunchKernelGGL(k_neighbors<true>, dim3(v.natoms), dim3(LWG), lds, st, v, (int *)nullptr, noff, neigh_j,
                     neigh_b, neigh_self, pair_atom, status);
  return (int)hipGetLastError();
}

int fbk_pair_disp(const DView &v, double *disp, hipStream_t st) {
  if (v.npairs == 0) return 0;
  hipLaunchKernelGGL(k_pair_disp, dim3((unsigned)((v.npairs + 255) / 256)), dim3(256), 0, st, v, disp);
  return (int)hipGetLastError();
}

int fbk_neigh_back(const DView &v, int *neigh_back, int *status, hipStream_t st) {
  if (v.npairs == 0) return 0;
  hipLaunchKernelGGL(k_neigh_back, dim3((unsigned)((v.npairs + 255) / 256)), dim3(256), 0, st, v, neigh_back,
                     status);
  return (int)hipGetLastError();
}

int fbk_common_count(const DView &v, int scan, int *ncommon, hipStream_t st) {
  const dim3 g((unsigned)v.natoms);
  if (scan)
    hipLaunchKernelGGL((k_common<false, true>), g, dim3(LWG), 0, st, v, ncommon, (const int64_t *)nullptr,
                       (int4 *)nullptr, (int *)nullptr);
  else
    hipLaunchKernelGGL((k_common<false, false>), g, dim3(LWG), 0, st, v, ncommon, (const int64_t *)nullptr,
                       (int4 *)nullptr, (int *)nullptr);
  return (int)hipGetLastError();
}

int fbk_common_fill(const DView &v, int scan, const int64_t *toff, int4 *trip, int *trip_pair, hipStream_t st) {
  const dim3 g((unsigned)v.natoms);
  if (scan)
    hipLaunchKernelGGL((k_common<true, true>), g, dim3(LWG), 0, st, v, (int *)nullptr, toff, trip, trip_pair);
  else
    hipLaunchKernelGGL((k_common<true, false>), g, dim3(LWG), 0, st, v, (int *)nullptr, toff, trip, trip_pair);
  return (int)hipGetLastError();
}

// most neighbours per atom that the target-order kernels take
int fbk_targets_nmax(void) { return TGT_NMAX; }

int fbk_targets_count(const DView &v, int nmax, TgtSum *sum, unsigned long long *mask, int *pcnt, int64_t *h_toff,
                      TgtSum *h_tot, int *h_status, hipStream_t st) {
  if (nmax > TGT_NMAX) return (int)hipErrorInvalidValue;
  const dim3 grid((unsigned)v.natoms);
  const size_t lds = TGT_LDS(false) * (size_t)nmax;
  if (v.natoms <= LIST_WIDE)
    hipLaunchKernelGGL((k_targets<false, 1024>), grid, dim3(1024), lds, st, v, sum, mask, (nmax + 63) / 64, pcnt,
                       TgtOut{});
  else
    hipLaunchKernelGGL((k_targets<false, LWG>), grid, dim3(LWG), lds, st, v, sum, mask, (nmax + 63) / 64, pcnt,
                       TgtOut{});
  hipLaunchKernelGGL(k_target_scan, dim3(1), dim3(1024), 0, st, v.natoms, sum, h_toff, h_tot, v.status,
                     h_status);
  return (int)hipGetLastError();
}

int fbk_targets_fill(const DView &v, int nmax, TgtSum *sum, unsigned long long *mask, int *pcnt, const TgtOut &out,
                     hipStream_t st) {
  if (nmax > TGT_NMAX) return (int)hipErrorInvalidValue;
  const dim3 grid((unsigned)v.natoms);
  const size_t lds = TGT_LDS(true) * (size_t)nmax;
  if (v.natoms <= LIST_WIDE)
    hipLaunchKernelGGL((k_targets<true, 1024>), grid, dim3(1024), lds, st, v, sum, mask, (nmax + 63) / 64, pcnt, out);
  else
    hipLaunchKernelGGL((k_targets<true, LWG>), grid, dim3(LWG), lds, st, v, sum, mask, (nmax + 63) / 64, pcnt, out);
  return (int)hipGetLastError();
}

// Lane order of the 2c workgroups (fb_2c_sp.h): within each 64-pair
// wavefront group of a workgroup item (the groups that pass c0 of item b
// forms: c0 + 64 w), the pairs by species pair, then bond length, then index,
// so that neighbouring lanes interpolate nearby rows of the same table.  perm[slot] is the
// group-relative index of the pair that the lane at slot takes.  Blocks and
// sums are placed by pair index, so any permutation gives the same bits.
__global__ __launch_bounds__(FB_2C_PCAP) void k_pair_perm(DView v, unsigned char *perm) {
  __shared__ double s_x[FB_2C_PCAP];
  __shared__ int s_k[FB_2C_PCAP];
  const int tid = threadIdx.x;
  const int64_t pb = v.noff[v.wg2c[blockIdx.x]], pe = v.noff[v.wg2c[blockIdx.x + 1]];
  for (int64_t c0 = pb; c0 < pe; c0 += FB_2C_PCAP) {
    const int64_t slot = c0 + tid;
    double x = 0.0;
    int key = 0;
    if (slot < pe) {
      const int4 pr = v.pair_rec[slot];
      key = pr.w;
      const double *xlp = v.xl + (int64_t)pr.z * 3;
      for (int q = 0; q < 3; q++) {
        const double d = v.ratom[3 * pr.y + q] + xlp[q] - v.ratom[3 * pr.x + q];
        x = x + d * d;
      }
    }
    __syncthreads();   // the previous pass has read s_x
    s_x[tid] = x;
    s_k[tid] = key;
    __syncthreads();
    if (slot < pe) {
      const int g0 = tid & ~63;
      const int n = (int)min((int64_t)64, pe - (c0 + g0));
      int rank = 0;
      for (int j = 0; j < n; j++) {
        const double xj = s_x[g0 + j];
        const int kj = s_k[g0 + j];
        rank += (kj < key || (kj == key && (xj < x || (xj == x && g0 + j < tid)))) ? 1 : 0;
      }
      perm[c0 + g0 + rank] = (unsigned char)(tid & 63);
    }
  }
}

int fbk_pair_perm(const DView &v, unsigned char *perm, hipStream_t st) {
  if (v.nwg2c == 0) return 0;
  hipLaunchKernelGGL(k_pair_perm, dim3((unsigned)v.nwg2c), dim3(FB_2C_PCAP), 0, st, v, perm);
  return (int)hipGetLastError();
}

int fbk_block_sizes(const DView &v, int64_t *sz, int4 *rec, hipStream_t st) {
  if (v.npairs == 0) return 0;
  hipLaunchKernelGGL(k_block_sizes, dim3((unsigned)((v.npairs + 255) / 256)), dim3(256), 0, st, v, sz, rec);
  return (int)hipGetLastError();
}

// exclusive prefix sums (int -> int64 and int64 -> int64); out has n+1 entries
int fbk_scan_i32(const int *in, int64_t *out, int64_t n, void *tmp, size_t *tmp_bytes, hipStream_t st) {
  // out[0] = 0, out[i+1] = sum(in[0..i])
  if (tmp == nullptr) {
    return (int)hipcub::DeviceScan::InclusiveSum(nullptr, *tmp_bytes, in, out + 1, (int)n, st);
  }
  hipError_t e = hipMemsetAsync(out, 0, sizeof(int64_t), st);
  if (e != hipSuccess) return (int)e;
  if (n == 0) return 0;
  return (int)hipcub::DeviceScan::InclusiveSum(tmp, *tmp_bytes, in, out + 1, (int)n, st);
}

int fbk_scan_i64(const int64_t *in, int64_t *out, int64_t n, void *tmp, size_t *tmp_bytes, hipStream_t st) {
  if (tmp == nullptr) {
    return (int)hipcub::DeviceScan::InclusiveSum(nullptr, *tmp_bytes, in, out + 1, (int)n, st);
  }
  hipError_t e = hipMemsetAsync(out, 0, sizeof(int64_t), st);
  if (e != hipSuccess) return (int)e;
  if (n == 0) return 0;
  return (int)hipcub::DeviceScan::InclusiveSum(tmp, *tmp_bytes, in, out + 1, (int)n, st);
}

// stable sort of triplet ids by target pair; then segments
int fbk_sort_pairs(const int *keys_in, int *keys_out, const int *vals_in, int *vals_out, int64_t n, int end_bit,
                   void *tmp, size_t *tmp_bytes, hipStream_t st) {
  return (int)hipcub::DeviceRadixSort::SortPairs(tmp, *tmp_bytes, keys_in, keys_out, vals_in, vals_out, (int)n,
                                                 0, end_bit, st);
}

int fbk_scan_incl_i32(const int *in, int *out, int64_t n, void *tmp, size_t *tmp_bytes, hipStream_t st) {
  return (int)hipcub::DeviceScan::InclusiveSum(tmp, *tmp_bytes, in, out, (int)n, st);
}

int fbk_iota(int *a, int64_t n, hipStream_t st) {
  if (n == 0) return 0;
  hipLaunchKernelGGL(k_iota, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, a);
  return (int)hipGetLastError();
}

int fbk_seg_mark(int64_t ntrip, const int *sorted_pair, int *flag, hipStream_t st) {
  if (ntrip == 0) return 0;
  hipLaunchKernelGGL(k_seg_mark, dim3((unsigned)((ntrip + 255) / 256)), dim3(256), 0, st, ntrip, sorted_pair,
                     flag);
  return (int)hipGetLastError();
}

int fbk_seg_fill(int64_t ntrip, const int *sorted_pair, const int *segid_incl, int64_t *seg_off, int *seg_pair,
                 int *trip_seg, int *pair_tgt, hipStream_t st) {
  if (ntrip == 0) return 0;
  hipLaunchKernelGGL(k_seg_fill, dim3((unsigned)((ntrip + 255) / 256)), dim3(256), 0, st, ntrip, sorted_pair,
                     segid_incl, seg_off, seg_pair, trip_seg, pair_tgt);
  return (int)hipGetLastError();
}

int fbk_gather_trip(int64_t ntrip, const int *perm, const int4 *in, int4 *out, hipStream_t st) {
  if (ntrip == 0) return 0;
  hipLaunchKernelGGL(k_gather_trip, dim3((unsigned)((ntrip + 255) / 256)), dim3(256), 0, st, ntrip, perm, in,
                     out);
  return (int)hipGetLastError();
}

}  // extern "C"

__global__ void k_fill_i32(int64_t n, int *a, int val) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) a[t] = val;
}

extern "C" int fbk_fill_i32(int *a, int64_t n, int val, hipStream_t st) {
  if (n == 0) return 0;
  hipLaunchKernelGGL(k_fill_i32, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, a, val);
  return (int)hipGetLastError();
}

// species group (neutral bcna) and structure of every sorted triplet
__global__ void k_trip_aux(DView v, int *aux) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= v.ntrip) return;
  const int4 tr = v.trip[t];
  const int in1 = v.imass[tr.y], in2 = v.imass[tr.z], in3 = v.imass[tr.x];
  int gid = v.idx3c[(((in1 - 1) * v.sp.ns + (in2 - 1)) * v.sp.ns + (in3 - 1)) * FB_MAXSUB3];
  aux[t] = (gid < 0 ? 0xffff : gid) | (v.atom_struct[tr.x] << 16);
}

// segment ownership of every tile of ch consecutive sorted triplets: the
// segments that start inside the tile, and the triplets they span
extern "C" int fbk_trip_aux(const DView &v, int *aux, hipStream_t st) {
  if (v.ntrip == 0) return 0;
  hipLaunchKernelGGL(k_trip_aux, dim3((unsigned)((v.ntrip + 255) / 256)), dim3(256), 0, st, v, aux);
  return (int)hipGetLastError();
}

