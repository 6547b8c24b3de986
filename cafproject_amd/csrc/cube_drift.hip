/*
 * cube_drift.hip -- update_x (W/update_particle.f90:16-256) on the whole box.
 *
 * The reference drifts tile by tile over the tile's extended region
 * (physical + ncb buffer cells, whose particles are copies of neighbouring
 * tiles), counts particles into new cells (pass 1), builds prefix sums
 * (spine_tile), and scatters them (pass 2) in the visit order
 * (ilayer, k, j, i, l) with ilayer = (k-(1-ncb)) mod nlayer; only particles
 * landing in physical cells survive.  Both passes decode with the same
 * arithmetic, so a particle's new cell is fixed by the coordinates of the
 * copy that lands.
 *
 * Here there are no buffer copies.  Each particle evaluates, per axis, the
 * copies the reference would hold of it (home coordinate c, and c-nt in the
 * next tile if c>nt-ncb, and c+nt in the previous tile if c<=ncb), with the
 * reference's FP64 expression ceiling(xq+dt_mid*v/ncell) in each copy's own
 * tile frame, and keeps the copies that land in [1,nt] (normally exactly
 * one).  Its order inside the destination cell is the 64-bit key
 *   ilayer(9) | k_src-k_dst+2ncb (5) | j.. (5) | i.. (5) | particle index (40)
 * which, for a fixed destination cell, sorts exactly like (ilayer,k,j,i,l).
 * Counting (atomics on integers), an exclusive scan, atomic slot placement
 * and a per-cell sort of the keys give the reference order independently of
 * the atomics' timing; a per-cell pass then accumulates vfield_new in that
 * order (FP64 add, FP32 store, as the reference's real(4) vfield_new) and
 * re-quantises x and v.
 */
#include "cube_internal.h"
#include <math.h>
#include <stdlib.h>
#include <string.h>
#include <algorithm>

#define DT 256
static const double WEIGHT_V = (double)0.1f; /* real(8),parameter :: weight_v=0.1 */

enum { DERR_RANGE = 1, DERR_KEY = 2, DERR_XOVER = 8 };

/* ---------------- small utilities ---------------- */
__global__ void k_fill_i64(int64_t *p, int64_t n, int64_t v) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}
static int fill_i64(cube_ctx *c, int64_t *p, int64_t n, int64_t v) {
  hipLaunchKernelGGL(k_fill_i64, dim3(64), dim3(256), 0, c->stream, p, n, v);
  CUBE_LAUNCH_CHECK();
  return CUBE_OK;
}

/* decoded residual velocity table: vdec[code+nvbin/2] =
   tan(pi*real(code)/real(nvbin-1)) / (sqrt(pi/2)/(sigma*vrel_boost)) */
__global__ void k_vdec(const float *tanf_tab, double *vdec, int nv, double vc, unsigned long long *zero, int nz) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nv) vdec[i] = (double)tanf_tab[i] / vc;
  if (i < nz) zero[i] = 0ull;
}
/* the table, and nz words cleared in the same launch */
int cube_vdec_table(cube_ctx *c, double *dst, float sigma, unsigned long long *zero, int nz) {
  const int nv = c->nvbin;
  hipLaunchKernelGGL(k_vdec, dim3((nv + 255) / 256), dim3(256), 0, c->stream, c->tanf_tab, dst, nv,
                     cube_vconst(sigma), zero, nz);
  CUBE_LAUNCH_CHECK();
  return CUBE_OK;
}

/* ---------------- exclusive scan of int32 counts -> int64 ---------------- */
#define SCAN_B 1024
/* largest cell whose keys the drift's finalize pass ranks, and that one wave sorts */
#define FB_LDS_SORT 64
#define MED_SORT 1024
__global__ __launch_bounds__(SCAN_B) void k_scan_blocks(const int32_t *cnt, int64_t n, int64_t *bsum,
                                                        unsigned long long *ctr) {
  __shared__ int64_t s[SCAN_B];
  const int64_t i = blockIdx.x * (int64_t)SCAN_B + threadIdx.x;
  const int v = i < n ? cnt[i] : 0;
  s[threadIdx.x] = v;
  if (ctr) { /* cells that will be listed: big in ctr[5], medium in ctr[6] */
    const uint64_t big = __ballot(v > MED_SORT), med = __ballot(v > FB_LDS_SORT) & ~big;
    if ((threadIdx.x & 63) == 0) {
      if (big) atomicAdd(ctr + 5, (unsigned long long)__popcll(big));
      if (med) atomicAdd(ctr + 6, (unsigned long long)__popcll(med));
    }
  }
  __syncthreads();
  for (int o = SCAN_B / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) s[threadIdx.x] += s[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) bsum[blockIdx.x] = s[0];
}
__global__ __launch_bounds__(SCAN_B) void k_scan_partials(int64_t *bsum, int64_t nb, int64_t *total,
                                                          const unsigned long long *ctr, unsigned long long *hres) {
  /* exclusive scan of nb block sums, one block, chunked */
  __shared__ int64_t s[SCAN_B];
  __shared__ int64_t carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (int64_t base = 0; base < nb; base += SCAN_B) {
    const int64_t i = base + threadIdx.x;
    const int64_t v = i < nb ? bsum[i] : 0;
    s[threadIdx.x] = v;
    __syncthreads();
    for (int o = 1; o < SCAN_B; o <<= 1) {
      const int64_t t = threadIdx.x >= o ? s[threadIdx.x - o] : 0;
      __syncthreads();
      s[threadIdx.x] += t;
      __syncthreads();
    }
    if (i < nb) bsum[i] = carry + s[threadIdx.x] - v;
    __syncthreads();
    if (threadIdx.x == SCAN_B - 1) carry += s[SCAN_B - 1];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    *total = carry;
    hres[HR_TOTAL] = (unsigned long long)carry;
  }
  if (ctr && threadIdx.x < 8) hres[HR_CTR + threadIdx.x] = ctr[threadIdx.x];
}
__global__ __launch_bounds__(SCAN_B) void k_scan_final(const int32_t *cnt, int64_t n, const int64_t *boff,
                                                     int64_t *start, const int64_t *total) {
  __shared__ int64_t s[SCAN_B];
  const int64_t i = blockIdx.x * (int64_t)SCAN_B + threadIdx.x;
  const int64_t v = i < n ? cnt[i] : 0;
  s[threadIdx.x] = v;
  __syncthreads();
  for (int o = 1; o < SCAN_B; o <<= 1) {
    const int64_t t = threadIdx.x >= o ? s[threadIdx.x - o] : 0;
    __syncthreads();
    s[threadIdx.x] += t;
    __syncthreads();
  }
  if (i < n) start[i] = boff[blockIdx.x] + s[threadIdx.x] - v;
  if (i == n - 1) start[n] = *total;
}
int cube_scan_counts(cube_ctx *c, const int32_t *cnt, int64_t *start, int64_t n, int64_t *total,
                     unsigned long long *ctr) {
  const int64_t nb = (n + SCAN_B - 1) / SCAN_B;
  int64_t *bsum = c->scanbuf;   /* nb + 1 entries */
  int64_t *tot = c->scanbuf + nb;
  hipLaunchKernelGGL(k_scan_blocks, dim3((unsigned)nb), dim3(SCAN_B), 0, c->stream, cnt, n, bsum, ctr);
  CUBE_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_scan_partials, dim3(1), dim3(SCAN_B), 0, c->stream, bsum, nb, tot, (const unsigned long long *)ctr,
                     c->hres);
  CUBE_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_scan_final, dim3((unsigned)nb), dim3(SCAN_B), 0, c->stream, cnt, n, bsum, start, tot);
  CUBE_LAUNCH_CHECK();
  CUBE_CHECK(hipStreamSynchronize(c->stream));
  if (total) *total = (int64_t)c->hres[HR_TOTAL];
  return CUBE_OK;
}

/* ---------------- per-tile sums over the extended box ---------------- */
/* particles of local cells [1-w, nt+w]^3 of tile t (periodic): a row of the
   box is a run of cells in each tile it crosses, so its sum is a difference of
   their starts.  BOX_WG workgroups share a tile's rows, the host adds their
   sums.  Latency bound: 4 us for small tiles, 9 for 8 of 128^3, where
   reading the cells' counts took 28 us on 8 tiles of 16^3 cells (784 rows of
   28 cells each, w = 6) and 83 us on 8 of 128^3 */
__global__ __launch_bounds__(256) void k_tile_boxsum(const int64_t *__restrict__ cstart, Geo g, int w,
                                                     int64_t *__restrict__ out) {
  const int t = blockIdx.y, nt = g.nt, e = nt + 2 * w;
  const int tz = t / (g.nnt * g.nnt), ty = (t / g.nnt) % g.nnt, tx = t % g.nnt;
  const int dn = (w + nt - 1) / nt; /* tiles the box reaches into on a side */
  int64_t s = 0;
  for (int q = blockIdx.x * 256 + threadIdx.x; q < e * e; q += BOX_WG * 256) {
    const int j = q % e - w, k = q / e - w;
    for (int d = -dn; d <= dn; ++d) { /* its part in tile tx + d: cells [i0, i1) of that tile */
      const int i0 = max(-w - d * nt, 0), i1 = min(nt + w - d * nt, nt);
      const int64_t row = cid_global(g, (tx + d) * nt, ty * nt + j, tz * nt + k);
      s += cstart[row + i1] - cstart[row + i0];
    }
  }
  __shared__ int64_t r[256];
  r[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) r[threadIdx.x] += r[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[t * BOX_WG + blockIdx.x] = r[0];
}
int cube_tile_boxsum(cube_ctx *c, int w, int64_t *host_out) {
  hipLaunchKernelGGL(k_tile_boxsum, dim3(BOX_WG, (unsigned)c->ntiles), dim3(256), 0, c->stream, c->cstart, geo_of(c), w,
                     (int64_t *)c->hres + HR_BOX);
  CUBE_LAUNCH_CHECK();
  CUBE_CHECK(hipStreamSynchronize(c->stream));
  const int64_t *part = (const int64_t *)c->hres + HR_BOX;
  for (int64_t t = 0; t < c->ntiles; ++t) {
    host_out[t] = 0;
    for (int b = 0; b < BOX_WG; ++b) host_out[t] += part[t * BOX_WG + b];
  }
  return CUBE_OK;
}

/* ---------------- pass 1: destination cell and order key ---------------- */
/* three interleaved components, read with one 12-byte load */
struct V3f {
  float x, y, z;
};

struct DriftP {
  Geo g;
  int nlayer;
  int nvh;        /* nvbin/2 */
  float dt_mid;
  double xres;
  double inv_xres4; /* 1/(xres*ncell), a power of two: multiplying by it is the division, exactly */
  int agg_cap;    /* largest row (particles) whose slots are aggregated in LDS */
};
#define AGG_CAP 4096

template <int IX, int IV>
__global__ __launch_bounds__(DT) void k_drift_dest(const typename IntOf<IX>::T *__restrict__ xp,
                                                   const typename IntOf<IV>::T *__restrict__ vp,
                                                   const float *__restrict__ vfield,
                                                   const int64_t *__restrict__ cstart,
                                                   const double *__restrict__ vdec, DriftP P,
                                                   int32_t *__restrict__ dest, uint64_t *__restrict__ key,
                                                   int32_t *__restrict__ cnt, int32_t *__restrict__ rank,
                                                   int32_t *__restrict__ xdest, uint64_t *__restrict__ xkey,
                                                   int32_t *__restrict__ xrank, int64_t xcap,
                                                   unsigned long long *__restrict__ counters) {
  /* counters: [0] extra copies, [1] lost, [2] error flags */
  const Geo g = P.g;
  const int nt = g.nt, ncb = g.ncb;
  const int64_t row = blockIdx.x;               /* j + nt*(k + nt*t) */
  const int j = (int)(row % nt), k = (int)((row / nt) % nt), t = (int)(row / ((int64_t)nt * nt));
  const int tz = t / (g.nnt * g.nnt), ty = (t / g.nnt) % g.nnt, tx = t % g.nnt;
  __shared__ int64_t cs[520];
  /* Slots inside destination cells: a main copy landing in the 3x3 rows of
     cells around this row (same tile) takes a local rank from an LDS
     counter, and each such cell then reserves its range with one global
     atomic; other copies take their slot with a global atomic directly. */
  extern __shared__ int dyn[];
  const int nwin = 9 * nt;
  int *lcnt = dyn;               /* nwin counters, then the reserved bases */
  /* per particle of the row: window cell << 19 | local rank, or ~0u */
  uint32_t *pslot = reinterpret_cast<uint32_t *>(dyn + nwin);
  const int64_t c0 = row * nt;
  for (int i = threadIdx.x; i <= nt; i += DT) cs[i] = cstart[c0 + i];
  for (int i = threadIdx.x; i < nwin; i += DT) lcnt[i] = 0;
  __syncthreads();
  const int64_t pbeg = cs[0], pend = cs[nt];
  const bool agg = pend - pbeg <= P.agg_cap;   /* uniform over the block */
  if (agg) { /* pslot first holds each particle's cell of the row */
    for (int c = threadIdx.x; c < nt; c += DT)
      for (int64_t q = cs[c]; q < cs[c + 1]; ++q) pslot[q - pbeg] = (uint32_t)c;
    __syncthreads();
  }
  for (int64_t p = pbeg + threadIdx.x; p < pend; p += DT) {
    /* cell of p: largest i with cs[i] <= p */
    int lo = 0, hi = nt;
    if (agg) {
      lo = (int)pslot[p - pbeg];
      pslot[p - pbeg] = ~0u;
    } else {
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (cs[mid] <= p) lo = mid; else hi = mid;
      }
    }
    const int i = lo;
    const int home[3] = {i + 1, j + 1, k + 1};   /* 1-based tile-local */
    const int tile[3] = {tx, ty, tz};
    int lcoord[3][3], lig[3][3], loff[3][3], nl[3];
    int err = 0;
    const V3f vcell = *reinterpret_cast<const V3f *>(vfield + 3 * (c0 + i)); /* one 12-byte load */
    const float vcf[3] = {vcell.x, vcell.y, vcell.z};
    int32_t xcode[3], vcode[3];
    code_split<IX>(code_word<IX>(xp, p), xcode);
    code_split<IV>(code_word<IV>(vp, p), vcode);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const int32_t xc = xcode[a];
      const int32_t vc = (int32_t)(typename IntOf<IV>::T)vcode[a];
      const double off = ((double)cube_ucode(IX, xc) + 0.5) * P.xres;
      const double vreal = vdec[vc + P.nvh] + (double)vcf[a];
      const double dx = ((double)P.dt_mid * vreal) / 4.0;
      nl[a] = 0;
      int cand[3] = {home[a], 0, 0}, coff[3] = {0, 0, 0}, nc = 1;
      if (home[a] >= nt - ncb + 1) { cand[nc] = home[a] - nt; coff[nc] = 1; ++nc; }
      if (home[a] <= ncb) { cand[nc] = home[a] + nt; coff[nc] = -1; ++nc; }
      for (int q = 0; q < nc; ++q) {
        const double xq = ((double)cand[q] - 1.0) + off;
        const double ig = ceil(xq + dx);
        if (ig < 1 - 2 * ncb || ig > nt + 2 * ncb) { err |= DERR_RANGE; continue; }
        const int igi = (int)ig;
        if (igi >= 1 && igi <= nt) {
          lcoord[a][nl[a]] = cand[q];
          lig[a][nl[a]] = igi;
          loff[a][nl[a]] = coff[q];
          ++nl[a];
        }
      }
    }
    const int ncopy = nl[0] * nl[1] * nl[2];
    if (ncopy == 0) {
      dest[p] = -1;
      atomicAdd(counters + 1, 1ull);
    }
    int w = 0;
    for (int qz = 0; qz < nl[2]; ++qz)
      for (int qy = 0; qy < nl[1]; ++qy)
        for (int qx = 0; qx < nl[0]; ++qx, ++w) {
          const int q[3] = {qx, qy, qz};
          int dt_[3], r[3];
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            dt_[a] = wrapi(tile[a] + loff[a][q[a]], g.nnt);
            r[a] = lcoord[a][q[a]] - lig[a][q[a]] + 2 * ncb;
            if (r[a] < 0 || r[a] > 31) err |= DERR_KEY;
          }
          const int il = (lcoord[2][qz] - (1 - ncb)) % P.nlayer;
          const int32_t dc = (int32_t)g.cid(lig[0][qx] - 1, lig[1][qy] - 1, lig[2][qz] - 1,
                                            dt_[0] + g.nnt * (dt_[1] + g.nnt * dt_[2]));
          const uint64_t kk = ((uint64_t)il << 55) | ((uint64_t)(r[2] & 31) << 50) |
                              ((uint64_t)(r[1] & 31) << 45) | ((uint64_t)(r[0] & 31) << 40) | (uint64_t)p;
          /* slots are taken in arrival order; the per-cell sort restores
             the reference order */
          if (w == 0) {
            dest[p] = dc;
            key[p] = kk;
            const int ddy = lig[1][qy] - 1 - j, ddz = lig[2][qz] - 1 - k;
            if (agg && dt_[0] == tx && dt_[1] == ty && dt_[2] == tz && ddy >= -1 && ddy <= 1 && ddz >= -1 &&
                ddz <= 1) {
              const int wi = ((ddz + 1) * 3 + (ddy + 1)) * nt + (lig[0][qx] - 1);
              const int lr = atomicAdd(lcnt + wi, 1);
              pslot[p - pbeg] = ((uint32_t)wi << 19) | (uint32_t)lr;
            } else {
              rank[p] = atomicAdd(cnt + dc, 1);
            }
          } else {
            const unsigned long long x = atomicAdd(counters + 0, 1ull);
            if ((int64_t)x < xcap) {
              xdest[x] = dc;
              xkey[x] = kk;
              xrank[x] = atomicAdd(cnt + dc, 1);
            } else {
              err |= DERR_XOVER;
            }
          }
        }
    if (err) atomicOr(counters + 2, (unsigned long long)err);
  }
  if (!agg) return; /* uniform */
  __syncthreads();
  /* reserve each window cell's range: one global atomic per cell */
  for (int wi = threadIdx.x; wi < nwin; wi += DT) {
    const int n = lcnt[wi];
    if (n > 0) {
      const int y = j + (wi / nt) % 3 - 1, z = k + (wi / nt) / 3 - 1;
      lcnt[wi] = atomicAdd(cnt + g.cid(wi % nt, y, z, t), n);
    }
  }
  __syncthreads();
  for (int64_t p = pbeg + threadIdx.x; p < pend; p += DT) {
    const uint32_t s = pslot[p - pbeg];
    if (s != ~0u) rank[p] = lcnt[s >> 19] + (int)(s & 0x7ffffu);
  }
}

/* ---------------- per-cell sort ---------------- */
#define BIG_SORT 16384
#define FB_CELLS 64      /* cells per finalize workgroup (the context sizes vpart for it) */
/* slots staged in LDS at once: an average workgroup's 512 and a quarter more, so
   that most go through their cells in one run; one with more takes runs of at
   most that many.  23.4 KB, 6 finalize workgroups a CU, which does not bind:
   their 93 registers allow 5 */
#define FB_CH 640
/* cells above FB_LDS_SORT, for the sorts of their own: big ones (above
   MED_SORT) from the front of the list, counted in counters[3], the others
   from its back, counted in counters[4] */
__device__ __forceinline__ void list_cell(int64_t c, int n, int64_t ncells, int32_t *__restrict__ list,
                                          unsigned long long *__restrict__ counters) {
  if (n > MED_SORT)
    list[atomicAdd(counters + 3, 1ull)] = (int32_t)c;
  else if (n > FB_LDS_SORT)
    list[ncells - 1 - (int64_t)atomicAdd(counters + 4, 1ull)] = (int32_t)c;
}
/* scatter to the slot taken at counting time: no second round of atomics; and
   (cnt given) the list of the cells that the finalize pass does not sort */
__global__ __launch_bounds__(256) void k_place_ranked(const int32_t *__restrict__ dest, const int32_t *__restrict__ rank,
                                                      const uint64_t *__restrict__ key, int64_t n,
                                                      const int64_t *__restrict__ start, uint64_t *__restrict__ out,
                                                      const int32_t *__restrict__ cnt, int64_t ncells,
                                                      int32_t *__restrict__ list,
                                                      unsigned long long *__restrict__ counters) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, nthr = (int64_t)gridDim.x * blockDim.x;
  if (cnt)
    for (int64_t c = t; c < ncells; c += nthr) list_cell(c, cnt[c], ncells, list, counters);
  for (int64_t p = t; p < n; p += nthr) {
    const int32_t d = dest[p];
    if (d < 0) continue;
    out[start[d] + rank[p]] = key[p];
  }
}
/* cells c_lo.. of a workgroup's ncl whose slots fit in FB_CH, at least one
   (the same in every wave); returns the cell past them */
__device__ __forceinline__ int seg_end(const int64_t *cst, int ncl, int c_lo) {
  const int c = c_lo + 1 + (int)(threadIdx.x & 63);
  return c_lo + max(1, (int)__popcll(__ballot(c <= ncl && cst[min(c, ncl)] - cst[c_lo] <= FB_CH)));
}
/* The keys of cells [c_lo, c_hi), which fit, into pix in order, with their
   cells in lcell.  A key's place in its cell is the number of smaller keys
   there (unique: they carry the particle index): every lane ranks its own
   slots at once instead of one lane per cell sorting serially.  Cells above
   FB_LDS_SORT come sorted (or, in k_sort_cells, are left to be). */
__device__ __forceinline__ void seg_sort(const uint64_t *__restrict__ keys, const int64_t *cst, int c_lo, int c_hi,
                                         uint64_t *pix, uint8_t *lcell) {
  const int tid = threadIdx.x;
  const int64_t s0 = cst[c_lo];
  const int n = (int)(cst[c_hi] - s0);
  for (int q = tid; q < n; q += 256) pix[q] = keys[s0 + q];
  if (c_lo + tid < c_hi) {
    const int lo = (int)(cst[c_lo + tid] - s0), hi = (int)(cst[c_lo + tid + 1] - s0);
    for (int q = lo; q < hi; ++q) lcell[q] = (uint8_t)(c_lo + tid);
  }
  __syncthreads();
  constexpr int PER = (FB_CH + 255) / 256;
  uint64_t kx[PER];
  int dst[PER];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int q = tid + 256 * u;
    dst[u] = -1;
    if (q < n) {
      const int c = lcell[q], lo = (int)(cst[c] - s0), hi = (int)(cst[c + 1] - s0);
      if (hi - lo <= FB_LDS_SORT) {
        const uint64_t x = pix[q];
        int r = 0;
        for (int w = lo; w < hi; ++w) r += pix[w] < x ? 1 : 0;
        kx[u] = x;
        dst[u] = lo + r;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < PER; ++u)
    if (dst[u] >= 0) pix[dst[u]] = kx[u];
  __syncthreads();
}
/* the keys of every cell up to FB_LDS_SORT in order, the others listed */
__global__ __launch_bounds__(256) void k_sort_cells(const int32_t *__restrict__ cnt, const int64_t *__restrict__ start,
                                                    int64_t ncells, uint64_t *__restrict__ keys, int32_t *__restrict__ list,
                                                    unsigned long long *__restrict__ counters) {
  __shared__ int64_t cst[FB_CELLS + 1];
  __shared__ uint64_t pix[FB_CH];
  __shared__ uint8_t lcell[FB_CH];
  const int tid = threadIdx.x;
  const int64_t c0 = (int64_t)blockIdx.x * FB_CELLS;
  const int ncl = (int)min((int64_t)FB_CELLS, ncells - c0);
  for (int i = tid; i <= ncl; i += 256) cst[i] = start[c0 + i];
  if (tid < ncl) list_cell(c0 + tid, cnt[c0 + tid], ncells, list, counters);
  __syncthreads();
  for (int c_lo = 0; c_lo < ncl;) {
    const int c_hi = seg_end(cst, ncl, c_lo);
    const int64_t s0 = cst[c_lo];
    const int n = (int)min(cst[c_hi] - s0, (int64_t)FB_CH + 1);
    if (n <= FB_CH) { /* uniform; else one crowded cell */
      seg_sort(keys, cst, c_lo, c_hi, pix, lcell);
      for (int q = tid; q < n; q += 256) keys[s0 + q] = pix[q];
      __syncthreads();
    }
    c_lo = c_hi;
  }
}

/* bitonic sort of sk[0..m) in LDS, m a power of two */
__device__ static void lds_bitonic(uint64_t *sk, int m) {
  for (int size = 2; size <= m; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int q = threadIdx.x; q < m; q += blockDim.x) {
        const int o = q ^ stride;
        if (o > q) {
          const bool up = (q & size) == 0;
          const uint64_t x = sk[q], y = sk[o];
          if ((x > y) == up) {
            sk[q] = y;
            sk[o] = x;
          }
        }
      }
      __syncthreads();
    }
}
/* number of elements of the ascending run r[0..n) below x */
__device__ static int lower_bound_u64(const uint64_t *r, int n, uint64_t x) {
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (r[mid] < x) lo = mid + 1; else hi = mid;
  }
  return lo;
}

/* One wave per medium cell (FB_LDS_SORT < n <= MED_SORT), four per
   workgroup, on a fixed grid (the count stays on the device): a bitonic sort of the cell's keys (padded to a power of two,
   at least 64) in the wave's 8 KB of LDS, the stages ordered by the wave
   itself -- no workgroup barriers, and 32 KB per workgroup so that five
   share a CU where a big cell's workgroup takes 128 KB. */
__global__ __launch_bounds__(256) void k_sort_med(const int32_t *__restrict__ cnt, const int64_t *__restrict__ start,
                                                  const int32_t *__restrict__ list, int64_t ncells,
                                                  const unsigned long long *__restrict__ counters,
                                                  uint64_t *__restrict__ a) {
  __shared__ uint64_t sm[4 * MED_SORT];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  uint64_t *sk = sm + wv * MED_SORT;
  const int64_t nlist = (int64_t)counters[4];
  for (int64_t i = (int64_t)blockIdx.x * 4 + wv; i < nlist; i += (int64_t)gridDim.x * 4) {
    const int32_t cidx = list[ncells - 1 - i];
    const int n = cnt[cidx];
    uint64_t *s = a + start[cidx];
    int m = 64;
    while (m < n) m <<= 1;
    for (int q = lane; q < m; q += 64) sk[q] = q < n ? s[q] : ~0ull;
    for (int size = 2; size <= m; size <<= 1)
      for (int stride = size >> 1; stride > 0; stride >>= 1) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        for (int q = lane; q < m; q += 64) { /* each pair (q, q^stride) has one owner */
          const int o = q ^ stride;
          if (o > q) {
            const bool up = (q & size) == 0;
            const uint64_t x = sk[q], y = sk[o];
            if ((x > y) == up) {
              sk[q] = y;
              sk[o] = x;
            }
          }
        }
      }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int q = lane; q < n; q += 64) s[q] = sk[q];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); /* the next cell's keys overwrite these */
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

/* One workgroup per big cell at a time, on a fixed grid.  Up to BIG_SORT keys: a bitonic sort in LDS.
   Larger cells (a collapsed halo core can hold more particles than LDS
   takes): BIG_SORT-key runs sorted in LDS, then pairwise merges of runs in
   global memory between the cell's segment and the same range of tmp (the
   placement keys, dead by now).  Keys within a cell are distinct (the low
   bits are the particle index), so an element's merged position is its
   index in its run plus its rank in the other run. */
__global__ __launch_bounds__(1024) void k_sort_big(const int32_t *__restrict__ cnt,
                                                   const int64_t *__restrict__ start,
                                                   const int32_t *__restrict__ biglist,
                                                   const unsigned long long *__restrict__ counters,
                                                   uint64_t *__restrict__ a, uint64_t *__restrict__ tmp) {
  extern __shared__ uint64_t sk[];
  const int64_t nlist = (int64_t)counters[3];
  for (int64_t i = blockIdx.x; i < nlist; i += gridDim.x) {
    const int32_t cidx = biglist[i];
    const int n = cnt[cidx];
    uint64_t *s = a + start[cidx];
    if (n <= BIG_SORT) {
      int m = 1;
      while (m < n) m <<= 1;
      for (int q = threadIdx.x; q < m; q += blockDim.x) sk[q] = q < n ? s[q] : ~0ull;
      __syncthreads();
      lds_bitonic(sk, m);
      for (int q = threadIdx.x; q < n; q += blockDim.x) s[q] = sk[q];
      __syncthreads();
      continue;
    }
    for (int c0 = 0; c0 < n; c0 += BIG_SORT) {
      const int len = min(BIG_SORT, n - c0);
      for (int q = threadIdx.x; q < BIG_SORT; q += blockDim.x) sk[q] = q < len ? s[c0 + q] : ~0ull;
      __syncthreads();
      lds_bitonic(sk, BIG_SORT);
      for (int q = threadIdx.x; q < len; q += blockDim.x) s[c0 + q] = sk[q];
      __syncthreads();
    }
    uint64_t *src = s, *dst = tmp + start[cidx];
    for (int w = BIG_SORT; w < n; w <<= 1) {
      for (int lo = 0; lo < n; lo += 2 * w) {
        const int mid = min(lo + w, n), hi = min(lo + 2 * w, n);
        for (int q = lo + (int)threadIdx.x; q < hi; q += blockDim.x) {
          const uint64_t x = src[q];
          const int pos = q < mid ? (q - lo) + lower_bound_u64(src + mid, hi - mid, x)
                                  : (q - mid) + lower_bound_u64(src + lo, mid - lo, x);
          dst[lo + pos] = x;
        }
      }
      __syncthreads();
      uint64_t *t = src;
      src = dst;
      dst = t;
    }
    if (src != s) {
      for (int q = threadIdx.x; q < n; q += blockDim.x) s[q] = src[q];
    }
    __syncthreads();
  }
}

/* ---------------- per-cell finalize ---------------- */
/*
 * Finalize by slot ranges: a workgroup owns FB_CELLS consecutive new cells
 * and the contiguous slot range of their particles, and goes through them in
 * runs of whole cells of at most FB_CH slots.  A run's keys are put in order
 * in LDS, lanes gather the decoded velocities of consecutive slots (one lane
 * per slot), one thread per cell then accumulates vfield_new serially in slot
 * order (the reference's order), and lanes write the re-quantised x, v and pid
 * of consecutive slots, so the stores are coalesced.  A cell above FB_CH is a
 * run of its own in pieces, all gathered for the sum and again for the stores.
 * Ranking every cell up to FB_LDS_SORT here replaced a lane per cell sorting in
 * scratch memory where a workgroup's cells did not fit in one run: with the
 * flags and the count read back 15 + 8 us on 16^3 cells, 113 us on 48^3 and 610
 * us on 128^3 at 16 particles a cell, against nothing but this kernel's own 21
 * -> 23, 54 -> 58 and 780 -> 820 us.  The velocity statistics
 * of the new state (W/update_particle.f90:172-224) are reduced on the way:
 * per workgroup in a fixed tree, then over workgroups in order.
 */
template <int IX, int IV>
__global__ __launch_bounds__(256) void k_drift_final2(
    const typename IntOf<IX>::T *__restrict__ xp, const typename IntOf<IV>::T *__restrict__ vp,
    const int32_t *__restrict__ pid, const float *__restrict__ vfield_old, const int64_t *__restrict__ start,
    const uint64_t *__restrict__ keys, const double *__restrict__ vdec, DriftP P, double venc,
    typename IntOf<IX>::T *__restrict__ xp2, typename IntOf<IV>::T *__restrict__ vp2,
    int32_t *__restrict__ pid2, float *__restrict__ vfield_new, int64_t ncells, double *__restrict__ part) {
  __shared__ int64_t cst[FB_CELLS + 1];
  __shared__ double vr[FB_CH][3]; /* decoded velocities; the final reduction reuses it */
  __shared__ uint64_t pix[FB_CH]; /* sorted keys, then source particle indices */
  __shared__ uint8_t lcell[FB_CH]; /* slot -> local cell */
  __shared__ int cgeo[FB_CELLS][4]; /* local i, j, k and tile of each cell */
  __shared__ float vn[FB_CELLS][3];
  const Geo g = P.g;
  const int nt = g.nt, ncb = g.ncb, tid = threadIdx.x;
  const int64_t c0 = (int64_t)blockIdx.x * FB_CELLS;
  const int ncl = (int)min((int64_t)FB_CELLS, ncells - c0);
  for (int i = tid; i <= ncl; i += 256) cst[i] = start[c0 + i];
  if (tid < ncl) {
    const int64_t cidx = c0 + tid;
    cgeo[tid][0] = (int)(cidx % nt);
    cgeo[tid][1] = (int)((cidx / nt) % nt);
    cgeo[tid][2] = (int)((cidx / ((int64_t)nt * nt)) % nt);
    cgeo[tid][3] = (int)(cidx / ((int64_t)nt * nt * nt));
  }
  __syncthreads();
  const int64_t S0 = cst[0];
  /* vfield_new: thread (component aa, cell ca) sums its cell's slots in
     slot order -- three independent serial chains per cell, so a crowded
     cell holds its workgroup a third as long */
  const int ca = tid & 63, aa = tid >> 6;
  double sr = 0, ss = 0;
  for (int c_lo = 0; c_lo < ncl;) {
    const int c_hi = seg_end(cst, ncl, c_lo);
    const int64_t s0 = cst[c_lo], s1 = cst[c_hi];
    const int np = max(1, (int)((s1 - s0 + FB_CH - 1) / FB_CH)), rounds = np > 1 ? 2 * np : 1; /* uniform */
    const bool accum = aa < 3 && ca >= c_lo && ca < c_hi;
    float acc = 0.f;
    if (accum) acc = (float)((double)vfield_old[3 * (c0 + ca) + aa] * WEIGHT_V);
#pragma unroll 1
    for (int u = 0; u < rounds; ++u) {
      const int64_t ch = s0 + (int64_t)(u < np ? u : u - np) * FB_CH, ce = min(ch + FB_CH, s1);
      /* slot s always belongs to the same lane: the sums' order */
      const int first = (tid - (int)(ch - S0)) & 255;
      if (np == 1) {
        seg_sort(keys, cst, c_lo, c_hi, pix, lcell);
      } else {
        for (int64_t s = ch + tid; s < ce; s += 256) {
          pix[s - ch] = keys[s];
          lcell[s - ch] = (uint8_t)c_lo;
        }
        __syncthreads();
      }
#pragma unroll 1
      for (int q = tid; q < (int)(ce - ch); q += 256) {
        const int lc = lcell[q], i = cgeo[lc][0], j = cgeo[lc][1], k = cgeo[lc][2], t = cgeo[lc][3];
        const uint64_t kk = pix[q];
        const int64_t p = (int64_t)(kk & KEY_PMASK);
        const int rx = (int)((kk >> 40) & 31), ry = (int)((kk >> 45) & 31), rz = (int)((kk >> 50) & 31);
        /* source cell = destination + (r - 2ncb), in the destination tile frame */
        const int sx = i + rx - 2 * ncb, sy = j + ry - 2 * ncb, sz = k + rz - 2 * ncb;
        int64_t sc;
        if (sx >= 0 && sx < nt && sy >= 0 && sy < nt && sz >= 0 && sz < nt) {
          sc = g.cid(sx, sy, sz, t);
        } else {
          const int tz = t / (g.nnt * g.nnt), ty = (t / g.nnt) % g.nnt, tx = t % g.nnt;
          sc = cid_global(g, tx * nt + sx, ty * nt + sy, tz * nt + sz);
        }
        const V3f vo = *reinterpret_cast<const V3f *>(vfield_old + 3 * sc); /* one 12-byte load */
        const float vof[3] = {vo.x, vo.y, vo.z};
        int32_t vcode[3];
        code_split<IV>(code_word<IV>(vp, p), vcode);
#pragma unroll
        for (int a = 0; a < 3; ++a)
          vr[q][a] = vdec[(int32_t)(typename IntOf<IV>::T)vcode[a] + P.nvh] + (double)vof[a];
        pix[q] = (uint64_t)p;
      }
      __syncthreads();
      if (u < np) { /* uniform */
        if (accum) {
          const int lo = (int)(max(cst[ca], ch) - ch), hi = (int)(min(cst[ca + 1], ce) - ch);
          for (int q = lo; q < hi; ++q) acc = (float)((double)acc + vr[q][aa]);
          if (u == np - 1) {
            const double n = (double)(cst[ca + 1] - cst[ca]);
            vn[ca][aa] = (float)((double)acc / (n + WEIGHT_V));
            vfield_new[3 * (c0 + ca) + aa] = vn[ca][aa];
          }
        }
        __syncthreads();
      }
      if (np == 1 || u >= np) {
#pragma unroll 1
        for (int q = first; q < (int)(ce - ch); q += 256) {
          const int lc = lcell[q];
          const int64_t p = (int64_t)pix[q], s = ch + q;
          const double vres[3] = {vr[q][0] - (double)vn[lc][0], vr[q][1] - (double)vn[lc][1],
                                  vr[q][2] - (double)vn[lc][2]};
          /* vp_new=nint(...atan(...*(vreal-vfield_new))...) (:116-117) */
          int32_t code[3];
          cube_encode_v3(IV, venc, vres, code);
          int32_t xcode[3];
          code_split<IX>(code_word<IX>(xp, p), xcode);
          double r[3];
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            /* xp_new=xp+nint(dt_mid*vreal/(x_resolution*ncell)) (:115) */
            const double qx = ((double)P.dt_mid * vr[q][a]) * P.inv_xres4;
            xp2[3 * s + a] = (typename IntOf<IX>::T)cube_wrap(IX, (int64_t)xcode[a] + (int64_t)cube_nint(qx)); /* modulo 2^8izipx */
            vp2[3 * s + a] = (typename IntOf<IV>::T)code[a];
            r[a] = vdec[code[a] + P.nvh];
          }
          if (pid) pid2[s] = pid[p];
          sr += (r[0] * r[0] + r[1] * r[1]) + r[2] * r[2];
          r[0] += (double)vn[lc][0];
          r[1] += (double)vn[lc][1];
          r[2] += (double)vn[lc][2];
          ss += (r[0] * r[0] + r[1] * r[1]) + r[2] * r[2];
        }
      }
      __syncthreads();
    }
    c_lo = c_hi;
  }
  double sc = 0;
  if (tid < ncl) {
    const float v0 = vn[tid][0], v1 = vn[tid][1], v2 = vn[tid][2];
    sc = (double)((v0 * v0 + v1 * v1) + v2 * v2);
  }
  /* vr is free: reduce through it */
  double(*red)[256] = reinterpret_cast<double(*)[256]>(&vr[0][0]);
  red[0][tid] = sc;
  red[1][tid] = sr;
  red[2][tid] = ss;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (tid < o)
      for (int a = 0; a < 3; ++a) red[a][tid] += red[a][tid + o];
    __syncthreads();
  }
  if (tid < 3) part[3 * blockIdx.x + tid] = red[tid][0];
}

/* fixed-order sum of nb triples: thread t sums a contiguous run of blocks,
   then a tree over the threads */
__global__ __launch_bounds__(1024) void k_sum_parts_tree(const double *__restrict__ part, int64_t nb,
                                                         double *__restrict__ out) {
  __shared__ double red[3][1024];
  const int t = threadIdx.x;
  /* thread t sums the partials b = t mod 1024 (a fixed order, so the sums
     repeat bit for bit; neighbouring lanes read neighbouring partials) */
  double s[3] = {0, 0, 0};
  for (int64_t b = t; b < nb; b += 1024)
#pragma unroll
    for (int a = 0; a < 3; ++a) s[a] += part[3 * b + a];
  for (int a = 0; a < 3; ++a) red[a][t] = s[a];
  __syncthreads();
  for (int o = 512; o > 0; o >>= 1) {
    if (t < o)
      for (int a = 0; a < 3; ++a) red[a][t] += red[a][t + o];
    __syncthreads();
  }
  if (t < 3) out[t] = red[t][0];
}

/* ---------------- velocity statistics (:172-224) ---------------- */
#define VS_BLOCKS 1024
template <int IV>
__global__ __launch_bounds__(256) void k_vstats(const typename IntOf<IV>::T *__restrict__ vp,
                                                const float *__restrict__ vfield, const int32_t *__restrict__ cnt,
                                                const int64_t *__restrict__ start, const double *__restrict__ vdec,
                                                int nvh, int64_t ncells, double *__restrict__ part) {
  double sc = 0, sr = 0, ss = 0;
  for (int64_t cidx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; cidx < ncells;
       cidx += (int64_t)gridDim.x * blockDim.x) {
    const float v0 = vfield[3 * cidx], v1 = vfield[3 * cidx + 1], v2 = vfield[3 * cidx + 2];
    sc += (double)((v0 * v0 + v1 * v1) + v2 * v2);
    const int n = cnt[cidx];
    const int64_t s0 = start[cidx];
    for (int q = 0; q < n; ++q) {
      double r[3];
#pragma unroll
      for (int a = 0; a < 3; ++a) r[a] = vdec[(int32_t)vp[3 * (s0 + q) + a] + nvh];
      sr += (r[0] * r[0] + r[1] * r[1]) + r[2] * r[2];
      r[0] += (double)v0;
      r[1] += (double)v1;
      r[2] += (double)v2;
      ss += (r[0] * r[0] + r[1] * r[1]) + r[2] * r[2];
    }
  }
  __shared__ double red[3][256];
  red[0][threadIdx.x] = sc;
  red[1][threadIdx.x] = sr;
  red[2][threadIdx.x] = ss;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o)
      for (int a = 0; a < 3; ++a) red[a][threadIdx.x] += red[a][threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x < 3) part[3 * blockIdx.x + threadIdx.x] = red[threadIdx.x][0];
}
__global__ void k_sum_parts(const double *part, int nb, double *out) {
  /* fixed-order final sum of the block partials */
  if (threadIdx.x < 3) {
    double s = 0;
    for (int b = 0; b < nb; ++b) s += part[3 * b + threadIdx.x];
    out[threadIdx.x] = s;
  }
}
int cube_vstats_run(cube_ctx *c, float sigma_vi, double *sums3) {
  int st = cube_vdec_table(c, c->vdec0, sigma_vi);
  if (st) return st;
  const int nvh = c->nvbin / 2;
  if (c->p.izipv == 1)
    hipLaunchKernelGGL(k_vstats<1>, dim3(VS_BLOCKS), dim3(256), 0, c->stream, (const int8_t *)c->vp, c->vfield,
                       c->rhoc, c->cstart, c->vdec0, nvh, c->ncells, c->dred);
  else
    hipLaunchKernelGGL(k_vstats<2>, dim3(VS_BLOCKS), dim3(256), 0, c->stream, (const int16_t *)c->vp, c->vfield,
                       c->rhoc, c->cstart, c->vdec0, nvh, c->ncells, c->dred);
  CUBE_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_sum_parts, dim3(1), dim3(64), 0, c->stream, c->dred, VS_BLOCKS, c->dred + 3 * VS_BLOCKS);
  CUBE_LAUNCH_CHECK();
  CUBE_CHECK(hipMemcpyAsync(sums3, c->dred + 3 * VS_BLOCKS, 3 * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  CUBE_CHECK(hipStreamSynchronize(c->stream));
  return CUBE_OK;
}

/* ---------------- helpers shared with the IC sort ---------------- */
__global__ void k_fill_zero_i32(int32_t *p, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0;
}
__global__ void k_place_keys(const int32_t *dest, const uint64_t *key, int64_t n, const int64_t *start, int32_t *fill,
                             uint64_t *out) {
  for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < n; p += (int64_t)gridDim.x * blockDim.x) {
    const int32_t d = dest[p];
    if (d < 0) continue;
    const int32_t s = atomicAdd(fill + d, 1);
    out[start[d] + s] = key[p];
  }
}
/* the cells that are listed: medium ones with a wave's bitonic sort, big ones
   with a workgroup's, huge ones by merging sorted runs, tmp the merge buffer.
   nmed and nbig bound their numbers; the lists' own counts are on the device */
static int sort_listed(cube_ctx *c, const int32_t *cnt, const int64_t *start, uint64_t *keys, const int32_t *list,
                       const unsigned long long *ctr, uint64_t *tmp, int64_t nmed, int64_t nbig) {
  if (nmed) {
    hipLaunchKernelGGL(k_sort_med, dim3((unsigned)std::min<int64_t>((nmed + 3) / 4, 1280)), dim3(256), 0, c->stream, cnt,
                       start, list, c->ncells, ctr, keys);
    CUBE_LAUNCH_CHECK();
  }
  if (nbig) {
    hipLaunchKernelGGL(k_sort_big, dim3((unsigned)std::min<int64_t>(nbig, 256)), dim3(1024), BIG_SORT * sizeof(uint64_t),
                       c->stream, cnt, start, list, ctr, keys, tmp);
    CUBE_LAUNCH_CHECK();
  }
  return CUBE_OK;
}
/* sort every cell's key segment ascending; c->key, dead once the keys are
   placed, is the merge buffer */
extern "C" int cube_sort_small_segments(cube_ctx *c, const int32_t *cnt, const int64_t *start, uint64_t *keys) {
  unsigned long long *ctr = (unsigned long long *)c->ured;
  int st = fill_i64(c, (int64_t *)ctr + 3, 2, 0);
  if (st) return st;
  hipLaunchKernelGGL(k_sort_cells, dim3((unsigned)((c->ncells + FB_CELLS - 1) / FB_CELLS)), dim3(256), 0, c->stream, cnt,
                     start, c->ncells, keys, (int32_t *)c->dest, ctr);
  CUBE_LAUNCH_CHECK();
  return sort_listed(c, cnt, start, keys, (const int32_t *)c->dest, ctr, c->key, c->ncells, c->ncells);
}

/* ---------------- driver ---------------- */
/* what the first pass reads: the decode table (as k_vdec), counts and counters cleared */
__global__ __launch_bounds__(256) void k_drift_prep(const float *__restrict__ tanf_tab, double *__restrict__ vdec, int nv,
                                                    double vc, int32_t *__restrict__ cnt, int64_t ncells,
                                                    unsigned long long *__restrict__ ctr) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, nthr = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = t; i < nv; i += nthr) vdec[i] = (double)tanf_tab[i] / vc;
  for (int64_t i = t; i < ncells; i += nthr) cnt[i] = 0;
  if (t < 8) ctr[t] = 0ull;
}
template <int IX, int IV> static int drift_impl(cube_ctx *c, DriftP P, double venc, int64_t *nxtra,
                                                unsigned long long *hc) {
  typedef typename IntOf<IX>::T TX;
  typedef typename IntOf<IV>::T TV;
  unsigned long long *ctr = (unsigned long long *)c->ured;
  int st;
  hipLaunchKernelGGL(k_drift_prep, dim3(1024), dim3(256), 0, c->stream, c->tanf_tab, c->vdec0, (int)c->nvbin, venc, c->rhoc2,
                     c->ncells, ctr);
  CUBE_LAUNCH_CHECK();
  const int64_t nrows = c->ncells / c->nt;
  const size_t dyn = (size_t)(9 * c->nt + P.agg_cap) * sizeof(int);
  hipLaunchKernelGGL((k_drift_dest<IX, IV>), dim3((unsigned)nrows), dim3(DT), dyn, c->stream, (const TX *)c->xp,
                     (const TV *)c->vp, c->vfield, c->cstart, c->vdec0, P, c->dest, c->key, c->rhoc2, c->rank,
                     c->xdest, c->xkey, c->xrank, c->xcap, ctr);
  CUBE_LAUNCH_CHECK();
  int64_t total = 0;
  if ((st = cube_scan_counts(c, c->rhoc2, c->cstart2, c->ncells, &total, ctr))) return st;
  memcpy(hc, c->hres + HR_CTR, 8 * sizeof(unsigned long long));
  if (hc[2] & (DERR_RANGE | DERR_KEY)) return CUBE_ERR_DISPLACEMENT;
  if (hc[2] & DERR_XOVER) return CUBE_ERR_IMAGE_OVERFLOW;
  if (total > c->cap) return CUBE_ERR_IMAGE_OVERFLOW;
  *nxtra = (int64_t)hc[0];
  int32_t *list = c->fill; /* the initial sort's, free here */
  hipLaunchKernelGGL(k_place_ranked, dim3(4096), dim3(256), 0, c->stream, c->dest, c->rank, c->key, c->nplocal,
                     c->cstart2, c->sortbuf, c->rhoc2, c->ncells, list, ctr);
  CUBE_LAUNCH_CHECK();
  if (hc[0]) {
    hipLaunchKernelGGL(k_place_ranked, dim3(64), dim3(256), 0, c->stream, c->xdest, c->xrank, c->xkey,
                       (int64_t)hc[0], c->cstart2, c->sortbuf, (const int32_t *)nullptr, c->ncells, list, ctr);
    CUBE_LAUNCH_CHECK();
  }
  /* key is dead after placement: the merge buffer */
  if ((st = sort_listed(c, c->rhoc2, c->cstart2, c->sortbuf, list, ctr, c->key, (int64_t)hc[6], (int64_t)hc[5]))) return st;
  const int64_t nfb = (c->ncells + FB_CELLS - 1) / FB_CELLS;
  hipLaunchKernelGGL((k_drift_final2<IX, IV>), dim3((unsigned)nfb), dim3(256), 0, c->stream, (const TX *)c->xp,
                     (const TV *)c->vp, c->p.has_pid ? c->pid : nullptr, c->vfield, c->cstart2, c->sortbuf,
                     c->vdec0, P, venc, (TX *)c->xp2, (TV *)c->vp2, c->pid2, c->vfield2, c->ncells,
                     c->vpart);
  CUBE_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_sum_parts_tree, dim3(1), dim3(1024), 0, c->stream, c->vpart, nfb, (double *)c->hres + HR_S3);
  CUBE_LAUNCH_CHECK();
  CUBE_CHECK(hipStreamSynchronize(c->stream));
  c->nplocal = total;
  return CUBE_OK;
}

int cube_drift(cube_ctx *c, float dt_old, float dt, float vz_max, float sigma_vi, cube_vstats *out) {
  /* dt_mid=(dt_old+dt)/2; nlayer=2*ceiling(dt_mid*vz_max/ncell)+1 (real(4)) */
  const float dt_mid = (dt_old + dt) / 2.0f;
  const int nlayer = 2 * (int)ceilf(dt_mid * vz_max / 4.0f) + 1;
  if (nlayer < 1 || nlayer > 511) return CUBE_ERR_DISPLACEMENT;
  /* tile overflow check (W/update_particle.f90:86-94): the copies in each
     tile's extended region must fit np_tile_max */
  int64_t *sums = (int64_t *)malloc(c->ntiles * sizeof(int64_t));
  tbeg(c);
  int st = cube_tile_boxsum(c, (int)c->ncb, sums);
  tend(c, CUBE_T_CHECKS);
  double ov = 0;
  int64_t mx = 0;
  for (int64_t t = 0; t < c->ntiles; ++t) {
    const double o = (double)((float)sums[t] / (float)c->np_tile_max);
    ov = o > ov ? o : ov;
    mx = sums[t] > mx ? sums[t] : mx;
  }
  free(sums);
  if (st) return st;
  if (mx > c->np_tile_max) return CUBE_ERR_TILE_OVERFLOW;
  tbeg(c);
  DriftP P;
  P.g = geo_of(c);
  P.nlayer = nlayer;
  P.nvh = c->nvbin / 2;
  P.dt_mid = dt_mid;
  P.xres = c->p.izipx == 1 ? 1.0 / 256.0 : 1.0 / 65536.0;
  P.inv_xres4 = c->p.izipx == 1 ? 64.0 : 16384.0;
  P.agg_cap = AGG_CAP;
  /* a lower cap sends more rows down the all-global slot path (used by the
     tests to cover both paths in one run) */
  if (const char *e = getenv("CUBE_DRIFT_AGG_CAP"); e && *e) P.agg_cap = std::min(AGG_CAP, atoi(e));
  const double venc = cube_vconst(sigma_vi);
  int64_t nxtra = 0;
  unsigned long long hc[8];
  const int64_t np_old = c->nplocal;
  if (c->p.izipx == 1 && c->p.izipv == 1) st = drift_impl<1, 1>(c, P, venc, &nxtra, hc);
  else if (c->p.izipx == 1) st = drift_impl<1, 2>(c, P, venc, &nxtra, hc);
  else if (c->p.izipv == 1) st = drift_impl<2, 1>(c, P, venc, &nxtra, hc);
  else st = drift_impl<2, 2>(c, P, venc, &nxtra, hc);
  if (st) return st;
  tend(c, CUBE_T_DRIFT);
  /* the new state becomes current */
  void *tx = c->xp; c->xp = c->xp2; c->xp2 = tx;
  void *tv = c->vp; c->vp = c->vp2; c->vp2 = tv;
  int32_t *tp = c->pid; c->pid = c->pid2; c->pid2 = tp;
  int32_t *tr = c->rhoc; c->rhoc = c->rhoc2; c->rhoc2 = tr;
  float *tf = c->vfield; c->vfield = c->vfield2; c->vfield2 = tf;
  int64_t *ts = c->cstart; c->cstart = c->cstart2; c->cstart2 = ts;
  /* std of the velocity field, FP64 sums (:171-224), reduced by the
     finalize kernel of the drift */
  double s3[3];
  memcpy(s3, c->hres + HR_S3, sizeof(s3));
  const double npg = (double)c->npglobal;
  cube_vstats v;
  memset(&v, 0, sizeof(v));
  v.sum_c = s3[0];
  v.sum_r = s3[1];
  v.sum_s = s3[2];
  v.std_vsim = sqrt(s3[2] / npg);
  v.std_vsim_c = sqrt(s3[0] / (double)c->nc / (double)c->nc / (double)c->nc);
  v.std_vsim_res = sqrt(s3[1] / npg);
  v.sigma_vi_new = (float)(v.std_vsim_res / (double)sqrtf(3.0f));
  v.nlayer = nlayer;
  v.nplocal = c->nplocal;
  v.lost = (int64_t)hc[1];
  v.overhead_tile = ov;
  (void)np_old;
  if (out) *out = v;
  if (c->nplocal != c->npglobal) return CUBE_ERR_COUNT;
  return CUBE_OK;
}
