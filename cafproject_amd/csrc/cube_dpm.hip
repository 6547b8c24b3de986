/*
 * cube_dpm.hip -- differentiable particle-mesh forward model and its
 * hand-written adjoint (include/cube_dpm.h).  No reference counterpart.
 *
 * A particle is held as its FP32 displacement d (in mesh cells) from its
 * lattice point q = (nf/ng) * l, l its lattice coordinates; particles keep
 * their slot for the whole run (no sorting), so the adjoint state is per
 * particle.  Slots go block by block of 4^3 lattice points, one wave each: a
 * wave reads its particles whole and finds them in a few cubic neighbouring
 * pieces of the mesh.  CIC convention: a particle at x = q + d touches mesh points
 * floor(x) and floor(x)+1 per axis (mod nf) with weights 1-f and f, formed
 * as q + floor(d) and f = d - floor(d): exact, and resolved to the
 * displacement's ulp rather than to the ulp of a position near nf, so far
 * fewer particles than with FP32 positions sit within rounding of a cell
 * edge, where the weights' slope (and so the gradient) jumps.
 *
 * Forward operators and their transposes:
 *   deposit  rho_c = sum_i W(x_i,c)          ^T: lam -> sum_c lam_c W(x_i,c)
 *   Poisson  F_d = (1/N^3) C2R[i K_d R2C(rho)]   ^T: K_d -> -K_d, summed over d
 *   gather   F_i = sum_c W(x_i,c) M_c         ^T (in M): S_c = sum_i W g_i
 *   and the position derivatives of deposit and gather use dW/dx.
 * K_d = k_d/k^2 (k = 2 pi m/N), zero at k=0 and on the Nyquist plane of
 * axis d, so every product spectrum stays Hermitian and the real
 * transforms are exact transposes of each other.
 */
#include "cube_dpm_internal.h"
#include "cube_dpm_mem.h"
#include <math.h>
#include <stdlib.h>
#include <string.h>
#include <algorithm>

#define PT 256

/* --------------------------- particles --------------------------- */
__device__ static inline float wrapf(float x, float n) {
  x = x - n * floorf(x / n);
  return x >= n ? x - n : x;
}
struct V3 { /* three interleaved components, read with one 12-byte load */
  float x, y, z;
};
__device__ __forceinline__ V3 ld3(const float *p) { return *reinterpret_cast<const V3 *>(p); }
__device__ __forceinline__ void st3(float *p, float x, float y, float z) { *reinterpret_cast<V3 *>(p) = V3{x, y, z}; }

/* the two mesh points i0, i1 of a row (adjacent but at the periodic edge), NC components each */
template <int NC> struct Pair {
  float v[2][NC];
};
template <int NC> __device__ __forceinline__ Pair<NC> ld_pair(const float *row, const int i[2]) {
  Pair<NC> r;
  struct P2 {
    float f[2 * NC];
  };
  const P2 a = *reinterpret_cast<const P2 *>(row + NC * (i[1] ? i[0] : i[0] - 1));
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    r.v[0][k] = a.f[k];
    r.v[1][k] = a.f[NC + k];
  }
  if (i[1] == 0) { /* the last point and the first */
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      r.v[0][k] = a.f[NC + k];
      r.v[1][k] = row[k];
    }
  }
  return r;
}

/* the particle lattice: ng^3 points r mesh cells apart, in nb^3 blocks of 4^3 */
struct Lat {
  int ng, r, nb, nblk;
};
/* block coordinates packed 10 bits each (cube_dpm_create bounds nb) */
__device__ __forceinline__ uint32_t blk_pack(const Lat &L, int b) {
  const uint32_t u = (uint32_t)b, n = (uint32_t)L.nb, q = u / n, z = q / n;
  return (u - q * n) | ((q - z * n) << 10) | (z << 20);
}
__device__ __forceinline__ int blk_of(const Lat &L, uint32_t pk) {
  return (int)(((pk >> 20) * (uint32_t)L.nb + ((pk >> 10) & 1023u)) * (uint32_t)L.nb + (pk & 1023u));
}
/* lattice coordinates of a lane of a block, and whether it is a particle */
__device__ __forceinline__ bool lat_of(const Lat &L, uint32_t pk, int lane, int l[3]) {
  l[0] = 4 * (int)(pk & 1023u) + (lane & 3);
  l[1] = 4 * (int)((pk >> 10) & 1023u) + ((lane >> 2) & 3);
  l[2] = 4 * (int)(pk >> 20) + (lane >> 4);
  return l[0] < L.ng && l[1] < L.ng && l[2] < L.ng;
}
__device__ __forceinline__ int64_t lat_index(const Lat &L, const int l[3]) {
  return ((int64_t)l[2] * L.ng + l[1]) * L.ng + l[0];
}
/* i mod n in [0, n): one addition for all but displacements beyond a box */
__device__ __forceinline__ int wrap_cell(int i, int n) {
  if ((unsigned)(i + n) < 3u * (unsigned)n) { /* [-n, 2n) */
    i += i < 0 ? n : 0;
    return i - (i >= n ? n : 0);
  }
  return ((i % n) + n) % n; /* always a valid mesh index, whatever d holds */
}
struct Cic {
  int i[3][2];   /* mesh indices per axis (periodic) */
  float w[3][2]; /* weights */
};
__device__ __forceinline__ Cic cic_of(V3 d, const int l[3], int r, int n) {
  const float dsp[3] = {d.x, d.y, d.z};
  Cic c;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float fl = floorf(dsp[a]);
    const float f = dsp[a] - fl;
    const int i0 = wrap_cell(r * l[a] + (int)fl, n);
    c.i[a][0] = i0;
    c.i[a][1] = i0 + 1 == n ? 0 : i0 + 1;
    c.w[a][0] = 1.f - f;
    c.w[a][1] = f;
  }
  return c;
}

/* --------------------------- tile lists ---------------------------
 * The deposit and its transpose gather: a workgroup owns a cubic tile of the
 * mesh, goes through the lattice blocks whose clouds reach it, and adds their
 * particles' terms in LDS.  Each kernel that moves particles appends every
 * block to the lists of the tiles it reaches (those in the bounding box of its
 * particles' cells, an interval of tiles per axis, or with more than 64 of
 * them those that a particle's cloud is in): about 5 lists per block with
 * 16-cell tiles and 13 with 8-cell ones (nf <= 128, where 16-cell tiles would
 * be too few workgroups).  A list that runs over (`cap` entries, several times
 * the mean) makes its tile test every block's interval instead, so nothing
 * depends on how clustered the box is.  There are two sets of list
 * lengths: the pass that reads one empties the other for the lists to come. */
struct Tiles {
  int T, nt, cap;  /* cells and tiles per axis, entries per list */
  int *cnt, *next; /* nt^3 list lengths, and those of the lists to come: zeroed by the pass that reads these */
  uint32_t *list;  /* nt^3 * cap packed blocks */
  uint64_t *range; /* per block: first tile and count per axis, 8 bits each */
};
/* append block b (lane `live`s with unwrapped base cells v) to its tiles */
__device__ __forceinline__ void bin_block(const Tiles &B, int b, uint32_t pk, int lane, bool live, const int v[3], int n) {
  int lo[3], hi[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    lo[a] = live ? v[a] : 0x7fffffff;
    hi[a] = live ? v[a] : -0x7fffffff - 1;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      lo[a] = min(lo[a], __shfl_xor(lo[a], o, 64));
      hi[a] = max(hi[a], __shfl_xor(hi[a], o, 64));
    }
  int t0[3], tc[3];
  uint64_t iv = 0;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int64_t len = (int64_t)hi[a] - lo[a] + 2; /* cells touched, the upper corner included */
    const int s = wrap_cell(lo[a], n);
    t0[a] = 0;
    tc[a] = B.nt;
    if (len < n) {
      const int e = s + (int)len - 1;
      t0[a] = s / B.T;
      tc[a] = e < n ? e / B.T - t0[a] + 1 : min(B.nt, B.nt - t0[a] + (e - n) / B.T + 1);
    }
    iv |= (uint64_t)((unsigned)t0[a] | ((unsigned)tc[a] << 8)) << (16 * a);
  }
  if (lane == 0) B.range[b] = iv;
  const int tot = tc[0] * tc[1] * tc[2];
  auto append = [&](int t) {
    const int q = atomicAdd(B.cnt + t, 1);
    if (q < B.cap) B.list[(int64_t)t * B.cap + q] = pk;
  };
  if (tot <= 64) {
    if (lane < tot) {
      const int ex = lane % tc[0], ey = (lane / tc[0]) % tc[1], ez = lane / (tc[0] * tc[1]);
      int x = t0[0] + ex, y = t0[1] + ey, z = t0[2] + ez;
      x -= x >= B.nt ? B.nt : 0;
      y -= y >= B.nt ? B.nt : 0;
      z -= z >= B.nt ? B.nt : 0;
      append((z * B.nt + y) * B.nt + x);
    }
    return;
  }
  /* A block whose particles have left one another: the box around them holds
     up to all tiles, where 64 scattered clouds reach 91 8-cell tiles.  Each
     tile they reach once: a lane's 8 corners are bits of `todo`, and a turn
     takes one corner's tile and clears it from every lane.  64^3 particles on
     128^3 points with displacements of 24 cells rms, forward and adjoint of
     three steps: 7.3 and 5.7 ms by the box, 0.76 and 0.62 so; 128^3 on 256^3
     12.3 and 16.5 against 3.6 and 4.1 */
  int t[3][2];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int c = wrap_cell(v[a], n);
    t[a][0] = c / B.T;
    t[a][1] = (c + 1 == n ? 0 : c + 1) / B.T;
  }
  unsigned todo = live ? 0xffu : 0u; /* bit 4z + 2y + x */
  if (t[0][0] == t[0][1]) todo &= 0x55u;
  if (t[1][0] == t[1][1]) todo &= 0x33u;
  if (t[2][0] == t[2][1]) todo &= 0x0fu;
  int mine = 0, m = 0;
  for (uint64_t any; (any = __ballot(todo != 0u)) != 0ull;) {
    const int src = __builtin_ctzll(any), k = __builtin_ctz((unsigned)__builtin_amdgcn_readlane((int)todo, src));
    const int X = __builtin_amdgcn_readlane(k & 1 ? t[0][1] : t[0][0], src),
              Y = __builtin_amdgcn_readlane(k & 2 ? t[1][1] : t[1][0], src),
              Z = __builtin_amdgcn_readlane(k & 4 ? t[2][1] : t[2][0], src);
    todo &= ~(((t[0][0] == X ? 0x55u : 0u) | (t[0][1] == X ? 0xaau : 0u)) &
              ((t[1][0] == Y ? 0x33u : 0u) | (t[1][1] == Y ? 0xccu : 0u)) &
              ((t[2][0] == Z ? 0x0fu : 0u) | (t[2][1] == Z ? 0xf0u : 0u)));
    if (lane == (m & 63)) mine = (Z * B.nt + Y) * B.nt + X;
    if ((++m & 63) == 0) append(mine);
  }
  if (lane < (m & 63)) append(mine);
}
__device__ __forceinline__ void base_cells(V3 d, const int l[3], int r, int v[3]) {
  v[0] = r * l[0] + (int)floorf(d.x);
  v[1] = r * l[1] + (int)floorf(d.y);
  v[2] = r * l[2] + (int)floorf(d.z);
}
__global__ void k_dpm_bin(const float *__restrict__ x, Lat L, int n, Tiles B) {
  const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  for (int b = blockIdx.x * nw + (threadIdx.x >> 6); b < L.nblk; b += gridDim.x * nw) {
    int l[3], v[3] = {0, 0, 0};
    const uint32_t pk = blk_pack(L, b);
    const bool live = lat_of(L, pk, lane, l);
    if (live) base_cells(ld3(x + 3 * ((int64_t)b * 64 + lane)), l, L.r, v);
    bin_block(B, b, pk, lane, live, v, n);
  }
}
/* empty lists and no maxima, before the first list of a pass is built */
__global__ void k_dpm_reset(int *cnt, int n, unsigned *gmx) {
  for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < n; q += gridDim.x * blockDim.x) cnt[q] = 0;
  if (blockIdx.x == 0 && threadIdx.x < 2 * DPM_GMX) gmx[threadIdx.x] = 0u;
}

/*
 * The deposit and its transpose add many particles' terms into mesh points in
 * no particular order.  They add 64-bit fixed-point integers, whose sums do
 * not depend on the order, and convert to FP32 once: the meshes, and so the
 * whole model, are the same bits run to run and in any launch shape or graph.
 * The deposit's terms are weights in [0, 1], kept with 32 fraction bits; the
 * transpose's terms w*g are scaled by a power of two that puts max|g| in
 * [2^39, 2^40) (found on the device before the scatter), so every sum of up
 * to 2^23 terms stays in range.  Each term is rounded once to the fixed-point
 * grid, finer than FP32 at the terms' scale; the conversion rounds the exact
 * sum once.
 */
#define FIX_DEPOSIT 0x1p32
/* the transpose's scale: 2^(40-e) for max|g| = m 2^e, m in [0.5, 1) */
__device__ static inline double fix_scale(unsigned gmx) {
  int e = 0;
  (void)frexp((double)__uint_as_float(gmx), &e);
  return ldexp(1.0, 40 - e);
}
/* nint (half to even) of |v| < 2^51 by the addition that leaves it in the low bits */
__device__ __forceinline__ unsigned long long fix_round(double v) {
  return (unsigned long long)(__double_as_longlong(v + 0x1.8p52) - 0x4338000000000000ll);
}
/* an accumulated sum as a double, exactly where it is below 2^51 (the inverse
   of fix_round's addition), rounded once beyond */
__device__ __forceinline__ double fix_double(unsigned long long a) {
  const long long v = (long long)a;
  if ((unsigned long long)(v + (1ll << 51)) < (1ull << 52))
    return __longlong_as_double(v + 0x4338000000000000ll) - 0x1.8p52;
  return (double)v;
}
__device__ __forceinline__ unsigned gmx_of(const unsigned *gmx, int lane) {
  unsigned m = 0;
  for (int q = lane; q < DPM_GMX; q += 64) m = max(m, gmx[q]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o, 64));
  return m;
}

/*
 * A tile of the mesh: NC = 1, rho = sum W (and delta = rho * inv_nbar - 1);
 * NC = 3, S_d = sum W g_d with g = coef * pbar.  The waves take the tile's
 * list entries in turn, a lane a particle; a cloud's 8 points are added where
 * they fall in the tile.  Against 64-bit atomics on the mesh (35e9 per second
 * whatever the launch shape, with a clear and a conversion pass): 128^3
 * particles on 256^3 points, deposit 0.56 -> 0.055 ms, transpose 1.7 -> 0.14.
 * Bound by VALU work (the terms' FP64 rounding, the tests, the conversion) and
 * by how many workgroups share a CU's LDS: the transpose's tile as two halves
 * of 8 planes keeps three workgroups of 8 waves (52 KB each) where the whole
 * one keeps a single one (0.18 ms).  LDS float additions are no way out: a
 * float add runs at a third of a lane per clock there, a 64-bit integer one at
 * five.
 */
template <int T, int NC, int ZS, int NT>
__global__ __launch_bounds__(NT) void k_dpm_tile(const float *__restrict__ x, const float *__restrict__ pbar, float coef,
                                               Lat L, int n, Tiles B, unsigned *__restrict__ gmx,
                                               unsigned *__restrict__ gmx_next, float *__restrict__ out,
                                               float *__restrict__ delta, float inv_nbar) {
  constexpr int TZ = T / ZS, T3 = T * T * TZ, NW = NT / 64;
  __shared__ __align__(16) unsigned long long acc[NC * T3];
  __shared__ int hits[NW][128]; /* per wave: slots whose clouds reach the tile */
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tile = blockIdx.x / ZS, zs = blockIdx.x % ZS; /* ZS workgroups share a tile's list, TZ planes each */
  const int lo[3] = {T * (tile % B.nt), T * ((tile / B.nt) % B.nt), T * (tile / (B.nt * B.nt))};
  const int t0[3] = {lo[0], lo[1], lo[2] + TZ * zs}, te[3] = {T, T, TZ};
  for (int q = tid; q < NC * T3 / 2; q += NT) reinterpret_cast<ulonglong2 *>(acc)[q] = make_ulonglong2(0ull, 0ull);
  const int cnt = B.cnt[tile];
  double scale = FIX_DEPOSIT;
  if constexpr (NC == 3) {
    scale = fix_scale(gmx_of(gmx, lane));
    if (tile == 0)
      for (int q = tid; q < DPM_GMX; q += NT) gmx_next[q] = 0u;
  }
  __syncthreads();
  /* Few of a listed block's particles reach the tile (a fifth at 16 cells), so
     the wave queues those that do and adds 64 at a time. */
  int *queue = hits[wv];
  int nq = 0;
  auto flush = [&](int m) { /* the first m <= 64 of the queue */
    wave_lds_sync();
    if (lane < m) {
      const int slot = queue[lane];
      int l[3];
      (void)lat_of(L, blk_pack(L, slot >> 6), slot & 63, l);
      const Cic c = cic_of(ld3(x + 3 * (int64_t)slot), l, L.r, n);
      float g[3] = {0.f, 0.f, 0.f};
      /* not finite: the weights (of a displacement that is not) or the
         cotangent.  Such a particle adds nothing: its terms have no integer */
      float odd = (c.w[0][1] + c.w[1][1]) + c.w[2][1];
      if constexpr (NC == 3) {
        const V3 pb = ld3(pbar + 3 * (int64_t)slot);
        g[0] = coef * pb.x;
        g[1] = coef * pb.y;
        g[2] = coef * pb.z;
        odd = fmaf(0.f, g[0], fmaf(0.f, g[1], fmaf(0.f, g[2], odd)));
      }
      int rel[3][2];
      bool in[3][2];
#pragma unroll
      for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          rel[a][u] = c.i[a][u] - t0[a];
          in[a][u] = (unsigned)rel[a][u] < (unsigned)te[a];
        }
      if (odd == odd)
#pragma unroll
      for (int z = 0; z < 2; ++z)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
          for (int xx = 0; xx < 2; ++xx)
            if (in[0][xx] && in[1][y] && in[2][z]) {
              const float w = c.w[0][xx] * c.w[1][y] * c.w[2][z];
              const int k = (rel[2][z] * T + rel[1][y]) * T + rel[0][xx];
              if constexpr (NC == 1) {
                atomicAdd(acc + k, fix_round((double)w * FIX_DEPOSIT));
              } else {
#pragma unroll
                for (int a = 0; a < 3; ++a) atomicAdd(acc + a * T3 + k, fix_round((double)(w * g[a]) * scale));
              }
            }
    }
    const int rest = queue[lane + 64];
    wave_lds_sync();
    if (lane + 64 < nq) queue[lane] = rest;
    nq = max(nq - 64, 0);
  };
  /* the particles of lattice block pk (uniform over the wave), at d */
  auto add = [&](uint32_t pk, V3 d) {
    int l[3];
    bool hit = lat_of(L, pk, lane, l);
    int v[3];
    base_cells(d, l, L.r, v);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      /* base cell in the tile or one below it: its distance from that one,
         modulo the box */
      int u = wrap_cell(v[a], n) - t0[a] + 1;
      u += u < 0 ? n : 0;
      u -= u >= n ? n : 0;
      hit = hit && (unsigned)u <= (unsigned)te[a];
    }
    const uint64_t m = __ballot(hit);
    if (hit) queue[nq + __popcll(m & ((1ull << lane) - 1ull))] = blk_of(L, pk) * 64 + lane;
    nq += __popcll(m);
    if (nq >= 64) flush(64);
  };
  if (cnt <= B.cap) {
    const uint32_t *list = B.list + (int64_t)tile * B.cap;
    for (int e0 = 0; e0 < cnt; e0 += NT) { /* a lane per entry, 64 a wave */
      const int mine = e0 + lane * NW + wv < cnt ? (int)list[e0 + lane * NW + wv] : 0;
      const int m = (min(cnt - e0, NT) - wv + NW - 1) / NW;
      for (int k = 0; k < m; k += 4) { /* four blocks' particles on their way at once */
        uint32_t pk[4];
        V3 d[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          pk[u] = (uint32_t)__builtin_amdgcn_readlane(mine, min(k + u, m - 1));
          d[u] = ld3(x + 3 * ((int64_t)blk_of(L, pk[u]) * 64 + lane));
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (k + u < m) add(pk[u], d[u]);
      }
    }
  } else { /* the list ran over: 64 blocks' intervals at a time */
    for (int e0 = wv * 64; e0 < L.nblk; e0 += NT) {
      bool hit = false;
      if (e0 + lane < L.nblk) {
        const uint64_t pk = B.range[e0 + lane];
        hit = true;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          int q = lo[a] / T - ((int)(pk >> (16 * a)) & 255);
          q += q < 0 ? B.nt : 0;
          hit = hit && q < ((int)(pk >> (16 * a + 8)) & 255);
        }
      }
      for (uint64_t m = __ballot(hit); m; m &= m - 1ull) {
        const int b = e0 + __builtin_ctzll(m);
        add(blk_pack(L, b), ld3(x + 3 * ((int64_t)b * 64 + lane)));
      }
    }
  }
  if (nq > 0) flush(nq);
  __syncthreads();
  if (zs == 0 && tid == 0) B.next[tile] = 0;
  const double inv = 1.0 / scale;
  const int64_t n3 = (int64_t)n * n * n;
  /* four points of a row at a time (mesh rows are multiples of 4 points) */
  for (int q4 = tid; q4 < NC * T3 / 4; q4 += NT) {
    const int q = 4 * q4, m = q % T3, X = t0[0] + m % T, Y = t0[1] + (m / T) % T, Z = t0[2] + m / (T * T);
    if (X >= n || Y >= n || Z >= n) continue;
    float v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = (float)(fix_double(acc[q + u]) * inv);
    const int64_t o = ((int64_t)Z * n + Y) * n + X;
    float *p = out + (q / T3) * n3 + o;
    if (n % 4 == 0) {
      *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
      for (int u = 0; u < 4 && X + u < n; ++u) p[u] = v[u];
    }
    if (NC == 1 && delta) /* the caller's array, of any alignment */
      for (int u = 0; u < 4 && X + u < n; ++u) delta[o + u] = v[u] * inv_nbar - 1.f;
  }
}

/* --------------------------- particle kernels --------------------------- */
/* Zel'dovich ICs from psi (three lattice planes): displacement and momentum */
__global__ void k_dpm_ic_particles(const float *__restrict__ psi, Lat L, int n, float r, float cx, float cp, float scale,
                                   float *__restrict__ x, float *__restrict__ p, Tiles B) {
  const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  const int64_t n3 = (int64_t)L.ng * L.ng * L.ng;
  for (int b = blockIdx.x * nw + (threadIdx.x >> 6); b < L.nblk; b += gridDim.x * nw) {
    int l[3], v[3] = {0, 0, 0};
    const uint32_t pk = blk_pack(L, b);
    const bool live = lat_of(L, pk, lane, l);
    if (live) {
      const int64_t i = lat_index(L, l), q = (int64_t)b * 64 + lane;
      const float s0 = psi[i] * scale * r, s1 = psi[n3 + i] * scale * r, s2 = psi[2 * n3 + i] * scale * r;
      const V3 d = {cx * s0, cx * s1, cx * s2}; /* displacement from the lattice point l*r */
      st3(x + 3 * q, d.x, d.y, d.z);
      st3(p + 3 * q, cp * s0, cp * s1, cp * s2);
      base_cells(d, l, L.r, v);
    }
    bin_block(B, b, pk, lane, live, v, n);
  }
}

/*
 * Around a force mesh: the closing half kick of the step before (cB), the
 * opening one of the next (cA), its drift (cD) into xout, and the new
 * positions' tile lists -- one pass over the particles and one gather, where
 * a step had two kicks, a drift and the lists' own pass.  p += c * F each time
 * with F = sum_c W F_c (interleaved, 3 per mesh point).  open = 0: the last
 * step's closing kick alone.  pkeep: p between the two kicks, the state of a
 * whole step (the steps that are recomputed start there).  128^3 particles on
 * 256^3 points: 0.11 ms where kick, kick, drift and copy took 0.16, a quarter
 * of it the lists; the address units' work on the gathers' scattered rows
 * bounds it (each reads the two points of a row together: 0.24 -> 0.16 ms in
 * k_dpm_grad, which reads a fourth component).
 */
__global__ void k_dpm_step(const float *x, float *__restrict__ p, const float *__restrict__ F, Lat L, int n,
                           int close, float cB, int open, float cA, float cD, float *xout /* may be x */,
                           float *__restrict__ pkeep, Tiles B) {
  const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  for (int b = blockIdx.x * nw + (threadIdx.x >> 6); b < L.nblk; b += gridDim.x * nw) {
    int l[3], v[3] = {0, 0, 0};
    const uint32_t pk = blk_pack(L, b);
    const bool live = lat_of(L, pk, lane, l);
    if (live) {
      const int64_t q = (int64_t)b * 64 + lane;
      const V3 d = ld3(x + 3 * q);
      const V3 p0 = ld3(p + 3 * q);
      const Cic c = cic_of(d, l, L.r, n);
      float f[3] = {0.f, 0.f, 0.f};
      Pair<3> m[2][2];
#pragma unroll
      for (int z = 0; z < 2; ++z)
#pragma unroll
        for (int y = 0; y < 2; ++y) m[z][y] = ld_pair<3>(F + 3 * ((int64_t)c.i[2][z] * n + c.i[1][y]) * n, c.i[0]);
#pragma unroll
      for (int z = 0; z < 2; ++z)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
          for (int xx = 0; xx < 2; ++xx) {
            const float w = c.w[0][xx] * c.w[1][y] * c.w[2][z];
#pragma unroll
            for (int a = 0; a < 3; ++a) f[a] += w * m[z][y].v[xx][a];
          }
      float pn[3] = {p0.x, p0.y, p0.z};
      if (close)
#pragma unroll
        for (int a = 0; a < 3; ++a) pn[a] += cB * f[a];
      if (pkeep) st3(pkeep + 3 * q, pn[0], pn[1], pn[2]);
      if (open) {
#pragma unroll
        for (int a = 0; a < 3; ++a) pn[a] += cA * f[a];
        /* the displacement needs no wrap: the mesh index is taken mod nf */
        const V3 dn = {d.x + cD * pn[0], d.y + cD * pn[1], d.z + cD * pn[2]};
        st3(xout + 3 * q, dn.x, dn.y, dn.z);
        base_cells(dn, l, L.r, v);
      }
      st3(p + 3 * q, pn[0], pn[1], pn[2]);
    }
    if (open) bin_block(B, b, pk, lane, live, v, n);
  }
}

/*
 * The backward counterpart, between two force meshes.  First the cotangent
 * that flows into the positions: xbar += sum_c dW(x,c)/dx (s_lam lam_c + g .
 * M_c) with g = coef * pbar (M null at the final density, where lam is the
 * loss gradient and xbar starts at zero).  Then the step below: pbar += cD *
 * xbar (drift^T), the maximum of |coef2 * pbar| for the transpose's scale and
 * the tile lists of that step's positions x2 (null: built by its own pass).
 * After the last step (psi) the initial conditions' psibar = r (cx xbar + cp
 * pbar) instead, three lattice planes.
 */
__global__ void k_dpm_grad(const float *__restrict__ x, Lat L, int n, const float *__restrict__ lam, float s_lam, float coef,
                           const float *__restrict__ M, int first, float *__restrict__ xbar, float *__restrict__ pbar,
                           float cD, float coef2, unsigned *__restrict__ gmx, const float *__restrict__ x2, Tiles B,
                           float *__restrict__ psi, float cx, float cp, float r) {
  const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  const int64_t n3 = (int64_t)L.ng * L.ng * L.ng;
  float mx = 0.f;
  for (int b = blockIdx.x * nw + (threadIdx.x >> 6); b < L.nblk; b += gridDim.x * nw) {
    int l[3], v2[3] = {0, 0, 0};
    const uint32_t pk = blk_pack(L, b);
    const bool live = lat_of(L, pk, lane, l);
    if (live) {
      const int64_t q = (int64_t)b * 64 + lane;
      const Cic c = cic_of(ld3(x + 3 * q), l, L.r, n);
      const V3 pb = first ? V3{0.f, 0.f, 0.f} : ld3(pbar + 3 * q), xb = first ? V3{0.f, 0.f, 0.f} : ld3(xbar + 3 * q);
      const float gv[3] = {coef * pb.x, coef * pb.y, coef * pb.z};
      float acc[3] = {0.f, 0.f, 0.f};
      Pair<1> lm[2][2];
      Pair<3> m[2][2];
#pragma unroll
      for (int z = 0; z < 2; ++z)
#pragma unroll
        for (int y = 0; y < 2; ++y) {
          const int64_t row = ((int64_t)c.i[2][z] * n + c.i[1][y]) * n;
          lm[z][y] = ld_pair<1>(lam + row, c.i[0]);
          if (M) m[z][y] = ld_pair<3>(M + 3 * row, c.i[0]);
        }
#pragma unroll
      for (int z = 0; z < 2; ++z)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
          for (int xx = 0; xx < 2; ++xx) {
            float v = s_lam * lm[z][y].v[xx][0];
            if (M) {
              const float *mv = m[z][y].v[xx];
              v += (gv[0] * mv[0] + gv[1] * mv[1]) + gv[2] * mv[2];
            }
            /* dW/dx_a: the weight of axis a replaced by its slope -1 (lower) or +1 (upper) */
            const float sx = xx ? 1.f : -1.f, sy = y ? 1.f : -1.f, sz = z ? 1.f : -1.f;
            acc[0] += v * (sx * c.w[1][y] * c.w[2][z]);
            acc[1] += v * (c.w[0][xx] * sy * c.w[2][z]);
            acc[2] += v * (c.w[0][xx] * c.w[1][y] * sz);
          }
      const float xn[3] = {xb.x + acc[0], xb.y + acc[1], xb.z + acc[2]};
      float pn[3] = {pb.x, pb.y, pb.z};
      if (psi) {
        const int64_t i = lat_index(L, l);
#pragma unroll
        for (int a = 0; a < 3; ++a) psi[a * n3 + i] = r * (cx * xn[a] + cp * pn[a]);
      } else {
        st3(xbar + 3 * q, xn[0], xn[1], xn[2]);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          pn[a] += cD * xn[a];
          mx = fmaxf(mx, fabsf(coef2 * pn[a]));
        }
        st3(pbar + 3 * q, pn[0], pn[1], pn[2]);
        if (x2) base_cells(ld3(x2 + 3 * q), l, L.r, v2);
      }
    }
    if (x2) bin_block(B, b, pk, lane, live, v2, n);
  }
  if (psi) return;
  /* non-negative floats order as their bits */
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  if (lane == 0 && mx > 0.f) atomicMax(gmx + (blockIdx.x * nw + (threadIdx.x >> 6)) % DPM_GMX, __float_as_uint(mx));
}

/* positions q + d wrapped into [0, nf) and momenta in lattice order, for cube_dpm_state */
__global__ void k_dpm_state(const float *x, const float *p, Lat L, int n, float *xo, float *po) {
  const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  for (int b = blockIdx.x * nw + (threadIdx.x >> 6); b < L.nblk; b += gridDim.x * nw) {
    int l[3];
    if (!lat_of(L, blk_pack(L, b), lane, l)) continue;
    const int64_t i = lat_index(L, l), q = (int64_t)b * 64 + lane;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      if (xo) xo[3 * i + a] = wrapf((float)(L.r * l[a]) + x[3 * q + a], (float)n);
      if (po) po[3 * i + a] = p[3 * q + a];
    }
  }
}
__global__ void k_dpm_scale_to(float *dst, const float *src, int64_t n, float coef) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x)
    dst[q] = coef * src[q];
}

/* --------------------------------- host --------------------------------- */
#define GRID 2048
/* a loop over the lattice blocks (a wave each) runs with the box's tuned
   shape, and no more workgroups than it has blocks for */
#define LAUNCH_P(k, ...)                                                                             \
  do {                                                                                               \
    const int wpb_ = d->block / 64;                                                                  \
    const int grid_ = std::min(d->grid, (d->nblk + wpb_ - 1) / wpb_);                                \
    hipLaunchKernelGGL(k, dim3(grid_), dim3(d->block), 0, d->c.stream, __VA_ARGS__);                 \
    CUBE_LAUNCH_CHECK();                                                                             \
  } while (0)

static Lat lat(const cube_dpm *d) { return Lat{d->p.ng, d->p.nf / d->p.ng, d->nb, d->nblk}; }
static Tiles tiles(const cube_dpm *d) {
  const int nt3 = d->ntile * d->ntile * d->ntile;
  return Tiles{d->tile, d->ntile, d->tcap, d->tcnt + d->tpar * nt3, d->tcnt + (1 - d->tpar) * nt3, d->tlist, d->trange};
}

/* rho of x (and delta), or the three cotangent meshes of coef*pbar */
static int tile_pass(cube_dpm *d, const float *x, int nc, float coef, int keep, unsigned *gmx, unsigned *gnext,
                     float *out, float *delta) {
  const int nt3 = d->ntile * d->ntile * d->ntile;
  const float inv_nbar = (float)((double)d->nf3 / (double)d->np);
#define TILE(T, NC, ZS, NT)                                                                                       \
  hipLaunchKernelGGL((k_dpm_tile<T, NC, ZS, NT>), dim3(nt3 * ZS), dim3(NT), 0, d->c.stream, x, d->pbar, coef, lat(d), \
                     d->p.nf, tiles(d), gmx, gnext, out, delta, inv_nbar)
  if (d->tile == 8) {
    if (nc == 1) TILE(8, 1, 1, 256);
    else TILE(8, 3, 1, 256);
  } else {
    if (nc == 1) TILE(16, 1, 1, 512);
    else TILE(16, 3, 2, 512); /* two workgroups per tile, 8 planes each */
  }
#undef TILE
  CUBE_LAUNCH_CHECK();
  if (!keep) d->tpar ^= 1; /* the next lists */
  return CUBE_OK;
}
static int reset(cube_dpm *d) {
  const int nt3 = d->ntile * d->ntile * d->ntile;
  hipLaunchKernelGGL(k_dpm_reset, dim3(std::min(256, (2 * nt3 + PT - 1) / PT)), dim3(PT), 0, d->c.stream, d->tcnt, 2 * nt3,
                     d->gmx);
  CUBE_LAUNCH_CHECK();
  d->tpar = 0;
  return CUBE_OK;
}
/* force mesh of the positions x, whose tile lists are built, into F (3 per
   point); rho stays in d->rho */
static int force_of(cube_dpm *d, const float *x, float *F, int keep, float *delta = nullptr) {
  int st = tile_pass(d, x, 1, 0.f, keep, nullptr, nullptr, d->rho, delta);
  if (st) return st;
  return cube_fft_poisson(&d->c, d->plan_f, d->rho, d->spec_f, d->work3_f, F, (float)d->p.nf);
}
/* the force mesh of the positions after s steps: kept for the adjoint, or the
   one buffer; after the last step in the cotangent meshes' room (unused by then) */
static float *force_slot(const cube_dpm *d, int s) {
  if (s == d->p.nsteps) return d->S;
  return d->force + (d->keep_force ? 3 * d->nf3 * s : 0);
}
/* where the positions after s steps are kept, or null; likewise the momenta */
static float *kept_x(const cube_dpm *d, int s) {
  if (s == d->p.nsteps) return d->xend;
  return s % d->every == 0 ? d->xs + (int64_t)(s / d->every) * d->npp * 3 : nullptr;
}
static float *kept_p(const cube_dpm *d, int s) {
  return d->ps && s < d->p.nsteps && s % d->every == 0 ? d->ps + (int64_t)(s / d->every) * d->npp * 3 : nullptr;
}

/* positions after s steps that were not kept, recomputed from the last kept
   step into d->x, their tile lists built */
static int recompute(cube_dpm *d, int s) {
  const int q0 = s - s % d->every;
  const float *x = kept_x(d, q0);
  CUBE_CHECK(hipMemcpyAsync(d->pw, kept_p(d, q0), d->npp * 3 * sizeof(float), hipMemcpyDeviceToDevice, d->c.stream));
  LAUNCH_P(k_dpm_bin, x, lat(d), d->p.nf, tiles(d));
  for (int q = q0; q < s; ++q) {
    int st = force_of(d, x, d->force, 0);
    if (st) return st;
    const double *c = d->steps + 3 * q;
    LAUNCH_P(k_dpm_step, x, d->pw, d->force, lat(d), d->p.nf, q > q0 ? 1 : 0, q > q0 ? (float)c[-1] : 0.f, 1, (float)c[0],
             (float)c[1], d->x, (float *)nullptr, tiles(d));
    x = d->x;
  }
  return CUBE_OK;
}

static int dalloc_f(float **p, int64_t n) {
  return hipMalloc((void **)p, (size_t)(n > 0 ? n : 1) * sizeof(float)) == hipSuccess ? CUBE_OK : CUBE_ERR_ALLOC;
}

extern "C" void cube_dpm_destroy(cube_dpm *d) {
  if (!d) return;
  void *ptrs[] = {d->amp, d->xs, d->ps, d->xend_own, d->x, d->pm, d->pw, d->rho, d->force, d->S, d->lam, d->spec_f,
                  d->work3_f, d->spec_g, d->work3_g, d->psi, d->xbar, d->pbar, d->gmx,
                  d->tcnt, d->tlist, d->trange};
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  cube_fft_destroy(d->plan_g);
  cube_fft_destroy(d->plan_f);
  if (d->c.stream) (void)hipStreamDestroy(d->c.stream);
  free(d->steps);
  free(d);
}

extern "C" int cube_dpm_create(const cube_dpm_params *p, cube_dpm **out) {
  if (!p || !out || p->ng < 4 || p->nf < p->ng || p->nf % p->ng || p->nsteps < 1) return CUBE_ERR_INVALID;
  static_assert(2048 / 4 <= 1023, "the largest lattice's blocks fit blk_pack's fields");
  CUBE_CHECK(hipSetDevice(p->device));
  cube_dpm *d = (cube_dpm *)calloc(1, sizeof(cube_dpm));
  if (!d) return CUBE_ERR_ALLOC;
  d->p = *p;
  d->c.device = p->device;
  d->grid = GRID;
  d->block = PT;
  d->np = d->ng3 = (int64_t)p->ng * p->ng * p->ng;
  d->nf3 = (int64_t)p->nf * p->nf * p->nf;
  d->sg = (int64_t)cube_spec_pitch(p->ng) * p->ng * p->ng;
  d->sf = (int64_t)cube_spec_pitch(p->nf) * p->nf * p->nf;
  d->steps = (double *)calloc(3 * p->nsteps, sizeof(double));
  int st = d->steps ? CUBE_OK : CUBE_ERR_ALLOC;
  if (!st && hipStreamCreate(&d->c.stream) != hipSuccess) st = CUBE_ERR_HIP;
  if (!st) st = cube_fft_create(&d->c, p->ng, &d->plan_g);
  if (!st) st = cube_fft_create(&d->c, p->nf, &d->plan_f);
  /* lattice blocks (a wave each; slots of lattice points past ng stay unused) and the mesh's tiles */
  d->nb = (p->ng + 3) / 4;
  d->nblk = d->nb * d->nb * d->nb;
  d->npp = (int64_t)d->nblk * 64;
  d->tile = p->nf <= 128 ? 8 : 16;
  d->ntile = (p->nf + d->tile - 1) / d->tile;
  const int nt3 = d->ntile * d->ntile * d->ntile;
  {
    /* room for 24 times the mean list (a box whose blocks spread over two more cells) */
    const double per = (4.0 * (p->nf / p->ng) + 4.0) / d->tile + 1.0;
    const double mean = (double)d->nblk * per * per * per / nt3;
    d->tcap = (int)std::min<double>(d->nblk, std::max(64.0, 24.0 * mean));
  }
  const int64_t np3 = d->npp * 3;
  /* What the adjoint finds.  checkpoint: the positions of every step, and
     their force meshes while there is room (dpm_keep_force), else they are
     formed again.  No checkpoint: the positions of every step if those after
     the initial ones take at most 24 bytes per mesh point, else position and
     momentum of every `every`-th step within those 24 bytes (of one step at
     least), recomputed from there with 36 bytes per slot to work in. */
  d->every = 1;
  int64_t nx = p->nsteps + 1, nps = 0;
  if (!p->checkpoint && p->nsteps * 12 * d->npp > 24 * d->nf3) {
    const int64_t k = std::max<int64_t>(1, 24 * d->nf3 / (24 * d->npp));
    d->every = (int)((p->nsteps + k - 1) / k);
    nx = (p->nsteps - 1) / d->every + 1;
    nps = nx;
  }
  const bool own_end = d->every > 1;
  int64_t base = 0; /* bytes of the arrays below */
  auto get = [&](float **q, int64_t n) {
    if (!st) st = dalloc_f(q, n);
    base += n * (int64_t)sizeof(float);
  };
  get(&d->amp, (int64_t)p->ng * p->ng * (p->ng / 2 + 1));
  get(&d->xs, nx * np3);
  if (nps) get(&d->ps, nps * np3);
  if (own_end) get(&d->xend_own, np3);
  if (!st) d->xend = own_end ? d->xend_own : d->xs + (int64_t)p->nsteps * np3;
  if (own_end) get(&d->x, np3);
  if (own_end) get(&d->pw, np3);
  get(&d->pm, np3);
  get(&d->rho, d->nf3);
  get(&d->S, 3 * d->nf3);
  get(reinterpret_cast<float **>(&d->gmx), 2 * DPM_GMX);
  get(&d->lam, d->nf3);
  get((float **)&d->spec_f, 2 * d->sf);
  get((float **)&d->work3_f, 6 * d->sf);
  get((float **)&d->spec_g, 2 * d->sg);
  get((float **)&d->work3_g, 6 * d->sg);
  get(&d->psi, 3 * d->ng3);
  get(&d->xbar, np3);
  get(&d->pbar, np3);
  get(reinterpret_cast<float **>(&d->tcnt), 2 * nt3);
  get(reinterpret_cast<float **>(&d->tlist), (int64_t)nt3 * d->tcap);
  get(reinterpret_cast<float **>(&d->trange), 2 * (int64_t)d->nblk);
  if (p->checkpoint && p->nsteps == 1) d->keep_force = 1; /* in the one mesh */
  if (!st && p->checkpoint && p->nsteps > 1) {
    const int64_t mesh = 3 * d->nf3 * (int64_t)sizeof(float), extra = (p->nsteps - 1) * mesh;
    size_t fr = 0, tot = 0;
    if (hipMemGetInfo(&fr, &tot) == hipSuccess && (int64_t)fr > mesh &&
        dpm_keep_force(fr - mesh, tot, base + mesh, extra, d->nf3, d->np)) {
      if (dalloc_f(&d->force, p->nsteps * 3 * d->nf3) == CUBE_OK)
        d->keep_force = 1;
      else
        (void)hipGetLastError(); /* no room after all: the one mesh below */
    }
  }
  if (!d->force) get(&d->force, 3 * d->nf3);
  if (!st && hipStreamSynchronize(d->c.stream) != hipSuccess) st = CUBE_ERR_HIP;
  if (st) {
    cube_dpm_destroy(d);
    return st;
  }
  *out = d;
  return CUBE_OK;
}

extern "C" int cube_dpm_set_amplitude(cube_dpm *d, const float *amp) {
  if (!d || !amp) return CUBE_ERR_INVALID;
  CUBE_CHECK(hipSetDevice(d->p.device));
  const int ng = d->p.ng;
  CUBE_CHECK(hipMemcpy(d->amp, amp, (size_t)ng * ng * (ng / 2 + 1) * sizeof(float), hipMemcpyHostToDevice));
  return CUBE_OK;
}

extern "C" int cube_dpm_set_schedule(cube_dpm *d, const double *ic, const double *steps) {
  if (!d || !ic || !steps) return CUBE_ERR_INVALID;
  d->ic[0] = ic[0];
  d->ic[1] = ic[1];
  memcpy(d->steps, steps, 3 * d->p.nsteps * sizeof(double));
  return CUBE_OK;
}

extern "C" int cube_dpm_forward(cube_dpm *d, const float *noise, float *delta) {
  if (!d || !noise || !delta) return CUBE_ERR_INVALID;
  CUBE_CHECK(hipSetDevice(d->p.device));
  const int S = d->p.nsteps, nf = d->p.nf;
  int st = reset(d);
  if (st) return st;
  if ((st = cube_fft_filter3(&d->c, d->plan_g, noise, d->amp, d->spec_g, d->work3_g, d->psi))) return st;
  const float *x = kept_x(d, 0);
  LAUNCH_P(k_dpm_ic_particles, d->psi, lat(d), nf, (float)nf / (float)d->p.ng, (float)d->ic[0], (float)d->ic[1],
           1.f / (float)d->ng3, kept_x(d, 0), d->pm, tiles(d));
  for (int s = 0; s <= S; ++s) {
    const int last = s == S;
    float *F = force_slot(d, s);
    /* the last density is the output's too */
    if ((st = force_of(d, x, F, 0, last ? delta : nullptr))) return st;
    const double *c = d->steps + 3 * s; /* c[-1]: the closing kick of the step before */
    float *xn = last ? nullptr : kept_x(d, s + 1);
    if (!last && !xn) xn = d->x;
    LAUNCH_P(k_dpm_step, x, d->pm, F, lat(d), nf, s > 0 ? 1 : 0, s > 0 ? (float)c[-1] : 0.f, last ? 0 : 1,
             last ? 0.f : (float)c[0], last ? 0.f : (float)c[1], xn, kept_p(d, s), tiles(d));
    x = xn;
  }
  d->has_forward = 1;
  return CUBE_OK;
}

extern "C" int cube_dpm_adjoint(cube_dpm *d, const float *delta_bar, float *noise_bar) {
  if (!d || !delta_bar || !noise_bar) return CUBE_ERR_INVALID;
  if (!d->has_forward) return CUBE_ERR_STATE;
  CUBE_CHECK(hipSetDevice(d->p.device));
  const int S = d->p.nsteps, nf = d->p.nf;
  const float r = (float)nf / (float)d->p.ng, cx = (float)d->ic[0], cp = (float)d->ic[1];
  /* the cotangent on F at step s: kick A of s and kick B of s-1 share it */
  auto coef = [&](int s) -> float {
    return (float)(d->steps[3 * s] + (s > 0 ? d->steps[3 * (s - 1) + 2] : 0.0));
  };
  auto drift = [&](int s) -> float { return (float)d->steps[3 * s + 1]; };
  unsigned *gmx[2] = {d->gmx, d->gmx + DPM_GMX};
  int st = reset(d);
  if (st) return st;
  /* final density: delta = rho/nbar - 1, then the last step's drift^T */
  LAUNCH_P(k_dpm_grad, d->xend, lat(d), nf, delta_bar, (float)((double)d->nf3 / (double)d->np), 0.f, (const float *)nullptr,
           1, d->xbar, d->pbar, drift(S - 1), coef(S - 1), gmx[(S - 1) & 1], (const float *)kept_x(d, S - 1), tiles(d),
           (float *)nullptr, 0.f, 0.f, 0.f);
  const float slam = 1.f / ((float)nf * (float)nf * (float)nf);
  for (int s = S - 1; s >= 0; --s) {
    const float *x = kept_x(d, s);
    if (!x) {
      if ((st = recompute(d, s))) return st;
      x = d->x;
    }
    const float *M = force_slot(d, s);
    if (!d->keep_force && (st = force_of(d, x, d->force, 1))) return st;
    if ((st = tile_pass(d, x, 3, coef(s), 0, gmx[s & 1], gmx[(s + 1) & 1], d->S, nullptr))) return st;
    if ((st = cube_fft_filter3_t(&d->c, d->plan_f, d->S, nullptr, d->spec_f, d->work3_f, d->lam))) return st;
    if (s > 0)
      LAUNCH_P(k_dpm_grad, x, lat(d), nf, d->lam, slam, coef(s), M, 0, d->xbar, d->pbar, drift(s - 1), coef(s - 1),
               gmx[(s - 1) & 1], (const float *)kept_x(d, s - 1), tiles(d), (float *)nullptr, 0.f, 0.f, 0.f);
    else
      LAUNCH_P(k_dpm_grad, x, lat(d), nf, d->lam, slam, coef(s), M, 0, d->xbar, d->pbar, 0.f, 0.f, gmx[0],
               (const float *)nullptr, tiles(d), d->psi, cx, cp, r);
  }
  /* ICs^T: noise_bar = (1/ng^3) IFFT[sum_d -i K_d A FFT(psibar_d)] */
  if ((st = cube_fft_filter3_t(&d->c, d->plan_g, d->psi, d->amp, d->spec_g, d->work3_g, noise_bar))) return st;
  hipLaunchKernelGGL(k_dpm_scale_to, dim3((unsigned)std::min<int64_t>(GRID, (d->ng3 + PT - 1) / PT)), dim3(PT), 0,
                     d->c.stream, noise_bar, noise_bar, d->ng3, 1.f / (float)d->ng3);
  CUBE_LAUNCH_CHECK();
  return CUBE_OK;
}

extern "C" int cube_dpm_state(cube_dpm *d, float *x, float *p) {
  if (!d) return CUBE_ERR_INVALID;
  if (!d->has_forward) return CUBE_ERR_STATE;
  CUBE_CHECK(hipSetDevice(d->p.device));
  if (x || p) LAUNCH_P(k_dpm_state, d->xend, d->pm, lat(d), d->p.nf, x, p); /* held as displacements */
  return CUBE_OK;
}

extern "C" int cube_dpm_sync(cube_dpm *d) {
  if (!d) return CUBE_ERR_INVALID;
  CUBE_CHECK(hipStreamSynchronize(d->c.stream));
  return CUBE_OK;
}
