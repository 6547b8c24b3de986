/*
 * cube_mesh.hip -- CIC deposits, force gathers (kicks) and the Green's
 * functions of particle_mesh (W/pm.f90) and kernel_f/kernel_c
 * (W/kernel_f.f90, W/kernel_c.f90) for a single image.
 *
 * Deposits are deterministic gathers: one thread per mesh cell walks the
 * few source coarse cells that can reach it in the reference's own visit
 * order (ilayer, k, j, i, l) with nlayer=3, re-evaluates each particle's
 * real(4) CIC weights with the reference's expression in the owning tile's
 * frame, and adds them in that order -- so every physical cell holds the
 * bit pattern the reference's layered OpenMP loop produces for it.
 */
#include "cube_internal.h"
#include <math.h>
#include <stdlib.h>
#include <string.h>

#define MT 256

/* the coarse CIC coordinate ((cell-1)+(x offset))-0.5 of W/pm.f90:213,335
   rounded to real(4); c = cell-1 (tile frame or global).  With 1-byte codes
   c + (u+0.5)/256 has at most 24 significant bits for c < 2^15, so the
   real(4) sums are exact and round as the real(8) form does; 2-byte codes
   keep the real(8) form. */
template <int IX> __device__ __forceinline__ float coarse_tempx(int c, int32_t code) {
  if constexpr (IX == 1)
    return ((float)c + ((float)cube_ucode(IX, code) + 0.5f) * 0x1p-8f) - 0.5f;
  else
    return (float)(((double)c + cube_xoff(IX, code)) - 0.5);
}
/* sum of nb partials in a fixed order (thread t takes b = t mod 64, then a
   tree over the threads), so the sum repeats bit for bit */
__global__ __launch_bounds__(64) void k_sum_parts1(const double *part, int nb, double *out) {
  __shared__ double r[64];
  const int t = threadIdx.x;
  double s = 0;
  for (int b = t; b < nb; b += 64) s += part[b];
  r[t] = s;
  __syncthreads();
  for (int o = 32; o > 0; o >>= 1) {
    if (t < o) r[t] += r[t + o];
    __syncthreads();
  }
  if (t == 0) *out = r[0];
}

__device__ __forceinline__ int rl_i(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
/*
 * Coarse deposit, W/pm.f90:205-267: one wave per block of 4x4x4 mesh cells of
 * a tile (clipped at the tile's high edge), one lane per mesh cell.  A mesh
 * cell sums the hits of its 3^3 source cells in the reference's order
 * (ilayer = k mod 3, j, i, l); the block's sources are the 6^3 cells around
 * it.  Source planes 3 apart have the same ilayer and no mesh cell needs
 * both, so the wave works in three phases of two planes each: every lane has
 * exactly one of the two planes to read in each phase, and the phases in
 * order of ilayer give every lane the reference's order.
 *
 * A phase stages its 12 rows of 6 cells in LDS, a row padded to batches of
 * 64 particles, as the own-cell weights in fixed point (one word per
 * particle) and three 64-bit ballots per batch: which particles sit in the
 * upper half of their cell on each axis.  A particle in the upper half
 * reaches its own and the next mesh cell, else its own and the one before, so
 * a lane gets the hits of three cells of a row from a few logic operations
 * and walks only those, in slot order = reference order.  A particle that
 * misses a mesh cell would add +0.0, which leaves a sum of non-negative
 * terms unchanged, so nothing is lost by not visiting it.
 *
 * A phase with more than `heavy_at` particles (a clustered region) or more
 * batches than are staged at once goes through its particles 64 at a time
 * instead: the wave forms the 27 terms of each (zero where it misses) in LDS
 * and each lane adds its column, two instructions per particle, so a halo of
 * thousands of particles costs its additions and not a walk each.
 *
 * PACK, for boxes of few particles: a phase of at most CD_PACK particles is
 * staged with its rows one behind the other, where a batch of its own for each
 * row of 6 cells was nearly empty.  One particle a cell: 210 instead of 260 us
 * on 128^3, 290 instead of 470 on one tile of 144^3 with 2-byte codes (where
 * rounding makes a slot's fields longest); 152 instead of 202 on 128^3 with one
 * particle in 8 cells.
 *
 * What bounds it: VALU work (the hit loop above all) at 16 waves per CU (9.4
 * KB of LDS per wave, 4 waves per SIMD by registers), on small meshes the one
 * chain of dependent loads of a wave, and with halos the additions of the
 * fullest block.  Alone on one MI355X, against one lane per 2^3 mesh cells
 * with the sources read where they lie: 32^3 particles 0.046 ms (was 0.24),
 * 128^3 0.08 (0.30), 256^3 with 2-byte codes at z = 3 0.92 (1.90), 512^3 2.2
 * (3.35), 128^3 at z = 0.5 with cells of up to 2300 particles 0.48 (4.6).
 */
template <int IX> struct CdWord;
template <> struct CdWord<1> { /* bytes q: own weight (2q+257)/512, the neighbour's (255-2q)/512 */
  typedef uint32_t T;
  static constexpr float H = 256.f, scale = 0x1p-27f; /* half a cell; 1/(2H)^3 */
  static constexpr int field = 8, NB = 16; /* NB: batches of 64 slots staged at once */
};
template <> struct CdWord<2> { /* 21-bit fields q: own weight (65536+q)/2^17, the neighbour's (65536-q)/2^17 */
  typedef uint64_t T;
  static constexpr float H = 65536.f, scale = 0x1p-51f;
  static constexpr int field = 21, NB = 14; /* 12 rows, a few of them over 64 particles */
};
/* the staged fields of a particle's codes (in the low bytes of `raw`) and a
   word with the top bit of axis a's field position set where corner 1 of the
   cloud is the particle's own cell (the upper half).  The own weight is d1
   there and 1-d1 in the lower half, both exact.  EX: tempx is exact in
   real(4) in every cell of the tile, so the weights are those of the code
   alone; else they come from tempx as the reference rounds it in cell c
   (0-based, tile frame) */
template <int IX, bool EX>
__device__ __forceinline__ typename CdWord<IX>::T cd_fields(typename CdWord<IX>::T raw, const int c[3], bool up[3]) {
  if constexpr (IX == 1) {
    /* upper: 255-u, lower: u, all three bytes at once */
    const uint32_t h = (raw >> 7) & 0x010101u;
#pragma unroll
    for (int a = 0; a < 3; ++a) up[a] = (raw & (0x80u << (8 * a))) != 0u;
    return (raw & 0xffffffu) ^ (h * 255u);
  } else {
    uint64_t w = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const uint32_t u = (uint32_t)(raw >> (16 * a)) & 0xffffu;
      uint32_t q;
      if constexpr (EX) {
        up[a] = u >= 32768u;
        q = (2u * u + 1u) ^ (up[a] ? 0x1ffffu : 0u); /* upper: 131071 - (2u+1), */
        q += up[a] ? 1u : 0u;                        /* so 131072 - (2u+1), 17 bits */
      } else {
        const float tempx = coarse_tempx<2>(c[a], (int32_t)u);
        const int i1 = (int)floorf(tempx) + 1;
        const float d1 = (float)i1 - tempx;
        up[a] = i1 == c[a] + 1;
        q = (uint32_t)((up[a] ? d1 : 1.0f - d1) * 131072.f) - 65536u;
      }
      w |= (uint64_t)q << (21 * a);
    }
    return w;
  }
}
/* axis a's field of a staged word, q of CdWord */
template <int IX> __device__ __forceinline__ float cd_q(typename CdWord<IX>::T w, int a) {
  if constexpr (IX == 1) return (float)((w >> (8 * a)) & 0xff);
  else return (float)(uint32_t)((w >> (21 * a)) & 0x1fffff);
}
/* a weight in units of 1/(2H), s = 1 the own cell's and -1 the neighbour's: H +
   s*t as q*cd_mul(s) + cd_add(s), t = 2q+1 (1-byte codes) or q */
template <int IX> __device__ __forceinline__ float cd_mul(float s) { return IX == 1 ? 2.f * s : s; }
template <int IX> __device__ __forceinline__ float cd_add(float s) { return IX == 1 ? CdWord<IX>::H + s : CdWord<IX>::H; }
/* the codes of particle p as stored: one 4- or 8-byte read of its 3 or 6
   bytes (the particle arrays end in padding) */
template <int IX>
__device__ __forceinline__ typename CdWord<IX>::T cd_load(const char *__restrict__ q) {
  typename CdWord<IX>::T v;
  __builtin_memcpy(&v, q, sizeof(v));
  return v;
}

template <int IX> struct CdLds { /* per wave */
  union {
    typename CdWord<IX>::T word[CdWord<IX>::NB * 64];
    float term[27 * 65 + 8]; /* 27 columns of 64 terms, in 27 different banks; read up to 7 past a column's end */
  };
  uint64_t up[CdWord<IX>::NB][3];
  int64_t start[36][3]; /* a row's first particle, and that of its cells iL and iE */
  int pre[36][7]; /* first particle of each cell of a row, counted from the row's first */
  int rb[12];     /* first slot (PACK) or batch of each row of the phase */
  int cax[3][6];  /* a source cell's id is the sum of its three axes' parts */
};
/* bits [0, p), p clipped to [0, 64] */
__device__ __forceinline__ uint64_t bits_below(int p) {
  p = max(p, 0);
  return p >= 64 ? ~0ull : (1ull << p) - 1ull;
}
__device__ __forceinline__ int64_t rl_i64(int64_t v, int l) {
  return (int64_t)(((uint64_t)(uint32_t)rl_i((int)(v >> 32), l) << 32) | (uint64_t)(uint32_t)rl_i((int)(v & 0xffffffff), l));
}

#define CD_PACK 128 /* largest phase whose rows are staged without padding */

template <int IX, bool EX, int NW, bool PACK>
__global__ __launch_bounds__(64 * NW, 4) void k_coarse_deposit(const typename IntOf<IX>::T *__restrict__ xp,
                                                            const int32_t *__restrict__ rhoc,
                                                            const int64_t *__restrict__ cstart, Geo g, float mass,
                                                            float *__restrict__ r3, double *__restrict__ part,
                                                            int nblk, int heavy_at) {
  typedef typename CdWord<IX>::T W;
  constexpr float H = CdWord<IX>::H, SC = CdWord<IX>::scale;
  constexpr int PB = 3 * IX; /* bytes per particle */
  __shared__ CdLds<IX> lds[NW];
  __shared__ double wsum[NW];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  CdLds<IX> &S = lds[wv];
  const char *xb8 = reinterpret_cast<const char *>(xp);
  const int nt = g.nt, nbt = (nt + 3) / 4;
  const int xi = lane & 3, yi = (lane >> 2) & 3, zi = lane >> 4;
  double tsum = 0;
  for (int b = blockIdx.x * NW + wv; b < nblk; b += gridDim.x * NW) {
    /* the block: tile T, first mesh cell m0 (0-based, tile frame) */
    const uint32_t ub = (uint32_t)b, un = (uint32_t)nbt, q1 = ub / un, q2 = q1 / un, t = q2 / un;
    const uint32_t tn = (uint32_t)g.nnt, t1 = t / tn;
    const int T[3] = {(int)(t - t1 * tn), (int)(t1 % tn), (int)(t1 / tn)};
    const int m0[3] = {4 * (int)(ub - q1 * un), 4 * (int)(q1 - q2 * un), 4 * (int)(q2 - t * un)};
    /* a row's particles are contiguous but for the cells of the neighbour
       tiles: cell 0 at the tile's low edge, cell iE on at its high edge */
    const int iL = m0[0] == 0 ? 1 : 0, iE = nt - (m0[0] - 1);
    const bool oneseg = iL == 0 && iE >= 6; /* uniform */
    /* starts of the 6^3 source cells m0-1..m0+4 (those past the tile's next
       cell are not needed: empty), then prefix sums along each row of 6 */
    if (lane < 18) {
      const int a = lane / 6, sc = (a == 0 ? m0[0] : a == 1 ? m0[1] : m0[2]) - 1 + lane % 6;
      int ta = a == 0 ? T[0] : a == 1 ? T[1] : T[2];
      int l = sc;
      if (sc < 0) { l = nt - 1; ta = ta > 0 ? ta - 1 : g.nnt - 1; }
      if (sc == nt) { l = 0; ta = ta < g.nnt - 1 ? ta + 1 : 0; }
      const int st = a == 0 ? 1 : a == 1 ? nt : nt * nt, ts = a == 0 ? 1 : a == 1 ? g.nnt : g.nnt * g.nnt;
      S.cax[a][lane % 6] = sc > nt ? -1 : l * st + nt * nt * nt * ts * ta;
    }
    wave_lds_sync();
    int cnt4[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int q = lane + 64 * u;
      cnt4[u] = 0;
      if (q < 216) {
        const int cx = S.cax[0][q % 6], cy = S.cax[1][(q / 6) % 6], cz = S.cax[2][q / 36];
        if ((cx | cy | cz) >= 0) {
          const int cc = cx + cy + cz;
          cnt4[u] = rhoc[cc];
          const int sx = q % 6;
          const int64_t st = cstart[cc];
          if (sx == 0) S.start[q / 6][0] = st;
          if (sx == iL) S.start[q / 6][1] = st;
          if (sx == iE) S.start[q / 6][2] = st;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (lane + 64 * u < 216) S.pre[(lane + 64 * u) / 6][(lane + 64 * u) % 6 + 1] = cnt4[u];
    wave_lds_sync();
    if (lane < 36) {
      int acc = 0;
      S.pre[lane][0] = 0;
#pragma unroll
      for (int q = 1; q < 7; ++q) {
        acc += S.pre[lane][q];
        S.pre[lane][q] = acc;
      }
    }
    wave_lds_sync();
    float acc = 0.f;
    const int k0 = m0[2] % 3; /* 1-based local k of source plane s is m0z + s */
#pragma unroll 1
    for (int il = 0; il < 3; ++il) {
      const int s0 = (il - k0 + 3) % 3;      /* planes s0 and s0+3 */
      const int sz = s0 >= zi ? s0 : s0 + 3; /* this lane's, offset sz-zi-1 from its cell */
      /* lane t < 12 keeps row t of the phase (y = t/2, plane s0 + 3*(t&1)):
         particles, and where they start in memory per segment */
      const int rt = lane < 12 ? (s0 + 3 * (lane & 1)) * 6 + (lane >> 1) : 0;
      const int nrow = lane < 12 ? S.pre[rt][6] : 0;
      const int64_t dA = S.start[rt][0];
      int64_t dB = 0, dC = 0;
      int sB = 0, sC = 0;
      if (!oneseg) {
        sB = iL ? S.pre[rt][1] : 0;
        sC = iE < 6 ? S.pre[rt][iE] : nrow;
        dB = S.start[rt][1] - sB;
        dC = iE < 6 ? S.start[rt][2] - sC : 0;
      }
      const int nbr = (nrow + 63) >> 6;
      const int bsc = wave_incl_scan(nbr), psc = wave_incl_scan(nrow);
      const int nbat = rl_i(bsc, 11), npart = rl_i(psc, 11);
      const bool packed = PACK && npart <= CD_PACK && npart <= heavy_at; /* uniform */
      const int rb = packed ? psc - nrow : (PACK ? 64 : 1) * (bsc - nbr); /* see CdLds */
      if (lane < 12) S.rb[lane] = rb;
      /* row tr of the phase, wave-uniform (read from its lane before any
         branch that turns lanes off), and its particle l's codes as stored */
      struct Seg {
        int64_t a, b, c;
        int sb, sc, n;
      };
      auto seg = [&](int tr) -> Seg {
        Seg e = {rl_i64(dA, tr), 0, 0, 0, 0, rl_i(nrow, tr)};
        if (!oneseg) {
          e.b = rl_i64(dB, tr);
          e.c = rl_i64(dC, tr);
          e.sb = rl_i(sB, tr);
          e.sc = rl_i(sC, tr);
        }
        return e;
      };
      auto load = [&](const Seg &e, int l) -> W {
        if (oneseg) return cd_load<IX>(xb8 + e.a * PB + (uint32_t)(l * PB));
        const int64_t d = l < e.sb ? e.a : (l < e.sc ? e.b : e.c);
        return cd_load<IX>(xb8 + (d + l) * PB);
      };
      /* its staged word and halves (the row's cell only where rounding asks for it) */
      auto fields = [&](W raw, int tr, int l, bool up[3]) -> W {
        int c[3] = {0, 0, 0};
        if constexpr (!EX) {
          const int r = (s0 + 3 * (tr & 1)) * 6 + (tr >> 1);
          c[0] = m0[0] - 1;
#pragma unroll
          for (int q = 1; q < 6; ++q) c[0] += S.pre[r][q] <= l ? 1 : 0;
          c[1] = m0[1] - 1 + (tr >> 1);
          c[2] = m0[2] - 1 + s0 + 3 * (tr & 1);
        }
        return cd_fields<IX, EX>(raw, c, up);
      };
      wave_lds_sync();
      if (packed || (nbat <= CdWord<IX>::NB && npart <= heavy_at)) {
        auto put = [&](W raw, int q, int tr, int l) {
          bool up[3];
          const W w = fields(raw, tr, l, up);
          const uint64_t u0 = __ballot(up[0]), u1 = __ballot(up[1]), u2 = __ballot(up[2]);
          S.word[q * 64 + lane] = w;
          if (lane < 3) S.up[q][lane] = lane == 0 ? u0 : (lane == 1 ? u1 : u2);
        };
        if (packed) {
#pragma unroll 1
          for (int q = 0; q * 64 < npart; ++q) {
            const int i = q * 64 + lane;
            int tr = 0; /* its row */
#pragma unroll
            for (int t = 1; t < 12; ++t) tr += rl_i(rb, t) <= i ? 1 : 0;
            const int l = i - S.rb[tr], r = (s0 + 3 * (tr & 1)) * 6 + (tr >> 1);
            W raw = 0;
            if (i < npart) {
              int64_t d = S.start[r][0];
              if (!oneseg) {
                const int eB = iL ? S.pre[r][1] : 0, eC = iE < 6 ? S.pre[r][iE] : npart;
                if (l >= eB) d = S.start[r][1] - eB;
                if (l >= eC) d = S.start[r][2] - eC;
              }
              raw = cd_load<IX>(xb8 + (d + l) * PB);
            }
            put(raw, q, tr, l);
          }
        } else {
          /* the first batch of every row is on its way before one is used */
          W raw[12];
#pragma unroll
          for (int tr = 0; tr < 12; ++tr) {
            raw[tr] = 0;
            const Seg e = seg(tr);
            if (lane < e.n) raw[tr] = load(e, lane);
          }
#pragma unroll
          for (int tr = 0; tr < 12; ++tr)
            if (rl_i(nrow, tr) > 0) put(raw[tr], rl_i(rb, tr) >> (PACK ? 6 : 0), tr, lane);
          if (__ballot(nrow > 64)) {
#pragma unroll 1
            for (int tr = 0; tr < 12; ++tr) {
              const Seg e = seg(tr);
              for (int o = 64; o < e.n; o += 64) {
                W w = 0;
                if (o + lane < e.n) w = load(e, o + lane);
                put(w, (rl_i(rb, tr) >> (PACK ? 6 : 0)) + (o >> 6), tr, o + lane);
              }
            }
          }
        }
        wave_lds_sync();
        const int oz = sz - zi - 1;
        const float zs = oz == 0 ? 1.f : -1.f, mz = cd_mul<IX>(zs) * SC, az = cd_add<IX>(zs) * SC;
#pragma unroll 1
        for (int j = 0; j < 3; ++j) { /* rows y-1, y, y+1 */
          const int sy = yi + j, r = sz * 6 + sy, tr = 2 * sy + (sz >= 3 ? 1 : 0);
          const int rb = S.rb[tr], r0 = PACK ? rb : 0, q0 = PACK ? 0 : rb;
          const int pA = r0 + S.pre[r][xi], pB = r0 + S.pre[r][xi + 1], pC = r0 + S.pre[r][xi + 2], pD = r0 + S.pre[r][xi + 3];
          const float ys = j == 1 ? 1.f : -1.f, my = cd_mul<IX>(ys), ay = cd_add<IX>(ys);
          for (int bb = pA >> 6; bb * 64 < pD; ++bb) {
            const int q = q0 + bb, o = 64 * bb;
            const uint64_t ux = S.up[q][0], uy = S.up[q][1], uz = S.up[q][2];
            const uint64_t fA = bits_below(pA - o), fB = bits_below(pB - o), fC = bits_below(pC - o), fD = bits_below(pD - o);
            uint64_t m = ((fB & ~fA) & ux) | (fC & ~fB) | ((fD & ~fC) & ~ux);
            m &= j == 0 ? uy : (j == 1 ? ~0ull : ~uy);
            m &= oz < 0 ? uz : (oz == 0 ? ~0ull : ~uz);
            const uint32_t xb = (uint32_t)(pB - o), xn = (uint32_t)(pC - pB);
            const W *wd = S.word + q * 64;
            /* two hits per turn, so that two words are on their way at once;
               without a second one its term is +0 */
            while (m) {
              const int i0 = __builtin_ctzll(m);
              m &= m - 1ull;
              const bool two = m != 0ull;
              const int i1 = two ? __builtin_ctzll(m) : i0;
              m &= m - 1ull; /* 0 stays 0 */
              const W w0 = wd[i0], w1 = wd[i1];
              const float s0x = (uint32_t)i0 - xb < xn ? 1.f : -1.f, s1x = (uint32_t)i1 - xb < xn ? 1.f : -1.f;
              const float x0 = fmaf(cd_q<IX>(w0, 0), cd_mul<IX>(s0x), cd_add<IX>(s0x));
              const float x1 = fmaf(cd_q<IX>(w1, 0), cd_mul<IX>(s1x), cd_add<IX>(s1x));
              const float y0 = fmaf(cd_q<IX>(w0, 1), my, ay), y1 = fmaf(cd_q<IX>(w1, 1), my, ay);
              const float z0 = fmaf(cd_q<IX>(w0, 2), mz, az), z1 = fmaf(cd_q<IX>(w1, 2), mz, az);
              /* the reference's ((wx*wy)*wz)*mass: the units are powers of two */
              const float e0 = x0 * y0 * z0 * mass, e1 = x1 * y1 * z1 * mass;
              acc = acc + e0;
              acc = acc + (two ? e1 : 0.f);
            }
          }
        }
      } else {
#pragma unroll 1
        for (int tr = 0; tr < 12; ++tr) {
          const int sy = tr >> 1, sp = s0 + 3 * (tr & 1), r = sp * 6 + sy;
          const Seg e = seg(tr);
          const int n = e.n;
          const bool mine = sp == sz && sy >= yi && sy <= yi + 2;
          const int col = ((sp - zi) * 3 + (sy - yi)) * 3; /* +0, 1, 2 for the cells x-1, x, x+1 */
          int pr[7];
#pragma unroll
          for (int q = 0; q < 7; ++q) pr[q] = __builtin_amdgcn_readfirstlane(S.pre[r][q]);
          W next = 0;
          if (lane < n) next = load(e, lane);
          for (int o = 0; o < n; o += 64) {
            const int m = min(64, n - o);
            const W raw = next; /* the next batch is on its way while this one is added */
            if (o + 64 + lane < n) next = load(e, o + 64 + lane);
            if (lane < m) {
              bool up[3];
              const W f = fields(raw, tr, o + lane, up);
              float w[3][3]; /* weights for a mesh cell one above, at and one below the particle's */
#pragma unroll
              for (int a = 0; a < 3; ++a) {
                const float q = cd_q<IX>(f, a), k = a == 2 ? SC : 1.f;
                const float nb = fmaf(q, cd_mul<IX>(-1.f), cd_add<IX>(-1.f)) * k;
                w[a][0] = up[a] ? nb : 0.f;
                w[a][1] = fmaf(q, cd_mul<IX>(1.f), cd_add<IX>(1.f)) * k;
                w[a][2] = up[a] ? 0.f : nb;
              }
#pragma unroll
              for (int y = 0; y < 3; ++y)
#pragma unroll
                for (int x = 0; x < 3; ++x) {
                  const float wxy = w[0][x] * w[1][y];
#pragma unroll
                  for (int z = 0; z < 3; ++z) S.term[((z * 3 + y) * 3 + x) * 65 + lane] = wxy * w[2][z] * mass;
                }
            }
            wave_lds_sync();
            /* cell by cell of the row, so that the slots are the same for
               every lane and a crowded cell is gone through once */
#pragma unroll
            for (int cx = 0; cx < 6; ++cx) {
              const int lo = max(pr[cx] - o, 0), hi = min(pr[cx + 1] - o, m);
              if (lo < hi && mine && (unsigned)(cx - xi) <= 2u) {
                const float *c = S.term + (col + cx - xi) * 65;
                for (int i = lo; i < hi; i += 8) {
                  float v[8];
#pragma unroll
                  for (int k = 0; k < 8; ++k) v[k] = c[i + k];
#pragma unroll
                  for (int k = 0; k < 8; ++k) acc = acc + (i + k < hi ? v[k] : 0.f);
                }
              }
            }
            wave_lds_sync();
          }
        }
      }
      wave_lds_sync(); /* rb, word and up are read until here */
    }
    if (m0[0] + xi < nt && m0[1] + yi < nt && m0[2] + zi < nt) {
      const int64_t X = T[0] * nt + m0[0] + xi, Y = T[1] * nt + m0[1] + yi, Z = T[2] * nt + m0[2] + zi;
      r3[(Z * g.nc + Y) * g.nc + X] = acc;
      tsum += (double)acc;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) tsum += __shfl_xor(tsum, o, 64);
  if constexpr (NW == 1) {
    if (lane == 0) part[blockIdx.x] = tsum;
  } else {
    if (lane == 0) wsum[wv] = tsum;
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int w = 1; w < NW; ++w) tsum += wsum[w];
      part[blockIdx.x] = tsum;
    }
  }
}

/*
 * Fine deposit, W/pm.f90:49-108: one wave per block of 4x4x4 coarse cells of
 * a tile, a lane per coarse cell owning its 4x4x4 fine cells.  Every particle
 * that reaches them lives in the 2x2x2 source cells {C-1,C} per axis; the lane
 * adds their terms in the reference's order -- z by (ilayer, k), then y, x,
 * l -- into LDS accumulators, so each fine cell holds the reference's bits.
 *
 * The block's 5^3 source cells go through LDS in three phases by ilayer (the
 * planes of one ilayer are 3 apart, so a lane needs at most one of them), as
 * raw codes in batches of 64 slots with three ballots each: which particles
 * sit in the last fine sub-cell (code >> sh == 3) on each axis.  Only those
 * reach the next coarse cell, so a lane's hits of two cells of a row are a few
 * logic operations.  Where the real(4) coordinate is inexact (EX false:
 * 2-byte codes, nt > 128) the top code of a lower sub-cell can round up onto
 * the boundary itself, and its weight past it is then exactly 0: leaving it
 * out drops only +0 terms.
 *
 * A hit's two planes per axis that lie in the cell are b, b+1 with b = 0..2
 * and weights that are 0 where a plane lies outside, so its 8 sums sit at
 * constant distances from one address and need no bounds checks; a +0 term
 * leaves a sum as it is.
 *
 * A cell whose 8 sources hold more than `heavy_at` particles would hold its
 * wave up: its lane sits out, and the block goes to a list for
 * k_fine_deposit_heavy with the mask of such cells.
 *
 * A row takes batches of its own, ten of which hold a phase of the usual 8
 * particles a cell; slots then need no offsets and no lane's rows straddle
 * batches.  PACK stages a phase's rows one behind the other instead.  With one
 * particle a cell the ten batches were nearly empty: 416 -> 322 us on 128^3
 * cells, 588 -> 470 on one tile of 144^3 with 2-byte codes.  With 27 a phase is
 * 30 batches, and staged ten at a time each window has work for the lanes of a
 * few rows only; packed into 24 at once 275 -> 141 us on 32^3, 670 -> 440 on 64^3
 * (11, 14 and 18 at a time 512, 516 and 569, however many more waves fit), 1.08
 * -> 0.97 ms with halos.
 *
 * Bound by VALU issue (some 4,000 instructions a block, half of them the hits)
 * with the 16 KiB of sums leaving 7 waves a CU to hide the rest.  Both kernels
 * and the sum, against a thread per coarse cell walking its 8 cells in global
 * memory with crowded cells handed round its wave: 5.12 -> 3.05 ms on the
 * 256^3 mesh of 512^3 particles, 1.79 -> 1.16 ms on
 * 128^3 at z = 3, 0.117 -> 0.086 ms on 64^3, 0.057 -> 0.045 ms on 16^3, 1.48
 * -> 0.68 ms on the clustered 128^3 at z = 0 with 1-byte codes.
 */
template <int IX, int NB> struct FdLds { /* per wave; NB: batches staged at once */
  float acc[64 * 64];                         /* fine cell q of lane t at q*64 + t: conflict free */
  typename CdWord<IX>::T word[NB * 64];
  uint64_t top[NB][3];
  int64_t start[25][2]; /* a row's first particle, and that of its second cell */
  int pre[25][6];
  int rb[2][10]; /* a row's first batch (PACK: first slot), by phase parity */
  int cax[3][5];
};
/* the two planes b, b+1 of an axis and their weights: a particle of code u in
   the lane's own cell, or (below) in the last sub-cell of the one below.  EX
   as in cd_fields; else ci is the particle's cell and C the lane's (1-based,
   tile frame) */
template <int IX, bool EX>
__device__ __forceinline__ void fd_axis(uint32_t u, bool below, int ci, int C, int &b, float &wa, float &wb) {
  if constexpr (EX) {
    constexpr int sh = IX == 1 ? 6 : 14;
    constexpr float s = 1.0f / (float)(1 << sh);
    const float k = (float)(u & ((1u << sh) - 1u));
    const float d1 = fmaf(k, -s, 1.0f - 0.5f * s), d2 = fmaf(k, s, 0.5f * s); /* exact */
    const int sub = (int)(u >> sh);
    const bool last = sub == 3;
    b = below ? 0 : min(sub, 2);
    wa = below ? d2 : (last ? 0.f : d1);
    wb = below ? 0.f : (last ? d1 : d2);
  } else {
    /* ncell*(i-1)+ncell*(x offset) rounded to real(4) (W/pm.f90:63): both terms
       are exact floats, so one float add rounds it */
    const float off4 = ((float)u + 0.5f) * (IX == 1 ? 0x1p-6f : 0x1p-14f);
    const float tempx = (float)(4 * (ci - 1)) + off4;
    const int i1 = (int)floorf(tempx) + 1, r = i1 - 4 * (C - 1) - 1;
    const float d1 = (float)i1 - tempx, d2 = 1.0f - d1;
    b = min(max(r, 0), 2);
    wa = r == b ? d1 : (r + 1 == b ? d2 : 0.f);
    wb = r == b + 1 ? d1 : (r == b ? d2 : 0.f);
  }
}
template <int IX> __device__ __forceinline__ uint32_t fd_code(typename CdWord<IX>::T w, int a) {
  return (uint32_t)(w >> (8 * IX * a)) & (IX == 1 ? 0xffu : 0xffffu);
}
/* lane's fine cells from LDS to the mesh, and their sum over the wave in a
   fixed order */
__device__ __forceinline__ double fd_store(const float *acc, int lane, bool live, int64_t X, int64_t Y, int64_t Z, int64_t nf,
                                           float *__restrict__ rho) {
  double t = 0;
  if (live) {
    for (int z = 0; z < 4; ++z)
      for (int y = 0; y < 4; ++y) {
        float4 v;
        v.x = acc[((z * 4 + y) * 4 + 0) * 64 + lane];
        v.y = acc[((z * 4 + y) * 4 + 1) * 64 + lane];
        v.z = acc[((z * 4 + y) * 4 + 2) * 64 + lane];
        v.w = acc[((z * 4 + y) * 4 + 3) * 64 + lane];
        *reinterpret_cast<float4 *>(rho + ((4 * Z + z) * nf + (4 * Y + y)) * nf + 4 * X) = v;
        t += ((double)v.x + (double)v.y) + ((double)v.z + (double)v.w);
      }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
  return t;
}
/* block b of the 4^3-cell blocks: tile T, first coarse cell m0 (0-based, tile frame) */
__device__ __forceinline__ void blk4(int b, const Geo &g, int nbt, int T[3], int m0[3]) {
  const uint32_t ub = (uint32_t)b, un = (uint32_t)nbt, q1 = ub / un, q2 = q1 / un, t = q2 / un;
  const uint32_t tn = (uint32_t)g.nnt, t1 = t / tn;
  T[0] = (int)(t - t1 * tn);
  T[1] = (int)(t1 % tn);
  T[2] = (int)(t1 / tn);
  m0[0] = 4 * (int)(ub - q1 * un);
  m0[1] = 4 * (int)(q1 - q2 * un);
  m0[2] = 4 * (int)(q2 - t * un);
}

template <int IX, bool EX, bool PACK, int NB>
__global__ __launch_bounds__(64) void k_fine_deposit(const typename IntOf<IX>::T *__restrict__ xp,
                                                     const int32_t *__restrict__ rhoc,
                                                     const int64_t *__restrict__ cstart, Geo g, float mass,
                                                     float *__restrict__ rho, double *__restrict__ bsum, int nblk,
                                                     int heavy_at, int32_t *__restrict__ hlist,
                                                     uint64_t *__restrict__ hmask,
                                                     unsigned long long *__restrict__ hcount) {
  typedef typename CdWord<IX>::T W;
  constexpr int PB = 3 * IX, sh = IX == 1 ? 6 : 14;
  __shared__ FdLds<IX, NB> S;
  const int lane = threadIdx.x;
  const char *xb8 = reinterpret_cast<const char *>(xp);
  const int nt = g.nt, nbt = (nt + 3) / 4;
  const int xi = lane & 3, yi = (lane >> 2) & 3, zi = lane >> 4;
  for (int b = blockIdx.x; b < nblk; b += gridDim.x) {
    int T[3], m0[3];
    blk4(b, g, nbt, T, m0);
    wave_lds_sync();
    /* the 5^3 source cells m0-1..m0+3, those past the tile empty */
    if (lane < 15) {
      const int a = lane / 5, sc = (a == 0 ? m0[0] : a == 1 ? m0[1] : m0[2]) - 1 + lane % 5;
      int ta = a == 0 ? T[0] : a == 1 ? T[1] : T[2], l = sc;
      if (sc < 0) {
        l = nt - 1;
        ta = ta > 0 ? ta - 1 : g.nnt - 1;
      }
      const int st = a == 0 ? 1 : a == 1 ? nt : nt * nt, ts = a == 0 ? 1 : a == 1 ? g.nnt : g.nnt * g.nnt;
      S.cax[a][lane % 5] = sc >= nt ? -1 : l * st + nt * nt * nt * ts * ta;
    }
    wave_lds_sync();
    const int i2 = m0[0] == 0 ? 1 : 0; /* at the tile's low edge cell 0 lies in the neighbour tile */
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int q = lane + 64 * u;
      if (q < 125) {
        int cnt = 0;
        const int cx = S.cax[0][q % 5], cy = S.cax[1][(q / 5) % 5], cz = S.cax[2][q / 25];
        if ((cx | cy | cz) >= 0) {
          const int cc = cx + cy + cz;
          cnt = rhoc[cc];
          if (q % 5 < 2) S.start[q / 5][q % 5] = cstart[cc];
        }
        S.pre[q / 5][q % 5 + 1] = cnt;
      }
    }
    wave_lds_sync();
    if (lane < 25) {
      int acc = 0;
      S.pre[lane][0] = 0;
#pragma unroll
      for (int q = 1; q < 6; ++q) {
        acc += S.pre[lane][q];
        S.pre[lane][q] = acc;
      }
    }
    wave_lds_sync();
    const int kz = (m0[2] - 2 + g.ncb + 3) % 3; /* ilayer of plane 0 (k = m0z, 1-based) */
    bool live = m0[0] + xi < nt && m0[1] + yi < nt && m0[2] + zi < nt;
    {
      int tot = 0; /* particles in the lane's 8 source cells */
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = (zi + (j >> 1)) * 5 + yi + (j & 1);
        tot += S.pre[r][xi + 2] - S.pre[r][xi];
      }
      const uint64_t hv = __ballot(live && tot > heavy_at);
      if (lane == 0) {
        hmask[b] = hv;
        if (hv) hlist[atomicAdd(hcount, 1ull)] = b;
      }
      live = live && tot <= heavy_at;
    }
#pragma unroll
    for (int q = 0; q < 16; ++q) reinterpret_cast<float4 *>(S.acc)[q * 64 + lane] = make_float4(0.f, 0.f, 0.f, 0.f);
    float *acc = S.acc + lane;
    /* lane t < 10: row t of the phase of ilayer il, y = t/2, plane p0 + 3*(t&1) */
    struct Phase {
      int nrow, sB, bsc, rb, nb;
      int64_t dA, dB;
      int p0, n; /* PACK: first plane, particles */
    };
    auto phase = [&](int il) -> Phase {
      const int p0 = (il - kz + 3) % 3; /* planes p0 and p0+3 (if below 5) have this ilayer */
      const bool on = lane < 10 && p0 + 3 * (lane & 1) < 5;
      const int rt = on ? (p0 + 3 * (lane & 1)) * 5 + (lane >> 1) : 0;
      Phase h;
      h.nrow = on ? S.pre[rt][5] : 0;
      if constexpr (PACK) {
        const int psc = wave_incl_scan(h.nrow);
        h.p0 = p0;
        h.rb = psc - h.nrow;
        h.n = rl_i(psc, 9);
        h.nb = (h.n + 63) >> 6;
        if (lane < 10) S.rb[il & 1][lane] = h.rb;
        return h;
      }
      h.sB = i2 ? S.pre[rt][1] : 0;
      h.dA = S.start[rt][0];
      h.dB = S.start[rt][1] - S.pre[rt][1];
      const int nbr = (h.nrow + 63) >> 6;
      h.bsc = wave_incl_scan(nbr);
      h.rb = h.bsc - nbr;
      h.nb = rl_i(h.bsc, 63); /* batches of 64 */
      if (lane < 10) S.rb[il & 1][lane] = h.rb;
      return h;
    };
    W raw[NB];
    /* batches q0.. of the phase's rows, in flight */
    auto fetch = [&](const Phase &h, int q0) {
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        raw[q] = 0;
        if (PACK && q0 + q < h.nb) {
          const int i = 64 * (q0 + q) + lane;
          int tr = 0, first = 0; /* its row and that row's first slot */
#pragma unroll
          for (int t = 1; t < 10; ++t) {
            const int f = rl_i(h.rb, t);
            if (f <= i) {
              tr = t;
              first = f;
            }
          }
          const int l = i - first, r = (h.p0 + 3 * (tr & 1)) * 5 + (tr >> 1);
          if (i < h.n) {
            int64_t p = S.start[r][0];
            if (i2) {
              const int sB = S.pre[r][1];
              if (l >= sB) p = S.start[r][1] - sB;
            }
            raw[q] = cd_load<IX>(xb8 + (p + l) * PB);
          }
        } else if (!PACK && q0 + q < h.nb) {
          const int tr = __popcll(__ballot(lane < 10 && h.bsc <= q0 + q)); /* its row */
          const int l = 64 * (q0 + q - rl_i(h.rb, tr)) + lane, n = rl_i(h.nrow, tr);
          int64_t p = rl_i64(h.dA, tr);
          if (i2) {
            const int64_t pb = rl_i64(h.dB, tr);
            if (l >= rl_i(h.sB, tr)) p = pb;
          }
          if (l < n) raw[q] = cd_load<IX>(xb8 + (p + l) * PB);
        }
      }
    };
    int il = 0, q0 = 0;
    Phase h = phase(0);
    fetch(h, 0);
#pragma unroll 1
    while (il < 3) {
      wave_lds_sync(); /* the reads of word and top are done */
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        if (q0 + q < h.nb) {
          const uint64_t t0 = __ballot((fd_code<IX>(raw[q], 0) >> sh) == 3u), t1 = __ballot((fd_code<IX>(raw[q], 1) >> sh) == 3u),
                         t2 = __ballot((fd_code<IX>(raw[q], 2) >> sh) == 3u);
          S.word[q * 64 + lane] = raw[q];
          if (lane < 3) S.top[q][lane] = lane == 0 ? t0 : (lane == 1 ? t1 : t2);
        }
      }
      wave_lds_sync();
      /* the next batches, or the next phase's first, fly during the sums */
      const int ci = il, c0 = q0;
      q0 += NB;
      if (q0 >= h.nb) {
        q0 = 0;
        if (++il < 3) h = phase(il);
      }
      if (il < 3) fetch(h, q0);
      const int p0 = (ci - kz + 3) % 3;
      /* this lane's plane: the one of zi (the cells below it), zi+1 (its own) that is p0 mod 3, or none */
      const int pl = zi % 3 == p0 ? zi : ((zi + 1) % 3 == p0 ? zi + 1 : -1);
      const bool zbelow = pl == zi;
      if (pl >= 0 && live) {
#pragma unroll 1
        for (int j = 0; j < 2; ++j) { /* rows y-1, y */
          const int r = pl * 5 + yi + j, r0 = S.rb[ci & 1][2 * (yi + j) + (pl >= 3 ? 1 : 0)];
          const int rb = (PACK ? 0 : r0) - c0, s0 = PACK ? r0 : 0; /* slots, counted from batch -rb's */
          const int pA = s0 + S.pre[r][xi], pB = s0 + S.pre[r][xi + 1], pC = s0 + S.pre[r][xi + 2];
          for (int bb = max(pA >> 6, -rb); bb * 64 < pC && rb + bb < NB; ++bb) {
            const int q = rb + bb, o = 64 * bb;
            const uint64_t fB = bits_below(pB - o);
            uint64_t m = bits_below(pC - o) & ~bits_below(pA - o) & (S.top[q][0] | ~fB);
            if (j == 0) m &= S.top[q][1];
            if (zbelow) m &= S.top[q][2];
            const W *wd = S.word + q * 64;
            if (!m) continue;
            int i = __builtin_ctzll(m);
            W wn = wd[i];
            while (m) {
              const W w = wn;
              const bool xbelow = o + i < pB;
              m &= m - 1ull;
              i = m ? __builtin_ctzll(m) : 0;
              wn = wd[i]; /* the next hit's codes are on their way */
              int bx, by, bz;
              float wx[2], wy[2], wz[2];
              fd_axis<IX, EX>(fd_code<IX>(w, 0), xbelow, m0[0] + xi + (xbelow ? 0 : 1), m0[0] + xi + 1, bx, wx[0], wx[1]);
              fd_axis<IX, EX>(fd_code<IX>(w, 1), j == 0, m0[1] + yi + j, m0[1] + yi + 1, by, wy[0], wy[1]);
              fd_axis<IX, EX>(fd_code<IX>(w, 2), zbelow, m0[2] + pl, m0[2] + zi + 1, bz, wz[0], wz[1]);
              float *a0 = acc + 64 * ((bz * 4 + by) * 4 + bx);
              float v[8];
#pragma unroll
              for (int k = 0; k < 8; ++k) v[k] = a0[64 * ((k >> 2) * 16 + ((k >> 1) & 1) * 4 + (k & 1))];
#pragma unroll
              for (int k = 0; k < 8; ++k) v[k] = v[k] + wx[k & 1] * wy[(k >> 1) & 1] * wz[k >> 2] * mass;
#pragma unroll
              for (int k = 0; k < 8; ++k) a0[64 * ((k >> 2) * 16 + ((k >> 1) & 1) * 4 + (k & 1))] = v[k];
            }
          }
        }
      }
    }
    const double t = fd_store(S.acc, lane, live, T[0] * nt + m0[0] + xi, T[1] * nt + m0[1] + yi, T[2] * nt + m0[2] + zi,
                              4 * g.nc, rho);
    if (lane == 0) bsum[b] = t;
  }
}

/*
 * The crowded cells of the listed blocks, FDH_W waves a block, each a workgroup
 * of its own that fits in beside whatever else runs: a wave takes one of its
 * cells at a time, lane f owning fine cell f = (z*4+y)*4+x, and
 * goes through the cell's 4 source rows (two cells of a row follow one another
 * in order) 64 particles at a time.  Ballots over the particles' sub-cells on
 * each axis give every lane the mask of the particles that reach its fine
 * cell, and it adds those alone, in order, four weight reads in flight.
 */
template <int IX, bool EX>
__global__ __launch_bounds__(64) void k_fine_deposit_heavy(const typename IntOf<IX>::T *__restrict__ xp,
                                                                   const int32_t *__restrict__ rhoc,
                                                                   const int64_t *__restrict__ cstart, Geo g, float mass,
                                                                   float *__restrict__ rho, double *__restrict__ hsum,
                                                                   const int32_t *__restrict__ hlist,
                                                                   const uint64_t *__restrict__ hmask,
                                                                   const unsigned long long *__restrict__ hcount) {
  typedef typename CdWord<IX>::T W;
  constexpr int PB = 3 * IX, sh = IX == 1 ? 6 : 14;
  __shared__ float wts[3][64]; /* d1 of the 64 particles at hand, per axis */
  const int lane = threadIdx.x;
  const char *xb8 = reinterpret_cast<const char *>(xp);
  const int nt = g.nt, nbt = (nt + 3) / 4;
  const int64_t nf = 4 * (int64_t)g.nc;
  const int fx = lane & 3, fy = (lane >> 2) & 3, fz = lane >> 4;
  const int64_t items = (int64_t)*hcount * FDH_W;
  for (int64_t h = blockIdx.x; h < items; h += gridDim.x) {
    const int b = hlist[h / FDH_W], wv = (int)(h % FDH_W);
    double hs = 0;
    const uint64_t cells = hmask[b];
    int T[3], m0[3];
    blk4(b, g, nbt, T, m0);
    int nth = 0;
    for (uint64_t rest = cells; rest; rest &= rest - 1ull, ++nth) {
      if (nth % FDH_W != wv) continue;
      const int L = __builtin_ctzll(rest);
      const int C[3] = {m0[0] + (L & 3), m0[1] + ((L >> 2) & 3), m0[2] + (L >> 4)}; /* 0-based */
      float sacc = 0.f;
      /* the source rows in order: the two z planes by ilayer, y-1 then y */
      const int ka = (C[2] - 2 + g.ncb + 3) % 3; /* ilayer of plane C-1 (k = C, 1-based) */
      /* lane 2r+i < 8: source cell i (x-1, x) of row r */
      int n8 = 0;
      int64_t s8 = 0;
      if (lane < 8) {
        const int i = lane & 1, y = (lane >> 1) & 1, zz = lane >> 2;
        const int oz = ka == 2 ? 1 - zz : zz; /* (2, 0): the upper plane first */
        const int64_t cc = cid_global(g, T[0] * nt + C[0] - 1 + i, T[1] * nt + C[1] - 1 + y, T[2] * nt + C[2] - 1 + oz);
        n8 = rhoc[cc];
        s8 = cstart[cc];
      }
#pragma unroll 1
      for (int r = 0; r < 4; ++r) {
        const int y = r & 1, oz = ka == 2 ? 1 - (r >> 1) : r >> 1;
        const int n0 = rl_i(n8, 2 * r), nn = n0 + rl_i(n8, 2 * r + 1);
        const int64_t s0 = rl_i64(s8, 2 * r), s1 = rl_i64(s8, 2 * r + 1) - n0;
        W next = 0;
        if (lane < nn) next = cd_load<IX>(xb8 + ((lane < n0 ? s0 : s1) + lane) * PB);
        for (int o = 0; o < nn; o += 64) {
          const W w = next;
          const int l = o + lane;
          if (l + 64 < nn) next = cd_load<IX>(xb8 + ((l + 64 < n0 ? s0 : s1) + l + 64) * PB);
          const bool xbelow = l < n0;
          const uint32_t u[3] = {fd_code<IX>(w, 0), fd_code<IX>(w, 1), fd_code<IX>(w, 2)};
          const bool below[3] = {xbelow, y == 0, oz == 0};
          bool pass = l < nn;
          int rr[3]; /* plane of corner 1 in the cell's frame, -1..4 */
          float d1[3];
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            pass = pass && (!below[a] || (u[a] >> sh) == 3u);
            if constexpr (EX) {
              constexpr float s = 1.0f / (float)(1 << sh);
              d1[a] = fmaf((float)(u[a] & ((1u << sh) - 1u)), -s, 1.0f - 0.5f * s);
              rr[a] = below[a] ? -1 : (int)(u[a] >> sh);
            } else {
              const int ci = C[a] + (below[a] ? 0 : 1);
              const float tempx = (float)(4 * (ci - 1)) + ((float)u[a] + 0.5f) * (IX == 1 ? 0x1p-6f : 0x1p-14f);
              const int i1 = (int)floorf(tempx) + 1;
              d1[a] = (float)i1 - tempx;
              rr[a] = i1 - 4 * C[a] - 1;
            }
          }
          wave_lds_sync(); /* the last batch's weights are read */
#pragma unroll
          for (int a = 0; a < 3; ++a) wts[a][lane] = d1[a];
          wave_lds_sync();
          /* particles whose corner 1 is this lane's plane (at), or the one below it (lo) */
          uint64_t at[3], lo[3];
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            const int f = a == 0 ? fx : (a == 1 ? fy : fz);
            uint64_t k[5];
#pragma unroll
            for (int q = 0; q < 5; ++q) k[q] = __ballot(rr[a] == q - 1);
            at[a] = f == 0 ? k[1] : (f == 1 ? k[2] : (f == 2 ? k[3] : k[4]));
            lo[a] = f == 0 ? k[0] : (f == 1 ? k[1] : (f == 2 ? k[2] : k[3]));
          }
          uint64_t m = __ballot(pass) & (at[0] | lo[0]) & (at[1] | lo[1]) & (at[2] | lo[2]);
          while (m) {
            float e[4][3];
            uint64_t bit[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const int i = m ? __builtin_ctzll(m) : 0;
              bit[k] = m & (0ull - m); /* 0: no particle left */
              m &= ~bit[k];
#pragma unroll
              for (int a = 0; a < 3; ++a) e[k][a] = wts[a][i];
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const float wx = at[0] & bit[k] ? e[k][0] : 1.0f - e[k][0], wy = at[1] & bit[k] ? e[k][1] : 1.0f - e[k][1],
                          wz = at[2] & bit[k] ? e[k][2] : 1.0f - e[k][2];
              const float s = sacc + wx * wy * wz * mass;
              sacc = bit[k] ? s : sacc;
            }
          }
        }
      }
      rho[((4 * (int64_t)(T[2] * nt + C[2]) + fz) * nf + 4 * (T[1] * nt + C[1]) + fy) * nf + 4 * (T[0] * nt + C[0]) + fx] = sacc;
      double t = (double)sacc;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
      hs += t;
    }
    if (lane == 0) hsum[(int64_t)b * FDH_W + wv] = hs; /* read if it had a cell */
  }
}
/* sum of the blocks' sums, those of their crowded cells among them, in a fixed
   order: a workgroup sums its stretch of blocks, the last to finish the
   workgroups' sums.  The list goes back to empty */
#define FDS_B 1024 /* blocks a workgroup takes before there is a second */
__global__ __launch_bounds__(256) void k_sum_blocks(const double *__restrict__ bsum, const uint64_t *__restrict__ hmask,
                                                    const double *__restrict__ hsum, int nb, int per,
                                                    double *__restrict__ part, double *__restrict__ out,
                                                    unsigned long long *__restrict__ hcount) {
  __shared__ double r[256];
  __shared__ bool last;
  const int t = threadIdx.x;
  const int64_t b0 = (int64_t)blockIdx.x * per, b1 = min(b0 + per, (int64_t)nb);
  double s = 0;
#pragma unroll 4
  for (int64_t b = b0 + t; b < b1; b += 256) {
    s += bsum[b];
    const int n = min(__popcll(hmask[b]), FDH_W);
    for (int k = 0; k < n; ++k) s += hsum[b * FDH_W + k];
  }
  r[t] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (t < o) r[t] += r[t + o];
    __syncthreads();
  }
  if (t == 0) {
    __hip_atomic_store(part + blockIdx.x, r[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last = __hip_atomic_fetch_add(hcount + 1, 1ull, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
  }
  __syncthreads();
  if (!last || t >= 64) return;
  s = t < (int)gridDim.x ? __hip_atomic_load(part + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if (t == 0) {
    *out = s;
    hcount[0] = 0ull;
    hcount[1] = 0ull;
  }
}

#define DEP_BLOCKS 2048
#define FD_GRID 16384
template <int IX, bool EX> static int fine_dep(cube_ctx *c, float mass, double *t) {
  /* a coarse cell whose 8 source cells hold more particles than this is formed
     by a wave of its own (CUBE_FD_HEAVY): a lane's hit costs its wave some 60
     instructions, a wave's pass over 64 candidates about 150 and the cell's 4
     rows as many each.  96 / 160 / 256 measured 2.02 / 1.36 / 1.16 ms on 128^3
     at z = 3, 0.120 / 0.105 / 0.099 ms on 48^3, 0.76 / 0.81 / 0.83 ms on the
     clustered 128^3 with 1-byte codes */
  int heavy_at = 256;
  if (const char *e = getenv("CUBE_FD_HEAVY"); e && *e) heavy_at = std::max(0, atoi(e));
  const int64_t nbt = (c->nt + 3) / 4, nblk = nbt * nbt * nbt * c->ntiles;
  const typename IntOf<IX>::T *xp = (const typename IntOf<IX>::T *)c->xp;
  unsigned long long *hcount = (unsigned long long *)c->ured + CUBE_URED_FDHEAVY;
  const int st = cube_words_open(c, CUBE_OPEN_FDLIST, hcount, 2);
  if (st) return st;
  /* by the mean density: a phase's 50 source cells in two batches, its rows of 5
     in one each, or more than that (see k_fine_deposit) */
  auto kern = 50 * c->nplocal <= 128 * c->ncells  ? k_fine_deposit<IX, EX, true, 4>
              : 5 * c->nplocal <= 64 * c->ncells ? k_fine_deposit<IX, EX, false, 10>
                                                 : k_fine_deposit<IX, EX, true, 24>;
  hipLaunchKernelGGL(kern, dim3((unsigned)std::min<int64_t>(nblk, FD_GRID)), dim3(64), 0, c->stream, xp, c->rhoc, c->cstart,
                     geo_of(c), mass, c->rho_f, c->fdsum, (int)nblk, heavy_at, c->fdlist, c->fdmask, hcount);
  CUBE_LAUNCH_CHECK();
  /* a fixed grid, four waves a SIMD: the count stays on the device */
  hipLaunchKernelGGL((k_fine_deposit_heavy<IX, EX>), dim3((unsigned)std::min<int64_t>(nblk * FDH_W, 4096)), dim3(64), 0,
                     c->stream, xp, c->rhoc, c->cstart, geo_of(c), mass, c->rho_f, c->fdheavy, c->fdlist, c->fdmask, hcount);
  CUBE_LAUNCH_CHECK();
  const int nw = (int)std::min<int64_t>(FDS_W, (nblk + FDS_B - 1) / FDS_B), per = (int)((nblk + nw - 1) / nw);
  hipLaunchKernelGGL(k_sum_blocks, dim3(nw), dim3(256), 0, c->stream, c->fdsum, c->fdmask, c->fdheavy, (int)nblk, per,
                     c->fdsum + nblk, c->dred + CUBE_DRED_FINE_SUM, hcount);
  CUBE_LAUNCH_CHECK();
  cube_words_close(c, CUBE_OPEN_FDLIST);
  if (t) {
    CUBE_CHECK(hipMemcpyAsync(t, c->dred + CUBE_DRED_FINE_SUM, sizeof(double), hipMemcpyDeviceToHost, c->stream));
    CUBE_CHECK(hipStreamSynchronize(c->stream));
  }
  return CUBE_OK;
}
int cube_fine_deposit(cube_ctx *c, float mass_p, double *testrhof) {
  if (c->p.izipx == 1) return fine_dep<1, true>(c, mass_p, testrhof);
  /* 2-byte codes: 4*(i-1) + (u+0.5)*2^-14 needs 15 fraction bits, exact in
     real(4) below 512, and the coordinate reaches 4 nt */
  return c->nt <= 128 ? fine_dep<2, true>(c, mass_p, testrhof) : fine_dep<2, false>(c, mass_p, testrhof);
}
template <int IX, bool EX> static int coarse_dep(cube_ctx *c, float mass, double *t) {
  /* partial sums in the upper half of dred, apart from the fine deposit's,
     so that the two deposits may run at the same time */
  double *part = c->dred + 4096;
  /* particles of a phase's 72 source cells above which it adds 64 particles'
     terms at a time (CUBE_CD_HEAVY); the staged batches hold no more */
  int heavy_at = 64 * CdWord<IX>::NB;
  if (const char *e = getenv("CUBE_CD_HEAVY"); e && *e) heavy_at = std::max(0, atoi(e));
  const int64_t nbt = (c->nt + 3) / 4, nblk = nbt * nbt * nbt * c->ntiles;
  /* small meshes: one wave per workgroup, so that few blocks spread over many
     CUs (with more than DEP_BLOCKS every CU has its waves either way, and
     there are no more partial sums than that); else four */
  const bool small = nblk <= DEP_BLOCKS;
  const int64_t want = small ? nblk : (nblk + 3) / 4;
  const unsigned grid = (unsigned)std::min<int64_t>(want, DEP_BLOCKS);
  const typename IntOf<IX>::T *xp = (const typename IntOf<IX>::T *)c->xp;
  /* few particles: the 72 source cells of an average phase fit CD_PACK.  With 8
     a cell a phase never does, and the other variant's slots need no offset (1
     to 2 % of the kernel) */
  const bool pack = 72 * c->nplocal <= CD_PACK * c->ncells;
  auto kern = small ? (pack ? k_coarse_deposit<IX, EX, 1, true> : k_coarse_deposit<IX, EX, 1, false>)
                    : (pack ? k_coarse_deposit<IX, EX, 4, true> : k_coarse_deposit<IX, EX, 4, false>);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(small ? 64 : 256), 0, c->stream, xp, c->rhoc, c->cstart, geo_of(c), mass,
                     c->rho_c, part, (int)nblk, heavy_at);
  CUBE_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_sum_parts1, dim3(1), dim3(64), 0, c->stream, part, (int)grid, c->dred + CUBE_DRED_COARSE_SUM);
  CUBE_LAUNCH_CHECK();
  if (t) {
    CUBE_CHECK(hipMemcpyAsync(t, c->dred + CUBE_DRED_COARSE_SUM, sizeof(double), hipMemcpyDeviceToHost, c->stream));
    CUBE_CHECK(hipStreamSynchronize(c->stream));
  }
  return CUBE_OK;
}
int cube_coarse_deposit(cube_ctx *c, float mass_p, double *testrhoc) {
  if (c->p.izipx == 1) return coarse_dep<1, true>(c, mass_p, testrhoc);
  /* 2-byte codes: c + (u+0.5)/65536 - 0.5 needs 17 fraction bits, exact in
     real(4) below 128, and a source cell's c reaches nt */
  return c->nt < 128 ? coarse_dep<2, true>(c, mass_p, testrhoc) : coarse_dep<2, false>(c, mass_p, testrhoc);
}

/* ---------------- kicks ---------------- */
#define KT 256
struct F3 {
  float x, y, z;
};

/* G = (((F*a_mid)*dt)/6)/pi per mesh value, the factor of every kick term
   (W/pm.f90:341-348); the coarse kick reads G so each coarse cell's value is
   formed once instead of by every particle whose cloud touches it */
__device__ __forceinline__ void kick_prescale(const float *__restrict__ F, int64_t n, float a_mid, float dt,
                                              float *__restrict__ G) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x) {
    const float a = (F[q] * a_mid) * dt;
    bool ok = true;
    const float v = div_6pi(a, ok);
    G[q] = ok ? v : (a / 6.0f) / CUBE_PI_F;
  }
}
__global__ void k_kick_prescale(const float *__restrict__ F, int64_t n, float a_mid, float dt, float *__restrict__ G) {
  kick_prescale(F, n, a_mid, dt, G);
}
/* all that the one-pass kicks read besides the state and the fine mesh, in one
   launch: G and both decode tables */
__global__ __launch_bounds__(256) void k_kick_prep(const float *__restrict__ F, int64_t n, float a_mid, float dt,
                                                   float *__restrict__ G, const float *__restrict__ tanf_tab, int nv,
                                                   double vc0, double vc1, double *__restrict__ vdec0,
                                                   double *__restrict__ vdec1) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nv; i += gridDim.x * blockDim.x) {
    vdec0[i] = (double)tanf_tab[i] / vc0; /* as k_vdec */
    vdec1[i] = (double)tanf_tab[i] / vc1;
  }
  kick_prescale(F, n, a_mid, dt, G);
}
/* a step's scalars to the host: vmax folded from its slots (left cleared), the
   mesh sums and max |F|^2 of both meshes */
__global__ __launch_bounds__(CUBE_SLOTS) void k_pm_result(unsigned long long *__restrict__ vsl, const double *__restrict__ dred,
                                                          const uint64_t *__restrict__ ured,
                                                          unsigned long long *__restrict__ hres) {
  __shared__ unsigned long long r[CUBE_SLOTS];
  const int t = threadIdx.x, reg = blockIdx.x;
  r[t] = vsl[reg * CUBE_SLOTS + t];
  vsl[reg * CUBE_SLOTS + t] = 0ull;
  __syncthreads();
  for (int o = CUBE_SLOTS / 2; o > 0; o >>= 1) {
    if (t < o) r[t] = r[t] > r[t + o] ? r[t] : r[t + o];
    __syncthreads();
  }
  if (t == 0) hres[HR_VMAX + reg] = r[0];
  if (reg == 0 && t == 1) hres[HR_SUM] = (unsigned long long)__double_as_longlong(dred[CUBE_DRED_FINE_SUM]);
  if (reg == 0 && t == 2) hres[HR_SUM + 1] = (unsigned long long)__double_as_longlong(dred[CUBE_DRED_COARSE_SUM]);
  if (reg == 0 && t == 3) hres[HR_F2] = ured[0]; /* two floats */
}

/* One kick of one particle: vreal[a] += the CIC gather of the mesh over
   the 8 corners in the order of W/pm.f90:146-153 (fine: force_f with
   ((((F*a_mid)*dt)/6)/pi)*wx*wy*wz per term; coarse: the prescaled G with
   G*wx*wy*wz, W/pm.f90:341-348).  loc: 1-based cell in the tile, tt: tile. */
template <int IX, bool FINE, bool PRE = false>
__device__ __forceinline__ void kick_particle(const int32_t code[3], const int loc[3], const int tt[3],
                                              const Geo &g, const float *__restrict__ force, float a_mid,
                                              float dt, double vreal[3]) {
  /* PRE: the fine mesh already holds (((F*a_mid)*dt)/6)/pi per value */
  constexpr bool DIV = FINE && !PRE;
  const int nt = g.nt, nfine = 4 * g.nc, nft = 4 * nt;
  int i1[3];
  float d1[3], d2[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    float tempx;
    if (FINE) /* ncell*((/i,j,k/)-1)+ncell*(...)*x_resolution, tile frame (W/pm.f90:138):
                 both terms are exact floats, so one float add rounds it */
      tempx = (float)(4 * (loc[a] - 1)) + ((float)cube_ucode(IX, code[a]) + 0.5f) * (IX == 1 ? 0x1p-6f : 0x1p-14f);
    else /* ((/itx,../)-1)*nt+((/i,../)-1)+(...)*x_resolution-0.5 (W/pm.f90:335) */
      tempx = coarse_tempx<IX>(tt[a] * nt + (loc[a] - 1), code[a]);
    i1[a] = (int)floorf(tempx) + 1;
    d1[a] = (float)i1[a] - tempx;
    d2[a] = 1.0f - d1[a];
  }
  /* 0-based periodic mesh coordinates of the two CIC planes per axis.
     tempx lies in (4(loc-1), 4 loc] (fine) or (g-1/2, g+1/2] around the
     global cell g (coarse), so the first plane is in [0, nfine] or
     [-1, nc-1] and one compare wraps each plane (no integer modulo) */
  const int n = FINE ? nfine : g.nc;
  int m1[3], m2[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int v = FINE ? tt[a] * nft + i1[a] - 1 : i1[a] - 1;
    m1[a] = v < 0 ? v + n : (v >= n ? v - n : v);
    m2[a] = v + 1 >= n ? v + 1 - n : v + 1;
  }
  /* corner order of W/pm.f90:146-153 */
  const int cx[8] = {0, 1, 0, 0, 0, 1, 1, 1}, cy[8] = {0, 0, 1, 0, 1, 0, 1, 1}, cz[8] = {0, 0, 0, 1, 1, 1, 0, 1};
  const double v0[3] = {vreal[0], vreal[1], vreal[2]};
  bool ok = true;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int X = cx[q] ? m2[0] : m1[0], Y = cy[q] ? m2[1] : m1[1], Z = cz[q] ? m2[2] : m1[2];
    const float wx = cx[q] ? d2[0] : d1[0], wy = cy[q] ? d2[1] : d1[1], wz = cz[q] ? d2[2] : d1[2];
    /* the corner's three components in one 12-byte load */
    const F3 Fv = *reinterpret_cast<const F3 *>(force + 3 * (((int64_t)Z * n + Y) * n + X));
    const float F[3] = {Fv.x, Fv.y, Fv.z};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const float gq = DIV ? div_6pi((F[a] * a_mid) * dt, ok) : F[a];
      const float inc = ((gq * wx) * wy) * wz;
      vreal[a] = vreal[a] + (double)inc;
    }
  }
  if (DIV && !ok) { /* a quotient outside the checked range: redo with divisions */
#pragma unroll
    for (int a = 0; a < 3; ++a) vreal[a] = v0[a];
    for (int q = 0; q < 8; ++q) {
      const int X = cx[q] ? m2[0] : m1[0], Y = cy[q] ? m2[1] : m1[1], Z = cz[q] ? m2[2] : m1[2];
      const float wx = cx[q] ? d2[0] : d1[0], wy = cy[q] ? d2[1] : d1[1], wz = cz[q] ? d2[2] : d1[2];
      const float *F = force + 3 * (((int64_t)Z * n + Y) * n + X);
      for (int a = 0; a < 3; ++a) {
        const float inc = ((((((F[a] * a_mid) * dt) / 6.0f) / CUBE_PI_F) * wx) * wy) * wz;
        vreal[a] = vreal[a] + (double)inc;
      }
    }
  }
}

/* max of |v + v_c| over the workgroup: wave shuffles, then the waves
   through LDS, one atomic per component into its slot region of
   vmax_bits (W/pm.f90:349) */
template <int THREADS> __device__ __forceinline__ void vmax_reduce(double vm[3], unsigned long long *__restrict__ vmax_bits) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
#pragma unroll
    for (int a = 0; a < 3; ++a) vm[a] = fmax(vm[a], __shfl_xor(vm[a], o, 64));
  __shared__ double red[3][THREADS / 64];
  if ((threadIdx.x & 63) == 0)
    for (int a = 0; a < 3; ++a) red[a][threadIdx.x >> 6] = vm[a];
  __syncthreads();
  if (threadIdx.x < 3) {
    double m = red[threadIdx.x][0];
    for (int w = 1; w < THREADS / 64; ++w) m = fmax(m, red[threadIdx.x][w]);
    atomicMax(cube_slot(vmax_bits + threadIdx.x * CUBE_SLOTS), (unsigned long long)__double_as_longlong(m));
  }
}

/* kicks, one workgroup per cell row (tile, k, j): particles of the row are
   contiguous; each thread finds its cell by binary search in LDS.  The one
   kick of FINE (decode with vdec, encode with venc), for callers that take
   the stages one by one; or (BOTH) a step's two in one pass, as k_kicks below
   but gathering from the meshes where they lie: for boxes of few particles, see
   kicks_impl. */
#define KICK_ROW 2048 /* particles of a row whose cells the kick tables in LDS (else a binary search) */
template <int IX, int IV, bool FINE, bool BOTH>
__global__ __launch_bounds__(KT) void k_kick(const typename IntOf<IX>::T *__restrict__ xp,
                                             typename IntOf<IV>::T *__restrict__ vp,
                                             const int64_t *__restrict__ cstart, const float *__restrict__ vfield,
                                             const float *__restrict__ force, const double *__restrict__ vdec,
                                             Geo g, int nvh, float a_mid, float dt, double venc,
                                             unsigned long long *__restrict__ vmax_bits,
                                             const float *__restrict__ force2, const double *__restrict__ vdec2) {
  const int nt = g.nt;
  const int64_t row = blockIdx.x;
  const int j = (int)(row % nt), k = (int)((row / nt) % nt), t = (int)(row / ((int64_t)nt * nt));
  const int tz = t / (g.nnt * g.nnt), ty = (t / g.nnt) % g.nnt, tx = t % g.nnt;
  __shared__ int64_t cs[520];
  __shared__ uint16_t lcell[KICK_ROW]; /* slot -> cell of the row, when it fits */
  const int64_t c0 = row * nt;
  for (int i = threadIdx.x; i <= nt; i += KT) cs[i] = cstart[c0 + i];
  __syncthreads();
  const bool tab = cs[nt] - cs[0] <= KICK_ROW; /* uniform */
  if (tab) {
    for (int i = threadIdx.x; i < nt; i += KT)
      for (int64_t q = cs[i]; q < cs[i + 1]; ++q) lcell[q - cs[0]] = (uint16_t)i;
    __syncthreads();
  }
  constexpr bool VMAX = !FINE || BOTH; /* the coarse kick reports vmax */
  double vm[3] = {0, 0, 0};
  for (int64_t p = cs[0] + threadIdx.x; p < cs[nt]; p += KT) {
    int lo = 0, hi = nt;
    if (tab) {
      lo = lcell[p - cs[0]];
    } else {
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (cs[mid] <= p) lo = mid; else hi = mid;
      }
    }
    const int loc[3] = {lo + 1, j + 1, k + 1};
    const int tt[3] = {tx, ty, tz};
    int32_t code[3];
    double vreal[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      code[a] = (int32_t)xp[3 * p + a];
      vreal[a] = vdec[(int32_t)vp[3 * p + a] + nvh];
    }
    kick_particle<IX, FINE, BOTH>(code, loc, tt, g, force, a_mid, dt, vreal);
    if (BOTH) { /* the code the fine kick would store, decoded again for the coarse kick */
      int32_t v1[3];
      cube_encode_v3(IV, venc, vreal, v1);
#pragma unroll
      for (int a = 0; a < 3; ++a) vreal[a] = vdec2[v1[a] + nvh];
      kick_particle<IX, false>(code, loc, tt, g, force2, a_mid, dt, vreal);
    }
    F3 vc = {0.f, 0.f, 0.f};
    if (VMAX) vc = *reinterpret_cast<const F3 *>(vfield + 3 * (c0 + lo)); /* one 12-byte load */
    const float vcf[3] = {vc.x, vc.y, vc.z};
    int32_t vcode[3];
    cube_encode_v3(IV, venc, vreal, vcode);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      if (VMAX) {
        const double av = fabs(vreal[a] + (double)vcf[a]);
        vm[a] = av > vm[a] ? av : vm[a];
      }
      vp[3 * p + a] = (typename IntOf<IV>::T)vcode[a];
    }
  }
  if (VMAX) vmax_reduce<KT>(vm, vmax_bits);
}

/*
 * The step's two kicks in one pass, W/pm.f90:129-159 then 322-354: the fine one
 * (decode with vdec) from the prescaled mesh that the step's force pipeline
 * leaves in force_f, then the coarse one on the code the fine one would store
 * (decoded again with vdec2), the intermediate codes in registers instead of
 * going through vp.
 *
 * One workgroup per block of 4x2x2 coarse cells of a tile.  Gathering 16
 * corners per particle from global memory, the mesh of a row of cells never in
 * L1 for long, was bound by those gathers.  Here the block's mesh values
 * (planes 0..16, 0..8, 0..8 of its 16x8x8 fine cells, and its coarse cells with
 * a ring) go to LDS in rows of 16-byte loads, and the gathers are LDS reads.
 * The first particles' words fly with them.  8 workgroups a CU hide one
 * another's loads; what bounds it now is VALU issue (some 840 instructions per
 * wave, at 4 ms of 7.4).  8x2x2 and 4x4x2 cells (4 workgroups a CU) took 8.7
 * and 7.7 ms, several blocks per workgroup 7.6 (99 registers).  With a
 * workgroup per row of cells, before -> after: 8.1 -> 7.4 ms on the 1024^3
 * fine mesh with 512^3 particles (13 GB of mesh), 1.29 -> 1.00 ms on
 * 512^3 with 256^3, 157 -> 141 us on 256^3 and 201 -> 148 us on its clustered
 * z = 0 state, 74 -> 51 us on 192^3; 8.9 -> 9.7 us on 64^3.
 */
#define KB 192 /* 16 cells at the usual 8 particles, and half as many again; 12 rows of 16 lanes load a plane */
template <int IX, int IV, bool EX>
__global__ __launch_bounds__(KB) void k_kicks(const typename IntOf<IX>::T *__restrict__ xp,
                                              typename IntOf<IV>::T *__restrict__ vp, const int64_t *__restrict__ cstart,
                                              const float *__restrict__ vfield, const float *__restrict__ force,
                                              const double *__restrict__ vdec, Geo g, int nvh, double venc,
                                              unsigned long long *__restrict__ vmax_bits,
                                              const float *__restrict__ force2, const double *__restrict__ vdec2) {
  /* EX: the real(4) coordinate is exact, so a particle's second plane is at
     most the first one past its cell; else it can round up to the one after.
     A row is CH chunks of 16 bytes, loaded by 16 lanes */
  constexpr int PL = EX ? 9 : 10, CH = EX ? 13 : 14, RF = 4 * CH;
  __shared__ float4 fm[PL * PL * CH];
  __shared__ float cm[4 * 4 * 18];
  __shared__ int64_t cs[4][5];
  __shared__ int pre[5];
  const int nt = g.nt, tid = threadIdx.x;
  /* consecutive blocks on one XCD, whose L2 then holds the planes they share */
  const unsigned nq = gridDim.x >> 3, nr = gridDim.x & 7, xcd = blockIdx.x & 7;
  const unsigned b = xcd * nq + min(xcd, nr) + (blockIdx.x >> 3);
  const unsigned nbx = (nt + 3) / 4, nby = (nt + 1) / 2, nbz = (nt + 1) / 2, q1 = b / nbx, q2 = q1 / nby, t = q2 / nbz;
  const int x0 = 4 * (int)(b - q1 * nbx), y0 = 2 * (int)(q1 - q2 * nby), z0 = 2 * (int)(q2 - t * nbz);
  const unsigned t1 = t / (unsigned)g.nnt;
  const int gx = (int)(t - t1 * g.nnt) * nt + x0, gy = (int)(t1 % (unsigned)g.nnt) * nt + y0,
            gz = (int)(t1 / (unsigned)g.nnt) * nt + z0; /* the block's first cell in the box */
  const int nf = 4 * g.nc, rowb = 12 * nf;
  if (tid < 64) { /* starts of the 4 rows' cells; those past the tile are empty */
    const int r = tid / 5, y = y0 + (r & 1), z = z0 + (r >> 1);
    int64_t v = 0;
    if (tid < 20) {
      const bool in = y < nt && z < nt;
      v = cstart[g.cid(0, in ? y : 0, in ? z : 0, (int)t) + (in ? min(x0 + tid % 5, nt) : 0)];
      cs[r][tid % 5] = v;
    }
    const int lo = 5 * min(tid, 3);
    const int n = (int)(__shfl(v, lo + 4, 64) - __shfl(v, lo, 64)); /* by the whole wave */
    const int sc = wave_incl_scan(tid < 4 ? n : 0);
    if (tid < 4) pre[tid + 1] = sc;
    if (tid == 63) pre[0] = 0;
  }
  __syncthreads();
  /* the mesh and the first particles fly together.  This lane's chunk of a
     plane; its row's bytes are a multiple of 48, so no chunk straddles its end */
  const int ry = tid >> 4, rc = tid & 15;
  const bool on = rc < CH && ry < PL;
  float4 raw[PL];
  {
    int x = 48 * gx + 16 * rc, y = 4 * gy + ry;
    while (x >= rowb) x -= rowb;
    while (y >= nf) y -= nf;
    const uint32_t off = (uint32_t)y * (uint32_t)rowb + (uint32_t)x; /* a plane is below 2^32 bytes */
#pragma unroll
    for (int z = 0; z < PL; ++z) raw[z] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (on)
#pragma unroll
      for (int z = 0; z < PL; ++z) {
        const int zz = 4 * gz + z;
        const char *plane = reinterpret_cast<const char *>(force) + (int64_t)(zz < nf ? zz : zz - nf) * nf * rowb;
        raw[z] = *reinterpret_cast<const float4 *>(plane + off);
      }
  }
  float rawc[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int q = min(tid + KB * u, 287), r = q / 18, f = q - 18 * r;
    int m[3] = {gx - 1 + f / 3, gy - 1 + (r & 3), gz - 1 + (r >> 2)};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      m[a] += m[a] < 0 ? g.nc : 0;
      while (m[a] >= g.nc) m[a] -= g.nc;
    }
    rawc[u] = force2[3 * ((int64_t)(m[2] * g.nc + m[1]) * g.nc + m[0]) + f % 3];
  }
  const int n = pre[4];
  int r = 0, ci = 0; /* the particle's row, its cell of the row's 4 */
  int64_t p = 0;
  int32_t code[3] = {0, 0, 0};
  double vreal[3] = {0, 0, 0};
  F3 vc = {0.f, 0.f, 0.f};
  auto fetch = [&](int q) {
    r = pre[2] <= q ? 2 : 0;
    r += pre[r + 1] <= q ? 1 : 0;
    p = cs[r][0] + (q - pre[r]);
    ci = (cs[r][1] <= p ? 1 : 0) + (cs[r][2] <= p ? 1 : 0) + (cs[r][3] <= p ? 1 : 0);
    const typename CdWord<IX>::T wx = cd_load<IX>(reinterpret_cast<const char *>(xp) + 3 * IX * p);
    const typename CdWord<IV>::T wv = cd_load<IV>(reinterpret_cast<const char *>(vp) + 3 * IV * p);
    vc = *reinterpret_cast<const F3 *>(vfield + 3 * g.cid(x0 + ci, y0 + (r & 1), z0 + (r >> 1), (int)t));
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      code[a] = (int32_t)fd_code<IX>(wx, a);
      vreal[a] = vdec[(int32_t)(typename IntOf<IV>::T)fd_code<IV>(wv, a) + nvh];
    }
  };
  if (tid < n) fetch(tid);
  if (on)
#pragma unroll
    for (int z = 0; z < PL; ++z) fm[(z * PL + ry) * CH + rc] = raw[z];
  cm[tid] = rawc[0];
  if (tid + KB < 288) cm[tid + KB] = rawc[1];
  __syncthreads();
  const float *ff = reinterpret_cast<const float *>(fm);
  /* corner order of W/pm.f90:146-153 */
  constexpr int ox[8] = {0, 1, 0, 0, 0, 1, 1, 1}, oy[8] = {0, 0, 1, 0, 1, 0, 1, 1}, oz[8] = {0, 0, 0, 1, 1, 1, 0, 1};
  double vm[3] = {0, 0, 0};
  for (int q = tid; q < n;) {
    const int lc[3] = {ci, r & 1, r >> 1}, l0[3] = {x0, y0, z0}, g0[3] = {gx, gy, gz};
    const float vcf[3] = {vc.x, vc.y, vc.z};
#pragma unroll
    for (int k = 0; k < 2; ++k) { /* the fine kick, the coarse kick */
      int m[3];
      float d1[3], d2[3];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        /* as in kick_particle; m: the first of the two planes in the staged block */
        const float tempx = k == 0 ? (float)(4 * (l0[a] + lc[a])) + ((float)cube_ucode(IX, code[a]) + 0.5f) * (IX == 1 ? 0x1p-6f : 0x1p-14f)
                                   : coarse_tempx<IX>(g0[a] + lc[a], code[a]);
        const float fl = floorf(tempx);
        m[a] = (int)fl - (k == 0 ? 4 * l0[a] : g0[a] - 1);
        d1[a] = (float)((int)fl + 1) - tempx;
        d2[a] = 1.0f - d1[a];
      }
      const float *F0 = k == 0 ? ff + (m[2] * PL + m[1]) * RF + 3 * m[0] : cm + (m[2] * 4 + m[1]) * 18 + 3 * m[0];
      const int sy = k == 0 ? RF : 18, sz = k == 0 ? PL * RF : 72;
#pragma unroll
      for (int q8 = 0; q8 < 8; ++q8) {
        const float *F = F0 + oz[q8] * sz + oy[q8] * sy + ox[q8] * 3;
        const float wx = ox[q8] ? d2[0] : d1[0], wy = oy[q8] ? d2[1] : d1[1], wz = oz[q8] ? d2[2] : d1[2];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const float inc = ((F[a] * wx) * wy) * wz;
          vreal[a] = vreal[a] + (double)inc;
        }
      }
      int32_t vcode[3];
      cube_encode_v3(IV, venc, vreal, vcode);
      if (k == 0) {
#pragma unroll
        for (int a = 0; a < 3; ++a) vreal[a] = vdec2[vcode[a] + nvh];
      } else {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const double av = fabs(vreal[a] + (double)vcf[a]);
          vm[a] = av > vm[a] ? av : vm[a];
          vp[3 * p + a] = (typename IntOf<IV>::T)vcode[a];
        }
      }
    }
    q += KB;
    if (q < n) fetch(q);
  }
  vmax_reduce<KB>(vm, vmax_bits);
}
template <int IX, int IV> static int kicks_impl(cube_ctx *c, const float *G, double venc, unsigned long long *vmb) {
  /* With few particles a block's staged mesh costs more than their gathers: with
     1, 2, 3, 4, 8 particles a cell k_kicks takes 598, 625, 658, 706, 880 us on
     128^3 cells and the rows 296, 482, 629, 753, 1149; on 48^3 56, 56, 57, 62, 70
     and 41, 49, 54, 58, 78; on 32^3 and below the two differ by 3 % */
  if (2 * c->nplocal <= 5 * c->ncells && c->nc >= 32) {
    hipLaunchKernelGGL((k_kick<IX, IV, true, true>), dim3((unsigned)(c->ncells / c->nt)), dim3(KT), 0, c->stream,
                       (const typename IntOf<IX>::T *)c->xp, (typename IntOf<IV>::T *)c->vp, c->cstart, c->vfield, c->force_f,
                       c->vdec0, geo_of(c), c->nvbin / 2, 0.f, 0.f, venc, vmb, G, c->vdec1);
    CUBE_LAUNCH_CHECK();
    return CUBE_OK;
  }
  const int64_t nt = c->nt, grid = ((nt + 3) / 4) * ((nt + 1) / 2) * ((nt + 1) / 2) * c->ntiles;
  auto kern = IX == 1 || nt <= 128 ? k_kicks<IX, IV, true> : k_kicks<IX, IV, IX == 1>; /* as in cube_fine_deposit */
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(KB), 0, c->stream, (const typename IntOf<IX>::T *)c->xp,
                     (typename IntOf<IV>::T *)c->vp, c->cstart, c->vfield, c->force_f, c->vdec0, geo_of(c), c->nvbin / 2,
                     venc, vmb, G, c->vdec1);
  CUBE_LAUNCH_CHECK();
  return CUBE_OK;
}

template <int IX, int IV, bool FINE>
static int kick_impl(cube_ctx *c, const float *force, float a_mid, float dt, double venc, unsigned long long *vmb) {
  const int64_t nrows = c->ncells / c->nt;
  hipLaunchKernelGGL((k_kick<IX, IV, FINE, false>), dim3((unsigned)nrows), dim3(KT), 0, c->stream,
                     (const typename IntOf<IX>::T *)c->xp, (typename IntOf<IV>::T *)c->vp, c->cstart, c->vfield, force,
                     c->vdec0, geo_of(c), c->nvbin / 2, a_mid, dt, venc, vmb, (const float *)nullptr, (const double *)nullptr);
  CUBE_LAUNCH_CHECK();
  return CUBE_OK;
}
template <bool FINE>
static int kick(cube_ctx *c, const float *force, float a_mid, float dt, double venc, unsigned long long *vmb) {
  const int x = c->p.izipx, v = c->p.izipv;
  if (x == 1 && v == 1) return kick_impl<1, 1, FINE>(c, force, a_mid, dt, venc, vmb);
  if (x == 1) return kick_impl<1, 2, FINE>(c, force, a_mid, dt, venc, vmb);
  if (v == 1) return kick_impl<2, 1, FINE>(c, force, a_mid, dt, venc, vmb);
  return kick_impl<2, 2, FINE>(c, force, a_mid, dt, venc, vmb);
}

/* fine kick, W/pm.f90:129-159: decode with sigma_vi, encode with sigma_vi_new */
int cube_fine_kick(cube_ctx *c, float a_mid, float dt, float sigma_vi, float sigma_vi_new, int sync) {
  int st = cube_vdec_table(c, c->vdec0, sigma_vi);
  if (st) return st;
  st = kick<true>(c, c->force_f, a_mid, dt, cube_vconst(sigma_vi_new), nullptr);
  if (st) return st;
  if (sync) CUBE_CHECK(hipStreamSynchronize(c->stream));
  return CUBE_OK;
}

/* The step's two kicks in one pass over the particles (W/pm.f90:129-159,
   then :193 and :322-387): the fine kick decodes with sigma_vi and encodes
   with sigma_vi_new, the coarse kick decodes and encodes with sigma_vi_new;
   vmax (W/pm.f90:349) as cube_coarse_kick.  force_f holds the fine kick's
   factors (((F*a_mid)*dt)/6)/pi, formed by the step's force pipeline for
   this a_mid and dt.  Equal to cube_fine_kick then
   cube_coarse_kick(sigma_vi_new) on the plain force bit for bit. */
int cube_pm_kicks(cube_ctx *c, float a_mid, float dt, float sigma_vi, float sigma_vi_new, float *vmax) {
  int st;
  unsigned long long *vsl = c->slots + CUBE_SLOT_VMAX * CUBE_SLOTS;
  if ((st = cube_slots_open(c, vsl, 3))) return st;
  float *G = reinterpret_cast<float *>(c->specd_c);
  hipLaunchKernelGGL(k_kick_prep, dim3(2048), dim3(256), 0, c->stream, c->force_c, 3 * c->ncells, a_mid, dt, G, c->tanf_tab,
                     (int)c->nvbin, cube_vconst(sigma_vi), cube_vconst(sigma_vi_new), c->vdec0, c->vdec1);
  CUBE_LAUNCH_CHECK();
  const double venc = cube_vconst(sigma_vi_new);
  const int ix = c->p.izipx, iv = c->p.izipv;
  if (ix == 1 && iv == 1) st = kicks_impl<1, 1>(c, G, venc, vsl);
  else if (ix == 1) st = kicks_impl<1, 2>(c, G, venc, vsl);
  else if (iv == 1) st = kicks_impl<2, 1>(c, G, venc, vsl);
  else st = kicks_impl<2, 2>(c, G, venc, vsl);
  if (st) return st;
  hipLaunchKernelGGL(k_pm_result, dim3(3), dim3(CUBE_SLOTS), 0, c->stream, vsl, c->dred, c->ured, c->hres);
  CUBE_LAUNCH_CHECK();
  cube_words_close(c, cube_slots_bits(c, vsl, 3));
  CUBE_CHECK(hipStreamSynchronize(c->stream));
  const unsigned long long *h = c->hres + HR_VMAX;
  for (int a = 0; a < 3; ++a) {
    double d;
    memcpy(&d, &h[a], sizeof(d));
    if (vmax) vmax[a] = (float)d; /* vmax is real(4) (W/variables.f90:35) */
  }
  return CUBE_OK;
}

/* coarse kick, W/pm.f90:322-387: decode and encode with sigma_vi */
int cube_coarse_kick(cube_ctx *c, float a_mid, float dt, float sigma_vi, float *vmax) {
  int st = cube_vdec_table(c, c->vdec0, sigma_vi);
  if (st) return st;
  unsigned long long *vsl = c->slots + CUBE_SLOT_VMAX * CUBE_SLOTS;
  if ((st = cube_slots_open(c, vsl, 3))) return st;
  /* G in the coarse spectra scratch, free once force_c is formed */
  float *G = reinterpret_cast<float *>(c->specd_c);
  hipLaunchKernelGGL(k_kick_prescale, dim3(2048), dim3(256), 0, c->stream, c->force_c, 3 * c->ncells, a_mid, dt, G);
  CUBE_LAUNCH_CHECK();
  st = kick<false>(c, G, a_mid, dt, cube_vconst(sigma_vi), vsl);
  if (st) return st;
  if ((st = cube_slots_fold(c, vsl, 3, 0, c->hres + HR_VMAX, nullptr))) return st;
  CUBE_CHECK(hipStreamSynchronize(c->stream));
  const unsigned long long *h = c->hres + HR_VMAX;
  for (int a = 0; a < 3; ++a) {
    double d;
    memcpy(&d, &h[a], sizeof(d));
    if (vmax) vmax[a] = (float)d; /* vmax is real(4) (W/variables.f90:35) */
  }
  return CUBE_OK;
}

/* ---------------- Green's functions ---------------- */
/* real-space fine kernel of component d on the nf^3 mesh: the 16^3 table at
   offsets 0..15, odd-mirrored in axis d and even in the others
   (W/kernel_f.f90:25-31), corner |o|<=pp_range zeroed when PP is on */
__global__ void k_fine_kernel_rs(float *rs, int n, const float *tab, int d, int pp_on, int pp_range) {
  const int64_t n3 = (int64_t)n * n * n;
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n3; q += (int64_t)gridDim.x * blockDim.x) {
    const int x = (int)(q % n), y = (int)((q / n) % n), z = (int)(q / ((int64_t)n * n));
    const int o[3] = {x <= n / 2 ? x : x - n, y <= n / 2 ? y : y - n, z <= n / 2 ? z : z - n};
    float v = 0.f;
    if (o[0] >= -15 && o[0] <= 15 && o[1] >= -15 && o[1] <= 15 && o[2] >= -15 && o[2] <= 15) {
      const int a0 = o[0] < 0 ? -o[0] : o[0], a1 = o[1] < 0 ? -o[1] : o[1], a2 = o[2] < 0 ? -o[2] : o[2];
      const bool zero = pp_on && a0 <= pp_range && a1 <= pp_range && a2 <= pp_range;
      if (!zero) {
        v = tab[((a2 * 16 + a1) * 16 + a0) * 3 + d];
        if (o[d] < 0) v = -v;
      }
    }
    rs[q] = v;
  }
}
/* keep Im of the positive-frequency octant 0..n/2 of component d in the
   blocked storage of cube_kernf_index (columns past n/2 of the last block
   hold zero) */
__global__ void k_extract_octant(const float2 *spec, int n, float *kern, int d) {
  const int h = n / 2 + 1;
  const int64_t kb = cube_kernf_blocks(h), tot = (int64_t)h * kb * h * 16;
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < tot; q += (int64_t)gridDim.x * blockDim.x) {
    const int kz = (int)((q / 16) % h), b = (int)((q / (16 * h)) % kb), ky = (int)(q / (16 * h * kb));
    const int kx = b * 16 + (int)(q % 16);
    kern[(int64_t)d * tot + q] = kx < h ? spec[((int64_t)kz * n + ky) * cube_spec_pitch(n) + kx].y : 0.f;
  }
}
/* uncorrected coarse kernel -r/r^3 in fine units (W/kernel_c.f90:16-28) and
   the table-corrected one (:31-72), component d */
__global__ void k_coarse_kernel_rs(float *rs_plain, float *rs_corr, int nc, const float *ctab, int d) {
  const int64_t n3 = (int64_t)nc * nc * nc;
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n3; q += (int64_t)gridDim.x * blockDim.x) {
    const int ii[3] = {(int)(q % nc), (int)((q / nc) % nc), (int)(q / ((int64_t)nc * nc))};
    float rx[3];
    for (int a = 0; a < 3; ++a) rx[a] = (float)(4 * ((ii[a] + nc / 2) % nc - nc / 2));
    const float r = sqrtf((rx[0] * rx[0] + rx[1] * rx[1]) + rx[2] * rx[2]);
    const float v = r == 0.f ? 0.f : -rx[d] / (r * (r * r));
    rs_plain[q] = v;
    /* octant copies of the 4^3 table: low block 0..3 or high block nc-3..nc-1
       (mirrored index nc-i), sign flipped for component d in a high block */
    int ti[3];
    bool in = true;
    float sgn = 1.f;
    for (int a = 0; a < 3; ++a) {
      if (ii[a] < 4) ti[a] = ii[a];
      else if (ii[a] >= nc - 3) {
        ti[a] = nc - ii[a];
        if (a == d) sgn = -sgn;
      } else in = false;
    }
    rs_corr[q] = in ? sgn * ctab[((ti[2] * 4 + ti[1]) * 4 + ti[0]) * 3 + d] : v;
  }
}
/* LRCKCORR (W/kernel_c.f90:301-325), all real(4) */
__global__ void k_lrckcorr(const float2 *spec_corr, const float2 *spec_plain, int nc, float *kern, int d) {
  const int nh = nc / 2 + 1;
  const int64_t tot = (int64_t)nh * nc * nc;
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < tot; q += (int64_t)gridDim.x * blockDim.x) {
    const int ix = (int)(q % nh), iy = (int)((q / nh) % nc), iz = (int)(q / ((int64_t)nh * nc));
    const int ki[3] = {(ix + nc / 2) % nc - nc / 2, (iy + nc / 2) % nc - nc / 2, (iz + nc / 2) % nc - nc / 2};
    float kx[3], ks[3];
    for (int a = 0; a < 3; ++a) {
      kx[a] = (float)ki[a];
      ks[a] = 2.0f * sinf(CUBE_PI_F * kx[a] / (float)nc);
    }
    const float kr = sqrtf((kx[0] * kx[0] + kx[1] * kx[1]) + kx[2] * kx[2]);
    const int64_t sq = ((int64_t)iz * nc + iy) * cube_spec_pitch(nc) + ix;
    const float kc = spec_corr[sq].y;
    const float cu = spec_plain[sq].y;
    float out = kc;
    /* for nc < 24 the |k|<=8 sphere reaches the Nyquist plane of axis d,
       where Im FFT of the odd kernel is exactly zero and the reference
       divides by it (NaN); those modes keep the uncorrected value */
    if (!(kr > 8.0f || ki[d] == 0 || 2 * ki[d] == -nc)) {
      const float ssum = (ks[0] * ks[0] + ks[1] * ks[1]) + ks[2] * ks[2];
      out = ((((kc * 0.25f) * CUBE_PI_F) * ks[d]) / ssum) / cu;
    }
    kern[(int64_t)d * tot + q] = out;
  }
}

int cube_green_init(cube_ctx *c, const float *wfxyzf, const float *wfxyzc) {
  float *dtab = nullptr, *dctab = nullptr;
  CUBE_CHECK(hipMalloc(&dtab, 16 * 16 * 16 * 3 * sizeof(float)));
  CUBE_CHECK(hipMalloc(&dctab, 4 * 4 * 4 * 3 * sizeof(float)));
  CUBE_CHECK(hipMemcpy(dtab, wfxyzf, 16 * 16 * 16 * 3 * sizeof(float), hipMemcpyHostToDevice));
  CUBE_CHECK(hipMemcpy(dctab, wfxyzc, 4 * 4 * 4 * 3 * sizeof(float), hipMemcpyHostToDevice));
  int st = CUBE_OK;
  const int nf = (int)c->nf, nc = (int)c->nc;
  for (int d = 0; d < 3 && !st; ++d) {
    hipLaunchKernelGGL(k_fine_kernel_rs, dim3(2048), dim3(256), 0, c->stream, c->rho_f, nf, dtab, d, c->p.pp_on,
                       c->p.pp_range);
    if (hipGetLastError() != hipSuccess) st = CUBE_ERR_HIP;
    if (!st) st = cube_fft_forward_full(c, c->plan_f, c->rho_f, c->spec_f);
    if (!st) {
      hipLaunchKernelGGL(k_extract_octant, dim3(2048), dim3(256), 0, c->stream, c->spec_f, nf, c->kern_f, d);
      if (hipGetLastError() != hipSuccess) st = CUBE_ERR_HIP;
    }
  }
  for (int d = 0; d < 3 && !st; ++d) {
    float *plain = c->rho_c, *corr = (float *)c->specd_c; /* specd_c is large enough for nc^3 floats */
    float2 *sp_plain = c->spec_c, *sp_corr = c->specd_c + (int64_t)cube_spec_pitch(nc) * nc * nc;
    hipLaunchKernelGGL(k_coarse_kernel_rs, dim3(1024), dim3(256), 0, c->stream, plain, corr, nc, dctab, d);
    if (hipGetLastError() != hipSuccess) st = CUBE_ERR_HIP;
    if (!st) st = cube_fft_forward_full(c, c->plan_c, plain, sp_plain);
    /* corr lives in specd_c plane 0; transform it into plane 1 */
    if (!st) st = cube_fft_forward_full(c, c->plan_c, corr, sp_corr);
    if (!st) {
      hipLaunchKernelGGL(k_lrckcorr, dim3(1024), dim3(256), 0, c->stream, sp_corr, sp_plain, nc, c->kern_c, d);
      if (hipGetLastError() != hipSuccess) st = CUBE_ERR_HIP;
    }
  }
  (void)hipStreamSynchronize(c->stream);
  (void)hipFree(dtab);
  (void)hipFree(dctab);
  return st;
}

/* ---------------- fine potential ----------------
 * The reference's main path never forms a potential (its fine force kernel
 * goes from i*K*rho_k straight to forces); it ships the fine potential
 * kernel table CUBEnu/kernels/wg1.ascii (CUBEnu/kernels/README:8-9), 16^3
 * values at offsets 0..15.  Mirrored evenly into the periodic nf^3 mesh
 * (zero beyond offset 15, the near corner zeroed with PP on as in the force
 * kernel) its spectrum is real, and phi = C2R(Re K * R2C(rho_f)) / nf^3,
 * divided by nf three times in real(4) like the force (W/pm.f90:122-123). */
__global__ void k_fine_pot_rs(float *rs, int n, const float *tab, int pp_on, int pp_range) {
  const int64_t n3 = (int64_t)n * n * n;
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n3; q += (int64_t)gridDim.x * blockDim.x) {
    const int x = (int)(q % n), y = (int)((q / n) % n), z = (int)(q / ((int64_t)n * n));
    const int a0 = min(x, n - x), a1 = min(y, n - y), a2 = min(z, n - z);
    float v = 0.f;
    if (a0 <= 15 && a1 <= 15 && a2 <= 15 && !(pp_on && a0 <= pp_range && a1 <= pp_range && a2 <= pp_range))
      v = tab[(a2 * 16 + a1) * 16 + a0];
    rs[q] = v;
  }
}
__global__ void k_mul_re(const float2 *spec, const float2 *kspec, float2 *out, int64_t n) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x) {
    const float2 s = spec[q];
    const float k = kspec[q].x;
    out[q] = make_float2(s.x * k, s.y * k);
  }
}
__global__ void k_div3(float *a, int64_t n3, float n) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n3; q += (int64_t)gridDim.x * blockDim.x) {
    float v = a[q];
    v = v / n;
    v = v / n;
    v = v / n;
    a[q] = v;
  }
}

int cube_fine_potential(cube_ctx *c, const float *wg1) {
  const int nf = (int)c->nf;
  const int64_t nf3 = (int64_t)nf * nf * nf, ns = (int64_t)cube_spec_pitch(nf) * nf * nf;
  float *dtab = nullptr;
  CUBE_CHECK(hipMalloc(&dtab, 16 * 16 * 16 * sizeof(float)));
  int st = CUBE_OK;
  if (hipMemcpy(dtab, wg1, 16 * 16 * 16 * sizeof(float), hipMemcpyHostToDevice) != hipSuccess) st = CUBE_ERR_HIP;
  /* rho_k in spec_f; the kernel in force_f's first nf^3 floats, its
     spectrum in force spectrum 0, the product back in spec_f; phi into
     force_f's first nf^3 floats */
  if (!st) st = cube_fft_forward_full(c, c->plan_f, c->rho_f, c->spec_f);
  if (!st) {
    hipLaunchKernelGGL(k_fine_pot_rs, dim3(2048), dim3(256), 0, c->stream, c->force_f, nf, dtab, c->p.pp_on,
                       c->p.pp_range);
    if (hipGetLastError() != hipSuccess) st = CUBE_ERR_HIP;
  }
  if (!st) st = cube_fft_forward_full(c, c->plan_f, c->force_f, c->specd_f);
  if (!st) {
    hipLaunchKernelGGL(k_mul_re, dim3(2048), dim3(256), 0, c->stream, c->spec_f, c->specd_f, c->spec_f, ns);
    if (hipGetLastError() != hipSuccess) st = CUBE_ERR_HIP;
  }
  if (!st) st = cube_fft_inverse_full(c, c->plan_f, c->spec_f, c->force_f);
  if (!st) {
    hipLaunchKernelGGL(k_div3, dim3(2048), dim3(256), 0, c->stream, c->force_f, nf3, (float)nf);
    if (hipGetLastError() != hipSuccess) st = CUBE_ERR_HIP;
  }
  (void)hipStreamSynchronize(c->stream);
  (void)hipFree(dtab);
  return st;
}
