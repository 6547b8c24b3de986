/*
 * cube_power.hip -- matter power spectrum of the particle state
 * (cube_power in include/cube.h), the analysis of WU/cicpower.f90:96-187 and
 * WU/powerspectrum.f90:28-135 on the GPU: cell-centred CIC in FP64,
 * delta = rho/mean - 1, FP32 FFT, then per-mode |delta_k|^2 binned in
 * linear |k| bins with the sinc^4 CIC window removed.
 */
#include "cube_internal.h"
#include <math.h>
#include <string.h>
#include <algorithm>
#include <mutex>
#include <type_traits>

#define PW_T 256

/*
 * Cell-centred CIC of the disjoint state: x = global coarse position, mesh
 * coordinate x*ng/nc - 0.5 (WU/cicpower.f90:113).
 *
 * Gathered, for a mesh at least as fine as the coarse cells: a workgroup owns
 * B^3 mesh cells, FP64 sums in LDS, and its waves take the rows of coarse cells
 * whose particles can reach them (6^3 cells for 16^3 mesh cells of a quarter
 * cell), 64 particles at a time.  Of these only what reaches its mesh cells (one
 * in three) goes to the wave's queue, whose words are deposited 64 at a time.
 * It writes delta itself, so the FP64 mesh, its clearing and a pass over it are
 * gone.  Bound by VALU (the test of what a row's particles reach, in FP64).
 * 128^3 particles on 256^3: 572 + 33 + 11 us with global FP64 atomics -> 86 us
 * (139 without the queue, 101 with the row's coordinates in vector registers).
 */
#define PG_B 16
#define PG_T 512
template <int IX>
__global__ __launch_bounds__(PG_T) void k_pw_gather(const typename IntOf<IX>::T *__restrict__ xp,
                                                    const int64_t *__restrict__ cstart, Geo g, int ng, int lb,
                                                    double inv_mean, float *__restrict__ delta) {
  __shared__ double acc[PG_B * PG_B * PG_B];
  __shared__ uint64_t queue[PG_T / 64][128]; /* per wave: codes (3 x 16 bits), cell (3 x 5) */
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int B = 1 << lb, nb = (ng + B - 1) >> lb;
  const int c0[3] = {(int)(blockIdx.x % nb) * B, (int)(blockIdx.x / nb % nb) * B, (int)(blockIdx.x / nb / nb) * B};
  const int nc = g.nc, nt = g.nt;
  int n[3], lo[3], nx[3]; /* own mesh cells; first coarse cell and their number, unwrapped: within [-1, nc] */
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    n[a] = min(B, ng - c0[a]);
    /* first planes c0-1..c0+n-1, so x*ng/nc in [c0-1/2, c0+n+1/2) */
    lo[a] = c0[a] == 0 ? -1 : (2 * c0[a] - 1) * nc / (2 * ng);
    nx[a] = (2 * (c0[a] + n[a]) + 1) * nc / (2 * ng) - lo[a] + 1; /* at most B + 3 */
  }
  for (int q = tid; q < B * B * B; q += PG_T) acc[q] = 0.0;
  /* a cell's id is the sum of its three axes' parts, lane i holding those of
     the i-th cell of each axis */
  int part[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int u = lo[a] + lane, gu = u < 0 ? u + nc : (u >= nc ? u - nc : u), t = gu / nt, l = gu - t * nt;
    part[a] = a == 0 ? l + nt * nt * nt * t : (a == 1 ? nt * l + nt * nt * nt * g.nnt * t
                                                    : nt * nt * l + nt * nt * nt * g.nnt * g.nnt * t);
  }
  __syncthreads();
  const double scale = (double)ng / (double)nc;
  /* one axis of a particle: its first plane among this workgroup's, and the
     weight of the second */
  auto axis = [&](int u, int a, uint32_t code, int &f, double &d2) {
    const int img = u < 0 ? -1 : (u >= nc ? 1 : 0);
    const double x = (double)(u - img * nc) + ((double)code + 0.5) * (IX == 1 ? 0x1p-8 : 0x1p-16); /* cube_xoff */
    const double m = x * scale - 0.5, fl = floor(m);
    d2 = m - fl;
    f = (int)fl + (img * ng - c0[a]);
  };
  /* the cells of row (y, z), one per lane */
  auto cells = [&](int y, int z, int64_t &first, int &cnt) {
    first = 0;
    cnt = 0;
    const int cc = part[0] + __builtin_amdgcn_readlane(part[1], y) + __builtin_amdgcn_readlane(part[2], z);
    if (z < nx[2] && lane < nx[0]) {
      first = cstart[cc];
      cnt = (int)(cstart[cc + 1] - first);
    }
  };
  int nq = 0; /* words queued */
  uint64_t *qw = queue[wv];
  auto drain = [&](int keep) { /* down to at most `keep` */
    while (nq > keep) {
      const int take = min(nq, 64);
      if (lane < take) {
        const uint64_t w = qw[nq - take + lane];
        int f[3];
        double wt[3][2];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          axis(lo[a] + (int)((w >> (48 + 5 * a)) & 31), a, (uint32_t)(w >> (16 * a)) & 0xffffu, f[a], wt[a][1]);
          wt[a][0] = 1.0 - wt[a][1];
        }
        double *at = acc + ((f[2] << lb) + f[1]) * B + f[0];
#pragma unroll
        for (int cz = 0; cz < 2; ++cz)
#pragma unroll
          for (int cy = 0; cy < 2; ++cy)
#pragma unroll
            for (int cx = 0; cx < 2; ++cx)
              if ((unsigned)(f[0] + cx) < (unsigned)n[0] && (unsigned)(f[1] + cy) < (unsigned)n[1] &&
                  (unsigned)(f[2] + cz) < (unsigned)n[2])
                atomicAdd(at + (cz * B + cy) * B + cx, wt[0][cx] * wt[1][cy] * wt[2][cz]);
      }
      nq -= take;
    }
  };
  int y = wv, z = 0, cnt;
  while (y >= nx[1]) y -= nx[1], ++z;
  int64_t first;
  cells(y, z, first, cnt);
  while (z < nx[2]) {
    const int sc = wave_incl_scan(cnt), total = __builtin_amdgcn_readlane(sc, 63);
    const int64_t off = first - (sc - cnt); /* a particle's number from its place in the row */
    const uint64_t yz = ((uint64_t)z << 58) | ((uint64_t)y << 53);
    const int uy = lo[1] + y, uz = lo[2] + z;
    y += PG_T / 64;
    while (y >= nx[1]) y -= nx[1], ++z;
    cells(y, z, first, cnt); /* the next row's, in flight */
    for (int o = 0; o < total; o += 64) {
      const int l = o + lane;
      int c = 0; /* its cell: the cells that end at or before it */
      for (int i = 0; i < nx[0] - 1; ++i) c += __builtin_amdgcn_readlane(sc, i) <= l ? 1 : 0;
      const int64_t p = __shfl(off, c, 64) + l;
      bool in = l < total;
      uint64_t w = yz | ((uint64_t)c << 48);
      if (in) {
        const int u[3] = {lo[0] + c, uy, uz};
        /* the arrays end in padding: one read of its 3 or 6 bytes */
        typename std::conditional<IX == 1, uint32_t, uint64_t>::type word;
        __builtin_memcpy(&word, xp + 3 * p, sizeof(word));
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const uint32_t code = (uint32_t)(word >> (8 * IX * a)) & (IX == 1 ? 0xffu : 0xffffu);
          int f;
          double d2;
          axis(u[a], a, code, f, d2);
          in = in && f >= -1 && f < n[a];
          w |= (uint64_t)code << (16 * a);
        }
      }
      const uint64_t hit = __ballot(in);
      if (in) qw[nq + __popcll(hit & ((1ull << lane) - 1ull))] = w;
      nq += __popcll(hit);
      wave_lds_sync();
      drain(63);
      wave_lds_sync();
    }
  }
  drain(0);
  __syncthreads();
  for (int q = tid; q < B * B * B; q += PG_T) {
    const int X = q & (B - 1), Y = (q >> lb) & (B - 1), Z = q >> (2 * lb);
    if (X < n[0] && Y < n[1] && Z < n[2])
      delta[((int64_t)(c0[2] + Z) * ng + c0[1] + Y) * ng + c0[0] + X] = (float)(acc[q] * inv_mean - 1.0);
  }
}
/* The same for a mesh coarser than the coarse cells, where few mesh cells take
   many particles each and a gathering workgroup would read too many cells: one
   workgroup per row of coarse cells, FP64 atomics into the mesh */
template <int IX>
__global__ __launch_bounds__(PW_T) void k_pw_deposit(const typename IntOf<IX>::T *__restrict__ xp,
                                                     const int64_t *__restrict__ cstart, Geo g, int ng,
                                                     double *__restrict__ rho) {
  const int nt = g.nt;
  const int64_t row = blockIdx.x;
  const int j = (int)(row % nt), k = (int)((row / nt) % nt), t = (int)(row / ((int64_t)nt * nt));
  const int tt[3] = {t % g.nnt, (t / g.nnt) % g.nnt, t / (g.nnt * g.nnt)};
  __shared__ int64_t cs[520];
  const int64_t c0 = row * nt;
  for (int i = threadIdx.x; i <= nt; i += PW_T) cs[i] = cstart[c0 + i];
  __syncthreads();
  const double scale = (double)ng / (double)g.nc;
  for (int64_t p = cs[0] + threadIdx.x; p < cs[nt]; p += PW_T) {
    int lo = 0, hi = nt;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (cs[mid] <= p) lo = mid; else hi = mid;
    }
    const int cell[3] = {tt[0] * nt + lo, tt[1] * nt + j, tt[2] * nt + k};
    int i1[3];
    double w[3][2];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const double x = (double)cell[a] + cube_xoff(IX, (int32_t)xp[3 * p + a]);
      const double m = x * scale - 0.5;
      const double fl = floor(m);
      const double d2 = m - fl;
      i1[a] = (int)fl;
      w[a][0] = 1.0 - d2;
      w[a][1] = d2;
    }
#pragma unroll
    for (int cz = 0; cz < 2; ++cz)
#pragma unroll
      for (int cy = 0; cy < 2; ++cy)
#pragma unroll
        for (int cx = 0; cx < 2; ++cx) {
          const int x = wrapi(i1[0] + cx, ng), y = wrapi(i1[1] + cy, ng), z = wrapi(i1[2] + cz, ng);
          atomicAdd(rho + ((int64_t)z * ng + y) * ng + x, w[0][cx] * w[1][cy] * w[2][cz]);
        }
  }
}

__global__ void k_pw_delta(const double *rho, int64_t n3, double inv_mean, float *delta) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n3; q += (int64_t)gridDim.x * blockDim.x)
    delta[q] = (float)(rho[q] * inv_mean - 1.0);
}

__device__ static inline double sincd(double k, int n) {
  if (k == 0.0) return 1.0;
  const double a = 3.14159265358979323846 * k / (double)n;
  return sin(a) / a;
}

/* bins 1..nbin of sum |k|, sum Delta^2, count (WU/powerspectrum.f90:60-133).
   A wave takes rows of modes (iy, iz), lanes along ix, the window factors of an
   axis from a table in LDS (their sines per mode were the kernel's work) and
   neighbouring lanes, whose modes often share a bin, on different copies of
   the bins; few large workgroups, as each adds all bins to the totals.  Bound
   by VALU (FP64 square root, division) and the read.  256^3: 149 -> 46 us. */
#define PWB_T 1024
__global__ __launch_bounds__(PWB_T) void k_pw_bin(const float2 *__restrict__ spec, int ng, int nl, int R,
                                                  double *__restrict__ ksum, double *__restrict__ psum,
                                                  unsigned long long *__restrict__ cnt) {
  /* R copies of the bins 1..nl, interleaved: R*(nl+1) sums each, as many
     counters, then ng/2+1 window factors */
  extern __shared__ double lsum[];
  double *lpow = lsum + R * (nl + 1), *win = lpow + 2 * R * (nl + 1);
  unsigned long long *lcnt = reinterpret_cast<unsigned long long *>(lpow + R * (nl + 1));
  for (int i = threadIdx.x; i < R * (nl + 1); i += PWB_T) {
    lsum[i] = 0.0;
    lpow[i] = 0.0;
    lcnt[i] = 0ull;
  }
  for (int i = threadIdx.x; i <= ng / 2; i += PWB_T) win[i] = sincd(i, ng); /* even in k */
  __syncthreads();
  const int ny = ng / 2, sp = cube_spec_pitch(ng);
  const double n3 = (double)ng * ng * ng;
  const int lane = threadIdx.x & 63, copy = lane % R;
  const bool pow2 = (ng & (ng - 1)) == 0; /* then 1/n3 is exact, and the product is the quotient */
  const double in3 = 1.0 / n3;
  auto mode = [&](int iz, int iy, int ix) {
    const int ky = iy < ny ? iy : iy - ng, kz = iz < ny ? iz : iz - ng;
    bool skip = ix == 0 && iy == 0 && iz == 0;
    const bool edge = ix == 0 || ix == ny;
    skip = skip || (edge && iy > ny) || (edge && (iy == 0 || iy == ny) && iz > ny);
    if (skip) return;
    const int kx = ix == ny ? -ny : ix;
    const double kr = sqrt((double)(kx * kx + ky * ky + kz * kz));
    const int ib = (int)rint(kr);
    if (ib < 1 || ib > nl) return;
    const float2 v = spec[((int64_t)iz * ng + iy) * sp + ix];
    const double re = pow2 ? (double)v.x * in3 : (double)v.x / n3, im = pow2 ? (double)v.y * in3 : (double)v.y / n3;
    const double s = win[ix] * win[abs(ky)] * win[abs(kz)];
    const double amp = (re * re + im * im) / (s * s * s * s) * 4.0 * 3.14159265358979323846 * kr * kr * kr;
    const int b = ib * R + copy;
    atomicAdd(lsum + b, kr);
    atomicAdd(lpow + b, amp);
    atomicAdd(lcnt + b, 1ull);
  };
  const int wave = blockIdx.x * (PWB_T / 64) + (int)(threadIdx.x >> 6), nw = gridDim.x * (PWB_T / 64);
  for (int row = wave; row < ng * ng; row += nw) {
    const int iz = row / ng, iy = row - iz * ng;
    for (int ix = lane; ix < ny; ix += 64) mode(iz, iy, ix);
  }
  for (int q = wave * 64 + lane; q < ng * ng; q += nw * 64) mode(q / ng, q % ng, ny); /* the last column */
  __syncthreads();
  for (int i = threadIdx.x; i <= nl; i += PWB_T) {
    double ks = 0.0, ps = 0.0;
    unsigned long long n = 0;
    for (int q = 0; q < R; ++q) {
      ks += lsum[i * R + q];
      ps += lpow[i * R + q];
      n += lcnt[i * R + q];
    }
    if (n) {
      atomicAdd(ksum + i, ks);
      atomicAdd(psum + i, ps);
      atomicAdd(cnt + i, n);
    }
  }
}

__global__ void k_pw_zero(double *a, int64_t n) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x)
    a[q] = 0.0;
}

/* Checks shared by both entry points. */
static int power_args(cube_ctx *c, int32_t ng, int32_t nbin, const double *ksum, const double *psum,
                      const int64_t *count) {
  if (!c || !ksum || !psum || !count || ng < 4 || ng > c->nf || c->nf % ng || nbin < 1) return CUBE_ERR_INVALID;
  if (!c->has_state) return CUBE_ERR_STATE;
  if (c->nt > 519) return CUBE_ERR_INVALID; /* k_pw_deposit stages nt+1 row offsets in LDS */
  /* room for an FP64 mesh in the force spectra, where ng < nc deposits (meshes
     refused for it stay refused where the gathering deposit needs none) */
  if ((size_t)ng * ng * ng * sizeof(double) >
      (size_t)c->fine_nspec * cube_spec_pitch((int)c->nf) * c->nf * c->nf * sizeof(float2))
    return CUBE_ERR_INVALID;
  return CUBE_OK;
}

/* Deposit, contrast, forward FFT and binning on the context's stream: the
   FP32 delta in rho_f (through an FP64 mesh in the force spectra where ng <
   nc), its spectrum in spec_f; bins = 3*(nbin+1) doubles (sum |k|, sum
   Delta^2, count), cleared here by a fill kernel. */
template <int IX>
static void power_deposit(cube_ctx *c, int32_t ng) {
  const int64_t n3 = (int64_t)ng * ng * ng;
  const double inv_mean = (double)n3 / (double)c->nplocal;
  const typename IntOf<IX>::T *xp = (const typename IntOf<IX>::T *)c->xp;
  if (ng >= c->nc) {
    /* 16^3 mesh cells a workgroup, 8^3 (half the particles read are its own)
       where that would be too few for 256 CUs, 4^3 where even these would be 64
       at most and each would go through its rows of particles one by one: a call
       on 16^3 of 32^3 particles takes 121 us with 8^3, 98 with 4^3 (103 by the
       atomics below), on 32^3 of 64^3 123 and 104 (140); on 48^3 of 24^3, 216
       workgroups of 8^3, 102 and 107 (108) */
    const int n16 = (ng + PG_B - 1) / PG_B, n8 = (ng + 7) / 8;
    const int lb = n16 * n16 * n16 >= 512 ? 4 : (n8 * n8 * n8 > 64 ? 3 : 2), nb = (ng + (1 << lb) - 1) >> lb;
    hipLaunchKernelGGL(k_pw_gather<IX>, dim3((unsigned)(nb * nb * nb)), dim3(PG_T), 0, c->stream, xp, c->cstart, geo_of(c),
                       ng, lb, inv_mean, c->rho_f);
    return;
  }
  double *rho = reinterpret_cast<double *>(c->specd_f);
  hipLaunchKernelGGL(k_pw_zero, dim3(1024), dim3(256), 0, c->stream, rho, n3);
  hipLaunchKernelGGL(k_pw_deposit<IX>, dim3((unsigned)(c->ncells / c->nt)), dim3(PW_T), 0, c->stream, xp, c->cstart,
                     geo_of(c), ng, rho);
  hipLaunchKernelGGL(k_pw_delta, dim3(1024), dim3(256), 0, c->stream, rho, n3, inv_mean, c->rho_f);
}
static int power_device(cube_ctx *c, int32_t ng, int32_t nbin, float2 *tw, double *bins) {
  hipLaunchKernelGGL(k_pw_zero, dim3(1), dim3(256), 0, c->stream, bins, (int64_t)3 * (nbin + 1));
  if (c->p.izipx == 1)
    power_deposit<1>(c, ng);
  else
    power_deposit<2>(c, ng);
  if (hipGetLastError() != hipSuccess) return CUBE_ERR_HIP;
  int st = cube_fft_forward_full_tw(c, ng, tw, c->rho_f, c->spec_f);
  if (st) return st;
  const size_t per_bin = 2 * sizeof(double) + sizeof(unsigned long long);
  if ((nbin + 1) * per_bin > 160 * 1024) return CUBE_ERR_HIP; /* what LDS holds of the bins asked for */
  const int nl = nbin < ng ? nbin : ng; /* |k| <= 0.87 ng: the bins above stay empty */
  /* as many copies as neighbouring lanes share bins, within 128 KiB */
  const int R = std::max(1, std::min(16, (int)(128 * 1024 / ((nl + 1) * per_bin))));
  const size_t lds = R * (nl + 1) * per_bin + (ng / 2 + 1) * sizeof(double);
  hipLaunchKernelGGL(k_pw_bin, dim3(256), dim3(PWB_T), lds, c->stream, c->spec_f, ng, nl, R, bins, bins + (nbin + 1),
                     (unsigned long long *)(bins + 2 * (nbin + 1)));
  return hipGetLastError() != hipSuccess ? CUBE_ERR_HIP : CUBE_OK;
}

extern "C" int cube_power(cube_ctx *c, int32_t ng, int32_t nbin, double *ksum, double *psum, int64_t *count) {
  if (c) c->pm_ahead = 0; /* forces formed ahead by ext_pp_force no longer apply */
  int st = power_args(c, ng, nbin, ksum, psum, count);
  if (st) return st;
  CUBE_CHECK(hipSetDevice(c->device));
  /* the bin sums in the force mesh, the twiddles in a plan of their own */
  double *bins = reinterpret_cast<double *>(c->force_f);
  if ((size_t)(3 * (nbin + 1)) * sizeof(double) > (size_t)3 * c->nf * c->nf * c->nf * sizeof(float))
    return CUBE_ERR_INVALID;
  FFTPlan *plan = nullptr;
  st = cube_fft_create(c, ng, &plan);
  if (st) return st;
  st = power_device(c, ng, nbin, cube_fft_plan_twiddles(plan), bins);
  if (!st) {
    double *h = new double[3 * (nbin + 1)];
    if (hipMemcpyAsync(h, bins, 3 * (nbin + 1) * sizeof(double), hipMemcpyDeviceToHost, c->stream) != hipSuccess ||
        hipStreamSynchronize(c->stream) != hipSuccess)
      st = CUBE_ERR_HIP;
    if (!st) {
      const unsigned long long *hc = reinterpret_cast<const unsigned long long *>(h + 2 * (nbin + 1));
      for (int b = 1; b <= nbin; ++b) {
        ksum[b - 1] = h[b];
        psum[b - 1] = h[nbin + 1 + b];
        count[b - 1] = (int64_t)hc[b];
      }
    }
    delete[] h;
  }
  (void)hipStreamSynchronize(c->stream);
  cube_fft_destroy(plan);
  return st;
}

/* ---------------- cube_power_noalloc ----------------
 * The same spectrum without any allocation in the call: the twiddle tables
 * of every built FFT size and the bin sums live in one file-scope device
 * array.  Host code never passes the array's name to a kernel or a copy
 * (on the host it is a stand-in, not a device address): the address of
 * each device's copy is taken once, at context creation on that device, and
 * kept per device.  Calls that overlap on one device share the array and
 * race; each call clears the bins it uses before the deposit. */
#define PW_TW_MAX 5632   /* float2 twiddles of all built sizes (5362) */
#define PW_NBIN_MAX 1774 /* nint(2048/2 * sqrt(3)): bins of the largest mesh */
#define PW_SCRATCH_DOUBLES (PW_TW_MAX + 3 * (PW_NBIN_MAX + 1))
#define PW_MAX_DEV 64

static __device__ __align__(256) double scratch[PW_SCRATCH_DOUBLES];

static std::mutex g_scratch_mu;
static double *g_scratch[PW_MAX_DEV];  /* device address of scratch, per device */
static int g_tw_off[2049];             /* float2 offset of size n's twiddles */

/* Once per device, with the device current: find scratch's address and
   write the twiddles of every built size into it. */
int cube_power_scratch_setup(int device) {
  if (device < 0 || device >= PW_MAX_DEV) return CUBE_ERR_INVALID;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch[device]) return CUBE_OK;
  double *ptr = nullptr;
  if (hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return CUBE_ERR_HIP;
  float2 h[2048];
  int off = 0;
  for (int n = 1; n <= 2048; ++n) {
    if (!cube_fft_supported(n)) continue;
    if (off + n > PW_TW_MAX) return CUBE_ERR_INVALID;
    cube_fft_twiddles(n, h);
    if (hipMemcpy(reinterpret_cast<float2 *>(ptr) + off, h, n * sizeof(float2), hipMemcpyHostToDevice) != hipSuccess)
      return CUBE_ERR_HIP;
    g_tw_off[n] = off;
    off += n;
  }
  g_scratch[device] = ptr;
  return CUBE_OK;
}

extern "C" int cube_power_noalloc(cube_ctx *c, int32_t ng, int32_t nbin, double *ksum, double *psum,
                                  int64_t *count) {
  if (c) c->pm_ahead = 0;
  int st = power_args(c, ng, nbin, ksum, psum, count);
  if (st) return st;
  if (nbin > PW_NBIN_MAX || ng > 2048) return CUBE_ERR_INVALID; /* beyond the scratch array */
  double *ptr;
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    ptr = (c->device >= 0 && c->device < PW_MAX_DEV) ? g_scratch[c->device] : nullptr;
  }
  if (!ptr) return CUBE_ERR_STATE; /* set up by cube_ctx_create on this device */
  CUBE_CHECK(hipSetDevice(c->device));
  float2 *tw = reinterpret_cast<float2 *>(ptr) + g_tw_off[ng];
  double *bins = ptr + PW_TW_MAX;
  st = power_device(c, ng, nbin, tw, bins);
  /* bins 1..nbin straight into the caller's arrays (the counts are
     unsigned 64-bit, the same bits as int64 below 2^63) */
  if (!st && (hipMemcpyAsync(ksum, bins + 1, nbin * sizeof(double), hipMemcpyDeviceToHost, c->stream) != hipSuccess ||
              hipMemcpyAsync(psum, bins + (nbin + 1) + 1, nbin * sizeof(double), hipMemcpyDeviceToHost,
                             c->stream) != hipSuccess ||
              hipMemcpyAsync(count, bins + 2 * (nbin + 1) + 1, nbin * sizeof(int64_t), hipMemcpyDeviceToHost,
                             c->stream) != hipSuccess))
    st = CUBE_ERR_HIP;
  if (hipStreamSynchronize(c->stream) != hipSuccess && !st) st = CUBE_ERR_HIP;
  return st;
}
