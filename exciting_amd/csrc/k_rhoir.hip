// Interstitial density of the occupied states (genrhoir.f90:28-89) without a full FFT: a basis fills only a
// small part of the grid's frequencies (its G lie in a box of half the grid's edge, since the grid holds every
// G - G'), so psi is transformed one direction at a time over the frequencies in use, as products with
// the DFT matrices on the FP64 matrix cores, and |psi|^2 is summed over the states before anything is
// stored:
//  * rhoir_map: the basis functions by their position in the box of G, and the range of each component;
//  * rhoir_x: z(x, s3, s2) = sum_s1 exp(2 pi i x s1 / n1) c(s1, s2, s3), gathering c straight from the
//    eigenvector, for s2, s3 in their ranges;
//  * rhoir_yz: a wave holds one x and 16 values of y and walks over states: the sum over s2 comes out
//    of the matrix cores in just the registers that the sum over s3 takes as its operand, so nothing lies in
//    between; t |psi|^2 stays in registers until the last state.  8 waves share the DFT matrices in LDS;
//  * rhoir_sum adds the groups of states to rho, in order.
// Only z (a quarter of the grid) crosses memory, where a batched FFT clears, scatters, transforms in
// three or four passes and reads the whole grid of every state: bound by the FP64 matrix cores, 0.85 n^4 complex
// multiply-adds a state on an n^3 grid.  200 states, 27 x 30 x 30 points, per k-point: 190 us with the batched
// FFT, 55 here; 64 states of 45 x 45 x 48 points 212 -> 103 us, 20 of 15^3 27 -> 18.
#include <math.h>

#include <algorithm>

#include "exc_common.h"

namespace {

constexpr int kKMax = 16;            // k-points per launch
constexpr int kTMax = 5;             // 16-wide tiles of a grid's edge: the DFT matrices of 80 points fill 120 KB of LDS

struct RhoK {
  const int *igpig;
  const cplx *evec;
  const double *occ;
  double wk;
  int ngp, ldv;
};
struct RhoArgs {
  RhoK k[kKMax];
  const int *ivg;
  int lo[3], n[3], nst, i0, ni;      // items i0 .. i0 + ni - 1: state i % nst of k-point i / nst
  double eps, omega;
  const cplx *f[3];                  // F_d(x, s) = exp(2 pi i x (lo_d + s) / n_d), x fastest
  int *inv, *rng;                    // per k-point: function + 1 at each G of the box (0: none); least and largest position
  cplx *z;                           // per item: n1 n2 n3
  double *part;                      // per k-point and group of states: (y, z, x)
};

// t1 of item i, or 0 for a state that does not count (genrhoir.f90:48)
__device__ __forceinline__ double weight(const RhoArgs &p, int k, int j) {
  const double t1 = p.k[k].wk * p.k[k].occ[j];
  return fabs(t1) > p.eps ? t1 : 0.0;
}

__device__ __forceinline__ void mac(d4_t &re, d4_t &im, cplx a, cplx b) {
  re = __builtin_amdgcn_mfma_f64_16x16x4f64(a.re, b.re, re, 0, 0, 0);
  im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.re, b.im, im, 0, 0, 0);
  re = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.im, b.im, re, 0, 0, 0);
  im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.im, b.re, im, 0, 0, 0);
}

__global__ __launch_bounds__(256) void rhoir_clear_kernel(RhoArgs p) {
  const int i = blockIdx.x * 256 + threadIdx.x, k = blockIdx.y, n = p.n[0] * p.n[1] * p.n[2];
  if (i < n) p.inv[(size_t)k * n + i] = 0;
  if (i < 6) p.rng[6 * k + i] = i < 3 ? 0x7fffffff : -1;
}

// (the ranges by workgroups of 1024: atomics of every wave on the six words took 30 us at 26000 functions)
constexpr int kMap = 1024;
__global__ __launch_bounds__(kMap) void rhoir_map_kernel(RhoArgs p) {
  __shared__ int r[kMap / 64][6];
  const int i = blockIdx.x * kMap + threadIdx.x, k = blockIdx.y, n = p.n[0] * p.n[1] * p.n[2];
  const int g = i < p.k[k].ngp ? p.k[k].igpig[i] - 1 : -1;
  const bool in = g >= 0 && g < n;
  int s[3] = {0x7fffffff, 0x7fffffff, 0x7fffffff}, h[3] = {-1, -1, -1};
  if (in) {
#pragma unroll
    for (int q = 0; q < 3; ++q) s[q] = h[q] = p.ivg[3 * g + q] - p.lo[q];
    p.inv[(size_t)k * n + s[0] + p.n[0] * (s[1] + p.n[1] * s[2])] = i + 1;
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      s[q] = min(s[q], __shfl_xor(s[q], o));
      h[q] = max(h[q], __shfl_xor(h[q], o));
    }
    if ((threadIdx.x & 63) == 0) {
      r[threadIdx.x >> 6][q] = s[q];
      r[threadIdx.x >> 6][3 + q] = h[q];
    }
  }
  __syncthreads();
  if (threadIdx.x >= 6) return;
  const bool low = threadIdx.x < 3;
  int v = r[0][threadIdx.x];
#pragma unroll
  for (int w = 1; w < kMap / 64; ++w) v = low ? min(v, r[w][threadIdx.x]) : max(v, r[w][threadIdx.x]);
  if (low) atomicMin(p.rng + 6 * k + threadIdx.x, v);
  else atomicMax(p.rng + 6 * k + threadIdx.x, v);
}

// a wave: 16 columns (s2, s3) of one item, all x
template <int XT>
__global__ __launch_bounds__(256) void rhoir_x_kernel(RhoArgs p) {
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int it = p.i0 + blockIdx.y, k = it / p.nst, j = it % p.nst;
  const int *rng = p.rng + 6 * k;
  if (rng[3] < 0 || weight(p, k, j) == 0.0) return;
  const int n1 = p.n[0], n2 = p.n[1], n = n1 * n2 * p.n[2];
  const int m1 = rng[3] - rng[0] + 1, m2 = rng[4] - rng[1] + 1, mc = m2 * (rng[5] - rng[2] + 1);
  const int c0 = 16 * (4 * blockIdx.x + wave);
  if (c0 >= mc) return;
  const int c = min(c0 + li, mc - 1), s3 = c / m2, s2 = c - s3 * m2;
  const int *inv = p.inv + (size_t)k * n + rng[0] + n1 * (rng[1] + s2 + n2 * (rng[2] + s3));
  const cplx *ev = p.k[k].evec + (size_t)p.k[k].ldv * j;
  const cplx *f = p.f[0] + (size_t)n1 * rng[0];
  d4_t re[XT], im[XT];
#pragma unroll
  for (int t = 0; t < XT; ++t) re[t] = im[t] = d4_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
  for (int s0 = 0; s0 < m1; s0 += 4) {
    const int s = min(s0 + lg, m1 - 1), g = s0 + lg < m1 ? inv[s] : 0;
    cplx b = ev[max(g, 1) - 1];
    if (!g) b = cplx{0.0, 0.0};
#pragma unroll
    for (int t = 0; t < XT; ++t) mac(re[t], im[t], f[min(16 * t + li, n1 - 1) + (size_t)n1 * s], b);
  }
  if (c0 + li >= mc) return;
  cplx *z = p.z + (size_t)blockIdx.y * n + c0 + li;
#pragma unroll
  for (int t = 0; t < XT; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int x = 16 * t + 4 * v + lg;
      if (x < n1) z[(size_t)x * mc] = cplx{re[t][v], im[t][v]};
    }
}

// workgroup (x, 16 values of y, k-point kk and group of states); LDS: F2 then F3 as operand registers, 1 KB a
// k-step of 4
template <int ZT>
__global__ __launch_bounds__(512) void rhoir_yz_kernel(RhoArgs p, int k0, int groups) {
  extern __shared__ cplx lds[];
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n1 = p.n[0], n2 = p.n[1], n3 = p.n[2], n = n1 * n2 * n3;
  const int x = blockIdx.x, y0 = 16 * blockIdx.y, k = k0 + blockIdx.z / groups, grp = blockIdx.z % groups;
  const int *rng = p.rng + 6 * k;
  const bool any = rng[3] >= 0;
  const int m2 = any ? rng[4] - rng[1] + 1 : 0, m3 = any ? rng[5] - rng[2] + 1 : 0;
  const int ks2 = (m2 + 3) / 4, ks3 = (m3 + 15) / 16 * 4;
  cplx *f2 = lds, *f3 = lds + 64 * ks2;
  for (int q = wave; q < ks2 + ZT * ks3; q += 8) {
    const bool two = q < ks2;
    const int zt = two ? 0 : (q - ks2) / ks3, s = 4 * (two ? q : (q - ks2) % ks3) + lg;
    const int r = (two ? y0 : 16 * zt) + li, nr = two ? n2 : n3;
    const bool in = r < nr && s < (two ? m2 : m3);
    lds[64 * q + lane] = in ? (two ? p.f[1] : p.f[2])[r + (size_t)nr * (s + rng[two ? 1 : 2])] : cplx{0.0, 0.0};
  }
  __syncthreads();
  double acc[ZT][4];
#pragma unroll
  for (int t = 0; t < ZT; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[t][v] = 0.0;
  const int first = max(p.i0, k * p.nst), last = min(p.i0 + p.ni, (k + 1) * p.nst);
  if (any)
#pragma unroll 1
    for (int it = first + grp * 8 + wave; it < last; it += 8 * groups) {
      const double t1 = weight(p, k, it - k * p.nst);
      if (t1 == 0.0) continue;
      const double t2 = t1 / p.omega;
      const cplx *z = p.z + (size_t)(it - p.i0) * n + (size_t)x * (m2 * m3);
      d4_t re[ZT], im[ZT];
#pragma unroll
      for (int t = 0; t < ZT; ++t) re[t] = im[t] = d4_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
      for (int s0 = 0; s0 < m3; s0 += 16) {
        const bool row = s0 + li < m3;
        const cplx *zr = z + (size_t)min(s0 + li, m3 - 1) * m2;
        d4_t qr = {0.0, 0.0, 0.0, 0.0}, qi = qr;
#pragma unroll 4
        for (int q = 0; q < ks2; ++q) {
          cplx a = zr[min(4 * q + lg, m2 - 1)];
          if (!row || 4 * q + lg >= m2) a = cplx{0.0, 0.0};
          mac(qr, qi, a, f2[64 * q + lane]);
        }
#pragma unroll
        for (int v = 0; v < 4; ++v)          // row 4 v + lane / 16 of the product: the operand of k-step v
#pragma unroll
          for (int t = 0; t < ZT; ++t) mac(re[t], im[t], f3[64 * (t * ks3 + s0 / 4 + v) + lane], cplx{qr[v], qi[v]});
      }
#pragma unroll
      for (int t = 0; t < ZT; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[t][v] += t2 * (re[t][v] * re[t][v] + im[t][v] * im[t][v]);
    }
  // the 8 waves' sums, a z tile at a time
  __shared__ double red[8][256];
  double *out = p.part + (size_t)blockIdx.z * n + (size_t)x * n2 * n3;
#pragma unroll
  for (int t = 0; t < ZT; ++t) {
    __syncthreads();
#pragma unroll
    for (int v = 0; v < 4; ++v) red[wave][64 * v + lane] = acc[t][v];
    __syncthreads();
    if (threadIdx.x < 256) {
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < 8; ++w) s += red[w][threadIdx.x];
      const int zz = 16 * t + 4 * wave + lg, y = y0 + li;
      if (zz < n3 && y < n2) out[y + n2 * zz] = s;
    }
  }
}

__global__ __launch_bounds__(256) void rhoir_sum_kernel(int n1, int n2, int n3, int parts, const double *__restrict__ part,
                                                        double *__restrict__ rho) {
  const int i = blockIdx.x * 256 + threadIdx.x, n = n1 * n2 * n3;
  if (i >= n) return;
  double s = 0.0;
#pragma unroll 8
  for (int q = 0; q < parts; ++q) s += part[(size_t)q * n + i];
  const int y = i % n2, z = i / n2 % n3, x = i / (n2 * n3);
  rho[x + n1 * (y + n2 * z)] += s;
}

template <int T>
void launch_x(const RhoArgs &p, dim3 g, hipStream_t s) {
  hipLaunchKernelGGL(rhoir_x_kernel<T>, g, dim3(256), 0, s, p);
}
template <int T>
int launch_yz(const RhoArgs &p, dim3 g, size_t lds, int k0, int groups, hipStream_t s) {
  if (lds > 64 * 1024)
    EXC_CHECK(hipFuncSetAttribute((const void *)rhoir_yz_kernel<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(rhoir_yz_kernel<T>, g, dim3(512), lds, s, p, k0, groups);
  return EXC_OK;
}

// groups of states of nk k-points with ns states each: two workgroups a CU, each wave at least one state
int rho_groups(const int *n, int nk, int ns, int ncu) {
  const int wg = n[0] * ((n[1] + 15) / 16) * nk, most = (ns + 7) / 8, want = (2 * ncu + wg - 1) / wg;
  return want < most ? want : most;
}

}  // namespace

// whether the grid's edges fit (above, a batched FFT: the DFT matrices no longer fit in LDS)
bool exc_rhoir_fits(const exc_dev &d) {
  return d.box_n[0] <= 16 * kTMax && d.box_n[1] <= 16 * kTMax && d.box_n[2] <= 16 * kTMax;
}

// Whether the products beat the FFT for nst states of a basis of ngp functions.  A workgroup of
// rhoir_yz takes a state a wave: with a few states most of it idles behind its loads of the DFT matrices,
// where the FFT of one state is a short job.  In us, W the complex multiply-adds of a state in
// millions (edges padded to 16, the basis a ball in the box), G the points in millions: products
// about 23 + 1.4 W + 0.16 W nst, FFT 28 + 28 G nst; below W = 3 both are mostly launches.  Measured (products, FFT):
// 48^3 points, N = 5898, 1 state 33, 25, 8 states 40, 57; 60^3, 13335, 1 44, 26, 8 56, 62; 60^3, 2000, 1 31, 27, 8 35, 60;
// 72^3 (the most padding, and the FFT's best edge), 18688, 8 104, 83, 40 286, 285; 75^3, 26046, 1 88, 46, 8 119, 113, 40
// 316, 563; 18 x 75 x 75, 5840, 1 42, 28, 8 54, 59; below the line 18 x 18 x 75, 1347, 1 32, 23, 8 40, 32, 16 40, 43.
bool exc_rhoir_pays(const exc_dev &d, int ngp, int nst) {
  auto pad = [](int n) { return (n + 15) / 16 * 16.0; };
  const double n1 = d.box_n[0], n2 = d.box_n[1], n3 = d.box_n[2], g = n1 * n2 * n3;
  const double f = std::min(1.0, cbrt(ngp / (g * (M_PI / 6.0))));
  const int m1 = (int)ceil(f * n1), m2 = (int)ceil(f * n2), m3 = (int)ceil(f * n3);
  const double w = 1e-6 * (pad(d.box_n[0]) * m1 * m2 * m3 +
                           n1 * pad(d.box_n[1]) * (m2 * pad(m3) + pad(d.box_n[2]) * pad(m3)));
  return w < 3.0 || nst * (28e-6 * g - 0.16 * w) >= 1.4 * w - 5.0;
}

// the items (states of all k-points) that z holds at a time: 256 MB, or the 64 states that the batched FFT takes
static long rho_chunk(size_t n, long items) {
  const long c = std::max((long)((size_t(256) << 20) / (sizeof(cplx) * n)), 64l);
  return std::min(std::min(c, items), 65535l);
}

size_t exc_rhoir_work_bytes(const exc_dev &d, int nk, int nst, int ncu) {
  const size_t n = (size_t)d.box_n[0] * d.box_n[1] * d.box_n[2];
  const int kc = std::min(nk, kKMax);
  size_t groups = 0;                                  // (a chunk may hold part of a k-point: any count up to kc)
  for (int k = 1; k <= kc; ++k) groups = std::max(groups, (size_t)k * rho_groups(d.box_n, k, nst, ncu));
  return sizeof(cplx) * n * rho_chunk(n, (long)kc * nst) + 8 * n * groups + 4 * (n * kc + 1) + 24 * kKMax;
}

// n1^2 + n2^2 + n3^2 elements
void exc_rhoir_tables(const exc_dev &d, cplx *f) {
  for (int q = 0; q < 3; ++q) {
    const int n = d.box_n[q];
    for (int s = 0; s < n; ++s)
      for (int x = 0; x < n; ++x) {
        const long long e = (((long long)x * (d.box_lo[q] + s)) % n + n) % n;
        const long double a = 2.0L * 3.14159265358979323846264338327950288L * e / n;
        *f++ = cplx{(double)cosl(a), (double)sinl(a)};
      }
  }
}

// rho += the density of nst states of nk k-points (host arrays of device pointers)
int exc_launch_rhoir(const exc_dev &d, int nk, const int *ngp, const int *const *igpig, int nst, const int *ldv,
                     const double *const *evec, const double *const *occ, const double *wkpt, double eps, const cplx *tab,
                     void *work, double *rho, int ncu, hipStream_t s) {
  const int n1 = d.box_n[0], n2 = d.box_n[1], n3 = d.box_n[2];
  const size_t n = (size_t)n1 * n2 * n3;
  if (!exc_rhoir_fits(d) || n == 0) return EXC_ERR_ARG;
  const int XT = (n1 + 15) / 16, YT = (n2 + 15) / 16, ZT = (n3 + 15) / 16;
  const size_t lds = sizeof(cplx) * 64 * ((n2 + 3) / 4 + (size_t)ZT * 4 * ZT);
  for (int k0 = 0; k0 < nk; k0 += kKMax) {
    const int kc = std::min(kKMax, nk - k0);
    RhoArgs p = {};
    int maxngp = 0;
    for (int k = 0; k < kc; ++k) {
      p.k[k] = {igpig[k0 + k], (const cplx *)evec[k0 + k], occ[k0 + k], wkpt[k0 + k], ngp[k0 + k], ldv[k0 + k]};
      maxngp = std::max(maxngp, ngp[k0 + k]);
    }
    if (maxngp == 0) continue;
    p.ivg = d.ivg;
    for (int q = 0; q < 3; ++q) {
      p.lo[q] = d.box_lo[q];
      p.n[q] = d.box_n[q];
    }
    p.nst = nst;
    p.eps = eps;
    p.omega = d.omega;
    p.f[0] = tab;
    p.f[1] = tab + n1 * n1;
    p.f[2] = p.f[1] + n2 * n2;
    const long items = (long)kc * nst, chunk = rho_chunk(n, items);
    p.z = (cplx *)work;
    p.rng = (int *)(p.z + n * rho_chunk(n, (long)std::min(nk, kKMax) * nst));
    p.inv = p.rng + 6 * kKMax;
    p.part = (double *)(p.inv + ((size_t)std::min(nk, kKMax) * n + 1) / 2 * 2);
    hipLaunchKernelGGL(rhoir_clear_kernel, dim3((unsigned)((n + 255) / 256), kc), dim3(256), 0, s, p);
    EXC_CHECK(hipGetLastError());
    hipLaunchKernelGGL(rhoir_map_kernel, dim3((maxngp + kMap - 1) / kMap, kc), dim3(kMap), 0, s, p);
    EXC_CHECK(hipGetLastError());
    for (long i0 = 0; i0 < items; i0 += chunk) {
      p.i0 = (int)i0;
      p.ni = (int)std::min(chunk, items - i0);
      const dim3 gx((n2 * n3 + 63) / 64, p.ni);
      switch (XT) {
        case 1: launch_x<1>(p, gx, s); break;
        case 2: launch_x<2>(p, gx, s); break;
        case 3: launch_x<3>(p, gx, s); break;
        case 4: launch_x<4>(p, gx, s); break;
        default: launch_x<5>(p, gx, s); break;
      }
      EXC_CHECK(hipGetLastError());
      const int ka = (int)(i0 / nst), kb = (int)((i0 + p.ni - 1) / nst), ks = kb - ka + 1;
      const int groups = rho_groups(d.box_n, ks, std::min((long)nst, (long)p.ni), ncu);
      const dim3 g(n1, YT, ks * groups);
      int rc;
      switch (ZT) {
        case 1: rc = launch_yz<1>(p, g, lds, ka, groups, s); break;
        case 2: rc = launch_yz<2>(p, g, lds, ka, groups, s); break;
        case 3: rc = launch_yz<3>(p, g, lds, ka, groups, s); break;
        case 4: rc = launch_yz<4>(p, g, lds, ka, groups, s); break;
        default: rc = launch_yz<5>(p, g, lds, ka, groups, s); break;
      }
      if (rc) return rc;
      EXC_CHECK(hipGetLastError());
      hipLaunchKernelGGL(rhoir_sum_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n1, n2, n3, ks * groups,
                         p.part, rho);
      EXC_CHECK(hipGetLastError());
    }
  }
  return EXC_OK;
}
