// Muffin-tin density of the direct route, rhovalk (rhovalk.f90:99-207, spinless; C holds the
// states' coefficients): per atom a and coarse radial point irc (mesh point ir = irc lradstep),
//   psi_j(lm)  = sum_io W(a, io, lm; j) u_{io,l}(ir) + sum_ilo C(lo(a, ilo, m); j) v_ilo(ir)
//                (wavefmt.f90:91-124; W = A^T C, the zdotu of apwalm with the coefficients),
//   rfmt(itp)  = sum_j w occ_j |sum_lm zbshtvr(itp, lm) psi_j(lm)|^2   (|w occ_j| > epsocc),
//   rhomt(:, ir, a) += rfshtvr rfmt                                 (rhovalk.f90:183-207).
// The transform is linear, so the sum over states factors through the radial functions
// f = (io, l <= lmaxvr) and the atom's local orbitals (the same sampled-point density, summed
// in another order):
//   P(itp, f, j) = sum_m zbshtvr(itp, lm(l_f, m)) coef_f(m, j)     coef: W rows or lo rows of C
//   z(itp, ir, j) = sum_f u_f(ir) P(itp, f, j)
//   rfmt(itp, ir) = sum_j t_j |z|^2 = sum_{f <= f'} u_f(ir) u_f'(ir) R(itp, f, f'),
//   R = (2 - delta_ff') Re sum_j t_j P(itp, f, j) conj(P(itp, f', j)),   t_j = w occ_j,
// with t_j = 0 for |w occ_j| <= epsocc.  Three kernels: rv_p (P), rv_q (R), rv_r (rfmt from R
// and u, then rfshtvr).  Flops per k-point 8 lmmaxvr (2 lmaxvr + 1) nf nst + 4 lmmaxvr nf^2 nst
// per atom and 2 lmmaxvr nf^2 + 2 lmmaxvr^2 per atom and mesh point, nf = apwordmax (lmaxvr + 1) +
// nlomax, instead of 8 lmmaxvr^2 per atom, mesh point and state.
//
// All three sums run on the FP64 matrix cores: they are a few GFLOP in many short products, so
// latency bounds them, and a 16 x 16 tile per wave with its operands straight from L2 (P is
// written and read with the states contiguous) leaves few loads in a row.  8 atoms, lmaxvr 8, 200
// states, 500 mesh points: rv_p 39 -> 16 us, rv_q 40 -> 16, rv_r 78 -> 24 (a thread per
// element with LDS operands before).
#include "exc_common.h"

namespace {

constexpr int kRvThreads = 256;
constexpr int kRvMaxF = 31;      // radial functions of an atom
constexpr int kRvMaxV = 81;      // lmmaxvr, lmaxvr <= 8
constexpr int kRvSteps = 5;      // groups of 4 of the 2 l + 1 <= 17 orders m

struct RvArgs {
  int lmv, lmaxvr, lradstep, nrmtmax, nlomax, lmaxapw, ao, naa, ldw, ngp, ldv, nst, nf, npair;
  const int *nrmt, *nlorb, *lorbl;   // per species; lorbl[ilo + nlomax is]
  const double *apwfr, *lofr;        // (nrmtmax, 2, ao, 0:lmaxapw, natm), (nrmtmax, 2, nlomax, natm)
  const cplx *w;                     // W(a naa + io + ao lm, j), leading dimension ldw
  const cplx *evec;                  // C(ldv, nst)
  const double *occ;
  double wk, eps;
  const cplx *zb;                    // zbshtvr(itp, lm), lmv x lmv column-major
  const double *rf;                  // rfshtvr(lm, itp), lmv x lmv column-major
  cplx *p;                           // P[((a lmv + itp) nf + f) nst + j]
  double *r;                         // R[(a npair + pair) lmv + itp], pairs f <= f' row by row
  double *rhomt;                     // (lmv, nrmtmax, natm)
};

// l of radial function f of species is (-1: none, an lo of another l range or beyond nlorb)
__device__ __forceinline__ int rv_fun_l(const RvArgs &p, int is, int f) {
  const int nfa = p.ao * (p.lmaxvr + 1);
  if (f < nfa) return f / p.ao;
  const int ilo = f - nfa;
  if (ilo >= p.nlorb[is]) return -1;
  const int l = p.lorbl[ilo + p.nlomax * is];
  return l <= p.lmaxvr ? l : -1;
}

__device__ __forceinline__ d4_t rv_mfma(double a, double b, d4_t c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// P for 16 points x 16 states of one atom: the radial functions of one l are a product of
// zbshtvr's 2 l + 1 columns with the coefficients; the waves share the l (a nearly equal number
// of orders m each) and the local orbitals
__global__ __launch_bounds__(kRvThreads) void rv_p_kernel(exc_dev d, RvArgs p) {
  const int j0 = 16 * blockIdx.x, i0 = 16 * blockIdx.y, a = blockIdx.z;
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int is = d.spidx[a], lmv = p.lmv, nfa = p.ao * (p.lmaxvr + 1);
  const int itp = min(i0 + li, lmv - 1), jc = min(j0 + li, p.nst - 1);
  // functions f0, f0 + 1 (the second if two) of angular momentum l, coefficient of order m at
  // c[m cs], the second's next to it
  auto put = [&](int f, const d4_t &re, const d4_t &im) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int i = i0 + 4 * v + lg;
      if (i < lmv && j0 + li < p.nst)
        p.p[(((size_t)a * lmv + i) * p.nf + f) * p.nst + j0 + li] = cplx{re[v], im[v]};
    }
  };
  auto fun = [&](int f0, bool two, int l, const cplx *c, int cs) {
    const int nm = 2 * l + 1;
    const cplx *zb = p.zb + itp + (size_t)lmv * (l * l);
    cplx z[kRvSteps], x[kRvSteps], y[kRvSteps];
#pragma unroll
    for (int g = 0; g < kRvSteps; ++g)
      if (4 * g < nm) {
        const int m = min(4 * g + lg, nm - 1);
        z[g] = zb[(size_t)lmv * m];
        x[g] = c[(size_t)cs * m];
        y[g] = c[(size_t)cs * m + (two ? 1 : 0)];
      }
    d4_t xr = {0.0, 0.0, 0.0, 0.0}, xi = xr, yr = xr, yi = xr;
#pragma unroll
    for (int g = 0; g < kRvSteps; ++g)
      if (4 * g < nm) {
        if (4 * g + lg >= nm) z[g] = x[g] = y[g] = cplx{0.0, 0.0};   // repeated orders
        xr = rv_mfma(z[g].re, x[g].re, xr);
        xi = rv_mfma(z[g].re, x[g].im, xi);
        xr = rv_mfma(-z[g].im, x[g].im, xr);
        xi = rv_mfma(z[g].im, x[g].re, xi);
        if (two) {
          yr = rv_mfma(z[g].re, y[g].re, yr);
          yi = rv_mfma(z[g].re, y[g].im, yi);
          yr = rv_mfma(-z[g].im, y[g].im, yr);
          yi = rv_mfma(z[g].im, y[g].re, yi);
        }
      }
    put(f0, xr, xi);
    if (two) put(f0 + 1, yr, yi);
  };
  const cplx *w = p.w + (size_t)p.ldw * jc + (size_t)a * p.naa;
  for (int t = 0; t <= p.lmaxvr; ++t) {
    if (((t & 7) < 4 ? (t & 7) : 7 - (t & 7)) != wave) continue;
    const int l = p.lmaxvr - t;
    for (int io = 0; io < p.ao; io += 2) fun(p.ao * l + io, io + 1 < p.ao, l, w + io + p.ao * (l * l), p.ao);
  }
  // the atom's lo rows: (ilo, m), m fastest (genidxlo order)
  const cplx *lo = p.evec + (size_t)p.ldv * jc + p.ngp + d.dm_lo[2 * a];
  int off = 0;
  for (int f = nfa; f < p.nf; ++f) {
    const int l = rv_fun_l(p, is, f);
    if ((f - nfa) % 4 == wave) {
      if (l >= 0) {
        fun(f, false, l, lo + off, 1);
      } else {
        const d4_t zero = {0.0, 0.0, 0.0, 0.0};
        put(f, zero, zero);
      }
    }
    if (f - nfa < p.nlorb[is]) off += 2 * p.lorbl[f - nfa + p.nlomax * is] + 1;
  }
}

// R of one point and atom: the pairs of functions as up to three 16 x 16 tiles (f <= f'), the
// real and imaginary parts of 4 states a k-step each, the states split over the waves
template <int TF>
__global__ __launch_bounds__(kRvThreads) void rv_q_kernel(RvArgs p) {
  constexpr int NT = TF * (TF + 1) / 2, U = 4;
  __shared__ double red[NT * 4][4][64];
  const int itp = blockIdx.x, a = blockIdx.y, nf = p.nf;
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const cplx *pa = p.p + ((size_t)a * p.lmv + itp) * nf * p.nst;
  const int ng = (p.nst + 3) / 4;
  double sum[NT][4] = {};
  for (int g0 = wave; g0 < ng; g0 += 4 * U) {
    cplx x[U][TF];
    double oc[U];
    d4_t acc[NT];                                      // of these 16 states: short sums, as chunks round less
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = d4_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = min(4 * (g0 + 4 * u) + lg, p.nst - 1);
      oc[u] = p.occ[j];
#pragma unroll
      for (int t = 0; t < TF; ++t) x[u][t] = pa[(size_t)min(16 * t + li, nf - 1) * p.nst + j];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool in = 4 * (g0 + 4 * u) + lg < p.nst;
      const double t1 = p.wk * oc[u], tw = in && fabs(t1) > p.eps ? t1 : 0.0;   // rhovalk.f90:101-102
#pragma unroll
      for (int t = 0; t < TF; ++t)
        if (!in) x[u][t] = cplx{0.0, 0.0};
#pragma unroll
      for (int t = 0, k = 0; t < TF; ++t)
#pragma unroll
        for (int q = t; q < TF; ++q, ++k) {
          acc[k] = rv_mfma(tw * x[u][t].re, x[u][q].re, acc[k]);
          acc[k] = rv_mfma(tw * x[u][t].im, x[u][q].im, acc[k]);
        }
    }
#pragma unroll
    for (int k = 0; k < NT; ++k)
#pragma unroll
      for (int v = 0; v < 4; ++v) sum[k][v] += acc[k][v];
  }
#pragma unroll
  for (int k = 0; k < NT; ++k)
#pragma unroll
    for (int v = 0; v < 4; ++v) red[4 * k + v][wave][lane] = sum[k][v];
  __syncthreads();
#pragma unroll
  for (int m = 0; m < NT; ++m) {
    const int e = wave * NT + m, k = e >> 2;   // tiles in the order (0, 0), (0, 1), (1, 1)
    const int f = 16 * (k == 2 ? 1 : 0) + 4 * (e & 3) + lg, g = 16 * (k > 0 ? 1 : 0) + li;
    if (f > g || g >= nf) continue;
    const double s = (red[e][0][lane] + red[e][1][lane]) + (red[e][2][lane] + red[e][3][lane]);
    const int q = f * nf - f * (f - 1) / 2 + g - f;
    p.r[((size_t)a * p.npair + q) * p.lmv + itp] = (f == g ? 1.0 : 2.0) * s;
  }
}

// 16 mesh points of one atom: rfmt = (u_f u_f') R over the pairs, then rfmt rfshtvr^T; a wave takes
// every fourth tile of 16 harmonics
__global__ __launch_bounds__(kRvThreads) void rv_r_kernel(exc_dev d, RvArgs p) {
  constexpr int NV = (kRvMaxV + 15) / 16, NW = (NV + 3) / 4, U = 4;
  __shared__ double us[kRvMaxF][17];
  __shared__ unsigned char pf[kRvMaxF * (kRvMaxF + 1) / 2], pg[kRvMaxF * (kRvMaxF + 1) / 2];
  __shared__ double rfm[kRvMaxV][17];
  const int a = blockIdx.y, nf = p.nf, lmv = p.lmv;
  const int is = d.spidx[a], nr = p.nrmt[is];
  const int irc0 = blockIdx.x * 16;
  if (irc0 * p.lradstep >= nr) return;   // uniform over the workgroup
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nfa = p.ao * (p.lmaxvr + 1);
  for (int e = threadIdx.x; e < 16 * nf; e += kRvThreads) {
    const int f = e >> 4, r = e & 15, ir = (irc0 + r) * p.lradstep;
    double u = 0.0;
    if (ir < nr && rv_fun_l(p, is, f) >= 0)
      u = f < nfa ? p.apwfr[ir + (size_t)p.nrmtmax * 2 * ((f % p.ao) + (size_t)p.ao * (f / p.ao + (size_t)(p.lmaxapw + 1) * a))]
                  : p.lofr[ir + (size_t)p.nrmtmax * 2 * ((f - nfa) + (size_t)p.nlomax * a)];
    us[f][r] = u;
  }
  for (int e = threadIdx.x; e < nf * nf; e += kRvThreads) {
    const int f = e / nf, g = e - f * nf;
    if (f > g) continue;
    const int q = f * nf - f * (f - 1) / 2 + g - f;
    pf[q] = (unsigned char)f;
    pg[q] = (unsigned char)g;
  }
  __syncthreads();
  const int nv = (lmv + 15) / 16;
  int vc[NW];   // this lane's column in each tile of this wave
#pragma unroll
  for (int w = 0; w < NW; ++w) vc[w] = min(16 * (wave + 4 * w) + li, lmv - 1);
  const d4_t zero = {0.0, 0.0, 0.0, 0.0};
  d4_t sum[NW], acc[NW];   // the sum and that of 16 of its terms (chunks round less)
#pragma unroll
  for (int w = 0; w < NW; ++w) sum[w] = zero;
  if (wave < nv) {
    const double *ra = p.r + (size_t)a * p.npair * lmv;
    for (int q0 = 0; q0 < p.npair; q0 += 4 * U) {
      double b[U][NW];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int q = min(q0 + 4 * u + lg, p.npair - 1);
#pragma unroll
        for (int w = 0; w < NW; ++w) b[u][w] = ra[(size_t)q * lmv + vc[w]];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int q = min(q0 + 4 * u + lg, p.npair - 1);
        const bool in = q0 + 4 * u + lg < p.npair;
        const double x = in ? us[pf[q]][li] * us[pg[q]][li] : 0.0;
#pragma unroll
        for (int w = 0; w < NW; ++w) acc[w] = rv_mfma(x, in ? b[u][w] : 0.0, u == 0 ? zero : acc[w]);
      }
#pragma unroll
      for (int w = 0; w < NW; ++w) sum[w] += acc[w];
    }
#pragma unroll
    for (int w = 0; w < NW; ++w)
      if (16 * (wave + 4 * w) + li < lmv)
#pragma unroll
        for (int v = 0; v < 4; ++v) rfm[16 * (wave + 4 * w) + li][4 * v + lg] = sum[w][v];
  }
  __syncthreads();
  if (wave >= nv) return;
  // rhomt(:, ir, a) += rfshtvr rfmt(:, ir)   (rhovalk.f90:183-207)
#pragma unroll
  for (int w = 0; w < NW; ++w) sum[w] = zero;
  for (int q0 = 0; q0 < lmv; q0 += 4 * U) {
    double b[U][NW];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int q = min(q0 + 4 * u + lg, lmv - 1);
#pragma unroll
      for (int w = 0; w < NW; ++w) b[u][w] = p.rf[vc[w] + (size_t)lmv * q];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int q = min(q0 + 4 * u + lg, lmv - 1);
      const bool in = q0 + 4 * u + lg < lmv;
      const double x = in ? rfm[q][li] : 0.0;
#pragma unroll
      for (int w = 0; w < NW; ++w) acc[w] = rv_mfma(x, in ? b[u][w] : 0.0, u == 0 ? zero : acc[w]);
    }
#pragma unroll
    for (int w = 0; w < NW; ++w) sum[w] += acc[w];
  }
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const int lm = 16 * (wave + 4 * w) + li;
    if (lm >= lmv) continue;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int ir = (irc0 + 4 * v + lg) * p.lradstep;
      if (ir < nr) p.rhomt[lm + (size_t)lmv * (ir + (size_t)p.nrmtmax * a)] += sum[w][v];
    }
  }
}

}  // namespace

size_t exc_rhovalk_work_bytes(const exc_dev &d, int lmaxvr, int nlomax, int nst) {
  const size_t lmv = (size_t)(lmaxvr + 1) * (lmaxvr + 1);
  const size_t nf = (size_t)d.apwordmax * (lmaxvr + 1) + (nlomax > 0 ? nlomax : 0);
  const size_t np = nf * (nf + 1) / 2;
  return ((sizeof(cplx) * d.natm * lmv * nst * nf + 255) & ~(size_t)255) + sizeof(double) * d.natm * np * lmv;
}

int exc_launch_rhovalk(const exc_dev &d, int lmaxvr, int lradstep, int nrmtmax, int nlomax, const int *nrmt,
                       const int *nlorb, const int *lorbl, const double *apwfr, const double *lofr, const cplx *w,
                       int ldw, int ngp, const cplx *evec, int ldv, int nst, const double *occ, double wk,
                       double eps, const cplx *zb, const double *rf, void *work, double *rhomt, hipStream_t s) {
  const int lmv = (lmaxvr + 1) * (lmaxvr + 1);
  if (nst <= 0) return EXC_OK;
  const int nl = nlomax > 0 ? nlomax : 0;
  RvArgs p;
  p.nf = d.apwordmax * (lmaxvr + 1) + nl;
  p.npair = p.nf * (p.nf + 1) / 2;
  if (lmaxvr > 8 || d.apwordmax > 4 || nl > 8 || p.nf > kRvMaxF || lradstep < 1 || d.natm > 65535 ||
      nst > 65535)
    return EXC_ERR_ARG;
  p.lmv = lmv;
  p.lmaxvr = lmaxvr;
  p.lradstep = lradstep;
  p.nrmtmax = nrmtmax;
  p.nlomax = nlomax > 0 ? nlomax : 1;
  p.lmaxapw = d.lmaxapw;
  p.ao = d.apwordmax;
  p.naa = d.naa;
  p.ldw = ldw;
  p.ngp = ngp;
  p.ldv = ldv;
  p.nst = nst;
  p.nrmt = nrmt;
  p.nlorb = nlorb;
  p.lorbl = lorbl;
  p.apwfr = apwfr;
  p.lofr = lofr;
  p.w = w;
  p.evec = evec;
  p.occ = occ;
  p.wk = wk;
  p.eps = eps;
  p.zb = zb;
  p.rf = rf;
  p.p = (cplx *)work;
  p.r = (double *)((char *)work + ((sizeof(cplx) * d.natm * (size_t)lmv * nst * p.nf + 255) & ~(size_t)255));
  p.rhomt = rhomt;
  hipLaunchKernelGGL(rv_p_kernel, dim3((nst + 15) / 16, (lmv + 15) / 16, d.natm), dim3(kRvThreads), 0, s, d, p);
  EXC_CHECK(hipGetLastError());
  if (p.nf <= 16)
    hipLaunchKernelGGL(rv_q_kernel<1>, dim3(lmv, d.natm), dim3(kRvThreads), 0, s, p);
  else
    hipLaunchKernelGGL(rv_q_kernel<2>, dim3(lmv, d.natm), dim3(kRvThreads), 0, s, p);
  EXC_CHECK(hipGetLastError());
  const int nrc = (nrmtmax + lradstep - 1) / lradstep;
  hipLaunchKernelGGL(rv_r_kernel, dim3((nrc + 15) / 16, d.natm), dim3(kRvThreads), 0, s, d, p);
  EXC_CHECK(hipGetLastError());
  return EXC_OK;
}
