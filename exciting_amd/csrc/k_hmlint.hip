// Muffin-tin Hamiltonian and overlap integrals of one SCF iteration, the producers of the
// setup's h_a (hmlint.f90:33-34 = mt_kin.f90 + mt_pot.f90; ValenceRelativity 'none',
// spinless) and of oalo / ololo (olprad.f90:90-125).
//
// Every radial integral of the reference is fderiv(-1) of a product on the species' mesh:
// the cubic spline of the product integrated interval by interval (fderiv.f90:64-72).  That
// functional is linear in the sampled values, so it is a fixed weight vector per mesh,
//     int f = sum_r wt_r f_r,
// computed on the host by the spline's recurrences (spline.f90:46-96) transposed.  On the device:
//  * hml_radial_kernel, one workgroup per (atom, q): for q < lmmaxvr the potential integrals
//    P_q(a, b) = sum_r wt_r r^2 V_q(r) u_a u_b (mt_pot.f90:142-212), q = lmmaxvr the kinetic
//    ones K(a, b) = sum_r wt_r (1/2 u_a' u_b' r^2 + 1/2 l(l+1) u_a u_b) for l_a = l_b
//    (mt_kin.f90:120-167), q = lmmaxvr + 1 the overlaps S(a, b) = sum_r wt_r r^2 u_a u_b
//    (olprad.f90:94-125); functions a: APW (l, io) io fastest for l <= lmaxmat, then lo;
//  * hml_assemble_kernel, one thread per matrix element:
//      h(f1, f3) = sum_lm2 G(lm1, lm2, lm3) P_lm2(a1, a3) + [lm1 = lm3] K(a1, a3)
//    with G the Gaunt coefficient int conj(Y_lm1) R_lm2 Y_lm3 (gauntyry.f90, nonzero only for
//    m2 = +-(m1 - m3)), stored per (lm1, lm3) as [l2][sign of m2]; rows and columns in the
//    setup's order (APW (l, m, io) io fastest, lo (ilo, m) m fastest); and oalo, ololo from S.
// And the reverse, the muffin-tin density from a density matrix (genrhomt.f90:34-150):
//  * rho_factor_kernel: F_lm2(a, b) = w sum_{m1, m3} Re(dm(f1, f3) conj(G(lm1, lm2, lm3)))
//    (w = 2 for APW-lo pairs, the lo-APW block then 0), one thread per (atom, a, b, l2);
//  * rho_radial_kernel: rho_lm2(r) = sum_{a, b} F_lm2(a, b) u_a(r) u_b(r), one thread per
//    (atom, lm2, r), on the radial functions of the last hmlint call.
#include <math.h>

#include <vector>

#include "exc_common.h"

namespace {

constexpr int kHT = 256;

__device__ __forceinline__ int isqrt_lm(int lm) {
  int l = (int)sqrt((double)lm);
  while (l * l > lm) --l;
  while ((l + 1) * (l + 1) <= lm) ++l;
  return l;
}

struct HmlArgs {
  int natm, ao, lmaxapw, lmaxmat, naf, nf, nlomax, lmv, nrmtmax, naa, maxnlo;
  const int *spidx, *nrmt, *nlorb, *lorbl;   // lorbl[is * nlomax + ilo]
  const double *wt, *spr, *apwfr, *lofr, *veffmt;
  double *rad;                                // [natm][lmv + 2][nf][nf]
  const cplx *gnt;                            // [lmmaxmat][lmmaxmat][lmaxvr + 1][2]
  const lo_desc *lod;
  const int *dm_lo;                           // [natm][2]: first lo, count
  cplx *haa, *loa, *lolo;
  double *oalo, *ololo;
  const cplx *dm;                             // genrhomt: dm(ws, ws, natm)
  int ws;
  double *rho;                                // genrhomt: rhomt(lmv, nrmtmax, natm)
};

__device__ __forceinline__ const double *radial_u(const HmlArgs &A, int atom, int a, int *l) {
  if (a < A.naf) {
    const int io = a % A.ao, la = a / A.ao;
    *l = la;
    return A.apwfr + (size_t)A.nrmtmax * 2 * (io + (size_t)A.ao * (la + (size_t)(A.lmaxapw + 1) * atom));
  }
  const int ilo = a - A.naf, is = A.spidx[atom];
  if (ilo >= A.nlorb[is]) return nullptr;
  *l = A.lorbl[is * A.nlomax + ilo];
  return A.lofr + (size_t)A.nrmtmax * 2 * (ilo + (size_t)A.nlomax * atom);
}

// 16 x 16 tiles of the pairs (a, b) on the matrix cores, r split over the waves: 8 atoms, 26 functions, 500
// points, lmaxvr 6 230 -> 54 us (a thread per pair, each walking the mesh before)
static_assert(kHT == 256, "four waves");
__global__ __launch_bounds__(kHT) void hml_radial_kernel(HmlArgs A) {
  const int q = blockIdx.x, atom = blockIdx.y;
  const int is = A.spidx[atom], nr = A.nrmt[is];
  extern __shared__ double sw[];   // [nr] weights of this block's integrand
  __shared__ double red[2][4][4][64];
  const double *wt = A.wt + (size_t)A.nrmtmax * is, *x = A.spr + (size_t)A.nrmtmax * is;
  for (int r = threadIdx.x; r < nr; r += kHT) {
    const double r2 = x[r] * x[r];
    double v;
    if (q < A.lmv) v = wt[r] * r2 * A.veffmt[q + (size_t)A.lmv * (r + (size_t)A.nrmtmax * atom)];
    else if (q == A.lmv) v = wt[r];          // kinetic: the r^2 and l(l+1) factors per pair
    else v = wt[r] * r2;
    sw[r] = v;
  }
  __syncthreads();
  double *out = A.rad + ((size_t)atom * (A.lmv + 2) + q) * A.nf * A.nf;
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int per = (nr + 15) / 16 * 4, rb = wave * per, re = min(nr, rb + per);
  // blocks of 32 x 32 pairs, I <= J: (2 I + i, 2 J + j) tiles of 16 functions, the one below the
  // diagonal of a diagonal block left out
  const int nblk = (A.nf + 31) / 32;
  for (int I = 0; I < nblk; ++I)
    for (int J = I; J < nblk; ++J) {
      const bool diag = I == J;
      const double *u[4];                                // functions 32 I + 16 t + li, then 32 J + ..., where there are
      bool has[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        int l;
        const int f = 32 * (t < 2 ? I : J) + 16 * (t & 1) + li;
        u[t] = f < A.nf ? radial_u(A, atom, f, &l) : nullptr;
        has[t] = u[t];
        if (!has[t]) u[t] = A.apwfr;
      }
      // sums over this wave's r of weight u_a u_b, ofs 0: the functions, nrmtmax: their derivatives
      // with 1/2 r^2
      d4_t acc[2][4];
      auto product = [&](d4_t *s, int ofs) {
#pragma unroll
        for (int k = 0; k < 4; ++k) s[k] = d4_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll 8
        for (int r0 = rb; r0 < re; r0 += 4) {
          const int r = min(r0 + lg, nr - 1);
          const bool in = r0 + lg < re;
          double w = sw[r], y[4];
          if (ofs) w *= 0.5 * (x[r] * x[r]);
#pragma unroll
          for (int t = 0; t < 4; ++t) y[t] = t < 2 || !diag ? u[t][r + ofs] : y[t - 2];
#pragma unroll
          for (int t = 0; t < 4; ++t) y[t] = in && has[t] ? y[t] : 0.0;
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
              if (i <= j || !diag)
                s[2 * i + j] = __builtin_amdgcn_mfma_f64_16x16x4f64(in ? w * y[i] : 0.0, y[2 + j], s[2 * i + j], 0, 0, 0);
        }
      };
      product(acc[0], 0);
      if (q == A.lmv) product(acc[1], A.nrmtmax);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        __syncthreads();                                 // the last tile's sums are read
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          red[0][v][wave][lane] = acc[0][k][v];
          if (q == A.lmv) red[1][v][wave][lane] = acc[1][k][v];
        }
        __syncthreads();
        // element 4 wave + lg of the rows, li of the columns; the lower triangle is the upper's mirror
        const int a = 32 * I + 16 * (k >> 1) + 4 * wave + lg, b = 32 * J + 16 * (k & 1) + li;
        if (a <= b && b < A.nf) {
          double f = 0.0;
#pragma unroll
          for (int w = 0; w < 4; ++w) f += red[0][wave][w][lane];
          if (q == A.lmv) {
            double g = 0.0;
            int la = 0, lb = 0;
#pragma unroll
            for (int w = 0; w < 4; ++w) g += red[1][wave][w][lane];
            radial_u(A, atom, a, &la);
            radial_u(A, atom, b, &lb);
            f = la == lb ? fma(0.5 * la * (la + 1), f, g) : 0.0;
          }
          out[a * A.nf + b] = f;
          out[b * A.nf + a] = f;
        }
      }
    }
}

// the Gaunt sum + kinetic term of one element; a1, a3 radial function indices
__device__ cplx hml_element(const HmlArgs &A, int atom, int l1, int m1, int a1, int l3, int m3, int a3) {
  const int lmm = (A.lmaxmat + 1) * (A.lmaxmat + 1), lmaxvr = isqrt_lm(A.lmv - 1);
  const int lm1 = l1 * l1 + l1 + m1, lm3 = l3 * l3 + l3 + m3;
  const cplx *g = A.gnt + ((size_t)lm1 * lmm + lm3) * (lmaxvr + 1) * 2;
  const double *P = A.rad + (size_t)atom * (A.lmv + 2) * A.nf * A.nf;
  const size_t ab = (size_t)a1 * A.nf + a3, qs = (size_t)A.nf * A.nf;
  const int d = m1 > m3 ? m1 - m3 : m3 - m1;
  cplx z = {0.0, 0.0};
  for (int l2 = d; l2 <= lmaxvr; ++l2) {
    const double pp = P[(size_t)(l2 * l2 + l2 + d) * qs + ab], pm = P[(size_t)(l2 * l2 + l2 - d) * qs + ab];
    const cplx gp = g[2 * l2], gm = g[2 * l2 + 1];
    z.re = fma(gp.re, pp, fma(gm.re, pm, z.re));
    z.im = fma(gp.im, pp, fma(gm.im, pm, z.im));
  }
  if (lm1 == lm3) z.re += P[(size_t)A.lmv * qs + ab];
  return z;
}

__global__ __launch_bounds__(kHT) void hml_assemble_kernel(HmlArgs A) {
  const int atom = blockIdx.y;
  const size_t e = (size_t)blockIdx.x * kHT + threadIdx.x;
  const size_t n_aa = (size_t)A.naa * A.naa, n_la = (size_t)A.maxnlo * A.naa, n_ll = (size_t)A.maxnlo * A.maxnlo;
  const size_t n_oa = (size_t)A.ao * A.nlomax, n_oo = (size_t)A.nlomax * A.nlomax;
  const int first = A.dm_lo[2 * atom], cnt = A.dm_lo[2 * atom + 1];
  auto apw = [&](int f, int *l, int *m, int *a) {
    const int io = f % A.ao, lm = f / A.ao;
    *l = isqrt_lm(lm);
    *m = lm - *l * *l - *l;
    *a = io + A.ao * *l;
  };
  if (e < n_aa) {
    const int f1 = (int)(e % A.naa), f3 = (int)(e / A.naa);
    int l1, m1, a1, l3, m3, a3;
    apw(f1, &l1, &m1, &a1);
    apw(f3, &l3, &m3, &a3);
    A.haa[(size_t)atom * n_aa + e] = hml_element(A, atom, l1, m1, a1, l3, m3, a3);
    return;
  }
  size_t i = e - n_aa;
  if (i < n_la) {
    const int r = (int)(i % A.maxnlo), f3 = (int)(i / A.maxnlo);
    cplx z = {0.0, 0.0};
    if (r < cnt) {
      const lo_desc q = A.lod[first + r];
      int l3, m3, a3;
      apw(f3, &l3, &m3, &a3);
      z = hml_element(A, atom, q.l, q.m, A.naf + q.ilo, l3, m3, a3);
    }
    A.loa[(size_t)atom * n_la + i] = z;
    return;
  }
  i -= n_la;
  if (i < n_ll) {
    const int r1 = (int)(i % A.maxnlo), r3 = (int)(i / A.maxnlo);
    cplx z = {0.0, 0.0};
    if (r1 < cnt && r3 < cnt) {
      const lo_desc q1 = A.lod[first + r1], q3 = A.lod[first + r3];
      z = hml_element(A, atom, q1.l, q1.m, A.naf + q1.ilo, q3.l, q3.m, A.naf + q3.ilo);
    }
    A.lolo[(size_t)atom * n_ll + i] = z;
    return;
  }
  i -= n_ll;
  const double *S = A.rad + ((size_t)atom * (A.lmv + 2) + A.lmv + 1) * A.nf * A.nf;
  const int is = A.spidx[atom];
  if (i < n_oa) {
    const int io = (int)(i % A.ao), ilo = (int)(i / A.ao);
    double v = 0.0;
    if (ilo < A.nlorb[is]) v = S[(size_t)(io + A.ao * A.lorbl[is * A.nlomax + ilo]) * A.nf + A.naf + ilo];
    A.oalo[(size_t)atom * n_oa + i] = v;
    return;
  }
  i -= n_oa;
  if (i < n_oo) {
    const int i1 = (int)(i % A.nlomax), i2 = (int)(i / A.nlomax);
    double v = 0.0;
    if (i1 < A.nlorb[is] && i2 < A.nlorb[is] && A.lorbl[is * A.nlomax + i1] == A.lorbl[is * A.nlomax + i2])
      v = S[(size_t)(A.naf + i1) * A.nf + A.naf + i2];
    A.ololo[(size_t)atom * n_oo + i] = v;
  }
}

// row of function a's m = -l in the density matrix: APW (l, io) at apwordmax l^2 + io (2l+1)
// (rows (l, io, m) m fastest, gendmatmt.f90:92-101), lo ilo after maxaa (ilo, m)
__device__ __forceinline__ int dm_row(const HmlArgs &A, int atom, int a) {
  if (a < A.naf) {
    const int io = a % A.ao, l = a / A.ao;
    return A.ao * l * l + io * (2 * l + 1);
  }
  const int is = A.spidx[atom];
  int r = A.naa;
  for (int i = 0; i < a - A.naf; ++i) r += 2 * A.lorbl[is * A.nlomax + i] + 1;
  return r;
}

constexpr int kMaxL2 = 16;   // lmaxvr supported by genrhomt

// F[atom][lm2][a][b] = w sum_{m1, m3} Re(dm(f1, f3) conj(G(lm1, lm2, lm3))) for the l2 of this
// thread (genrhomt.f90:60-71, 96-107, 131-142; w = 2 for APW-lo, the lo-APW block is 0)
__global__ __launch_bounds__(kHT) void rho_factor_kernel(HmlArgs A) {
  const int atom = blockIdx.y, L2 = isqrt_lm(A.lmv - 1) + 1;
  const int t = blockIdx.x * kHT + threadIdx.x;
  if (t >= A.nf * A.nf * L2) return;
  const int l2 = t % L2, ab = t / L2, a = ab / A.nf, b = ab % A.nf;
  const int lmm = (A.lmaxmat + 1) * (A.lmaxmat + 1);
  double *F = A.rad + (size_t)atom * A.lmv * A.nf * A.nf + (size_t)a * A.nf + b;
  const size_t qs = (size_t)A.nf * A.nf;
  double acc[2 * kMaxL2 + 1];
  for (int i = 0; i <= 2 * l2; ++i) acc[i] = 0.0;
  int la = 0, lb = 0;
  const double *ua = radial_u(A, atom, a, &la), *ub = radial_u(A, atom, b, &lb);
  if (ua && ub && !(a >= A.naf && b < A.naf)) {
    const double w = (a < A.naf && b >= A.naf) ? 2.0 : 1.0;
    const int o1 = dm_row(A, atom, a), o3 = dm_row(A, atom, b);
    const cplx *dm = A.dm + (size_t)atom * A.ws * A.ws;
    for (int m1 = -la; m1 <= la; ++m1)
      for (int m3 = -lb; m3 <= lb; ++m3) {
        const int d = m1 > m3 ? m1 - m3 : m3 - m1;
        if (d > l2) continue;
        const cplx z = dm[(o1 + m1 + la) + (size_t)A.ws * (o3 + m3 + lb)];
        const cplx *g = A.gnt + (((size_t)(la * la + la + m1) * lmm + (lb * lb + lb + m3)) * L2 + l2) * 2;
        acc[l2 + d] = fma(z.re, g[0].re, fma(z.im, g[0].im, acc[l2 + d]));
        if (d > 0) acc[l2 - d] = fma(z.re, g[1].re, fma(z.im, g[1].im, acc[l2 - d]));
      }
    for (int i = 0; i <= 2 * l2; ++i) acc[i] *= w;
  }
  for (int m2 = -l2; m2 <= l2; ++m2) F[(size_t)(l2 * l2 + l2 + m2) * qs] = acc[l2 + m2];
}

// rhomt(lm2, r, atom) = sum_{a, b} F[atom][lm2][a][b] u_a(r) u_b(r) (genrhomt.f90:72-77)
__global__ __launch_bounds__(kHT) void rho_radial_kernel(HmlArgs A) {
  const int r = blockIdx.x * kHT + threadIdx.x, lm2 = blockIdx.y, atom = blockIdx.z;
  if (r >= A.nrmtmax) return;
  const int nr = A.nrmt[A.spidx[atom]];
  double s = 0.0;
  if (r < nr) {
    const double *F = A.rad + ((size_t)atom * A.lmv + lm2) * A.nf * A.nf;
    for (int a = 0; a < A.nf; ++a) {
      int la;
      const double *ua = radial_u(A, atom, a, &la);
      if (!ua) continue;
      const double va = ua[r];
      double t = 0.0;
      for (int b = 0; b < A.nf; ++b) {
        int lb;
        const double *ub = radial_u(A, atom, b, &lb);
        if (ub) t = fma(F[a * A.nf + b], ub[r], t);
      }
      s = fma(va, t, s);
    }
  }
  A.rho[lm2 + (size_t)A.lmv * (r + (size_t)A.nrmtmax * atom)] = s;
}

// ------------------------------------------------------------------ host helpers

long double lfact(int n) {
  long double f = 1.0L;
  for (int i = 2; i <= n; ++i) f *= i;
  return f;
}

// (j1 j2 j3; m1 m2 m3) by the Racah formula
double wigner3j(int j1, int j2, int j3, int m1, int m2, int m3) {
  if (m1 + m2 + m3 != 0 || abs(m1) > j1 || abs(m2) > j2 || abs(m3) > j3) return 0.0;
  if (j3 < abs(j1 - j2) || j3 > j1 + j2) return 0.0;
  const long double tri = lfact(j1 + j2 - j3) * lfact(j1 - j2 + j3) * lfact(-j1 + j2 + j3) / lfact(j1 + j2 + j3 + 1);
  const long double pre = tri * lfact(j1 + m1) * lfact(j1 - m1) * lfact(j2 + m2) * lfact(j2 - m2) * lfact(j3 + m3) *
                          lfact(j3 - m3);
  long double s = 0.0L;
  for (int k = 0; k <= j1 + j2 + j3; ++k) {
    const int d[6] = {k, j3 - j2 + k + m1, j3 - j1 + k - m2, j1 + j2 - j3 - k, j1 - k - m1, j2 - k + m2};
    bool ok = true;
    long double den = 1.0L;
    for (int v : d) {
      if (v < 0) {
        ok = false;
        break;
      }
      den *= lfact(v);
    }
    if (ok) s += ((k & 1) ? -1.0L : 1.0L) / den;
  }
  const long double sign = ((j1 - j2 - m3) & 1) ? -1.0L : 1.0L;
  return (double)(sign * sqrtl(pre) * s);
}

// int conj(Y_l1m1) Y_l2m2 Y_l3m3 dOmega
double gaunt_c(int l1, int l2, int l3, int m1, int m2, int m3) {
  if (m1 - m2 - m3 != 0 || ((l1 + l2 + l3) & 1)) return 0.0;
  const double t = sqrt((2.0 * l1 + 1.0) * (2.0 * l2 + 1.0) * (2.0 * l3 + 1.0) / (4.0 * M_PI));
  return ((m1 & 1) ? -t : t) * wigner3j(l1, l2, l3, 0, 0, 0) * wigner3j(l1, l2, l3, -m1, m2, m3);
}

// int conj(Y_l1m1) R_l2m2 Y_l3m3 dOmega, R_lm = sqrt2 Re Y_lm (m > 0), Y_l0, sqrt2 Im Y_lm (m < 0)
cplx gaunt_yry(int l1, int l2, int l3, int m1, int m2, int m3) {
  const double c1 = 0.70710678118654752440;
  if (m2 > 0) {
    const double t1 = (m2 % 2 == 0) ? 1.0 : -1.0;
    return {c1 * (gaunt_c(l1, l2, l3, m1, m2, m3) + t1 * gaunt_c(l1, l2, l3, m1, -m2, m3)), 0.0};
  }
  if (m2 < 0) {
    const double t1 = ((-m2) % 2 == 0) ? 1.0 : -1.0;
    return {0.0, -c1 * (gaunt_c(l1, l2, l3, m1, m2, m3) - t1 * gaunt_c(l1, l2, l3, m1, -m2, m3))};
  }
  return {gaunt_c(l1, l2, l3, m1, m2, m3), 0.0};
}

}  // namespace

// Integration weights of fderiv(-1) on the mesh x (n >= 4 points): the integral of the spline is
//   sum_i dx_i (f_i + f_{i+1}) / 2 - dx_i^3 / 12 (c2_i + c2_{i+1}),
// linear in f, so its weights are the transposed recurrences of spline.f90 run backwards from the
// coefficients of the c2: O(n).  (Run forwards on the n unit vectors, O(n^2), they took 0.5 ms of the
// host for each species of 500 points, before anything of an SCF iteration could be launched.)
void exc_hml_spline_weights(int n, const double *x, double *wt) {
  std::vector<double> w(n - 1), c2s(n), t2(n), g(n, 0.0), c1(n - 1, 0.0);
  for (int i = 0; i < n - 1; ++i) w[i] = 1.0 / (x[i + 1] - x[i]);
  // the elimination's factors: r_i = 3 (c1_i - c1_{i-1}) w_i - t2_i r_{i-1}, c2_i = c2s_i s_i,
  // s_i = r_i - c2s_{i+1} s_{i+1} (1 <= i < n - 1), s_0 = r_0, s_{n-1} = r_{n-1}
  c2s[0] = c2s[n - 1] = 1.0;
  double t1 = (x[1] - x[0]) * w[1];
  t2[1] = t1;
  c2s[1] = 1.0 / (2.0 * (t1 + 1.0));
  for (int i = 2; i < n - 1; ++i) {
    t1 = (x[i] - x[i - 1]) * w[i];
    t2[i] = t1 * c2s[i - 1];
    c2s[i] = 1.0 / (2.0 * t1 + 2.0 - t2[i]);
  }
  // derivatives of the integral: by the c2 (times c2s: by the s), then by the r
  for (int i = 0; i < n - 1; ++i) {
    const double dx = x[i + 1] - x[i], d = -dx * dx * dx / 12.0;
    g[i] += d;
    g[i + 1] += d;
  }
  for (int i = 0; i < n; ++i) g[i] *= c2s[i];
  for (int i = 1; i < n - 1; ++i) g[i + 1] -= c2s[i + 1] * g[i];
  // by the c1 (first differences of f times w)
  const double ge = g[n - 1] / (x[n - 1] - x[n - 3]);
  c1[n - 2] += ge;
  c1[n - 3] -= ge;
  for (int i = n - 2; i >= 1; --i) {
    const double d = 3.0 * w[i] * g[i];
    c1[i] += d;
    c1[i - 1] -= d;
    g[i - 1] -= t2[i] * g[i];
  }
  const double gb = g[0] / (x[2] - x[0]);
  c1[1] += gb;
  c1[0] -= gb;
  for (int i = 0; i < n; ++i) wt[i] = 0.0;
  for (int i = 0; i < n - 1; ++i) {
    const double half = 0.5 * (x[i + 1] - x[i]), d = w[i] * c1[i];
    wt[i] += half - d;
    wt[i + 1] += half + d;
  }
}

// G[((lm1 * lmmaxmat + lm3) * (lmaxvr + 1) + l2) * 2 + s] = gauntyry(l1, l2, l3, m1, m2, m3)
// with m2 = +d (s = 0) and m2 = -d (s = 1, zero when d = 0), d = |m1 - m3|
void exc_hml_gaunt_table(int lmaxmat, int lmaxvr, cplx *g) {
  const int lmm = (lmaxmat + 1) * (lmaxmat + 1);
  for (int l1 = 0; l1 <= lmaxmat; ++l1)
    for (int m1 = -l1; m1 <= l1; ++m1)
      for (int l3 = 0; l3 <= lmaxmat; ++l3)
        for (int m3 = -l3; m3 <= l3; ++m3) {
          const int lm1 = l1 * l1 + l1 + m1, lm3 = l3 * l3 + l3 + m3, d = abs(m1 - m3);
          cplx *o = g + ((size_t)lm1 * lmm + lm3) * (lmaxvr + 1) * 2;
          for (int l2 = 0; l2 <= lmaxvr; ++l2) {
            o[2 * l2] = o[2 * l2 + 1] = {0.0, 0.0};
            if (d > l2) continue;
            o[2 * l2] = gaunt_yry(l1, l2, l3, m1, d, m3);
            if (d > 0) o[2 * l2 + 1] = gaunt_yry(l1, l2, l3, m1, -d, m3);
          }
        }
}

namespace {
HmlArgs hml_args(const exc_dev &d, int lmv, int nrmtmax, const int *nrmt, const int *nlorb, const int *lorbl,
                 const double *wt, const double *spr, const double *apwfr, const double *lofr, const double *veffmt,
                 double *rad, const cplx *gnt) {
  HmlArgs A;
  A.natm = d.natm;
  A.ao = d.apwordmax;
  A.lmaxapw = d.lmaxapw;
  A.lmaxmat = d.lmaxmat;
  A.naf = d.apwordmax * (d.lmaxmat + 1);
  A.nlomax = d.nlomax > 0 ? d.nlomax : 0;
  A.nf = A.naf + A.nlomax;
  A.lmv = lmv;
  A.nrmtmax = nrmtmax;
  A.naa = d.naa;
  A.maxnlo = d.maxnlo;
  A.spidx = d.spidx;
  A.nrmt = nrmt;
  A.nlorb = nlorb;
  A.lorbl = lorbl;
  A.wt = wt;
  A.spr = spr;
  A.apwfr = apwfr;
  A.lofr = lofr;
  A.veffmt = veffmt;
  A.rad = rad;
  A.gnt = gnt;
  A.lod = d.lod;
  A.dm_lo = d.dm_lo;
  A.haa = d.haa;
  A.loa = d.loa;
  A.lolo = d.lolo;
  A.oalo = d.oalo;
  A.ololo = d.ololo;
  A.dm = nullptr;
  A.ws = 0;
  A.rho = nullptr;
  return A;
}
}  // namespace

int exc_launch_hmlint(const exc_dev &d, int lmv, int nrmtmax, const int *nrmt, const int *nlorb, const int *lorbl,
                      const double *wt, const double *spr, const double *apwfr, const double *lofr,
                      const double *veffmt, double *rad, const cplx *gnt, hipStream_t s) {
  HmlArgs A = hml_args(d, lmv, nrmtmax, nrmt, nlorb, lorbl, wt, spr, apwfr, lofr, veffmt, rad, gnt);
  if (d.natm > 65535 || lmv + 2 > 65535) return EXC_ERR_ARG;
  if ((size_t)nrmtmax * sizeof(double) > 64 * 1024) return EXC_ERR_ARG;
  hipLaunchKernelGGL(hml_radial_kernel, dim3(lmv + 2, d.natm), dim3(kHT), nrmtmax * sizeof(double), s, A);
  EXC_CHECK(hipGetLastError());
  const size_t n = (size_t)d.naa * d.naa + (size_t)d.maxnlo * d.naa + (size_t)d.maxnlo * d.maxnlo +
                   (size_t)A.ao * A.nlomax + (size_t)A.nlomax * A.nlomax;
  hipLaunchKernelGGL(hml_assemble_kernel, dim3((unsigned)((n + kHT - 1) / kHT), d.natm), dim3(kHT), 0, s, A);
  EXC_CHECK(hipGetLastError());
  return EXC_OK;
}

int exc_launch_genrhomt(const exc_dev &d, int lmv, int nrmtmax, const int *nrmt, const int *nlorb, const int *lorbl,
                        const double *apwfr, const double *lofr, const cplx *gnt, const cplx *dm, int ws, double *fbuf,
                        double *rhomt, hipStream_t s) {
  HmlArgs A = hml_args(d, lmv, nrmtmax, nrmt, nlorb, lorbl, nullptr, nullptr, apwfr, lofr, nullptr, fbuf, gnt);
  A.dm = dm;
  A.ws = ws;
  A.rho = rhomt;
  const int L2 = (int)lround(sqrt((double)lmv));
  if (L2 - 1 > kMaxL2 || d.natm > 65535 || lmv > 65535 || ws < d.naa + A.maxnlo) return EXC_ERR_ARG;
  const size_t nt = (size_t)A.nf * A.nf * L2;
  hipLaunchKernelGGL(rho_factor_kernel, dim3((unsigned)((nt + kHT - 1) / kHT), d.natm), dim3(kHT), 0, s, A);
  EXC_CHECK(hipGetLastError());
  hipLaunchKernelGGL(rho_radial_kernel, dim3((nrmtmax + kHT - 1) / kHT, lmv, d.natm), dim3(kHT), 0, s, A);
  EXC_CHECK(hipGetLastError());
  return EXC_OK;
}
