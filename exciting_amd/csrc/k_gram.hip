// The Gram form's table of the modular split (exc_setup_batched_dev, EXC_BATCH_SPLIT_CRT): per
// atom the extreme eigenvalues of h_a, which fix the shift sigma, and the lower Cholesky factor
// of h_a + sigma in the Y stage's summation order.  It is made again for every new h_a, once per
// SCF iteration, and everything after it waits.
//
// One workgroup of 8 or 16 waves per atom: the matrices (242 x 242 at lmax 10) are far too small to
// spread over the chip, and a library solve of the whole batch spends its time on the ~1000
// launches of its column steps and on eigenvectors nobody needs (8 atoms, naa 242: about 8 ms; here
// 1.8 ms for the extremes and 0.37 for the factor).  Bound by one CU's path to L2 and by the chain of barriers.
//  * gram_extremes_kernel: Householder tridiagonalization, then the smallest and the largest
//    eigenvalue by Sturm counts of 128 points each at a time.  A step reads the trailing matrix once for
//    its matrix-vector product, both triangles, so that every access runs along columns and no sum
//    crosses lanes; the rank-2 updates wait in LDS, corrected for in the products, and are applied 8 at a
//    time on the matrix cores (1.82 ms; 2.24 with each step's update applied in the next one's
//    pass, a read and a write of the matrix a step).
//  * gram_chol_kernel: left-looking by panels of 16 columns.
#include "reflector.h"
#include "wave_sum.h"

namespace {

constexpr int kCT = 512, kCW = kCT / 64;    // the Cholesky kernel: a row of the panel per lane in registers
constexpr int kNMax = 338;           // naa at lmax 12
constexpr int kNB = 16;              // Cholesky panel

// eigenvalues of the tridiagonal (d, e^2 in e2) below x.  The quotient may be a few ulp off (as
// if e^2 were): the reciprocal is refined twice from the hardware's estimate.
__device__ __forceinline__ int sturm(int n, const double *d, const double *e2, double pivmin, double x) {
  int c = 0;
  double q = d[0] - x;
  if (fabs(q) < pivmin) q = -pivmin;
  c += q < 0.0;
  for (int i = 1; i < n; ++i) {
    double r = __builtin_amdgcn_rcp(q);
    r = fma(fma(-q, r, 1.0), r, r);
    r = fma(fma(-q, r, 1.0), r, r);
    q = fma(-e2[i - 1], r, d[i] - x);
    if (fabs(q) < pivmin) q = -pivmin;
    c += q < 0.0;
  }
  return c;
}

// R: 64-row chunks of n.  h: the upper triangles are read; m: n x n scratch per atom; ext[2 a]:
// the smallest and largest eigenvalue of atom a (NaN where h is not finite)
template <int R, int kGT = R <= 4 ? 1024 : 512, int NB = R <= 4 ? 8 : 6>       // (the larger orders need the registers and LDS)
__global__ __launch_bounds__(kGT) void gram_extremes_kernel(int n, const cplx *__restrict__ h, cplx *__restrict__ m,
                                                            double *__restrict__ ext) {
  constexpr int kGW = kGT / 64;
  __shared__ cplx pv[NB][64 * R], pw[NB][64 * R];       // v, w of the panel: the matrix lacks their updates
  __shared__ cplx vn[64 * R];                           // v of this step
  __shared__ cplx red[kGW][64 * R];
  __shared__ cplx col[64 * R];                          // the next column, short of the panel's updates
  __shared__ double d[64 * R], e2[64 * R], buf[2][kGW];
  __shared__ cplx s_alpha, sab[2 * NB];                 // w_q^H v, then v_q^H v
  __shared__ int cnt[2][2];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const cplx *H = h + (size_t)n * n * blockIdx.x;
  cplx *M = m + (size_t)n * n * blockIdx.x;
  for (int k = wave; k < n; k += kGW)
    for (int i = lane; i < n; i += 64) {
      const cplx a = i <= k ? H[i + (size_t)n * k] : H[k + (size_t)n * i];
      const cplx x = i < k ? a : i > k ? cplx{a.re, -a.im} : cplx{a.re, 0.0};
      M[i + (size_t)n * k] = x;
      if (k == 0) col[i] = x;
    }
  __syncthreads();
  int p = 0;                                            // steps since the last update of the matrix
  for (int j = 0; j < n - 1; ++j) {
    // column j with the panel's updates, and its Householder vector (thread i: row i)
    cplx x = {0.0, 0.0};
    if (tid >= j && tid < n) {
      x = col[tid];
#pragma unroll 2
      for (int q = 0; q < p; ++q) {
        const cplx v = pv[q][tid], w = pw[q][tid], vj = pv[q][j], wj = pw[q][j];
        x.re -= v.re * wj.re + v.im * wj.im + w.re * vj.re + w.im * vj.im;
        x.im -= v.im * wj.re - v.re * wj.im + w.im * vj.re - w.re * vj.im;
      }
    }
    if (wave < R) {                                     // the waves that hold rows
      if (tid == j) d[j] = x.re;
      if (tid == j + 1) s_alpha = x;
      const double t = wave_sum(tid > j + 1 ? x.re * x.re + x.im * x.im : 0.0);
      if (lane == 0) buf[0][wave] = t;
    }
    __syncthreads();
    cplx tau = {0.0, 0.0};
    if (wave < R) {                                     // (the others would only take turns at the FP64 units)
      double xn2 = 0.0;
#pragma unroll
      for (int w = 0; w < R; ++w) xn2 += buf[0][w];
      const cplx al = s_alpha;
      double rf[5];                                     // (a column below 1e-145 counts as zero)
      reflector(al.re, al.im, xn2, rf);
      tau = cplx{rf[1], rf[2]};
      const cplx sc = {rf[3], rf[4]};
      const double beta = rf[0];
      if (tid == 0) e2[j] = beta * beta;
      vn[tid] = tid == j + 1 ? cplx{1.0, 0.0} : (tid > j + 1 && tid < n) ? cmul(x, sc) : cplx{0.0, 0.0};
    }
    __syncthreads();
    // this wave's columns' share of A v
    cplx acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = cplx{0.0, 0.0};
#pragma unroll 4
    for (int k = j + 1 + wave; k < n; k += kGW) {
      const cplx v = vn[k];
      const cplx *cl = M + (size_t)n * k;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int i = lane + 64 * r;
        if (64 * r + 63 <= j || i >= n) continue;       // rows above the trailing matrix: whole chunks skipped
        const cplx a = cl[i];
        if (k == j + 1) col[i] = a;                     // wave 0's first column: the next step's
        acc[r].re = fma(a.re, v.re, fma(-a.im, v.im, acc[r].re));
        acc[r].im = fma(a.re, v.im, fma(a.im, v.re, acc[r].im));
      }
    }
    // the panel's products with v, one a wave
    for (int t = wave; t < 2 * p; t += kGW) {
      const cplx *b = t < p ? pw[t] : pv[t - p];
      cplx s = {0.0, 0.0};
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const cplx y = b[lane + 64 * r], v = vn[lane + 64 * r];
        s.re += y.re * v.re + y.im * v.im;
        s.im += y.re * v.im - y.im * v.re;
      }
      s = cplx{wave_sum(s.re), wave_sum(s.im)};
      if (lane == 0) sab[t] = s;
    }
    double vav = 0.0;                                   // this wave's share of v^H A v (real)
#pragma unroll
    for (int r = 0; r < R; ++r) {
      red[wave][lane + 64 * r] = acc[r];
      const cplx v = vn[lane + 64 * r];
      vav += v.re * acc[r].re + v.im * acc[r].im;
    }
    vav = wave_sum(vav);
    if (lane == 0) buf[1][wave] = vav;
    __syncthreads();
    // z = A v less the panel's updates of A, w = tau z - 1/2 |tau|^2 (v^H z) v
    if (tid < 64 * R) {
      cplx w = {0.0, 0.0}, v = {0.0, 0.0};
      if (tid > j && tid < n) {
        v = vn[tid];
        cplx z = {0.0, 0.0};
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < kGW; ++q) {
          z.re += red[q][tid].re;
          z.im += red[q][tid].im;
          s += buf[1][q];
        }
#pragma unroll 2
        for (int q = 0; q < p; ++q) {
          const cplx a = sab[q], b = sab[p + q], x = pv[q][tid], y = pw[q][tid];
          z.re -= x.re * a.re - x.im * a.im + y.re * b.re - y.im * b.im;
          z.im -= x.re * a.im + x.im * a.re + y.re * b.im + y.im * b.re;
          s -= 2.0 * (a.re * b.re + a.im * b.im);
        }
        const double hk = -0.5 * (tau.re * tau.re + tau.im * tau.im) * s;
        w = cmul(tau, z);
        w = cplx{fma(hk, v.re, w.re), fma(hk, v.im, w.im)};
      }
      pv[p][tid] = v;
      pw[p][tid] = w;
    }
    __syncthreads();
    if (++p < NB) continue;
    // A -= V W^H + W V^H below and right of (j, j): the 16 x 16 tiles on and below the diagonal dealt to
    // the waves, their conjugates stored above it
    p = 0;
    const int li = lane & 15, lg = lane >> 4, t0 = (j + 1) / 16, nt = (n + 15) / 16 - t0;
    for (int tile = wave; tile < nt * (nt + 1) / 2; tile += kGW) {
      int ti = (int)((sqrtf(8.0f * tile + 1.0f) - 1.0f) * 0.5f);   // ti >= tk, row by row
      ti += (ti + 1) * (ti + 2) / 2 <= tile;
      ti -= ti * (ti + 1) / 2 > tile;
      const int tk = tile - ti * (ti + 1) / 2, k0 = 16 * (t0 + tk), i = 16 * (t0 + ti) + li;
      cplx a[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) a[v] = M[min(i, n - 1) + (size_t)n * min(k0 + 4 * v + lg, n - 1)];
      d4_t re = {0.0, 0.0, 0.0, 0.0}, im = re;
#pragma unroll
      for (int q0 = 0; q0 < NB; q0 += 4) {
        const int q = min(q0 + lg, NB - 1);
        const bool in = q0 + lg < NB;
        auto mac = [&](cplx y, cplx x) {                // + x conj(y)
          if (!in) x = y = cplx{0.0, 0.0};
          re = __builtin_amdgcn_mfma_f64_16x16x4f64(y.re, x.re, re, 0, 0, 0);
          im = __builtin_amdgcn_mfma_f64_16x16x4f64(y.re, x.im, im, 0, 0, 0);
          re = __builtin_amdgcn_mfma_f64_16x16x4f64(y.im, x.im, re, 0, 0, 0);
          im = __builtin_amdgcn_mfma_f64_16x16x4f64(-y.im, x.re, im, 0, 0, 0);
        };
        mac(pw[q][k0 + li], pv[q][i]);
        mac(pv[q][k0 + li], pw[q][i]);
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int k = k0 + 4 * v + lg;
        if (i <= j || k <= j || i >= n || k >= n) continue;
        const cplx x = {a[v].re - re[v], a[v].im - im[v]};
        M[i + (size_t)n * k] = x;
        if (k == j + 1) col[i] = x;
        if (ti > tk) M[k + (size_t)n * i] = cplx{x.re, -x.im};
      }
    }
    __syncthreads();
  }
  const int j = n - 1;
  if (tid == 0) {
    double x = col[j].re;
    for (int q = 0; q < p; ++q) x -= 2.0 * (pv[q][j].re * pw[q][j].re + pv[q][j].im * pw[q][j].im);
    d[j] = x;
  }
  __syncthreads();
  // bounds (Gershgorin), and whether all is finite; 4 waves from here on
  if (wave >= 4) return;
  double bound = 0.0, emax2 = 0.0;
  for (int i = lane; i < n; i += 64) {
    const double l2 = i > 0 ? e2[i - 1] : 0.0, r2 = i < n - 1 ? e2[i] : 0.0;
    const double g = fabs(d[i]) + sqrt(l2) + sqrt(r2);
    bound = g > bound || !(g == g) ? g : bound;
    emax2 = fmax(emax2, r2);
  }
  bool fin = bound < 1e300;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    bound = fmax(bound, __shfl_xor(bound, o));
    emax2 = fmax(emax2, __shfl_xor(emax2, o));
  }
  if (!__all(fin)) {                                    // NaN and infinities end here (every wave alike)
    if (tid < 2) ext[2 * blockIdx.x + tid] = __builtin_nan("");
    return;
  }
  bound = bound * (1.0 + 1e-14) + 1e-300;
  const double pivmin = fmax(1e-290, 2.3e-308 * emax2);
  // waves 0, 1 close in on the smallest, 2, 3 on the largest: each round keeps the one of 129
  // subintervals that holds it
  const int half = tid >> 7, t = tid & 127;
  double lo = -bound, hi = bound;
  for (int it = 0; it < 8; ++it) {                      // 129^8 > 2^56
    if (tid < 2) cnt[it & 1][tid] = 0;
    __syncthreads();
    const double x = lo + (hi - lo) * ((t + 1) * (1.0 / 129.0));
    const int c = sturm(n, d, e2, pivmin, x);
    const bool left = half ? c < n : c == 0;            // the eigenvalue is not below x
    const unsigned long long b = __ballot(left);
    if (lane == 0) atomicAdd(&cnt[it & 1][half], __popcll(b));
    __syncthreads();
    const int k = cnt[it & 1][half];                    // it lies in subinterval k
    const double w = hi - lo;
    hi = k < 128 ? lo + w * ((k + 1) * (1.0 / 129.0)) : hi;
    lo = k > 0 ? lo + w * (k * (1.0 / 129.0)) : lo;
  }
  if (t == 0) ext[2 * blockIdx.x + half] = 0.5 * (lo + hi);
}

// sigma from every atom's extremes (the caller's formula), NaN if any is not finite
__device__ __forceinline__ double gram_shift(int natm, const double *ext) {
  double lmin = 0.0, lmax = 0.0;
  for (int a = 0; a < natm; ++a) {
    const double x = ext[2 * a], y = ext[2 * a + 1];
    if (!(x == x) || !(y == y)) return __builtin_nan("");
    lmin = fmin(lmin, fmin(x, y));
    lmax = fmax(lmax, fmax(fabs(x), fabs(y)));
  }
  return (lmin < 0.0 ? -lmin * (1.0 + 1e-6) : 0.0) + 1e-10 * lmax;
}

// lane q's value of v in every lane
__device__ __forceinline__ double lane_of(double v, int q) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, q), hi = __builtin_amdgcn_readlane((int)(b >> 32), q);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// L L^H = P (h + sigma) P^T per atom, P the order fperm; info[a] nonzero if it is not positive
// definite (or not finite).  Per panel: each wave forms 16 x 16 blocks of the panel less the
// finished columns' part (FP64 MFMA, operands from L2), one wave factors the diagonal block in
// registers, then a thread per row solves against it.
__global__ __launch_bounds__(kCT) void gram_chol_kernel(int n, int natm, const cplx *__restrict__ h,
                                                        const int *__restrict__ fperm, const double *__restrict__ ext,
                                                        cplx *__restrict__ lf, double *__restrict__ sig,
                                                        int *__restrict__ info) {
  __shared__ cplx pan[kNMax + 14][kNB + 1];          // the panel from its diagonal down (whole 16-row blocks)
  __shared__ cplx dg[kNB][kNB + 1];                  // the panel's diagonal block, factored
  __shared__ double rinv[kNB];
  __shared__ int fp[kNMax], bad;
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const cplx *H = h + (size_t)n * n * blockIdx.x;
  cplx *L = lf + (size_t)n * n * blockIdx.x;
  const double sigma = gram_shift(natm, ext);
  if (blockIdx.x == 0 && tid == 0) *sig = sigma;
  if (!(sigma == sigma)) {
    if (tid == 0) info[blockIdx.x] = 1;
    return;
  }
  for (int i = tid; i < n; i += kCT) fp[i] = fperm[i];
  if (tid == 0) bad = 0;
  __syncthreads();
  for (int c0 = 0; c0 < n; c0 += kNB) {
    const int nb = min(kNB, n - c0);
    for (int r0 = c0 + 16 * wave; r0 < n; r0 += 16 * kCW) {
      // the block of h + sigma: rows 4 v + lane / 16, column lane % 16, as the MFMA leaves its sums
      cplx a[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = r0 + 4 * v + lk, c = c0 + li;
        a[v] = cplx{0.0, 0.0};
        if (r < n && c < n) {
          a[v] = H[fp[r] + (size_t)n * fp[c]];
          if (r == c) a[v].re += sigma;
        }
      }
      d4_t re = {0.0, 0.0, 0.0, 0.0}, im = {0.0, 0.0, 0.0, 0.0};
      const cplx *pr = L + min(r0 + li, n - 1), *pc = L + min(c0 + li, n - 1);
      constexpr int U = 8;
      for (int k0 = 0; k0 < c0; k0 += 4 * U) {         // c0 is a multiple of 16: k-steps whole, groups not
        cplx x[U], y[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const size_t o = (size_t)n * min(k0 + 4 * u + lk, c0 - 1);
          x[u] = pr[o];
          y[u] = pc[o];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (k0 + 4 * u >= c0) break;
          re = __builtin_amdgcn_mfma_f64_16x16x4f64(x[u].re, y[u].re, re, 0, 0, 0);
          im = __builtin_amdgcn_mfma_f64_16x16x4f64(x[u].im, y[u].re, im, 0, 0, 0);
          re = __builtin_amdgcn_mfma_f64_16x16x4f64(x[u].im, y[u].im, re, 0, 0, 0);
          im = __builtin_amdgcn_mfma_f64_16x16x4f64(-x[u].re, y[u].im, im, 0, 0, 0);
        }
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) pan[r0 - c0 + 4 * v + lk][li] = cplx{a[v].re - re[v], a[v].im - im[v]};
    }
    __syncthreads();
    if (wave == 0) {                                 // factor the diagonal block: lane = row, its 16 columns in registers
      cplx x[kNB];
#pragma unroll
      for (int c = 0; c < kNB; ++c) x[c] = pan[li][c];
      bool ok = true;
#pragma unroll
      for (int c = 0; c < kNB; ++c) {
        if (c < nb && ok) {
          const double p = lane_of(x[c].re, c);
          ok = p > 0.0;                              // uniform
          const double s = sqrt(p), si = 1.0 / s;
          if (lane == c) rinv[c] = si;
          x[c] = li == c ? cplx{s, 0.0} : cplx{x[c].re * si, x[c].im * si};
          __builtin_amdgcn_sched_barrier(0);         // column by column: hoisted broadcasts would spill
#pragma unroll
          for (int q = c + 1; q < kNB; ++q) {
            const double br = lane_of(x[c].re, q), bi = lane_of(x[c].im, q);
            x[q].re -= x[c].re * br + x[c].im * bi;
            x[q].im -= x[c].im * br - x[c].re * bi;
          }
        }
      }
      if (lane < kNB)
#pragma unroll
        for (int c = 0; c < kNB; ++c) dg[lane][c] = x[c];
      if (lane == 0 && !ok) bad = 1;
    }
    __syncthreads();
    if (bad) break;                                  // uniform
    for (int r = c0 + tid; r < n; r += kCT) {
      cplx x[kNB];
      if (r < c0 + kNB) {
#pragma unroll
        for (int c = 0; c < kNB; ++c) x[c] = c <= r - c0 ? dg[r - c0][c] : cplx{0.0, 0.0};
      } else {
#pragma unroll
        for (int c = 0; c < kNB; ++c) x[c] = pan[r - c0][c];   // nb = 16: rows follow the panel
#pragma unroll
        for (int c = 0; c < kNB; ++c) {
          __builtin_amdgcn_sched_barrier(0);
          x[c] = cplx{x[c].re * rinv[c], x[c].im * rinv[c]};
#pragma unroll
          for (int q = c + 1; q < kNB; ++q) {
            const cplx b = dg[q][c];
            x[q].re -= x[c].re * b.re + x[c].im * b.im;
            x[q].im -= x[c].im * b.re - x[c].re * b.im;
          }
        }
      }
#pragma unroll
      for (int c = 0; c < kNB; ++c)
        if (c < nb) L[r + (size_t)n * (c0 + c)] = x[c];
    }
    __syncthreads();
  }
  if (tid == 0) info[blockIdx.x] = bad;
}

// T(r, fperm[kk]) = conj(L(kk, r)) for kk >= r and 0 above, L the lower Cholesky factor: the Y
// stage on T forms E = A_p conj(L), conj(E) E^T = conj(A) (h + sigma) A^T, and the sum of a
// column tile starting at r0 may start at position r0 of the order
__global__ __launch_bounds__(256) void gram_tri_kernel(int naa, const cplx *__restrict__ L,
                                                       const int *__restrict__ fperm, cplx *__restrict__ T) {
  const int r = blockIdx.x * 256 + threadIdx.x, kk = blockIdx.y, at = blockIdx.z;
  if (r >= naa) return;
  const size_t o = (size_t)at * naa * naa;
  cplx v = {0.0, 0.0};
  if (kk >= r) {
    const cplx l = L[o + kk + (size_t)naa * r];
    v = cplx{l.re, -l.im};
  }
  T[o + r + (size_t)naa * fperm[kk]] = v;
}

}  // namespace

// ext: 2 natm, info: natm, sig: 1 (device); scratch and T: naa x naa x natm
int exc_launch_gram(const exc_dev &d, cplx *scratch, cplx *T, double *ext, double *sig, int *info, hipStream_t s) {
  const int n = d.naa;
  if (n < 1 || n > kNMax) return EXC_ERR_UNSUPPORTED;
  const dim3 g(d.natm), b(1024), b5(512);
  switch ((n + 63) / 64) {
    case 1: hipLaunchKernelGGL(gram_extremes_kernel<1>, g, b, 0, s, n, d.haa, scratch, ext); break;
    case 2: hipLaunchKernelGGL(gram_extremes_kernel<2>, g, b, 0, s, n, d.haa, scratch, ext); break;
    case 3: hipLaunchKernelGGL(gram_extremes_kernel<3>, g, b, 0, s, n, d.haa, scratch, ext); break;
    case 4: hipLaunchKernelGGL(gram_extremes_kernel<4>, g, b, 0, s, n, d.haa, scratch, ext); break;
    case 5: hipLaunchKernelGGL(gram_extremes_kernel<5>, g, b5, 0, s, n, d.haa, scratch, ext); break;
    default: hipLaunchKernelGGL(gram_extremes_kernel<6>, g, b5, 0, s, n, d.haa, scratch, ext); break;
  }
  EXC_CHECK(hipGetLastError());
  hipLaunchKernelGGL(gram_chol_kernel, g, dim3(kCT), 0, s, n, d.natm, d.haa, d.fperm, ext, scratch, sig, info);
  EXC_CHECK(hipGetLastError());
  hipLaunchKernelGGL(gram_tri_kernel, dim3((n + 255) / 256, n, d.natm), dim3(256), 0, s, n, scratch, d.fperm, T);
  EXC_CHECK(hipGetLastError());
  return EXC_OK;
}
