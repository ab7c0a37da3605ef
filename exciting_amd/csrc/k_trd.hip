// Tridiagonal reduction C = Q T Q^H of a strided batch of Hermitian matrices (both triangles
// stored), with the reflectors, d, e and tau where zhetrd('U') leaves them: for column c = n-1 .. 1
// the reflector H = I - tau v v^H, v(c-1) = 1, zero below, annihilates A(0:c-2, c); v(0:c-2) is
// stored there, e(c-1) at A(c-1, c).
//
// The reduction is a chain of n columns, each a matrix-vector product with what is left: bound by
// the launches and load latencies of one column, then by reading the leading block (n^2/3 elements on
// average) once a column.  So a column is two launches for the whole batch, and everything that
// would need another (norms, the corrections' dot products, the scaling of v) is a small sum each
// workgroup repeats:
//  * trd_col: finishes the last column's w (w = tau z + hk v, z = A v less the panel's corrections,
//    hk = -1/2 |tau|^2 v^H z) for 64 rows, updates column c with the panel's V and W, and sums
//    its norm over those rows;
//  * trd_mv: beta, tau and the scale of v from the norm; then a wave for every two columns k of the
//    leading block: (A v)_k = sum_r conj(A(r, k)) v_r, lanes along the column, no sum across waves.
//    The panel's columns go the same way (W^H v, V^H v).
// Every kPanel columns trd_update applies V W^H + W V^H to both triangles of the rest (FP64 MFMA).
// 4 matrices, n = 1258: 17.7 ms (14 us a column); rocSOLVER's zhetrd_strided_batched about 35 (five launches and
// 27 us a column, 3.4 ms of updates).
#include "reflector.h"
#include "wave_sum.h"

namespace {

constexpr int kPanel = 32;

struct TrdArgs {
  int n;
  cplx *a;             // n x n at n n k
  cplx *v, *w;         // n x kPanel at n kPanel k
  cplx *x, *y;         // n; n + 2 kPanel
  double *part;        // norms of x, one per 64 rows: (n + 63) / 64
  double *vav;         // parts of v^H A v, one per workgroup of trd_mv: trd_groups(n, kPanel)
  double *d, *e;       // n each
  cplx *tau;           // n
};

// workgroups of trd_mv for column c with p panel columns before it: 8 columns each, and 256 rows of v; a
// multiple of 8, so that a column of A is read through the same XCD's L2 every time
__host__ __device__ inline int trd_groups(int c, int p) {
  const int a = (c + 2 * p + 7) / 8, b = (c + 255) / 256;
  return ((a > b ? a : b) + 7) / 8 * 8;
}

__device__ __forceinline__ TrdArgs trd_of(TrdArgs t, int k) {
  const size_t n = t.n;
  t.a += n * n * k;
  t.v += n * kPanel * k;
  t.w += n * kPanel * k;
  t.x += n * k;
  t.y += (n + 2 * kPanel) * k;
  t.part += (n + 63) / 64 * k;
  t.vav += (size_t)trd_groups(t.n, kPanel) * k;
  t.d += n * k;
  t.e += n * k;
  t.tau += n * k;
  return t;
}

// acc -= x y, acc -= x conj(y)
__device__ __forceinline__ void msub(cplx &acc, cplx x, cplx y) {
  acc.re -= x.re * y.re - x.im * y.im;
  acc.im -= x.re * y.im + x.im * y.re;
}
__device__ __forceinline__ void msubc(cplx &acc, cplx x, cplx y) {
  acc.re -= x.re * y.re + x.im * y.im;
  acc.im -= x.im * y.re - x.re * y.im;
}

// p: the panel's columns that have V (fin: the last of them still lacks W, its product is in y).
// upd: column c updated into x, its norm above row c - 1 into part, d(c).  groups: trd_mv's for that product
__global__ __launch_bounds__(256) void trd_col_kernel(TrdArgs args, int c, int p, int fin, int upd, int groups) {
  const TrdArgs t = trd_of(args, blockIdx.y);
  __shared__ cplx rz[4][64], rx[4][64], rc[4];
  __shared__ double rs[4];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = blockIdx.x * 64 + lane, rr = min(r, c);
  const size_t n = t.n;
  const int m = c + 1, pf = p - 1;                       // rows of the last v; panel columns with W
  cplx z = {0.0, 0.0}, x = {0.0, 0.0}, zc = {0.0, 0.0};
  cplx ac = {0.0, 0.0}, tau = ac, yr = ac, yc = ac, v = ac;   // for the end, loaded with the rest
  double s = 0.0;
  if (upd) ac = t.a[rr + n * c];
  if (fin) {
    tau = t.tau[c];
    yr = t.y[rr];
    yc = t.y[c];
    v = t.v[rr + n * pf];
    double f = 0.0;                                        // v^H A v
    for (int i = threadIdx.x; i < groups; i += 256) f += t.vav[i];
#pragma unroll 8
    for (int q = wave; q < pf; q += 4) {
      const cplx vr = t.v[rr + n * q], wr = t.w[rr + n * q], vc = t.v[c + n * q], wc = t.w[c + n * q];
      const cplx a = t.y[m + q], b = t.y[m + pf + q];      // W_q^H v, V_q^H v
      msub(z, vr, a);
      msub(z, wr, b);
      msub(zc, vc, a);
      msub(zc, wc, b);
      msubc(x, vr, wc);
      msubc(x, wr, vc);
      s -= 2.0 * (a.re * b.re + a.im * b.im);
    }
    s += wave_sum(f);
  }
  rz[wave][lane] = z;
  rx[wave][lane] = x;
  if (lane == 0) {
    rc[wave] = zc;
    rs[wave] = s;
  }
  __syncthreads();
  if (wave) return;
#pragma unroll
  for (int w = 1; w < 4; ++w) {
    z.re += rz[w][lane].re;
    z.im += rz[w][lane].im;
    x.re += rx[w][lane].re;
    x.im += rx[w][lane].im;
  }
  x.re += ac.re;
  x.im += ac.im;
  if (fin) {
    const double hk = -0.5 * (tau.re * tau.re + tau.im * tau.im) * (((rs[0] + rs[1]) + rs[2]) + rs[3]);
    z.re += yr.re;
    z.im += yr.im;
    zc = cplx{((rc[0].re + rc[1].re) + rc[2].re) + rc[3].re + yc.re, ((rc[0].im + rc[1].im) + rc[2].im) + rc[3].im + yc.im};
    cplx w = cmul(tau, z), wc = cmul(tau, zc);             // v(c) = 1
    w = cplx{fma(hk, v.re, w.re), fma(hk, v.im, w.im)};
    wc.re += hk;
    if (r <= c) t.w[r + n * pf] = w;
    msubc(x, v, wc);
    x.re -= w.re;
    x.im -= w.im;
  }
  if (!upd) return;
  if (r <= c) t.x[r] = x;
  if (r == c) t.d[c] = x.re;
  const double f = wave_sum(r < c - 1 ? x.re * x.re + x.im * x.im : 0.0);
  if (lane == 0) t.part[blockIdx.x] = f;
}

// reflector of column c >= 1 (x, part) and y = A(0:c-1, 0:c-1) v, then W^H v and V^H v of the
// panel's p columns
__global__ __launch_bounds__(256) void trd_mv_kernel(TrdArgs args, int c, int p) {
  const TrdArgs t = trd_of(args, blockIdx.y);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const size_t n = t.n;
  // the norm, needed only after the sums: the row c - 1 of v is not x's, its term is added at the end
  const int np = (c + 64) / 64;                            // workgroups of trd_col: rows 0 .. c
  double xn2 = 0.0;
  for (int i = lane; i < np; i += 64) xn2 += t.part[i];
  const cplx al = t.x[c - 1];
  const int k = (blockIdx.x * 4 + wave) * 2, tot = c + 2 * p;
  auto column = [&](int q) -> const cplx * {
    return q < c ? t.a + n * q : q < c + p ? t.w + n * (q - c) : t.v + n * (q - c - p);
  };
  const bool work = k < tot;
  cplx s0 = {0.0, 0.0}, s1 = s0, l0 = s0, l1 = s0, x0 = s0, x1 = s0;
  if (work) {
    const cplx *a0 = column(k), *a1 = column(min(k + 1, tot - 1));
    l0 = a0[c - 1];
    l1 = a1[c - 1];
    if (k < c) x0 = t.x[k];
    if (k + 1 < c) x1 = t.x[k + 1];
#pragma unroll 8
    for (int r = lane; r < c - 1; r += 64) {
      const cplx x = t.x[r], b0 = a0[r], b1 = a1[r];
      s0.re += b0.re * x.re + b0.im * x.im;
      s0.im += b0.re * x.im - b0.im * x.re;
      s1.re += b1.re * x.re + b1.im * x.im;
      s1.im += b1.re * x.im - b1.im * x.re;
    }
  }
  xn2 = wave_sum(xn2);
  s0 = cplx{wave_sum(s0.re), wave_sum(s0.im)};
  s1 = cplx{wave_sum(s1.re), wave_sum(s1.im)};
  double rf[5];                                            // (a column below 1e-145 counts as zero)
  reflector(al.re, al.im, xn2, rf);
  const cplx tau = {rf[1], rf[2]}, sc = {rf[3], rf[4]};
  const double beta = rf[0];
  double vav = 0.0;                                        // of v^H A v: conj(v_k) y_k, real part
  __shared__ double sv[4];
  if (work) {
    auto done = [&](int q, cplx s, cplx l, cplx x) {       // (A v)_q = sc s + conj(l), v = 1 at row c - 1
      const cplx y = cmul(sc, s), z = {y.re + l.re, y.im - l.im};
      if (q >= tot) return;
      if (lane == 0) t.y[q] = z;
      const cplx v = q == c - 1 ? cplx{1.0, 0.0} : cmul(sc, x);
      if (q < c) vav += v.re * z.re + v.im * z.im;
    };
    done(k, s0, l0, x0);
    done(k + 1, s1, l1, x1);
  }
  if (lane == 0) sv[wave] = vav;
  __syncthreads();
  if (threadIdx.x == 0) t.vav[blockIdx.x] = (sv[0] + sv[1]) + (sv[2] + sv[3]);
  // the reflector itself, by 256 rows a workgroup
  const int r = blockIdx.x * 256 + threadIdx.x;
  if (r < c) {
    const cplx v = r == c - 1 ? cplx{1.0, 0.0} : cmul(sc, t.x[r]);
    t.v[r + n * p] = v;
    t.a[r + n * c] = r == c - 1 ? cplx{beta, 0.0} : v;
    if (r == c - 1) {
      t.tau[r] = tau;
      t.e[r] = beta;
    }
  }
}

// A(0:m-1, 0:m-1) -= V W^H + W V^H over p columns: a 64 x 64 tile per workgroup, 32 x 32 a wave, the
// operands from L2
__global__ __launch_bounds__(256) void trd_update_kernel(TrdArgs args, int m, int p) {
  const TrdArgs t = trd_of(args, blockIdx.z);
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const size_t n = t.n;
  const int r0 = blockIdx.x * 64 + 32 * (wave & 1), k0 = blockIdx.y * 64 + 32 * (wave >> 1);
  if (r0 >= m || k0 >= m) return;
  int rr[2], kk[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    rr[i] = min(r0 + 16 * i + li, m - 1);
    kk[i] = min(k0 + 16 * i + li, m - 1);
  }
  d4_t re[2][2], im[2][2];                                 // (column tile, row tile)
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) re[i][j] = im[i][j] = d4_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll 2
  for (int q0 = 0; q0 < p; q0 += 4) {
    const bool in = q0 + lg < p;
    const size_t q = n * min(q0 + lg, p - 1);
    cplx vr[2], wr[2], vk[2], wk[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      vr[i] = t.v[rr[i] + q];
      wr[i] = t.w[rr[i] + q];
      vk[i] = t.v[kk[i] + q];
      wk[i] = t.w[kk[i] + q];
    }
    if (!in) vr[0] = vr[1] = wr[0] = wr[1] = vk[0] = vk[1] = wk[0] = wk[1] = cplx{0.0, 0.0};
    auto mac = [&](d4_t &cr, d4_t &ci, cplx y, cplx x) {   // + x conj(y)
      cr = __builtin_amdgcn_mfma_f64_16x16x4f64(y.re, x.re, cr, 0, 0, 0);
      ci = __builtin_amdgcn_mfma_f64_16x16x4f64(y.re, x.im, ci, 0, 0, 0);
      cr = __builtin_amdgcn_mfma_f64_16x16x4f64(y.im, x.im, cr, 0, 0, 0);
      ci = __builtin_amdgcn_mfma_f64_16x16x4f64(-y.im, x.re, ci, 0, 0, 0);
    };
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        mac(re[i][j], im[i][j], wk[i], vr[j]);
        mac(re[i][j], im[i][j], vk[i], wr[j]);
      }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = r0 + 16 * j + li, k = k0 + 16 * i + 4 * v + lg;
        if (r < m && k < m) {
          cplx *a = t.a + r + n * k;
          *a = cplx{a->re - re[i][j][v], a->im - im[i][j][v]};
        }
      }
}

}  // namespace

size_t exc_trd_work_bytes(int n, int nb) {
  return ((size_t)n * (2 * kPanel + 2) + 2 * kPanel) * nb * sizeof(cplx) +
         ((size_t)(n + 63) / 64 + trd_groups(n, kPanel)) * nb * sizeof(double);
}

// a: nb matrices n x n; d, e: n and tau: n per matrix
int exc_launch_trd(int n, int nb, cplx *a, double *d, double *e, cplx *tau, void *work, hipStream_t s) {
  if (n <= 0 || nb <= 0) return EXC_OK;
  if (nb > 65535 || (n + 63) / 64 > 65535) return EXC_ERR_ARG;
  TrdArgs t;
  t.n = n;
  t.a = a;
  t.v = (cplx *)work;
  t.w = t.v + (size_t)n * kPanel * nb;
  t.x = t.w + (size_t)n * kPanel * nb;
  t.y = t.x + (size_t)n * nb;
  t.part = (double *)(t.y + ((size_t)n + 2 * kPanel) * nb);
  t.vav = t.part + (size_t)(n + 63) / 64 * nb;
  t.d = d;
  t.e = e;
  t.tau = tau;
  auto col = [&](int c, int p, int fin, int upd) {
    hipLaunchKernelGGL(trd_col_kernel, dim3(c / 64 + 1, nb), dim3(256), 0, s, t, c, p, fin, upd, trd_groups(c + 1, p - 1));
  };
  int c = n - 1;
  while (c > 0) {
    int p = 0;
    col(c, 0, 0, 1);
    for (;;) {
      hipLaunchKernelGGL(trd_mv_kernel, dim3(trd_groups(c, p), nb), dim3(256), 0, s, t, c, p);
      ++p;
      --c;
      const bool last = p == kPanel || c == 0;
      col(c, p, 1, !last);
      if (last) break;
    }
    const int g = c / 64 + 1;
    hipLaunchKernelGGL(trd_update_kernel, dim3(g, g, nb), dim3(256), 0, s, t, c + 1, p);
    EXC_CHECK(hipGetLastError());
  }
  col(0, 0, 0, 1);                                         // d(0)
  EXC_CHECK(hipGetLastError());
  return EXC_OK;
}
