// Device helpers of the generalized eigensolve (exc_eigen_dev, exc_eigen_batched_dev).
//
// solvewithlapack (modfvsystem.f90:585-720) hands ZHEGVX the upper triangles of H and O.
// The level-3 reduction C = U^-H H U^-1 multiplies by the whole of H, so the lower triangle
// is first made the conjugate of the upper one (and the diagonal real, as ZHETRD assumes).
//
// The grouped solve of many k-points copies every k-point's pair into a strided batch of
// one common order n = max nmat_k, padded as
//     H_pad = [H_k 0; 0 sigma I],   O_pad = [O_k 0; 0 I],
// for the strided-batched Cholesky, triangular inverse, trmm and tridiagonal reduction (one
// launch per step for all k-points; the per-k-point reduction is thousands of small
// launches, one column at a time).  The pad stays out of the leading nmat_k block of every
// result: the Cholesky factor and its inverse are block diagonal with an identity block, the
// reduced matrix is [C_k 0; 0 sigma I], the Householder reflectors of the columns of C_k touch
// only rows above their column, and those of the pad columns annihilate vectors that are
// already zero (tau = 0).  The leading nmat_k part of the tridiagonal matrix, the reflectors
// and U^-1 are therefore those of the k-point alone (to rounding: the blocking of the
// batched routines follows n), and the rest of the solve runs per k-point on that part only.
#include "exc_common.h"

namespace {

constexpr int kET = 32;          // tile edge of the fill and pad kernels
constexpr int kEThreads = 256;   // 32 rows x 8 column groups
constexpr int kSelThreads = 1024;

__device__ __forceinline__ cplx czero() { return {0.0, 0.0}; }

// In place: h(r, c) = conj(h(c, r)) for r > c, Im h(c, c) = 0.  Block (ti, tj), ti <= tj,
// reads tile (ti, tj) of the upper triangle and writes its conjugate transpose at (tj, ti).
__global__ __launch_bounds__(kEThreads) void herm_fill_kernel(cplx *h, int n, int ldh) {
  const int ti = blockIdx.x, tj = blockIdx.y;
  if (ti > tj) return;
  __shared__ cplx s[kET][kET + 1];   // s[c][r] = h(row0 + r, col0 + c)
  const int r = threadIdx.x % kET, cg = threadIdx.x / kET;
  const int row0 = ti * kET, col0 = tj * kET;
  for (int c = cg; c < kET; c += kEThreads / kET) {
    const int R = row0 + r, C = col0 + c;
    s[c][r] = (R < n && C < n) ? h[R + (size_t)C * ldh] : czero();
  }
  __syncthreads();
  // destination (col0 + r, row0 + c) = conj(h(row0 + c, col0 + r)) = conj(s[r][c]),
  // for destination rows strictly below the diagonal
  for (int c = cg; c < kET; c += kEThreads / kET) {
    const int R = col0 + r, C = row0 + c;
    if (R >= n || C >= n) continue;
    if (R > C) {
      h[R + (size_t)C * ldh] = cconj(s[r][c]);
    } else if (R == C) {
      h[R + (size_t)C * ldh].im = 0.0;
    }
  }
}

// Padded copy of matrix `which` (0: H with pad sigma, 1: O with pad 1) of every k-point of
// the batch into p + k * n * n (leading dimension n), both triangles from the upper one.
__global__ __launch_bounds__(kEThreads) void eig_pad_kernel(const eig_kdesc *ks, int n, cplx *p, int which,
                                                            double sigma) {
  const int ti = blockIdx.x, tj = blockIdx.y, k = blockIdx.z;
  if (ti > tj) return;
  const eig_kdesc kd = ks[k];
  const cplx *src = which ? kd.o : kd.h;
  const double dpad = which ? 1.0 : sigma;
  cplx *dst = p + (size_t)k * n * n;
  __shared__ cplx s[kET][kET + 1];
  const int r = threadIdx.x % kET, cg = threadIdx.x / kET;
  const int row0 = ti * kET, col0 = tj * kET;
  for (int c = cg; c < kET; c += kEThreads / kET) {
    const int R = row0 + r, C = col0 + c;
    if (R >= n || C >= n) continue;
    cplx v;
    if (R > C) {
      v = czero();   // below the diagonal of a diagonal tile: written from s below
    } else if (C < kd.n) {
      v = src[R + (size_t)C * kd.ldh];
      if (R == C) v.im = 0.0;
    } else {
      v = R == C ? cplx{dpad, 0.0} : czero();
    }
    s[c][r] = v;
    if (R <= C) dst[R + (size_t)C * n] = v;
  }
  __syncthreads();
  for (int c = cg; c < kET; c += kEThreads / kET) {
    const int R = col0 + r, C = row0 + c;
    if (R >= n || C >= n || R <= C) continue;
    dst[R + (size_t)C * n] = cconj(s[r][c]);
  }
}

// zc(:, j) = zr(:, j) for j < ncols (m rows): real eigenvectors of the tridiagonal matrix
// into the complex workspace of the back-transform
__global__ __launch_bounds__(256) void eig_r2c_kernel(const double *zr, int m, int ldr, cplx *zc, int ldc) {
  const int r = blockIdx.x * 256 + threadIdx.x, j = blockIdx.y;
  if (r >= m) return;
  zc[r + (size_t)j * ldc] = {zr[r + (size_t)j * ldr], 0.0};
}

// Block i0 .. i0+ib-1 of the reflectors of the upper tridiagonal reduction (zhetrd 'U':
// reflector i has v(0:i-1) = A(0:i-1, i+1), v(i) = 1, zero below) as explicit columns,
// V[k sv + r + n c] for r < m = i0 + ib, of every k-point k of the batch
__global__ __launch_bounds__(256) void eig_vblock_kernel(const cplx *A, int n, int i0, int ib, size_t sv, cplx *V) {
  const int r = blockIdx.x * 256 + threadIdx.x, c = blockIdx.y, k = blockIdx.z;
  const int m = i0 + ib;
  if (r >= m) return;
  const int i = i0 + c;
  cplx v = {0.0, 0.0};
  if (r < i) v = A[(size_t)k * n * n + r + (size_t)n * (i + 1)];
  else if (r == i) v.re = 1.0;
  V[(size_t)k * sv + r + (size_t)n * c] = v;
}

// G = V^H V (lower triangle) of every block of kTB reflectors of every k-point, V as above straight from A:
// a 16 x 16 tile per workgroup, the rows split over its 4 waves (FP64 MFMA, operands from L2).  All blocks in one
// launch: as a product per block, 64 x 64 results leave the chip idle for 20 of them in turn.
constexpr int kTB = 64;
__global__ __launch_bounds__(256) void eig_vhv_kernel(const cplx *A, int n, cplx *G) {
  const int tile = blockIdx.x, nblk = gridDim.y, blk = blockIdx.y, k = blockIdx.z;
  int ti = 0, tj = tile;                                   // ti >= tj, row by row
  while (tj > ti) tj -= ++ti;
  const int i0 = blk * kTB, ib = min(kTB, n - 1 - i0), mb = i0 + ib;
  if (16 * ti >= ib) return;
  __shared__ cplx red[4][4][64];
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int fi = i0 + min(16 * ti + li, ib - 1), fj = i0 + min(16 * tj + li, ib - 1);   // reflectors
  const cplx *pi = A + (size_t)k * n * n + (size_t)n * (fi + 1), *pj = A + (size_t)k * n * n + (size_t)n * (fj + 1);
  d4_t re = {0.0, 0.0, 0.0, 0.0}, im = re;
#pragma unroll 4
  for (int r0 = 4 * wave; r0 < mb; r0 += 16) {
    const int r = r0 + lg, rc = min(r, mb - 1);
    cplx x = pi[rc], y = pj[rc];
    x = r < fi ? x : cplx{r == fi ? 1.0 : 0.0, 0.0};
    y = r < fj ? y : cplx{r == fj ? 1.0 : 0.0, 0.0};
    re = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re, y.re, re, 0, 0, 0);
    im = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re, y.im, im, 0, 0, 0);
    re = __builtin_amdgcn_mfma_f64_16x16x4f64(x.im, y.im, re, 0, 0, 0);
    im = __builtin_amdgcn_mfma_f64_16x16x4f64(-x.im, y.re, im, 0, 0, 0);
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) red[v][wave][lane] = cplx{re[v], im[v]};
  __syncthreads();
  cplx s = {0.0, 0.0};
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    s.re += red[wave][w][lane].re;
    s.im += red[wave][w][lane].im;
  }
  const int i = 16 * ti + 4 * wave + lg, j = 16 * tj + li;
  if (i < ib && j < ib) G[((size_t)k * nblk + blk) * kTB * kTB + i + kTB * j] = s;
}

// T (ib x ib, lower triangular) of the block reflector H(i0+ib-1) ... H(i0) = I - V T V^H from
// G = V^H V and tau (zlarft, direct 'B', storev 'C').  T^-1 has the diagonal 1 / tau_r and the lower
// triangle of G, so column i of T is a forward substitution of its own:
//   T(i, i) = tau_i,  T(r, i) = -tau_r sum_{i <= q < r} G(r, q) T(q, i).
// The reflectors of k-point k beyond its own order (i >= nmat_k - 1: the pad columns and the
// coupling column, zero vectors) are left out (tau taken as 0).  One workgroup per block and k-point: lane
// i holds column i, its rows dealt to the 4 waves' registers, G in LDS.  A chain of ib sums either
// way: 158 us a block by zlarft's order on one wave, 58 here, and all blocks in one launch.
__global__ __launch_bounds__(4 * kTB) void eig_tblock_kernel(const eig_kdesc *ks, const cplx *G, const cplx *tau, int n,
                                                             cplx *T) {
  const int nblk = gridDim.x, blk = blockIdx.x, k = blockIdx.y, i = threadIdx.x & (kTB - 1);
  const int i0 = blk * kTB, ib = min(kTB, n - 1 - i0);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kTB);
  const int last = ks[k].n - 1;   // reflectors i0 + i < last are the k-point's
  const cplx *g = G + ((size_t)k * nblk + blk) * kTB * kTB;
  cplx *t = T + ((size_t)blk * gridDim.y + k) * kTB * kTB;   // a block's T of all k-points together
  __shared__ cplx sg[kTB][kTB];          // G(r, q) at [q][r]
  __shared__ cplx red[2][4][kTB], st[kTB];
  for (int e = threadIdx.x; e < kTB * ib; e += 4 * kTB) sg[e / kTB][e % kTB] = g[e];
  if (threadIdx.x < kTB) st[i] = i < ib && i0 + i < last ? tau[(size_t)k * n + i0 + i] : czero();
  __syncthreads();
  cplx col[kTB / 4];                     // T(4 j + wave, i)
#pragma unroll
  for (int j = 0; j < kTB / 4; ++j) col[j] = czero();
#pragma unroll 1
  for (int r = 0; r < ib; ++r) {
    cplx s = {0.0, 0.0};
#pragma unroll
    for (int j = 0; j < kTB / 4; ++j)
      if (4 * j + wave < r) {
        const cplx p = cmul(sg[4 * j + wave][r], col[j]);
        s.re += p.re;
        s.im += p.im;
      }
    red[r & 1][wave][i] = s;
    __syncthreads();
    if ((r & 3) != wave) continue;
    const cplx tr = st[r];
    cplx v = {0.0, 0.0};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      v.re += red[r & 1][w][i].re;
      v.im += red[r & 1][w][i].im;
    }
    v = cmul(tr, v);
    v = i < r ? cplx{-v.re, -v.im} : i == r ? tr : czero();
#pragma unroll
    for (int j = 0; j < kTB / 4; ++j)
      if (4 * j + wave == r) col[j] = v;
    if (i < ib) t[r + kTB * i] = v;
  }
}

// Eigenpairs of a tridiagonal matrix from bisection and inverse iteration (dstebz with eorder
// 'blocks', then dstein), ordered by split-off block; *nfound >= nev of them (the bisection
// keeps a whole cluster of equal eigenvalues at the upper end of the index range).  Column j
// moves to its rank among the nfound eigenvalues (ties by index) if that is below nev:
// x(r, rank_j) = z(r, j) as complex for r < m, eval(rank_j) = w(j).  Every workgroup of
// column j counts the rank itself (nfound reads); the grid covers m columns.
__global__ __launch_bounds__(256) void eig_sort_r2c_kernel(const double *zr, int m, int nev, int ldr,
                                                           const int *nfound, const double *w, cplx *x, int ldx,
                                                           double *eval) {
  const int r = blockIdx.x * 256 + threadIdx.x, j = blockIdx.y;
  const int nf = min(*nfound, m);
  if (j >= nf) return;   // uniform over the workgroup
  __shared__ int part[256];
  const double wj = w[j];
  int cnt = 0;
  for (int i = threadIdx.x; i < nf; i += 256) cnt += (w[i] < wj) || (w[i] == wj && i < j);
  part[threadIdx.x] = cnt;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (threadIdx.x < h) part[threadIdx.x] += part[threadIdx.x + h];
    __syncthreads();
  }
  const int rank = part[0];
  if (rank >= nev) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) eval[rank] = wj;
  if (r < m) x[r + (size_t)rank * ldx] = {zr[r + (size_t)j * ldr], 0.0};
}

// evec_k(r, j) = x(r, j) for r < nmat_k, j < nev (x: n x nev per k-point, leading dimension n)
__global__ __launch_bounds__(256) void eig_copyout_kernel(const eig_kdesc *ks, int n, int nev, const cplx *x) {
  const int r = blockIdx.x * 256 + threadIdx.x, j = blockIdx.y, k = blockIdx.z;
  const eig_kdesc kd = ks[k];
  if (r >= kd.n) return;
  kd.evec[r + (size_t)j * kd.ldv] = x[(size_t)k * n * nev + r + (size_t)j * n];
}

inline int tiles(int n) { return (n + kET - 1) / kET; }

}  // namespace

int exc_launch_eig_hermfill(cplx *h, int n, int ldh, hipStream_t s) {
  if (n <= 0) return EXC_OK;
  if (ldh < n || tiles(n) > 65535) return EXC_ERR_ARG;
  hipLaunchKernelGGL(herm_fill_kernel, dim3(tiles(n), tiles(n)), dim3(kEThreads), 0, s, h, n, ldh);
  EXC_CHECK(hipGetLastError());
  return EXC_OK;
}

int exc_launch_eig_pad(const eig_kdesc *ks, int nb, int n, cplx *ph, cplx *po, double sigma, hipStream_t s) {
  if (nb <= 0 || n <= 0) return EXC_OK;
  if (nb > 65535 || tiles(n) > 65535) return EXC_ERR_ARG;
  const dim3 grid(tiles(n), tiles(n), nb);
  hipLaunchKernelGGL(eig_pad_kernel, grid, dim3(kEThreads), 0, s, ks, n, ph, 0, sigma);
  EXC_CHECK(hipGetLastError());
  hipLaunchKernelGGL(eig_pad_kernel, grid, dim3(kEThreads), 0, s, ks, n, po, 1, sigma);
  EXC_CHECK(hipGetLastError());
  return EXC_OK;
}

int exc_launch_eig_r2c(const double *zr, int m, int ncols, int ldr, cplx *zc, int ldc, hipStream_t s) {
  if (m <= 0 || ncols <= 0) return EXC_OK;
  if (ncols > 65535 || ldr < m || ldc < m) return EXC_ERR_ARG;
  hipLaunchKernelGGL(eig_r2c_kernel, dim3((m + 255) / 256, ncols), dim3(256), 0, s, zr, m, ldr, zc, ldc);
  EXC_CHECK(hipGetLastError());
  return EXC_OK;
}

int exc_launch_eig_vblock(const cplx *A, int nb, int n, int i0, int ib, size_t sv, cplx *V, hipStream_t s) {
  if (nb <= 0 || ib <= 0) return EXC_OK;
  if (sv < (size_t)n * ib) return EXC_ERR_ARG;
  if (nb > 65535 || ib > 64 || i0 < 0 || i0 + ib > n - 1) return EXC_ERR_ARG;   // reflector i in column i + 1
  hipLaunchKernelGGL(eig_vblock_kernel, dim3((i0 + ib + 255) / 256, ib, nb), dim3(256), 0, s, A, n, i0, ib, sv, V);
  EXC_CHECK(hipGetLastError());
  return EXC_OK;
}

// T of every block of kTB reflectors: block b of k-point k at (b nb + k) kTB^2, leading dimension kTB; G: as much
int exc_launch_eig_tblock(const eig_kdesc *ks, const cplx *A, const cplx *tau, int nb, int n, cplx *G, cplx *T,
                          hipStream_t s) {
  if (nb <= 0 || n < 2) return EXC_OK;
  const int nblk = (n - 1 + kTB - 1) / kTB, t = kTB / 16;
  if (nblk > 65535 || nb > 65535) return EXC_ERR_ARG;
  hipLaunchKernelGGL(eig_vhv_kernel, dim3(t * (t + 1) / 2, nblk, nb), dim3(256), 0, s, A, n, G);
  EXC_CHECK(hipGetLastError());
  hipLaunchKernelGGL(eig_tblock_kernel, dim3(nblk, nb), dim3(4 * kTB), 0, s, ks, G, tau, n, T);
  EXC_CHECK(hipGetLastError());
  return EXC_OK;
}

int exc_launch_eig_sort_r2c(const double *zr, int m, int nev, int ldr, const int *nfound, const double *w, cplx *x,
                            int ldx, double *eval, hipStream_t s) {
  if (m <= 0 || nev <= 0) return EXC_OK;
  if (m > 65535 || nev > m) return EXC_ERR_ARG;
  hipLaunchKernelGGL(eig_sort_r2c_kernel, dim3((m + 255) / 256, m), dim3(256), 0, s, zr, m, nev, ldr, nfound, w, x,
                     ldx, eval);
  EXC_CHECK(hipGetLastError());
  return EXC_OK;
}

int exc_launch_eig_copyout(const eig_kdesc *ks, int nb, int n, int nev, const cplx *x, hipStream_t s) {
  if (nb <= 0 || nev <= 0) return EXC_OK;
  if (nb > 65535 || nev > 65535) return EXC_ERR_ARG;
  hipLaunchKernelGGL(eig_copyout_kernel, dim3((n + 255) / 256, nev, nb), dim3(256), 0, s, ks, n, nev, x);
  EXC_CHECK(hipGetLastError());
  return EXC_OK;
}
