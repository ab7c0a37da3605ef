// X = U^-1 of O = U^H U for a strided batch of Hermitian positive definite matrices (upper triangles read,
// X in their place): the first half of the grouped eigensolve's reduction to standard form.
//
// Cholesky factor and inverse come from the same elimination: with Y = U^-H, block row b of [U | Y] is
// Y_bb [A_b | R_b], and every later row i subtracts U_bi^H [U_b | Y_b] from [A_i | R_i].  R needs the blocks
// below the diagonal only, which are free, and U itself is needed for one step.  Per 64 columns two
// launches for the whole batch:
//  * chol_panel: row b's product with Y_bb, kept as 64 x n with the columns running (the update's
//    operand), and X's block column b = Y_b^H into the upper triangle;
//  * chol_update: the 64 x 64 blocks of the later rows, 32 x 32 a wave on the FP64 matrix cores, operands
//    from L2.  The workgroup of the next diagonal block factors and inverts it on the spot, in LDS by the
//    same elimination in blocks of 16, while the others are at work.
// Bound by the chain of diagonal blocks on small orders, by the matrix cores on large ones.
#include "exc_common.h"

namespace {

constexpr int kB = 64, kBS = 16, kLd = kB + 1;

struct CholArgs {
  int n, nb;
  cplx *a;             // n x n at n n k
  cplx *p;             // kB x n at kB n k: row b of [Y | U], columns fastest
  cplx *y;             // kB x kB at kB^2 k: Y_bb, (row, column) at row + kB column
  int *info;           // per matrix: order of the first leading minor that is not positive, or 0
};

__device__ __forceinline__ double lane_of(double v, int q) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, q), hi = __builtin_amdgcn_readlane((int)(b >> 32), q);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// + x y, + conj(x) y and + x conj(y); x: rows of the result, y: columns
__device__ __forceinline__ void mac(d4_t &re, d4_t &im, cplx x, cplx y) {
  re = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re, y.re, re, 0, 0, 0);
  im = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re, y.im, im, 0, 0, 0);
  re = __builtin_amdgcn_mfma_f64_16x16x4f64(-x.im, y.im, re, 0, 0, 0);
  im = __builtin_amdgcn_mfma_f64_16x16x4f64(x.im, y.re, im, 0, 0, 0);
}
__device__ __forceinline__ void macc(d4_t &re, d4_t &im, cplx x, cplx y) { mac(re, im, cplx{x.re, -x.im}, y); }

// S (column c, row r at S[c][r]): the upper triangle of a 64 x 64 block of A in, Y = U^-H out (in the lower
// one).  The order of the first minor that is not positive, or 0, in every thread.
__device__ int factor_block(cplx (*S)[kLd], cplx (*L)[kBS + 1], double *rinv, int *bad) {
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (threadIdx.x == 0) *bad = 0;
  __syncthreads();
#pragma unroll 1
  for (int s = 0; s < kB / kBS; ++s) {
    const int c0 = kBS * s;
    if (wave == 0) {                 // L = U^H of the diagonal 16 x 16: lane = row, its columns in registers
      cplx x[kBS];
#pragma unroll
      for (int c = 0; c < kBS; ++c) {
        const cplx v = S[c0 + li][c0 + min(c, li)];
        x[c] = cplx{v.re, -v.im};
      }
      int first = 0;
#pragma unroll
      for (int c = 0; c < kBS; ++c) {
        if (first) continue;         // uniform
        const double p = lane_of(x[c].re, c);
        if (!(p > 0.0)) {
          first = c0 + c + 1;
          continue;
        }
        const double r = sqrt(p), ri = 1.0 / r;
        if (lane == c) rinv[c] = ri;
        x[c] = li == c ? cplx{r, 0.0} : cplx{x[c].re * ri, x[c].im * ri};
        __builtin_amdgcn_sched_barrier(0);   // column by column: hoisted broadcasts would spill
#pragma unroll
        for (int q = c + 1; q < kBS; ++q) {
          const double br = lane_of(x[c].re, q), bi = lane_of(x[c].im, q);
          x[q].re -= x[c].re * br + x[c].im * bi;
          x[q].im -= x[c].im * br - x[c].re * bi;
        }
      }
      if (lane < kBS)
#pragma unroll
        for (int c = 0; c < kBS; ++c) L[lane][c] = x[c];
      if (lane == 0 && first) *bad = first;
    }
    __syncthreads();
    if (*bad) return *bad;           // uniform
    if (wave == 0) {                 // its inverse: a column per lane
      cplx y[kBS];
#pragma unroll
      for (int r = 0; r < kBS; ++r) {
        cplx t = {r == li ? 1.0 : 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < r; ++q) {
          const cplx l = L[r][q];
          t.re -= l.re * y[q].re - l.im * y[q].im;
          t.im -= l.re * y[q].im + l.im * y[q].re;
        }
        y[r] = cplx{t.re * rinv[r], t.im * rinv[r]};
        __builtin_amdgcn_sched_barrier(0);
      }
      if (lane < kBS)
#pragma unroll
        for (int r = 0; r < kBS; ++r) S[c0 + lane][c0 + r] = y[r];
    }
    __syncthreads();
    if (wave < 3) {                  // row s: a 16 x 16 block per wave
      const int j = wave < s ? wave : wave + 1;
      d4_t re = {0.0, 0.0, 0.0, 0.0}, im = re;
#pragma unroll
      for (int m = 0; m < kBS; m += 4) mac(re, im, S[c0 + m + lg][c0 + li], S[16 * j + li][c0 + m + lg]);
#pragma unroll
      for (int v = 0; v < 4; ++v) S[16 * j + li][c0 + 4 * v + lg] = cplx{re[v], im[v]};
    }
    __syncthreads();
    int t = 0;
#pragma unroll 1
    for (int i = s + 1; i < kB / kBS; ++i)
#pragma unroll 1
      for (int j = 0; j < kB / kBS; ++j) {
        if (j > s && j < i) continue;
        if ((t++ & 3) != wave) continue;
        d4_t re = {0.0, 0.0, 0.0, 0.0}, im = re;
#pragma unroll
        for (int m = 0; m < kBS; m += 4) macc(re, im, S[16 * i + li][c0 + m + lg], S[16 * j + li][c0 + m + lg]);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          cplx *e = &S[16 * j + li][16 * i + 4 * v + lg];
          const cplx o = j == s ? cplx{0.0, 0.0} : *e;
          *e = cplx{o.re - re[v], o.im - im[v]};
        }
      }
    __syncthreads();
  }
  return 0;
}

// block row i > b, block column j <= b or j >= i: A_ij (R_ij) -= U_bi^H [U_b | Y_b]_j; b = -1: the first
// diagonal block is factored and nothing else
__global__ __launch_bounds__(256) void chol_update_kernel(CholArgs g, int b, int nblk) {
  const int k = blockIdx.x, i = b + 1 + blockIdx.z, jq = blockIdx.y + b + 1, j = jq < nblk ? jq : jq - nblk;
  if (j > b && j < i) return;
  const bool diag = i == b + 1 && j == i;
  if (b >= 0 && g.info[k]) return;
  __shared__ cplx S[kB][kLd], L[kBS][kBS + 1];
  __shared__ double rinv[kBS];
  __shared__ int bad;
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = g.n;
  cplx *a = g.a + (size_t)n * n * k;
  const cplx *p = g.p + (size_t)kB * n * k;
  const int r0 = kB * i + 32 * (wave & 1), c0 = kB * j + 32 * (wave >> 1);
  int rr[2], cc[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    rr[q] = min(r0 + 16 * q + li, n - 1);
    cc[q] = min(c0 + 16 * q + li, n - 1);
  }
  d4_t re[2][2], im[2][2];                                 // (column tile, row tile)
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int r = 0; r < 2; ++r) re[q][r] = im[q][r] = d4_t{0.0, 0.0, 0.0, 0.0};
  if (b >= 0)
#pragma unroll 4
    for (int m = 0; m < kB; m += 4) {
      const cplx *pm = p + (size_t)n * (m + lg);
      cplx x[2], y[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        x[q] = pm[cc[q]];
        y[q] = pm[rr[q]];
        y[q].im = -y[q].im;
      }
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int r = 0; r < 2; ++r) mac(re[q][r], im[q][r], x[q], y[r]);
    }
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = r0 + 16 * r + li, col = c0 + 16 * q + 4 * v + lg;
        const bool in = row < n && col < n;
        cplx *e = a + min(row, n - 1) + (size_t)n * min(col, n - 1);
        cplx o = {0.0, 0.0};
        if (j != b && in) o = *e;
        o = cplx{o.re - re[q][r][v], o.im - im[q][r][v]};
        if (diag)
          S[col - kB * j][row - kB * i] = in ? o : cplx{row == col ? 1.0 : 0.0, 0.0};
        else if (in)
          *e = o;
      }
  if (!diag) return;
  const int f = factor_block(S, L, rinv, &bad);
  if (threadIdx.x == 0) g.info[k] = f ? kB * i + f : 0;
  if (f) return;
  cplx *y = g.y + (size_t)kB * kB * k;
  for (int e = threadIdx.x; e < kB * kB; e += 256) {
    const int r = e & (kB - 1), c = e / kB, row = kB * i + r, col = kB * i + c;
    const cplx v = r >= c ? S[c][r] : cplx{0.0, 0.0};
    y[e] = v;
    const cplx t = S[r][c];                                // X(r, c) = conj(Y(c, r))
    if (r <= c && col < n) a[row + (size_t)n * col] = cplx{t.re, -t.im};
  }
}

// row b of [Y | U] = Y_bb [R | A]: a wave takes 16 columns
__global__ __launch_bounds__(256) void chol_panel_kernel(CholArgs g, int b) {
  const int k = blockIdx.x;
  if (g.info[k]) return;
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = g.n, j0 = kB * b, j = kB * blockIdx.y + 16 * wave + li, jc = min(j, n - 1);
  cplx *a = g.a + (size_t)n * n * k;
  cplx *p = g.p + (size_t)kB * n * k;
  const cplx *y = g.y + (size_t)kB * kB * k;
  if (blockIdx.y == (unsigned)b) {
    if (j < n)
      for (int r = lg; r < kB; r += 4) p[(size_t)n * r + j] = y[r + kB * (j - j0)];
    return;
  }
  d4_t re[4], im[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) re[t] = im[t] = d4_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int m0 = 0; m0 < kB; m0 += 16)
#pragma unroll
    for (int m = m0; m < m0 + 16; m += 4) {
      const int row = j0 + m + lg;
      cplx x = a[min(row, n - 1) + (size_t)n * jc];
      if (row >= n) x = cplx{0.0, 0.0};
#pragma unroll
      for (int t = m0 / 16; t < 4; ++t) mac(re[t], im[t], y[16 * t + li + kB * (m + lg)], x);   // Y is lower triangular
    }
  if (j >= n) return;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int r = 16 * t + 4 * v + lg;
      p[(size_t)n * r + j] = cplx{re[t][v], im[t][v]};
      if (j < j0 && j0 + r < n) a[j + (size_t)n * (j0 + r)] = cplx{re[t][v], -im[t][v]};
    }
}

}  // namespace

size_t exc_chol_work_bytes(int n, int nb) { return sizeof(cplx) * ((size_t)kB * n + kB * kB) * nb; }

// a: nb matrices n x n; info: nb
int exc_launch_chol_inverse(int n, int nb, cplx *a, int *info, void *work, hipStream_t s) {
  if (n <= 0 || nb <= 0) return EXC_OK;
  const int nblk = (n + kB - 1) / kB;
  if (nblk > 65535) return EXC_ERR_ARG;
  CholArgs g;
  g.n = n;
  g.nb = nb;
  g.a = a;
  g.p = (cplx *)work;
  g.y = g.p + (size_t)kB * n * nb;
  g.info = info;
  hipLaunchKernelGGL(chol_update_kernel, dim3(nb, 1, 1), dim3(256), 0, s, g, -1, nblk);
  EXC_CHECK(hipGetLastError());
  for (int b = 0; b < nblk; ++b) {
    hipLaunchKernelGGL(chol_panel_kernel, dim3(nb, nblk), dim3(256), 0, s, g, b);
    EXC_CHECK(hipGetLastError());
    if (b + 1 < nblk) {
      hipLaunchKernelGGL(chol_update_kernel, dim3(nb, nblk, nblk - 1 - b), dim3(256), 0, s, g, b, nblk);
      EXC_CHECK(hipGetLastError());
    }
  }
  return EXC_OK;
}
