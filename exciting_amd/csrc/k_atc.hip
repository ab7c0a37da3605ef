// X^T Y of column-major complex matrices on gfx950: the products of apwalm with eigenvectors,
// sum_G A(G, f) C(G, n) (the adjoint's U, the coefficients of the densities), whose summation
// index runs along the columns.
//
// A workgroup takes a (16 TI) x (16 TJ) tile of the result and its 4 waves a quarter of the sum
// each (added in wave order through LDS): the result is small (a few hundred 32 x 32 tiles) and
// the sum long, so one wave per SIMD on every CU is what there is to have.  Operands go
// straight to registers, two to three groups of 16 G ahead; a load covers 4 consecutive G (64 bytes) of 16
// columns (with each lane's 4 loads side by side instead, 64 lines a load, it took 110 us below).  Three real products
// per complex product.  Bound by the FP64 MFMA rate; measured at 64 states, N = 2500, 16
// atoms: 102 us (49 TFLOP/s in four-product flops; 242 tiles, one per CU).
#include "mt_wave.h"

namespace {

using setup_dev::wdv2;

template <int TI, int TJ>
__global__ __launch_bounds__(256, 1) void xty_kernel(int n, const cplx *__restrict__ X, int ldx, int ni, size_t xs,
                                                  const cplx *__restrict__ Y, int ldy, int nj, size_t ys,
                                                  cplx *__restrict__ out, size_t si, size_t os) {
  struct Group {
    wdv2 a[4][TI], b[4][TJ];
  };
  __shared__ cplx red[TI * TJ * 4][4][64];
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i0 = blockIdx.x * 16 * TI, j0 = blockIdx.y * 16 * TJ;
  X += xs * blockIdx.z;
  Y += ys * blockIdx.z;
  const cplx *px[TI], *py[TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i) px[i] = X + (size_t)min(i0 + 16 * i + li, ni - 1) * ldx;   // columns past the end: the last again
#pragma unroll
  for (int j = 0; j < TJ; ++j) py[j] = Y + (size_t)min(j0 + 16 * j + li, nj - 1) * ldy;
  const int per = (n + 63) / 64 * 16;
  const int kb = wave * per, ke = min(n, kb + per);
  d4_t p1[TI][TJ], p2[TI][TJ], p3[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) p1[i][j] = p2[i][j] = p3[i][j] = d4_t{0.0, 0.0, 0.0, 0.0};
  auto load = [&](Group &g, int k0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = min(k0 + 4 * u + lg, n - 1);
#pragma unroll
      for (int i = 0; i < TI; ++i) g.a[u][i] = *(const wdv2 *)(px[i] + k);
#pragma unroll
      for (int j = 0; j < TJ; ++j) g.b[u][j] = *(const wdv2 *)(py[j] + k);
    }
  };
  auto step = [&](const Group &g, int k0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool in = k0 + 4 * u + lg < ke;
      double ar[TI], ai[TI], as[TI], br[TJ], bi[TJ], bs[TJ];
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        ar[i] = in ? g.a[u][i].x : 0.0;
        ai[i] = in ? g.a[u][i].y : 0.0;
        as[i] = ar[i] + ai[i];
      }
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        br[j] = in ? g.b[u][j].x : 0.0;
        bi[j] = in ? g.b[u][j].y : 0.0;
        bs[j] = br[j] + bi[j];
      }
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
          p1[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[i], br[j], p1[i][j], 0, 0, 0);
          p2[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai[i], bi[j], p2[i][j], 0, 0, 0);
          p3[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(as[i], bs[j], p3[i][j], 0, 0, 0);
        }
    }
  };
  // three groups in turn, each refilled right after its use: a copy from one to the next
  // would wait for the loads in flight.  Groups past the wave's share multiply zeros.
  Group g0, g1, g2;
  load(g0, kb);
  load(g1, kb + 16);
  load(g2, kb + 32);
#pragma unroll 1
  for (int k0 = kb; k0 < ke; k0 += 48) {
    step(g0, k0);
    load(g0, k0 + 48);
    step(g1, k0 + 16);
    load(g1, k0 + 64);
    step(g2, k0 + 32);
    load(g2, k0 + 80);
  }
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        red[4 * (TJ * i + j) + v][wave][lane] =
            cplx{p1[i][j][v] - p2[i][j][v], (p3[i][j][v] - p1[i][j][v]) - p2[i][j][v]};
  __syncthreads();
#pragma unroll
  for (int m = 0; m < TI * TJ; ++m) {
    const int e = wave * TI * TJ + m;
    const int i = i0 + 16 * (e / (4 * TJ)) + 4 * (e & 3) + lg, j = j0 + 16 * (e / 4 % TJ) + li;
    if (i >= ni || j >= nj) continue;
    cplx s = red[e][0][lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) {
      s.re += red[e][w][lane].re;
      s.im += red[e][w][lane].im;
    }
    out[os * blockIdx.z + i * si + j] = s;
  }
}

template <int TI, int TJ>
void launch_t(int nb, int n, const cplx *X, int ldx, int ni, size_t xs, const cplx *Y, int ldy, int nj, size_t ys,
              cplx *out, size_t si, size_t os, hipStream_t s) {
  hipLaunchKernelGGL((xty_kernel<TI, TJ>), dim3((ni + 16 * TI - 1) / (16 * TI), (nj + 16 * TJ - 1) / (16 * TJ), nb),
                     dim3(256), 0, s, n, X, ldx, ni, xs, Y, ldy, nj, ys, out, si, os);
}

}  // namespace

// out[b os + i si + j] = sum_k X(k, i) Y(k, j), k < n, for nb pairs at strides xs, ys: 32 x 32
// tiles, or 16 x 32 ones where those would be fewer than one per CU
int exc_launch_xty(int nb, int n, const cplx *X, int ldx, int ni, size_t xs, const cplx *Y, int ldy, int nj, size_t ys,
                   cplx *out, size_t si, size_t os, int ncu, hipStream_t s) {
  if (nb <= 0 || n <= 0 || ni <= 0 || nj <= 0) return EXC_OK;
  if ((nj + 15) / 16 > 65535 || nb > 65535) return EXC_ERR_ARG;
  const long tiles = (long)nb * ((ni + 31) / 32) * ((nj + 31) / 32);
  if (10 * tiles < 9 * ncu)
    launch_t<1, 2>(nb, n, X, ldx, ni, xs, Y, ldy, nj, ys, out, si, os, s);
  else
    launch_t<2, 2>(nb, n, X, ldx, ni, xs, Y, ldy, nj, ys, out, si, os, s);
  EXC_CHECK(hipGetLastError());
  return EXC_OK;
}
