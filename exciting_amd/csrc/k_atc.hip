// X^T Y of column-major complex matrices on gfx950: the products of apwalm with eigenvectors,
// sum_G A(G, f) C(G, n) (the adjoint's U, the coefficients of the densities), whose summation
// index runs along the columns.
//
// A workgroup takes a (16 TI) x (16 TJ) tile of the result and its 4 waves a quarter of the sum
// each (added in wave order through LDS): the result is small (a few hundred 32 x 32 tiles) and
// the sum long, so one wave per SIMD on every CU is what there is to have.  Operands go
// straight to registers, two to three groups of 8 G ahead; a load covers 4 consecutive G (64 bytes) of 16
// columns (with each lane's 4 loads side by side instead, 64 lines a load, it took 110 us below).  Measured with three
// real products per complex product at 64 states, N = 2500, 16 atoms: 90 us (56 TFLOP/s in
// four-product flops; 242 tiles, one per CU; 50 us of MFMA), 102 with groups of 16 G, whose registers
// were copied between turns.
#include <algorithm>

#include "mt_wave.h"

namespace {

using setup_dev::wdv2;

template <int TI, int TJ, bool G3>
__global__ __launch_bounds__(256, TI == 1 ? 2 : 1) void xty_kernel(
    int nb, int n, const cplx *__restrict__ X, int ldx, int ni, size_t xs, const cplx *__restrict__ Y, int ldy, int nj,
    size_t ys, cplx *__restrict__ out, size_t si, size_t os) {
  // workgroups b, b + 8, ... run on one XCD: a contiguous eighth of the tiles, the direction with
  // fewer of them fastest, so that those of the same columns read them through one L2
  const int gi = (ni + 16 * TI - 1) / (16 * TI), gj = (nj + 16 * TJ - 1) / (16 * TJ);
  const int chunk = gridDim.x / 8, tile = (blockIdx.x & 7) * chunk + (blockIdx.x >> 3);
  if (tile >= gi * gj * nb) return;
  const int fast = gi < gj ? gi : gj, f1 = tile % fast, f2 = tile / fast % (gi + gj - fast), b = tile / (gi * gj);
  const int bi = gi < gj ? f1 : f2, bj = gi < gj ? f2 : f1;
  constexpr int U = 2;                            // k-steps (of 4) per group of loads
  struct Group {
    wdv2 a[U][TI], b[U][TJ];
  };
  __shared__ cplx red[TI * TJ * 4][4][64];
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i0 = bi * 16 * TI, j0 = bj * 16 * TJ;
  X += xs * b;
  Y += ys * b;
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
    for (int u = 0; u < U; ++u) {
      const int k = min(k0 + 4 * u + lg, n - 1);
#pragma unroll
      for (int i = 0; i < TI; ++i) g.a[u][i] = *(const wdv2 *)(px[i] + k);
#pragma unroll
      for (int j = 0; j < TJ; ++j) g.b[u][j] = *(const wdv2 *)(py[j] + k);
    }
  };
  auto step = [&](const Group &g, int k0, bool full) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool in = full || k0 + 4 * u + lg < ke;
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
          if constexpr (G3) {
            p2[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai[i], bi[j], p2[i][j], 0, 0, 0);
            p3[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(as[i], bs[j], p3[i][j], 0, 0, 0);
          } else {
            p3[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[i], bi[j], p3[i][j], 0, 0, 0);
            p1[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(-ai[i], bi[j], p1[i][j], 0, 0, 0);
            p3[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai[i], br[j], p3[i][j], 0, 0, 0);
          }
        }
    }
  };
  // three groups in turn, each refilled right after its use: a copy from one to the next would wait
  // for the loads in flight, and so would a load moved across a step (the scheduling barriers), or
  // accumulators that do not fit beside the groups in 256 registers (copied each turn).
  // Past the last whole turn the elements past the wave's share are taken as zeros.
  Group g0, g1, g2;
  load(g0, kb);
  load(g1, kb + 4 * U);
  load(g2, kb + 8 * U);
  int k0 = kb;
#pragma unroll 1
  for (; k0 + 12 * U <= ke; k0 += 12 * U) {
    __builtin_amdgcn_sched_barrier(0);
    step(g0, k0, true);
    __builtin_amdgcn_sched_barrier(0);
    load(g0, k0 + 12 * U);
    __builtin_amdgcn_sched_barrier(0);
    step(g1, k0 + 4 * U, true);
    __builtin_amdgcn_sched_barrier(0);
    load(g1, k0 + 16 * U);
    __builtin_amdgcn_sched_barrier(0);
    step(g2, k0 + 8 * U, true);
    __builtin_amdgcn_sched_barrier(0);
    load(g2, k0 + 20 * U);
  }
  step(g0, k0, false);
  step(g1, k0 + 4 * U, false);
  step(g2, k0 + 8 * U, false);
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        red[4 * (TJ * i + j) + v][wave][lane] =
            G3 ? cplx{p1[i][j][v] - p2[i][j][v], (p3[i][j][v] - p1[i][j][v]) - p2[i][j][v]}
               : cplx{p1[i][j][v], p3[i][j][v]};
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
    out[os * b + i * si + j] = s;
  }
}

template <int TI, int TJ, bool G3>
void launch_t(int nb, int n, const cplx *X, int ldx, int ni, size_t xs, const cplx *Y, int ldy, int nj, size_t ys,
              cplx *out, size_t si, size_t os, hipStream_t s) {
  const long tiles = (long)nb * ((ni + 16 * TI - 1) / (16 * TI)) * ((nj + 16 * TJ - 1) / (16 * TJ));
  hipLaunchKernelGGL((xty_kernel<TI, TJ, G3>), dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(256), 0, s, nb, n, X, ldx, ni, xs, Y,
                     ldy, nj, ys, out, si, os);
}

}  // namespace

// out[b os + i si + j] = sum_k X(k, i) Y(k, j), k < n, for nb pairs at strides xs, ys, by three real
// products (Gauss) or four, which round the imaginary parts less: 32 x 32 tiles, one workgroup per CU
// at a time, or 16 x 32 ones, two per CU and 0.7 of the time each, where those fill the chip better
// (162 x 200 for each of 8 atoms, N = 1200: three products, 336 tiles 80 us, 624 half tiles 69; four, half
// tiles 75, the library's product 136; three products, 3872 x 64, N = 2500: 242 tiles 90, 484 half tiles 131)
int exc_launch_xty(int nb, int n, const cplx *X, int ldx, int ni, size_t xs, const cplx *Y, int ldy, int nj, size_t ys,
                   cplx *out, size_t si, size_t os, bool three, int ncu, hipStream_t s) {
  if (nb <= 0 || n <= 0 || ni <= 0 || nj <= 0) return EXC_OK;
  const long tiles = (long)nb * ((ni + 31) / 32) * ((nj + 31) / 32);
  if (tiles > 0x3fffffff) return EXC_ERR_ARG;
  const long half = (long)nb * ((ni + 15) / 16) * ((nj + 31) / 32);
  const bool narrow = 7 * std::max(half, (long)ncu) < 10 * ncu * ((tiles + ncu - 1) / ncu);
  auto launch = three ? (narrow ? launch_t<1, 2, true> : launch_t<2, 2, true>)
                      : (narrow ? launch_t<1, 2, false> : launch_t<2, 2, false>);
  launch(nb, n, X, ldx, ni, xs, Y, ldy, nj, ys, out, si, os, s);
  EXC_CHECK(hipGetLastError());
  return EXC_OK;
}
