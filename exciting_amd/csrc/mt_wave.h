// Narrow FP64 MFMA tiles for small bases: the muffin-tin tile and the Y-stage tile of mt_dma.h
// where the 64-wide tiles leave most of the chip idle.
//
// A workgroup takes one (16 TB) x (16 TB) tile; its 4 waves (one per SIMD) split the sum over
// k and are added in wave order through LDS at the end.  The operands go from global memory
// (L2) straight to registers in the MFMA layout (16 rows of 16 bytes contiguous per k), U
// to 2 U k-steps of 4 ahead of their use: no LDS staging and no barrier in the K loop, so a wave's time
// is its MFMA chain plus one memory latency per U steps, and the interstitial values of the
// elements a wave finishes are looked up before the K loop (three dependent loads).
// Gauss's three real products per complex product, as the 64-wide default.
#pragma once
#include "setup_dev.h"

namespace setup_dev {

typedef double wdv2 __attribute__((ext_vector_type(2)));

// C(i, j) = sum_k op(A(i, k)) B(j, k): this wave's quarter of k, (re, im) of its TB x TB blocks
template <int TB, bool CONJA>
struct WaveCore {
  static constexpr int U = TB == 1 ? 8 : 4;       // k-steps (of 4) per group of loads
  static constexpr int T = 16 * TB;
  static constexpr int E = TB * TB * 4;           // accumulator registers of a tile and lane
  struct Red {
    cplx v[E][4][64];
  };

  struct Group {
    wdv2 a[U][TB], b[U][TB];
  };

  __device__ __forceinline__ static void cols(int (&kc)[U], const int *__restrict__ kperm, int k0, int klast) {
    const int lk = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int u = 0; u < U; ++u) kc[u] = kperm[min(k0 + 4 * u + lk, klast)];
  }
  __device__ __forceinline__ static void load(Group &g, const int (&kc)[U], const cplx *const (&pa)[TB], int lda,
                                              const cplx *const (&pb)[TB], int ldb) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < TB; ++i) {
        g.a[u][i] = *(const wdv2 *)(pa[i] + (size_t)kc[u] * lda);
        g.b[u][i] = *(const wdv2 *)(pb[i] + (size_t)kc[u] * ldb);
      }
  }

  // rows past mrows / nrows read row 0 (never stored); the k's past this wave's share count zero
  __device__ __forceinline__ static void run(const cplx *__restrict__ A, int lda, int row0, int mrows,
                                             const cplx *__restrict__ B, int ldb, int col0, int nrows, int ktot,
                                             const int *__restrict__ kperm, d4_t (&cr)[TB][TB], d4_t (&ci)[TB][TB]) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int per = (ktot + 15) / 16 * 4;          // k's per wave, whole k-steps
    sum(A, lda, row0, mrows, B, ldb, col0, nrows, ktot, wave * per, min(ktot, (wave + 1) * per), kperm, cr, ci);
  }

  // the same for k in [kb, ke)
  __device__ __forceinline__ static void sum(const cplx *__restrict__ A, int lda, int row0, int mrows,
                                             const cplx *__restrict__ B, int ldb, int col0, int nrows, int ktot, int kb,
                                             int ke, const int *__restrict__ kperm, d4_t (&cr)[TB][TB],
                                             d4_t (&ci)[TB][TB]) {
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const cplx *pa[TB], *pb[TB];
#pragma unroll
    for (int i = 0; i < TB; ++i) {
      const int r = row0 + 16 * i + li, c = col0 + 16 * i + li;
      pa[i] = A + (r < mrows ? r : 0);
      pb[i] = B + (c < nrows ? c : 0);
    }
    d4_t p1[TB][TB], p2[TB][TB], p3[TB][TB];
#pragma unroll
    for (int i = 0; i < TB; ++i)
#pragma unroll
      for (int j = 0; j < TB; ++j) p1[i][j] = p2[i][j] = p3[i][j] = d4_t{0.0, 0.0, 0.0, 0.0};
    const int klast = ktot - 1;
    auto step = [&](const Group &g, int k0) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (k0 + 4 * u >= ke) break;
        const bool in = k0 + 4 * u + lk < ke;
        double ar[TB], ai[TB], as[TB], br[TB], bi[TB], bs[TB];
#pragma unroll
        for (int i = 0; i < TB; ++i) {
          ar[i] = in ? g.a[u][i].x : 0.0;
          ai[i] = in ? g.a[u][i].y : 0.0;
          as[i] = CONJA ? ar[i] - ai[i] : ar[i] + ai[i];
          br[i] = in ? g.b[u][i].x : 0.0;
          bi[i] = in ? g.b[u][i].y : 0.0;
          bs[i] = br[i] + bi[i];
        }
#pragma unroll
        for (int i = 0; i < TB; ++i)
#pragma unroll
          for (int j = 0; j < TB; ++j) {
            p1[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[i], br[j], p1[i][j], 0, 0, 0);
            p2[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai[i], bi[j], p2[i][j], 0, 0, 0);
            p3[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(as[i], bs[j], p3[i][j], 0, 0, 0);
          }
      }
    };
    // two groups in turn, each refilled right after its use (a copy from one to the next would
    // wait for the loads in flight); past the end they load the last k's again, unused
    int kc[U];
    Group g0, g1;
    cols(kc, kperm, kb, klast);
    load(g0, kc, pa, lda, pb, ldb);
    cols(kc, kperm, kb + 4 * U, klast);
    load(g1, kc, pa, lda, pb, ldb);
    cols(kc, kperm, kb + 8 * U, klast);
#pragma unroll 1
    for (int k0 = kb; k0 < ke; k0 += 8 * U) {
      step(g0, k0);
      load(g0, kc, pa, lda, pb, ldb);
      cols(kc, kperm, k0 + 12 * U, klast);
      if (k0 + 4 * U >= ke) break;
      step(g1, k0 + 4 * U);
      load(g1, kc, pa, lda, pb, ldb);
      cols(kc, kperm, k0 + 16 * U, klast);
    }
#pragma unroll
    for (int i = 0; i < TB; ++i)
#pragma unroll
      for (int j = 0; j < TB; ++j) {
        cr[i][j] = CONJA ? p1[i][j] + p2[i][j] : p1[i][j] - p2[i][j];
        ci[i][j] = CONJA ? (p3[i][j] - p1[i][j]) + p2[i][j] : (p3[i][j] - p1[i][j]) - p2[i][j];
      }
  }

  // every wave's partial sums into LDS; element e of lane `lane` afterwards is total(red, e).
  // e = 4 (TB i + j) + v sits at row 16 i + 4 v + lane / 16, column 16 j + lane % 16; wave w
  // finishes the elements e = w TB^2 .. (w + 1) TB^2 - 1
  __device__ __forceinline__ static void share(Red &red, const d4_t (&cr)[TB][TB], const d4_t (&ci)[TB][TB]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < TB; ++i)
#pragma unroll
      for (int j = 0; j < TB; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) red.v[4 * (TB * i + j) + v][wave][lane] = cplx{cr[i][j][v], ci[i][j][v]};
    __syncthreads();
  }
  __device__ __forceinline__ static cplx total(const Red &red, int e) {
    const int lane = threadIdx.x & 63;
    cplx s = red.v[e][0][lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) {
      const cplx p = red.v[e][w][lane];
      s.re += p.re;
      s.im += p.im;
    }
    return s;
  }
  __device__ __forceinline__ static int row_of(int e) {
    return 16 * (e / (4 * TB)) + 4 * (e & 3) + ((threadIdx.x & 63) >> 4);
  }
  __device__ __forceinline__ static int col_of(int e) { return 16 * (e / 4 % TB) + (threadIdx.x & 15); }
};

// one (tile, H-or-O) item: the counterpart of MtTileDMA::run
template <int TB>
struct MtTileWave {
  using C = WaveCore<TB, true>;
  __device__ static void run(typename C::Red &red, int ngp, int ktot, const cplx *__restrict__ apwalm, int ldg,
                             const cplx *__restrict__ yt, int ldy, const int *__restrict__ igpig,
                             const double *__restrict__ vgpc, const GTab &gt, cplx *__restrict__ h,
                             cplx *__restrict__ o, int ldh, const int *__restrict__ kperm, int ti, int tj, int which) {
    constexpr int M = TB * TB;
    const int row0 = ti * C::T, col0 = tj * C::T;
    const int e0 = (threadIdx.x >> 6) * M;
    cplx add[M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int r = row0 + C::row_of(e0 + m), c = col0 + C::col_of(e0 + m);
      add[m] = cplx{0.0, 0.0};
      if (r <= c && c < ngp) {
        const int *gr = gt.ivg + 3 * (igpig[r] - 1), *gc = gt.ivg + 3 * (igpig[c] - 1);
        const int ig = lookup_g(gt, gr[0] - gc[0], gr[1] - gc[1], gr[2] - gc[2]);
        if (ig) {
          const double *vr = vgpc + 3 * r, *vc = vgpc + 3 * c;
          if (which) {
            add[m] = olp_theta(gt, ig, vr, vc);
          } else {
            const cplx vv = gt.veffig[ig - 1], kn = gt.kinig[ig - 1];
            const double t1 = 0.5 * (vr[0] * vc[0] + vr[1] * vc[1] + vr[2] * vc[2]);
            add[m] = cplx{vv.re + t1 * kn.re, vv.im + t1 * kn.im};
          }
        }
      }
    }
    d4_t cr[TB][TB], ci[TB][TB];
    C::run(apwalm, ldg, row0, ngp, which ? apwalm : yt, which ? ldg : ldy, col0, ngp, ktot, kperm, cr, ci);
    C::share(red, cr, ci);
    cplx *out = which ? o : h;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int r = row0 + C::row_of(e0 + m), c = col0 + C::col_of(e0 + m);
      if (r > c || c >= ngp) continue;
      const cplx s = C::total(red, e0 + m);
      const double re = s.re + add[m].re, im = s.im + add[m].im;
      out[r + (size_t)c * ldh] = cplx{re, im};
      if (r < c) out[c + (size_t)r * ldh] = cplx{re, -im};
    }
  }
};

// one tile of Yt_a = A_a h_a^T, the tile's rows (basis functions) along the lanes; kfirst as in
// YTileDMA
template <int TB>
struct YTileWave {
  using C = WaveCore<TB, false>;
  __device__ static void run(typename C::Red &red, int ngp, int naa, const cplx *__restrict__ A, int ldg,
                             const cplx *__restrict__ ha, cplx *__restrict__ Y, int ldy, int row0, int col0,
                             const int *__restrict__ fperm, int kfirst) {
    constexpr int M = TB * TB;
    d4_t cr[TB][TB], ci[TB][TB];
    C::run(ha, naa, col0, naa, A, ldg, row0, ngp, naa - kfirst, fperm + kfirst, cr, ci);
    C::share(red, cr, ci);
    const int e0 = (threadIdx.x >> 6) * M;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int c = col0 + C::row_of(e0 + m), r = row0 + C::col_of(e0 + m);
      if (r < ngp && c < naa) Y[r + (size_t)c * ldy] = C::total(red, e0 + m);
    }
  }
};

}  // namespace setup_dev
