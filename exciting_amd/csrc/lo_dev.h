// Device code of the APW-lo and lo-lo blocks of H and O, shared by the per-k and the
// grouped kernels.
//
//  H(N+lo, i)  = sum_f loa_a(lo, f) A_a(i, f)          (hamiltonsetup.f90:131-145)
//  H(i, N+lo)  = conj(H(N+lo, i))                         (hamiltonsetup.f90:147-149)
//  O(i, N+lo)  = sum_io conj(A_a(i, io, lm)) oalo(io, ilo) (overlapsetup.f90:119-131)
//  O(N+lo, i)  = conj(O(i, N+lo))
//  H(lo, lo')  = lolo_a block on the atom diagonal, 0 elsewhere (hamiltonsetup.f90:154-161)
//  O(lo, lo')  = ololo(ilo, ilo') for equal atom, l and m (overlapsetup.f90:136-148)
// with the strict lower triangle of the lo-lo block set to conj(upper) as
// hamiltonoverlapocopy_UL.f90:15-27 leaves it.
#pragma once
#include "exc_common.h"

namespace lo_dev {

constexpr int kMaxLo = 16;          // lo functions per atom supported
constexpr int kRows = 64;           // APW rows (G+k) per workgroup: one wave's lanes
constexpr int kWaves = 8;           // waves of a workgroup, each summing its share of f
constexpr int kThreads = 64 * kWaves;
constexpr int kChunk = 4;           // lo functions reduced through LDS at a time

// One workgroup = 64 rows of one atom (lane = row) or, blockIdx.x = 0, the atom's columns of
// the lo-lo block (one launch for both).  The sum over the atom's naa APW functions is split
// over 8 waves and added in wave order through LDS, kChunk lo functions at a time; A's loads
// are one 1 KiB row segment per f and wave, the loa coefficients wave-uniform (scalar loads).
// The kernel is bound by reading A once; at small N by the chain of its loads, which the
// split over f shortens (one thread per row summing all of f, after one thread had scanned
// the lo table: 113 us at N = 97, 2 atoms, 93 us at N = 260, 5 atoms x 8 k-points, 1.26 ms at
// N = 5000, 32 atoms x 8 k-points, now 14 us, 15 us and 1.16 ms).  The (lo, row) elements
// are written with the lo index fastest, kChunk contiguous ones per row.  Products are
// explicit FMAs so that the per-k and the grouped kernels, which inline this body, round
// identically.
struct ApwLoShared {
  cplx red[kWaves][kChunk][kRows];
  cplx fin[2][kRows][kChunk + 1];
};

template <int MAXLO>
__device__ __forceinline__ void lo_apw_body(ApwLoShared &sh, int bx, int ias, int ngp, int naa, int maxnlo, int nlomax,
                                            int apwordmax, const int *__restrict__ dlo, const lo_desc *__restrict__ lod,
                                            const cplx *__restrict__ apwalm, int ldg, const cplx *__restrict__ loa,
                                            const double *__restrict__ oalo, const double *__restrict__ h1loa,
                                            cplx *__restrict__ h, cplx *__restrict__ o, int ldh) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int first = dlo[2 * ias], cnt = dlo[2 * ias + 1];
  const int row0 = bx * kRows;
  if (cnt == 0 || row0 >= ngp) return;              // uniform over the workgroup
  const int i = row0 + lane;
  const cplx *A = apwalm + (size_t)ldg * naa * ias;
  const cplx *la = loa + (size_t)maxnlo * naa * ias;
  double hr[MAXLO], hi[MAXLO];
#pragma unroll
  for (int q = 0; q < MAXLO; ++q) hr[q] = hi[q] = 0.0;
  if (h) {
    const int per = (naa + kWaves - 1) / kWaves;
    const int f1 = min(naa, (wave + 1) * per);
    const cplx *Ai = A + min(i, ngp - 1);            // rows past N read a valid row, never stored
#pragma unroll 4
    for (int f = wave * per; f < f1; ++f) {
      const cplx a = Ai[(size_t)f * ldg];
#pragma unroll
      for (int q = 0; q < MAXLO; ++q) {
        if (q < cnt) {
          const cplx w = la[q + (size_t)maxnlo * f];   // loa row q of the atom = its q-th lo function
          hr[q] = fma(w.re, a.re, hr[q]);
          hr[q] = fma(-w.im, a.im, hr[q]);
          hi[q] = fma(w.re, a.im, hi[q]);
          hi[q] = fma(w.im, a.re, hi[q]);
        }
      }
    }
  }
  const size_t nlo0 = (size_t)ngp + first;
#pragma unroll
  for (int c0 = 0; c0 < MAXLO; c0 += kChunk) {
    if (c0 >= cnt) break;
#pragma unroll
    for (int q = 0; q < kChunk; ++q) sh.red[wave][q][lane] = cplx{hr[c0 + q], hi[c0 + q]};
    __syncthreads();
    // (row, lo), contiguous over the rows: O primary, H = conj(H(lo, row)).  Waves 0 .. 3 add
    // up H's partial sums, waves 4 .. 7 form O's element, one lo function each.  h or o is
    // null when only the other matrix is set up (a uniform branch).
    const int q = wave & 3, lo = c0 + q;
    if (lo < cnt) {
      const size_t rl = (size_t)i + (nlo0 + lo) * ldh;
      if (wave < 4) {
        cplx v = sh.red[0][q][lane];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) {
          v.re += sh.red[w][q][lane].re;
          v.im += sh.red[w][q][lane].im;
        }
        sh.fin[0][lane][q] = v;
        if (h && i < ngp) h[rl] = cplx{v.re, -v.im};
      } else {
        const lo_desc dq = lod[first + lo];
        double orr = 0.0, oi = 0.0;
        if (i < ngp) {
          for (int io = 0; io < apwordmax; ++io) {
            const cplx a = A[i + (size_t)(io + apwordmax * dq.lm) * ldg];
            // oalo + h1loa ('iora*', overlapsetup.f90:126; h1loa is zero otherwise)
            const size_t wi = io + apwordmax * (dq.ilo + nlomax * ias);
            const double w = h1loa ? oalo[wi] + h1loa[wi] : oalo[wi];
            orr = fma(a.re, w, orr);
            oi = fma(-a.im, w, oi);
          }
          if (o) o[rl] = cplx{orr, oi};
        }
        sh.fin[1][lane][q] = cplx{orr, -oi};
      }
    }
    __syncthreads();
    // (lo, row): H primary (loa . A^T), O = conj(O(row, lo)); kChunk lo functions of a row
    // from consecutive lanes
    const int t = threadIdx.x & 255, r = t / kChunk, qq = t % kChunk;
    cplx *out = threadIdx.x < 256 ? h : o;
    if (out && row0 + r < ngp && c0 + qq < cnt)
      out[(nlo0 + c0 + qq) + (size_t)(row0 + r) * ldh] = sh.fin[threadIdx.x < 256 ? 0 : 1][r][qq];
  }
}

__device__ __forceinline__ void lo_lo_body(int r, int c, int ngp, int nlotot, int maxnlo, int nlomax,
                                           const lo_desc *__restrict__ lod, const cplx *__restrict__ lolo,
                                           const double *__restrict__ ololo, const double *__restrict__ h1lolo,
                                           cplx *__restrict__ h, cplx *__restrict__ o, int ldh) {
  const lo_desc dr = lod[r], dc = lod[c];
  cplx hv = {0.0, 0.0}, ov = {0.0, 0.0};
  if (dr.ias == dc.ias) {
    const cplx *ll = lolo + (size_t)maxnlo * maxnlo * dr.ias;
    if (r <= c) {
      hv = ll[dr.row + maxnlo * dc.row];
    } else {
      const cplx t = ll[dc.row + maxnlo * dr.row];
      hv = cplx{t.re, -t.im};
    }
    if (dr.l == dc.l && dr.m == dc.m) {
      // ololo + h1lolo ('iora*', overlapsetup.f90:144)
      const size_t base = (size_t)nlomax * nlomax * dr.ias;
      const size_t oi = base + ((r <= c) ? dr.ilo + nlomax * dc.ilo : dc.ilo + nlomax * dr.ilo);
      ov.re = h1lolo ? ololo[oi] + h1lolo[oi] : ololo[oi];
    }
  }
  const size_t idx = (size_t)(ngp + r) + (size_t)(ngp + c) * ldh;
  if (h) h[idx] = hv;
  if (o) o[idx] = ov;
}

// the lo-lo block's columns of atom ias, all rows, by one workgroup
__device__ __forceinline__ void lo_lo_atom(int ias, const int *__restrict__ dlo, int ngp, int nlotot, int maxnlo,
                                           int nlomax, const lo_desc *__restrict__ lod, const cplx *__restrict__ lolo,
                                           const double *__restrict__ ololo, const double *__restrict__ h1lolo,
                                           cplx *__restrict__ h, cplx *__restrict__ o, int ldh) {
  const int first = dlo[2 * ias], cnt = dlo[2 * ias + 1];
  for (int c = 0; c < cnt; ++c)
    for (int r = threadIdx.x; r < nlotot; r += kThreads)
      lo_lo_body(r, first + c, ngp, nlotot, maxnlo, nlomax, lod, lolo, ololo, h1lolo, h, o, ldh);
}

}  // namespace lo_dev
