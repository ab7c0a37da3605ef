// Adjoint (vector-Jacobian product) of the setup on gfx950: dL/dtau and dL/dV(G) of
// L = Re sum_ij (D_ji H_ij + W_ji O_ij) for cotangents of rank nst,
//   D = C diag(wh) C^H,   W = C diag(wo) C^H,
// which with wh = w_k f and wo = -w_k f e is the k-point's contribution to dE/dtau, i.e.
// minus forcek's IBS force (forcek.f90:267-383, F = -dE/dtau).
//
// With q_i = G_i + k, U = C_apw^T A and, per atom a (columns of A_a) and state n,
//   Z_nf = wh_n ((h_a U_n)_f + sum_{lo j of a} C_jn conj(loa_jf))
//        + wo_n (U_nf + sum_{lo j of a, lm_j = lm_f} C_jn oalo(io_f, ilo_j)),
//  MT         :  2 sum_G q_l(G) sum_n Im(conj(C_Gn) sum_f conj(A_Gf) Z_nf)
//  Theta(G)   :  sum_ij (q_il - q_jl) Im(-ffac_a(G_i-G_j) conj(S_ia) S_ja (dp_ij D_ji + W_ji))
//                (the tau dependence of Theta(G) = delta_G0 - sum_a exp(-iG.r_a) ffac_a(G))
//  dL/dV(g)   =  sum_{ij: G_i - G_j = g} D_ji  (holomorphic partial over the full matrix)
// The MT line is one product with A for U and one back (the derivative's factor q_l sits on the
// G side, so the three directions share it): vjp_back_kernel forms sum_f conj(A) Z on FP64 MFMA
// tiles and contracts it with q_l conj(C) in its epilogue, storing nothing.  The Theta and V
// lines need D and W over pairs only through their sums per G_i - G_j = g: dw_kernel adds
// D_ji and dp_ij D_ji + W_ji of the upper triangle into per-g sums (the other triangle is the
// conjugate at -g), theta_kernel then walks the few 10^4 g instead of every pair for every atom.
// Measured, 16 atoms, N = 2500, 64 states (us): U 90, back 95, h_a U 21, dw 165, theta 12, the rest 25;
// with a q-scaled library product for each direction, U and V_l together 320, the contraction
// per (atom, state) 119 and the pairs times all atoms with four atomics each 788.
// U and the product back take three real products per complex one (Gauss), which round the imaginary
// parts more than the library's four did; dE/dtau as a whole came closer to 64-bit values all the same (16 atoms, N = 2500:
// 4.0e-15 -> 3.2e-15 relative).
#include "setup_dev.h"
#include "mt_dma.h"

namespace {

using namespace zf64;
using setup_dev::GTab;
using setup_dev::lookup_g;
using setup_dev::DmaCore;

// Z in place of h_a U (hu), both nst x (natm naa) with n fastest
__global__ __launch_bounds__(256) void vjp_z_kernel(int ngp, int nst, int naa, int maxnlo, int nlomax, int apwordmax,
                                                    const int *__restrict__ dlo, const lo_desc *__restrict__ lod,
                                                    const cplx *__restrict__ loa, const double *__restrict__ oalo,
                                                    const cplx *__restrict__ evec, int ldc,
                                                    const double *__restrict__ wh, const double *__restrict__ wo,
                                                    const cplx *__restrict__ u, cplx *__restrict__ hu) {
  const int n = blockIdx.x * 64 + (threadIdx.x & 63), f = blockIdx.y * 4 + (threadIdx.x >> 6), ias = blockIdx.z;
  if (n >= nst || f >= naa) return;
  const size_t at = n + (size_t)nst * (f + (size_t)naa * ias);
  cplx x = hu[at], y = u[at];
  const int first = dlo[2 * ias], cnt = dlo[2 * ias + 1];
  for (int q = first; q < first + cnt; ++q) {
    const lo_desc d = lod[q];
    const cplx c = evec[ngp + q + (size_t)n * ldc];
    const cplx w = loa[d.row + (size_t)maxnlo * (f + (size_t)naa * ias)];
    x.re += c.re * w.re + c.im * w.im;              // C conj(loa)
    x.im += c.im * w.re - c.re * w.im;
    if (d.lm == f / apwordmax) {
      const double o = oalo[f % apwordmax + apwordmax * (d.ilo + nlomax * ias)];
      y.re += c.re * o;
      y.im += c.im * o;
    }
  }
  hu[at] = cplx{wh[n] * x.re + wo[n] * y.re, wh[n] * x.im + wo[n] * y.im};
}

// sum over the workgroup's W waves of 3 values, added to out[0..2] times fac
template <int W>
__device__ __forceinline__ void add3(double (&acc)[3], double (&red)[W][3], double fac, double *out) {
#pragma unroll
  for (int l = 0; l < 3; ++l) {
    double v = acc[l];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][l] = v;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    double v = 0.0;
#pragma unroll
    for (int w = 0; w < W; ++w) v += red[w][threadIdx.x];
    atomicAdd(out + threadIdx.x, fac * v);
  }
}

// one 64 x 64 tile (G, state) of sum_f conj(A_a(G, f)) Z_a(n, f) (the muffin-tin tile's LDS-DMA
// core), contracted with q_l conj(C)
__global__ __launch_bounds__(512) void vjp_back_kernel(int ngp, int nst, int naa, const cplx *__restrict__ apwalm,
                                                       int ldg, const cplx *__restrict__ z,
                                                       const cplx *__restrict__ evec, int ldc,
                                                       const double *__restrict__ vgpc, const int *__restrict__ fperm,
                                                       double *__restrict__ dedtau) {
  using C = DmaCore<64, 64, 16, 2, 2, 4, true, true>;
  using St = typename C::Stage;
  EXC_DMA_STAGES(St, 2)
  __shared__ double sr[8][3];
  const int ias = blockIdx.z, row0 = blockIdx.x * 64, col0 = blockIdx.y * 64;
  d4_t cr[C::MB][C::NB], ci[C::MB][C::NB];
  C::run(EXC_DMA_STAGE_ARGS(St), apwalm + (size_t)ldg * naa * ias, ldg, row0, ngp, z + (size_t)nst * naa * ias, nst,
         col0, nst, naa, fperm, cr, ci);
  const int wave = threadIdx.x >> 6, wr = wave / 4, wc = wave % 4;
  double acc[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int i = 0; i < C::MB; ++i)
#pragma unroll
    for (int j = 0; j < C::NB; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = row0 + C::row_of(wr, i, v), n = col0 + C::col_of(wc, j);
        if (r >= ngp || n >= nst) continue;
        const cplx c = evec[r + (size_t)n * ldc];
        const double t = c.re * ci[i][j][v] - c.im * cr[i][j][v];      // Im(conj(C) B)
#pragma unroll
        for (int l = 0; l < 3; ++l) acc[l] += vgpc[3 * r + l] * t;
      }
  add3<8>(acc, sr, 2.0, dedtau + 3 * ias);
}

// ---------------------------------------------------------------------------------------
// dw: tiles of D^T (i,j) = D_ji and W^T over the upper triangle of the APW block
// ---------------------------------------------------------------------------------------
constexpr int DBM = 64, DBK = 16;
using DCore = Core<DBM, DBM, DBK, 2, 2, true>;

// The basis is taken in the order of its position in the G box, lines along the box's longest
// axis first (perm): a 64 x 64 tile then covers a handful of line segments on either side,
// whose pairs share their differences (about 600 different g for 4096 pairs).  The pairs of a
// tile are added up per (row line, column line, difference along the line) in LDS and each
// sum goes to memory once: straight atomics per pair took 460 us where the products take 50
// (N = 2500).  A tile with more than kSlots such sums (a basis of short lines) adds its
// pairs directly.
constexpr int kSlots = 1024;

// keys: position in the G box with axis ax fastest; the per-g sums and pairs cleared
__global__ __launch_bounds__(256) void vjp_clear_kernel(int ngp, const int *__restrict__ igpig, GTab gt, int ax,
                                                        int *__restrict__ key, double *__restrict__ s,
                                                        unsigned long long *__restrict__ rep) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < gt.ngvec) {
#pragma unroll
    for (int q = 0; q < 4; ++q) s[q * (size_t)gt.ngvec + i] = 0.0;
    rep[i] = ~0ull;
  }
  if (i < ngp) {
    const int *g = gt.ivg + 3 * (igpig[i] - 1);
    const int p[3] = {g[0] - gt.lo0, g[1] - gt.lo1, g[2] - gt.lo2}, n[3] = {gt.n0, gt.n1, gt.n2};
    const int b = ax == 2 ? 0 : ax + 1, c = 3 - ax - b;
    key[i] = p[ax] + n[ax] * (p[b] + n[b] * p[c]);
  }
}

// perm[rank of key i] = i (equal keys, a basis with a repeated G, in index order): 64 rows per
// workgroup, the comparisons split over its 16 waves
__global__ __launch_bounds__(1024) void vjp_rank_kernel(int ngp, const int *__restrict__ key, int *__restrict__ perm) {
  __shared__ int cnt[16][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = blockIdx.x * 64 + lane;
  const int k = key[min(i, ngp - 1)], per = (ngp + 15) / 16, j1 = min(ngp, (wave + 1) * per);
  int c = 0;
#pragma unroll 8
  for (int j = wave * per; j < j1; ++j) c += key[j] < k || (key[j] == k && j < i) ? 1 : 0;
  cnt[wave][lane] = c;
  __syncthreads();
  if (wave == 0 && i < ngp) {
    int r = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) r += cnt[w][lane];
    perm[r] = i;
  }
}

// the rows of C in perm's order: as they are, times wh and times wo
__global__ __launch_bounds__(256) void scale_cols_kernel(int ngp, int nst, const cplx *__restrict__ evec, int ldc,
                                                         const int *__restrict__ perm, const double *__restrict__ wh,
                                                         const double *__restrict__ wo, cplx *__restrict__ ch,
                                                         cplx *__restrict__ cf, cplx *__restrict__ cg) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  const int n = blockIdx.y;
  if (i >= ngp) return;
  const cplx c = evec[perm[i] + (size_t)n * ldc];
  ch[i + (size_t)n * ngp] = c;
  cf[i + (size_t)n * ngp] = cplx{c.re * wh[n], c.im * wh[n]};
  cg[i + (size_t)n * ngp] = cplx{c.re * wo[n], c.im * wo[n]};
}

// per-g sums over the pairs i <= j (in perm's order): s = (D re, D im, X re, X im) per g, X =
// dp D + W, the diagonal with weight 1/2; rep[g] a pair with G_i - G_j = g (any of them: q_i -
// q_j and conj(S_i) S_j are the same for all up to rounding).  sg -1: the pair's difference is
// outside the G set (counted) and its mirror pair's, -g, is taken instead.
struct DwOut {
  double *s;
  unsigned long long *rep;
};
__device__ __forceinline__ void dw_add(const DwOut &o, const GTab &gt, int d0, int d1, int d2, int r, int c, double dr,
                                       double di, double xr, double xi, bool theta) {
  const size_t nv = gt.ngvec;
  double sg = 1.0;
  int ig = lookup_g(gt, d0, d1, d2);
  if (!ig) {
    ig = lookup_g(gt, -d0, -d1, -d2);
    if (!ig) return;
    sg = -1.0;
  }
  double *t = o.s + (ig - 1);
  atomicAdd(t, dr);
  atomicAdd(t + nv, sg * di);
  if (theta) {                                        // the diagonal (G = 0) has no Theta term
    atomicAdd(t + 2 * nv, xr);
    atomicAdd(t + 3 * nv, sg * xi);
    o.rep[ig - 1] = sg > 0.0 ? ((unsigned long long)r << 32) | (unsigned)c : ((unsigned long long)c << 32) | (unsigned)r;
  }
}

// (two workgroups a CU: left to itself the compiler takes 284 registers and one fits; a pass of the 16-atom case at
// N = 2500, two k-points, 587 -> 577 us.  Bound by the LDS atomics of the sums.)
__global__ __launch_bounds__(256, 2) void dw_kernel(int ngp, int nst, const cplx *__restrict__ ch,
                                                 const cplx *__restrict__ cf, const cplx *__restrict__ cg,
                                                 const int *__restrict__ perm, const int *__restrict__ igpig,
                                                 const double *__restrict__ vgpc, GTab gt, int ax, DwOut o) {
  struct Sums {
    double v[4][kSlots];
    int rep[kSlots];
  };
  __shared__ union U {                                // the operands' stage, then the sums
    Smem<DBM, DBM, DBK> sm;
    Sums su;
    __device__ U() {}
  } un;
  __shared__ int s_g[2][DBM][3], s_ix[2][DBM];        // rows, columns: G, index in the caller's basis
  __shared__ double s_q[2][DBM][3];
  __shared__ int s_z0[2][DBM], s_z1[2][DBM], s_n[2];  // first and last position of each line, number of lines
  __shared__ int2 s_slot[2][DBM];                     // see below
  int ti, tj;
  setup_dev::tri_decode(blockIdx.x, ti, tj);
  const int row0 = ti * DBM, col0 = tj * DBM;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wr = wave >> 1, wc = wave & 1;
  int line = 0;
  if (wave < 2) {                                     // wave 0: the rows, wave 1: the columns
    const int idx = (wave ? col0 : row0) + lane;
    const bool in = idx < ngp;
    int g[3] = {0, 0, 0}, ix = 0;
    if (in) {
      ix = perm[idx];
      const int ig = igpig[ix] - 1;
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        g[q] = gt.ivg[3 * ig + q];
        s_q[wave][lane][q] = vgpc[3 * ix + q];
      }
    }
    s_ix[wave][lane] = ix;
#pragma unroll
    for (int q = 0; q < 3; ++q) s_g[wave][lane][q] = g[q];
    const int b = ax == 2 ? 0 : ax + 1, c = 3 - ax - b;
    const int z = ax == 0 ? g[0] : ax == 1 ? g[1] : g[2];
    const int gb = b == 0 ? g[0] : b == 1 ? g[1] : g[2], gc = c == 0 ? g[0] : c == 1 ? g[1] : g[2];
    // a line starts where another coordinate than the fast one changes; positions rise along it
    const int pb = __shfl_up(gb, 1), pc = __shfl_up(gc, 1);
    const bool start = in && (lane == 0 || gb != pb || gc != pc);
    const unsigned long long m = __ballot(start), valid = __ballot(in);
    const unsigned long long upto = lane == 63 ? ~0ull : (1ull << (lane + 1)) - 1;
    line = max(0, __popcll(m & upto) - 1);
    if (start) s_z0[wave][line] = z;
    const bool last = in && (lane == 63 || !((valid >> (lane + 1)) & 1) || ((m >> (lane + 1)) & 1));
    if (last) s_z1[wave][line] = z;
    if (lane == 0) s_n[wave] = __popcll(m);
  }
  __syncthreads();
  // slots: for row line a, column line b the differences z_r - z_c from z0_a - z1_b to z1_a - z0_b,
  // a-major.  With the widths w = z1 - z0 a pair's slot is s_slot[0][r].x + b w_a + s_slot[1][c].x,
  // (.y: w_a for a row, b for a column)
  const int na = s_n[0], nb = s_n[1];
  int wsum = 0, total = 0;                            // sum of the column lines' w + 1; number of slots
  for (int b = 0; b < nb; ++b) wsum += s_z1[1][b] - s_z0[1][b] + 1;
  for (int a = 0; a < na; ++a) total += nb * (s_z1[0][a] - s_z0[0][a]) + wsum;
  const bool lds = total <= kSlots;                   // uniform
  if (wave < 2) {
    const int z = s_g[wave][lane][ax];
    int x = 0;
    if (wave == 0)
      for (int a = 0; a < line; ++a) x += nb * (s_z1[0][a] - s_z0[0][a]) + wsum;
    else
      for (int b = 0; b < line; ++b) x += s_z1[1][b] - s_z0[1][b] + 1;
    s_slot[wave][lane] = wave == 0 ? make_int2(x + z - s_z0[0][line], s_z1[0][line] - s_z0[0][line])
                                   : make_int2(x - z + s_z1[1][line], line);
  }
  // D^T tile: out(i, j) = sum_n conj(C_in wh_n) C_jn;  W^T with wo
  DCore cd, cw;
  cd.run(un.sm, cf, ngp, row0, ngp, ch, ngp, col0, ngp, nst, nullptr);
  cw.run(un.sm, cg, ngp, row0, ngp, ch, ngp, col0, ngp, nst, nullptr);
  __syncthreads();
  if (lds) {
    for (int e = tid; e < total; e += 256) {
      un.su.rep[e] = -1;
#pragma unroll
      for (int q = 0; q < 4; ++q) un.su.v[q][e] = 0.0;
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < DCore::MB; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int rl = DCore::row_of(wr, i, v), r = row0 + rl;
      const int2 sr = s_slot[0][rl];
#pragma unroll
      for (int j = 0; j < DCore::NB; ++j) {
        const int cl = DCore::col_of(wc, j), c = col0 + cl;
        if (r > c || c >= ngp) continue;
        const double w = r == c ? 0.5 : 1.0;
        const double dr = w * cd.cr[i][j][v], di = w * cd.ci[i][j][v];
        const double dp = 0.5 * (s_q[0][rl][0] * s_q[1][cl][0] + s_q[0][rl][1] * s_q[1][cl][1] + s_q[0][rl][2] * s_q[1][cl][2]);
        const double xr = dp * dr + cw.cr[i][j][v], xi = dp * di + cw.ci[i][j][v];
        if (lds) {
          const int2 sc = s_slot[1][cl];
          const int slot = sr.x + sc.y * sr.y + sc.x;
          atomicAdd(&un.su.v[0][slot], dr);
          atomicAdd(&un.su.v[1][slot], di);
          if (r < c) {
            atomicAdd(&un.su.v[2][slot], xr);
            atomicAdd(&un.su.v[3][slot], xi);
          }
          un.su.rep[slot] = rl * DBM + cl;            // any of the slot's pairs
        } else {
          dw_add(o, gt, s_g[0][rl][0] - s_g[1][cl][0], s_g[0][rl][1] - s_g[1][cl][1], s_g[0][rl][2] - s_g[1][cl][2],
                 s_ix[0][rl], s_ix[1][cl], dr, di, xr, xi, r < c);
        }
      }
    }
  if (!lds) return;
  __syncthreads();
  for (int e = tid; e < total; e += 256) {
    const int p = un.su.rep[e];
    if (p < 0) continue;
    const int rl = p / DBM, cl = p % DBM;
    dw_add(o, gt, s_g[0][rl][0] - s_g[1][cl][0], s_g[0][rl][1] - s_g[1][cl][1], s_g[0][rl][2] - s_g[1][cl][2],
           s_ix[0][rl], s_ix[1][cl], un.su.v[0][e], un.su.v[1][e], un.su.v[2][e], un.su.v[3][e],
           row0 + rl < col0 + cl);
  }
}

// per g: dL/dV(g) += S(g) + conj(S(-g)) (by the workgroups of atom 0), and atom y's Theta term
__global__ __launch_bounds__(256) void theta_kernel(const double *__restrict__ s,
                                                    const unsigned long long *__restrict__ rep,
                                                    const double *__restrict__ vgpc, const cplx *__restrict__ sfacgp,
                                                    int ldg, const int *__restrict__ spidx,
                                                    const double *__restrict__ ffacg, GTab gt,
                                                    double *__restrict__ dedtau, double *__restrict__ dedv) {
  __shared__ double sr[4][3];
  const int g = blockIdx.x * 256 + threadIdx.x, a = blockIdx.y;
  const size_t nv = gt.ngvec;
  double acc[3] = {0.0, 0.0, 0.0};
  if (g < gt.ngvec) {
    const int a0 = -gt.ivg[3 * g] - gt.lo0, a1 = -gt.ivg[3 * g + 1] - gt.lo1, a2 = -gt.ivg[3 * g + 2] - gt.lo2;
    int m = 0;                                        // -g in the set (1-based), 0 if not
    if ((unsigned)a0 < (unsigned)gt.n0 && (unsigned)a1 < (unsigned)gt.n1 && (unsigned)a2 < (unsigned)gt.n2)
      m = gt.ivgig[a0 + gt.n0 * (a1 + gt.n1 * a2)];
    if (m > gt.ngvec) m = 0;
    if (a == 0) {
      double re = s[g], im = s[nv + g];
      if (m > 0) {
        re += s[m - 1];
        im -= s[nv + m - 1];
      }
      // atomic: calls on other streams may be adding their k-points to the same array
      if (re != 0.0) atomicAdd(dedv + 2 * g, re);
      if (im != 0.0) atomicAdd(dedv + 2 * g + 1, im);
    }
    const unsigned long long pair = rep[g];
    if (pair != ~0ull) {
      const int i = (int)(pair >> 32), j = (int)(pair & 0xffffffffu);
      const cplx si = sfacgp[i + (size_t)ldg * a], sj = sfacgp[j + (size_t)ldg * a];
      // p = conj(S_i) S_j = exp(-i (G_i - G_j).r_a); the term of (i, j) is Im(-ffac p X) and that
      // of (j, i), at -g, the same
      const double pr = si.re * sj.re + si.im * sj.im, pi = si.re * sj.im - si.im * sj.re;
      const double th = -(m > 0 ? 2.0 : 1.0) * ffacg[g + nv * spidx[a]];
      const double v = th * (pr * s[3 * nv + g] + pi * s[2 * nv + g]);
#pragma unroll
      for (int l = 0; l < 3; ++l) acc[l] = (vgpc[3 * i + l] - vgpc[3 * j + l]) * v;
      if (a == 0 && m <= 0 && gt.miss) atomicAdd(gt.miss, 1u);   // the mirror pairs are outside the G set
    }
  }
  add3<4>(acc, sr, 1.0, dedtau + 3 * a);
}

}  // namespace

// work: exc_vjp_work_elems(d, ngp, nst) elements; yv: the Y-stage variant for h_a U
int exc_launch_vjp(const exc_dev &d, int ngp, int nst, const cplx *apwalm, int ldg, const int *igpig,
                   const double *vgpc, const cplx *sfacgp, const cplx *evec, int ldc, const double *wh,
                   const double *wo, cplx *work, double *dedtau, double *dedv, int ncu, int yv, hipStream_t s) {
  if (ngp <= 0 || nst <= 0) return EXC_OK;
  if (nst > 65535) return EXC_ERR_ARG;
  if (d.naa > 256 || d.nlotot > 256) return EXC_ERR_UNSUPPORTED;
  const int ktot = d.natm * d.naa;
  cplx *u = work, *hu = u + (size_t)nst * ktot;        // nst x K each
  cplx *ch = hu + (size_t)nst * ktot;                  // ngp x nst each
  cplx *cf = ch + (size_t)ngp * nst, *cg = cf + (size_t)ngp * nst;
  double *sums = (double *)(cg + (size_t)ngp * nst);   // 4 ngvec
  unsigned long long *rep = (unsigned long long *)(sums + 4 * (size_t)d.ngvec);
  int *key = (int *)(rep + d.ngvec), *perm = key + ngp;
  const GTab gt = setup_dev::make_gtab(d);
  int rc;
  if ((rc = exc_launch_xty(1, ngp, apwalm, ldg, ktot, 0, evec, ldc, nst, 0, u, nst, 0, true, ncu, s))) return rc;
  if ((rc = exc_launch_ystage(d, nst, u, nst, hu, nst, yv, s))) return rc;
  hipLaunchKernelGGL(vjp_z_kernel, dim3((nst + 63) / 64, (d.naa + 3) / 4, d.natm), dim3(256), 0, s, ngp, nst, d.naa,
                     d.maxnlo, d.nlomax, d.apwordmax, d.dm_lo, d.lod, d.loa, d.oalo, evec, ldc, wh, wo, u, hu);
  EXC_CHECK(hipGetLastError());
  hipLaunchKernelGGL(vjp_back_kernel, dim3((ngp + 63) / 64, (nst + 63) / 64, d.natm), dim3(512), 0, s, ngp, nst, d.naa,
                     apwalm, ldg, hu, evec, ldc, vgpc, d.fperm, dedtau);
  EXC_CHECK(hipGetLastError());
  const int ax = d.box_n[0] >= d.box_n[1] ? (d.box_n[0] >= d.box_n[2] ? 0 : 2) : (d.box_n[1] >= d.box_n[2] ? 1 : 2);
  hipLaunchKernelGGL(vjp_clear_kernel, dim3((std::max(d.ngvec, ngp) + 255) / 256), dim3(256), 0, s, ngp, igpig, gt, ax,
                     key, sums, rep);
  EXC_CHECK(hipGetLastError());
  hipLaunchKernelGGL(vjp_rank_kernel, dim3((ngp + 63) / 64), dim3(1024), 0, s, ngp, key, perm);
  EXC_CHECK(hipGetLastError());
  hipLaunchKernelGGL(scale_cols_kernel, dim3((ngp + 255) / 256, nst), dim3(256), 0, s, ngp, nst, evec, ldc, perm, wh, wo,
                     ch, cf, cg);
  EXC_CHECK(hipGetLastError());
  const int nt = (ngp + DBM - 1) / DBM;
  hipLaunchKernelGGL(dw_kernel, dim3(nt * (nt + 1) / 2), dim3(256), 0, s, ngp, nst, ch, cf, cg, perm, igpig, vgpc, gt, ax,
                     DwOut{sums, rep});
  EXC_CHECK(hipGetLastError());
  hipLaunchKernelGGL(theta_kernel, dim3((d.ngvec + 255) / 256, d.natm), dim3(256), 0, s, sums, rep, vgpc, sfacgp, ldg,
                     d.spidx, d.ffacg, gt, dedtau, dedv);
  EXC_CHECK(hipGetLastError());
  return EXC_OK;
}

// U and h U (nst x K each), the three copies of C (ngp x nst each), the per-g sums and pairs, the
// order of the basis
size_t exc_vjp_work_elems(const exc_dev &d, int ngp, int nst) {
  return 2 * (size_t)nst * d.natm * d.naa + 3 * (size_t)ngp * nst + (5 * (size_t)d.ngvec + 1) / 2 + ((size_t)ngp + 1) / 2;
}
