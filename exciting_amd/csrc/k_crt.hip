// Modular split of the muffin-tin contraction on gfx950 (EXC_BATCH_SPLIT_CRT).
//
// H_MT = conj(A) Yt^T (and O_MT = conj(A) A^T) from exact integer products instead of FP64
// MFMA, the other terms of the setup staying FP64.  The plain FP64 path takes the same route at
// large sizes with 16 moduli (beta = 57, exc_setup_batched_dev's exact_pays); rows the integers cannot
// represent (not finite, norms outside 1e-125 .. 1e145) are marked and their tiles left to
// FP64 MFMA (bmt_fix_kernel).  An element then enters with an absolute error of 2^-58 of the power of
// two above its row's norm: with all its 53 bits down to 2^-4 of the norm, with 45 at 2^-12, about the
// median element of an lmax 10 basis.  The sums are exact, so H_ij is within 2^-56 sqrt(2K) |A_i| |Yt_j|
// and one rounding: a bound relative to the rows' norms, not to H_ij.  (8 atoms, lmax 10, N = 260, against 80-bit
// sums, per |A_i| |Yt_j|: rms 7e-18, largest 2.3e-17; FP64 products 3.3e-17, 1.4e-16; 5 of 100
// elements come out further off than by FP64, the smallest of a row by up to a digit of their own.)
//
// The steps:
//
//  scale : per row i of an operand X (N x K complex, K = natm naa) the exponent e_i with
//          |X_i|_2 < 2^e_i and s_i = beta - e_i, beta the largest with 2^(2 beta + 2) <= P,
//          P = m_0 ... m_(n-1) the product of the pairwise coprime moduli (241, 233, 229, ...).
//  split : X'_ik = rint(Re X_ik 2^s_i) + i rint(Im X_ik 2^s_i), exact integers below 2^beta.
//          Every modulus m is odd with prime factors 1 mod 4, so it has a square root iota of
//          -1 and Z_m[i] splits into two copies of Z_m by the ring maps x + iy -> x +- iota y.
//          Per modulus the two planes of an operand are those maps, as int8 residues (within
//          m / 2 + 2 of zero, lowres): Re X' - iota Im X' and Re X' + iota Im X' for the conjugated left operand,
//          Re X' + iota Im X' and Re X' - iota Im X' for the right one; layout
//          [m][plane][K/16][row][16 bytes]: one 16-byte k-chunk of 64 consecutive rows is one
//          1 KiB wave-wide DMA.
//  gemm  : per modulus, tile and map, U = u_a u_b^T or V = v_a v_b^T by
//          v_mfma_i32_32x32x32_i8 with exact int32 accumulation (|P| <= K 122^2 < 2^31),
//          reduced modulo m to int8 residues: two real products per modulus, where Gauss's
//          form needs three.
//  merge : per tile element Re = (U + V)/2, Im = (U - V)/(2 iota) modulo each m, then
//          Garner's mixed-radix digits of Re', Im' in [-(P-1)/2, (P-1)/2] (exact:
//          |Re'|, |Im'| <= |A'_i| |B'_j| < P/2), the FP64 value correctly rounded as
//          fma(x_hi, M_6, x_lo), times 2^-(s_i + t_j); then the interstitial term and the
//          Hermitian mirror exactly as the FP64 epilogue (hmlistln.f90:74-84,
//          olpistln.f90:69-82, hamiltonoverlapocopy_UL.f90:15-27).
// Integer sums do not depend on their order, so every variant of every kernel gives the
// same bits; the only rounding between the inputs and H_MT is that of the operands to
// beta-bit integers and the final conversion.
//
// Gram form (the default where it applies): with a shift sigma >= -min lambda(h_a) and h_a +
// sigma = L_a L_a^H, E_a = A_a conj(L_a) (the Y stage on that table instead of h_a, k_gram.hip)
// gives conj(E) E^T = conj(A) (h + sigma) A^T = H_MT + sigma O_APW, so
// H_MT = conj(E) E^T - sigma O_APW with O_APW the FP64 addition-theorem overlap (O minus
// its interstitial term).  One operand is split instead of two, and the right operand's
// planes are the left's swapped, as for O = conj(A) A^T; merge items of this form carry
// which = 2.
#include "setup_dev.h"
#include "mt_dma.h"

namespace {

using setup_dev::GTab;
using setup_dev::stage_barrier;
using setup_dev::wait_vm_lgkm0;

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void;

// symmetric residue of an exact integer held in a double, |x| < 2^52, modulo an odd m
// (|x/m| is never within 1/(2m) of a half-integer, far above the rounding of x/m)
__device__ __forceinline__ int dres(double x, int m, double minv) { return (int)fma(-(double)m, rint(x * minv), x); }

// ---------------------------------------------------------------------------------------
// scale: the per-row exponents s = beta - e, |X_i| < 2^e, of Yt, and of A when the caller
// supplies apwalm (with the grouped match, crt_expo_kernel sums A's from the norms the match
// wrote): one workgroup per (k, 64 rows); each of its 16 waves sums |x|^2 over a part of K, the
// parts added in wave order (a fixed order: the exponents do not depend on timing).  Bound by
// reading X; 16 waves since a batch of small k-points has few row blocks (N = 1200, 8
// k-points: 152 workgroups; 241 us with 4 waves, 86 us with 16; N = 5000, 32 atoms, 8 k-points
// 1.13 -> 0.87 ms, 5.7 TB/s).
// ---------------------------------------------------------------------------------------
constexpr int kScaleWaves = 16;

__global__ __launch_bounds__(64 * kScaleWaves) void crt_scale_kernel(const kdesc *__restrict__ ks, int ktot, int beta,
                                                                     int op, int exact) {
  const kdesc k = ks[blockIdx.z];             // op 0: A (apwalm), 1: Yt, 2: E (in Yt's place) as the left operand
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = blockIdx.x * 64 + lane;
  __shared__ double part[kScaleWaves][64];
  __shared__ int some[64];                    // the row has a nonzero value
  if (blockIdx.x * 64 >= k.cnp) return;       // uniform over the workgroup
  if (wave == 0) some[lane] = 0;
  const cplx *src = op ? k.yt : k.apwalm;
  const int ld = op ? k.ldy : k.ldg;
  const int kq = (ktot + kScaleWaves - 1) / kScaleWaves, k0 = wave * kq, k1 = min(ktot, k0 + kq);   // op 2 writes xa
  double acc = 0.0;
  bool nz = false;
  if (row < k.ngp) {
#pragma unroll 8
    for (int c = k0; c < k1; ++c) {
      const cplx v = src[row + (size_t)c * ld];
      acc = fma(v.re, v.re, acc);
      acc = fma(v.im, v.im, acc);
      nz = nz || v.re != 0.0 || v.im != 0.0;
    }
  }
  part[wave][lane] = acc;
  __syncthreads();
  if (nz) some[lane] = 1;
  __syncthreads();
  if (wave == 0) {
    double s2 = 0.0;
#pragma unroll
    for (int w = 0; w < kScaleWaves; ++w) s2 += part[w][lane];
    int e = 0;
    if (s2 > 0.0) frexp(sqrt(s2), &e);       // |X_i| < 2^e
    int x = beta - e;
    // not finite, or so large or small that the squares' sum is not the norm's
    if (exact && (!(s2 < 1e290) || (s2 < 1e-250 && some[lane]))) x = kBadRow;
    (op == 1 ? k.xy : k.xa)[row] = row < k.ngp ? x : 0;
  }
}

// A's exponents from the squared norms per (atom, row) that the grouped match wrote (in
// closed form), summed in atom order: no pass over A.  One thread per row.
__global__ __launch_bounds__(256) void crt_expo_kernel(const kdesc *__restrict__ ks, int natm, int beta, int exact) {
  const kdesc k = ks[blockIdx.z];
  const int row = blockIdx.x * 256 + threadIdx.x;
  if (row >= k.cnp) return;
  double s2 = 0.0;
  if (row < k.ngp)
    for (int a = 0; a < natm; ++a) s2 += k.pa2[(size_t)a * k.cnp + row];
  int e = 0;
  if (s2 > 0.0) frexp(sqrt(s2), &e);
  const int x = exact && !(s2 < 1e290 && s2 > 1e-250) ? kBadRow : beta - e;
  k.xa[row] = row < k.ngp ? x : 0;
}

// ---------------------------------------------------------------------------------------
// split: 4 waves; wave w of workgroup (bx, by) converts rows 64 bx .. +63 of k-chunk
// 4 by + w (16 values of k) into the residue planes of every modulus
// ---------------------------------------------------------------------------------------
// the low bytes of four ints as one word (byte 0 from a)
__device__ __forceinline__ unsigned pack4(int a, int b, int c, int d) {
  return __builtin_amdgcn_perm((unsigned)b, (unsigned)a, 0x0c0c0400u) |
         __builtin_amdgcn_perm((unsigned)d, (unsigned)c, 0x04000c0cu);
}

// the four balanced 16-bit limbs of an integer |x| < 2^58 held in a double, two a word, from the
// lowest up: each in [-2^15, 2^15), the carries exact (x / 2^16 + 1/2 rounds only where its
// sum leaves x / 2^16's binade, and then not past an integer)
__device__ __forceinline__ void limbs(double x, int (&w)[2]) {
  const double h1 = floor(fma(x, 0x1p-16, 0.5)), l0 = fma(-h1, 0x1p16, x);
  const double h2 = floor(fma(h1, 0x1p-16, 0.5)), l1 = fma(-h2, 0x1p16, h1);
  const double h3 = floor(fma(h2, 0x1p-16, 0.5)), l2 = fma(-h3, 0x1p16, h2);
  w[0] = __builtin_amdgcn_perm((unsigned)(int)l1, (unsigned)(int)l0, 0x05040100u);
  w[1] = __builtin_amdgcn_perm((unsigned)(int)h3, (unsigned)(int)l2, 0x05040100u);
}

typedef short s16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ int dot2(int a, int b, int c) {
  return __builtin_amdgcn_sdot2(__builtin_bit_cast(s16x2, a), __builtin_bit_cast(s16x2, b), c, false);
}

// a residue of |t| < 2^25 modulo m in the low byte (the upper ones are not part of it): t - q m
// with q = rint(t / m) in the low bits of the float 1.5 2^23 + q, whose other bits are a multiple
// of 2^22 and drop out modulo 256.  |t - q m| <= m / 2 + 2: the float quotient is within 1/64 of
// t / m
__device__ __forceinline__ int lowres(int t, int m, float finv) {
  return t - __mul24(__float_as_int(fmaf((float)t, finv, 12582912.0f)), m);
}

// The residue planes of every modulus for 16 values of k of one row: the maps Re X' + sg iota
// Im X' and Re X' - sg iota Im X' (sg = -1 for the conjugated left operand A, +1 for the right
// operand Yt).  Modulo m the parts are sums of four limbs times the residues of 2^0 .. 2^48 (for
// Im X' times iota): |sum| < 4 2^15 120 < 2^24, two v_dot2_i32_i16 each, exact, and their sum and
// difference are reduced once: 14 32-bit operations per complex value and modulus, where reducing
// the integers in FP64 took 11 FP64 ones and 2 conversions.
template <int SG>
__device__ __forceinline__ void split_planes(const int (&xr)[16][2], const int (&xi)[16][2], const CrtTab &t,
                                             signed char *base, size_t pstride, size_t off) {
#pragma unroll 1
  for (int l = 0; l < t.n; ++l) {
    const int m = t.m[l], a0 = t.wr[l][0], a1 = t.wr[l][1], b0 = t.wi[l][0], b1 = t.wi[l][1];
    const float fi = t.finv[l];
    unsigned w[2][4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      int ru[4], rv[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int p = dot2(xr[4 * g + b][0], a0, dot2(xr[4 * g + b][1], a1, 0));
        const int q = dot2(xi[4 * g + b][0], b0, dot2(xi[4 * g + b][1], b1, 0));
        ru[b] = lowres(SG > 0 ? p + q : p - q, m, fi);
        rv[b] = lowres(SG > 0 ? p - q : p + q, m, fi);
      }
      w[0][g] = pack4(ru[0], ru[1], ru[2], ru[3]);
      w[1][g] = pack4(rv[0], rv[1], rv[2], rv[3]);
    }
#pragma unroll
    for (int p = 0; p < 2; ++p)
      *(uint4 *)(base + (size_t)(2 * l + p) * pstride + off) = make_uint4(w[p][0], w[p][1], w[p][2], w[p][3]);
  }
}

// gram: one operand per k-point (grid z = k), E from Yt's buffer into the left planes
__global__ __launch_bounds__(256) void crt_split_kernel(const kdesc *__restrict__ ks, int ktot, int kp, CrtTab t,
                                                        int gram) {
  const kdesc k = ks[gram ? blockIdx.z : blockIdx.z >> 1];
  const int op = gram ? 0 : blockIdx.z & 1;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = blockIdx.x * 64 + lane;
  const int kc = blockIdx.y * 4 + wave;
  if (blockIdx.x * 64 >= k.cnp || kc * 16 >= kp) return;
  const cplx *src = (op || gram) ? k.yt : k.apwalm;
  const int ld = (op || gram) ? k.ldy : k.ldg;
  const int s = row < k.ngp ? (op ? k.xy : k.xa)[row] : 0;
  int xr[16][2], xi[16][2];
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const int c = kc * 16 + q;
    cplx v = {0.0, 0.0};
    if (row < k.ngp && c < ktot) v = src[row + (size_t)c * ld];
    limbs(rint(ldexp(v.re, s)), xr[q]);
    limbs(rint(ldexp(v.im, s)), xi[q]);
  }
  signed char *base = (signed char *)(op ? k.qy : k.qa);
  const size_t pstride = (size_t)kp * k.cnp;            // bytes of one plane
  const size_t off = ((size_t)kc * k.cnp + row) * 16;
  if (op)
    split_planes<1>(xr, xi, t, base, pstride, off);
  else
    split_planes<-1>(xr, xi, t, base, pstride, off);
}

// ---------------------------------------------------------------------------------------
// gemm: one real residue product (tile, modulus, product p) per workgroup on an XCD-mapped
// grid (workgroup b runs on XCD b % 8 and takes the next work of that XCD's contiguous eighth
// of the list; the list keeps the tiles of one (k-point, modulus, product) in 4 x 4 blocks, so
// the workgroups an XCD runs together share their row and column panels in its L2).  BT x BT
// tiles, WR x WC waves with (BT / WR) x (BT / WC) wave tiles of 32 x 32 MFMA blocks, LDS
// stages of BK bytes of k of one plane of both panels, filled by DMA, NST stages in flight.
//   p = 0: U = u_a u_b^T, p = 1: V = v_a v_b^T (the two maps of Z_m[i]), each reduced modulo
//   m to int8 residues; the merge combines them.
// ---------------------------------------------------------------------------------------
template <int BT, int BK, int NST, int WR, int WC>
struct GemmCfg {
  static constexpr int kWaves = WR * WC, kThreads = 64 * kWaves;
  static constexpr int KC = BK / 16;                          // 16-byte k-chunks per stage
  static constexpr int PB = KC * BT * 16;                     // bytes of one panel per stage
  static constexpr int NL = 2 * KC * (BT / 64);               // wave-wide 1 KiB DMAs per stage
  static constexpr int L = NL / kWaves;
  static constexpr int MI = BT / WR / 32, NJ = BT / WC / 32;
  static_assert(NL % kWaves == 0 && BK % 32 == 0 && BT % 64 == 0, "DMA split / MFMA k-step");
  struct __attribute__((aligned(16))) Stage {
    unsigned char a[PB];
    unsigned char b[PB];
  };
};

template <int BT, int BK, int NST, int WR, int WC>
__device__ __forceinline__ void gemm_issue(typename GemmCfg<BT, BK, NST, WR, WC>::Stage *st, const unsigned char *pa,
                                           const unsigned char *pb, size_t chunk_stride, int row0, int col0,
                                           int kc0) {
  using C = GemmCfg<BT, BK, NST, WR, WC>;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
  for (int q = 0; q < C::L; ++q) {
    const int j = wave + C::kWaves * q;               // 0 .. NL-1: (panel, chunk, 64-row quarter)
    const bool isb = j >= C::NL / 2;
    const int jj = isb ? j - C::NL / 2 : j;
    const int h = jj % (BT / 64), kc = jj / (BT / 64);
    const unsigned char *src = (isb ? pb : pa) + (size_t)(kc0 + kc) * chunk_stride +
                               (size_t)((isb ? col0 : row0) + 64 * h + lane) * 16;
    unsigned char *dst = (isb ? st->b : st->a) + kc * (BT * 16) + h * 1024;
    __builtin_amdgcn_global_load_lds((const void *)src, (lds_void *)dst, 16, 0, 0);
  }
}

template <int BT, int BK, int NST, int WR, int WC>
__device__ __forceinline__ void gemm_compute(const typename GemmCfg<BT, BK, NST, WR, WC>::Stage *st,
                                             v16i (&acc)[GemmCfg<BT, BK, NST, WR, WC>::MI][GemmCfg<BT, BK, NST, WR, WC>::NJ],
                                             int wr, int wc) {
  using C = GemmCfg<BT, BK, NST, WR, WC>;
  const int lane = threadIdx.x & 63;
  const int r = lane & 31, hk = lane >> 5;
#pragma unroll
  for (int s = 0; s < BK / 32; ++s) {
    v4i af[C::MI], bf[C::NJ];
#pragma unroll
    for (int i = 0; i < C::MI; ++i)
      af[i] = *(const v4i *)(st->a + ((2 * s + hk) * BT + wr * (32 * C::MI) + 32 * i + r) * 16);
#pragma unroll
    for (int j = 0; j < C::NJ; ++j)
      bf[j] = *(const v4i *)(st->b + ((2 * s + hk) * BT + wc * (32 * C::NJ) + 32 * j + r) * 16);
#pragma unroll
    for (int i = 0; i < C::MI; ++i)
#pragma unroll
      for (int j = 0; j < C::NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[i], bf[j], acc[i][j], 0, 0, 0);
  }
}

template <int BT, int BK, int NST, int WR, int WC, int MINW>
__global__ __launch_bounds__(64 * WR * WC, MINW) void crt_gemm_kernel(const kdesc *__restrict__ ks,
                                                                      const mt_item *__restrict__ items,
                                                                      const int2 *__restrict__ work, int nwork, int kp,
                                                                      CrtTab t, signed char *__restrict__ res) {
  using C = GemmCfg<BT, BK, NST, WR, WC>;
  using St = typename C::Stage;
  EXC_DMA_STAGES(St, NST)
  const int chunk = (nwork + 7) / 8;
  const int x = blockIdx.x % 8, qb = blockIdx.x / 8;
  const int wi = x * chunk + qb;
  if (qb >= chunk || wi >= nwork) return;
  const int2 wk = work[wi];                      // (item, 4 * modulus + product)
  const mt_item it = items[wk.x];
  const kdesc k = ks[it.k];
  const int l = wk.y >> 2, p = wk.y & 3;
  const size_t pstride = (size_t)kp * k.cnp, chunk_stride = (size_t)k.cnp * 16;
  // left operand conj(A): its planes u, v; right operand Yt (H): its planes u, v; or A (O),
  // whose maps as a right operand are the left planes swapped
  const unsigned char *pa = (const unsigned char *)k.qa + (size_t)(2 * l + p) * pstride;
  const unsigned char *pb = it.which ? (const unsigned char *)k.qa + (size_t)(2 * l + 1 - p) * pstride
                                     : (const unsigned char *)k.qy + (size_t)(2 * l + p) * pstride;
  const int row0 = it.ti * BT, col0 = it.tj * BT;
  const int wave = threadIdx.x >> 6, wr = wave / WC, wc = wave % WC;
  v16i acc[C::MI][C::NJ];
#pragma unroll
  for (int i = 0; i < C::MI; ++i)
#pragma unroll
    for (int j = 0; j < C::NJ; ++j) acc[i][j] = v16i{};
  St *st[4] = {&s0_, &s1_, (St *)&s2_, (St *)&s3_};
  const int nsteps = kp / BK;
#pragma unroll
  for (int u = 0; u < NST - 1; ++u)
    if (u < nsteps) gemm_issue<BT, BK, NST, WR, WC>(st[u], pa, pb, chunk_stride, row0, col0, u * C::KC);
  for (int base = 0; base < nsteps; base += NST) {
#pragma unroll
    for (int u = 0; u < NST; ++u) {
      const int step = base + u;
      if (step < nsteps) {
        // stage `step` has landed once at most the DMAs of the NST-2 later stages are out
        if (step + NST - 2 < nsteps)
          wait_vm_lgkm0<(NST - 2) * C::L>();
        else
          wait_vm_lgkm0<0>();
        stage_barrier();
        if (step + NST - 1 < nsteps)
          gemm_issue<BT, BK, NST, WR, WC>(st[(u + NST - 1) % NST], pa, pb, chunk_stride, row0, col0,
                                          (step + NST - 1) * C::KC);
        gemm_compute<BT, BK, NST, WR, WC>(st[u], acc, wr, wc);
      }
    }
  }
  // residues modulo m of one 32 x 32 block and lane are 16 contiguous bytes:
  // res[item][modulus][product][wave][block][lane][16]
  const int m = t.m[l];
  const double mi = t.dminv[l];
  const int lane = threadIdx.x & 63;
  signed char *out = res + (((size_t)wk.x * t.n + l) * 2 + p) * (size_t)(BT * BT);
#pragma unroll
  for (int i = 0; i < C::MI; ++i)
#pragma unroll
    for (int j = 0; j < C::NJ; ++j) {
      unsigned u4[4] = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int v = 0; v < 16; ++v) u4[v >> 2] |= (unsigned)(dres((double)acc[i][j][v], m, mi) & 255) << (8 * (v & 3));
      const int blk = wave * (C::MI * C::NJ) + i * C::NJ + j;
      *(uint4 *)(out + ((size_t)blk * 64 + lane) * 16) = make_uint4(u4[0], u4[1], u4[2], u4[3]);
    }
}

// ---------------------------------------------------------------------------------------
// gemm, register-pipelined form for one wave per SIMD (4 waves, 2 x 2, 128 x 128 wave tiles:
// 8 LDS fragment reads per 16 MFMAs instead of 6 per 8 — the LDS, read by the MFMA operands
// and written by the DMA, bounds the 2 x 4 form).  With no second wave on the SIMD to cover
// the LDS latency, the fragments of MFMA k-step s + 1 are read while the MFMAs of step s run
// (two register sets), and the workgroup barrier that hands an LDS stage over to the DMA is
// taken once per stage, at its last k-step, after its last fragments are in registers:
//   wait for the next stage's DMA | barrier | read its first fragments | half of the DMA into the stage
//   just finished (the other half during the next stage's first k-step) | MFMAs of the last k-step
// so that the next stage's first fragments are in flight during those MFMAs, and a DMA follows every
// fourth MFMA: issued together, the wave waits at the full queue of the L1 instead.  Same
// products, same integer sums, same output layout as crt_gemm_kernel with a 2 x 2 wave grid.
// N = 5000, 32 atoms, 8 k-points, 10 moduli: MFMA alone takes 10.3 ms (1.8 GHz: power), the DMA alone 9.1,
// with the buffers chosen at run time both in turn 19.2, here 15.0; N = 2500, 16 atoms, 16 moduli 4.84 -> 3.70.
// ---------------------------------------------------------------------------------------
template <int BT, int BK, int NST, int WR, int WC>
__device__ __forceinline__ void gemm_frags(const typename GemmCfg<BT, BK, NST, WR, WC>::Stage *st, int s,
                                           v4i (&af)[GemmCfg<BT, BK, NST, WR, WC>::MI],
                                           v4i (&bf)[GemmCfg<BT, BK, NST, WR, WC>::NJ], int wr, int wc) {
  using C = GemmCfg<BT, BK, NST, WR, WC>;
  const int lane = threadIdx.x & 63;
  const int r = lane & 31, hk = lane >> 5;
#pragma unroll
  for (int i = 0; i < C::MI; ++i)
    af[i] = *(const v4i *)(st->a + ((2 * s + hk) * BT + wr * (32 * C::MI) + 32 * i + r) * 16);
#pragma unroll
  for (int j = 0; j < C::NJ; ++j)
    bf[j] = *(const v4i *)(st->b + ((2 * s + hk) * BT + wc * (32 * C::NJ) + 32 * j + r) * 16);
}

template <int BT, int BK, int NST, int WR, int WC>
__device__ __forceinline__ void gemm_mfma(const v4i (&af)[GemmCfg<BT, BK, NST, WR, WC>::MI],
                                          const v4i (&bf)[GemmCfg<BT, BK, NST, WR, WC>::NJ],
                                          v16i (&acc)[GemmCfg<BT, BK, NST, WR, WC>::MI][GemmCfg<BT, BK, NST, WR, WC>::NJ]) {
  using C = GemmCfg<BT, BK, NST, WR, WC>;
#pragma unroll
  for (int i = 0; i < C::MI; ++i)
#pragma unroll
    for (int j = 0; j < C::NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[i], bf[j], acc[i][j], 0, 0, 0);
}

// the L wave-wide DMAs of one stage from per-slot sources fixed for the tile (slot q: panel,
// 16-byte chunk, 64-row quarter), `off` bytes further along k: no address arithmetic at the
// hand-over beyond one add per slot
template <int BT, int BK, int NST, int WR, int WC, int Q0, int Q1>
__device__ __forceinline__ void gemm_issue_pre(typename GemmCfg<BT, BK, NST, WR, WC>::Stage *st, const unsigned char *pak,
                                               const unsigned char *pbk,
                                               const unsigned (&voff)[GemmCfg<BT, BK, NST, WR, WC>::L],
                                               const int (&doff)[GemmCfg<BT, BK, NST, WR, WC>::L]) {
  using C = GemmCfg<BT, BK, NST, WR, WC>;
  static_assert((C::NL / 2) % C::kWaves == 0, "slot q of every wave in one panel");
#pragma unroll
  for (int q = Q0; q < Q1; ++q)
    __builtin_amdgcn_global_load_lds((const void *)((q * C::kWaves >= C::NL / 2 ? pbk : pak) + voff[q]),
                                     (lds_void *)((unsigned char *)st + doff[q]), 16, 0, 0);
}

template <int BT, int BK, int NST, int WR, int WC>
__global__ __launch_bounds__(64 * WR * WC, 1) void crt_gemm_pipe_kernel(const kdesc *__restrict__ ks,
                                                                        const mt_item *__restrict__ items,
                                                                        const int2 *__restrict__ work, int nwork,
                                                                        int kp, CrtTab t, signed char *__restrict__ res) {
  using C = GemmCfg<BT, BK, NST, WR, WC>;
  using St = typename C::Stage;
  constexpr int S = BK / 32;                    // MFMA k-steps per stage
  constexpr int D = C::L / S;                   // DMA slots per k-step
  static_assert(S == 2 && C::L % S == 0 && NST >= 2 && NST <= 4, "register sets alternate within a stage; LDS size");
  EXC_DMA_STAGES(St, NST)
  const int chunk = (nwork + 7) / 8;
  const int x = blockIdx.x % 8, qb = blockIdx.x / 8;
  const int wi = x * chunk + qb;
  if (qb >= chunk || wi >= nwork) return;
  const int2 wk = work[wi];
  const mt_item it = items[wk.x];
  const kdesc k = ks[it.k];
  const int l = wk.y >> 2, p = wk.y & 3;
  const size_t pstride = (size_t)kp * k.cnp, chunk_stride = (size_t)k.cnp * 16;
  const unsigned char *pa = (const unsigned char *)k.qa + (size_t)(2 * l + p) * pstride;
  const unsigned char *pb = it.which ? (const unsigned char *)k.qa + (size_t)(2 * l + 1 - p) * pstride
                                     : (const unsigned char *)k.qy + (size_t)(2 * l + p) * pstride;
  const int row0 = it.ti * BT, col0 = it.tj * BT;
  const int wave = threadIdx.x >> 6, wr = wave / WC, wc = wave % WC;
  v16i acc[C::MI][C::NJ];
#pragma unroll
  for (int i = 0; i < C::MI; ++i)
#pragma unroll
    for (int j = 0; j < C::NJ; ++j) acc[i][j] = v16i{};
  St *st[4] = {&s0_, &s1_, (St *)&s2_, (St *)&s3_};
  const int nsteps = kp / BK;
  // DMA slot q of this wave: panel (A for the first half of the slots), 16-byte k-chunk kc
  // and 64-row quarter h; its source is the panel's base for the stage plus voff[q] (below
  // 2^32: kc < KC, rows < cnp), its destination doff[q] bytes into the stage
  unsigned voff[C::L];
  int doff[C::L];
  {
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int q = 0; q < C::L; ++q) {
      const int j = wv + C::kWaves * q;
      const bool isb = j >= C::NL / 2;
      const int jj = isb ? j - C::NL / 2 : j;
      const int h = jj % (BT / 64), kc = jj / (BT / 64);
      voff[q] = (unsigned)((size_t)kc * chunk_stride + (size_t)((isb ? col0 : row0) + 64 * h + lane) * 16);
      doff[q] = (isb ? C::PB : 0) + kc * (BT * 16) + h * 1024;
    }
  }
  const size_t sstride = (size_t)C::KC * chunk_stride;       // bytes of k per stage
  // stage j's DMA is issued from the hand-over of stage j - NST on (stages 0 .. NST-2 here, the first
  // half of NST-1 at the first hand-over below); stages past the end load the last one again (never read),
  // so that exactly NST - 2 stages' DMA after the next one is in flight at every hand-over
  const size_t klast = (size_t)(nsteps - 1) * sstride;
#pragma unroll
  for (int u = 0; u < NST - 1; ++u) {
    const size_t o = std::min((size_t)u * sstride, klast);
    gemm_issue_pre<BT, BK, NST, WR, WC, 0, C::L>(st[u], pa + o, pb + o, voff, doff);
  }
  v4i fa[2][C::MI], fb[2][C::NJ];
  // hand-over before stage 0
  wait_vm_lgkm0<(NST - 2) * C::L>();
  stage_barrier();
  gemm_frags<BT, BK, NST, WR, WC>(st[0], 0, fa[0], fb[0], wr, wc);
  {
    const size_t o = std::min((size_t)(NST - 1) * sstride, klast);
    gemm_issue_pre<BT, BK, NST, WR, WC, 0, D>(st[NST - 1], pa + o, pb + o, voff, doff);
  }
  // no branch around an MFMA: the accumulators never flow through one (they would be copied between
  // register files), and the scheduler can put one fragment read and one DMA between two MFMAs.  The
  // last stage hands over too (its reads unused).
  size_t koff = std::min((size_t)(NST - 1) * sstride, klast);   // k offset of stage min(step + NST - 1, nsteps - 1)
  auto stage = [&](St *cs, St *ns, St *ps) __attribute__((always_inline)) {
    const size_t kprev = koff;
    koff = koff + sstride < klast ? koff + sstride : klast;    // stage min(step + NST, nsteps - 1)
    // 16 MFMAs, a fragment read after each of the first eight, a DMA after every fourth
    auto order = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < C::MI * C::NJ; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (q < C::MI + C::NJ) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        if (q % 4 == 2 && q / 4 < D) __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
      }
    };
    __builtin_amdgcn_sched_barrier(0);
    gemm_frags<BT, BK, NST, WR, WC>(cs, 1, fa[1], fb[1], wr, wc);
    gemm_issue_pre<BT, BK, NST, WR, WC, D, C::L>(ps, pa + kprev, pb + kprev, voff, doff);
    gemm_mfma<BT, BK, NST, WR, WC>(fa[0], fb[0], acc);
    order();
    __builtin_amdgcn_sched_barrier(0);
    // hand-over: stage step + 1 has landed once at most the DMA of the NST - 2 stages after it is out
    wait_vm_lgkm0<(NST - 2) * C::L>();
    stage_barrier();
    gemm_frags<BT, BK, NST, WR, WC>(ns, 0, fa[0], fb[0], wr, wc);
    gemm_issue_pre<BT, BK, NST, WR, WC, 0, D>(cs, pa + koff, pb + koff, voff, doff);
    gemm_mfma<BT, BK, NST, WR, WC>(fa[1], fb[1], acc);
    order();
  };
  // the stages rotate by name: with a buffer chosen at run time the compiler cannot tell the fragment
  // reads from the DMA in flight into another stage and drains it before each stage's reads
  // (s_waitcnt vmcnt(0): load and MFMA then took turns)
  int step = 0;
#pragma unroll 1
  for (; step + NST <= nsteps; step += NST) {
#pragma unroll
    for (int u = 0; u < NST; ++u) stage(st[u], st[(u + 1) % NST], st[(u + NST - 1) % NST]);
  }
  // the last nsteps % NST of them
  if (step < nsteps) stage(st[0], st[1], st[NST - 1]);
  if (NST > 2 && step + 1 < nsteps) stage(st[1], st[2], st[0]);
  if (NST > 3 && step + 2 < nsteps) stage(st[2], st[3], st[1]);
  wait_vm_lgkm0<0>();                            // no DMA into this workgroup's LDS outlives it
  const int m = t.m[l];
  const double mi = t.dminv[l];
  const int lane = threadIdx.x & 63;
  signed char *out = res + (((size_t)wk.x * t.n + l) * 2 + p) * (size_t)(BT * BT);
#pragma unroll
  for (int i = 0; i < C::MI; ++i)
#pragma unroll
    for (int j = 0; j < C::NJ; ++j) {
      unsigned u4[4] = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int v = 0; v < 16; ++v) u4[v >> 2] |= (unsigned)(dres((double)acc[i][j][v], m, mi) & 255) << (8 * (v & 3));
      const int blk = wave * (C::MI * C::NJ) + i * C::NJ + j;
      *(uint4 *)(out + ((size_t)blk * 64 + lane) * 16) = make_uint4(u4[0], u4[1], u4[2], u4[3]);
    }
}

// ---------------------------------------------------------------------------------------
// merge: one 32 x 32 block of the gemm layout per wave (wave-major as the gemm wrote them, decoded
// with that variant's wave grid), one lane per gemm lane with its 16 values.  Waves share
// nothing: the rows' data sit in the wave's own LDS slice, the column's in registers, so there
// is no barrier and a small batch still fills the chip (with a tile per workgroup and its blocks
// in turn: 104 us for 5 atoms, N = 260, 8 k-points, 36 here; N = 5000, 32 atoms, 8 k: 2.56 ms, 2.26
// here; with 16 moduli, N = 2500, 16 atoms, 8 k: 1.19 ms with a multiply-add per pair of
// digits, 0.71).  Bound by Garner's 32-bit arithmetic and by reading the residues and O and writing H.
// ---------------------------------------------------------------------------------------
// The moduli and Garner's tables are fixed at compile time for each modulus count (the
// moduli list is constant; only how many of them is chosen), so every reduction below
// multiplies by immediates.  Moduli: odd, pairwise coprime, every prime factor 1 mod 4
// (221 = 13 17, 205 = 5 41), the largest first.
constexpr int kModList[kMaxMod] = {241, 233, 229, 221, 205, 197, 193, 181, 173, 157, 149, 137, 113, 109, 101, 97};

constexpr int inv_mod(int a, int m) {   // a^-1 mod m, gcd(a, m) = 1 (extended Euclid)
  int r0 = m, r1 = ((a % m) + m) % m, t0 = 0, t1 = 1;
  while (r1) {
    const int q = r0 / r1, r2 = r0 - q * r1, t2 = t0 - q * t1;
    r0 = r1; r1 = r2; t0 = t1; t1 = t2;
  }
  return t0 < 0 ? t0 + m : t0;
}

constexpr int iota_of(int m) {          // the smallest square root of -1 modulo m
  for (int x = 1; x < m; ++x)
    if ((x * x + 1) % m == 0) return x;
  return 0;
}

// Garner's mixed-radix digits d_l = (r_l - sum_j d_j M_j) M_l^-1 mod m_l (M_j = m_0 ... m_(j-1))
// of Re' and Im', from U and V: r_l = (U + V) 2^-1 for Re, (U - V) (2 iota_l)^-1 for Im, so
// the digit is s_l c_l - sum_j d_j w[l][j] reduced once, with s_l = U +- V unreduced,
// c_l = (2^-1 or (2 iota_l)^-1) M_l^-1 mod m_l and w[l][j] = (M_j mod m_l) M_l^-1 mod m_l.
template <int NM>
struct GarnerTab {
  int w[NM][(NM + 3) / 4];   // -w_lj symmetric modulo m_l, a byte each, four j a word (0 for j >= l)
  int cre[NM], cim[NM];
  double mk;        // M_6 (or P for fewer moduli): x = x_hi M_6 + x_lo
  double mh, ml;    // M_12 = mh + ml
  constexpr GarnerTab() : w(), cre(), cim(), mk(1.0), mh(0.0), ml(0.0) {
    for (int l = 0; l < NM; ++l) {
      const int m = kModList[l];
      long long ml = 1;
      int mj[NM] = {};
      for (int j = 0; j < l; ++j) {
        mj[j] = (int)(ml % m);
        ml = ml * kModList[j] % m;
      }
      const int v = inv_mod((int)ml, m);
      for (int j = 0; j < l; ++j) {
        int x = m - mj[j] * v % m;
        if (x > m / 2) x -= m;
        w[l][j / 4] |= (int)((unsigned)(x & 0xff) << (8 * (j % 4)));
      }
      cre[l] = inv_mod(2, m) * v % m;
      cim[l] = inv_mod(2 * iota_of(m) % m, m) * v % m;
    }
    for (int j = 0; j < (NM < kCrtLoDigits ? NM : kCrtLoDigits); ++j) mk *= kModList[j];
    if (NM > 2 * kCrtLoDigits) {
      __int128 m12 = 1;
      for (int j = 0; j < 2 * kCrtLoDigits; ++j) m12 *= kModList[j];
      mh = (double)m12;
      ml = (double)(m12 - (__int128)mh);
    }
  }
};

// symmetric residue modulo m = kModList[L] of |x| < 2^22; the float quotient is within
// 2^-21 |x| / m of x / m, far inside the 1/(2m) margin of the rounding
template <int L>
__device__ __forceinline__ int cres(int x) {
  constexpr int m = kModList[L];
  constexpr float finv = 1.0f / (float)m;
  return x - __mul24((int)rintf((float)x * finv), m);
}

// |s_l c_l| <= 240 240 and |d_j w| <= 120 120: the sum stays below 2^22 for up to 16 moduli.  The
// digits are packed four a word as they come, so that a dot product of bytes takes four of them (a
// multiply-add each was half of the merge's instructions, and more code than the instruction cache holds).
template <int NM, int L, bool IM>
__device__ __forceinline__ void garner_digit(int (&d)[NM], int (&dp)[(NM + 3) / 4], const int (&s)[NM]) {
  constexpr GarnerTab<NM> G{};
  int acc = __mul24(s[L], IM ? G.cim[L] : G.cre[L]);
#pragma unroll
  for (int j = 0; j < (L + 3) / 4; ++j) acc = __builtin_amdgcn_sdot4(dp[j], G.w[L][j], acc, false);
  d[L] = cres<L>(acc);
  if constexpr (L + 1 < NM) {
    // byte L % 4 of word L / 4
    if constexpr (L % 4 == 0) dp[L / 4] = d[L] & 0xff;
    else dp[L / 4] = __builtin_amdgcn_perm((unsigned)d[L], (unsigned)dp[L / 4], L % 4 == 1 ? 0x0c0c0400u : L % 4 == 2 ? 0x0c040100u : 0x04020100u);
    garner_digit<NM, L + 1, IM>(d, dp, s);
  }
}

// Re' (IM false) or Im' in [-(P-1)/2, (P-1)/2] from s_l = U + V (or U - V) modulo each m_l:
// Garner's digits, then the correctly rounded fma(x_hi, M_6, x_lo), the two parts exact in
// FP64 (|x_lo| < M_6 / 2 < 2^52)
template <int NM, bool IM>
__device__ __forceinline__ double garner(const int (&s)[NM]) {
  constexpr GarnerTab<NM> G{};
  int d[NM], dp[(NM + 3) / 4];
  garner_digit<NM, 0, IM>(d, dp, s);
  constexpr int NLO = NM < kCrtLoDigits ? NM : kCrtLoDigits, NMID = NM < 2 * kCrtLoDigits ? NM : 2 * kCrtLoDigits;
  double lo = (double)d[NLO - 1];
#pragma unroll
  for (int j = NLO - 2; j >= 0; --j) lo = fma(lo, (double)kModList[j], (double)d[j]);
  double mid = 0.0;
#pragma unroll
  for (int j = NMID - 1; j >= NLO; --j) mid = fma(mid, (double)kModList[j], (double)d[j]);
  const double x = fma(mid, G.mk, lo);
  if constexpr (NM <= NMID) {
    return x;
  } else {
    // beyond 12 moduli a third part x_hi M_12, M_12 = mh + ml to 106 bits: |x| <= M_12 / 2, so the
    // sum is within two roundings of the exact value
    double hi = 0.0;
#pragma unroll
    for (int j = NM - 1; j >= NMID; --j) hi = fma(hi, (double)kModList[j], (double)d[j]);
    return fma(hi, G.mh, fma(hi, G.ml, x));
  }
}

template <int NM>
__global__ __launch_bounds__(256) void crt_merge_kernel(const kdesc *__restrict__ ks, const mt_item *__restrict__ items,
                                                        int nitems, const signed char *__restrict__ res, int bt,
                                                        int wr_n, int wc_n, GTab gt, const double *__restrict__ gsig) {
  struct Slice {
    // Element (row, col) of a block sits in lane (col mod 32) of the gemm layout, so the
    // conjugate store at (col, row) is coalesced along the lanes; the store at (row, col) goes
    // through LDS, 16 rows of the block at a time: stored [col][row] with one pad element per
    // column, read back with 16 lanes along a column (256 contiguous bytes)
    cplx t[32 * 17];
    double v[32][3];
    int g[32][3], ex[32];
  };
  __shared__ Slice sl[4];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  Slice &sw = sl[wave];
  const int bpt = (bt / 32) * (bt / 32);                    // blocks of a tile: a multiple of 4
  const int item = blockIdx.x / (bpt / 4), blk = blockIdx.x % (bpt / 4) * 4 + wave;
  const mt_item it = items[item];
  const kdesc k = ks[it.k];
  const int ngp = k.ngp;
  const int mi_n = bt / wr_n / 32, nj_n = bt / wc_n / 32, per_wave = mi_n * nj_n;
  const int wv = blk / per_wave, bi = (blk % per_wave) / nj_n, bj = blk % nj_n;
  const int row0 = it.ti * bt + (wv / wc_n) * (32 * mi_n) + 32 * bi;     // the block's origin
  const int col0 = it.tj * bt + (wv % wc_n) * (32 * nj_n) + 32 * bj;
  if (row0 > col0 + 31 || col0 >= ngp) return;              // below the diagonal or past the basis (uniform)
  const size_t ptile = (size_t)bt * bt;                     // residue bytes of one (modulus, product)
  const signed char *base = res + (size_t)item * NM * 2 * ptile + ((size_t)blk * 64 + lane) * 16;
  cplx *out = it.which == 1 ? k.o : k.h;
  const double sig = it.which == 2 ? *gsig : 0.0;           // Gram form: H_MT = conj(E) E^T - sigma O_APW
  if (lane < 32) {
    const int idx = row0 + lane;
    int ig = 0, ex = 0;
    if (idx < ngp) {
      ig = k.igpig[idx] - 1;
      ex = k.xa[idx];
#pragma unroll
      for (int q = 0; q < 3; ++q) sw.v[lane][q] = k.vgpc[3 * idx + q];
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) sw.g[lane][q] = gt.ivg[3 * ig + q];
    sw.ex[lane] = ex;
  }
  const int col = col0 + (lane & 31);
  int gc[3] = {0, 0, 0}, exc = 0;
  double vc[3] = {0.0, 0.0, 0.0};
  if (col < ngp) {
    const int ig = k.igpig[col] - 1;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      gc[q] = gt.ivg[3 * ig + q];
      vc[q] = k.vgpc[3 * col + q];
    }
    exc = it.which ? k.xa[col] : k.xy[col];
  }
  auto fence = [] {                                         // orders this wave's LDS stores and loads
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  constexpr bool kWhole = NM <= 12;                         // more moduli: half a block's residues at a time (registers)
  uint4 q1[kWhole ? NM : 1], q2[kWhole ? NM : 1];
  if constexpr (kWhole) {
#pragma unroll
    for (int l = 0; l < NM; ++l) {
      q1[l] = *(const uint4 *)(base + (size_t)l * 2 * ptile);
      q2[l] = *(const uint4 *)(base + (size_t)l * 2 * ptile + ptile);
    }
  }
  unsigned miss = 0;
  fence();
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    uint2 p1[NM], p2[NM];
#pragma unroll
    for (int l = 0; l < NM; ++l) {
      if constexpr (kWhole) {
        p1[l] = h ? make_uint2(q1[l].z, q1[l].w) : make_uint2(q1[l].x, q1[l].y);
        p2[l] = h ? make_uint2(q2[l].z, q2[l].w) : make_uint2(q2[l].x, q2[l].y);
      } else {
        p1[l] = *(const uint2 *)(base + (size_t)l * 2 * ptile + 8 * h);
        p2[l] = *(const uint2 *)(base + (size_t)l * 2 * ptile + ptile + 8 * h);
      }
    }
    // the interstitial indices of this half's 8 elements (lookup_g without its branches: the loads
    // go out together), -1 where nothing is stored
    int ig[8];
#pragma unroll
    for (int vv = 0; vv < 8; ++vv) {
      const int rl = 16 * h + 8 * (vv >> 2) + 4 * (lane >> 5) + (vv & 3), row = row0 + rl;
      const int d0 = sw.g[rl][0] - gc[0] - gt.lo0, d1 = sw.g[rl][1] - gc[1] - gt.lo1, d2 = sw.g[rl][2] - gc[2] - gt.lo2;
      const bool in = (unsigned)d0 < (unsigned)gt.n0 && (unsigned)d1 < (unsigned)gt.n1 && (unsigned)d2 < (unsigned)gt.n2;
      const int v = gt.ivgig[in ? d0 + gt.n0 * (d1 + gt.n1 * d2) : 0];
      ig[vv] = in && v > 0 && v <= gt.ngvec ? v : 0;
      if (!(col < ngp && row <= col)) ig[vv] = -1;
      miss += ig[vv] == 0;
    }
    // Gram form: this half's eight O elements, loaded together ahead of the reconstruction;
    // read at (col, row), O's conjugate mirror (bit for bit), where the lanes are contiguous
    cplx om[8];
    if (it.which == 2) {
#pragma unroll
      for (int vv = 0; vv < 8; ++vv) {
        const int row = row0 + 16 * h + 8 * (vv >> 2) + 4 * (lane >> 5) + (vv & 3);
        om[vv] = ig[vv] >= 0 ? k.o[col + (size_t)row * k.ldh] : cplx{0.0, 0.0};
      }
    }
#pragma unroll
    for (int vv = 0; vv < 8; ++vv) {
      const int rh = 8 * (vv >> 2) + 4 * (lane >> 5) + (vv & 3);   // row within the half
      const int rl = 16 * h + rh, row = row0 + rl;
      cplx val = {0.0, 0.0};
      {
        // conj(a) b: Re = (U + V)/2, Im = (U - V)/(2 iota) modulo each m
        const int sh = 8 * (vv & 3);
        int sr[NM], si[NM];
#pragma unroll
        for (int l = 0; l < NM; ++l) {
          const unsigned w1 = vv < 4 ? p1[l].x : p1[l].y, w2 = vv < 4 ? p2[l].x : p2[l].y;
          const int u = (signed char)(w1 >> sh), v = (signed char)(w2 >> sh);
          sr[l] = u + v;
          si[l] = u - v;
        }
        const int sc = -(sw.ex[rl] + exc);
        double re = ldexp(garner<NM, false>(sr), sc);
        double im = ldexp(garner<NM, true>(si), sc);
        const bool has = ig[vv] > 0;
        const int g = max(ig[vv], 1);
        if (it.which == 2) {
          // O_APW = O - its interstitial term, O as the overlap kernel wrote it
          cplx oa = {om[vv].re, -om[vv].im};
          const cplx tho = setup_dev::olp_theta(gt, g, sw.v[rl], vc);
          oa = cplx{oa.re - (has ? tho.re : 0.0), oa.im - (has ? tho.im : 0.0)};
          re = fma(-sig, oa.re, re);
          im = fma(-sig, oa.im, im);
        }
        if (it.which == 1) {
          const cplx th = gt.cfunig[g - 1];
          re += has ? th.re : 0.0;
          im += has ? th.im : 0.0;
        } else {
          const cplx vv2 = gt.veffig[g - 1], kin = gt.kinig[g - 1];
          const double t1 = 0.5 * (sw.v[rl][0] * vc[0] + sw.v[rl][1] * vc[1] + sw.v[rl][2] * vc[2]);
          re += has ? vv2.re + t1 * kin.re : 0.0;
          im += has ? vv2.im + t1 * kin.im : 0.0;
        }
        val = cplx{re, im};
        if (row < col && col < ngp) out[col + (size_t)row * k.ldh] = cplx{re, -im};
      }
      sw.t[(lane & 31) * 17 + rh] = val;
    }
    fence();
    // 16 rows x 32 columns of this half: lane -> row (lane & 15), columns (lane >> 4) + 4 i
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int cc = (lane >> 4) + 4 * i, r = lane & 15;
      const int grow = row0 + 16 * h + r, gcol = col0 + cc;
      if (gcol < ngp && grow <= gcol) out[grow + (size_t)gcol * k.ldh] = sw.t[cc * 17 + r];
    }
    fence();                                                // the slice is rewritten next
  }
  if (miss && gt.miss) atomicAdd(gt.miss, miss);
}

template <int NM>
int launch_merge_t(const exc_dev &d, const kdesc *ks, const mt_item *items, int nitems, const CrtTab &t,
                   const signed char *res, int bt, int wr, int wc, const double *gsig, hipStream_t s) {
  hipLaunchKernelGGL((crt_merge_kernel<NM>), dim3(nitems * (bt * bt / 4096)), dim3(256), 0, s, ks, items, nitems, res, bt,
                     wr, wc, setup_dev::make_gtab(d), gsig);
  EXC_CHECK(hipGetLastError());
  return EXC_OK;
}

template <int BT, int BK, int NST, int WR, int WC, int MINW>
int launch_gemm_t(const kdesc *ks, const mt_item *items, const int2 *work, int nwork, int kp, const CrtTab &t,
                  signed char *res, hipStream_t s) {
  if (kp % BK) return EXC_ERR_UNSUPPORTED;      // the k loop runs whole stages of BK bytes
  const int chunk = (nwork + 7) / 8;
  hipLaunchKernelGGL((crt_gemm_kernel<BT, BK, NST, WR, WC, MINW>), dim3(8 * chunk), dim3(64 * WR * WC), 0, s, ks,
                     items, work, nwork, kp, t, res);
  EXC_CHECK(hipGetLastError());
  return EXC_OK;
}

template <int BT, int BK, int NST>
int launch_gemm_pipe_t(const kdesc *ks, const mt_item *items, const int2 *work, int nwork, int kp, const CrtTab &t,
                       signed char *res, hipStream_t s) {
  if (kp % BK) return EXC_ERR_UNSUPPORTED;
  const int chunk = (nwork + 7) / 8;
  hipLaunchKernelGGL((crt_gemm_pipe_kernel<BT, BK, NST, 2, 2>), dim3(8 * chunk), dim3(256), 0, s, ks, items, work,
                     nwork, kp, t, res);
  EXC_CHECK(hipGetLastError());
  return EXC_OK;
}

}  // namespace

void exc_crt_tables(int n, CrtTab *t) {
  *t = CrtTab{};
  t->n = n;
  double lp = 0.0;
  for (int l = 0; l < n; ++l) {
    t->m[l] = kModList[l];
    t->iota[l] = iota_of(kModList[l]);
    t->dminv[l] = 1.0 / kModList[l];
    t->finv[l] = 1.0f / (float)kModList[l];
    const int m = kModList[l];
    long long w = 1;
    int sr[4], si[4];
    for (int q = 0; q < 4; ++q) {
      const int a = (int)w, b = (int)(w * t->iota[l] % m);
      sr[q] = a > m / 2 ? a - m : a;
      si[q] = b > m / 2 ? b - m : b;
      w = w * 65536 % m;
    }
    for (int q = 0; q < 2; ++q) {
      t->wr[l][q] = (int)(((unsigned)sr[2 * q + 1] << 16) | ((unsigned)sr[2 * q] & 0xffffu));
      t->wi[l][q] = (int)(((unsigned)si[2 * q + 1] << 16) | ((unsigned)si[2 * q] & 0xffffu));
    }
    lp += log2((double)kModList[l]);
  }
  // beta: the largest b with 2^(2b + 2) <= P, from log2 P with a margin against its rounding
  t->beta = (int)floor((lp - 2.0 - 1e-9) / 2.0);
}

// a_parts: the grouped match wrote A's squared norms per atom (else A takes a pass of its
// own, as Yt always does); gram: E in Yt's buffer is the only operand; exact: rows the integers
// cannot hold are marked (kBadRow)
int exc_launch_crt_prep(const exc_dev &d, int nk, int maxnp, const kdesc *ks, const CrtTab &t, bool a_parts,
                        bool gram, bool exact, hipStream_t s) {
  if (nk <= 0 || maxnp <= 0) return EXC_OK;
  const int ex = exact;
  const int ktot = d.natm * d.naa, kp = exc_crt_kpad(ktot);
  if (gram) {
    hipLaunchKernelGGL(crt_scale_kernel, dim3(maxnp / 64, 1, nk), dim3(64 * kScaleWaves), 0, s, ks, ktot, t.beta, 2, ex);
    EXC_CHECK(hipGetLastError());
    hipLaunchKernelGGL(crt_split_kernel, dim3(maxnp / 64, kp / 64, nk), dim3(256), 0, s, ks, ktot, kp, t, 1);
    EXC_CHECK(hipGetLastError());
    return EXC_OK;
  }
  if (a_parts) {
    hipLaunchKernelGGL(crt_expo_kernel, dim3((maxnp + 255) / 256, 1, nk), dim3(256), 0, s, ks, d.natm, t.beta, ex);
    EXC_CHECK(hipGetLastError());
  } else {
    hipLaunchKernelGGL(crt_scale_kernel, dim3(maxnp / 64, 1, nk), dim3(64 * kScaleWaves), 0, s, ks, ktot, t.beta, 0, ex);
    EXC_CHECK(hipGetLastError());
  }
  hipLaunchKernelGGL(crt_scale_kernel, dim3(maxnp / 64, 1, nk), dim3(64 * kScaleWaves), 0, s, ks, ktot, t.beta, 1, ex);
  EXC_CHECK(hipGetLastError());
  hipLaunchKernelGGL(crt_split_kernel, dim3(maxnp / 64, kp / 64, 2 * nk), dim3(256), 0, s, ks, ktot, kp, t, 0);
  EXC_CHECK(hipGetLastError());
  return EXC_OK;
}

// variants: (tile edge, k bytes per LDS stage, stages, wave grid, minimum waves per SIMD)
//   0: 256, 64, 3, 2 x 4 (128 x 64 wave tiles), 1    1: 256, 32, 4, 2 x 4, 1
//   2: 128, 64, 3, 2 x 2 (64 x 64 wave tiles), 2     3: 256, 64, 2, 2 x 4, 1
//   4: 128, 32, 4, 2 x 2, 2
//   5: 256, 64, 3, 2 x 2 (128 x 128 wave tiles: two thirds of the LDS reads per MFMA), 1
//   6: 256, 32, 4, 2 x 2, 1                           7: 256, 64, 4, 2 x 2, 1
//   8: 256, 64, 3, 2 x 2, register-pipelined          9: 256, 64, 2, 2 x 2, register-pipelined
//  10: 256, 64, 4, 2 x 2, register-pipelined
int exc_crt_shape(int variant, int *bt, int *wr, int *wc) {
  switch (variant) {
    case 0: case 1: case 3: *bt = 256; *wr = 2; *wc = 4; return EXC_OK;
    case 5: case 6: case 7: case 8: case 9: case 10: *bt = 256; *wr = 2; *wc = 2; return EXC_OK;
    case 2: case 4: *bt = 128; *wr = 2; *wc = 2; return EXC_OK;
    default: return EXC_ERR_ARG;
  }
}

int exc_launch_crt_gemm(const exc_dev &d, const kdesc *ks, const mt_item *items, const int2 *work, int nwork,
                        const CrtTab &t, signed char *res, int variant, hipStream_t s) {
  if (nwork <= 0) return EXC_OK;
  const int kp = exc_crt_kpad(d.natm * d.naa);
  switch (variant) {
    case 0: return launch_gemm_t<256, 64, 3, 2, 4, 1>(ks, items, work, nwork, kp, t, res, s);
    case 1: return launch_gemm_t<256, 32, 4, 2, 4, 1>(ks, items, work, nwork, kp, t, res, s);
    case 2: return launch_gemm_t<128, 64, 3, 2, 2, 2>(ks, items, work, nwork, kp, t, res, s);
    case 3: return launch_gemm_t<256, 64, 2, 2, 4, 1>(ks, items, work, nwork, kp, t, res, s);
    case 4: return launch_gemm_t<128, 32, 4, 2, 2, 2>(ks, items, work, nwork, kp, t, res, s);
    case 5: return launch_gemm_t<256, 64, 3, 2, 2, 1>(ks, items, work, nwork, kp, t, res, s);
    case 6: return launch_gemm_t<256, 32, 4, 2, 2, 1>(ks, items, work, nwork, kp, t, res, s);
    case 7: return launch_gemm_t<256, 64, 4, 2, 2, 1>(ks, items, work, nwork, kp, t, res, s);
    case 8: return launch_gemm_pipe_t<256, 64, 3>(ks, items, work, nwork, kp, t, res, s);
    case 9: return launch_gemm_pipe_t<256, 64, 2>(ks, items, work, nwork, kp, t, res, s);
    case 10: return launch_gemm_pipe_t<256, 64, 4>(ks, items, work, nwork, kp, t, res, s);
    default: return EXC_ERR_ARG;
  }
}

int exc_launch_crt_merge(const exc_dev &d, const kdesc *ks, const mt_item *items, int nitems, const CrtTab &t,
                         const signed char *res, int variant, const double *gsig, hipStream_t s) {
  if (nitems <= 0) return EXC_OK;
  int bt = 0, wr = 0, wc = 0;
  if (exc_crt_shape(variant, &bt, &wr, &wc)) return EXC_ERR_ARG;
  switch (t.n) {
    case 8: return launch_merge_t<8>(d, ks, items, nitems, t, res, bt, wr, wc, gsig, s);
    case 9: return launch_merge_t<9>(d, ks, items, nitems, t, res, bt, wr, wc, gsig, s);
    case 10: return launch_merge_t<10>(d, ks, items, nitems, t, res, bt, wr, wc, gsig, s);
    case 11: return launch_merge_t<11>(d, ks, items, nitems, t, res, bt, wr, wc, gsig, s);
    case 12: return launch_merge_t<12>(d, ks, items, nitems, t, res, bt, wr, wc, gsig, s);
    case kExactMod: return launch_merge_t<kExactMod>(d, ks, items, nitems, t, res, bt, wr, wc, gsig, s);
    default: return EXC_ERR_ARG;
  }
}
