// APW-lo and lo-lo blocks of one k-point on gfx950 (device code in lo_dev.h).
#include "lo_dev.h"

namespace {

using namespace lo_dev;

template <int MAXLO>
__global__ __launch_bounds__(kThreads) void lo_kernel(int ngp, int naa, int maxnlo, int nlomax, int apwordmax,
                                                      int nlotot, const int *__restrict__ dlo,
                                                      const lo_desc *__restrict__ lod, const cplx *__restrict__ apwalm,
                                                      int ldg, const cplx *__restrict__ loa,
                                                      const double *__restrict__ oalo, const double *__restrict__ h1loa,
                                                      const cplx *__restrict__ lolo, const double *__restrict__ ololo,
                                                      const double *__restrict__ h1lolo, cplx *__restrict__ h,
                                                      cplx *__restrict__ o, int ldh) {
  __shared__ ApwLoShared sh;
  if (blockIdx.x == 0)
    lo_lo_atom(blockIdx.y, dlo, ngp, nlotot, maxnlo, nlomax, lod, lolo, ololo, h1lolo, h, o, ldh);
  else
    lo_apw_body<MAXLO>(sh, blockIdx.x - 1, blockIdx.y, ngp, naa, maxnlo, nlomax, apwordmax, dlo, lod, apwalm, ldg, loa,
                       oalo, h1loa, h, o, ldh);
}

template <int MAXLO>
void launch_lo_t(const exc_dev &d, int ngp, const cplx *apwalm, int ldg, cplx *h, cplx *o, int ldh, hipStream_t s) {
  const dim3 grid(1 + (ngp + kRows - 1) / kRows, d.natm);
  hipLaunchKernelGGL(lo_kernel<MAXLO>, grid, dim3(kThreads), 0, s, ngp, d.naa, d.maxnlo, d.nlomax, d.apwordmax,
                     d.nlotot, d.dm_lo, d.lod, apwalm, ldg, d.loa, d.oalo, (d.iora & 2) ? d.h1loa : nullptr, d.lolo,
                     d.ololo, (d.iora & 2) ? d.h1lolo : nullptr, h, o, ldh);
}

}  // namespace

int exc_launch_lo(const exc_dev &d, int ngp, const cplx *apwalm, int ldg, cplx *h, cplx *o, int ldh, hipStream_t s) {
  if (d.nlotot == 0) return EXC_OK;
  if (d.maxnlo > kMaxLo) return EXC_ERR_UNSUPPORTED;
  // the accumulators of a thread are sized for the most lo functions an atom has
  if (d.dm_maxlo <= 4) launch_lo_t<4>(d, ngp, apwalm, ldg, h, o, ldh, s);
  else if (d.dm_maxlo <= 8) launch_lo_t<8>(d, ngp, apwalm, ldg, h, o, ldh, s);
  else launch_lo_t<16>(d, ngp, apwalm, ldg, h, o, ldh, s);
  EXC_CHECK(hipGetLastError());
  return EXC_OK;
}
