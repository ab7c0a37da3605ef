// Sum over a wave without LDS: DPP moves within the rows of 16 lanes and across them.
#pragma once
#include "exc_common.h"

namespace {

// v of another lane of the row / half by DPP (no LDS round trip), 0 where there is none
template <int CTRL, int RM>
__device__ __forceinline__ double dpp_add(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, RM, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, RM, 0xf, false);
  return v + __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// sum over the wave, in every lane: within the rows of 16, then across them, lane 63 last
__device__ __forceinline__ double wave_sum(double v) {
  v = dpp_add<0x111, 0xf>(v);   // row_shr 1, 2, 4, 8: lane 15 of a row holds its sum
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);   // row_bcast15 into rows 1 and 3
  v = dpp_add<0x143, 0xc>(v);   // row_bcast31 into rows 2 and 3
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, 63), hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

}  // namespace
