// The scalars of an elementary reflector, as zlarfg forms them: H = I - tau v v^H with v = (1, sc x)
// takes the vector (al, x) to (beta, 0), beta real, xn2 = |x|^2.  Host and device.
#pragma once
#include <math.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define EXC_HD __host__ __device__ __forceinline__
#else
#define EXC_HD inline
#endif

// Below this |al|^2 + |x|^2 is no longer a normal number to full precision, and 1 / |al - beta|^2
// would overflow: the vector, below 1e-145, counts as zero, tau = sc = 0 and beta = Re al.  (zlarfg
// scales such vectors up; a branch for that in the matrix-vector kernel cost 2 % of an eigensolve, for
// elements 130 orders below what an eigenvalue of any Hamiltonian is known to.)
constexpr double kReflectorTiny = 1e-290;

EXC_HD bool reflector_tiny(double are, double aim, double xn2) {
  return are * are + aim * aim + xn2 < kReflectorTiny;
}

// z: beta, Re tau, Im tau, Re sc, Im sc
EXC_HD void reflector(double are, double aim, double xn2, double (&z)[5]) {
  z[0] = are;
  z[1] = z[2] = z[3] = z[4] = 0.0;
  if ((xn2 == 0.0 && aim == 0.0) || reflector_tiny(are, aim, xn2)) return;
  const double beta = -copysign(sqrt(are * are + aim * aim + xn2), are), bi = 1.0 / beta;
  const double dr = are - beta, q = 1.0 / (dr * dr + aim * aim);
  z[0] = beta;
  z[1] = (beta - are) * bi;
  z[2] = -aim * bi;
  z[3] = dr * q;
  z[4] = -aim * q;
}
