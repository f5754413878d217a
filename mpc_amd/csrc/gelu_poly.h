/*
 * gelu_poly.h -- the polynomial of the inference path's GELU (fno_device.h:
 * gelu_fast), host and device, so that its error can be checked on the CPU.
 *
 * M(a) = -log2(erfc(a / sqrt 2)) / a for a >= 0, so that erfc(a / sqrt 2) =
 * 2^(-a M(a)).  A deviation dM moves 0.5 a erfc(a / sqrt 2), GELU's tail, by ln 2
 * a erfc(a / sqrt 2) dM of a / 2; these degree-9 coefficients make the largest of
 * that over 0 <= a <= 7 least (a linear program on 4001 Chebyshev points):
 * 1.3e-10, and 1e-9 with the coefficients rounded to FP32.  Beyond 7 erfc is
 * below 3e-12 and the polynomial keeps growing.
 */
#ifndef MPC_GELU_POLY_H
#define MPC_GELU_POLY_H

#include <cmath>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define MPC_GELU_HD __host__ __device__ __forceinline__
#else
#define MPC_GELU_HD inline
#endif

template <class T> MPC_GELU_HD T gelu_poly(T a) {
    T q = std::fma(a, (T)5.96657586e-08f, (T)-1.44687669e-06f);
    q = std::fma(q, a, (T)1.56093301e-05f);
    q = std::fma(q, a, (T)-9.60515536e-05f);
    q = std::fma(q, a, (T)0.000327383692f);
    q = std::fma(q, a, (T)-6.75654228e-05f);
    q = std::fma(q, a, (T)-0.00689349789f);
    q = std::fma(q, a, (T)0.0524200164f);
    q = std::fma(q, a, (T)0.459224194f);
    return std::fma(q, a, (T)1.15110409f);
}

#endif
