/*
 * One Newton-Raphson step for a reciprocal, with fused multiply-adds: from an
 * estimate within an ulp it gives the correctly rounded quotient but for single
 * mantissas (P. Markstein, "Computation of elementary functions on the IBM RISC
 * System/6000 processor", IBM J. Res. Dev. 34, 1990).  From the gfx950
 * estimate it does for every mantissa, where the estimate alone is an ulp
 * off for 11% of them.  (Also compiled for the host, where a test runs it over
 * every mantissa and the floats around its reciprocal.)
 */
#ifndef LRH_RCP_H
#define LRH_RCP_H

#include <math.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define LRH_RCP __device__ __forceinline__
#else
#define LRH_RCP inline
#endif

// 1/d from the estimate r
LRH_RCP float lrhRefineRcp(float d, float r) { return fmaf(fmaf(-d, r, 1.0f), r, r); }

#endif
