// Functions that the kernels share with host code.
#pragma once

#ifdef __HIPCC__
#define DMHM_HD __host__ __device__ inline __attribute__((always_inline))
#else
#define DMHM_HD inline
#endif
