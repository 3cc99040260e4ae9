// In place of <hip/hip_runtime.h>: the library's device headers as ordinary
// C++, one work item at a time, so that the code the kernels are built from runs
// on the CPU.  The hardware's estimates are the correctly rounded values moved
// by host_ulps units in the last place; what looks at other lanes of a wavefront
// is only declared.
#pragma once
#include <hip/hip_runtime_api.h>
#include <math.h>
#include <stdint.h>
#include <string.h>

#undef __device__
#undef __host__
#undef __global__
#undef __forceinline__
#define __device__
#define __host__
#define __global__
#define __forceinline__ inline

inline int host_ulps = 0;
inline float host_moved(float v) {
  if (!isfinite(v) || v == 0.f) return v;
  int32_t b;
  memcpy(&b, &v, 4);
  b += host_ulps;
  memcpy(&v, &b, 4);
  return v;
}
inline float __builtin_amdgcn_rcpf(float x) { return host_moved(1.0f / x); }
inline float __builtin_amdgcn_sqrtf(float x) { return host_moved(sqrtf(x)); }
inline float __builtin_amdgcn_rsqf(float x) { return host_moved(1.0f / sqrtf(x)); }
inline float __builtin_amdgcn_fmed3f(float a, float b, float c) { return fmaxf(fminf(a, b), fminf(fmaxf(a, b), c)); }
inline uint32_t __float_as_uint(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }
inline int __float_as_int(float f) { int u; memcpy(&u, &f, 4); return u; }
inline float __uint_as_float(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
inline float __int_as_float(int u) { float f; memcpy(&f, &u, 4); return f; }
inline uint32_t __umul24(uint32_t a, uint32_t b) { return (a & 0xFFFFFFu) * (b & 0xFFFFFFu); }
inline bool __any(bool b) { return b; }
inline bool __all(bool b) { return b; }

int __builtin_amdgcn_update_dpp(int, int, int, int, int, bool);
int __builtin_amdgcn_readlane(int, int);
uint32_t __builtin_amdgcn_mbcnt_hi(uint32_t, uint32_t);
uint32_t __builtin_amdgcn_mbcnt_lo(uint32_t, uint32_t);
