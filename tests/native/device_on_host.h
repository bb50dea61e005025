// device_on_host.h -- what the device functions of the library's headers need
// to run on the CPU, one lane at a time (g++, the HIP headers' host types).
// A file defines the thread it plays in threadIdx, blockIdx and blockDim.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstring>

#ifndef __forceinline__
#define __forceinline__ inline
#endif

struct HostDim3 { unsigned x = 0, y = 0, z = 0; };
static HostDim3 threadIdx, blockIdx, blockDim, gridDim;

template <class T> static T atomicCAS(T* p, T want, T v) { const T o = *p; if (o == want) *p = v; return o; }
template <class T> static T atomicMax(T* p, T v) { const T o = *p; if (o < v) *p = v; return o; }
template <class T> static T __shfl_down(T v, int, int = 64) { return v; }
template <class T> static T __shfl_up(T v, int, int = 64) { return v; }
static inline unsigned __umulhi(unsigned a, unsigned b) { return (unsigned)(((unsigned long long)a * b) >> 32); }
static inline double __longlong_as_double(long long v) { double d; std::memcpy(&d, &v, 8); return d; }
static inline void __syncthreads() {}
#define __HIP_MEMORY_SCOPE_AGENT 4
#define __hip_atomic_load(p, order, scope) (*(p))
#define __builtin_amdgcn_readfirstlane(x) (x)
using std::max;
using std::min;
