// What fft_small.h needs of the HIP headers, for a one-thread CPU build.
#pragma once
#define __device__
#define __host__
#define __forceinline__ inline
struct float2 { float x, y; };
inline float2 make_float2(float x, float y) { return float2{x, y}; }
struct Index { int x; };
static Index threadIdx = {0};
inline void __syncthreads() {}
