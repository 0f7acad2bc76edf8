// What the kernels need of HIP to compile as ordinary C++ for the host, one
// lane at a time (lane_order_check.cpp runs the lanes and the waits between them).
#pragma once
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <cstring>

#define __device__
#define __host__
#define __global__
#define __shared__ static
#define __forceinline__ inline
#define __launch_bounds__(...)
#define hipLaunchKernelGGL(kernel, ...) host_launch(kernel, __VA_ARGS__)

struct dim3 {
    unsigned x, y, z;
    dim3(unsigned x_ = 1, unsigned y_ = 1, unsigned z_ = 1) : x(x_), y(y_), z(z_) {}
};
typedef void* hipStream_t;
enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1 };
inline hipError_t hipGetLastError() { return hipSuccess; }

extern dim3 threadIdx, blockIdx, blockDim, gridDim;
void host_wave_wait();   // every lane of the caller's wave is here
void host_block_wait();  // every lane of the block is here
template <class... P, class... A>
void host_launch(void (*kernel)(P...), dim3 grid, dim3 block, int shared, hipStream_t, A... args);

inline void __syncthreads() { host_block_wait(); }
#define __builtin_amdgcn_wave_barrier() host_wave_wait()
#define __builtin_amdgcn_fence(order, scope) ((void)0)
#define __builtin_amdgcn_readfirstlane(x) (x)
inline uint64_t __umul64hi(uint64_t a, uint64_t b) { return (uint64_t)((unsigned __int128)a * b >> 64); }
inline uint32_t __umulhi(uint32_t a, uint32_t b) { return (uint32_t)((uint64_t)a * b >> 32); }
inline uint32_t __brev(uint32_t x) { return __builtin_bitreverse32(x); }
inline double __longlong_as_double(long long x) { double d; std::memcpy(&d, &x, 8); return d; }
inline long long __double_as_longlong(double x) { long long l; std::memcpy(&l, &x, 8); return l; }
