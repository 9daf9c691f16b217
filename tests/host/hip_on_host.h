// Stands in for hip/hip_runtime.h when the GEMM sources are compiled as plain C++: a launch runs every
// lane of every workgroup in turn on the CPU, and the buffer instructions check the addresses they would
// read instead of reading.  Values are zero throughout: this is for addresses, not results.
//
// A raw buffer read is in range when its lane offset is below num_records - uniform offset, an unsigned
// 32-bit subtraction; a read that passes that test must lie in the span, and a span in its operand.
#pragma once
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <type_traits>
#include <vector>

#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ static
#define __align__(n) __attribute__((aligned(n)))
#define HIP_SYMBOL(s) (&(s))

struct dim3 {
    unsigned x, y, z;
    dim3(unsigned x_ = 1, unsigned y_ = 1, unsigned z_ = 1) : x(x_), y(y_), z(z_) {}
};
struct uint2 { uint32_t x, y; };
struct uint4 { uint32_t x, y, z, w; };
struct float2 { float x, y; };
struct float4 { float x, y, z, w; };
inline uint2 make_uint2(uint32_t x, uint32_t y) { return {x, y}; }
inline uint4 make_uint4(uint32_t x, uint32_t y, uint32_t z, uint32_t w) { return {x, y, z, w}; }
inline float2 make_float2(float x, float y) { return {x, y}; }
inline float4 make_float4(float x, float y, float z, float w) { return {x, y, z, w}; }

typedef void* hipStream_t;
typedef int hipError_t;
constexpr int hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorInvalidDevice = 101, hipErrorInvalidSymbol = 13;
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { return *d = 0; }
template <class T>
hipError_t hipGetSymbolAddress(void** p, T* symbol) { return *p = symbol, hipSuccess; }

inline dim3 threadIdx, blockIdx, blockDim, gridDim;
using std::max;
using std::min;
inline float __uint_as_float(uint32_t v) { float f; memcpy(&f, &v, 4); return f; }
inline uint32_t __float_as_uint(float f) { uint32_t v; memcpy(&v, &f, 4); return v; }
inline float __int_as_float(int v) { return __uint_as_float((uint32_t)v); }
inline int __float_as_int(float f) { return (int)__float_as_uint(f); }
inline float __shfl_xor(float v, int, int) { return v; }
inline float rsqrtf(float v) { return 1.f / sqrtf(v); }
inline void __syncthreads() {}

// -------------------------------------------------------------- what the launch may touch
struct Operand {
    const char* base;
    size_t bytes;
};
inline std::vector<Operand> operands;
inline long violations;
inline void violation(const char* what, long long a, long long b) {
    if (violations++ < 3)
        printf("block %u thread %u: %s (%lld against %lld)\n", blockIdx.x, threadIdx.x, what, a, b);
}

struct __amdgpu_buffer_rsrc_t {
    const char* base;
    uint32_t bytes;
};
inline __amdgpu_buffer_rsrc_t __builtin_amdgcn_make_buffer_rsrc(void* base, short, uint32_t bytes, int) {
    const char* b = (const char*)base;
    bool inside = bytes == 0;
    for (const Operand& o : operands) inside |= b >= o.base && b + bytes <= o.base + o.bytes;
    if (!inside) violation("a span leaves its operand", bytes, 0);
    return {b, bytes};
}
inline void check_read(const __amdgpu_buffer_rsrc_t& s, uint32_t voff, uint32_t soff, uint32_t size) {
    const bool passes = voff < s.bytes - soff;
    const unsigned long long end = (unsigned long long)voff + soff + size;
    if (passes && end > s.bytes) violation("a read past its span passes the range check", (long long)end, s.bytes);
}
typedef unsigned int host_u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int host_u32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 host_bf16x2 __attribute__((ext_vector_type(2)));
inline host_u32x4 __builtin_amdgcn_raw_buffer_load_b128(__amdgpu_buffer_rsrc_t s, uint32_t v, uint32_t u, int) {
    return check_read(s, v, u, 16), host_u32x4{0, 0, 0, 0};
}
inline host_u32x2 __builtin_amdgcn_raw_buffer_load_b64(__amdgpu_buffer_rsrc_t s, uint32_t v, uint32_t u, int) {
    return check_read(s, v, u, 8), host_u32x2{0, 0};
}
inline uint16_t __builtin_amdgcn_raw_buffer_load_b16(__amdgpu_buffer_rsrc_t s, uint32_t v, uint32_t u, int) {
    return check_read(s, v, u, 2), 0;
}
inline uint8_t __builtin_amdgcn_raw_buffer_load_b8(__amdgpu_buffer_rsrc_t s, uint32_t v, uint32_t u, int) {
    return check_read(s, v, u, 1), 0;
}
inline void __builtin_amdgcn_raw_ptr_buffer_load_lds(__amdgpu_buffer_rsrc_t s, void*, int size, uint32_t v, uint32_t u,
                                                     int, int) {
    check_read(s, v, u, size);
}

// -------------------------------------------------------------- instructions without an address
inline int __builtin_amdgcn_readfirstlane(int v) { return v; }
inline void __builtin_amdgcn_sched_barrier(int) {}
inline void __builtin_amdgcn_s_waitcnt(int) {}
inline void __builtin_amdgcn_s_barrier() {}
inline void __builtin_amdgcn_global_load_lds(const void*, void*, int, int, int) {}
inline int __builtin_amdgcn_update_dpp(int, int v, int, int, int, bool) { return v; }
inline int __builtin_amdgcn_sdot4(int, int, int c, bool) { return c; }
inline uint32_t __builtin_amdgcn_perm(uint32_t a, uint32_t, uint32_t) { return a; }
inline host_u32x2 __builtin_amdgcn_permlane16_swap(uint32_t a, uint32_t b, bool, bool) { return {a, b}; }
inline host_u32x2 __builtin_amdgcn_permlane32_swap(uint32_t a, uint32_t b, bool, bool) { return {a, b}; }
inline float __builtin_amdgcn_fdot2_f32_bf16(host_bf16x2, host_bf16x2, float c, bool) { return c; }
inline host_bf16x2 __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(uint32_t, float, bool) { return {0, 0}; }
template <class A, class C>
C __builtin_amdgcn_mfma_f32_32x32x16_bf16(A, A, C c, int, int, int) { return c; }
template <class A, class C>
C __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, A, C c, int, int, int) { return c; }

// -------------------------------------------------------------- a launch
inline bool run_launches = true;
inline unsigned last_blocks = ~0u;  // run only this many
struct Launched {
    const char* kernel;
    unsigned blocks;
};
inline std::vector<Launched> launched;
template <class F>
void host_launch(const char* kernel, dim3 grid, dim3 block, F lane) {
    launched.push_back({kernel, grid.x * grid.y});
    if (!run_launches) return;
    gridDim = grid;
    blockDim = block;
    for (blockIdx.y = 0; blockIdx.y < grid.y; ++blockIdx.y)
        for (blockIdx.x = grid.x > last_blocks ? grid.x - last_blocks : 0; blockIdx.x < grid.x; ++blockIdx.x)
            for (threadIdx.x = 0; threadIdx.x < block.x; ++threadIdx.x) lane();
}
#define hipLaunchKernelGGL(kernel, grid, block, lds, stream, ...) \
    host_launch(#kernel, grid, block, [&] { kernel(__VA_ARGS__); })
