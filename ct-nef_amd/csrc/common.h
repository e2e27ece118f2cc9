// Shared device/host helpers for the nefct HIP kernels (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/nefct_hip.h"

#define NEFCT_WAVE 64

// Raw buffer resource over [p, p + nbytes): loads past the end return 0 and
// atomics past the end are dropped by the texture address unit, so a wrong
// index can never fault the device.  Dword 3 = 0x00020000 is the raw-buffer
// format word for the gfx9 family (CDNA3/4).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, uint32_t nbytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)nbytes, 0x00020000);
}

__device__ __forceinline__ float buf_load(__amdgpu_buffer_rsrc_t r, int byte_off)
{
    // the b32 builtin returns the raw bits as an unsigned int
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, byte_off, 0, 0));
}

// four floats from a byte offset that is a multiple of 4
__device__ __forceinline__ float4 buf_load4(__amdgpu_buffer_rsrc_t r, int byte_off)
{
    return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, byte_off, 0, 0));
}

// One dword per lane from byte offset lane_off + off of a raw buffer straight
// into LDS at lds + 4 lane (no registers; past the buffer's end: 0).  All of
// off, lds and the buffer are wave-uniform and every lane is active.  Written
// as assembly because the compiler holds back every later LDS read until such
// loads have landed: the caller waits with lds_loads_done() before the barrier
// that hands the cells over.
// A buffer load may read a scalar register five wait states after a vector
// instruction (readfirstlane) wrote it at the earliest, and inside assembly
// nothing keeps that distance: the buffer's words are waited for once, where
// they are made, and the offset goes through a scalar move, which also is the
// wait state between m0 and the load (1 % of the FDK backprojection of
// 512 x 512 x 256 voxels; a five-state wait in every load: 2 %).
typedef int rsrc_words __attribute__((ext_vector_type(4)));
__device__ __forceinline__ rsrc_words make_rsrc_words(const void* p, uint32_t nbytes)
{
    const uint64_t a = (uint64_t)p;
    rsrc_words r;
    r.x = __builtin_amdgcn_readfirstlane((int)(uint32_t)a);
    r.y = __builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32) & 0xffff);
    r.z = __builtin_amdgcn_readfirstlane((int)nbytes);
    r.w = 0x00020000;
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("s_nop 4" : : "s"(r));
#endif
    return r;
}

__device__ __forceinline__ void buf_load_lds(rsrc_words r, int lane_off, unsigned off, unsigned lds)
{
#ifdef __HIP_DEVICE_COMPILE__
    int at;
    asm volatile("s_mov_b32 m0, %1\n\ts_mov_b32 %0, %4\n\tbuffer_load_dword %2, %3, %0 offen lds"
                 : "=&s"(at)
                 : "s"(__builtin_amdgcn_readfirstlane((int)lds)), "v"(lane_off), "s"(r),
                   "s"(__builtin_amdgcn_readfirstlane((int)off))
                 : "memory", "m0");
#endif
}

__device__ __forceinline__ void lds_loads_done()
{
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#endif
}

__device__ __forceinline__ void buf_atomic_add(__amdgpu_buffer_rsrc_t r, int byte_off, float v)
{
    __builtin_amdgcn_raw_ptr_buffer_atomic_fadd_f32(v, r, byte_off, 0, 0);
}

__device__ __forceinline__ int wave_min_i32(int v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, NEFCT_WAVE));
    return v;
}

__device__ __forceinline__ int wave_max_i32(int v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, NEFCT_WAVE));
    return v;
}

// 1/x in FP64 from the hardware reciprocal and two Newton steps (a few ulp at
// most, against ~10 instructions for a correctly rounded division).
__device__ __forceinline__ double rcp64(double x)
{
    double r = __builtin_amdgcn_rcp(x);
    double e = fma(-x, r, 1.0);
    r = fma(r, e, r);
    e = fma(-x, r, 1.0);
    return fma(r, e, r);
}

// v unchanged, but opaque to the optimiser: it cannot fuse the product that
// made v into a later addition (an FMA contraction rounds once instead of
// twice), which it may do in one kernel and not in another.
__device__ __forceinline__ float no_contract(float v)
{
    asm("" : "+v"(v));
    return v;
}

#define NEFCT_CHECK_LAUNCH()                                        \
    do {                                                            \
        hipError_t e_ = hipGetLastError();                          \
        if (e_ != hipSuccess) return NEFCT_ERR_LAUNCH;              \
    } while (0)
