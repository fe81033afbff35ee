/*
 * What splattar_amd/csrc/gs_internal.h needs of HIP to be compiled for the
 * host (test infrastructure only): the vector types and the device functions
 * that its inline math calls. The approximate ones err by their documented
 * bound, up or down by a hash of the argument, so that a replay on the host
 * meets roundings at least as bad as the device's.
 */
#pragma once

#include <cmath>
#include <cstdint>
#include <cstring>

#define __device__
#define __host__
#define __forceinline__ inline
#define __align__(n) __attribute__((aligned(n)))

struct float2 { float x, y; };
struct float3 { float x, y, z; };
struct __attribute__((aligned(16))) float4 { float x, y, z, w; };
struct uint2 { uint32_t x, y; };
struct __attribute__((aligned(16))) uint4 { uint32_t x, y, z, w; };
inline float3 make_float3(float x, float y, float z) { return {x, y, z}; }
inline float4 make_float4(float x, float y, float z, float w) { return {x, y, z, w}; }
inline uint4 make_uint4(uint32_t x, uint32_t y, uint32_t z, uint32_t w) { return {x, y, z, w}; }

typedef struct host_hip_stream* hipStream_t;
typedef int hipError_t;
constexpr hipError_t hipSuccess = 0;

inline int min(int a, int b) { return a < b ? a : b; }
inline int max(int a, int b) { return a > b ? a : b; }
inline uint32_t min(uint32_t a, uint32_t b) { return a < b ? a : b; }
inline uint32_t max(uint32_t a, uint32_t b) { return a > b ? a : b; }
struct HostDim { uint32_t x; };
constexpr HostDim gridDim{1}, blockIdx{0};
inline uint32_t atomicAdd(uint32_t* p, uint32_t v) { const uint32_t o = *p; *p += v; return o; }

inline float __fsqrt_rn(float x) { return std::sqrt(x); }
inline float __fdiv_rn(float a, float b) { return a / b; }

// x moved by -ulps, 0 or +ulps units in the last place.
inline float host_nudge(float x, int ulps) {
    uint32_t u;
    std::memcpy(&u, &x, 4);
    const uint32_t exponent = u >> 23 & 0xFFu;
    if (exponent < 2u || exponent > 252u) return x;
    u += (uint32_t)(((int)((u * 2654435761u) >> 24) % 3 - 1) * ulps);
    std::memcpy(&x, &u, 4);
    return x;
}
inline float host_rcpf(float x) { return host_nudge(1.0f / x, 1); }
inline float host_sqrtf(float x) { return host_nudge(std::sqrt(x), 1); }
#define __builtin_amdgcn_rcpf host_rcpf
#define __builtin_amdgcn_sqrtf host_sqrtf
inline float host_expf(float x) { return host_nudge(std::exp(x), 2); }
inline float host_logf(float x) { return host_nudge(std::log(x), 2); }
#define __expf host_expf
#define __logf host_logf
