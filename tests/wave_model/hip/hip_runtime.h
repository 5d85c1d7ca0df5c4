// hip/hip_runtime.h — what the fixed-dt kernels use of HIP, for a build of their source by the
// host compiler in which every lane is a fiber (wave_model.cpp): the wave operations meet all
// 64 lanes of a wave, __syncthreads all waves of the workgroup, and between two of them the
// waves run in whatever order the test asks for.  Test infrastructure only.
#pragma once

#include <math.h>
#include <stddef.h>
#include <stdint.h>
#include <string.h>

#define __device__
#define __host__
#define __global__
#define __shared__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __align__(n)

namespace wave_model {

enum Op : uint32_t { kBallot = 1, kReadFirst, kReadLane, kDpp, kShfl, kShflUp, kShflXor, kWaveBarrier,
                     kWorkgroupBarrier = 0x10000 };
struct Index { unsigned x; };
Index thread_index();
Index block_index();
int lane();
// Waits for the wave's 64 lanes (a workgroup barrier: op | line, for all its waves too); the
// values they brought.
const uint64_t* meet(uint32_t op, uint64_t v);

}  // namespace wave_model

#define threadIdx (::wave_model::thread_index())
#define blockIdx (::wave_model::block_index())
#define __syncthreads() ((void)::wave_model::meet(::wave_model::kWorkgroupBarrier | __LINE__, 0))

struct float4 { float x, y, z, w; };
struct uint2 { uint32_t x, y; };
struct uint4 { uint32_t x, y, z, w; };
struct dim3 { unsigned x, y, z; dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {} };
inline float4 make_float4(float x, float y, float z, float w) { return {x, y, z, w}; }
inline uint2 make_uint2(uint32_t x, uint32_t y) { return {x, y}; }

template <class To, class From> inline To bits_as(From v)
{
    static_assert(sizeof(To) == sizeof(From), "a cast of bits");
    To r;
    memcpy(&r, &v, sizeof r);
    return r;
}
inline uint32_t __float_as_uint(float v) { return bits_as<uint32_t>(v); }
inline float __uint_as_float(uint32_t v) { return bits_as<float>(v); }
inline float __int_as_float(int v) { return bits_as<float>(v); }
inline long long __double_as_longlong(double v) { return bits_as<long long>(v); }
inline double __longlong_as_double(long long v) { return bits_as<double>(v); }
inline int __popcll(unsigned long long v) { return __builtin_popcountll(v); }
template <class T> inline T min(T a, T b) { return b < a ? b : a; }
template <class T> inline T max(T a, T b) { return a < b ? b : a; }

// ---- wave operations (every lane of the wave takes part) -----------------------------
inline unsigned __lane_id() { return (unsigned)wave_model::lane(); }
inline uint64_t __ballot(bool p)
{
    const uint64_t* v = wave_model::meet(wave_model::kBallot, p ? 1u : 0u);
    uint64_t m = 0;
    for (int l = 0; l < 64; ++l) m |= v[l] << l;
    return m;
}
inline int __builtin_amdgcn_readfirstlane(int v)
{
    return (int)(uint32_t)wave_model::meet(wave_model::kReadFirst, (uint32_t)v)[0];
}
inline int __builtin_amdgcn_readlane(int v, int l)
{
    return (int)(uint32_t)wave_model::meet(wave_model::kReadLane, (uint32_t)v)[l & 63];
}
inline uint32_t __builtin_amdgcn_mbcnt_lo(uint32_t m, uint32_t c)
{
    const int l = wave_model::lane();
    return c + (uint32_t)__builtin_popcount(l >= 32 ? m : m & ((1u << l) - 1u));
}
inline uint32_t __builtin_amdgcn_mbcnt_hi(uint32_t m, uint32_t c)
{
    const int l = wave_model::lane();
    return c + (uint32_t)__builtin_popcount(l <= 32 ? 0u : m & ((1u << (l - 32)) - 1u));
}
// quad_perm, row_mirror, row_half_mirror and row_shr: what the kernels use
inline int __builtin_amdgcn_update_dpp(int old, int v, int ctrl, int, int, bool zero)
{
    const uint64_t* b = wave_model::meet(wave_model::kDpp, (uint32_t)v);
    const int l = wave_model::lane(), row = l & 48, q = l & 15;
    int src = -1;
    if (ctrl < 0x100) src = (l & ~3) | ((ctrl >> (2 * (l & 3))) & 3);
    else if (ctrl == 0x140) src = row | (15 - q);
    else if (ctrl == 0x141) src = (l & ~7) | (7 - (l & 7));
    else if (ctrl > 0x110 && ctrl < 0x120) src = q >= ctrl - 0x110 ? l - (ctrl - 0x110) : -1;
    else __builtin_trap();
    return src < 0 ? (zero ? 0 : old) : (int)(uint32_t)b[src];
}
template <class T> inline T shuffled(const uint64_t* b, int src)
{
    return bits_as<T>((uint32_t)b[src & 63]);
}
template <class T> inline T __shfl(T v, int src, int = 64)
{
    return shuffled<T>(wave_model::meet(wave_model::kShfl, bits_as<uint32_t>(v)), src);
}
template <class T> inline T __shfl_up(T v, int off)
{
    const int l = wave_model::lane();
    return shuffled<T>(wave_model::meet(wave_model::kShflUp, bits_as<uint32_t>(v)), l >= off ? l - off : l);
}
template <class T> inline T __shfl_xor(T v, int off, int = 64)
{
    const int l = wave_model::lane();
    return shuffled<T>(wave_model::meet(wave_model::kShflXor, bits_as<uint32_t>(v)), l ^ off);
}
inline void __builtin_amdgcn_wave_barrier() { wave_model::meet(wave_model::kWaveBarrier, 0); }
inline void __builtin_amdgcn_fence(int, const char*, const char* = nullptr) {}

// ---- atomics (a lane runs alone between two meetings) --------------------------------
template <class T> inline T atomicAdd(T* p, T v) { const T o = *p; *p = o + v; return o; }
template <class T> inline T atomicOr(T* p, T v) { const T o = *p; *p = o | v; return o; }
inline uint32_t atomicMin(uint32_t* p, uint32_t v) { const uint32_t o = *p; if (v < o) *p = v; return o; }

// ---- host names that the headers declare or call -------------------------------------
typedef int hipError_t;
typedef struct ihipStream_t* hipStream_t;
constexpr hipError_t hipSuccess = 0, hipErrorInvalidValue = 1;
constexpr int hipFuncAttributeMaxDynamicSharedMemorySize = 0;
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipFuncSetAttribute(const void*, int, int) { return hipSuccess; }
inline hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t)
{
    *n = 1;
    return hipSuccess;
}
#define hipLaunchKernelGGL(...) ((void)0)
