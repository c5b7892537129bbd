// lanes.h -- device helpers shared by kernels.hip and paths.hip: global-memory
// accesses, block order and rig look-up, packed 16-bit pairs, DPP moves and
// reductions over groups of lanes.
#pragma once
#include <hip/hip_runtime.h>
#include "rig.h"

namespace sister {

// Device buffers reached through the rig table are generic pointers; casting
// them to the global address space lets the compiler use global_load/store
// with a scalar base (flat accesses need 64-bit per-lane addresses and also
// hold the LDS counter).
template <typename T> using gptr = __attribute__((address_space(1))) T*;
template <typename T> __device__ __forceinline__ gptr<T> G(T* p) { return (gptr<T>)p; }
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint4 LD16(const void* p)
{
    const u32x4 v = *(gptr<const u32x4>)p;
    return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ void ST16(void* p, uint4 v) { *(gptr<u32x4>)p = u32x4{v.x, v.y, v.z, v.w}; }

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x3 __attribute__((ext_vector_type(3)));
template <int N> struct Vec;
template <> struct Vec<1> { typedef uint32_t T; };
template <> struct Vec<2> { typedef u32x2 T; };
template <> struct Vec<3> { typedef u32x3 T; };
template <> struct Vec<4> { typedef u32x4 T; };


// Raw buffers: a base and a size in bytes; an access of N dwords at a lane
// offset past the size reads 0 and stores nothing, so a lane that has nothing
// to move takes kDropped instead of a branch.
constexpr uint32_t kDropped = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf(uint8_t* base, uint32_t bytes = 0x7FFFFFFFu)
{
    return __builtin_amdgcn_make_buffer_rsrc(base, 0, (int)bytes, 0x00020000);
}
template <int N> __device__ __forceinline__ void buf_store(const uint32_t* w, __amdgpu_buffer_rsrc_t r, uint32_t off)
{
    if constexpr (N == 1) __builtin_amdgcn_raw_buffer_store_b32(w[0], r, off, 0, 0);
    else if constexpr (N == 2) __builtin_amdgcn_raw_buffer_store_b64(u32x2{w[0], w[1]}, r, off, 0, 0);
    else if constexpr (N == 3) __builtin_amdgcn_raw_buffer_store_b96(u32x3{w[0], w[1], w[2]}, r, off, 0, 0);
    else __builtin_amdgcn_raw_buffer_store_b128(u32x4{w[0], w[1], w[2], w[3]}, r, off, 0, 0);
}
template <int N> __device__ __forceinline__ void buf_load(uint32_t* w, __amdgpu_buffer_rsrc_t r, uint32_t off)
{
    if constexpr (N == 1) {
        w[0] = __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
    } else {
        typename Vec<N>::T v;
        if constexpr (N == 2) v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
        else if constexpr (N == 3) v = __builtin_amdgcn_raw_buffer_load_b96(r, off, 0, 0);
        else v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
#pragma unroll
        for (int i = 0; i < N; i++) w[i] = v[i];
    }
}

// Block index b of an n-block grid taken in XCD-contiguous order: with
// round-robin dispatch block b runs on XCD b % 8, so the XCD gets the
// consecutive logical blocks [start(b % 8), start(b % 8 + 1)) (the first
// n % 8 XCDs one more than the others).  A bijection of [0, n).
__device__ __forceinline__ int xcd_order(int b, int n)
{
    const int x = b & 7, k = b >> 3, q = n >> 3, r = n & 7;
    return x < r ? x * (q + 1) + k : r * (q + 1) + (x - r) * q + k;
}

__device__ __forceinline__ int find_rig(const int* __restrict__ bs, int n, int b)
{
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if (bs[mid] <= b) lo = mid; else hi = mid;
    }
    return lo;
}

// compile-time loop: f(integral_constant<int, I>) for I in [B, E), so register
// arrays indexed by I are never indexed at run time
template <int I> struct IC { static constexpr int value = I; };
template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f)
{
    if constexpr (B < E) {
        f(IC<B>{});
        static_for<B + 1, E>(f);
    }
}

typedef unsigned short us2 __attribute__((ext_vector_type(2)));
constexpr uint32_t kGuard2 = 0x3FFF3FFFu;

__device__ __forceinline__ us2 U2(uint32_t v) { return __builtin_bit_cast(us2, v); }
__device__ __forceinline__ uint32_t W2(us2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ us2 umin2(us2 a, us2 b) { return __builtin_elementwise_min(a, b); }
__device__ __forceinline__ us2 umax2(us2 a, us2 b) { return __builtin_elementwise_max(a, b); }
// minimum and maximum of three pairs in one instruction.  gfx950 has packed
// three-input forms for halves only; non-negative halves order like their bit
// patterns, and finite ones (patterns below 0x7C00) pass through unchanged,
// denormals included (f16 denormals are on by default): exact for integers
// below 0x7C00.
__device__ __forceinline__ us2 umin3(us2 a, us2 b, us2 c)
{
    uint32_t r;
    asm("v_pk_minimum3_f16 %0, %1, %2, %3" : "=v"(r) : "v"(__builtin_bit_cast(uint32_t, a)),
        "v"(__builtin_bit_cast(uint32_t, b)), "v"(__builtin_bit_cast(uint32_t, c)));
    return __builtin_bit_cast(us2, r);
}
__device__ __forceinline__ us2 umax3(us2 a, us2 b, us2 c)
{
    uint32_t r;
    asm("v_pk_maximum3_f16 %0, %1, %2, %3" : "=v"(r) : "v"(__builtin_bit_cast(uint32_t, a)),
        "v"(__builtin_bit_cast(uint32_t, b)), "v"(__builtin_bit_cast(uint32_t, c)));
    return __builtin_bit_cast(us2, r);
}
// bytes b0,b1 of w -> pair (b0, b1); bytes b2,b3 -> pair (b2, b3)
__device__ __forceinline__ uint32_t bytes01(uint32_t w) { return __builtin_amdgcn_perm(w, w, 0x0c010c00u); }
__device__ __forceinline__ uint32_t bytes23(uint32_t w) { return __builtin_amdgcn_perm(w, w, 0x0c030c02u); }
// low bytes of pairs a, b -> one word (a.lo, a.hi, b.lo, b.hi)
__device__ __forceinline__ uint32_t pack4(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x06040200u); }
__device__ __forceinline__ uint32_t dup16(uint32_t v) { return v | (v << 16); }
// 255 -> 0 in both halves (paramInvalidDispCost, sgm.cpp:109-110,146-147)
__device__ __forceinline__ uint32_t tilde2(uint32_t p)
{
    uint32_t lo = (p & 0xFFFFu) == 255u ? 0u : (p & 0xFFFFu);
    uint32_t hi = (p >> 16) == 255u ? 0u : (p >> 16);
    return lo | (hi << 16);
}

// unpack one 16-byte chunk of a u8 volume into 8 pairs, and back
__device__ __forceinline__ void unpack16(const uint4& v, uint32_t (&p)[8])
{
    p[0] = bytes01(v.x); p[1] = bytes23(v.x);
    p[2] = bytes01(v.y); p[3] = bytes23(v.y);
    p[4] = bytes01(v.z); p[5] = bytes23(v.z);
    p[6] = bytes01(v.w); p[7] = bytes23(v.w);
}
__device__ __forceinline__ uint4 pack16(const uint32_t (&p)[8])
{
    return make_uint4(pack4(p[0], p[1]), pack4(p[2], p[3]), pack4(p[4], p[5]), pack4(p[6], p[7]));
}

// DPP within a 16-lane row: lane i gets lane i-1 (shr) / i+1 (shl); 0 where
// the source is outside the row (one DPP move, no fill value to materialise)
__device__ __forceinline__ uint32_t row_shr1(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, true);
}
__device__ __forceinline__ uint32_t row_shl1(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x101, 0xF, 0xF, true);
}
// the same over the wave's 64 lanes
__device__ __forceinline__ uint32_t wave_from_left(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x138, 0xF, 0xF, true);
}
__device__ __forceinline__ uint32_t wave_from_right(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x130, 0xF, 0xF, true);
}
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_min(uint32_t v)
{
    return min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, CTRL, 0xF, 0xF, false));
}
// minimum over each aligned group of KL lanes (KL in 1,2,4,8,16), in every lane
template <int KL>
__device__ __forceinline__ uint32_t group_min(uint32_t v)
{
    if (KL >= 2) v = dpp_min<0xB1>(v);    // quad_perm [1,0,3,2]
    if (KL >= 4) v = dpp_min<0x4E>(v);    // quad_perm [2,3,0,1]
    if (KL >= 8) v = dpp_min<0x141>(v);   // row_half_mirror
    if (KL >= 16) v = dpp_min<0x140>(v);  // row_mirror
    return v;
}


}  // namespace sister
