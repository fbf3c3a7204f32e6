// fs_mg_device.hpp -- helpers shared by the multigrid kernels.
#pragma once
#include "fs_device.hpp"

namespace fsim {

namespace {

__device__ __forceinline__ float inv_or_zero(float d) { return d > 0.f ? __builtin_amdgcn_rcpf(d) : 0.f; }

// Loads and stores of multigrid storage formats; arithmetic is FP32.  Stores round to nearest even.
__device__ __forceinline__ float ldv(float v) { return v; }
__device__ __forceinline__ float ldv(half16 v) { return (float)__builtin_bit_cast(_Float16, v.bits); }
__device__ __forceinline__ float ldv(bf16 v) { return __uint_as_float((unsigned)v.bits << 16); }
template <class T> __device__ __forceinline__ T stv(float f);
template <> __device__ __forceinline__ float stv<float>(float f) { return f; }
template <> __device__ __forceinline__ half16 stv<half16>(float f)
{
    return half16{__builtin_bit_cast(unsigned short, (_Float16)f)};
}
template <> __device__ __forceinline__ bf16 stv<bf16>(float f)
{
    // round to nearest even on the 16 bits dropped (finite inputs: the levels hold no NaN)
    const unsigned u = __float_as_uint(f);
    return bf16{(unsigned short)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16)};
}

// Two neighbouring values, element-aligned (one load where the hardware allows it).
template <class T> struct __attribute__((packed, aligned(alignof(T)))) Pair {
    T a, b;
};

// XCD-aware tile order.  Workgroups of a launch are dealt to the 8 XCDs round-robin (workgroup b runs
// on XCD b % 8), each XCD with its own L2.  Mapping the workgroups an XCD receives onto a contiguous
// run of row-major tiles keeps neighbouring tiles, whose 8-cell halos overlap, on the same L2.  The
// launch is one-dimensional with exactly gx * gy workgroups; the map is a bijection onto the tiles.
constexpr int kXcds = 8;
__device__ __forceinline__ void xcd_tile(int gx, int gy, int& bx, int& by)
{
    const int n = gx * gy;
    const int b = blockIdx.x;
    const int per = n / kXcds, rem = n % kXcds;
    const int xcd = b % kXcds, q = b / kXcds;
    const int t = xcd * per + min(xcd, rem) + q;
    by = t / gx;
    bx = t - by * gx;
}

}  // namespace

}  // namespace fsim
