// kernel_util.h -- device helpers shared by the kernels (address spaces,
// cross-lane moves, coefficient planes) and the launch helpers.
#pragma once

#include <hip/hip_runtime.h>

#include "engine.h"
#include "hip_check.h"

namespace aw {

// Pointers read out of DevInst are generic; accesses through them compile to
// flat instructions, which count against the LDS wait counter too, so every
// LDS wait would also drain outstanding HBM stores.  gp() restores the
// global address space so loads and stores become global_* instructions.
#define AW_GLOBAL __attribute__((address_space(1)))
template <class X>
__device__ inline AW_GLOBAL X *gp(X *p)
{
    return (AW_GLOBAL X *)p;
}

#define AW_LDS __attribute__((address_space(3)))

// Read-only data indexed by wave-uniform values (block bounds, uniforms)
// goes through the constant address space so it is fetched with scalar loads.
#define AW_CONST __attribute__((address_space(4)))
template <class X>
__device__ inline AW_CONST const X *cp(const X *p)
{
    return (AW_CONST const X *)p;
}

// index i such that off[i] <= x < off[i+1]
template <class PT, class X>
__device__ inline int find_owner(PT off, int n, X x)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= x) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

//===========================================================================
// cross-lane moves (DPP).  A lane whose source is outside the wave (wave
// shifts) or outside its 16-lane row (row shifts) receives 0.

constexpr int DPP_ROW_SHR1 = 0x111, DPP_ROW_SHR2 = 0x112, DPP_ROW_SHR4 = 0x114,
              DPP_ROW_SHR8 = 0x118, DPP_WAVE_SHL1 = 0x130, DPP_WAVE_SHR1 = 0x138;

template <int CTRL>
__device__ __forceinline__ int dpp_i(int x)
{
    return __builtin_amdgcn_mov_dpp(x, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ float dpp_r(float x)
{
    return __int_as_float(dpp_i<CTRL>(__float_as_int(x)));
}
template <int CTRL>
__device__ __forceinline__ double dpp_r(double x)
{
    const long long v = __double_as_longlong(x);
    const unsigned lo = (unsigned)dpp_i<CTRL>((int)v);
    const unsigned hi = (unsigned)dpp_i<CTRL>((int)(v >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

__device__ __forceinline__ double readlane_d(double x, int l)
{
    const long long v = __double_as_longlong(x);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)v, l);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(v >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// the slots of a lane in a lane-run row (slot_pos), loaded and stored up to 16
// bytes at a time
template <class X, int R>
struct SlotPiece {
    static constexpr int N = slot_vec(R) * sizeof(X) <= 16 ? slot_vec(R) : 16 / sizeof(X);
    typedef X type __attribute__((ext_vector_type(N)));
};
template <int R, class X>
__device__ __forceinline__ void slots_load(const AW_GLOBAL X *row, int lane, X (&x)[R])
{
    using P = SlotPiece<X, R>;
#pragma unroll
    for (int r = 0; r < R; r += P::N) {
        const auto v = *(const AW_GLOBAL typename P::type *)(row + slot_pos(r, lane, R));
#pragma unroll
        for (int k = 0; k < P::N; k++) x[r + k] = v[k];
    }
}
template <int R, class X>
__device__ __forceinline__ void slots_store(AW_GLOBAL X *row, int lane, const X (&x)[R])
{
    using P = SlotPiece<X, R>;
#pragma unroll
    for (int r = 0; r < R; r += P::N) {
        typename P::type v;
#pragma unroll
        for (int k = 0; k < P::N; k++) v[k] = x[r + k];
        *(AW_GLOBAL typename P::type *)(row + slot_pos(r, lane, R)) = v;
    }
}

template <class Real>
__device__ __forceinline__ const AW_GLOBAL Real *planes(const DevInst &d, int b, int RW)
{
    if (sizeof(Real) == 4)
        return (const AW_GLOBAL Real *)(gp(d.lcoef32) + (size_t)b * NCOEF * RW);
    return (const AW_GLOBAL Real *)(gp(d.lcoef) + (size_t)b * NCOEF * RW);
}

__device__ __forceinline__ float readlane_r(float x, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}
__device__ __forceinline__ double readlane_r(double x, int l)
{
    return readlane_d(x, l);
}

// x of the lane addr / 4 (ds_bpermute)
__device__ __forceinline__ float bperm_r(float x, int addr)
{
    return __int_as_float(__builtin_amdgcn_ds_bpermute(addr, __float_as_int(x)));
}
__device__ __forceinline__ double bperm_r(double x, int addr)
{
    const long long v = __double_as_longlong(x);
    const unsigned lo = (unsigned)__builtin_amdgcn_ds_bpermute(addr, (int)v);
    const unsigned hi = (unsigned)__builtin_amdgcn_ds_bpermute(addr, (int)(v >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Raises a kernel's dynamic-LDS limit to sh bytes (engine.hip): it only ever
// rises, under one lock, so a batch on another host thread that set a larger
// limit for the same kernel is never undercut between its call and its launch.
int set_lds_limit(const void *kern, size_t sh);

}  // namespace aw
