// Grid geometry and memory accessors shared by the search kernels.
#pragma once
#include "pgeof_device.hpp"
#include "pgeof_internal.hpp"

namespace pgeof_amd
{

__device__ __forceinline__ int cell_coord(double v, double lo, double inv_h, int g)
{
    double t = (v - lo) * inv_h;
    t = fmin(fmax(t, 0.0), (double)(g - 1));  // NaN -> 0
    return (int)t;
}

// ------------------------------------------------- global-memory access ----
// Pointers that reach a kernel through a table in device memory (the levels
// of the pyramid, moved to scalar registers) lose their address space, and
// the compiler then reads them with flat loads.  A flat load also counts
// against the LDS wait counter, so every LDS access of the heaps would wait
// for the candidate loads in flight; these helpers read and write through
// global-address-space pointers instead (global_load / global_store).
#define PGEOF_GLOBAL __attribute__((address_space(1)))
typedef float pgeof_f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned long long pgeof_u64x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float4 gload(const float4* p, size_t i)
{
    const pgeof_f32x4 v = ((const PGEOF_GLOBAL pgeof_f32x4*)p)[i];
    return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint32_t gload(const uint32_t* p, size_t i)
{
    return ((const PGEOF_GLOBAL uint32_t*)p)[i];
}
__device__ __forceinline__ uint64_t gload(const uint64_t* p, size_t i)
{
    return ((const PGEOF_GLOBAL unsigned long long*)p)[i];
}
// two consecutive 8-byte entries at p (16-byte aligned)
__device__ __forceinline__ ulonglong2 gload2(const uint64_t* p)
{
    const pgeof_u64x2 v = *(const PGEOF_GLOBAL pgeof_u64x2*)p;
    return make_ulonglong2(v.x, v.y);
}
__device__ __forceinline__ void gstore(uint64_t* p, size_t i, uint64_t v)
{
    ((PGEOF_GLOBAL unsigned long long*)p)[i] = v;
}

// distance from v to the slab [lo + c h, lo + (c+1) h], less a safety margin
__device__ __forceinline__ double axis_gap(double v, int c, double lo, double h, double margin)
{
    const double a = lo + (double)c * h, b = a + h;
    const double g = fmax(fmax(a - v, v - b), 0.0) - margin;
    return g > 0.0 ? g : 0.0;
}

// LDS visibility between the lanes of one wavefront
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct Box
{
    int x0, x1, y0, y1, z0, z1;  // inclusive cell ranges; empty when x0 > x1
};

__device__ __forceinline__ Box empty_box() { return Box{1, 0, 1, 0, 1, 0}; }

__device__ __forceinline__ Box cube_box(int cx, int cy, int cz, int n, const Level& G)
{
    return Box{max(cx - n, 0), min(cx + n, G.g[0] - 1), max(cy - n, 0), min(cy + n, G.g[1] - 1), max(cz - n, 0),
               min(cz + n, G.g[2] - 1)};
}

// t-th element (t in [0, hi - lo]) of the order c, c-1, c+1, c-2, c+2, ...
// over [lo, hi] with c in [lo, hi]: alternating while both sides last, then
// the longer side outwards
__device__ __forceinline__ int nth_near(int t, int c, int lo, int hi)
{
    const int below = c - lo, above = hi - c, m = min(below, above);
    if (t <= 2 * m)
    {
        const int d = (t + 1) >> 1;
        return (t & 1) ? c - d : c + d;
    }
    const int r = t - m;
    return below > above ? c - r : c + r;
}

}  // namespace pgeof_amd
