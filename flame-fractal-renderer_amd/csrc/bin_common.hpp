// Device helpers of the binning kernels (bin_kernels.hip, miss_kernels.hip).
#pragma once

#include "walk.hpp"

namespace ffr {

// Workgroup barriers that order the LDS only: loads and stores of device
// memory stay in flight across them.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The LDS word of cell c of a tile: c with its low five bits (its bank)
// turned by a hash of the rest.  Cells that flames occupy often share their
// low bits (the Sierpinski tetrahedron's occupied cells of a row have x
// digits that avoid y's and z's, so a few banks held them all and the
// counts' atomics queued on them); the hash spreads each group of 32 cells
// over the banks, one bank each.
__device__ __forceinline__ unsigned tile_word(unsigned c)
{
    return c ^ (((c >> 5) * 0x9E3779B1u) >> 27);
}

// reals of a record's words
template <typename PR> __device__ __forceinline__ void put_real(unsigned *w, PR v);
template <> __device__ __forceinline__ void put_real(unsigned *w, float v)
{
    w[0] = __float_as_uint(v);
}
template <> __device__ __forceinline__ void put_real(unsigned *w, double v)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    w[0] = (unsigned)b;
    w[1] = (unsigned)(b >> 32);
}
template <typename PR> __device__ __forceinline__ double get_real(const unsigned *w);
template <> __device__ __forceinline__ double get_real<float>(const unsigned *w)
{
    return (double)__uint_as_float(w[0]);
}
template <> __device__ __forceinline__ double get_real<double>(const unsigned *w)
{
    return __longlong_as_double((long long)(((unsigned long long)w[1] << 32) | w[0]));
}

// the last t in [0, n) with first[t] <= w
__device__ __forceinline__ int last_not_above(const unsigned *first, int n, unsigned w)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (first[mid] <= w)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// Exclusive scan, in place, of an LDS array of n counts by the 1024 lanes
// of a workgroup (per lane, per wave, across the waves); returns the total.
// wsum: 16 words of LDS.  Barriers inside; none after the last write.
__device__ __forceinline__ unsigned lds_scan(unsigned *off, int n, unsigned *wsum)
{
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int per = (n + 1023) / 1024;
    const int t0 = tid * per;
    unsigned mine = 0;
    for (int j = 0; j < per; ++j)
        if (t0 + j < n)
            mine += off[t0 + j];
    unsigned incl = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned y = __shfl_up(incl, d, 64);
        if (lane >= d)
            incl += y;
    }
    if (lane == 63)
        wsum[wave] = incl;
    lds_barrier();
    unsigned before = 0, total = 0;
    for (int w = 0; w < 16; ++w) {
        const unsigned ws = wsum[w];
        before += w < wave ? ws : 0u;
        total += ws;
    }
    unsigned run = before + incl - mine;
    for (int j = 0; j < per; ++j)
        if (t0 + j < n) {
            const unsigned m = off[t0 + j];
            off[t0 + j] = run;
            run += m;
        }
    return total;
}

} // namespace ffr
