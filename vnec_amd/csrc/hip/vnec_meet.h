// vnec_meet.h — sums of rows that several tiles share, joined by the tiles'
// own workgroups.
#pragma once
#include "vnec_common.h"

// An empty slot: a NaN that no sum is stored as (sums that are NaN are stored
// as the quiet NaN).
#define MEET_EMPTY64 0x7FF4DEADBEEF0001ull
#define MEET_EMPTY32 0x7FA4DEADu

static __global__ void k_meet_empty(int64_t n, int fp32, void *__restrict__ slot)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (fp32) ((uint32_t *)slot)[i] = MEET_EMPTY32;
    else ((uint64_t *)slot)[i] = MEET_EMPTY64;
}

// Partial sums of a row cut by tile boundaries meet pairwise: the row's n
// tiles are the leaves of a binary tree whose node between leaves m - 1 and m
// owns slot[(t0 + m) k].  Of a node's two sides the first to arrive leaves its sum
// in the slot and is done; the second takes it, empties the slot for the next
// launch and goes on with the total.  The tree fixes the order of the sums,
// one atomic exchange carries both the value and its arrival, and nothing is
// waited for.  Launches that share slots must follow one another, and each run
// to its end: every entry of the library puts a plan's on its one stream.
__device__ __forceinline__ bool meet_swap(double *slot, double &s)
{
    typedef unsigned long long u64;
    const u64 mine = s != s ? 0x7FF8000000000000ull : (u64)__double_as_longlong(s);
    const u64 old = __hip_atomic_exchange((u64 *)slot, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (old == MEET_EMPTY64) return false;
    __hip_atomic_store((u64 *)slot, MEET_EMPTY64, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s += __longlong_as_double((long long)old);
    return true;
}
__device__ __forceinline__ bool meet_swap(float *slot, float &s)
{
    const uint32_t mine = s != s ? 0x7FC00000u : (uint32_t)__float_as_int(s);
    const uint32_t old = __hip_atomic_exchange((uint32_t *)slot, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (old == MEET_EMPTY32) return false;
    __hip_atomic_store((uint32_t *)slot, MEET_EMPTY32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s += __int_as_float((int)old);
    return true;
}

template <typename F>
__device__ __forceinline__ void meet_rows(F *slot, int k, int t0, int n, int leaf, F s, F *yrow)
{
    int i = leaf;  // first leaf of the node whose sum is s
    for (int z = 1; z < n; z <<= 1) {
        int m = i + z;  // first leaf of the node's right side
        if (i & z) {
            m = i;
            i -= z;
        } else if (m >= n) {
            continue;  // no right side
        }
        if (!meet_swap(slot + (int64_t)(t0 + m) * k, s)) return;
    }
    *yrow = s;
}
