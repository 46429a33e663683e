// Work items of grids no taller than the row span, for the kernels that build
// them (bh_force.hip, bh_summ.hip).
#pragma once
#include "bh_common.h"
#include "bh_kernels.h"

// The i-th run of pitem particles of column x, whose rows start at o[0 .. G].
__device__ __forceinline__ Item run_item(const int32_t* __restrict__ o, int G, int s, int x, int i,
                                         int pitem)
{
    Item it;
    it.p0 = o[0] + i * pitem;
    it.np = min(pitem, o[G] - it.p0);
    it.sys = s;
    it.cx = x;
    // rows of the first and last particle: the last row that starts at or before it
    int y[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int p = u ? it.p0 + it.np - 1 : it.p0;
        int lo = 0, hi = G - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (o[mid] <= p) lo = mid; else hi = mid - 1;
        }
        y[u] = lo;
    }
    it.y0 = y[0];
    it.y1 = y[1];
    it.pad0 = 0;
    it.pad1 = 0;
    return it;
}

// Where no item can reach the row span (every grid at most yspan rows), a
// column's items are its runs of pitem particles: item t of the pass, in column
// col, starts pitem (t - at) particles into it (at: the column's first item).
__device__ __forceinline__ void write_run(const SysDev* __restrict__ sys, int S, int col, int t,
                                          int at, const int32_t* __restrict__ offsets, int pitem,
                                          Item* __restrict__ items)
{
    const int s = sys_of_col(sys, S, col);
    const SysDev& d = sys[s];
    const int x = (int)(col - d.col_off);
    items[t] = run_item(offsets + d.c_off + (int64_t)x * d.G, d.G, s, x, t - at, pitem);
}

__device__ __forceinline__ int col_of_item(const int32_t* col_off, int ncols, int t)
{
    int lo = 0, hi = ncols - 1;   // the last column whose first item is at or before t
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (col_off[mid] <= t) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// Counts and scans the runs of ncols <= COLS columns by one block of THREADS, and
// writes the items too where they are few (write != 0).
template <int THREADS, int COLS>
__device__ __forceinline__ void items_runs(const SysDev* __restrict__ sys, int S, int ncols,
                                           const int32_t* __restrict__ offsets, int pitem,
                                           int32_t* col_off, Item* __restrict__ items,
                                           int64_t max_items, int32_t* stats, int write,
                                           int32_t* at, int* wsum)
{
    constexpr int R = COLS / THREADS;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int v[R], sum = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int col = threadIdx.x * R + r;
        v[r] = 0;
        if (col < ncols) {
            const SysDev& d = sys[sys_of_col(sys, S, col)];
            const int32_t* o = offsets + d.c_off + (int64_t)(col - d.col_off) * d.G;
            v[r] = (o[d.G] - o[0] + pitem - 1) / pitem;
        }
        sum += v[r];
    }
    int inc = sum;
#pragma unroll
    for (int o = 1; o < BH_WAVE; o <<= 1) {
        const int a = __shfl_up(inc, o, BH_WAVE);
        if (lane >= o) inc += a;
    }
    if (lane == BH_WAVE - 1) wsum[w] = inc;
    __syncthreads();
    int before = 0, total = 0;
#pragma unroll
    for (int k = 0; k < THREADS / BH_WAVE; ++k) {
        if (k < w) before += wsum[k];
        total += wsum[k];
    }
    int e = before + inc - sum;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int col = threadIdx.x * R + r;
        if (col < ncols) {
            at[col] = e;
            col_off[col] = e;
        }
        e += v[r];
    }
    const int n = (int)min((int64_t)total, max_items);
    if (threadIdx.x == 0) {
        col_off[ncols] = total;
        stats[ST_NITEMS] = n;
        if (total > max_items) atomicOr(&stats[ST_ERR], BH_ERR_ITEMS);
    }
    if (!write) return;
    __syncthreads();
    for (int t = threadIdx.x; t < n; t += THREADS) {
        const int col = col_of_item(at, ncols, t);
        write_run(sys, S, col, t, at[col], offsets, pitem, items);
    }
}
