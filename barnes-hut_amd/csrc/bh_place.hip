// Placement phase: bounding box -> cell keys + histogram -> offsets ->
// ordered permutation -> gather.  Replaces python-bh's
//   set_particles_bounding_box   barneshut/implementations/base.py:211-239
//   g_place_particles            barneshut/kernels/grid_decomposition/gpu/grid.py:15-50
//   g_calculate_box_cumm         .../gpu/grid.py:52-60
//   g_sort_particles             .../gpu/grid.py:62-76
// with the ordering of the sequential path (implementations/sequential.py:32-50):
// x-major cell key, and inside a cell numpy's structured-sort tie rule
// (px, py, mass, vx, vy, ax, ay, pid), so the permutation is deterministic.
#include <limits.h>

#include "bh_common.h"
#include "bh_kernels.h"

// ---------------------------------------------------------------- fills
__global__ void k_fill_i32(int32_t* p, int64_t n, int32_t v)
{
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = v;
}

__global__ void k_fill_f64(double* p, int64_t n, double v)
{
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = v;
}

// Everything a placement clears: the stats block, the cell counts and the
// bounding boxes (one launch).
__global__ __launch_bounds__(256) void k_place_init(int32_t* stats, int32_t* counts, int64_t C,
                                                    uint64_t* bb, int S)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    if (t < ST_COUNT) stats[t] = 0;
    for (int64_t s = t; s < S; s += stride) {
        bb[4 * s + 0] = ~0ull;   // min x (ordered key)
        bb[4 * s + 1] = ~0ull;   // min y
        bb[4 * s + 2] = 0ull;    // max x
        bb[4 * s + 3] = 0ull;    // max y
    }
    for (int64_t c = t; c < C; c += stride) counts[c] = 0;
}

// ---------------------------------------------------------------- bbox
// Atomic min/max of the ordered keys; skipped when the stored value already
// bounds ours (stored minima only fall and maxima only rise, so a stale read
// can only cause an unneeded atomic, never a missed one).
// By lanes 0 to 3, an extreme each: one after the other they made k_bbox 6.8 instead
// of 5.2 us on 16,384 particles, 11 instead of 6.5 us on 40 systems.
__device__ __forceinline__ void bbox_flush(uint64_t* bb, int s, double mnx, double mny, double mxx,
                                           double mxy)
{
    const int k = threadIdx.x & 63;
    if (k >= 4) return;
    unsigned long long* b = (unsigned long long*)&bb[4 * s + k];
    const unsigned long long key = bh_ord_key(k == 0 ? mnx : k == 1 ? mny : k == 2 ? mxx : mxy);
    const unsigned long long had = __atomic_load_n(b, __ATOMIC_RELAXED);
    if (k < 2 && key < had) atomicMin(b, key);
    if (k >= 2 && key > had) atomicMax(b, key);
}

// Each wave covers `rounds` runs of 64 R consecutive particles, all of a run's
// loads issued before the first is used; min/max are exact, so the reduction
// order does not matter.  Two blocks a CU with as many rounds as it takes: a
// block's look at the stored extremes costs ~15 ns of one cache line's time, so a
// block per 2048 rows took 157 us on 10M particles, 116 on 4.2M and 245 on 512
// systems, against 58, 40 and 181 (the rows: 43, 18 and 115 at copy rate).
// Rows of one system are consecutive: a wave reduces when the system changes
// (a block of one system reduces over the block).
template <int R>
__global__ __launch_bounds__(256) void k_bbox(const double* __restrict__ px,
                                              const double* __restrict__ py,
                                              const int32_t* __restrict__ sys_of, int64_t N,
                                              int rounds, uint64_t* bb, int32_t* stats)
{
    const double inf = __longlong_as_double(0x7ff0000000000000ll);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    int cur = -1;   // system of the running extremes (wave-uniform)
    double mnx = inf, mny = inf, mxx = -inf, mxy = -inf;
    bool bad = false;
    auto reduce = [&]() {
        mnx = wave_min(mnx);
        mny = wave_min(mny);
        mxx = wave_max(mxx);
        mxy = wave_max(mxy);
    };
    auto flush = [&]() {
        if (cur < 0) return;
        reduce();
        bbox_flush(bb, cur, mnx, mny, mxx, mxy);
        mnx = inf; mny = inf; mxx = -inf; mxy = -inf;
    };
    // a wave's rows: `rounds` runs of 64 R, one after the other
    int64_t base = ((int64_t)blockIdx.x * 4 + wid) * (64 * R) * rounds;
    for (int k = 0; k < rounds && base < N; ++k, base += 64 * R) {
        int sv[R];
        double xv[R], yv[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int64_t i = base + 64 * r + lane;
            const bool in = i < N;
            sv[r] = in ? sys_of[i] : -1;
            xv[r] = in ? px[i] : 0.0;
            yv[r] = in ? py[i] : 0.0;
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const bool fin = isfinite(xv[r]) && isfinite(yv[r]);
            if (sv[r] >= 0 && !fin) bad = true;
            unsigned long long todo = __ballot(sv[r] >= 0);
            while (todo) {   // the systems of these 64 rows, nearly always one
                const int s = __builtin_amdgcn_readlane(sv[r], __ffsll((long long)todo) - 1);
                if (s != cur) {
                    flush();
                    cur = s;
                }
                if (sv[r] == s && fin) {
                    mnx = fmin(mnx, xv[r]);
                    mxx = fmax(mxx, xv[r]);
                    mny = fmin(mny, yv[r]);
                    mxy = fmax(mxy, yv[r]);
                }
                todo &= ~__ballot(sv[r] == s);
            }
        }
    }
    __shared__ double red[4][4];
    __shared__ int wsys[4];
    if (cur >= 0) reduce();
    if (lane == 0) {
        wsys[wid] = cur;
        red[wid][0] = mnx;
        red[wid][1] = mny;
        red[wid][2] = mxx;
        red[wid][3] = mxy;
    }
    if (__any(bad) && lane == 0) atomicOr(&stats[ST_ERR], BH_ERR_NONFINITE);
    __syncthreads();
    if (wid > 0) return;
    for (int v = 0; v < 4; ++v) {   // waves of one system meet here
        if (wsys[v] < 0) continue;
        if (v + 1 < 4 && wsys[v + 1] == wsys[v]) {
            if (lane < 4)
                red[v + 1][lane] = lane < 2 ? fmin(red[v + 1][lane], red[v][lane])
                                            : fmax(red[v + 1][lane], red[v][lane]);
            __builtin_amdgcn_wave_barrier();
        } else {
            bbox_flush(bb, wsys[v], red[v][0], red[v][1], red[v][2], red[v][3]);
        }
    }
}

template __global__ void k_bbox<4>(const double*, const double*, const int32_t*, int64_t, int,
                                   uint64_t*, int32_t*);
template __global__ void k_bbox<8>(const double*, const double*, const int32_t*, int64_t, int,
                                   uint64_t*, int32_t*);

// ---------------------------------------------------------------- keys + histogram
struct Box {
    double min_x, min_y, max_x, max_y, step;
    int64_t c_off;
    int32_t G;
};

// A system's box from its extremes: helpers/grid.py:15-22 square-up,
// base.py:237 step, exactly in FP64.
__device__ __forceinline__ Box square_box(const SysDev& sys, double min_x, double min_y,
                                          double max_x, double max_y)
{
    Box d;
    d.min_x = min_x;
    d.min_y = min_y;
    d.max_x = max_x;
    d.max_y = max_y;
    const double xe = d.max_x - d.min_x, ye = d.max_y - d.min_y;
    if (xe > ye) {
        d.max_y += (xe - ye);
    } else if (ye > xe) {
        d.max_x += (ye - xe);
    }
    d.G = sys.G;
    d.c_off = sys.c_off;
    d.step = (d.max_x - d.min_x) / (double)d.G;
    return d;
}

__device__ __forceinline__ Box box_of(const SysDev* sys, const uint64_t* bb, int s)
{
    return square_box(sys[s], bh_ord_val(bb[4 * s + 0]), bh_ord_val(bb[4 * s + 1]),
                      bh_ord_val(bb[4 * s + 2]), bh_ord_val(bb[4 * s + 3]));
}

// Whether the box has an extent.
__device__ __forceinline__ bool store_box(SysDev& sys, const Box& d)
{
    sys.min_x = d.min_x;
    sys.min_y = d.min_y;
    sys.max_x = d.max_x;
    sys.max_y = d.max_y;
    sys.step = d.step;
    sys.com_out = 0;
    return d.step > 0.0 && isfinite(d.step);
}

// sequential.py:32-34: g = clip(floor((p - min) / step), 0, G-1), IEEE division.
__device__ __forceinline__ int32_t cell_key(double x, double y, const Box& d)
{
    double fx = floor((x - d.min_x) / d.step);
    double fy = floor((y - d.min_y) / d.step);
    double gm = (double)(d.G - 1);
    fx = fx < 0.0 ? 0.0 : (fx > gm ? gm : fx);
    fy = fy < 0.0 ? 0.0 : (fy > gm ? gm : fy);
    int gx = (int)fx, gy = (int)fy;
    // second clamp keeps a NaN coordinate (already flagged) inside the grid
    gx = gx < 0 ? 0 : (gx > d.G - 1 ? d.G - 1 : gx);
    gy = gy < 0 ? 0 : (gy > d.G - 1 ? d.G - 1 : gy);
    return (int32_t)(d.c_off + (int64_t)gx * d.G + gy);
}

__device__ __forceinline__ void block_minmax(int& kmin, int& kmax, int* red)
{
    kmin = wave_min(kmin);
    kmax = wave_max(kmax);
    int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        red[w] = kmin;
        red[4 + w] = kmax;
    }
    __syncthreads();
    kmin = min(min(red[0], red[1]), min(red[2], red[3]));
    kmax = max(max(red[4], red[5]), max(red[6], red[7]));
    __syncthreads();
}

// Keys of 256 R consecutive particles per block, the cells' counts, and each
// row's rank among its cell's rows (in no fixed order; the scatter places rows
// by it, so that it needs no counters of its own).  Rows are counted in LDS first
// and each cell goes to global memory once a block: in a window of keys when the
// block's fit one (the input is the previous step's sorted order, so they are
// nearly contiguous), else in a hash table (unsorted input; rows that find no
// place in four probes go to global memory by themselves).  Bound by latency and,
// unsorted, by additions to the same words: 262,144 unsorted particles with 9,900
// in one cell 202 -> 44 us with k_scatter; 10M sorted ones 370 -> 333 us.  Each row's box comes straight from the
// extremes; the thread of a system's first row stores it (a kernel of its own, or
// a last block behind a device fence, costs more than the division).
template <int R>
__global__ __launch_bounds__(256) void k_keys_hist(const double* __restrict__ px,
                                                   const double* __restrict__ py,
                                                   const int32_t* __restrict__ sys_of,
                                                   SysDev* sys, const uint64_t* __restrict__ bb,
                                                   int64_t N, int32_t* __restrict__ key_out,
                                                   int32_t* __restrict__ rank_out,
                                                   int32_t* __restrict__ counts, int32_t* stats)
{
    __shared__ int32_t hist[HIST_BINS];
    __shared__ int red[8];
    int64_t base = (int64_t)blockIdx.x * (256 * R);
    int kk[R], sr[R];
    double xr[R], yr[R];
    int kmin = INT_MAX, kmax = INT_MIN;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int64_t i = min(base + r * 256 + threadIdx.x, N - 1);
        sr[r] = sys_of[i];
        xr[r] = px[i];
        yr[r] = py[i];
    }
    int cur = sr[0];
    Box d = box_of(sys, bb, cur);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        int64_t i = base + r * 256 + threadIdx.x;
        kk[r] = -1;
        if (i < N) {
            if (sr[r] != cur) {
                cur = sr[r];
                d = box_of(sys, bb, cur);
            }
            if (i == sys[cur].p_off) {
                if (!store_box(sys[cur], d)) atomicOr(&stats[ST_ERR], BH_ERR_DEGENERATE);
            }
            int k = cell_key(xr[r], yr[r], d);
            key_out[i] = k;
            kk[r] = k;
            kmin = min(kmin, k);
            kmax = max(kmax, k);
        }
    }
    block_minmax(kmin, kmax, red);
    if (kmax < kmin) return;   // empty block
    int slot[R], lr[R];
    if ((int64_t)kmax - kmin < HIST_BINS) {
        int span = kmax - kmin + 1;
        for (int b = threadIdx.x; b < span; b += 256) hist[b] = 0;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < R; ++r) lr[r] = kk[r] >= 0 ? atomicAdd(&hist[kk[r] - kmin], 1) : 0;
        __syncthreads();
        for (int b = threadIdx.x; b < span; b += 256)
            if (hist[b]) hist[b] = atomicAdd(&counts[kmin + b], hist[b]);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (kk[r] >= 0) rank_out[base + r * 256 + threadIdx.x] = hist[kk[r] - kmin] + lr[r];
    } else {
        // hist holds HASH keys, then their counts
        constexpr int HASH = R > 2 ? HIST_BINS / 2 : HIST_BINS / 8;
        int32_t* hk = hist;
        int32_t* hc = hist + HASH;
        for (int b = threadIdx.x; b < HASH; b += 256) {
            hk[b] = -1;
            hc[b] = 0;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < R; ++r) {
            slot[r] = -1;
            if (kk[r] < 0) continue;
            unsigned h = ((unsigned)kk[r] * 2654435761u) >> 16;
            for (int t = 0; t < 4 && slot[r] < 0; ++t, ++h) {
                const int old = atomicCAS(&hk[h & (HASH - 1)], -1, kk[r]);
                if (old == -1 || old == kk[r]) slot[r] = h & (HASH - 1);
            }
            if (slot[r] >= 0) lr[r] = atomicAdd(&hc[slot[r]], 1);
        }
        __syncthreads();
        for (int b = threadIdx.x; b < HASH; b += 256)
            if (hc[b]) hc[b] = atomicAdd(&counts[hk[b]], hc[b]);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (kk[r] >= 0)
                rank_out[base + r * 256 + threadIdx.x] =
                    slot[r] >= 0 ? hc[slot[r]] + lr[r] : atomicAdd(&counts[kk[r]], 1);
    }
}

template __global__ void k_keys_hist<2>(const double*, const double*, const int32_t*, SysDev*,
                                        const uint64_t*, int64_t, int32_t*, int32_t*, int32_t*,
                                        int32_t*);
template __global__ void k_keys_hist<8>(const double*, const double*, const int32_t*, SysDev*,
                                        const uint64_t*, int64_t, int32_t*, int32_t*, int32_t*,
                                        int32_t*);

// ---------------------------------------------------------------- scan
// Block-wide exclusive scan of two int sequences (256 or 1024 threads).
__device__ __forceinline__ void block_excl_scan2(int v, int f, int& ev, int& ef, int& tv, int& tf,
                                                 int* sh /* >= 2*16 + 2 ints */)
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
    int iv = v, jf = f;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        int a = __shfl_up(iv, o, BH_WAVE);
        int b = __shfl_up(jf, o, BH_WAVE);
        if (lane >= o) {
            iv += a;
            jf += b;
        }
    }
    if (lane == 63) {
        sh[wid] = iv;
        sh[16 + wid] = jf;
    }
    __syncthreads();
    if (wid == 0) {
        int a = lane < nw ? sh[lane] : 0;
        int b = lane < nw ? sh[16 + lane] : 0;
        int ia = a, ib = b;
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) {
            int x = __shfl_up(ia, o, BH_WAVE);
            int y = __shfl_up(ib, o, BH_WAVE);
            if (lane >= o) {
                ia += x;
                ib += y;
            }
        }
        if (lane < nw) {
            sh[lane] = ia - a;
            sh[16 + lane] = ib - b;
        }
        if (lane == nw - 1) {
            sh[32] = ia;
            sh[33] = ib;
        }
    }
    __syncthreads();
    ev = sh[wid] + iv - v;
    ef = sh[16 + wid] + jf - f;
    tv = sh[32];
    tf = sh[33];
    __syncthreads();
}

// Phase 1: per-tile sums of v = in[c] and f = (in[c] > 0), plus the max.
template <bool CNT>
__global__ __launch_bounds__(256) void k_scan_reduce(const int32_t* __restrict__ in, int64_t n,
                                                     int32_t* bsum, int32_t* bne, int32_t* stats)
{
    __shared__ int sh[40];
    int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * (SCAN_TILE / 256);
    int v = 0, f = 0, mx = 0;
#pragma unroll
    for (int r = 0; r < SCAN_TILE / 256; ++r) {
        int64_t i = base + r;
        if (i < n) {
            int c = in[i];
            v += c;
            f += c > 0;
            mx = max(mx, c);
        }
    }
    int ev, ef, tv, tf;
    block_excl_scan2(v, f, ev, ef, tv, tf, sh);
    if (CNT) {
        // at most one atomic a block, and only if it raises the maximum: one per
        // wave, all on one word, made this kernel 28 us for 1M cells instead of 10
        mx = wave_max(mx);
        if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = mx;
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        bsum[blockIdx.x] = tv;
        if (CNT) {
            bne[blockIdx.x] = tf;
            mx = max(max(sh[0], sh[1]), max(sh[2], sh[3]));
            if (mx > __atomic_load_n(&stats[ST_MAXCOUNT], __ATOMIC_RELAXED))
                atomicMax(&stats[ST_MAXCOUNT], mx);
        }
    }
}

// Phase 2: one block scans the tile sums in place (exclusive).
template <bool CNT>
__global__ __launch_bounds__(1024) void k_scan_blocks(int32_t* bsum, int32_t* bne, int64_t nb,
                                                      int32_t* stats, int total_slot)
{
    __shared__ int sh[40];
    int cv = 0, cf = 0;
    for (int64_t c0 = 0; c0 < nb; c0 += 1024) {
        int64_t i = c0 + threadIdx.x;
        int v = i < nb ? bsum[i] : 0;
        int f = (CNT && i < nb) ? bne[i] : 0;
        int ev, ef, tv, tf;
        block_excl_scan2(v, f, ev, ef, tv, tf, sh);
        if (i < nb) {
            bsum[i] = cv + ev;
            if (CNT) bne[i] = cf + ef;
        }
        cv += tv;
        cf += tf;
    }
    if (threadIdx.x == 0) {
        if (CNT) stats[ST_NCELLS_NE] = cf;
        if (total_slot >= 0) stats[total_slot] = cv;
    }
}

// What the cells' scan leaves for the phases after it, besides the prefixes:
// the list of non-empty cells and zeros in the dense COM array (k_com writes the
// non-empty cells).
__device__ __forceinline__ void clear_com(double* com_dense, int64_t c0, int64_t c1, int threads)
{
    for (int64_t i = 3 * c0 + threadIdx.x; i < 3 * c1; i += threads) com_dense[i] = 0.0;
}

// Phase 3: exclusive prefix per element; out has n + 1 entries.
template <bool CNT>
__global__ __launch_bounds__(256) void k_scan_final(const int32_t* __restrict__ in, int64_t n,
                                                    const int32_t* bsum, const int32_t* bne,
                                                    int32_t* out_v, int32_t* out_f,
                                                    int32_t* ne_list, double* com_dense)
{
    __shared__ int sh[40];
    constexpr int R = SCAN_TILE / 256;
    int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * R;
    int cv[R];
    int v = 0, f = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        int64_t i = base + r;
        cv[r] = i < n ? in[i] : 0;
        v += cv[r];
        f += cv[r] > 0;
    }
    int ev, ef, tv, tf;
    block_excl_scan2(v, f, ev, ef, tv, tf, sh);
    int av = bsum[blockIdx.x] + ev;
    int af = CNT ? bne[blockIdx.x] + ef : 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        int64_t i = base + r;
        if (i < n) {
            out_v[i] = av;
            if (CNT) {
                out_f[i] = af;
                if (cv[r] > 0) ne_list[af] = (int32_t)i;
            }
            av += cv[r];
            af += cv[r] > 0;
            if (i == n - 1) {
                out_v[n] = av;
                if (CNT) out_f[n] = af;
            }
        }
    }
    if (CNT) {
        const int64_t c0 = (int64_t)blockIdx.x * SCAN_TILE;
        clear_com(com_dense, c0, min(n, c0 + SCAN_TILE), 256);
    }
}

// Exclusive scan of n <= 1024 R counts and of their non-empty flags by one block:
// get(i) gives count i, put(i, count, before, non-empty before) takes its place.
// A wave's elements are R rows of 64, so that both ends are contiguous across the
// lanes.  Returns the totals and the largest count.
struct ScanTotals {
    int v, f, mx;
};

template <int R, typename Get, typename Put>
__device__ __forceinline__ ScanTotals scan_block(int n, int* sh /* 48 ints */, Get&& get, Put&& put)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, base = w * (64 * R) + lane;
    const unsigned long long below = (1ull << lane) - 1ull;
    int cv[R], inc[R], v = 0, f = 0, mx = 0;
    unsigned long long ne[R];
#pragma unroll
    for (int r = 0; r < R; ++r) cv[r] = base + 64 * r < n ? get(base + 64 * r) : 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        inc[r] = cv[r];
        mx = max(mx, cv[r]);
        ne[r] = __ballot(cv[r] > 0);
        f += __popcll(ne[r]);
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int a = __shfl_up(inc[r], o, BH_WAVE);
            if (lane >= o) inc[r] += a;
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) v += __builtin_amdgcn_readlane(inc[r], 63);
    mx = wave_max(mx);
    if (lane == 0) {
        sh[w] = v;
        sh[16 + w] = f;
        sh[32 + w] = mx;
    }
    __syncthreads();
    ScanTotals t = {0, 0, 0};
    int av = 0, af = 0;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        if (k == w) {
            av = t.v;
            af = t.f;
        }
        t.v += sh[k];
        t.f += sh[16 + k];
        t.mx = max(t.mx, sh[32 + k]);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int i = base + 64 * r;
        if (i < n) put(i, cv[r], av + inc[r] - cv[r], af + __popcll(ne[r] & below));
        av += __builtin_amdgcn_readlane(inc[r], 63);
        af += __popcll(ne[r]);
    }
    return t;
}

// scan_block with as few rows as hold n.
template <int RMAX, typename Get, typename Put>
__device__ __forceinline__ ScanTotals scan_fit(int n, int* sh, Get&& get, Put&& put)
{
    if (n <= 1024) return scan_block<1>(n, sh, get, put);
    if (n <= 4096) return scan_block<4>(n, sh, get, put);
    return scan_block<RMAX>(n, sh, get, put);
}

// The three phases in one block, for n <= SCAN_ONE (three launches cost more
// than the scan: 13,603 cells 16 us, in one block 13.5; 1,024 cells 3.0).  max_total >= 0: the total is kept within it,
// BH_ERR_ITEMS raised beyond.
template <bool CNT>
__global__ __launch_bounds__(1024) void k_scan_one(const int32_t* __restrict__ in, int n,
                                                   int32_t* out_v, int32_t* out_f, int32_t* ne_list,
                                                   double* com_dense, int32_t* stats,
                                                   int total_slot, int64_t max_total)
{
    __shared__ int sh[48];
    const ScanTotals t = scan_fit<SCAN_ONE / 1024>(
        n, sh, [&](int i) { return in[i]; },
        [&](int i, int c, int av, int af) {
            out_v[i] = av;
            if (CNT) {
                out_f[i] = af;
                if (c > 0) ne_list[af] = i;
            }
        });
    if (threadIdx.x == 0) {
        out_v[n] = t.v;
        if (CNT) {
            out_f[n] = t.f;
            stats[ST_NCELLS_NE] = t.f;
            if (t.mx > 0) atomicMax(&stats[ST_MAXCOUNT], t.mx);
        }
        if (total_slot >= 0) {
            const bool over = max_total >= 0 && t.v > max_total;
            stats[total_slot] = over ? (int32_t)max_total : t.v;
            if (over) atomicOr(&stats[ST_ERR], BH_ERR_ITEMS);
        }
    }
    if (CNT) clear_com(com_dense, 0, n, 1024);
}

template __global__ void k_scan_reduce<true>(const int32_t*, int64_t, int32_t*, int32_t*, int32_t*);
template __global__ void k_scan_reduce<false>(const int32_t*, int64_t, int32_t*, int32_t*, int32_t*);
template __global__ void k_scan_blocks<true>(int32_t*, int32_t*, int64_t, int32_t*, int);
template __global__ void k_scan_blocks<false>(int32_t*, int32_t*, int64_t, int32_t*, int);
template __global__ void k_scan_final<true>(const int32_t*, int64_t, const int32_t*, const int32_t*,
                                            int32_t*, int32_t*, int32_t*, double*);
template __global__ void k_scan_final<false>(const int32_t*, int64_t, const int32_t*,
                                             const int32_t*, int32_t*, int32_t*, int32_t*, double*);
template __global__ void k_scan_one<true>(const int32_t*, int, int32_t*, int32_t*, int32_t*,
                                          double*, int32_t*, int, int64_t);
template __global__ void k_scan_one<false>(const int32_t*, int, int32_t*, int32_t*, int32_t*,
                                           double*, int32_t*, int, int64_t);

// 64-bit key ordered as numpy orders doubles: -0.0 equals +0.0, every NaN is
// equal to every other NaN and sorts after all numbers.
__device__ __forceinline__ uint64_t sort_key(double d)
{
    if (isnan(d)) return ~0ull;
    return bh_ord_key(d == 0.0 ? 0.0 : d);
}

// ---------------------------------------------------------------- scatter
// Counting-sort scatter into cell order: a row's place is its cell's first plus
// its rank among the cell's rows, which k_keys_hist kept; the order inside a
// cell is fixed afterwards by k_sort_units.
// Each row's px and py sort keys travel with it, so that pass reads them
// contiguously (rows clipped to the box edge tie in px by the thousand).
template <int R>
__global__ __launch_bounds__(256) void k_scatter(const int32_t* __restrict__ key, int64_t N,
                                                 const int32_t* __restrict__ offsets,
                                                 const int32_t* __restrict__ rank,
                                                 int32_t* __restrict__ idx_out,
                                                 int32_t* __restrict__ key_sorted,
                                                 const double* __restrict__ px,
                                                 const double* __restrict__ py,
                                                 uint64_t* __restrict__ pxkey_out,
                                                 uint64_t* __restrict__ pykey_out)
{
    const int64_t base = (int64_t)blockIdx.x * (256 * R) + threadIdx.x;
    int kr[R], rr[R];
    double xr[R], yr[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {   // clamped, so that all loads are under way at once
        const int64_t i = min(base + r * 256, N - 1);
        kr[r] = key[i];
        rr[r] = rank[i];
        xr[r] = px[i];
        yr[r] = py[i];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int64_t i = base + r * 256;
        if (i >= N) break;
        const int64_t pos = (int64_t)offsets[kr[r]] + rr[r];
        idx_out[pos] = (int32_t)i;
        key_sorted[pos] = kr[r];
        pxkey_out[pos] = sort_key(xr[r]);
        pykey_out[pos] = sort_key(yr[r]);
    }
}

template __global__ void k_scatter<1>(const int32_t*, int64_t, const int32_t*, const int32_t*,
                                      int32_t*, int32_t*, const double*, const double*, uint64_t*,
                                      uint64_t*);
template __global__ void k_scatter<8>(const int32_t*, int64_t, const int32_t*, const int32_t*,
                                      int32_t*, int32_t*, const double*, const double*, uint64_t*,
                                      uint64_t*);

// ---------------------------------------------------------------- small systems
// Box, keys, counts, scan and scatter of one system of at most PLACE_ONE rows and
// PLACE_CELLS cells in one block: five launches of 2 to 5 us each otherwise, most of
// it latency.  2,000 particles on 11^2 cells: 9.6 us instead of 16; 16,384 on 32^2
// would take 32 instead of 20.
__global__ __launch_bounds__(1024) void k_place_one(
    const double* __restrict__ px, const double* __restrict__ py, SysDev* sys, int N, int C,
    int32_t* __restrict__ key_out, int32_t* __restrict__ rank_out, int32_t* __restrict__ counts,
    int32_t* __restrict__ offsets, int32_t* __restrict__ neprefix, int32_t* __restrict__ ne_list,
    double* __restrict__ com_dense, int32_t* __restrict__ idx_out, int32_t* __restrict__ key_sorted,
    uint64_t* __restrict__ pxkey, uint64_t* __restrict__ pykey, int32_t* __restrict__ stats)
{
    constexpr int RP = PLACE_ONE / 1024;
    __shared__ int32_t cell[PLACE_CELLS];   // counts, then offsets
    __shared__ double red[4][16];
    __shared__ int sh[48], err;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const double inf = __longlong_as_double(0x7ff0000000000000ll);
    double x[RP], y[RP], mnx = inf, mny = inf, mxx = -inf, mxy = -inf;
    if (tid == 0) err = 0;
    for (int c = tid; c < C; c += 1024) cell[c] = 0;
#pragma unroll
    for (int r = 0; r < RP; ++r) {   // clamped: a row past the end repeats the last
        const int i = min(tid + 1024 * r, N - 1);
        x[r] = px[i];
        y[r] = py[i];
    }
    bool bad = false;
#pragma unroll
    for (int r = 0; r < RP; ++r) {
        if (!isfinite(x[r]) || !isfinite(y[r])) {
            bad = true;
            continue;
        }
        mnx = fmin(mnx, x[r]);
        mxx = fmax(mxx, x[r]);
        mny = fmin(mny, y[r]);
        mxy = fmax(mxy, y[r]);
    }
    mnx = wave_min(mnx);
    mny = wave_min(mny);
    mxx = wave_max(mxx);
    mxy = wave_max(mxy);
    __syncthreads();
    if (lane == 0) {
        red[0][w] = mnx;
        red[1][w] = mny;
        red[2][w] = mxx;
        red[3][w] = mxy;
    }
    if (bad) atomicOr(&err, BH_ERR_NONFINITE);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        mnx = fmin(mnx, red[0][k]);
        mny = fmin(mny, red[1][k]);
        mxx = fmax(mxx, red[2][k]);
        mxy = fmax(mxy, red[3][k]);
    }
    const Box d = square_box(sys[0], mnx, mny, mxx, mxy);
    int key[RP], lr[RP];
#pragma unroll
    for (int r = 0; r < RP; ++r) {
        const int i = tid + 1024 * r;
        if (i >= N) continue;
        key[r] = cell_key(x[r], y[r], d);
        lr[r] = atomicAdd(&cell[key[r]], 1);
        key_out[i] = key[r];
        rank_out[i] = lr[r];
    }
    __syncthreads();
    if (tid == 0 && !store_box(sys[0], d)) atomicOr(&err, BH_ERR_DEGENERATE);
    const ScanTotals t = scan_fit<PLACE_CELLS / 1024>(
        C, sh, [&](int i) { return cell[i]; },
        [&](int i, int c, int av, int af) {
            counts[i] = c;
            offsets[i] = av;
            neprefix[i] = af;
            cell[i] = av;
            if (c > 0) ne_list[af] = i;
        });
    clear_com(com_dense, 0, C, 1024);
    __syncthreads();
    if (tid < ST_COUNT) {
        int st = 0;
        if (tid == ST_ERR) st = err;
        if (tid == ST_NCELLS_NE) st = t.f;
        if (tid == ST_MAXCOUNT) st = t.mx;
        stats[tid] = st;
    }
    if (tid == 0) {
        offsets[C] = t.v;
        neprefix[C] = t.f;
    }
#pragma unroll
    for (int r = 0; r < RP; ++r) {
        const int i = tid + 1024 * r;
        if (i >= N) continue;
        const int pos = cell[key[r]] + lr[r];
        idx_out[pos] = i;
        key_sorted[pos] = key[r];
        pxkey[pos] = sort_key(x[r]);
        pykey[pos] = sort_key(y[r]);
    }
}

// ---------------------------------------------------------------- within-cell order
// numpy's structured-sort tie rule after (gx, gy): px, py, mass, vx, vy, ax,
// ay, pid (internals/particle.py:3-9); equal rows keep input order (stable).
// Doubles compare as numpy sorts them: NaN after every number, NaNs equal,
// so the order is total and the ranks always form a permutation.
__device__ __forceinline__ int dcmp(double u, double v)
{
    const bool un = isnan(u), vn = isnan(v);
    if (un || vn) return (int)un - (int)vn;
    return (u < v) ? -1 : (u > v ? 1 : 0);
}

__device__ __forceinline__ bool tie_less(const SortFields& F, int a, int b)
{
    int c;
    if ((c = dcmp(F.py[a], F.py[b]))) return c < 0;
    if ((c = dcmp(F.m[a], F.m[b]))) return c < 0;
    if ((c = dcmp(F.vx[a], F.vx[b]))) return c < 0;
    if ((c = dcmp(F.vy[a], F.vy[b]))) return c < 0;
    if ((c = dcmp(F.ax[a], F.ax[b]))) return c < 0;
    if ((c = dcmp(F.ay[a], F.ay[b]))) return c < 0;
    if (F.pid[a] != F.pid[b]) return F.pid[a] < F.pid[b];
    return a < b;
}

__device__ __forceinline__ bool row_less(const SortFields& F, int a, int b)
{
    int c = dcmp(F.px[a], F.px[b]);
    if (c) return c < 0;
    return tie_less(F, a, b);
}

// A "unit" is a whole cell when the cell holds <= SORT_W particles, else one
// SORT_W-long chunk of it (chunks counted from the cell start).  Every unit
// starts in exactly one aligned SORT_W window; the block owning that window
// ranks the unit's rows in LDS (all of them lie in [w0, w0 + 2*SORT_W)) on
// their px keys, then py keys; the remaining fields are read only for rows
// equal in both.  Bound by the compares: a row's rank is the count of smaller
// px keys of its unit, two instructions a key, eight keys read ahead.  Only
// rows that end up in one slot, that is rows of equal px keys, are looked at a
// second time.  10M particles in cells of 700: 0.85 ms; 3.0 with every key also
// tested for equality in the one loop.  2k in cells of 64: 4.6 us; 8.7.
__global__ __launch_bounds__(SORT_THREADS) void k_sort_units(SortFields F, int64_t N,
                                                    const int32_t* __restrict__ idx_in,
                                                    const int32_t* __restrict__ key_sorted,
                                                    const uint64_t* __restrict__ pxkey,
                                                    const uint64_t* __restrict__ pykey,
                                                    const int32_t* __restrict__ offsets,
                                                    int32_t* __restrict__ idx_out)
{
    __shared__ uint64_t lkx[2 * SORT_W];
    __shared__ uint64_t lky[2 * SORT_W];
    __shared__ int taken[2 * SORT_W];
    __shared__ int64_t lend;
    const int64_t w0 = (int64_t)blockIdx.x * SORT_W;
    if (threadIdx.x == 0) {
        // rows past the window belong to this block only up to the end of the
        // unit that holds the window's last row
        const int64_t ql = min((int64_t)N, w0 + SORT_W) - 1;
        const int k = key_sorted[ql];
        const int64_t a = offsets[k], b = offsets[k + 1];
        int64_t ub = b;
        if (b - a > SORT_W) ub = min(b, a + ((ql - a) / SORT_W) * SORT_W + SORT_W);
        lend = max(ql + 1, ub);
    }
    __syncthreads();
    const int64_t wend = min(lend, w0 + 2 * SORT_W);   // > w0: the window holds a row
    // Each thread's rows t = threadIdx.x + SORT_THREADS r.  Every load below reads a
    // row clamped into [w0, wend), so it is always in bounds and needs no
    // branch: the loads of all rows are issued before the first is waited on
    // (a guarded load per row would wait for each one in turn).
    constexpr int RPT = 2 * SORT_W / SORT_THREADS;
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
        const int t = threadIdx.x + SORT_THREADS * r;
        const int64_t q = min(w0 + t, wend - 1);
        // slots past wend get the last row's keys; no rank reads them (every
        // unit this block ranks ends at or before wend)
        lkx[t] = pxkey[q];
        lky[t] = pykey[q];
        taken[t] = 0;
    }
    __syncthreads();
    // the rows' cells and source rows, then the cells' bounds
    int kr[RPT], er[RPT];
    int64_t ar[RPT], br[RPT];
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
        const int64_t q = min(w0 + threadIdx.x + SORT_THREADS * r, wend - 1);
        kr[r] = key_sorted[q];
        er[r] = idx_in[q];
    }
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
        ar[r] = offsets[kr[r]];
        br[r] = offsets[kr[r] + 1];
    }
    int rank[RPT], j0[RPT], j1[RPT];
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
        const int t = threadIdx.x + SORT_THREADS * r;
        const int64_t q = w0 + t;
        const int64_t a = ar[r], b = br[r];
        int64_t ua = a, ub = b;
        if (b - a > SORT_W) {
            ua = a + ((q - a) / SORT_W) * SORT_W;
            ub = min(b, ua + SORT_W);
        }
        rank[r] = -1;
        // past the block's rows, or a unit owned by another block
        if (q >= wend || ua < w0 || ua >= w0 + SORT_W) continue;
        j0[r] = (int)(ua - w0);
        j1[r] = (int)(ub - w0);
        const uint64_t x = lkx[t];
        int less = 0;
        int j = j0[r];
        for (; j + 7 < j1[r]; j += 8) {
            uint64_t y[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) y[k] = lkx[j + k];
#pragma unroll
            for (int k = 0; k < 8; ++k) less += y[k] < x;
        }
        for (; j < j1[r]; ++j) less += lkx[j] < x;
        rank[r] = j0[r] + less;
        atomicAdd(&taken[rank[r]], 1);   // rows of equal keys meet in one slot
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
        if (rank[r] < 0) continue;
        const int t = threadIdx.x + SORT_THREADS * r;
        const int e = er[r];
        int place = rank[r];
        if (taken[place] > 1) {
            const uint64_t x = lkx[t], xy = lky[t];
            for (int j = j0[r]; j < j1[r]; ++j) {
                if (lkx[j] != x) continue;
                const uint64_t yy = lky[j];
                if (yy < xy || (yy == xy && j != t && tie_less(F, idx_in[w0 + j], e))) ++place;
            }
        }
        idx_out[w0 + place] = e;
    }
}

// Merge pass for cells longer than SORT_W: runs of length R = SORT_W *
// SORT_WAYS^L, counted from the cell start, are merged SORT_WAYS at a time: a
// row's place is its place in its own run plus, by binary search, the rows
// before it in each of the others.  Only rows of such cells are touched; the
// pass is a no-op once R >= max count.  (Pairwise merging searches less per row
// but takes four times the launches, and most of them find nothing to do: 12 at
// 4.5 us on 4.2M particles.  8 at a time: one launch more at 16,384, 262,144 and
// 4.2M particles, 2 to 5 us each; 32 saves one more at 1M but searches twice as
// many runs per row of the largest cells.)
__global__ __launch_bounds__(256) void k_sort_merge(SortFields F, int64_t N,
                                                    const int32_t* __restrict__ idx_in,
                                                    const int32_t* __restrict__ key_sorted,
                                                    const int32_t* __restrict__ offsets,
                                                    int32_t* __restrict__ idx_out, int64_t R,
                                                    const int32_t* __restrict__ stats)
{
    if (R >= stats[ST_MAXCOUNT]) return;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < N; q += stride) {
        int k = key_sorted[q];
        int64_t a = offsets[k], b = offsets[k + 1];
        if (b - a <= SORT_W) continue;
        const int e = idx_in[q];
        const int64_t W0 = a + ((q - a) / (SORT_WAYS * R)) * (SORT_WAYS * R);
        const int own = (int)((q - W0) / R);
        int64_t place = q - (W0 + own * R);
        for (int r = 0; r < SORT_WAYS; ++r) {
            if (r == own) continue;
            const int64_t p0 = W0 + r * R, p1 = min(b, p0 + R);
            if (p0 >= b) break;
            int64_t lo = p0, hi = p1;
            while (lo < hi) {
                const int64_t m = (lo + hi) >> 1;
                if (row_less(F, idx_in[m], e)) lo = m + 1; else hi = m;
            }
            place += lo - p0;
        }
        idx_out[W0 + place] = e;
    }
}

// ---------------------------------------------------------------- gather
// dst[q] = src[perm[q]] for every field.  Rows of cells <= SORT_W are final
// in idx_b; longer cells went through npass merge passes b->a->b...
__global__ __launch_bounds__(256) void k_gather(SortFields S, BhParticles D, int64_t N,
                                                const int32_t* __restrict__ idx_a,
                                                const int32_t* __restrict__ idx_b,
                                                const int32_t* __restrict__ key_sorted,
                                                const int32_t* __restrict__ offsets,
                                                const int32_t* __restrict__ stats,
                                                int32_t* __restrict__ perm_out)
{
    int mc = stats[ST_MAXCOUNT];
    int npass = 0;
    for (int64_t R = SORT_W; R < mc; R *= SORT_WAYS) ++npass;
    const int32_t* big = (npass & 1) ? idx_a : idx_b;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < N; q += stride) {
        int k = key_sorted[q];
        int e = (offsets[k + 1] - offsets[k] <= SORT_W) ? idx_b[q] : big[q];
        if ((uint32_t)e >= (uint32_t)N) e = 0;   // never taken: the ranks form a permutation
        D.px[q] = S.px[e];
        D.py[q] = S.py[e];
        D.m[q] = S.m[e];
        D.vx[q] = S.vx[e];
        D.vy[q] = S.vy[e];
        D.ax[q] = S.ax[e];
        D.ay[q] = S.ay[e];
        D.pid[q] = S.pid[e];
        if (perm_out) perm_out[q] = e;
    }
}
