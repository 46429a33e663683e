// Force evaluation: work items + persistent force kernels (FP64 and FP32).
//
// Replaces g_evaluate_boxes (python-bh/barneshut/kernels/grid_decomposition/
// gpu/grid.py:116-156, with d_is_neighbor :187-192 and the d_*_grav device
// functions :211-268).  For a particle i in cell (cx, cy):
//   near: every particle j != i of the 3x3 cell block around (cx, cy),
//   far:  the COM of every NON-EMPTY cell outside that block (the empty-cell
//         skip of seq/evaluation.py:86-95),
//   a_i += Gc * sum m_j (x_j - x_i) w(r2),  w(s) = 1/(s + eps2)  [LAW 0]
//                                           w(s) = s > r2cut ? 1/(s + eps2) : 0  [LAW 1]
// and the result is added to the existing acceleration, as the reference
// accumulates in place (gpu/grid.py:227-230).
//
// Work decomposition: a work item is a run of <= 64*P consecutive sorted
// particles of one column cx spanning rows [y0, y1] (y1 - y0 < yspan).  One wave (a 64-thread
// workgroup) takes items from a queue (atomic cursor; optional order array),
// stages the item's neighbour particles and then the system's compact COM
// list through LDS in 64-entry tiles, and every lane evaluates its P
// particles against each staged entry (LDS broadcast reads).  The COM
// entries that fall in some lane's 3x3 block lie in three compact ranges
// (columns cx-1..cx+1, rows y0-1..y1+1); only tiles meeting those ranges
// take the per-lane masked path.
#include "bh_common.h"
#include "bh_items.h"
#include "bh_kernels.h"

// ---------------------------------------------------------------- items
// One wave per grid column (all systems).  The column's sorted particles
// are cut, in order, into runs of pitem particles (a run may start or end
// inside a cell); a run is closed early when its next particle lies yspan or
// more rows below its first one, and at the end of the column.  Pass 1
// (WRITE = false) counts items per column; pass 2 writes them at the scanned
// column offsets.
//
// Where no run of pitem particles reaches the row span, those are the column's
// items, found a lane each.  Else the wave goes from item to item, the row of a
// particle found by 64 lanes at a time.  The two passes, and with a walk of the
// column's rows: 700k particles on 601^2 cells 13 us, 95; 4.2M in clusters on
// 1024^2 39 us, 181; 512 systems 36 us, 220.

// The row of a column that particle p lies in: the last with o[y] <= p, o[0 .. G].
__device__ __forceinline__ int row_of(const int32_t* __restrict__ o, int G, int p)
{
    const int lane = threadIdx.x & 63;
    int lo = 0, n = G;   // the row is in [lo, lo + n)
    while (n > 1) {
        const int step = (n + 63) >> 6;
        const bool in = lane * step < n;
        const unsigned long long b = __ballot(in && o[lo + (in ? lane * step : 0)] <= p);
        const int k = __popcll(b) - 1;
        n = min(step, n - k * step);
        lo += k * step;
    }
    return lo;
}

template <bool WRITE>
__device__ __forceinline__ int column_items(const SysDev* __restrict__ sys, int S, int64_t col,
                                            const int32_t* __restrict__ offsets, int pitem,
                                            int yspan, int64_t out, Item* __restrict__ items,
                                            int64_t max_items, int32_t* stats)
{
    const int lane = threadIdx.x & 63;
    const int s = sys_of_col(sys, S, col);
    const SysDev& d = sys[s];
    const int G = d.G;
    const int x = (int)(col - d.col_off);
    const int32_t* o = offsets + d.c_off + (int64_t)x * G;
    const int pb = uniform_int(o[G]);
    int p = uniform_int(o[0]);
    const int runs = (pb - p + pitem - 1) / pitem;
    bool wide = false;
    for (int i = lane; i < runs && G > yspan; i += BH_WAVE) {
        const Item it = run_item(o, G, s, x, i, pitem);
        wide = wide || it.y1 - it.y0 >= yspan;
    }
    if (!__any(wide)) {
        for (int i = lane; WRITE && i < runs; i += BH_WAVE) {
            if (out + i < max_items) items[out + i] = run_item(o, G, s, x, i, pitem);
            else atomicOr(&stats[ST_ERR], BH_ERR_ITEMS);
        }
        return runs;
    }
    int n_out = 0;
    while (p < pb) {   // the same on every lane; lane 0 writes
        Item it;
        it.p0 = p;
        it.y0 = row_of(o, G, p);
        const int end = it.y0 + yspan < G ? uniform_int(o[it.y0 + yspan]) : pb;
        p = min(p + pitem, end);
        if (WRITE) {
            it.np = p - it.p0;
            it.y1 = row_of(o, G, p - 1);
            it.sys = s;
            it.cx = x;
            it.pad0 = 0;
            it.pad1 = 0;
            if (lane == 0) {
                if (out + n_out < max_items) items[out + n_out] = it;
                else atomicOr(&stats[ST_ERR], BH_ERR_ITEMS);
            }
        }
        ++n_out;
    }
    return n_out;
}

template <bool WRITE>
__global__ __launch_bounds__(64) void k_items(const SysDev* __restrict__ sys, int S, int64_t ncols,
                                              const int32_t* __restrict__ offsets, int pitem,
                                              int yspan, int32_t* __restrict__ col_items,
                                              Item* __restrict__ items, int64_t max_items,
                                              int32_t* stats)
{
    const int64_t col = blockIdx.x;
    if (col >= ncols) return;
    const int n = column_items<WRITE>(sys, S, col, offsets, pitem, yspan,
                                      WRITE ? col_items[col] : 0, items, max_items, stats);
    if (!WRITE && threadIdx.x == 0) col_items[col] = n;
}

template __global__ void k_items<false>(const SysDev*, int, int64_t, const int32_t*, int, int,
                                        int32_t*, Item*, int64_t, int32_t*);
template __global__ void k_items<true>(const SysDev*, int, int64_t, const int32_t*, int, int,
                                       int32_t*, Item*, int64_t, int32_t*);

// items_runs as a launch of its own: the count, scan, clamp and write of a
// 16,384-particle step were six launches and 24 us.
__global__ __launch_bounds__(1024) void k_items_runs(const SysDev* __restrict__ sys, int S,
                                                     int ncols, const int32_t* __restrict__ offsets,
                                                     int pitem, int32_t* col_off,
                                                     Item* __restrict__ items, int64_t max_items,
                                                     int32_t* stats, int write)
{
    __shared__ int32_t at[SCAN_ONE];
    __shared__ int wsum[16];
    items_runs<1024, SCAN_ONE>(sys, S, ncols, offsets, pitem, col_off, items, max_items, stats,
                               write, at, wsum);
}

__global__ __launch_bounds__(256) void k_items_fill(const SysDev* __restrict__ sys, int S,
                                                    int ncols, const int32_t* __restrict__ offsets,
                                                    int pitem, const int32_t* __restrict__ col_off,
                                                    Item* __restrict__ items,
                                                    const int32_t* __restrict__ stats)
{
    const int n = stats[ST_NITEMS];
    for (int t = blockIdx.x * 256 + threadIdx.x; t < n; t += gridDim.x * 256) {
        const int col = col_of_item(col_off, ncols, t);
        write_run(sys, S, col, t, col_off[col], offsets, pitem, items);
    }
}

// Keeps the item count within the allocated capacity (flags the overflow).
__global__ void k_clamp_items(int32_t* stats, int64_t max_items)
{
    if (threadIdx.x == 0 && blockIdx.x == 0 && stats[ST_NITEMS] > max_items) {
        stats[ST_NITEMS] = (int32_t)max_items;
        stats[ST_ERR] |= BH_ERR_ITEMS;
    }
}

// ---------------------------------------------------------------- common pieces
struct NearE {
    double x, y, m;
    int32_t row, idx;
};

__device__ __forceinline__ void kahan_add(float& s, float& c, float v)
{
    float y = v - c;
    float t = s + y;
    c = (t - s) - y;
    s = t;
}

__device__ __forceinline__ int next_item(int32_t* stats, int lane)
{
    int q = 0;
    if (lane == 0) q = atomicAdd(&stats[ST_QUEUE], 1);
    q = __shfl(q, 0, BH_WAVE);
    return uniform_int(q);
}

// Queue positions [begin, end) of launch `part` of `nparts`: contiguous
// ranges of the `total` positions (the launches of one pass run one after
// the other on one stream; each particle's sums do not depend on the split).
__device__ __forceinline__ void part_range(int total, int part, int nparts, int& begin, int& end)
{
    begin = (int)(((int64_t)total * part) / nparts);
    end = (int)(((int64_t)total * (part + 1)) / nparts);
}

__device__ __forceinline__ bool meets(int b0, int b1, int lo, int hi)
{
    return lo < hi && b0 < hi && b1 > lo;
}

// M w(s2) of a far entry from its reciprocal mass rM = 1 / M (+inf for the
// padding and zero-mass cells, whose terms are then exactly 0).
template <int LAW>
__device__ __forceinline__ float far_t32(float wx, float wy, float rM, float eps2c, float r2c)
{
    if (LAW == 0) return __builtin_amdgcn_rcpf(fmaf(wx, wx, fmaf(wy, wy, eps2c)) * rM);
    const float s2 = fmaf(wx, wx, wy * wy);
    return (s2 > r2c) ? __builtin_amdgcn_rcpf((s2 + eps2c) * rM) : 0.0f;
}

// ---------------------------------------------------------------- FP64
// Far-field weights M0 / q0 and M1 / q1 of two COM entries for one particle
// from one reciprocal: Q = q0 q1, R = 1/Q from v_rcp_f64 refined as in
// wdiv64, then M0 / q0 = (M0 R) q1 and M1 / q1 = (M1 R) q0.  That is the VALU
// count of two separate refined weights with half the reciprocals (v_rcp_f64
// takes four issue cycles of its own), at four roundings per weight instead
// of two.  Needs every kept q >= 1, which the FP64 kernel's far entries have in
// units of 1 / sig (their cell is at least one cell away); an entry the
// particle does not keep (k0 / k1 false: inside its 3x3 block) enters the pair
// as q = 1 and gets weight 0, so the other weight is the same as in any pair
// with it.
template <int LAW>
__device__ __forceinline__ void pair_w64(double wx0, double wy0, double M0, bool k0, double wx1,
                                         double wy1, double M1, bool k1, double eps2,
                                         double r2cut, double& w0, double& w1)
{
    const double s0 = fma(wx0, wx0, wy0 * wy0), s1 = fma(wx1, wx1, wy1 * wy1);
    double q0 = (LAW == 0) ? fma(wx0, wx0, fma(wy0, wy0, eps2)) : s0 + eps2;
    double q1 = (LAW == 0) ? fma(wx1, wx1, fma(wy1, wy1, eps2)) : s1 + eps2;
    q0 = k0 ? q0 : 1.0;
    q1 = k1 ? q1 : 1.0;
    const double Q = q0 * q1;
    const double R0 = __builtin_amdgcn_rcp(Q);
    const double e = fma(-Q, R0, 1.0);
    const double R = fma(R0, fma(e, e, e), R0);
    w0 = (M0 * R) * q1;
    w1 = (M1 * R) * q0;
    if (LAW == 1) {
        w0 = s0 > r2cut ? w0 : 0.0;
        w1 = s1 > r2cut ? w1 : 0.0;
    }
    w0 = k0 ? w0 : 0.0;
    w1 = k1 ? w1 : 0.0;
}

// FAST 1: far-field weights in pairs (pair_w64), near-field weights by
// wdiv64, positions in units of a power of two near the cell size; FAST 0:
// IEEE division per weight, physical units (fp64_ieee).
template <int P, int LAW, int FAST>
__global__ __launch_bounds__(64) void k_force64(ForceArgs A)
{
    __shared__ Com64 ftile[BH_WAVE];
    __shared__ NearE ntile[BH_WAVE];
    const int lane = threadIdx.x;
    const int nitems = A.stats[ST_NITEMS];
    int qb, qe;
    part_range(nitems, A.qpart, A.nqparts, qb, qe);
    for (;;) {
        const int q = qb + next_item(A.stats, lane);
        if (q >= qe) break;
        const long long t0 = A.cost_log ? (long long)wall_clock64() : 0;
        const int itx = A.order ? uniform_int(A.order[q]) : q;
        if ((unsigned)itx >= (unsigned)nitems) continue;   // malformed order entry
        const Item it = A.items[itx];
        const SysDev& d = A.sys[it.sys];
        const int G = d.G;
        const int64_t coff = d.c_off;
        const int cx = it.cx;
        const int ylo = max(it.y0 - 1, 0), yhi = min(it.y1 + 1, G - 1);
        // FAST: positions in units of 1 / sig, sig a power of two with
        // step * sig in [1, 2).  The scaling is exact, so every difference and
        // product rounds as in physical units, and a far-field q is >= 1.
        double sig = 1.0;
        if (FAST && d.step > 0.0 && d.step < __builtin_huge_val()) {
            int e2;
            (void)frexp(d.step, &e2);
            sig = ldexp(1.0, 1 - e2);
        }
        const double eps2 = A.eps2 * sig * sig, r2cut = A.r2cut * sig * sig;
        // past the list: zero mass far away (the term is exactly 0).  In units of
        // 1 / sig a padding q is ~2e120, so a pair of two padding entries keeps
        // Q ~ 4e240 finite (an infinite Q would give R = NaN through
        // fma(-inf, 0, 1)), and particles up to 1e59 cells from the origin stay
        // far from it
        const double pad = FAST ? 1e60 : 1e150;

        double xi[P], yi[P], sx[P], sy[P];
        int cy[P], gi[P];
        bool act[P];
#pragma unroll
        for (int k = 0; k < P; ++k) {
            int slot = lane + BH_WAVE * k;
            act[k] = slot < it.np;
            gi[k] = it.p0 + slot;
            xi[k] = 0.0;
            yi[k] = 0.0;
            cy[k] = -100000;
            sx[k] = 0.0;
            sy[k] = 0.0;
            if (act[k]) {
                xi[k] = A.x[gi[k]] * sig;
                yi[k] = A.y[gi[k]] * sig;
                cy[k] = (int)(A.key_sorted[gi[k]] - coff) - cx * G;
            }
        }

        // near field: particles of columns cx-1..cx+1, rows ylo..yhi
        for (int dx = -1; dx <= 1; ++dx) {
            const int xc = cx + dx;
            if (xc < 0 || xc >= G) continue;
            const int64_t cl = coff + (int64_t)xc * G;
            const int pa = A.offsets[cl + ylo], pb = A.offsets[cl + yhi + 1];
            for (int base = pa; base < pb; base += BH_WAVE) {
                const int j = base + lane;
                NearE e;
                if (j < pb) {
                    e.x = A.x[j] * sig;
                    e.y = A.y[j] * sig;
                    e.m = A.m[j];
                    e.row = (int)(A.key_sorted[j] - cl);
                    e.idx = j;
                } else {
                    e.x = 0.0;
                    e.y = 0.0;
                    e.m = 0.0;
                    e.row = -100000;
                    e.idx = -1;
                }
                ntile[lane] = e;
                __syncthreads();
                const int cnt = min(BH_WAVE, pb - base);
                for (int jj = 0; jj < cnt; ++jj) {
                    const NearE f = ntile[jj];
#pragma unroll
                    for (int k = 0; k < P; ++k) {
                        const bool keep = (f.idx != gi[k]) && (abs(f.row - cy[k]) <= 1);
                        const double wx = f.x - xi[k], wy = f.y - yi[k];
                        double w = near_w64<LAW, FAST>(wx, wy, f.m, eps2, r2cut);
                        w = keep ? w : 0.0;
                        sx[k] = fma(wx, w, sx[k]);
                        sy[k] = fma(wy, w, sy[k]);
                    }
                }
                __syncthreads();
            }
        }

        // far field: compact COM list of the system, minus the 3x3 blocks
        const int ne0 = A.neprefix[coff], ne1 = A.neprefix[coff + (int64_t)G * G];
        int mlo[3], mhi[3];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const int xc = cx + t - 1;
            if (xc >= 0 && xc < G) {
                const int64_t cl = coff + (int64_t)xc * G;
                mlo[t] = A.neprefix[cl + ylo];
                mhi[t] = A.neprefix[cl + yhi + 1];
            } else {
                mlo[t] = 0;
                mhi[t] = 0;
            }
        }
        auto stage = [&](int e) {
            Com64 c;
            if (e < ne1) {
                c = A.l64[e];
                c.X *= sig;
                c.Y *= sig;
            } else {
                c.X = pad; c.Y = pad; c.M = 0.0; c.kx = -100000; c.ky = -100000;
            }
            return c;
        };
        Com64 nxt = stage(ne0 + lane);
        for (int base = ne0; base < ne1; base += BH_WAVE) {
            ftile[lane] = nxt;
            __syncthreads();
            nxt = stage(base + BH_WAVE + lane);
            const int b1 = base + BH_WAVE;
            const bool masked = meets(base, b1, mlo[0], mhi[0]) || meets(base, b1, mlo[1], mhi[1]) ||
                                meets(base, b1, mlo[2], mhi[2]);
            if (FAST) {
                // entries in pairs (fixed by their index, so every particle
                // gets the same pairs under any launch shape) sharing one
                // reciprocal; masked tiles give an entry a particle does not
                // keep q = 1 inside the pair, so the kept one rounds exactly
                // as in an unmasked tile
                if (!masked) {
#pragma unroll 2
                    for (int j = 0; j < BH_WAVE; j += 2) {
                        const Com64 f0 = ftile[j], f1 = ftile[j + 1];
#pragma unroll
                        for (int k = 0; k < P; ++k) {
                            const double wx0 = f0.X - xi[k], wy0 = f0.Y - yi[k];
                            const double wx1 = f1.X - xi[k], wy1 = f1.Y - yi[k];
                            double w0, w1;
                            pair_w64<LAW>(wx0, wy0, f0.M, true, wx1, wy1, f1.M, true, eps2, r2cut,
                                          w0, w1);
                            sx[k] = fma(wx0, w0, sx[k]);
                            sy[k] = fma(wy0, w0, sy[k]);
                            sx[k] = fma(wx1, w1, sx[k]);
                            sy[k] = fma(wy1, w1, sy[k]);
                        }
                    }
                } else {
                    for (int j = 0; j < BH_WAVE; j += 2) {
                        const Com64 f0 = ftile[j], f1 = ftile[j + 1];
                        const bool cn0 = abs(f0.kx - cx) <= 1, cn1 = abs(f1.kx - cx) <= 1;
#pragma unroll
                        for (int k = 0; k < P; ++k) {
                            const bool k0 = !(cn0 && abs(f0.ky - cy[k]) <= 1);
                            const bool k1 = !(cn1 && abs(f1.ky - cy[k]) <= 1);
                            const double wx0 = f0.X - xi[k], wy0 = f0.Y - yi[k];
                            const double wx1 = f1.X - xi[k], wy1 = f1.Y - yi[k];
                            double w0, w1;
                            pair_w64<LAW>(wx0, wy0, f0.M, k0, wx1, wy1, f1.M, k1, eps2, r2cut, w0,
                                          w1);
                            sx[k] = fma(wx0, w0, sx[k]);
                            sy[k] = fma(wy0, w0, sy[k]);
                            sx[k] = fma(wx1, w1, sx[k]);
                            sy[k] = fma(wy1, w1, sy[k]);
                        }
                    }
                }
            } else if (!masked) {
#pragma unroll 4
                for (int j = 0; j < BH_WAVE; ++j) {
                    const Com64 f = ftile[j];
#pragma unroll
                    for (int k = 0; k < P; ++k) {
                        const double wx = f.X - xi[k], wy = f.Y - yi[k];
                        const double w = far_w64<LAW, 0>(wx, wy, f.M, eps2, r2cut);
                        sx[k] = fma(wx, w, sx[k]);
                        sy[k] = fma(wy, w, sy[k]);
                    }
                }
            } else {
                for (int j = 0; j < BH_WAVE; ++j) {
                    const Com64 f = ftile[j];
                    const bool colnear = abs(f.kx - cx) <= 1;
#pragma unroll
                    for (int k = 0; k < P; ++k) {
                        const bool keep = !(colnear && abs(f.ky - cy[k]) <= 1);
                        const double wx = f.X - xi[k], wy = f.Y - yi[k];
                        double w = far_w64<LAW, 0>(wx, wy, f.M, eps2, r2cut);
                        w = keep ? w : 0.0;
                        sx[k] = fma(wx, w, sx[k]);
                        sy[k] = fma(wy, w, sy[k]);
                    }
                }
            }
            __syncthreads();
        }

#pragma unroll
        for (int k = 0; k < P; ++k) {
            if (act[k]) {
                A.ax[gi[k]] += A.Gc * (sx[k] * sig);
                A.ay[gi[k]] += A.Gc * (sy[k] * sig);
            }
        }
        if (A.cost_log && lane == 0) A.cost_log[itx] = (long long)wall_clock64() - t0;
    }
}

// ---------------------------------------------------------------- FP64, shared chunks
// The terms of k_force64<.., FAST 1>, with the work of 64 particles shared by
// the W waves of a block: each wave takes every W-th group of near candidates
// and the w-th slice of the COM list, and the waves' sums are added in wave
// order.  A pass has N / 64 W waves instead of N / 128 and each a W-th of the
// chain, so small passes fill the chip; the terms come by scalar loads, so
// they cost neither LDS reads nor a staging round per tile.  A chunk is 64
// consecutive sorted particles of one system: in passes of this form a particle's
// terms and their order depend on its system alone.
//
// Near candidates: if the chunk lies in one column and spans two rows at most
// (dense cells), its waves walk the union of the lanes' cells, four candidates
// at a time; else each lane walks its own three ranges with vector loads.
//
// Force pass against the one-wave kernel (uniform particles): 2,000 on 11^2
// cells 90 -> 16 us, 16,384 on 32^2 152 -> 21 us, 262,144 on 256^2 10.4 -> 6.0 ms
// (2.9e12 terms/s, with terms in pairs; quads save 2 to 4 % more), 1M on 32^2 (8.8e9 near pairs) 7.3 -> 4.3 ms; no size was
// slower, so only the cost log, which times work items, still takes k_force64.
// Loading each quad one ahead of its use is worth 15 % and, where the
// candidates of a cell exceed an XCD's L2, a third.  W = 4 and 16 are within
// 10 % of W = 8 from 65k particles on and slower below (W = 4: 29 against 24 us
// at 16,384) or above (W = 16).
// At most 80 registers, so that three blocks share a CU: with 81 under a cutoff,
// 184,442 particles on 46^2 cells took 438 instead of 393 us.
typedef double fd4a __attribute__((ext_vector_type(4), aligned(8)));

struct Four {   // four candidates in scalar registers
    double X[4], Y[4], M[4];
};

// Candidates j .. j + 3 of [j, b); those past b are copies of j without mass.
__device__ __forceinline__ Four load_four(const double* x, const double* y, const double* m, int j,
                                          int b, int N)
{
    Four f;
    if (j + 4 <= N) {
        const fd4a X = *(cptr<fd4a>)as_const(x + j), Y = *(cptr<fd4a>)as_const(y + j);
        const fd4a M = *(cptr<fd4a>)as_const(m + j);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            f.X[u] = X[u];
            f.Y[u] = Y[u];
            f.M[u] = M[u];
        }
    } else {   // the last rows of the arrays
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int k = min(j + u, N - 1);
            f.X[u] = as_const(x)[k];
            f.Y[u] = as_const(y)[k];
            f.M[u] = as_const(m)[k];
        }
    }
#pragma unroll
    for (int u = 1; u < 4; ++u)
        if (j + u >= b) {
            f.X[u] = f.X[0];
            f.Y[u] = f.Y[0];
            f.M[u] = 0.0;
        }
    return f;
}

template <int LAW, bool OWN>
__device__ __forceinline__ void near_four(const Four& f, int j, int b, int gi, double x, double y,
                                          double sig, double eps2, double r2cut, double& sx,
                                          double& sy)
{
    double wx[4], wy[4];
    bool keep[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        wx[u] = fma(f.X[u], sig, -x);
        wy[u] = fma(f.Y[u], sig, -y);
        keep[u] = (j + u < b ? j + u : j) != gi;
    }
    quad_terms<LAW, OWN>(wx, wy, f.M, keep, eps2, r2cut, sx, sy);
}

// Every (4 W)-th group of four of [j, b), the next one loaded ahead.
template <int W, int LAW, bool OWN>
__device__ __forceinline__ void near_cell(const ForceArgs& A, int j, int b, int N, int gi, double x,
                                          double y, double sig, double eps2, double r2cut,
                                          double& sx, double& sy)
{
    if (j >= b) return;
    Four f = load_four(A.x, A.y, A.m, j, b, N);
    for (;;) {
        const int jn = j + 4 * W;
        Four n = f;
        if (jn < b) n = load_four(A.x, A.y, A.m, jn, b, N);
        near_four<LAW, OWN>(f, j, b, gi, x, y, sig, eps2, r2cut, sx, sy);
        if (jn >= b) break;
        f = n;
        j = jn;
    }
}

template <int W, int LAW>
__global__ __launch_bounds__(64 * W, 6) void k_force64s(ForceArgs A, int S)
{
    __shared__ double part[2][W][BH_WAVE];
    __shared__ int bad[W];
    const int lane = threadIdx.x & 63, w = uniform_int(threadIdx.x >> 6);
    const int64_t ci = A.chunk0 + blockIdx.x;
    int s = 0;
    if (S > 1) {   // the system of the chunk
        int hi = S - 1;
        while (s < hi) {
            const int mid = (s + hi + 1) >> 1;
            if (A.sys[mid].k_off <= ci) s = mid; else hi = mid - 1;
        }
        s = uniform_int(s);
    }
    if (blockIdx.x == 0 && threadIdx.x < 4) A.stats[ST_NRECOMP + threadIdx.x] = 0;
    const SysDev& d = A.sys[s];
    const int G = d.G;
    const int64_t coff = d.c_off;
    const int rank = (int)(ci - d.k_off) * 64 + lane;
    const bool act = rank < d.n;
    const int gi = act ? (int)d.p_off + rank : -1;
    const double sig = step_scale(d.step);
    const double eps2 = A.eps2 * sig * sig, r2cut = A.r2cut * sig * sig;
    double x = 0.0, y = 0.0, sx = 0.0, sy = 0.0;
    int cx = -100000, cy = -100000;
    if (act) {
        x = A.x[gi];
        y = A.y[gi];
        const int key = A.key_sorted[gi] - (int)coff;
        cx = key / G;
        cy = key - cx * G;
    }
    const bool plain = placed_apart<LAW>(d, r2cut, act, (x - d.min_x) / d.step - cx,
                                         (y - d.min_y) / d.step - cy);
    x *= sig;
    y *= sig;
    const int cxl = uniform_int(wave_min(act ? cx : 0x7fffffff));
    const int cxh = uniform_int(wave_max(act ? cx : -1));
    const int cyl = uniform_int(wave_min(act ? cy : 0x7fffffff));
    const int cyh = uniform_int(wave_max(act ? cy : -1));

    // near candidates
    if (cxl == cxh && cyh - cyl < 2) {
        int turn = 0;   // groups of four so far, dealt to the waves in turn
        for (int dx = -1; dx <= 1; ++dx) {
            const int xc = cxl + dx;
            if (xc < 0 || xc >= G) continue;
            const int64_t cl = coff + (int64_t)xc * G;
            for (int row = max(cyl - 1, 0); row <= min(cyh + 1, G - 1); ++row) {
                const int a = uniform_int(A.offsets[cl + row]);
                const int b = uniform_int(A.offsets[cl + row + 1]);
                const int first = (w - turn) & (W - 1);
                turn += (b - a + 3) >> 2;
                if (!(act && abs(row - cy) <= 1)) continue;
                if (dx == 0 && row >= cyl && row <= cyh)   // some lanes' own cell
                    near_cell<W, LAW, true>(A, a + 4 * first, b, (int)A.part_n, gi, x, y, sig, eps2,
                                            r2cut, sx, sy);
                else
                    near_cell<W, LAW, false>(A, a + 4 * first, b, (int)A.part_n, gi, x, y, sig, eps2,
                                             r2cut, sx, sy);
            }
        }
    } else if (act) {
        int n0 = 0, n1 = 0, n2 = 0, o0 = 0, o1 = 0, o2 = 0;   // the three ranges as one list
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const int xc = cx + t - 1;
            int a = 0, b = 0;
            if (xc >= 0 && xc < G) {
                const int64_t cl = coff + (int64_t)xc * G;
                a = A.offsets[cl + max(cy - 1, 0)];
                b = A.offsets[cl + min(cy + 1, G - 1) + 1];
            }
            if (t == 0) { o0 = a; n0 = b - a; }
            if (t == 1) { o1 = a - n0; n1 = n0 + b - a; }
            if (t == 2) { o2 = a - n1; n2 = n1 + b - a; }
        }
        for (int k = 2 * w; k < n2; k += 2 * W) {
            const int k1 = min(k + 1, n2 - 1);
            const int j0 = k + (k < n0 ? o0 : (k < n1 ? o1 : o2));
            const int j1 = k1 + (k1 < n0 ? o0 : (k1 < n1 ? o1 : o2));
            pair_terms<LAW, true>(fma(A.x[j0], sig, -x), fma(A.y[j0], sig, -y), A.m[j0],
                                  fma(A.x[j1], sig, -x), fma(A.y[j1], sig, -y),
                                  k + 1 < n2 ? A.m[j1] : 0.0, j0 != gi, j1 != gi, eps2, r2cut, sx,
                                  sy);
        }
    }

    // COM list: this wave's slice, a whole number of quads
    const int ne0 = uniform_int(A.neprefix[coff]);
    const int ne1 = uniform_int(A.neprefix[coff + (int64_t)G * G]);
    const int mlo = uniform_int(A.neprefix[coff + (int64_t)max(cxl - 1, 0) * G]);
    const int mhi = uniform_int(A.neprefix[coff + (int64_t)min(cxh + 2, G) * G]);
    const int per = (((ne1 - ne0 + W - 1) / W) + 3) & ~3;
    const int f0 = min(ne1, ne0 + w * per), f1 = min(ne1, f0 + per);
    if (f0 < f1) {
        // the list is padded by a quad, so whole quads are in bounds
        fd8 p = *(cptr<fd8>)(as_const(A.l64) + f0), q = *(cptr<fd8>)(as_const(A.l64) + f0 + 2);
        for (int e = f0; e < f1; e += 4) {
            const int en = e + 4 < f1 ? e + 4 : e;
            const fd8 pn = *(cptr<fd8>)(as_const(A.l64) + en);
            const fd8 qn = *(cptr<fd8>)(as_const(A.l64) + en + 2);
            if (e + 4 > f1) {   // past the slice: its first entry again, without mass
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if (u != 2 && e + 1 >= f1) p[4 + u] = p[u];
                    if (u != 2 && e + 2 >= f1) q[u] = p[u];
                    if (u != 2 && e + 3 >= f1) q[4 + u] = p[u];
                }
                if (e + 1 >= f1) p[6] = 0.0;
                if (e + 2 >= f1) q[2] = 0.0;
                q[6] = 0.0;
            }
            const double wx[4] = {fma(p[0], sig, -x), fma(p[4], sig, -x), fma(q[0], sig, -x),
                                  fma(q[4], sig, -x)};
            const double wy[4] = {fma(p[1], sig, -y), fma(p[5], sig, -y), fma(q[1], sig, -y),
                                  fma(q[5], sig, -y)};
            const double m[4] = {p[2], p[6], q[2], q[6]};
            if (plain && (e + 4 <= mlo || e >= mhi)) {
                quad_terms<0, false>(wx, wy, m, {true, true, true, true}, eps2, r2cut, sx, sy);
            } else {
                auto far = [&](double kxy) {
                    const long long c = __double_as_longlong(kxy);
                    return (unsigned)((int)c - cx + 1) > 2u ||
                           (unsigned)((int)(c >> 32) - cy + 1) > 2u;
                };
                quad_terms<LAW, true>(wx, wy, m, {far(p[3]), far(p[7]), far(q[3]), far(q[7])},
                                      eps2, r2cut, sx, sy);
            }
            p = pn;
            q = qn;
        }
    }
    part[0][w][lane] = sx;
    part[1][w][lane] = sy;
    if (lane == 0) bad[w] = 0;
    if (!is_finite(sx, sy)) bad[w] = 1;
    __syncthreads();
    // one by one, by all waves of the block (see one_term); told by a word a wave
    // beside the sums, since a barrier of its own costs 1 % of a short block
    if (__any(bad[lane & (W - 1)])) {
        sx = sy = 0.0;
        for (int xc = max(cx - 1, 0); act && xc <= min(cx + 1, G - 1); ++xc) {
            const int64_t cl = coff + (int64_t)xc * G;
            const int b = A.offsets[cl + min(cy + 1, G - 1) + 1];
#pragma unroll 1
            for (int j = A.offsets[cl + max(cy - 1, 0)] + w; j < b; j += W)
                one_term<LAW>(fma(A.x[j], sig, -x), fma(A.y[j], sig, -y), A.m[j], j != gi, eps2,
                              r2cut, sx, sy);
        }
#pragma unroll 1
        for (int e = f0; e < f1; ++e) {
            const Com64 f = A.l64[e];
            one_term<LAW>(fma(f.X, sig, -x), fma(f.Y, sig, -y), f.M,
                          abs(f.kx - cx) > 1 || abs(f.ky - cy) > 1, eps2, r2cut, sx, sy);
        }
        part[0][w][lane] = sx;
        part[1][w][lane] = sy;
        __syncthreads();
    }
    if (w < 2 && act) {   // wave 0 adds x, wave 1 adds y
        double t = 0.0;
#pragma unroll
        for (int v = 0; v < W; ++v) t += part[w][v][lane];
        double* a = w ? A.ay : A.ax;
        a[gi] += A.Gc * (t * sig);
    }
}

// ---------------------------------------------------------------- FP32
// Positions in cell units relative to the item origin (cx, oy), oy = the
// item's middle row: the integer cell offsets are exact in FP32, so a far
// term's separation carries a relative error of a few ulp.  Near-field
// separations are formed in FP64 and rounded once.  KAHAN: 0 plain FP32
// sums; 1 FP32 partial per 64-entry tile, tiles Kahan-summed; 2 Kahan per term.
//
// Far field without a cutoff (LAW 0) in mass-scaled form: with c = s / M per
// COM entry (s a power of two per item),
//     t = c (a - u),   M (a - u) / (|a - u|^2 + eps2) = s * t / (|t|^2 + c^2 eps2),
// so the tile holds (c a_x, c a_y, -c, c^2 eps2) and each term costs two fma
// for t, two for |t|^2, v_rcp_f32 and two fma into the sums: one VALU
// instruction fewer than forming M * w.  Scaling by the power of two s is
// exact, so s only keeps c^2 |a - u|^2 inside the FP32 range (s = 2^e with
// M <= 2^e < 2 M for the item's own cell; any power of two gives the same
// sums bit for bit); near-field terms are divided by s (exactly) to share the
// sums, and the sums are multiplied by s at the end.  c = s * rM from the
// list's reciprocal mass equals the correctly rounded s / M (a power-of-two
// scaling commutes with rounding), so staging a tile takes no division.
// Zero-mass entries and the padding past the list hold (1e30, 1e30, 0, 0):
// |t|^2 overflows to inf, v_rcp_f32 gives 0 and the term adds exactly 0.
// Minimum resident waves per SIMD the FP32 kernel is compiled for (bounds its
// VGPRs so that more waves hide the reciprocal's latency): 5 for 4 particles
// per lane, 8 for 1 or 2 (one fewer with per-term Kahan sums, which hold more
// registers).  At 2 particles per lane the 8-wave build keeps a few per-item
// values in scratch and still runs 1.4 % faster than the 7-wave one.
template <int P, int KAHAN>
struct F32Waves {
    static constexpr int value = (P >= 4 ? 5 : 8) - (KAHAN == 2 ? 1 : 0);
};

template <int P, int LAW, int KAHAN>
__global__ __launch_bounds__(64, (F32Waves<P, KAHAN>::value)) void k_force32(ForceArgs A)
{
    constexpr int FT = 2 * BH_WAVE;            // far-field tile: two entries staged per lane
    __shared__ float4 ftile[FT];
    __shared__ int32_t ktile[FT];              // kx << 16 | ky (LAW 0 masked tiles)
    __shared__ NearE ntile[BH_WAVE];
    const int lane = threadIdx.x;
    const int nitems = A.stats[ST_NITEMS];
    const int S = A.split > 1 ? A.split : 1;
    const int nt = S > 1 ? min(A.n_tail, nitems) : 0;
    const int nu = nitems - nt;
    const int total = nu + nt * S;
    int qb, qe;
    part_range(total, A.qpart, A.nqparts, qb, qe);
    for (;;) {
        const int q = qb + next_item(A.stats, lane);
        if (q >= qe) break;
        int pos = q, part = -1;
        if (q >= nu) {   // slice-major: every tail item's slice 0, then slice 1, ...
            const int r = q - nu;
            part = r / nt;
            pos = nu + (r - part * nt);
        }
        const long long t0 = A.cost_log ? (long long)wall_clock64() : 0;
        const int itx = A.order ? uniform_int(A.order[pos]) : pos;
        if ((unsigned)itx >= (unsigned)nitems) continue;   // malformed order entry
        const Item it = A.items[itx];
        const SysDev& d = A.sys[it.sys];
        const int G = d.G;
        const int64_t coff = d.c_off;
        const int cx = it.cx;
        const int oy = (it.y0 + it.y1) >> 1;
        const int ylo = max(it.y0 - 1, 0), yhi = min(it.y1 + 1, G - 1);
        const double step = d.step;
        const double inv_step = 1.0 / step;
        const float eps2c = (float)(A.eps2 * inv_step * inv_step);
        const float r2c = (float)(A.r2cut * inv_step * inv_step);
        // mass scale s (LAW 0): 1 / (the power of two at or below 1 / M of the
        // item's own cell), i.e. M <= s < 2 M
        float msc = 1.0f;
        if (LAW == 0) {
            const int64_t own = coff + (int64_t)cx * G + it.y0;
            const float r0 = fabsf(A.l32[A.neprefix[own]].rM);
            const float p2 = __int_as_float(__float_as_int(r0) & 0x7f800000);
            if (p2 >= 1.0e-37f && p2 <= 1.0e37f) msc = 1.0f / p2;
        }
        const float inv_msc = 1.0f / msc;

        double xi[P], yi[P];
        float ux[P], uy[P], Sx[P], Sy[P], Cx[P], Cy[P], tx[P], ty[P], s2n[P];
        int cy[P], gi[P];
        bool act[P];
#pragma unroll
        for (int k = 0; k < P; ++k) {
            int slot = lane + BH_WAVE * k;
            act[k] = slot < it.np;
            gi[k] = it.p0 + slot;
            xi[k] = 0.0;
            yi[k] = 0.0;
            ux[k] = 0.0f;
            uy[k] = 0.0f;
            cy[k] = -100000;
            if (act[k]) {
                xi[k] = A.x[gi[k]];
                yi[k] = A.y[gi[k]];
                cy[k] = (int)(A.key_sorted[gi[k]] - coff) - cx * G;
                ux[k] = (float)((xi[k] - d.min_x) / step - (double)cx);
                uy[k] = (float)((yi[k] - d.min_y) / step - (double)oy);
            }
            Sx[k] = Sy[k] = Cx[k] = Cy[k] = tx[k] = ty[k] = s2n[k] = 0.0f;
        }

        // near field (separations in FP64, rounded once to FP32); part 0 of a split item.
        // s2n sums fm * t = fm^2 / (s2 + eps2c) >= |term|^2 for the recompute's estimate.
        for (int dx = -1; dx <= (part <= 0 ? 1 : -2); ++dx) {
            const int xc = cx + dx;
            if (xc < 0 || xc >= G) continue;
            const int64_t cl = coff + (int64_t)xc * G;
            const int pa = A.offsets[cl + ylo], pb = A.offsets[cl + yhi + 1];
            for (int base = pa; base < pb; base += BH_WAVE) {
                const int j = base + lane;
                NearE e;
                if (j < pb) {
                    e.x = A.x[j];
                    e.y = A.y[j];
                    e.m = A.m[j];
                    e.row = (int)(A.key_sorted[j] - cl);
                    e.idx = j;
                } else {
                    e.x = 0.0;
                    e.y = 0.0;
                    e.m = 0.0;
                    e.row = -100000;
                    e.idx = -1;
                }
                ntile[lane] = e;
                __syncthreads();
                const int cnt = min(BH_WAVE, pb - base);
                for (int jj = 0; jj < cnt; ++jj) {
                    const NearE f = ntile[jj];
                    const float fm = (float)f.m * inv_msc;
#pragma unroll
                    for (int k = 0; k < P; ++k) {
                        const bool keep = (f.idx != gi[k]) && (abs(f.row - cy[k]) <= 1);
                        const float wx = (float)((f.x - xi[k]) * inv_step);
                        const float wy = (float)((f.y - yi[k]) * inv_step);
                        const float s2 = fmaf(wx, wx, wy * wy);
                        float t = fm * __builtin_amdgcn_rcpf(s2 + eps2c);
                        if (LAW == 1) t = (s2 > r2c) ? t : 0.0f;
                        t = keep ? t : 0.0f;
                        s2n[k] = fmaf(fm, t, s2n[k]);
                        if (KAHAN == 2) {
                            kahan_add(Sx[k], Cx[k], wx * t);
                            kahan_add(Sy[k], Cy[k], wy * t);
                        } else {
                            tx[k] = fmaf(wx, t, tx[k]);
                            ty[k] = fmaf(wy, t, ty[k]);
                        }
                    }
                }
                if (KAHAN == 1) {
#pragma unroll
                    for (int k = 0; k < P; ++k) {
                        kahan_add(Sx[k], Cx[k], tx[k]);
                        kahan_add(Sy[k], Cy[k], ty[k]);
                        tx[k] = 0.0f;
                        ty[k] = 0.0f;
                    }
                }
                __syncthreads();
            }
        }

        if (A.rc && part <= 0) {
#pragma unroll
            for (int k = 0; k < P; ++k)
                if (act[k]) A.ay[A.part_n + gi[k]] = (double)s2n[k] * ((double)msc * (double)msc);
        }

        // far field (a split item's part covers one 64-aligned slice of the list)
        int ne0 = A.neprefix[coff], ne1 = A.neprefix[coff + (int64_t)G * G];
        if (part >= 0) {
            const int chunk = (((ne1 - ne0 + S - 1) / S) + BH_WAVE - 1) & ~(BH_WAVE - 1);
            ne0 = ne0 + part * chunk;
            ne1 = min(ne1, ne0 + chunk);
        }
        int mlo[3], mhi[3];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const int xc = cx + t - 1;
            if (xc >= 0 && xc < G) {
                const int64_t cl = coff + (int64_t)xc * G;
                mlo[t] = A.neprefix[cl + ylo];
                mhi[t] = A.neprefix[cl + yhi + 1];
            } else {
                mlo[t] = 0;
                mhi[t] = 0;
            }
        }
        Com32 nxt[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int e = ne0 + lane + h * BH_WAVE;
            if (e < ne1) nxt[h] = A.l32[e];
            else { nxt[h].fx = 1e18f; nxt[h].fy = 1e18f; nxt[h].rM = __builtin_huge_valf(); nxt[h].kxy = 0x7fff7fff; }
        }
        for (int base = ne0; base < ne1; base += FT) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const Com32 en = nxt[h];
                const int kx = en.kxy >> 16, ky = en.kxy & 0xffff;
                const float ex = (float)(kx - cx) + en.fx;
                const float ey = (float)(ky - oy) + en.fy;
                float4 v;
                if (LAW == 0) {
                    if (fabsf(en.rM) != __builtin_huge_valf()) {   // M != 0 (NaN passes)
                        const float c = msc * en.rM;
                        v.x = ex * c;
                        v.y = ey * c;
                        v.z = -c;
                        v.w = (c * c) * eps2c;
                    } else {
                        v.x = 1e30f;
                        v.y = 1e30f;
                        v.z = 0.0f;
                        v.w = 0.0f;
                    }
                    ktile[lane + h * BH_WAVE] = en.kxy;
                } else {
                    v.x = ex;
                    v.y = ey;
                    v.z = en.rM;
                    v.w = __int_as_float(en.kxy);
                }
                ftile[lane + h * BH_WAVE] = v;
            }
            __syncthreads();
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int e = base + FT + lane + h * BH_WAVE;
                if (e < ne1) nxt[h] = A.l32[e];
                else { nxt[h].fx = 1e18f; nxt[h].fy = 1e18f; nxt[h].rM = __builtin_huge_valf(); nxt[h].kxy = 0x7fff7fff; }
            }
            const int b1 = base + FT;
            const bool masked = meets(base, b1, mlo[0], mhi[0]) || meets(base, b1, mlo[1], mhi[1]) ||
                                meets(base, b1, mlo[2], mhi[2]);
            if (!masked) {
#pragma unroll 8
                for (int j = 0; j < FT; ++j) {
                    const float4 f = ftile[j];
#pragma unroll
                    for (int k = 0; k < P; ++k) {
                        float wx, wy, t;
                        if (LAW == 0) {
                            wx = fmaf(ux[k], f.z, f.x);
                            wy = fmaf(uy[k], f.z, f.y);
                            t = __builtin_amdgcn_rcpf(fmaf(wx, wx, fmaf(wy, wy, f.w)));
                        } else {
                            wx = f.x - ux[k];
                            wy = f.y - uy[k];
                            t = far_t32<LAW>(wx, wy, f.z, eps2c, r2c);
                        }
                        if (KAHAN == 2) {
                            kahan_add(Sx[k], Cx[k], wx * t);
                            kahan_add(Sy[k], Cy[k], wy * t);
                        } else {
                            tx[k] = fmaf(wx, t, tx[k]);
                            ty[k] = fmaf(wy, t, ty[k]);
                        }
                    }
                }
            } else {
                for (int j = 0; j < FT; ++j) {
                    const float4 f = ftile[j];
                    const int kxy = LAW == 0 ? ktile[j] : __float_as_int(f.w);
                    const bool colnear = abs((kxy >> 16) - cx) <= 1;
                    const int ky = kxy & 0xffff;
#pragma unroll
                    for (int k = 0; k < P; ++k) {
                        const bool keep = !(colnear && abs(ky - cy[k]) <= 1);
                        float wx, wy, t;
                        if (LAW == 0) {
                            wx = fmaf(ux[k], f.z, f.x);
                            wy = fmaf(uy[k], f.z, f.y);
                            t = __builtin_amdgcn_rcpf(fmaf(wx, wx, fmaf(wy, wy, f.w)));
                        } else {
                            wx = f.x - ux[k];
                            wy = f.y - uy[k];
                            t = far_t32<LAW>(wx, wy, f.z, eps2c, r2c);
                        }
                        t = keep ? t : 0.0f;
                        if (KAHAN == 2) {
                            kahan_add(Sx[k], Cx[k], wx * t);
                            kahan_add(Sy[k], Cy[k], wy * t);
                        } else {
                            tx[k] = fmaf(wx, t, tx[k]);
                            ty[k] = fmaf(wy, t, ty[k]);
                        }
                    }
                }
            }
            if (KAHAN == 1) {
#pragma unroll
                for (int k = 0; k < P; ++k) {
                    kahan_add(Sx[k], Cx[k], tx[k]);
                    kahan_add(Sy[k], Cy[k], ty[k]);
                    tx[k] = 0.0f;
                    ty[k] = 0.0f;
                }
            }
            __syncthreads();
        }

        const double scale = A.Gc * inv_step * (double)msc;
#pragma unroll
        for (int k = 0; k < P; ++k) {
            if (act[k]) {
                double rx, ry;
                if (KAHAN == 0) {
                    rx = (double)tx[k];
                    ry = (double)ty[k];
                } else {
                    rx = (double)Sx[k] - (double)Cx[k];
                    ry = (double)Sy[k] - (double)Cy[k];
                }
                if (part < 0) {
                    A.ax[gi[k]] += scale * rx;
                    A.ay[gi[k]] += scale * ry;
                } else {
                    const int64_t o = ((int64_t)part * A.part_n + gi[k]) * 2;
                    A.part[o] = scale * rx;
                    A.part[o + 1] = scale * ry;
                }
            }
        }
        if (A.cost_log && lane == 0 && part < 0) A.cost_log[itx] = (long long)wall_clock64() - t0;
    }
}

// Adds the parts of the split tail items, in part order (deterministic).
__global__ __launch_bounds__(256) void k_force_combine(const Item* __restrict__ items,
                                                       const int32_t* __restrict__ order,
                                                       const int32_t* __restrict__ stats,
                                                       int split, int n_tail, int pslots,
                                                       const double* __restrict__ part,
                                                       int64_t part_n,
                                                       double* __restrict__ ax,
                                                       double* __restrict__ ay)
{
    const int nitems = stats[ST_NITEMS];
    const int nt = min(n_tail, nitems);
    const int nu = nitems - nt;
    const int64_t total = (int64_t)nt * pslots;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += stride) {
        const int j = (int)(g / pslots), slot = (int)(g - (int64_t)j * pslots);
        const int pos = nu + j;
        const int itx = order ? order[pos] : pos;
        if ((unsigned)itx >= (unsigned)nitems) continue;
        const Item it = items[itx];
        if (slot >= it.np) continue;
        const int64_t gi = (int64_t)it.p0 + slot;
        double sx = 0.0, sy = 0.0;
        for (int s = 0; s < split; ++s) {
            const int64_t o = ((int64_t)s * part_n + gi) * 2;
            sx += part[o];
            sy += part[o + 1];
        }
        ax[gi] += sx;
        ay[gi] += sy;
    }
}

// ---------------------------------------------------------------- FP32, shared chunks
// The terms of k_force32 (tile sums carried in FP64 instead of Kahan pairs),
// with the work of 64 particles shared by the W waves of a block, as in
// k_force64s.  Near separations are formed in FP64 in units of 1 / sig and
// rounded once; far entries are staged per wave in LDS in mass-scaled,
// cell-relative form (origin: the chunk's first cell), 64 at a time, the next
// 64 on their way.
// Force pass with the recompute against k_force32 (default launch shape):
// 2,000 particles on 11^2 cells 165 -> 70 us, 16,384 on 32^2 210 -> 72 us, in
// clusters 486 -> 143 us; 262,144 on 256^2 3.47 -> 3.31 ms, 1M on 100^2 2.74 ->
// 2.46 ms and 14.2 -> 7.6 ms in clusters.
template <int LAW, bool OWN>
__device__ __forceinline__ void near_four32(const Four& f, int j, int b, int gi, double x, double y,
                                            double sig, double inv_msc, float eps2, float r2cut,
                                            double& sx, double& sy, float& s2n)
{
    float tx = 0.0f, ty = 0.0f;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const float wx = (float)fma(f.X[u], sig, -x), wy = (float)fma(f.Y[u], sig, -y);
        const float fm = (float)(f.M[u] * inv_msc);
        float q;
        bool keep = true;
        if (LAW == 1) {
            const float s2 = fmaf(wx, wx, wy * wy);
            keep = s2 > r2cut;
            q = s2 + eps2;
        } else {
            q = fmaf(wx, wx, fmaf(wy, wy, eps2));
        }
        float t = fm * __builtin_amdgcn_rcpf(q);
        if (OWN) keep = keep && (j + u < b ? j + u : j) != gi;
        // past the end: a copy of the first without mass
        if (LAW == 1 || OWN) t = keep ? t : 0.0f;
        s2n = fmaf(fm, t, s2n);
        tx = fmaf(wx, t, tx);
        ty = fmaf(wy, t, ty);
    }
    sx += (double)tx;
    sy += (double)ty;
}

template <int W, int LAW, bool OWN>
__device__ __forceinline__ void near_cell32(const ForceArgs& A, int j, int b, int N, int gi,
                                            double x, double y, double sig, double inv_msc,
                                            float eps2, float r2cut, double& sx, double& sy,
                                            float& s2n)
{
    if (j >= b) return;
    Four f = load_four(A.x, A.y, A.m, j, b, N);
    for (;;) {
        const int jn = j + 4 * W;
        Four n = f;
        if (jn < b) n = load_four(A.x, A.y, A.m, jn, b, N);
        near_four32<LAW, OWN>(f, j, b, gi, x, y, sig, inv_msc, eps2, r2cut, sx, sy, s2n);
        if (jn >= b) break;
        f = n;
        j = jn;
    }
}

template <int W, int LAW>
__global__ __launch_bounds__(64 * W) void k_force32s(ForceArgs A, int S)
{
    __shared__ float4 ftile[W][BH_WAVE];
    __shared__ int32_t ktile[W][BH_WAVE];
    __shared__ double part[2][W][BH_WAVE];
    __shared__ float part2[W][BH_WAVE];
    const int lane = threadIdx.x & 63, w = uniform_int(threadIdx.x >> 6);
    const int64_t ci = A.chunk0 + blockIdx.x;
    int s = 0;
    if (S > 1) {   // the system of the chunk
        int hi = S - 1;
        while (s < hi) {
            const int mid = (s + hi + 1) >> 1;
            if (A.sys[mid].k_off <= ci) s = mid; else hi = mid - 1;
        }
        s = uniform_int(s);
    }
    const SysDev& d = A.sys[s];
    const int G = d.G;
    const int64_t coff = d.c_off;
    const int rank = (int)(ci - d.k_off) * 64 + lane;
    const bool act = rank < d.n;
    const int gi = act ? (int)d.p_off + rank : -1;
    const double step = d.step, inv_step = 1.0 / step, sig = step_scale(step);
    const float eps2n = (float)(A.eps2 * sig * sig), r2cn = (float)(A.r2cut * sig * sig);
    const float eps2c = (float)(A.eps2 * inv_step * inv_step);
    const float r2c = (float)(A.r2cut * inv_step * inv_step);
    double x = 0.0, y = 0.0, sx = 0.0, sy = 0.0, fx = 0.0, fy = 0.0;
    float s2n = 0.0f, ux = 0.0f, uy = 0.0f;
    int cx = -100000, cy = -100000, key = 0;
    if (act) {
        x = A.x[gi];
        y = A.y[gi];
        key = A.key_sorted[gi] - (int)coff;
        cx = key / G;
        cy = key - cx * G;
    }
    const int ox = __builtin_amdgcn_readfirstlane(cx), oy = __builtin_amdgcn_readfirstlane(cy);
    const int own = __builtin_amdgcn_readfirstlane(key);
    // mass scale, as in k_force32: the power of two at or above the own cell's mass
    float msc = 1.0f;
    {
        const float r0 = fabsf(A.l32[A.neprefix[coff + own]].rM);
        const float p2 = __int_as_float(__float_as_int(r0) & 0x7f800000);
        if (p2 >= 1.0e-37f && p2 <= 1.0e37f) msc = 1.0f / p2;
    }
    const double inv_msc = 1.0 / (double)msc;
    if (act) {
        ux = (float)((x - d.min_x) * inv_step - (double)ox);
        uy = (float)((y - d.min_y) * inv_step - (double)oy);
        x *= sig;
        y *= sig;
    }
    const int cxl = uniform_int(wave_min(act ? cx : 0x7fffffff));
    const int cxh = uniform_int(wave_max(act ? cx : -1));
    const int cyl = uniform_int(wave_min(act ? cy : 0x7fffffff));
    const int cyh = uniform_int(wave_max(act ? cy : -1));

    // near candidates
    if (cxl == cxh && cyh - cyl < 2) {
        int turn = 0;   // groups of four so far, dealt to the waves in turn
        for (int dx = -1; dx <= 1; ++dx) {
            const int xc = cxl + dx;
            if (xc < 0 || xc >= G) continue;
            const int64_t cl = coff + (int64_t)xc * G;
            for (int row = max(cyl - 1, 0); row <= min(cyh + 1, G - 1); ++row) {
                const int a = uniform_int(A.offsets[cl + row]);
                const int b = uniform_int(A.offsets[cl + row + 1]);
                const int first = (w - turn) & (W - 1);
                turn += (b - a + 3) >> 2;
                if (!(act && abs(row - cy) <= 1)) continue;
                if (dx == 0 && row >= cyl && row <= cyh)   // some lanes' own cell
                    near_cell32<W, LAW, true>(A, a + 4 * first, b, (int)A.part_n, gi, x, y, sig,
                                              inv_msc, eps2n, r2cn, sx, sy, s2n);
                else
                    near_cell32<W, LAW, false>(A, a + 4 * first, b, (int)A.part_n, gi, x, y, sig,
                                               inv_msc, eps2n, r2cn, sx, sy, s2n);
            }
        }
    } else if (act) {
        int n0 = 0, n1 = 0, n2 = 0, o0 = 0, o1 = 0, o2 = 0;   // the three ranges as one list
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const int xc = cx + t - 1;
            int a = 0, b = 0;
            if (xc >= 0 && xc < G) {
                const int64_t cl = coff + (int64_t)xc * G;
                a = A.offsets[cl + max(cy - 1, 0)];
                b = A.offsets[cl + min(cy + 1, G - 1) + 1];
            }
            if (t == 0) { o0 = a; n0 = b - a; }
            if (t == 1) { o1 = a - n0; n1 = n0 + b - a; }
            if (t == 2) { o2 = a - n1; n2 = n1 + b - a; }
        }
#pragma unroll 2
        for (int k = w; k < n2; k += W) {
            const int j = k + (k < n0 ? o0 : (k < n1 ? o1 : o2));
            const float wx = (float)fma(A.x[j], sig, -x), wy = (float)fma(A.y[j], sig, -y);
            const float fm = (float)(A.m[j] * inv_msc);
            const float s2 = fmaf(wx, wx, wy * wy);
            float t = fm * __builtin_amdgcn_rcpf(s2 + eps2n);
            const bool keep = j != gi && (LAW == 0 || s2 > r2cn);
            t = keep ? t : 0.0f;
            s2n = fmaf(fm, t, s2n);
            sx += (double)(wx * t);
            sy += (double)(wy * t);
        }
    }

    // COM list: this wave's slice
    const int ne0 = uniform_int(A.neprefix[coff]);
    const int ne1 = uniform_int(A.neprefix[coff + (int64_t)G * G]);
    const int mlo = uniform_int(A.neprefix[coff + (int64_t)max(cxl - 1, 0) * G]);
    const int mhi = uniform_int(A.neprefix[coff + (int64_t)min(cxh + 2, G) * G]);
    const int per = (((ne1 - ne0 + W - 1) / W) + 7) & ~7;
    const int f0 = min(ne1, ne0 + w * per), f1 = min(ne1, f0 + per);
    auto fetch = [&](int e) {
        Com32 c;
        if (e < f1) {
            c = A.l32[e];
        } else {
            c.fx = 1e18f; c.fy = 1e18f; c.rM = __builtin_huge_valf(); c.kxy = 0x7fff7fff;
        }
        return c;
    };
    Com32 nxt = fetch(f0 + lane);
    for (int base = f0; base < f1; base += BH_WAVE) {
        const int kx = nxt.kxy >> 16, ky = nxt.kxy & 0xffff;
        const float ex = (float)(kx - ox) + nxt.fx, ey = (float)(ky - oy) + nxt.fy;
        float4 v;
        if (LAW == 0) {
            v.x = 1e30f; v.y = 1e30f; v.z = 0.0f; v.w = 0.0f;
            if (fabsf(nxt.rM) != __builtin_huge_valf()) {   // M != 0 (NaN passes)
                const float c = msc * nxt.rM;
                v.x = ex * c;
                v.y = ey * c;
                v.z = -c;
                v.w = (c * c) * eps2c;
            }
        } else {
            v.x = ex; v.y = ey; v.z = nxt.rM; v.w = 0.0f;
        }
        ftile[w][lane] = v;
        ktile[w][lane] = nxt.kxy;
        __builtin_amdgcn_wave_barrier();
        nxt = fetch(base + BH_WAVE + lane);
        const int cnt = min(BH_WAVE, (f1 - base + 7) & ~7);   // padded with nothing
        float tx = 0.0f, ty = 0.0f;
        auto term = [&](const float4& f, bool keep) {
            float wx, wy, t;
            if (LAW == 0) {
                wx = fmaf(ux, f.z, f.x);
                wy = fmaf(uy, f.z, f.y);
                t = __builtin_amdgcn_rcpf(fmaf(wx, wx, fmaf(wy, wy, f.w)));
            } else {
                wx = f.x - ux;
                wy = f.y - uy;
                t = far_t32<LAW>(wx, wy, f.z, eps2c, r2c);
            }
            t = keep ? t : 0.0f;
            tx = fmaf(wx, t, tx);
            ty = fmaf(wy, t, ty);
        };
        if (!meets(base, base + BH_WAVE, mlo, mhi)) {
#pragma unroll 8
            for (int j = 0; j < cnt; ++j) term(ftile[w][j], true);
        } else {
            for (int j = 0; j < cnt; ++j) {
                const int k = ktile[w][j];
                term(ftile[w][j], (unsigned)((k >> 16) - cx + 1) > 2u ||
                                      (unsigned)((k & 0xffff) - cy + 1) > 2u);
            }
        }
        fx += (double)tx;
        fy += (double)ty;
        __builtin_amdgcn_wave_barrier();
    }
    // near sums are in units of msc / (1 / sig), far ones of msc / step (LAW 0) or 1 / step
    const double fs = LAW == 0 ? inv_step * (double)msc : inv_step;
    part[0][w][lane] = sx * (sig * (double)msc) + fx * fs;
    part[1][w][lane] = sy * (sig * (double)msc) + fy * fs;
    part2[w][lane] = s2n;
    __syncthreads();
    if (!act) return;
    if (w < 2) {   // wave 0 adds x, wave 1 adds y
        double t = 0.0;
#pragma unroll
        for (int v = 0; v < W; ++v) t += part[w][v][lane];
        double* a = w ? A.ay : A.ax;
        if (A.rc) a[gi] = A.Gc * t;   // a scratch plane: the recompute adds it
        else a[gi] += A.Gc * t;
    } else if (w == 2 && A.rc) {   // sum of (m / r)^2, r in cells
        double t = 0.0;
#pragma unroll
        for (int v = 0; v < W; ++v) t += (double)part2[v][lane];
        const double ms = (double)msc * (step * sig);
        A.ay[A.part_n + gi] = t * (ms * ms);
    }
}

// ---------------------------------------------------------------- FP32 + matrix cores
// Same decomposition and coordinates as k_force32, with the far-field sum
// split as  sum_k M_k r_k (a_k - u) = sum_k r_k (M_k a_k) - u sum_k r_k M_k,
// r_k = 1/(|a_k - u|^2 + eps2).  Per COM entry the tile holds
// B_k = (M a_x, M a_y, M, 0); every lane computes r_k for its particle (2 sub,
// r^2 as mul+fma, v_rcp_f32) and v_mfma_f32_4x4x1f32 adds B_k * r_k into the
// lane's own column: with A from lane 4b+c and B from lane l, lane l's
// register c receives A(lane 4*(l/4) + c) * B(lane l).  So lane 4b+c supplies
// component c of B_k as the A operand and its own r_k as the B operand.  The matrix unit accumulates one
// 64-entry tile (FP32); tiles are Kahan-summed; the final combination
// sum r M a - u sum r M is done in FP64.  Near field as in k_force32.
typedef float mf4 __attribute__((ext_vector_type(4)));

template <int P, int LAW>
__global__ __launch_bounds__(64) void k_force32m(ForceArgs A)
{
    __shared__ float2 atile[BH_WAVE];          // (a_x, a_y) relative to the item origin
    __shared__ float btile[BH_WAVE][4];        // (M a_x, M a_y, M, 0)
    __shared__ int32_t ktile[BH_WAVE];         // kx << 16 | ky
    __shared__ NearE ntile[BH_WAVE];
    const int lane = threadIdx.x;
    const int bc = lane & 3;
    const int nitems = A.stats[ST_NITEMS];
    int qb, qe;
    part_range(nitems, A.qpart, A.nqparts, qb, qe);
    for (;;) {
        const int q = qb + next_item(A.stats, lane);
        if (q >= qe) break;
        const long long t0 = A.cost_log ? (long long)wall_clock64() : 0;
        const int itx = A.order ? uniform_int(A.order[q]) : q;
        if ((unsigned)itx >= (unsigned)nitems) continue;
        const Item it = A.items[itx];
        const SysDev& d = A.sys[it.sys];
        const int G = d.G;
        const int64_t coff = d.c_off;
        const int cx = it.cx;
        const int oy = (it.y0 + it.y1) >> 1;
        const int ylo = max(it.y0 - 1, 0), yhi = min(it.y1 + 1, G - 1);
        const double step = d.step;
        const double inv_step = 1.0 / step;
        const float eps2c = (float)(A.eps2 * inv_step * inv_step);
        const float r2c = (float)(A.r2cut * inv_step * inv_step);

        double xi[P], yi[P];
        float ux[P], uy[P], Sx[P], Sy[P], Cx[P], Cy[P], tx[P], ty[P];
        float Fx[P], Fy[P], Fm[P], Gx[P], Gy[P], Gm[P];   // far sums (Kahan) of r M a_x, r M a_y, r M
        int cy[P], gi[P];
        bool act[P];
#pragma unroll
        for (int k = 0; k < P; ++k) {
            int slot = lane + BH_WAVE * k;
            act[k] = slot < it.np;
            gi[k] = it.p0 + slot;
            xi[k] = 0.0;
            yi[k] = 0.0;
            ux[k] = 0.0f;
            uy[k] = 0.0f;
            cy[k] = -100000;
            if (act[k]) {
                xi[k] = A.x[gi[k]];
                yi[k] = A.y[gi[k]];
                cy[k] = (int)(A.key_sorted[gi[k]] - coff) - cx * G;
                ux[k] = (float)((xi[k] - d.min_x) / step - (double)cx);
                uy[k] = (float)((yi[k] - d.min_y) / step - (double)oy);
            }
            Sx[k] = Sy[k] = Cx[k] = Cy[k] = tx[k] = ty[k] = 0.0f;
            Fx[k] = Fy[k] = Fm[k] = Gx[k] = Gy[k] = Gm[k] = 0.0f;
        }

        // near field (separations in FP64, rounded once to FP32)
        for (int dx = -1; dx <= 1; ++dx) {
            const int xc = cx + dx;
            if (xc < 0 || xc >= G) continue;
            const int64_t cl = coff + (int64_t)xc * G;
            const int pa = A.offsets[cl + ylo], pb = A.offsets[cl + yhi + 1];
            for (int base = pa; base < pb; base += BH_WAVE) {
                const int j = base + lane;
                NearE e;
                if (j < pb) {
                    e.x = A.x[j];
                    e.y = A.y[j];
                    e.m = A.m[j];
                    e.row = (int)(A.key_sorted[j] - cl);
                    e.idx = j;
                } else {
                    e.x = 0.0;
                    e.y = 0.0;
                    e.m = 0.0;
                    e.row = -100000;
                    e.idx = -1;
                }
                ntile[lane] = e;
                __syncthreads();
                const int cnt = min(BH_WAVE, pb - base);
                for (int jj = 0; jj < cnt; ++jj) {
                    const NearE f = ntile[jj];
                    const float fm = (float)f.m;
#pragma unroll
                    for (int k = 0; k < P; ++k) {
                        const bool keep = (f.idx != gi[k]) && (abs(f.row - cy[k]) <= 1);
                        const float wx = (float)((f.x - xi[k]) * inv_step);
                        const float wy = (float)((f.y - yi[k]) * inv_step);
                        const float s2 = fmaf(wx, wx, wy * wy);
                        float t = fm * __builtin_amdgcn_rcpf(s2 + eps2c);
                        if (LAW == 1) t = (s2 > r2c) ? t : 0.0f;
                        t = keep ? t : 0.0f;
                        tx[k] = fmaf(wx, t, tx[k]);
                        ty[k] = fmaf(wy, t, ty[k]);
                    }
                }
#pragma unroll
                for (int k = 0; k < P; ++k) {
                    kahan_add(Sx[k], Cx[k], tx[k]);
                    kahan_add(Sy[k], Cy[k], ty[k]);
                    tx[k] = 0.0f;
                    ty[k] = 0.0f;
                }
                __syncthreads();
            }
        }

        // far field
        const int ne0 = A.neprefix[coff], ne1 = A.neprefix[coff + (int64_t)G * G];
        int mlo[3], mhi[3];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const int xc = cx + t - 1;
            if (xc >= 0 && xc < G) {
                const int64_t cl = coff + (int64_t)xc * G;
                mlo[t] = A.neprefix[cl + ylo];
                mhi[t] = A.neprefix[cl + yhi + 1];
            } else {
                mlo[t] = 0;
                mhi[t] = 0;
            }
        }
        Com32 nxt;
        {
            const int e = ne0 + lane;
            if (e < ne1) nxt = A.l32[e];
            else { nxt.fx = 1e18f; nxt.fy = 1e18f; nxt.rM = __builtin_huge_valf(); nxt.kxy = 0x7fff7fff; }
        }
        for (int base = ne0; base < ne1; base += BH_WAVE) {
            {
                const int kx = nxt.kxy >> 16, ky = nxt.kxy & 0xffff;
                const float ax_ = (float)(kx - cx) + nxt.fx;
                const float ay_ = (float)(ky - oy) + nxt.fy;
                atile[lane] = make_float2(ax_, ay_);
                const float Mv = 1.0f / nxt.rM;
                btile[lane][0] = Mv * ax_;
                btile[lane][1] = Mv * ay_;
                btile[lane][2] = Mv;
                btile[lane][3] = 0.0f;
                ktile[lane] = nxt.kxy;
            }
            __syncthreads();
            {
                const int e = base + BH_WAVE + lane;
                if (e < ne1) nxt = A.l32[e];
                else { nxt.fx = 1e18f; nxt.fy = 1e18f; nxt.rM = __builtin_huge_valf(); nxt.kxy = 0x7fff7fff; }
            }
            const int b1 = base + BH_WAVE;
            const bool masked = meets(base, b1, mlo[0], mhi[0]) || meets(base, b1, mlo[1], mhi[1]) ||
                                meets(base, b1, mlo[2], mhi[2]);
            mf4 acc[P];
#pragma unroll
            for (int k = 0; k < P; ++k) acc[k] = (mf4){0.0f, 0.0f, 0.0f, 0.0f};
            if (!masked) {
#pragma unroll
                for (int j = 0; j < BH_WAVE; ++j) {
                    const float2 a = atile[j];
                    const float bj = btile[j][bc];
#pragma unroll
                    for (int k = 0; k < P; ++k) {
                        const float wx = a.x - ux[k], wy = a.y - uy[k];
                        float r;
                        if (LAW == 0) {
                            r = __builtin_amdgcn_rcpf(fmaf(wx, wx, fmaf(wy, wy, eps2c)));
                        } else {
                            const float s2 = fmaf(wx, wx, wy * wy);
                            r = (s2 > r2c) ? __builtin_amdgcn_rcpf(s2 + eps2c) : 0.0f;
                        }
                        acc[k] = __builtin_amdgcn_mfma_f32_4x4x1f32(bj, r, acc[k], 0, 0, 0);
                    }
                }
            } else {
                for (int j = 0; j < BH_WAVE; ++j) {
                    const float2 a = atile[j];
                    const float bj = btile[j][bc];
                    const int kxy = ktile[j];
                    const bool colnear = abs((kxy >> 16) - cx) <= 1;
                    const int ky = kxy & 0xffff;
#pragma unroll
                    for (int k = 0; k < P; ++k) {
                        const bool keep = !(colnear && abs(ky - cy[k]) <= 1);
                        const float wx = a.x - ux[k], wy = a.y - uy[k];
                        float r;
                        if (LAW == 0) {
                            r = __builtin_amdgcn_rcpf(fmaf(wx, wx, fmaf(wy, wy, eps2c)));
                        } else {
                            const float s2 = fmaf(wx, wx, wy * wy);
                            r = (s2 > r2c) ? __builtin_amdgcn_rcpf(s2 + eps2c) : 0.0f;
                        }
                        r = keep ? r : 0.0f;
                        acc[k] = __builtin_amdgcn_mfma_f32_4x4x1f32(bj, r, acc[k], 0, 0, 0);
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < P; ++k) {
                kahan_add(Fx[k], Gx[k], acc[k][0]);
                kahan_add(Fy[k], Gy[k], acc[k][1]);
                kahan_add(Fm[k], Gm[k], acc[k][2]);
            }
            __syncthreads();
        }

        const double scale = A.Gc * inv_step;
#pragma unroll
        for (int k = 0; k < P; ++k) {
            if (act[k]) {
                const double sm = (double)Fm[k] - (double)Gm[k];
                const double fx = ((double)Fx[k] - (double)Gx[k]) - (double)ux[k] * sm;
                const double fy = ((double)Fy[k] - (double)Gy[k]) - (double)uy[k] * sm;
                const double rx = fx + ((double)Sx[k] - (double)Cx[k]);
                const double ry = fy + ((double)Sy[k] - (double)Cy[k]);
                A.ax[gi[k]] += scale * rx;
                A.ay[gi[k]] += scale * ry;
            }
        }
        if (A.cost_log && lane == 0) A.cost_log[itx] = (long long)wall_clock64() - t0;
    }
}

// ---------------------------------------------------------------- dispatch table
typedef void (*force_fn)(ForceArgs);

#define F64(P, L) (force_fn)k_force64<P, L, 1>
#define F64I(P, L) (force_fn)k_force64<P, L, 0>
#define F32(P, L, K) (force_fn)k_force32<P, L, K>
#define F32M(P, L) (force_fn)k_force32m<P, L>

// [precision: 0 fp64, 1..3 fp32 kahan mode 1,2,0, 4 fp32 matrix-core, 5 fp64 IEEE
// division][P index][law]
static const force_fn g_force[6][3][2] = {
    {{F64(1, 0), F64(1, 1)}, {F64(2, 0), F64(2, 1)}, {F64(4, 0), F64(4, 1)}},
    {{F32(1, 0, 1), F32(1, 1, 1)}, {F32(2, 0, 1), F32(2, 1, 1)}, {F32(4, 0, 1), F32(4, 1, 1)}},
    {{F32(1, 0, 2), F32(1, 1, 2)}, {F32(2, 0, 2), F32(2, 1, 2)}, {F32(4, 0, 2), F32(4, 1, 2)}},
    {{F32(1, 0, 0), F32(1, 1, 0)}, {F32(2, 0, 0), F32(2, 1, 0)}, {F32(4, 0, 0), F32(4, 1, 0)}},
    {{F32M(1, 0), F32M(1, 1)}, {F32M(2, 0), F32M(2, 1)}, {F32M(4, 0), F32M(4, 1)}},
    {{F64I(1, 0), F64I(1, 1)}, {F64I(2, 0), F64I(2, 1)}, {F64I(4, 0), F64I(4, 1)}},
};

const void* bh_force_kernel(int precision, int pidx, int law)
{
    if (precision < 0 || precision > 5 || pidx < 0 || pidx > 2 || law < 0 || law > 1) return nullptr;
    return (const void*)g_force[precision][pidx][law];
}

void bh_force64s(const ForceArgs& A, int law, int S, int64_t nchunks, hipStream_t st)
{
    const dim3 g((unsigned)nchunks), b(64 * F64S_WAVES);
    if (law) hipLaunchKernelGGL((k_force64s<F64S_WAVES, 1>), g, b, 0, st, A, S);
    else hipLaunchKernelGGL((k_force64s<F64S_WAVES, 0>), g, b, 0, st, A, S);
}

void bh_force32s(const ForceArgs& A, int law, int S, int64_t nchunks, hipStream_t st)
{
    const dim3 g((unsigned)nchunks), b(64 * F32S_WAVES);
    if (law) hipLaunchKernelGGL((k_force32s<F32S_WAVES, 1>), g, b, 0, st, A, S);
    else hipLaunchKernelGGL((k_force32s<F32S_WAVES, 0>), g, b, 0, st, A, S);
}
