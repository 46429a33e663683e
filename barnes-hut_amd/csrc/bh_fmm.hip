// Grouped far field: the same sums as the term-by-term force kernels, with
// the COMs of distant cells taken in groups.
//
// A system's grid is covered by square tiles of T cells per side (fmm_tile).  A
// particle's terms split into
//   near     the particles of its 3x3 cells, one by one;
//   mid      the COMs of the other non-empty cells of its 3x3 tiles, one by one;
//   distant  the COMs of all other cells, at least T cells away.
// The law's weight 1 / (r^2 + eps2) is smooth over the distant part (softening
// only makes it smoother), so that part is interpolated: on each tile, and on
// each square of 2^l tiles per side, a P x P Chebyshev grid carries the
// sources up (anterpolated masses at the nodes) and the field down (ax, ay at
// the nodes).  Two squares interact directly (the law between their nodes) at
// the coarsest level where they are not neighbours while their parents are.
// Interpolating across a gap of one square converges as 5.8^-P: P = 12 leaves
// 1.3e-10 of the far field (the FP32 precision's own rounding was 4e-8), and
// P = 20 leaves 1e-15, below the rounding of a term-by-term FP64 sum over
// 10^4 cells and more.  Across a gap of two squares, or past a corner, it
// converges as 9.9^-F or 8.6^-F, so these 15 of a square's 27 take F = 10 or 16
// nodes a side for the same remainder.  Everything here is FP64.
//
// Work per pass: 12 node-to-node products of (2 P^2) x P^2 and 15 of (2 F^2) x
// F^2 per square instead of one term per (particle, cell): 4.2M particles on
// 1024^2 cells go from 2.0e12 far terms to ~4e9 terms and ~4.4e5 products.
#include "bh_common.h"
#include "bh_kernels.h"

#define FMM_IN 1.0001   // |coordinate| on a square up to which it counts as inside

typedef double fd4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- tiles
// Eight lanes per tile add up its columns' particles and non-empty cells; the
// block reserves runs of the chunk list (64 particles of one tile each) and of
// the tile-ordered COM list with one atomic each.  Chunks of dense tiles, whose
// particles have many near candidates, fill the chunk list from its start (a
// block shares each of them), the others from its end (a wave each).  The
// order of the runs varies from launch to launch; no result depends on it.
__global__ __launch_bounds__(256) void k_fmm_tiles(FmmArgs A)
{
    __shared__ int wc[4], we[4], wd[4], base_c, base_e, base_d;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int64_t t = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> 3;
    const int sub = threadIdx.x & 7;
    int np = 0, ne = 0;
    float n2 = 0.0f;   // sum of squared cell counts
    FmmTile tl = {0, 0, 0};
    if (t < A.nleaf) {
        tl = A.tiles[t];
        const SysDev& d = A.sys[tl.sys];
        const int T = A.fsys[tl.sys].T;
        const int x0 = tl.tx * T, y0 = tl.ty * T;
        const int x1 = min(x0 + T, d.G), y1 = min(y0 + T, d.G);
        for (int x = x0 + sub; x < x1; x += 8) {
            const int64_t cl = d.c_off + (int64_t)x * d.G;
            int a = A.offsets[cl + y0];
            for (int y = y0; y < y1; ++y) {
                const int b = A.offsets[cl + y + 1];
                n2 += (float)(b - a) * (float)(b - a);
                np += b - a;
                a = b;
            }
            ne += A.neprefix[cl + y1] - A.neprefix[cl + y0];
        }
    }
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) {
        np += __shfl_xor(np, o, BH_WAVE);
        ne += __shfl_xor(ne, o, BH_WAVE);
        n2 += __shfl_xor(n2, o, BH_WAVE);
    }
    const bool dense = n2 > (float)FMM_DENSE * (float)np;
    const int nch = (np + 63) >> 6;
    const int nc = dense ? 0 : nch, nd = dense ? nch : 0;
    const int ner = (ne + 3) & ~3;   // a tile's run of the list is padded to whole quads
    // exclusive prefix over the wave's eight tiles
    int pc = nc, pe = ner, pd = nd;
#pragma unroll
    for (int o = 8; o < 64; o <<= 1) {
        const int a = __shfl_up(pc, o, BH_WAVE), b = __shfl_up(pe, o, BH_WAVE);
        const int g = __shfl_up(pd, o, BH_WAVE);
        if (lane >= o) {
            pc += a;
            pe += b;
            pd += g;
        }
    }
    if (lane == 63) {
        wc[wid] = pc;
        we[wid] = pe;
        wd[wid] = pd;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int c = 0, e = 0, g = 0;
        for (int w = 0; w < 4; ++w) {
            const int a = wc[w], b = we[w], v = wd[w];
            wc[w] = c;
            we[w] = e;
            wd[w] = g;
            c += a;
            e += b;
            g += v;
        }
        base_c = c ? atomicAdd(&A.cnt[FMM_LIGHT], c) : 0;
        base_e = e ? atomicAdd(&A.cnt[FMM_LIST], e) : 0;
        base_d = g ? atomicAdd(&A.cnt[FMM_HEAVY], g) : 0;
    }
    __syncthreads();
    if (t >= A.nleaf) return;
    const int c0 = base_c + wc[wid] + pc - nc, d0 = base_d + wd[wid] + pd - nd;
    const int e0 = base_e + we[wid] + pe - ner;
    if (sub == 0) {
        A.tcnt[t] = np;
        A.tstart[t] = e0;
        A.tne[t] = ne;
    }
    for (int k = sub; k < nch; k += 8) {
        FmmChunk c;
        c.tile = (int32_t)t;
        c.k = k;
        A.chunks[dense ? d0 + k : A.max_chunks - 1 - (c0 + k)] = c;
    }
}

// ---------------------------------------------------------------- small products
#define FMM_THREADS 128   // of the kernels that take a square per block

// For NF pairs A_z (M x K, at A + z az) and B_z (K x N, at B + z bz), row-major in
// LDS on 16 bytes: C_z[m][n] = sum_k A_z[m][k] B_z[k][n], handed to put(z, m, n, C)
// in pieces of 2 x NB.  A thread's piece takes 6 bytes of LDS reads a multiply-add
// (16 with an element per thread); these reads bound the kernels below.  One
// element per thread, 256 threads: 4.2M FP64 particles on 1024^2 cells p2m 181, m2m
// 5 x 24.7, l2l 6 x 39 us; in pieces 129, 5 x 23 and 6 x 22.  512 systems: 413, 3 x
// 60, 4 x 80; 382, 3 x 64 and 4 x 55.
template <int N>
constexpr int piece() { return N % 4 == 0 ? 4 : 2; }

template <int M, int N, int K, int NF, int TH = FMM_THREADS, typename Put>
__device__ __forceinline__ void products(const double* A, int az, const double* B, int bz,
                                         Put&& put)
{
    constexpr int NB = piece<N>(), PM = M / 2, PN = N / NB;
    static_assert(M % 2 == 0 && N % NB == 0 && K % 2 == 0, "whole pieces");
    for (int u = threadIdx.x; u < NF * PM * PN; u += TH) {
        const int z = u / (PM * PN), r = u - z * (PM * PN);
        const int m = 2 * (r / PN), n = NB * (r % PN);
        const double *a = A + z * az + m * K, *b = B + z * bz + n;
        double c[2][NB] = {};
#pragma unroll
        for (int k = 0; k < K; k += 2) {
            const double2 a0 = *(const double2*)(a + k);
            const double2 a1 = *(const double2*)(a + K + k);
#pragma unroll
            for (int v = 0; v < NB; v += 2) {
                const double2 b0 = *(const double2*)(b + k * N + v);
                const double2 b1 = *(const double2*)(b + (k + 1) * N + v);
                c[0][v] = fma(a0.y, b1.x, fma(a0.x, b0.x, c[0][v]));
                c[0][v + 1] = fma(a0.y, b1.y, fma(a0.x, b0.y, c[0][v + 1]));
                c[1][v] = fma(a1.y, b1.x, fma(a1.x, b0.x, c[1][v]));
                c[1][v + 1] = fma(a1.y, b1.y, fma(a1.x, b0.y, c[1][v + 1]));
            }
        }
        put(z, m, n, c);
    }
}

// A piece into a row-major N-wide matrix in LDS.
template <int N, int NB>
__device__ __forceinline__ void put_lds(double* D, int m, int n, const double (&c)[2][NB])
{
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
        for (int v = 0; v < NB; ++v) D[(m + w) * N + n + v] = c[w][v];
}

// An R x C table from global memory, and its transpose.
template <int R, int C, int TH = FMM_THREADS>
__device__ __forceinline__ void load_table(const double* __restrict__ g, double* t, double* tt)
{
    for (int q = threadIdx.x; q < R * C; q += TH) {
        const double v = g[q];
        if (t) t[q] = v;
        if (tt) tt[(q % C) * R + q / C] = v;
    }
}

// ---------------------------------------------------------------- sources up
// A square's node masses C (P^2, in LDS) anterpolated to its F x F coarser nodes
// (fine[I][i]: the coarse cardinal I at node i; fineT its transpose); V: scratch
// for F P.  By the whole block.
template <int P, int F, int TH = FMM_THREADS>
__device__ __forceinline__ void coarse_masses(const double* C, double* V, const double* fine,
                                              const double* fineT, double* M, int64_t plane)
{
    __syncthreads();
    products<F, P, P, 1, TH>(fine, 0, C, 0, [&](int, int m, int n, const auto& c) {
        put_lds<P>(V, m, n, c);
    });
    __syncthreads();
    products<F, F, P, 1, TH>(V, 0, fineT, 0, [&](int, int m, int n, const auto& c) {
#pragma unroll
        for (int w = 0; w < 2; ++w)
#pragma unroll
            for (int v = 0; v < piece<F>(); ++v) M[((m + w) * F + n + v) * plane] = c[w][v];
    });
}

// One block per tile: the tile's COMs into the tile-ordered list, and their
// masses anterpolated to the tile's nodes: Chebyshev moments
// W_kl = sum M T_k(x) T_l(y) over the entries, then nodes = C^T W C.
template <int P>
__global__ __launch_bounds__(FMM_THREADS) void k_fmm_p2m(FmmArgs A,
                                                         const double* __restrict__ ctab,
                                                         const double* __restrict__ ftab)
{
    constexpr int Q = P * P, F = fmm_far(P), EB = 32, NB = piece<P>();
    // tx, ty: T_k of the entries; afterwards scratch and the coarser nodes' tables
    __shared__ alignas(16) double tx[P * EB], ty[EB * P], W[Q], ct[Q], ctT[Q];
    static_assert(Q <= P * EB && 2 * F * P <= P * EB, "room in tx and ty");
    double *V = tx, *fine = ty, *fineT = ty + F * P;
    const int tid = threadIdx.x;
    const int64_t t = blockIdx.x;
    const FmmTile tl = A.tiles[t];
    const SysDev& d = A.sys[tl.sys];
    const FmmSys& fs = A.fsys[tl.sys];
    const int T = fs.T, ne = A.tne[t], e0 = A.tstart[t];
    const int x0 = tl.tx * T, y0 = tl.ty * T;
    const int x1 = min(x0 + T, d.G), y1 = min(y0 + T, d.G);
    const double sig = step_scale(d.step);
    double *M = nullptr, *MF = nullptr;   // node q's mass goes to M[q * plane]
    int64_t plane = 0;
    const bool up = fs.nlev > 0;
    if (up) {
        plane = fmm_plane(fs.n[0]);
        M = A.mult + fs.moff[0] * Q + fmm_slot(fs.n[0], tl.tx, tl.ty);
        MF = A.multf + fs.moff[0] * (F * F) + fmm_slot(fs.n[0], tl.tx, tl.ty);
        if (ne > 0) load_table<P, P>(ctab, ct, ctT);
    }
    const double h = (double)T * d.step;
    // a thread's piece of the moments, over all entries
    constexpr int PN = P / NB;
    const int pm = 2 * (tid / PN), pn = NB * (tid % PN);
    double acc[2][NB] = {};
    int cx = x0, cb = A.neprefix[d.c_off + (int64_t)x0 * d.G + y0];
    int cn = A.neprefix[d.c_off + (int64_t)x0 * d.G + y1] - cb, cpre = 0;
    for (int b = 0; b < ne; b += EB) {
        const int nb = min(EB, ne - b);
        const int el = tid & (EB - 1);   // threads 0 .. 31 take x, 32 .. 63 y
        if (tid < 2 * EB && el < nb) {
            const int r = b + el;   // entry rank in the tile, columns in order
            while (r - cpre >= cn && cx + 1 < x1) {
                cpre += cn;
                ++cx;
                const int64_t cl = d.c_off + (int64_t)cx * d.G;
                cb = A.neprefix[cl + y0];
                cn = A.neprefix[cl + y1] - cb;
            }
            const Com64 c = A.l64[cb + (r - cpre)];
            const double ux = 2.0 * ((c.X - d.min_x) / h - tl.tx) - 1.0;
            const double uy = 2.0 * ((c.Y - d.min_y) / h - tl.ty) - 1.0;
            if (tid < EB) {
                FmmCom f;
                f.X = c.X * sig;
                f.Y = c.Y * sig;
                f.M = c.M;
                f.kx = c.kx;
                f.ky = c.ky;
                if (c.M == 0.0) {   // no COM: any point of the cell, at weight 0
                    f.X = fma((double)c.kx + 0.5, d.step, d.min_x) * sig;
                    f.Y = fma((double)c.ky + 0.5, d.step, d.min_y) * sig;
                }
                A.list[e0 + r] = f;
                // masses of both signs can put a COM outside its tile, where
                // the interpolation does not hold: that system goes term by term
                if (up && c.M != 0.0 && !(fabs(ux) <= FMM_IN && fabs(uy) <= FMM_IN))
                    A.sbad[tl.sys] = 1;
            }
            // T_k(x) M and T_k(y)
            const double u = tid < EB ? ux : uy;
            double t0 = tid < EB ? c.M : 1.0, t1 = t0 * u;
            if (c.M == 0.0) t0 = t1 = 0.0;
            double* dst = tid < EB ? tx + el : ty + el * P;
            const int step = tid < EB ? EB : 1;
#pragma unroll
            for (int k = 0; k < P; ++k) {
                dst[k * step] = t0;
                const double tn = fma(2.0 * u, t1, -t0);
                t0 = t1;
                t1 = c.M == 0.0 ? 0.0 : tn;
            }
        } else if (tid < 2 * EB && el == nb) {   // past an odd last entry: nothing
            for (int k = 0; k < P; ++k) {
                if (tid < EB) tx[k * EB + el] = 0.0;
                else ty[el * P + k] = 0.0;
            }
        }
        if (!up) continue;
        __syncthreads();
        if (pm < P) {
#pragma unroll 4
            for (int e = 0; e < nb; e += 2) {
                const double2 a0 = *(const double2*)(tx + pm * EB + e);
                const double2 a1 = *(const double2*)(tx + (pm + 1) * EB + e);
#pragma unroll
                for (int v = 0; v < NB; ++v) {
                    const double b0 = ty[e * P + pn + v], b1 = ty[(e + 1) * P + pn + v];
                    acc[0][v] = fma(a0.y, b1, fma(a0.x, b0, acc[0][v]));
                    acc[1][v] = fma(a1.y, b1, fma(a1.x, b0, acc[1][v]));
                }
            }
        }
        __syncthreads();
    }
    if (tid < (-ne & 3)) {   // padding: no mass, far away (three in a product of four)
        FmmCom f;
        f.X = 1e30;
        f.Y = 1e30;
        f.M = 0.0;
        f.kx = 0x3fffffff;   // after the last column
        f.ky = 0x3fffffff;
        A.list[e0 + ne + tid] = f;
    }
    if (!up) return;
    if (ne == 0) {   // uniform over the block
        for (int q = tid; q < Q; q += FMM_THREADS) M[q * plane] = 0.0;
        for (int q = tid; q < F * F; q += FMM_THREADS) MF[q * plane] = 0.0;
        return;
    }
    if (pm < P) put_lds<P>(W, pm, pn, acc);
    load_table<F, P>(ftab, fine, fineT);
    __syncthreads();
    products<P, P, P, 1>(ctT, 0, W, 0, [&](int, int m, int n, const auto& c) {
        put_lds<P>(V, m, n, c);
    });
    __syncthreads();
    products<P, P, P, 1>(V, 0, ct, 0, [&](int, int m, int n, const auto& c) {
        put_lds<P>(W, m, n, c);
#pragma unroll
        for (int w = 0; w < 2; ++w)
#pragma unroll
            for (int v = 0; v < NB; ++v) M[((m + w) * P + n + v) * plane] = c[w][v];
    });
    coarse_masses<P, F>(W, V, fine, fineT, MF, plane);
}

// One block per square of level lev: its children's node masses anterpolated
// to its own nodes (shift[a][i][I]: the parent's cardinal i at child node I).  The
// four children are read and taken through the first product together: the few
// squares of the upper levels are a chain of latencies.
template <int P>
__global__ __launch_bounds__(256) void k_fmm_m2m(FmmArgs A, const double* __restrict__ shift,
                                                 const double* __restrict__ ftab, int lev)
{
    constexpr int Q = P * P, F = fmm_far(P), TH = 256;
    __shared__ alignas(16) double S[2 * Q], ST[2 * Q], C[4 * Q], V[4 * Q];
    const int tid = threadIdx.x;
    const int64_t t = A.lev_off[lev] + blockIdx.x;
    const FmmTile tl = A.tiles[t];
    const FmmSys& fs = A.fsys[tl.sys];
    const int nc = fs.n[lev - 1];
    const int64_t cplane = fmm_plane(nc), plane = fmm_plane(fs.n[lev]);
    int np = 0;
    bool has[4];
#pragma unroll
    for (int ch = 0; ch < 4; ++ch) {
        const int cx = 2 * tl.tx + (ch >> 1), cy = 2 * tl.ty + (ch & 1);
        int n = 0;
        if (cx < nc && cy < nc) n = A.tcnt[fs.off[lev - 1] + (int64_t)cx * nc + cy];
        has[ch] = n != 0;
        np += n;
    }
    if (tid == 0) A.tcnt[t] = np;
    double* M = A.mult + fs.moff[lev] * Q + fmm_slot(fs.n[lev], tl.tx, tl.ty);
    double* MF = A.multf + fs.moff[lev] * (F * F) + fmm_slot(fs.n[lev], tl.tx, tl.ty);
    if (np == 0) {   // uniform over the block
        for (int q = tid; q < Q; q += TH) M[q * plane] = 0.0;
        for (int q = tid; q < F * F; q += TH) MF[q * plane] = 0.0;
        return;
    }
#pragma unroll
    for (int ch = 0; ch < 4; ++ch) {
        const double* src = A.mult + fs.moff[lev - 1] * Q +
                            fmm_slot(nc, 2 * tl.tx + (ch >> 1), 2 * tl.ty + (ch & 1));
        for (int q = tid; q < Q; q += TH) C[ch * Q + q] = has[ch] ? src[q * cplane] : 0.0;
    }
    load_table<P, P, TH>(shift, S, ST);
    load_table<P, P, TH>(shift + Q, S + Q, ST + Q);
    __syncthreads();
    auto in_V = [&](int c, int m, int n, const auto& v) { put_lds<P>(V + c * Q, m, n, v); };
    products<P, P, P, 2, TH>(S, 0, C, Q, in_V);
    products<P, P, P, 2, TH>(S + Q, 0, C + 2 * Q, Q, [&](int c, int m, int n, const auto& v) {
        put_lds<P>(V + (c + 2) * Q, m, n, v);
    });
    __syncthreads();
    // children (0, b) and (1, b) by the shift of b, then the four are added
#pragma unroll
    for (int b = 0; b < 2; ++b)
        products<P, P, P, 2, TH>(V + b * Q, 2 * Q, ST + b * Q, 0,
                                 [&](int a, int m, int n, const auto& v) {
                                     put_lds<P>(C + (2 * a + b) * Q, m, n, v);
                                 });
    __syncthreads();
    for (int q = tid; q < Q; q += TH) {
        const double s = ((C[q] + C[Q + q]) + C[2 * Q + q]) + C[3 * Q + q];
        V[q] = s;
        M[q * plane] = s;
    }
    load_table<F, P, TH>(ftab, S, S + Q);
    coarse_masses<P, F, TH>(V, V + Q, S, S + Q, MF, plane);
}

// ---------------------------------------------------------------- node to node
// One wave per (64 targets of one level and child position, 16 target nodes,
// near or far offsets).  For each of its 12 or 15 offsets a wave forms its 16 x Q
// slice of the law between target and source nodes in registers, one entry per
// lane and step (two components), and multiplies it with the 64 sources' node
// masses on the FP64 matrix unit: A = 16 target nodes x 4 source nodes, B = 4
// source nodes x 16 squares, four B blocks per A.  Forming an entry costs ~11
// issue slots per lane, the eight products it feeds 8 x 16, so the matrix unit is
// the bound.  Softening enters relative to the square's size, which differs by
// level and system; forming the slice on the fly needs no table of them.
// 4.2M particles, 1024^2 cells, tiles of 8: P = 20 4.6 ms (7.0 with all 27 offsets
// at P), 55 TFLOP/s (a large FP64 matrix product reaches 73; the unit is busy 0.74
// of the cycles, at 2.27 GHz), P = 12 0.76 ms (0.98); 512 systems 2.3 ms (2.7).  F = 8
// for P = 12 would take 0.56 and 1.6 ms but leaves 1e-9 of the far field, and
// single particles whose terms cancel up to 6e-6.  Tried: sources square-major
// (one line per 16 bytes read: 76 ms at P = 20 with 27 offsets, against 7.0);
// waves of several node rows sharing a workgroup (8.5 ms: its waves spread
// unevenly over the SIMDs); node rows of a group kept on one XCD (6.8 ms, but
// 4.3 instead of 2.8 ms on 512 systems, whose groups differ in size).
// NB: blocks of 16 targets (no branch inside: a branch around a product would
// copy its accumulators).
template <int P, int NB, bool FAR>
__device__ __forceinline__ void m2l_wave(const FmmArgs& A, const FmmGroup& gr, int rb, double eps2,
                                         const double* hn)
{
    constexpr int Q = P * P, QP = P / 4;
    constexpr int U = P % 4 == 0 ? 2 : 1;   // products between loads
    static_assert(Q % 4 == 0, "a lane group takes a quarter of the nodes");
    const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
    const FmmSys& fs = A.fsys[gr.sys];
    const int lev = gr.lev, n = fs.n[lev], off = fs.off[lev];
    const int ny = (n - gr.b + 1) >> 1;   // targets of this child position: columns of ny
    const int w = fmm_pitch(n);
    const int64_t plane = fmm_plane(n);
    const double* M = (FAR ? A.multf : A.mult) + fs.moff[lev] * Q;
    const double h = (double)fs.T * A.sys[gr.sys].step * (double)(1 << lev);
    const double e2 = eps2 / (h * h);
    int tx[NB], ty[NB], tg[NB];
    unsigned pos[NB];   // byte offset of the target's place in a class, plus the lane's first node
    bool any = false;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int t = gr.t0 + 16 * b + c;
        const bool ok = 16 * b + c < gr.cnt;
        const int i = ok ? t / ny : 0, j = ok ? t - i * ny : 0;
        tx[b] = 2 * i + gr.a;
        ty[b] = 2 * j + gr.b;
        tg[b] = ok ? off + tx[b] * n + ty[b] : -1;
        if (ok && A.tcnt[tg[b]] == 0) tg[b] = -1;
        pos[b] = (unsigned)(((i + 1) * w + j + 1 + g * (Q / 4) * plane) * sizeof(double));
        any = any || tg[b] >= 0;
    }
    if (!__any(any)) return;
    const int row = min(16 * rb + c, Q - 1);   // the last block may repeat the last node
    const double xt = hn[row / P], yt = hn[row % P];
    fd4 ax[NB] = {}, ay[NB] = {};
    for (int o = 0; o < 36; ++o) {
        const int pi = o / 12 - 1, ca = (o / 6) & 1, pj = (o % 6) / 2 - 1, cb = o & 1;
        const int ox = 2 * pi + ca - gr.a, oy = 2 * pj + cb - gr.b;
        if (abs(ox) <= 1 && abs(oy) <= 1) continue;
        if (fmm_is_far(ox, oy) != FAR) continue;
        bool act = false;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int sx = tx[b] + ox, sy = ty[b] + oy;
            const bool in = tg[b] >= 0 && sx >= 0 && sx < n && sy >= 0 && sy < n;
            act = act || (in && A.tcnt[in ? off + sx * n + sy : 0] > 0);
        }
        if (!__any(act)) continue;
        // the sources' class, shifted by (pi, pj)
        const char* mp = (const char*)(M + ((2 * ca + cb) * w + pi) * w + pj);
        const double dy0 = (double)oy - yt;
        double m[U][NB];   // the next step's node masses, on their way
        auto load = [&]() {
#pragma unroll
            for (int u = 0; u < U; ++u) {
#pragma unroll
                for (int b = 0; b < NB; ++b) m[u][b] = *(const double*)(mp + pos[b]);
                mp += plane * sizeof(double);
            }
        };
        auto products = [&](const double (&mc)[U][NB], const double (&kx)[U],
                            const double (&ky)[U]) {
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    ax[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(kx[u], mc[u][b], ax[b], 0, 0, 0);
                    ay[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(ky[u], mc[u][b], ay[b], 0, 0, 0);
                }
        };
        load();
        double mc[U][NB], kx[U], ky[U];
        if (P % 4 == 0) {   // a lane's quarter is whole columns of nodes
#pragma unroll 1
            for (int k = 0; k < QP; ++k) {
                const double dx = ((double)ox - xt) + hn[g * QP + k];
                const double dx2 = fma(dx, dx, e2);
#pragma unroll 1
                for (int j = 0; j < P; j += U) {
#pragma unroll
                    for (int u = 0; u < U; ++u) {
#pragma unroll
                        for (int b = 0; b < NB; ++b) mc[u][b] = m[u][b];
                        const double dy = hn[j + u] + dy0;
                        const double r = rcp64(fma(dy, dy, dx2));
                        kx[u] = dx * r;
                        ky[u] = dy * r;
                    }
                    if (k < QP - 1 || j + U < P) load();
                    products(mc, kx, ky);
                }
            }
        } else {
            int i = g * (Q / 4) / P, j = g * (Q / 4) % P;
#pragma unroll 1
            for (int k = 0; k < Q / 4; ++k) {
                const double dx = ((double)ox - xt) + hn[i], dy = hn[j] + dy0;
                const double r = rcp64(fma(dy, dy, fma(dx, dx, e2)));
#pragma unroll
                for (int b = 0; b < NB; ++b) mc[0][b] = m[0][b];
                kx[0] = dx * r;
                ky[0] = dy * r;
                j = j + 1 < P ? j + 1 : 0;
                i += j == 0;
                if (k + 1 < Q / 4) load();
                products(mc, kx, ky);
            }
        }
    }
    const double inv_h = 1.0 / h;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        if (tg[b] < 0) continue;
        double* L = (FAR ? A.locf : A.loc) + (int64_t)tg[b] * (2 * Q) + 16 * rb;
#pragma unroll
        for (int v = 0; v < 4; ++v) {   // register v of lane (c, g): row 4 v + g, column c
            if (Q % 16 && 16 * rb + 4 * v + g >= Q) continue;
            L[4 * v + g] = ax[b][v] * inv_h;
            L[Q + 4 * v + g] = ay[b][v] * inv_h;
        }
    }
}

// Blocks of 16 target nodes of a square with P^2.
__host__ __device__ constexpr int m2l_rows(int P) { return (P * P + 15) / 16; }

template <int P, bool FAR>
__device__ __forceinline__ void m2l_group(const FmmArgs& A, int64_t blk, const double* __restrict__ nodes, double eps2,
                                          double* hn)
{
    constexpr int RB = m2l_rows(P);
    if (threadIdx.x < P) hn[threadIdx.x] = 0.5 * nodes[threadIdx.x];
    __syncthreads();
    const int gi = (int)(blk / RB), rb = (int)(blk - (int64_t)gi * RB);
    const FmmGroup gr = A.groups[gi];
    const int cnt = gr.cnt;
    if (cnt > 32) m2l_wave<P, 4, FAR>(A, gr, rb, eps2, hn);
    else if (cnt > 16) m2l_wave<P, 2, FAR>(A, gr, rb, eps2, hn);
    else m2l_wave<P, 1, FAR>(A, gr, rb, eps2, hn);
}

// The longer waves, those of the near offsets, come first.
template <int P>
__global__ __launch_bounds__(64, 3) void k_fmm_m2l(FmmArgs A, int ngroups,
                                                   const double* __restrict__ nodes,
                                                   const double* __restrict__ fnodes, double eps2)
{
    constexpr int F = fmm_far(P);
    __shared__ double hn[P];   // nodes on [-1/2, 1/2]
    const int64_t near = (int64_t)ngroups * m2l_rows(P);
    if (blockIdx.x < near) m2l_group<P, false>(A, blockIdx.x, nodes, eps2, hn);
    else m2l_group<F, true>(A, blockIdx.x - near, fnodes, eps2, hn);
}

// ---------------------------------------------------------------- field down
// One block per square of level lev: adds the far offsets' field, from the coarser
// nodes, and the parent's, interpolated at the square's nodes; on tiles (lev 0)
// the sum becomes Chebyshev coefficients.
template <int P>
__global__ __launch_bounds__(FMM_THREADS) void k_fmm_l2l(FmmArgs A,
                                                         const double* __restrict__ shift,
                                                         const double* __restrict__ ctab,
                                                         const double* __restrict__ ftab, int lev)
{
    constexpr int Q = P * P, F = fmm_far(P), QF = F * F, NB = piece<P>();
    constexpr int PM = P / 2, PN = P / NB;
    static_assert(2 * PM * PN <= FMM_THREADS && F * P <= Q, "a piece per thread; room in S");
    __shared__ alignas(16) double S[2 * Q], C[2 * Q], V[2 * Q];
    const int tid = threadIdx.x;
    const int64_t t = A.lev_off[lev] + blockIdx.x;
    if (A.tcnt[t] == 0) return;
    const FmmTile tl = A.tiles[t];
    const FmmSys& fs = A.fsys[tl.sys];
    if (fs.nlev <= lev) return;
    const bool par = lev + 1 < fs.nlev;
    double* L = A.loc + t * (int64_t)(2 * Q);
    // this thread's piece of the field
    const int z = tid / (PM * PN), r = tid - z * (PM * PN);
    const int at = z * Q + 2 * (r / PN) * P + NB * (r % PN);
    double acc[2][NB];
    auto add = [&](int, int, int, const auto& c) {
#pragma unroll
        for (int w = 0; w < 2; ++w)
#pragma unroll
            for (int v = 0; v < NB; ++v) acc[w][v] += c[w][v];
    };
    auto in_V = [&](int f, int m, int n, const auto& c) { put_lds<P>(V + f * Q, m, n, c); };
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
        for (int v = 0; v < NB; ++v) acc[w][v] = z < 2 ? L[at + w * P + v] : 0.0;
    load_table<F, P>(ftab, S, S + Q);
    for (int q = tid; q < 2 * QF; q += FMM_THREADS) C[q] = A.locf[t * (2 * QF) + q];
    __syncthreads();
    // V[i][J] = sum_I fine[I][i] C[I][J], then over J
    products<P, F, F, 2>(S + Q, 0, C, QF, [&](int f, int m, int n, const auto& c) {
        put_lds<F>(V + f * P * F, m, n, c);
    });
    __syncthreads();
    products<P, P, F, 2>(V, P * F, S, 0, add);
    __syncthreads();
    if (par) {
        const int64_t pt = fs.off[lev + 1] + (int64_t)(tl.tx >> 1) * fs.n[lev + 1] + (tl.ty >> 1);
        load_table<P, P>(shift + (tl.tx & 1) * Q, nullptr, S);
        load_table<P, P>(shift + (tl.ty & 1) * Q, S + Q, nullptr);
        for (int q = tid; q < 2 * Q; q += FMM_THREADS) C[q] = A.loc[pt * (2 * Q) + q];
        __syncthreads();
        products<P, P, P, 2>(S, 0, C, Q, in_V);   // V[I][j] = sum_i shift_a[i][I] C[i][j]
        __syncthreads();
        products<P, P, P, 2>(V, Q, S + Q, 0, add);
        __syncthreads();
    }
    if (lev == 0) {
        if (z < 2)
#pragma unroll
            for (int w = 0; w < 2; ++w)
#pragma unroll
                for (int v = 0; v < NB; ++v) {
                    C[at + w * P + v] = acc[w][v];
                    acc[w][v] = 0.0;
                }
        load_table<P, P>(ctab, S, S + Q);
        __syncthreads();
        products<P, P, P, 2>(S, 0, C, Q, in_V);   // V[k][J] = sum_I ct[k][I] C[I][J]
        __syncthreads();
        products<P, P, P, 2>(V, Q, S + Q, 0, add);
    }
    if (z < 2)
#pragma unroll
        for (int w = 0; w < 2; ++w)
#pragma unroll
            for (int v = 0; v < NB; ++v) L[at + w * P + v] = acc[w][v];
}

// ---------------------------------------------------------------- particles
__global__ __launch_bounds__(256) void k_fmm_pack(FmmArgs A)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < A.N; i += stride) {
        const double sig = step_scale(A.sys[A.sys_of[i]].step);
        FmmPart p;
        p.x = A.x[i] * sig;
        p.y = A.y[i] * sig;
        p.m = A.m[i];
        p.pad = 0.0;
        A.pack[i] = p;
    }
}

// Quads of a cell's particles from j on, `step` apart, before b, as near
// candidates of the whole wave, by scalar loads.  Only quads that hold some of the
// wave's own particles (g0 to g1) are tested for the particle itself: with every
// quad of the lanes' own cells tested, 10M particles in cells of 700 took 23.7 ms
// instead of 22.8, 1M in cells of 100 under a cutoff 0.98 instead of 0.86.  (In
// k_force64s, which loads ahead, the branch costs 5 to 8 % on clusters.)
// (Loading a quad ahead, as k_force64s does, is 5 % slower here: the second set of
// registers spills scalars that the outer loops hold.)
template <int LAW, bool SQ>
__device__ __forceinline__ void near_cell(const FmmPart* pack, int j, int b, int g0, int g1, int gi,
                                          double x, double y, double eps2, double r2cut, int step,
                                          double& sx, double& sy, double& s2)
{
    const cptr<FmmPart> E = as_const(pack);
    for (; j + 3 < b; j += step) {
        const fd8 p = *(cptr<fd8>)(E + j), q = *(cptr<fd8>)(E + j + 2);
        const double wx[4] = {p[0] - x, p[4] - x, q[0] - x, q[4] - x};
        const double wy[4] = {p[1] - y, p[5] - y, q[1] - y, q[5] - y};
        const double m[4] = {p[2], p[6], q[2], q[6]};
        if (j + 3 < g0 || j > g1)
            quad_terms<LAW, false, SQ>(wx, wy, m, {true, true, true, true}, eps2, r2cut, sx, sy, &s2);
        else
            quad_terms<LAW, true, SQ>(wx, wy, m, {j != gi, j + 1 != gi, j + 2 != gi, j + 3 != gi},
                                  eps2, r2cut, sx, sy, &s2);
    }
    if (j + 1 < b) {
        const fd8 p = *(cptr<fd8>)(E + j);
        pair_terms<LAW, true, SQ>(p[0] - x, p[1] - y, p[2], p[4] - x, p[5] - y, p[6], j != gi,
                              j + 1 != gi, eps2, r2cut, sx, sy, &s2);
        j += 2;
    }
    if (j < b)   // the last of an odd count, with a copy of itself without mass
        pair_terms<LAW, true, SQ>(E[j].x - x, E[j].y - y, E[j].m, E[j].x - x, E[j].y - y, 0.0, j != gi,
                              j != gi, eps2, r2cut, sx, sy, &s2);
}

// A lane's own near candidates in column xc (OWN: its own column, which holds
// the particle itself), every W-th pair from the w-th on.  gi < 0: no particle.
template <int LAW, bool OWN, bool SQ>
__device__ __forceinline__ void near_range(const FmmArgs& A, int64_t coff, int G, int xc, int cy,
                                           int gi, int w, int W, double x, double y, double eps2,
                                           double r2cut, double& sx, double& sy, double& s2)
{
    if (gi < 0 || xc < 0 || xc >= G) return;
    const int64_t cl = coff + (int64_t)xc * G;
    int j = A.offsets[cl + max(cy - 1, 0)] + 2 * w;
    const int b = A.offsets[cl + min(cy + 1, G - 1) + 1];
    const FmmPart* E = A.pack + j;
    for (; j < b; j += 2 * W, E += 2 * W) {
        const bool two = j + 1 < b;
        const FmmPart* E1 = two ? E + 1 : E;
        const double m1 = two ? E1->m : 0.0;
        pair_terms<LAW, OWN, SQ>(E->x - x, E->y - y, E->m, E1->x - x, E1->y - y, m1, j != gi,
                             (two ? j + 1 : j) != gi, eps2, r2cut, sx, sy, &s2);
    }
}

// The terms of chunk ci's particles that fall to wave w of the W that share it
// (a power of two): gi is the lane's particle (-1: none), (rx, ry) its sum.  The
// tile's coefficients and the mid entries are the same for every lane: scalar
// loads of whole quads (128 bytes), no test per lane in quads that no lane's 3x3
// cells touch (a test and its selects double a quad's instructions).  Near
// candidates: if the chunk lies in one column and spans at most
// FMM_UNIFORM_ROWS rows, the union of its lanes' ranges is walked with scalar
// loads and a row test; otherwise each lane walks its own three ranges with
// vector loads (a union would spend most of its terms on the test).  Terms go in
// quads, or a lane's own in pairs, that share a reciprocal; only quads that hold
// the lanes themselves are tested for the particle itself.  SQ: r2 is the sum of
// the near terms' (m / r)^2, r in cell sides, for the FP64 recompute's bound: 2 to 3
// % (4.2M FP32 particles over 1024^2 cells 2.14 -> 2.20 ms, 512 systems 7.14 -> 7.27).
template <int P, int LAW, bool SQ>
__device__ __forceinline__ void chunk_terms(const FmmArgs& A, int ci, int w, int W, double eps2p,
                                            double r2cutp, int& gi, double& rx, double& ry,
                                            double& r2)
{
    constexpr int Q = P * P;
    const int lane = threadIdx.x & 63;
    const FmmChunk ch = A.chunks[ci];
    const int t = uniform_int(ch.tile);
    const FmmTile tl = A.tiles[t];
    const int s = uniform_int(tl.sys);
    const int ttx = uniform_int(tl.tx), tty = uniform_int(tl.ty);
    const SysDev& d = A.sys[s];
    const FmmSys& fs = A.fsys[s];
    const int G = d.G, T = fs.T;
    const int64_t coff = d.c_off;
    const double step = d.step, sig = step_scale(step);
    const double eps2 = eps2p * sig * sig, r2cut = r2cutp * sig * sig;
    const double h = (double)T * step;
    const int x0 = ttx * T, y0 = tty * T, x1 = min(x0 + T, G), y1 = min(y0 + T, G);

    // lane -> particle: rank 64 k + lane in the tile, columns in order
    int r = 64 * uniform_int(ch.k) + lane;
    gi = -1;
    for (int x = x0; x < x1; ++x) {
        const int64_t cl = coff + (int64_t)x * G;
        const int a = A.offsets[cl + y0], b = A.offsets[cl + y1];
        if (gi < 0 && r < b - a) gi = a + r;
        r -= b - a;
    }
    const bool act = gi >= 0;
    double x = 0.0, y = 0.0, sx = 0.0, sy = 0.0, s2 = 0.0, fx = 0.0, fy = 0.0;
    int cx = -100000, cy = -100000;
    if (act) {
        const FmmPart p = A.pack[gi];
        x = p.x;
        y = p.y;
        const int key = A.key_sorted[gi] - (int)coff;
        cx = key / G;
        cy = key - cx * G;
    }
    const int cxl = uniform_int(wave_min(act ? cx : 0x7fffffff));
    const int cxh = uniform_int(wave_max(act ? cx : -1));
    const int cyl = uniform_int(wave_min(act ? cy : 0x7fffffff));
    const int cyh = uniform_int(wave_max(act ? cy : -1));

    // the particle on its tile, [-1, 1]^2
    const double ux = 2.0 * ((x / sig - d.min_x) / h - ttx) - 1.0;
    const double uy = 2.0 * ((y / sig - d.min_y) / h - tty) - 1.0;

    // near pairs
    if (cxl == cxh && cyh - cyl < FMM_UNIFORM_ROWS) {
        const int g0 = uniform_int(wave_min(act ? gi : 0x7fffffff));
        const int g1 = uniform_int(wave_max(gi));
        int turn = 0;   // quads so far, dealt to the waves in turn
        for (int dx = -1; dx <= 1; ++dx) {
            const int xc = cxl + dx;
            if (xc < 0 || xc >= G) continue;
            const int64_t cl = coff + (int64_t)xc * G;
            for (int row = max(cyl - 1, 0); row <= min(cyh + 1, G - 1); ++row) {
                const int a = uniform_int(A.offsets[cl + row]);
                const int b = uniform_int(A.offsets[cl + row + 1]);
                const int j = a + 4 * ((w - turn) & (W - 1));
                turn += (b - a + 3) >> 2;
                if (!(act && abs(row - cy) <= 1)) continue;
                near_cell<LAW, SQ>(A.pack, j, b, g0, g1, gi, x, y, eps2, r2cut, 4 * W, sx, sy,
                                   s2);
            }
        }
    } else {
        near_range<LAW, false, SQ>(A, coff, G, cx - 1, cy, gi, w, W, x, y, eps2, r2cut, sx, sy, s2);
        near_range<LAW, true, SQ>(A, coff, G, cx, cy, gi, w, W, x, y, eps2, r2cut, sx, sy, s2);
        near_range<LAW, false, SQ>(A, coff, G, cx + 1, cy, gi, w, W, x, y, eps2, r2cut, sx, sy, s2);
    }

    // mid entries: 3x3 tiles, or every tile where the grouped part does not
    // hold: a system of one tile, a cutoff that reaches past a tile, COMs
    // outside their tiles, particles that left theirs since they were placed
    const bool in = !act || (fabs(ux) <= FMM_IN && fabs(uy) <= FMM_IN);
    // (0.9995: FMM_IN lets either end be 5e-5 of a tile nearer)
    const bool all = fs.nlev == 0 || (LAW == 1 && !(r2cutp < 0.9995 * h * h)) ||
                     uniform_int(A.sbad[s]) != 0 || __ballot(!in) != 0ull;
    const bool plain = placed_apart<LAW>(d, r2cut, act, (0.5 * (ux + 1.0) + ttx) * T - cx,
                                         (0.5 * (uy + 1.0) + tty) * T - cy);
    const int nt = fs.n[0];
    const int mx0 = all ? 0 : max(ttx - 1, 0), mx1 = all ? nt - 1 : min(ttx + 1, nt - 1);
    const int my0 = all ? 0 : max(tty - 1, 0), my1 = all ? nt - 1 : min(tty + 1, nt - 1);
    for (int mx = mx0; mx <= mx1; ++mx) {
        for (int my = my0; my <= my1; ++my) {
            const int mt = fs.off[0] + mx * nt + my;
            const int e0 = uniform_int(A.tstart[mt]), ne = uniform_int(A.tne[mt]);
            const cptr<fd8> E = (cptr<fd8>)(as_const(A.list) + e0);
            // a tile that some lane's 3x3 cells may touch: each entry is tested
            const bool touch = mx * T <= cxh + 1 && mx * T + T > cxl - 1 &&
                               my * T <= cyh + 1 && my * T + T > cyl - 1;
            if (!touch && plain) {
                for (int e = 4 * w; e < ne; e += 4 * W) {
                    const fd8 p = E[e >> 1], q = E[(e >> 1) + 1];
                    quad_terms<0, false>({p[0] - x, p[4] - x, q[0] - x, q[4] - x},
                                         {p[1] - y, p[5] - y, q[1] - y, q[5] - y},
                                         {p[2], p[6], q[2], q[6]}, {true, true, true, true}, eps2,
                                         r2cut, sx, sy);
                }
            } else {
                auto far = [&](double kxy) {
                    const long long c = __double_as_longlong(kxy);
                    return (unsigned)((int)c - cx + 1) > 2u ||
                           (unsigned)((int)(c >> 32) - cy + 1) > 2u;
                };
                for (int e = 4 * w; e < ne; e += 4 * W) {
                    const fd8 p = E[e >> 1], q = E[(e >> 1) + 1];
                    // the quad's cells, in column order: does one of them lie
                    // in some lane's 3x3?
                    const long long c0 = __double_as_longlong(p[3]);
                    const long long c3 = __double_as_longlong(q[7]);
                    const int kx0 = (int)c0, kx3 = (int)c3, ky0 = (int)(c0 >> 32),
                              ky3 = (int)(c3 >> 32);
                    const bool meet = kx3 >= cxl - 1 && kx0 <= cxh + 1 &&
                                      (kx0 != kx3 || (ky3 >= cyl - 1 && ky0 <= cyh + 1));
                    const double wx[4] = {p[0] - x, p[4] - x, q[0] - x, q[4] - x};
                    const double wy[4] = {p[1] - y, p[5] - y, q[1] - y, q[5] - y};
                    const double m[4] = {p[2], p[6], q[2], q[6]};
                    if (plain && !meet)
                        quad_terms<0, false>(wx, wy, m, {true, true, true, true}, eps2, r2cut, sx,
                                             sy);
                    else if (LAW == 1 && !meet)   // a wide cutoff: one test a quad
                        quad_terms<LAW, false>(wx, wy, m, {true, true, true, true}, eps2, r2cut,
                                               sx, sy);
                    else
                        quad_terms<LAW, true>(wx, wy, m,
                                              {far(p[3]), far(p[7]), far(q[3]), far(q[7])}, eps2,
                                              r2cut, sx, sy);
                }
            }
        }
    }

    // terms one by one (see one_term), by all waves of the chunk (SQ: the
    // recompute takes particles whose sums are not finite)
    const bool bad = !SQ && !is_finite(sx, sy);
    if (!SQ && (W > 1 ? (bool)__syncthreads_or(bad) : __any(bad))) {
        sx = sy = 0.0;
        for (int xc = max(cx - 1, 0); act && xc <= min(cx + 1, G - 1); ++xc) {
            const int64_t cl = coff + (int64_t)xc * G;
            const int b = A.offsets[cl + min(cy + 1, G - 1) + 1];
#pragma unroll 1
            for (int j = A.offsets[cl + max(cy - 1, 0)] + w; j < b; j += W) {
                const FmmPart q = A.pack[j];
                one_term<LAW>(q.x - x, q.y - y, q.m, j != gi, eps2, r2cut, sx, sy);
            }
        }
        for (int mx = mx0; mx <= mx1; ++mx) {
            for (int my = my0; my <= my1; ++my) {
                const int mt = fs.off[0] + mx * nt + my;
                const int e0 = A.tstart[mt], ne = A.tne[mt];
#pragma unroll 1
                for (int e = e0 + w; e < e0 + ne; e += W) {
                    const FmmCom f = A.list[e];
                    one_term<LAW>(f.X - x, f.Y - y, f.M, abs(f.kx - cx) > 1 || abs(f.ky - cy) > 1,
                                  eps2, r2cut, sx, sy);
                }
            }
        }
    }

    // distant part: the tile's Chebyshev series
    if (!all && act) {
        double ty[P];
        ty[0] = 1.0;
        ty[1] = uy;
#pragma unroll
        for (int l = 2; l < P; ++l) ty[l] = fma(2.0 * uy, ty[l - 1], -ty[l - 2]);
        cptr<double> L = as_const(A.loc) + (int64_t)t * (2 * Q);
        double a0 = 1.0, a1 = ux;
        for (int k = 0; k < P; ++k) {
            if ((k & (W - 1)) == w) {
                double vx = 0.0, vy = 0.0;
#pragma unroll
                for (int l = 0; l < P; ++l) {
                    vx = fma(L[k * P + l], ty[l], vx);
                    vy = fma(L[Q + k * P + l], ty[l], vy);
                }
                fx = fma(a0, vx, fx);
                fy = fma(a0, vy, fy);
            }
            const double an = fma(2.0 * ux, a1, -a0);
            a0 = a1;
            a1 = an;
        }
    }
    rx = fma(sx, sig, fx);
    ry = fma(sy, sig, fy);
    if (SQ) r2 = s2 * ((step * sig) * (step * sig));
}

// A particle's sums as the pass leaves them: added to its acceleration, or (SQ)
// in the recompute's planes, which add them or the FP64 terms in their place.
template <bool SQ>
__device__ __forceinline__ void put_sum(double* a, int gi, double v)
{
    if (SQ) a[gi] = v;
    else a[gi] += v;
}

// Chunks of dense tiles, each shared by the eight waves of a block: a particle
// of a cluster's core may have 10^4 near candidates where the others have a
// hundred, and on a wave of its own such a chunk would outlast the rest of the
// pass.  1M particles, 400^2 cells, cores of 10^3 a cell: 10.7 -> 7.9 ms.
template <int P, int LAW, bool SQ>
__global__ __launch_bounds__(64 * FMM_WAVES) void k_fmm_dense(FmmArgs A, double Gc, double eps2,
                                                              double r2cut, int qpart, int nqparts)
{
    __shared__ double part[SQ ? 3 : 2][FMM_WAVES][BH_WAVE];
    __shared__ int unit;
    const int lane = threadIdx.x & 63, w = uniform_int(threadIdx.x >> 6);
    const int64_t n = A.cnt[FMM_HEAVY];
    const int q0 = (int)(n * qpart / nqparts), q1 = (int)(n * (qpart + 1) / nqparts);
    if (q0 >= q1) return;
    for (;;) {
        if (threadIdx.x == 0) unit = q0 + atomicAdd(&A.cnt[FMM_QHEAVY], 1);
        __syncthreads();
        const int ci = uniform_int(unit);
        if (ci >= q1) break;
        int gi;
        double rx, ry, r2;
        chunk_terms<P, LAW, SQ>(A, ci, w, FMM_WAVES, eps2, r2cut, gi, rx, ry, r2);
        part[0][w][lane] = rx;
        part[1][w][lane] = ry;
        if (SQ) part[SQ ? 2 : 0][w][lane] = r2;
        __syncthreads();
        if (w < (SQ ? 3 : 2) && gi >= 0) {   // wave 0 adds x, wave 1 y, wave 2 the near squares
            double t = 0.0;
#pragma unroll
            for (int v = 0; v < FMM_WAVES; ++v) t += part[w][v][lane];
            if (SQ && w == 2) A.s2n[gi] = t;
            else put_sum<SQ>(w ? A.ay : A.ax, gi, Gc * t);
        }
    }
}

// The other chunks, a wave each.  The chunks are left to the hardware's
// dispatch: a queue cursor (one atomic on the same word every ~15 ns) took 4.2M
// particles from 2.2 to 3.5 ms, a fixed deal 512 systems from 10.0 to 12.4 ms.
// Bound by FP64 issue (the vector units are busy 91 % of the time on 4.2M
// clustered particles over 1024^2 cells): with tiles of 8 cells 2.02 ms there, 8.8
// ms on 512 systems (7.1 with tiles of 6); 2.16 and 9.9 ms with terms in pairs
// and every entry of a tile that the 3x3 cells touch tested, 2.8 and 12.8 ms with
// entries loaded one by one.
template <int P, int LAW, bool SQ>
__global__ __launch_bounds__(64) void k_fmm_force(FmmArgs A, double Gc, double eps2, double r2cut,
                                                  int qpart, int nqparts)
{
    const int64_t n = A.cnt[FMM_LIGHT];
    const int q0 = (int)(n * qpart / nqparts), q1 = (int)(n * (qpart + 1) / nqparts);
    for (int u = q0 + blockIdx.x; u < q1; u += gridDim.x) {
        int gi;
        double rx, ry, r2;
        chunk_terms<P, LAW, SQ>(A, (int)(A.max_chunks - 1 - u), 0, 1, eps2, r2cut, gi, rx, ry, r2);
        if (gi >= 0) {
            put_sum<SQ>(A.ax, gi, Gc * rx);
            put_sum<SQ>(A.ay, gi, Gc * ry);
            if (SQ) A.s2n[gi] = r2;
        }
    }
}

// ---------------------------------------------------------------- launches
template <int P>
static void fmm_prepare(const FmmArgs& A, const FmmPlan& pl, double eps2, int num_cu,
                        hipStream_t st)
{
    const FmmTables& tb = pl.tab;
    hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(64), 0, st, A.cnt,
                       (int64_t)(FMM_NCNT + A.S), 0);
    hipLaunchKernelGGL(k_fmm_tiles, dim3((unsigned)((A.nleaf * 8 + 255) / 256)), dim3(256), 0, st,
                       A);
    const unsigned pg = (unsigned)((A.N + 255) / 256);
    hipLaunchKernelGGL(k_fmm_pack, dim3(pg < (unsigned)num_cu * 16 ? pg : num_cu * 16), dim3(256),
                       0, st, A);
    hipLaunchKernelGGL(k_fmm_p2m<P>, dim3((unsigned)A.nleaf), dim3(FMM_THREADS), 0, st, A, tb.cheb,
                       tb.fine);
    for (int l = 1; l < pl.nlev; ++l)
        hipLaunchKernelGGL(k_fmm_m2m<P>, dim3((unsigned)(A.lev_off[l + 1] - A.lev_off[l])),
                           dim3(256), 0, st, A, tb.shift, tb.fine, l);
    constexpr int F = fmm_far(P);
    hipLaunchKernelGGL(k_fmm_m2l<P>, dim3((unsigned)pl.ngroups * (m2l_rows(P) + m2l_rows(F))),
                       dim3(64), 0, st, A, (int)pl.ngroups, tb.nodes, tb.fnodes, eps2);
    for (int l = pl.nlev - 1; l >= 0; --l)
        hipLaunchKernelGGL(k_fmm_l2l<P>, dim3((unsigned)(A.lev_off[l + 1] - A.lev_off[l])),
                           dim3(FMM_THREADS), 0, st, A, tb.shift, tb.cheb, tb.fine, l);
}

template <int P, int LAW, bool SQ>
static void fmm_force(const FmmArgs& A, double Gc, double eps2, double r2cut, int part, int nparts,
                      int num_cu, hipStream_t st)
{
    if (part > 0)   // the queue of this launch
        hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(64), 0, st, A.cnt + FMM_QHEAVY, (int64_t)1, 0);
    const int64_t cap = A.max_chunks, most = (int64_t)num_cu * 256;
    hipLaunchKernelGGL((k_fmm_dense<P, LAW, SQ>), dim3(num_cu * 4), dim3(64 * FMM_WAVES), 0, st, A,
                       Gc, eps2, r2cut, part, nparts);
    hipLaunchKernelGGL((k_fmm_force<P, LAW, SQ>), dim3((unsigned)(cap < most ? cap : most)),
                       dim3(64), 0, st, A, Gc, eps2, r2cut, part, nparts);
}

void bh_fmm_pass(const FmmArgs& A, const FmmPlan& pl, bool fp64, double Gc, double eps2,
                 double r2cut, int part, int nparts, int num_cu, hipStream_t st)
{
    if (part == 0) {
        if (fp64) fmm_prepare<FMM_P64>(A, pl, eps2, num_cu, st);
        else fmm_prepare<FMM_P32>(A, pl, eps2, num_cu, st);
    }
    const bool law = r2cut > 0.0, sq = A.s2n != nullptr;
    const auto force = fp64 ? (law ? fmm_force<FMM_P64, 1, false> : fmm_force<FMM_P64, 0, false>)
                     : sq   ? (law ? fmm_force<FMM_P32, 1, true> : fmm_force<FMM_P32, 0, true>)
                            : (law ? fmm_force<FMM_P32, 1, false> : fmm_force<FMM_P32, 0, false>);
    force(A, Gc, eps2, r2cut, part, nparts, num_cu, st);
}
