// Cloud-to-cloud direct gravity: the reference's gravity plugin
//   fn(self_cloud, other_cloud, G, update_other)
// (python-bh/barneshut/kernels/gravity/cpu_numba.py:8-92, selected by
// gravity/__init__.py:6-41 and called from internals/cloud.py:113-114).
//
// A cloud is n rows of ld doubles in the reference's particle row layout
// (px, py, mass, vx, vy, ax, ay, ...; internals/particle.py:3-15), in device
// memory.  For every target row i the kernel adds
//     G * sum_j m_j (x_j - x_i) w(|x_j - x_i|^2)
// over the source rows j (j != i when targets and sources are one cloud) to
// the row's ax, ay, with the law's w (bh_law: cutoff r2_cut > 0 drops pairs
// with r^2 <= r2_cut, as the reference's CPU kernel does at 1e-5).
//
// One 256-thread block owns P * G' consecutive targets (G' = 256 / L groups of
// L lanes, P = 1 or 2 targets per lane).  Sources are staged through LDS in tiles of
// 256 rows; lane l of a group takes the tile rows l, l + L, l + 2L, ... for
// its P targets (with one group per block, L = 256, the lanes read their rows
// straight from memory instead), and the L partial sums of a target are added
// by a fixed tree.  The shape (P, L) is a function of the two cloud sizes only, so a
// result never depends on timing.  FP64 throughout; each weight m / q by the
// refined hardware reciprocal (wdiv64, within about one ulp of the quotient), or
// in large clouds two weights by one (cloud_pair).  Bound by FP64 issue: 2.0e12
// terms/s on 100,003 rows (5.1 ms; 5.9 with a reciprocal per term), ~15 slots a
// term.  Tried and slower: rows by scalar loads (80-byte strides miss the scalar
// cache: 7.7 ms), four targets per lane (169 registers: 5.8 ms).

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>

#include "bh_common.h"
#include "bh_kernels.h"
#include "../../include/bh_hip.h"

int bh_ctx_fail(int code, const char* msg);

#define CL_THREADS 256
#define CL_MIN_BLOCKS 2048   // blocks a launch aims for before lanes are widened
#define CL_PAIRS 6000        // rows on both sides from which sources go in pairs
#define CL_HUGE 81920        // targets from which pairs take the full CL_MIN_BLOCKS
#define CL_MIN_PER_LANE 8    // fewest source rows a lane is given when widening

namespace {

// Reference row columns (internals/particle.py:3-15).
constexpr int COL_X = 0, COL_Y = 1, COL_M = 2, COL_AX = 5, COL_AY = 6;

struct CloudArgs {
    const double* src;   // source rows (px, py, mass read)
    int64_t ns, lds;
    double* tgt;         // target rows (px, py read; ax, ay added to)
    int64_t nt, ldt;
    int32_t mask_self;   // 1: row i of the sources is target i, skip it by index
    int32_t llog2;       // log2 of the lanes per target
    double G, eps2, r2cut;
};

// m w(r^2) of the law: LAW 1 drops r^2 <= r2cut; SOFT 0 has eps2 = 0 (the
// reference laws), so r^2 + eps2 is not formed.
template <int LAW, int SOFT>
__device__ __forceinline__ double cloud_w(double wx, double wy, double m, double eps2,
                                          double r2cut)
{
    const double s2 = fma(wx, wx, wy * wy);
    const double w = wdiv64(m, SOFT ? s2 + eps2 : s2);
    return LAW ? ((s2 > r2cut) ? w : 0.0) : w;
}

// One source row for P targets, by itself: the exact form.
template <int LAW, int SOFT, int P, int MASK>
__device__ __forceinline__ void cloud_one(double x, double y, double m, int64_t j,
                                          const int64_t* ti, const double* xi, const double* yi,
                                          double* ax, double* ay, double eps2, double r2cut)
{
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const double wx = x - xi[p], wy = y - yi[p];
        double w = cloud_w<LAW, SOFT>(wx, wy, m, eps2, r2cut);
        if (MASK) w = (j == ti[p]) ? 0.0 : w;
        ax[p] = fma(wx, w, ax[p]);
        ay[p] = fma(wy, w, ay[p]);
    }
}

// Two source rows for P targets.  Their weights come from one reciprocal, of
// Q = q0 q1 (see pair_terms), where no lane of the wave drops either row and Q
// is well inside the range of a double; else each row by itself.  12.5 issue
// slots a term instead of 18 with a reciprocal, a compare and a select each.
template <int LAW, int SOFT, int P>
__device__ __forceinline__ void cloud_pair(double x0, double y0, double m0, double x1, double y1,
                                           double m1, const double* xi, const double* yi,
                                           double* ax, double* ay, double eps2, double r2cut)
{
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const double wx0 = x0 - xi[p], wy0 = y0 - yi[p];
        const double wx1 = x1 - xi[p], wy1 = y1 - yi[p];
        const double s0 = fma(wx0, wx0, wy0 * wy0), s1 = fma(wx1, wx1, wy1 * wy1);
        const double q0 = SOFT ? s0 + eps2 : s0, q1 = SOFT ? s1 + eps2 : s1;
        const double Q = q0 * q1;
        double w0, w1;
        // under a cutoff of 1e-140 and more the products of kept rows are fine
        const bool plain = LAW ? fmin(s0, s1) > fmax(r2cut, 1e-140) : Q > 1e-290;
        if (!__any(!plain)) {
            const double R = rcp64(Q);
            w0 = (m0 * R) * q1;
            w1 = (m1 * R) * q0;
        } else {
            w0 = cloud_w<LAW, SOFT>(wx0, wy0, m0, eps2, r2cut);
            w1 = cloud_w<LAW, SOFT>(wx1, wy1, m1, eps2, r2cut);
        }
        ax[p] = fma(wx0, w0, ax[p]);
        ay[p] = fma(wy0, w0, ay[p]);
        ax[p] = fma(wx1, w1, ax[p]);
        ay[p] = fma(wy1, w1, ay[p]);
    }
}

// FAST: rows in pairs; otherwise, and under MASK, one by one.
template <int LAW, int SOFT, int P, int MASK, int FAST>
__device__ __forceinline__ void cloud_tile(const double* sx, const double* sy, const double* sm,
                                           int cnt, int lane, int L, int64_t t0,
                                           const int64_t* ti, const double* xi, const double* yi,
                                           double* ax, double* ay, double eps2, double r2cut)
{
    int k = lane;
    if (FAST && !MASK)
#pragma unroll 2
        for (; k + L < cnt; k += 2 * L)
            cloud_pair<LAW, SOFT, P>(sx[k], sy[k], sm[k], sx[k + L], sy[k + L], sm[k + L], xi, yi,
                                     ax, ay, eps2, r2cut);
    for (; k < cnt; k += L)
        cloud_one<LAW, SOFT, P, MASK>(sx[k], sy[k], sm[k], t0 + k, ti, xi, yi, ax, ay, eps2, r2cut);
}

// Source rows lane, lane + 256, ... read straight from memory (L = 256), one by
// one: the loads bound this loop, and a branch per pair keeps them from being
// issued ahead (64 rows against 200,000: 127 us, in pairs 173).
template <int LAW, int SOFT, int P, int MASK>
__device__ __forceinline__ void cloud_direct(const CloudArgs& A, int lane, const int64_t* ti,
                                             const double* xi, const double* yi, double* ax,
                                             double* ay)
{
#pragma unroll 4
    for (int64_t j = lane; j < A.ns; j += CL_THREADS) {
        const double* r = A.src + j * A.lds;
        cloud_one<LAW, SOFT, P, MASK>(r[COL_X], r[COL_Y], r[COL_M], j, ti, xi, yi, ax, ay, A.eps2,
                                      A.r2cut);
    }
}

// All sources on the block's targets.
template <int LAW, int SOFT, int P, int FAST>
__device__ __forceinline__ void cloud_sum(const CloudArgs& A, double* buf, int64_t base, int lane,
                                          const int64_t* ti, const double* xi, const double* yi,
                                          double* ax, double* ay)
{
    double *sx = buf, *sy = buf + CL_THREADS, *sm = buf + 2 * CL_THREADS;
    const int tid = threadIdx.x, L = 1 << A.llog2, groups = CL_THREADS >> A.llog2;
#pragma unroll
    for (int p = 0; p < P; ++p) {
        ax[p] = 0.0;
        ay[p] = 0.0;
    }
    if (groups == 1) {
        // one target group per block: a tile would serve only its P targets,
        // so each lane reads its own source rows (unrolled, loads in flight)
        if (A.mask_self)
            cloud_direct<LAW, SOFT, P, 1>(A, lane, ti, xi, yi, ax, ay);
        else
            cloud_direct<LAW, SOFT, P, 0>(A, lane, ti, xi, yi, ax, ay);
        return;
    }
    for (int64_t t0 = 0; t0 < A.ns; t0 += CL_THREADS) {
        __syncthreads();   // every lane is done with the previous tile
        const int64_t j = t0 + tid;
        if (j < A.ns) {
            const double* r = A.src + j * A.lds;
            sx[tid] = r[COL_X];
            sy[tid] = r[COL_Y];
            sm[tid] = r[COL_M];
        }
        __syncthreads();
        const int cnt = (int)std::min<int64_t>(CL_THREADS, A.ns - t0);
        // the index test only where the tile holds the block's own rows
        if (A.mask_self && t0 < base + P * groups && t0 + CL_THREADS > base)
            cloud_tile<LAW, SOFT, P, 1, FAST>(sx, sy, sm, cnt, lane, L, t0, ti, xi, yi, ax, ay,
                                              A.eps2, A.r2cut);
        else if (FAST) {
            // a tile's sum first: fewer lanes per target make each lane's chain
            // longer, and in one chain its rounding grew with it (70,000 rows: 9e-16
            // of the sums, 4.5e-16 on twice the lanes, 1.8e-16 by tiles)
            double tx[P] = {}, ty[P] = {};
            cloud_tile<LAW, SOFT, P, 0, FAST>(sx, sy, sm, cnt, lane, L, t0, ti, xi, yi, tx, ty,
                                              A.eps2, A.r2cut);
#pragma unroll
            for (int p = 0; p < P; ++p) {
                ax[p] += tx[p];
                ay[p] += ty[p];
            }
        } else
            cloud_tile<LAW, SOFT, P, 0, FAST>(sx, sy, sm, cnt, lane, L, t0, ti, xi, yi, ax, ay,
                                              A.eps2, A.r2cut);
    }
}

// Block blk's targets.
template <int LAW, int SOFT, int P, int FAST>
__device__ __forceinline__ void cloud_block(const CloudArgs& A, int64_t blk)
{
    // tiles use 3 x 256 doubles, the final tree 2 P x 256
    __shared__ double buf[4 * CL_THREADS];
    const int tid = threadIdx.x;
    const int L = 1 << A.llog2;
    const int lane = tid & (L - 1);
    const int groups = CL_THREADS >> A.llog2;
    const int grp = tid >> A.llog2;
    const int64_t base = blk * (P * groups);

    int64_t ti[P];
    double xi[P], yi[P], ax[P], ay[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        ti[p] = base + (int64_t)p * groups + grp;
        const bool live = ti[p] < A.nt;
        xi[p] = live ? A.tgt[ti[p] * A.ldt + COL_X] : 0.0;
        yi[p] = live ? A.tgt[ti[p] * A.ldt + COL_Y] : 0.0;
    }
    cloud_sum<LAW, SOFT, P, FAST>(A, buf, base, lane, ti, xi, yi, ax, ay);
    if (FAST) {
        // a product Q beyond a double's range leaves a NaN: row by row then, which
        // also says what the sum is where it is not finite by itself
        int bad = 0;
#pragma unroll
        for (int p = 0; p < P; ++p) bad |= !(fabs(ax[p]) < 1e308 && fabs(ay[p]) < 1e308);
        if (__syncthreads_or(bad))
            cloud_sum<LAW, SOFT, P, 0>(A, buf, base, lane, ti, xi, yi, ax, ay);
    }

    __syncthreads();
#pragma unroll
    for (int p = 0; p < P; ++p) {
        buf[(2 * p) * CL_THREADS + tid] = ax[p];
        buf[(2 * p + 1) * CL_THREADS + tid] = ay[p];
    }
    __syncthreads();
    for (int s = L >> 1; s > 0; s >>= 1) {
        if (lane < s) {
#pragma unroll
            for (int q = 0; q < 2 * P; ++q)
                buf[q * CL_THREADS + tid] += buf[q * CL_THREADS + tid + s];
        }
        __syncthreads();
    }
    if (lane == 0) {
#pragma unroll
        for (int p = 0; p < P; ++p) {
            if (ti[p] < A.nt) {
                double* r = A.tgt + ti[p] * A.ldt;
                r[COL_AX] += A.G * buf[(2 * p) * CL_THREADS + tid];
                r[COL_AY] += A.G * buf[(2 * p + 1) * CL_THREADS + tid];
            }
        }
    }
}

template <int LAW, int SOFT, int P, int FAST>
__global__ __launch_bounds__(CL_THREADS, 6) void k_cloud(CloudArgs A)
{
    cloud_block<LAW, SOFT, P, FAST>(A, blockIdx.x);
}

// Both directions of a call: blocks [0, nblk0) run A0, the others A1.
template <int LAW, int SOFT, int P, int FAST>
__global__ __launch_bounds__(CL_THREADS) void k_cloud_both(CloudArgs A0, CloudArgs A1, int nblk0)
{
    if ((int)blockIdx.x < nblk0) cloud_block<LAW, SOFT, P, FAST>(A0, blockIdx.x);
    else cloud_block<LAW, SOFT, P, FAST>(A1, blockIdx.x - nblk0);
}

inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Shape of one launch from the two sizes: 2 targets per lane (one LDS read
// and the loop's bookkeeping serve both) once there are 2 per thread of a
// block, and more lanes per target while blocks are fewer than CL_MIN_BLOCKS
// and every lane keeps at least CL_MIN_PER_LANE source rows.  Large clouds take
// rows in pairs that share a reciprocal, and up to CL_HUGE targets half as many
// lanes (a cloud on itself, microseconds, rows one by one / in pairs / in pairs
// on half the lanes: 8,000 85 / 109 / 66, 16,000 227 / 218 / 184, 32,000 684 /
// 627 / 578, 64,000 2365 / 2106 / 2046, 100,003 5839 / 5015 / 5770, 131,072
// 9161 / 8016 / 8589); below, the shorter loop is the faster one.
void cloud_shape(int64_t nt, int64_t ns, int* P, int* llog2, int* pairs)
{
    *P = nt >= 2LL * CL_THREADS ? 2 : 1;
    *pairs = nt >= CL_PAIRS && ns >= CL_PAIRS;
    const int64_t want = *pairs && nt < CL_HUGE ? CL_MIN_BLOCKS / 2 : CL_MIN_BLOCKS;
    int l = 0;
    while (l < 8 && cdiv(nt, (int64_t)*P * (CL_THREADS >> l)) < want &&
           ((int64_t)CL_MIN_PER_LANE << (l + 1)) <= ns)
        ++l;
    *llog2 = l;
}

struct CloudJob {
    CloudArgs A;
    int P, pairs;
    int64_t blocks;
};

CloudJob cloud_job(const bh_cloud* tgt, const bh_cloud* src, int mask_self, const bh_law* law)
{
    CloudJob j;
    j.A.src = src->rows;
    j.A.ns = src->n;
    j.A.lds = src->ld;
    j.A.tgt = tgt->rows;
    j.A.nt = tgt->n;
    j.A.ldt = tgt->ld;
    j.A.mask_self = mask_self;
    j.A.G = law->G;
    j.A.eps2 = law->eps2;
    j.A.r2cut = law->r2_cut;
    int l;
    cloud_shape(j.A.nt, j.A.ns, &j.P, &l, &j.pairs);
    j.A.llog2 = l;
    j.blocks = cdiv(j.A.nt, (int64_t)j.P * (CL_THREADS >> l));
    return j;
}

// One launch for a, and for b (of a's P) too if it is given.
int launch_cloud(const CloudJob& a, const CloudJob* b, const bh_law* law, hipStream_t st)
{
    const int64_t blocks = a.blocks + (b ? b->blocks : 0);
    if (blocks > 0x7fffffffLL) return bh_ctx_fail(BH_EINVAL, "cloud too large for one launch");
    typedef void (*One)(CloudArgs);
    typedef void (*Both)(CloudArgs, CloudArgs, int);
    // [cutoff][softened][1 or 2 targets per lane, 2 with rows in pairs]
#define CL_TABLE(K)                                                                        \
    {{{K<0, 0, 1, 0>, K<0, 0, 2, 0>, K<0, 0, 2, 1>}, {K<0, 1, 1, 0>, K<0, 1, 2, 0>, K<0, 1, 2, 1>}}, \
     {{K<1, 0, 1, 0>, K<1, 0, 2, 0>, K<1, 0, 2, 1>}, {K<1, 1, 1, 0>, K<1, 1, 2, 0>, K<1, 1, 2, 1>}}}
    static const One one[2][2][3] = CL_TABLE(k_cloud);
    static const Both both[2][2][3] = CL_TABLE(k_cloud_both);
#undef CL_TABLE
    const int lc = law->r2_cut > 0.0, ls = law->eps2 > 0.0, shape = a.P - 1 + a.pairs;
    if (b)
        hipLaunchKernelGGL(both[lc][ls][shape], dim3((unsigned)blocks), dim3(CL_THREADS), 0, st,
                           a.A, b->A, (int)a.blocks);
    else
        hipLaunchKernelGGL(one[lc][ls][shape], dim3((unsigned)blocks), dim3(CL_THREADS), 0, st,
                           a.A);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : bh_ctx_fail(BH_EHIP, hipGetErrorString(e));
}

// Whether the memory of two clouds' rows overlaps (views of one array).
bool overlap(const bh_cloud* a, const bh_cloud* b)
{
    const uintptr_t a0 = (uintptr_t)a->rows, a1 = (uintptr_t)(a->rows + (a->n - 1) * a->ld + 7);
    const uintptr_t b0 = (uintptr_t)b->rows, b1 = (uintptr_t)(b->rows + (b->n - 1) * b->ld + 7);
    return a0 < b1 && b0 < a1;
}

int check_cloud(const bh_cloud* c, const char* name)
{
    char msg[160];
    if (c->n < 0 || c->ld < 7 || (c->n > 0 && !c->rows) ||
        (c->n > 0 && c->n > INT64_MAX / c->ld)) {
        snprintf(msg, sizeof msg, "%s cloud needs n >= 0, ld >= 7 and rows (n=%lld, ld=%lld)",
                 name, (long long)c->n, (long long)c->ld);
        return bh_ctx_fail(BH_EINVAL, msg);
    }
    return 0;
}

}  // namespace

extern "C" int bh_cloud_gravity(const bh_cloud* self, const bh_cloud* other, int32_t same,
                                const bh_law* law, int32_t update_other, void* stream)
{
    if (!self || !law || (!same && !other)) return bh_ctx_fail(BH_EINVAL, "NULL argument");
    if (!(law->eps2 >= 0.0) || !(law->r2_cut >= 0.0) || !std::isfinite(law->G))
        return bh_ctx_fail(BH_EINVAL, "law needs finite G, eps2 >= 0, r2_cut >= 0");
    int rc = check_cloud(self, "self");
    if (rc) return rc;
    if (!same && (rc = check_cloud(other, "other"))) return rc;
    hipStream_t st = (hipStream_t)stream;
    if (same) {
        // the self term has r^2 = 0: the cutoff drops it and softening makes
        // it 0 * w; only the plain law (0 / 0) needs it skipped by index
        const int mask = !(law->r2_cut > 0.0) && !(law->eps2 > 0.0);
        return self->n > 0 ? launch_cloud(cloud_job(self, self, mask, law), nullptr, law, st) : 0;
    }
    if (self->n == 0 || other->n == 0) return 0;
    const CloudJob a = cloud_job(self, other, 0, law);
    if (!update_other) return launch_cloud(a, nullptr, law, st);
    // both directions read positions and masses only and add to rows of their
    // own: one launch, unless a row is in both clouds or their shapes differ
    const CloudJob b = cloud_job(other, self, 0, law);
    if (a.P == b.P && a.pairs == b.pairs && a.blocks + b.blocks <= 0x7fffffffLL && !overlap(self, other))
        return launch_cloud(a, &b, law, st);
    if ((rc = launch_cloud(a, nullptr, law, st))) return rc;
    return launch_cloud(b, nullptr, law, st);
}
