// Kernel declarations and tile constants shared by the .hip translation units.
#pragma once
#include "bh_common.h"

// Particles per block in bbox / keys / scatter: 256 R.  Large sets take R = 8
// (a block's rows share its histogram window); below PLACE_SMALL that leaves
// too few blocks and each thread's rows come one after the other (k_bbox: 9.8
// us for 16,384 particles in 8 blocks).
#define PLACE_SMALL 262144
#define HIST_BINS 8192     // LDS histogram window (keys) per block
#define SCAN_TILE 2048     // elements per block in the scans
#define SCAN_ONE 16384     // elements that one block scans in one launch
#define PLACE_CELLS 8192   // cells of a system that one block places (k_place_one)
#define PLACE_ONE 4096     // rows of a system that one block places (k_place_one)
#define SORT_WAYS 16       // runs that a merge pass joins
#define ITEMS_COLS 1024    // columns whose items a block of k_com_items builds
#define ITEMS_ONE 65536    // particles up to which one block builds a step's items
#define COM_BIG 1024       // rows from which a cell's sums are a block's work (k_com)
#define SORT_W 1024        // within-cell rank window (rows)
#define SORT_THREADS 1024  // threads of a k_sort_units block (2 rows of the 2 SORT_W window each)

struct SortFields {
    const double *px, *py, *m, *vx, *vy, *ax, *ay;
    const int32_t* pid;
};

// Arguments of the force kernels (passed by value).
struct ForceArgs {
    const Item* items;
    const int32_t* order;      // queue position -> item (NULL: identity)
    int32_t* stats;
    const SysDev* sys;
    const int32_t* offsets;    // cell -> first sorted particle (C + 1)
    const int32_t* neprefix;   // cell -> first compact non-empty index (C + 1)
    const int32_t* key_sorted; // sorted particle -> global cell
    const double *x, *y, *m;
    const Com64* l64;
    const Com32* l32;
    double *ax, *ay;
    double Gc, eps2, r2cut;
    long long* cost_log;       // per item duration (wall clock ticks) or NULL
    // tail split (FP32 kernels): the last n_tail queue positions are each run
    // as `split` far-field parts, issued slice-major so that resident waves
    // share one slice of the COM list in L2; part holds their sums, one plane
    // of part_n particles x 2 doubles per slice (element ((s * part_n) + i) * 2),
    // added in slice order by k_force_combine.  split == 1: off.
    int split, n_tail;
    double* part;
    int64_t part_n;
    // this launch covers queue positions [total * qpart / nqparts,
    // total * (qpart + 1) / nqparts) (one launch: part 0 of 1)
    int qpart, nqparts;
    // FP64 recompute on (FP32 kernels): ax / ay point at zeroed scratch
    // planes of part_n doubles, and ay[part_n + i] receives particle i's sum
    // over its near-field terms of (m_j / r_ij)^2 (an upper bound of sum
    // |term|^2 under any softening or cutoff); the recompute then adds the
    // FP32 or the FP64 result to the particles' accelerations.  A flag rather
    // than a third pointer keeps the kernel's scalar registers unchanged.
    int rc;
    int64_t chunk0;   // k_force64s: first chunk of 64 particles of this launch (k_force32s too)
};

#define F64S_WAVES 8   // waves that share 64 particles (a power of two)
#define F32S_WAVES 8
void bh_force32s(const ForceArgs& A, int law, int S, int64_t nchunks, hipStream_t st);
// k_force64s over nchunks chunks from A.chunk0 on.
void bh_force64s(const ForceArgs& A, int law, int S, int64_t nchunks, hipStream_t st);

// Arguments of the grid-method potential (bh_potential.hip).
struct PotArgs {
    const Item* items;
    int32_t* stats;
    const SysDev* sys;
    const int32_t* offsets;
    const int32_t* neprefix;
    const int32_t* key_sorted;
    const double *x, *y, *m, *vx, *vy;
    const Com64* l64;
    const Com32* l32;
    const double* msys;   // total mass per system
    double eps2;
    double *u, *k;        // m_i phi_i and m_i |v_i|^2 per particle
};

// ---- grouped far field (bh_fmm.hip)
#define FMM_TILE 8           // cells per side of a tile at ~4 (fp32) or 30 (fp64) particles a cell
#define FMM_TILE_MIN 4       // and its range (fmm_tile)
#define FMM_TILE_MAX 24
#define FMM_SIDE_MAX 1024    // most tiles a side: a level's node masses are addressed with 32 bits
#define FMM_P32 12           // Chebyshev nodes per side, FP32 precision
#define FMM_P64 20           // and FP64 precision
#define FMM_LEVELS 13        // levels of squares (grid_dim <= 32767)
#define FMM_MIN_GRID 32      // smaller grids are one tile, every COM taken on its own
#define FMM_WAVES 8          // waves that share a chunk of a dense tile (a power of two)
#define FMM_DENSE 512        // mean cell count a particle sees from which its tile is dense
#define FMM_UNIFORM_ROWS 2   // rows a wave may span to walk its near candidates together

// A system: T cells per tile side, nlev levels of squares (0: one tile, no
// grouped part), n[l] squares per side at level l (level 0: the tiles), the
// first of them at off[l] of the square index space.
struct FmmSys {
    int32_t T, nlev;
    int32_t n[FMM_LEVELS];
    int32_t off[FMM_LEVELS];
    int64_t moff[FMM_LEVELS];   // first node-mass slot of the level (see fmm_slot)
};
struct FmmTile {
    int32_t sys;
    int16_t tx, ty;
};
struct FmmChunk {   // particles [64 k, 64 k + 64) of a tile
    int32_t tile, k;
};
struct FmmGroup {   // targets t0 .. t0 + cnt - 1 (at most 64) of a level's squares (2 i + a, 2 j + b)
    int32_t sys, t0, cnt;
    int16_t lev;
    int8_t a, b;
};
struct alignas(32) FmmCom {   // COM in units of step_scale, tile order
    double X, Y, M;
    int32_t kx, ky;
};
struct alignas(32) FmmPart {
    double x, y, m, pad;
};

enum {   // FmmArgs::cnt: chunks of dense tiles, of the others, list entries, dense queue cursor
    FMM_HEAVY,
    FMM_LIGHT,
    FMM_LIST,
    FMM_QHEAVY,
    FMM_NCNT
};

struct FmmArgs {
    const SysDev* sys;
    const FmmSys* fsys;
    const int32_t *sys_of, *offsets, *neprefix, *key_sorted;
    const Com64* l64;
    const double *x, *y, *m;
    double *ax, *ay;
    double* s2n;               // the near terms' (m / r)^2, if the recompute follows
    const FmmTile* tiles;      // every square, level by level
    const FmmGroup* groups;
    int32_t *tcnt;             // per square: particles
    int32_t *tstart, *tne;     // per tile: its run of list
    int32_t* cnt;              // FMM_HEAVY .. FMM_QHEAVY, then per system sbad
    int32_t* sbad;             // != 0: a COM lies outside its tile
    FmmChunk* chunks;
    FmmCom* list;
    FmmPart* pack;
    double* mult;              // node masses, node-major (fmm_slot)
    double* multf;             // the same on the coarser nodes of far offsets
    double* loc;               // per square: P^2 ax, P^2 ay
    double* locf;              // the part of far offsets, F^2 ax, F^2 ay
    int32_t S;
    int64_t N, nleaf, ntiles, max_chunks;
    int64_t lev_off[FMM_LEVELS + 1];
};

// Of the 27 squares that a square takes directly, the 15 with a gap of two
// squares or past a corner converge faster and take fewer nodes per side: across
// (3, 0) and (2, 2), 16 leave 4e-15 (20 across (2, 0) 2e-15) and 10 leave 4e-11
// and 2e-10 (12 across (2, 0) 6e-10).
__host__ __device__ constexpr int fmm_far(int P) { return P == FMM_P64 ? 16 : 10; }
__host__ __device__ inline bool fmm_is_far(int ox, int oy)
{
    const int a = ox < 0 ? -ox : ox, b = oy < 0 ? -oy : oy;
    return a + b >= 4 || a > 2 || b > 2;
}

// Node masses of a level of n^2 squares: node-major planes, so that the squares
// a wave reads together are neighbours in memory.  A plane holds the squares by
// child position (x & 1, y & 1), each class a (np + 2)^2 array with a border of
// zeros (np = (n + 1) / 2) that stands for the squares outside the grid.
__host__ __device__ inline int fmm_pitch(int n) { return (n + 1) / 2 + 2; }
__host__ __device__ inline int64_t fmm_plane(int n)
{
    return 4 * (int64_t)fmm_pitch(n) * fmm_pitch(n);
}
// Slot of square (x, y) in a plane.
__host__ __device__ inline int fmm_slot(int n, int x, int y)
{
    const int w = fmm_pitch(n);
    return ((2 * (x & 1) + (y & 1)) * w + (x >> 1) + 1) * w + (y >> 1) + 1;
}

struct FmmTables {
    const double *nodes;   // P Chebyshev nodes on [-1, 1]
    const double *cheb;    // [k][i]: c_k T_k(node i), c_0 = 1 / P, c_k = 2 / P
    const double *shift;   // [a][i][I]: cardinal i of a square at node I of its child half a
    const double *fnodes;  // F = fmm_far(P) nodes
    const double *fine;    // [I][i]: cardinal I of the F nodes at node i of the P
};
struct FmmPlan {
    int nlev = 0;
    int64_t ngroups = 0;
    FmmTables tab;
};
void bh_fmm_pass(const FmmArgs& A, const FmmPlan& pl, bool fp64, double Gc, double eps2,
                 double r2cut, int part, int nparts, int num_cu, hipStream_t st);

// m / q to FP64 accuracy without the IEEE division sequence: v_rcp_f64 gives
// r0 with e = 1 - q r0 small (|e| < 2^-22), and 1/q = r0 (1 + e + e^2 + e^3 + ...),
// so m r0 (1 + e + e^2) differs from m / q by the relative e^3 plus the
// roundings of m r0 and of the final fma: within about one ulp.  Three VALU
// instructions and the reciprocal, against ten and the reciprocal for the
// correctly rounded quotient.  q = 0 gives NaN (m / 0 * 0 is NaN as well).
__device__ __forceinline__ double wdiv64(double m, double q)
{
    const double r0 = __builtin_amdgcn_rcp(q);
    const double e = fma(-q, r0, 1.0);
    const double ee = fma(e, e, e);
    const double w0 = m * r0;
    return fma(w0, ee, w0);
}

// One FP64 weight m * w(r2) of the law (LAW 0: no cutoff; LAW 1: r2 <= r2cut
// gives 0).  FAST 1: the quotient by wdiv64 (the FP64 kernel's near field);
// FAST 0: the IEEE division (the fp64_ieee kernel).
template <int FAST>
__device__ __forceinline__ double qdiv64(double m, double q)
{
    return FAST ? wdiv64(m, q) : m / q;
}

template <int LAW, int FAST>
__device__ __forceinline__ double far_w64(double wx, double wy, double M, double eps2, double r2cut)
{
    if (LAW == 0) return qdiv64<FAST>(M, fma(wx, wx, fma(wy, wy, eps2)));
    const double s2 = fma(wx, wx, wy * wy);
    return (s2 > r2cut) ? qdiv64<FAST>(M, s2 + eps2) : 0.0;
}

template <int LAW, int FAST>
__device__ __forceinline__ double near_w64(double wx, double wy, double m, double eps2, double r2cut)
{
    const double s2 = fma(wx, wx, wy * wy);
    if (LAW == 0) return qdiv64<FAST>(m, s2 + eps2);
    return (s2 > r2cut) ? qdiv64<FAST>(m, s2 + eps2) : 0.0;
}

// Wave-uniform reads through the constant address space: scalar loads, so
// every lane gets the value from a scalar register.
typedef double fd8 __attribute__((ext_vector_type(8)));
template <typename T>
using cptr = const T __attribute__((address_space(4)))*;

template <typename T>
__device__ __forceinline__ cptr<T> as_const(const T* p)
{
    return (cptr<T>)(uintptr_t)p;
}

// The power of two that brings the cell side into [1, 2): positions scaled by
// it are exact, and a distance to another cell's COM is at least 1.
__device__ __forceinline__ double step_scale(double step)
{
    if (!(step > 0.0) || !(step < __builtin_huge_val())) return 1.0;
    int e2;
    (void)frexp(step, &e2);
    return ldexp(1.0, 1 - e2);
}

// Whether (fx, fy), in cell sides from a cell's corner, lies in the cell, up to
// a thousandth of it (rounding of a COM's sums).
__device__ __forceinline__ bool in_cell(double fx, double fy)
{
    return fabs(fx - 0.5) <= 0.501 && fabs(fy - 0.5) <= 0.501;
}

// Whether every COM outside a lane's 3x3 cells is beyond the cutoff r2cut (in
// units of step_scale) for all lanes of the wave, so that its term needs no
// test: the cutoff is below a cell side (at least 1; 0.996 squared with
// in_cell's margins), the system's COMs lie in their cells and the lanes'
// particles, (fx, fy) in cell sides from the corner of the cell that they were
// placed in, are still there.
template <int LAW>
__device__ __forceinline__ bool placed_apart(const SysDev& d, double r2cut, bool act, double fx,
                                             double fy)
{
    if (LAW == 0) return true;
    if (!(r2cut < 0.99) || d.com_out != 0) return false;
    return __ballot(act && !in_cell(fx, fy)) == 0ull;
}

// 1 / q as in wdiv64.
__device__ __forceinline__ double rcp64(double q)
{
    const double r0 = __builtin_amdgcn_rcp(q);
    const double e = fma(-q, r0, 1.0);
    return fma(r0, fma(e, e, e), r0);
}

// Two terms of the law from one reciprocal: Q = q0 q1, R = 1 / Q, so the
// weights are (m0 R) q1 and (m1 R) q0.  An entry that the particle does not
// keep enters as q = 1 with weight 0.  (wx, wy): from the particle.  Under a
// cutoff, a wave none of whose lanes drops either term (all but the closest
// pairs) takes the plain form after one test of the smaller distance: ~14 issue
// slots a term instead of 19 with a select per q and weight.
// SQ: s2 gains the sum of m w, which is (m / r)^2, r softened.
template <int LAW, bool MASK, bool SQ = false>
__device__ __forceinline__ void pair_terms(double wx0, double wy0, double m0, double wx1,
                                           double wy1, double m1, bool k0, bool k1, double eps2,
                                           double r2cut, double& sx, double& sy,
                                           double* s2 = nullptr)
{
    double q0, q1;
    bool sel = MASK;   // wave-uniform
    if (LAW == 1) {
        const double s0 = fma(wx0, wx0, wy0 * wy0), s1 = fma(wx1, wx1, wy1 * wy1);
        q0 = s0 + eps2;
        q1 = s1 + eps2;
        if (MASK) {
            k0 = k0 && s0 > r2cut;
            k1 = k1 && s1 > r2cut;
        } else if (__any(!(fmin(s0, s1) > r2cut))) {
            sel = true;
            k0 = s0 > r2cut;
            k1 = s1 > r2cut;
        }
    } else {
        q0 = fma(wx0, wx0, fma(wy0, wy0, eps2));
        q1 = fma(wx1, wx1, fma(wy1, wy1, eps2));
    }
    if (sel) {
        q0 = k0 ? q0 : 1.0;
        q1 = k1 ? q1 : 1.0;
    }
    const double R = rcp64(q0 * q1);
    double w0 = (m0 * R) * q1, w1 = (m1 * R) * q0;
    if (sel) {
        w0 = k0 ? w0 : 0.0;
        w1 = k1 ? w1 : 0.0;
    }
    sx = fma(wx0, w0, sx);
    sy = fma(wy0, w0, sy);
    sx = fma(wx1, w1, sx);
    sy = fma(wy1, w1, sy);
    if (SQ) *s2 = fma(m1, w1, fma(m0, w0, *s2));
}

// Four terms from one reciprocal: pairs are brought to common denominators,
// (m0 q1) w0 + (m1 q0) w1 over q0 q1, and R = 1 / (q0 q1 q2 q3).  33
// instructions and one reciprocal (of several issue slots) after the
// separations, where two pairs take 34 and two: 10M particles over 120^2 cells,
// 6.7e10 terms, 26.5 -> 24.3 ms.
template <int LAW, bool MASK, bool SQ = false>
__device__ __forceinline__ void quad_terms(const double (&wx)[4], const double (&wy)[4],
                                           const double (&m)[4], const bool (&keep)[4],
                                           double eps2, double r2cut, double& sx, double& sy,
                                           double* s2 = nullptr)
{
    double q[4], t[4];
    bool k[4] = {keep[0], keep[1], keep[2], keep[3]};
    bool sel = MASK;   // wave-uniform
    if (LAW == 1) {
        double s[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            s[u] = fma(wx[u], wx[u], wy[u] * wy[u]);
            q[u] = s[u] + eps2;
        }
        if (MASK || __any(!(fmin(fmin(s[0], s[1]), fmin(s[2], s[3])) > r2cut))) {
            sel = true;
#pragma unroll
            for (int u = 0; u < 4; ++u) k[u] = (!MASK || k[u]) && s[u] > r2cut;
        }
    } else {
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = fma(wx[u], wx[u], fma(wy[u], wy[u], eps2));
    }
    if (sel) {
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = k[u] ? q[u] : 1.0;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        t[u] = m[u] * q[u ^ 1];
        if (sel) t[u] = k[u] ? t[u] : 0.0;
    }
    const double Q0 = q[0] * q[1], Q1 = q[2] * q[3];
    const double nx0 = fma(wx[1], t[1], wx[0] * t[0]), ny0 = fma(wy[1], t[1], wy[0] * t[0]);
    const double nx1 = fma(wx[3], t[3], wx[2] * t[2]), ny1 = fma(wy[3], t[3], wy[2] * t[2]);
    const double R = rcp64(Q0 * Q1);
    const double u0 = R * Q1, u1 = R * Q0;
    sx = fma(nx0, u0, sx);
    sy = fma(ny0, u0, sy);
    sx = fma(nx1, u1, sx);
    sy = fma(ny1, u1, sy);
    if (SQ) {
        *s2 = fma(fma(m[1], t[1], m[0] * t[0]), u0, *s2);
        *s2 = fma(fma(m[3], t[3], m[2] * t[2]), u1, *s2);
    }
}

// One term, by a reciprocal of its own.  The products above leave a double's
// range where softening is below ~1e-77 cell sides squared (and particles
// coincide) or above 1e77, and then leave an infinite or NaN sum: the kernels
// take such a wave's or block's terms again, one by one, which says what the sum
// is where it is not finite by itself.
template <int LAW>
__device__ __forceinline__ void one_term(double wx, double wy, double m, bool keep, double eps2,
                                         double r2cut, double& sx, double& sy)
{
    double w = near_w64<LAW, 1>(wx, wy, m, eps2, r2cut);
    w = keep ? w : 0.0;
    sx = fma(wx, w, sx);
    sy = fma(wy, w, sy);
}

__device__ __forceinline__ bool is_finite(double sx, double sy)
{
    return fabs(sx) < __builtin_huge_val() && fabs(sy) < __builtin_huge_val();
}

// grid-method potential
__global__ void k_sys_mass(const SysDev* sys, const int32_t* neprefix, const Com64* l64,
                           double* msys);
template <int P>
__global__ void k_potential(PotArgs A);

// placement
__global__ void k_fill_i32(int32_t* p, int64_t n, int32_t v);
__global__ void k_fill_f64(double* p, int64_t n, double v);
__global__ void k_place_init(int32_t* stats, int32_t* counts, int64_t C, uint64_t* bb, int S);
template <int R>
__global__ void k_bbox(const double* px, const double* py, const int32_t* sys_of, int64_t N, int rounds,
                       uint64_t* bb, int32_t* stats);
template <int R>
__global__ void k_keys_hist(const double* px, const double* py, const int32_t* sys_of, SysDev* sys,
                            const uint64_t* bb, int64_t N, int32_t* key_out, int32_t* rank_out,
                            int32_t* counts, int32_t* stats);
template <bool CNT>
__global__ void k_scan_reduce(const int32_t* in, int64_t n, int32_t* bsum, int32_t* bne,
                              int32_t* stats);
template <bool CNT>
__global__ void k_scan_blocks(int32_t* bsum, int32_t* bne, int64_t nb, int32_t* stats,
                              int total_slot);
template <bool CNT>
__global__ void k_scan_final(const int32_t* in, int64_t n, const int32_t* bsum, const int32_t* bne,
                             int32_t* out_v, int32_t* out_f, int32_t* ne_list, double* com_dense);
template <bool CNT>
__global__ void k_scan_one(const int32_t* in, int n, int32_t* out_v, int32_t* out_f,
                           int32_t* ne_list, double* com_dense, int32_t* stats, int total_slot,
                           int64_t max_total);
template <int R>
__global__ void k_scatter(const int32_t* key, int64_t N, const int32_t* offsets,
                          const int32_t* rank, int32_t* idx_out, int32_t* key_sorted, const double* px,
                          const double* py, uint64_t* pxkey_out, uint64_t* pykey_out);
__global__ void k_place_one(const double* px, const double* py, SysDev* sys, int N, int C,
                            int32_t* key_out, int32_t* rank_out, int32_t* counts, int32_t* offsets,
                            int32_t* neprefix, int32_t* ne_list, double* com_dense,
                            int32_t* idx_out, int32_t* key_sorted, uint64_t* pxkey,
                            uint64_t* pykey, int32_t* stats);
__global__ void k_sort_units(SortFields F, int64_t N, const int32_t* idx_in,
                             const int32_t* key_sorted, const uint64_t* pxkey,
                             const uint64_t* pykey, const int32_t* offsets, int32_t* idx_out);
__global__ void k_sort_merge(SortFields F, int64_t N, const int32_t* idx_in,
                             const int32_t* key_sorted, const int32_t* offsets, int32_t* idx_out,
                             int64_t R, const int32_t* stats);
__global__ void k_gather(SortFields S, BhParticles D, int64_t N, const int32_t* idx_a,
                         const int32_t* idx_b, const int32_t* key_sorted, const int32_t* offsets,
                         const int32_t* stats, int32_t* perm_out);

// summarize + tick
__global__ void k_com(SysDev* sys, int S, const int32_t* ne_list, const int32_t* stats,
                      const int32_t* offsets, const double* x, const double* y, const double* m,
                      double* com_dense, Com64* l64, Com32* l32);
// k_com, and in its last block the items (k_items_runs) of at most ITEMS_COLS columns
__global__ void k_com_items(SysDev* sys, int S, const int32_t* ne_list, int32_t* stats,
                            const int32_t* offsets, const double* x, const double* y,
                            const double* m, double* com_dense, Com64* l64, Com32* l32, int ncols,
                            int pitem, int32_t* col_off, Item* items, int64_t max_items, int write);
__global__ void k_tick(double* x, double* y, double* vx, double* vy, double* ax, double* ay,
                       int64_t N, double dt);
__global__ void k_interactions(const SysDev* sys, int S, const int32_t* counts,
                               const int32_t* neprefix, int64_t C,
                               unsigned long long* out /* 2*S + 2 */);
__global__ void k_energy(const double* x, const double* y, const double* m, const double* vx,
                         const double* vy, int64_t p0, int64_t n, double eps2, double* u,
                         double* k);

// force
__global__ void k_clamp_items(int32_t* stats, int64_t max_items);
__global__ void k_force_combine(const Item* items, const int32_t* order, const int32_t* stats,
                                int split, int n_tail, int pslots, const double* part,
                                int64_t part_n, double* ax, double* ay);
// FP64 recompute of the particles whose FP32 rounding-error estimate is
// large against their acceleration
__global__ void k_rc_grouped(int32_t* stats);
__global__ void k_rc_sums(const SysDev* sys, int S, int64_t nblocks, int64_t ntiles, int nb,
                          const double* com_dense, double* blk, double* tl, int32_t* rc_cnt,
                          int32_t* stats);
__global__ void k_rc_blockfar(const SysDev* sys, int S, int64_t nblocks, const double* blk,
                              double* bfar);
template <int W>
__global__ void k_rc_flag(const Item* items, const SysDev* sys, const int32_t* key_sorted,
                          const int32_t* neprefix, const Com64* l64, const double* x,
                          const double* y, const double* com, const double* tl,
                          const double* blk, const double* bfar, const double* a32x,
                          const double* a32y, const double* s2n, double Gc, double kappa2,
                          const int32_t* stats, int32_t* rc_cnt, int32_t* list, double* ax,
                          double* ay);
__global__ void k_rc_groups(const int32_t* rc_cnt, int S, int32_t* gofs, int32_t* stats);
template <int LAW>
__global__ void k_rc_fix64(const int32_t* stats, const int32_t* rc_cnt, const int32_t* gofs,
                           int S, const int32_t* list, const SysDev* sys,
                           const int32_t* key_sorted, const int32_t* offsets,
                           const int32_t* neprefix, const Com64* l64, const double* x,
                           const double* y, const double* m, double Gc, double eps2,
                           double r2cut, double* part, double* ax, double* ay);
__global__ void k_rc_combine(const int32_t* stats, const int32_t* rc_cnt, const int32_t* gofs,
                             int S, const int32_t* list, const SysDev* sys, const double* part,
                             double Gc, double* ax, double* ay);

template <bool WRITE>
__global__ void k_items(const SysDev* sys, int S, int64_t ncols, const int32_t* offsets, int pitem,
                        int yspan, int32_t* col_items, Item* items, int64_t max_items,
                        int32_t* stats);
__global__ void k_items_runs(const SysDev* sys, int S, int ncols, const int32_t* offsets, int pitem,
                             int32_t* col_off, Item* items, int64_t max_items, int32_t* stats,
                             int write);
__global__ void k_items_fill(const SysDev* sys, int S, int ncols, const int32_t* offsets, int pitem,
                             const int32_t* col_off, Item* items, const int32_t* stats);
