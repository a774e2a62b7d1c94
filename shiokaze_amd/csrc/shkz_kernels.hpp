// shkz_kernels.hpp -- HIP kernels of the MI355X pressure projection (gfx950).
//
// Stages, in the order of macpressuresolver3::project (src/projection/macpressuresolver3.cpp):
//   k_any_negative     levelset_exist() of both level sets (array_utility3.h:112-122)
//   k_curvature,
//   k_surface_tension  surface-tension impulse (:85-115)
//   k_flags            unknown labelling (:121-156) + which 8^3 bricks hold unknowns
//   k_operator         matrix-free assembly (:159-199): conductances, Dirichlet sums, rhs
//   k_coarsen, k_idiag multigrid operators (no counterpart: they stand in for MIC(0))
//   k_defect4 ... k_update_p, V-cycle kernels
//                      Krylov solve (stands in for PCGSolver::solve, pcg_solver.h:246-295)
//   k_output           m_pressure (:245-248) and velocity update (:252-268)
//
// Build and output kernels work on dense arrays, up to twelve grids in a launch.  Solver kernels work on a batch: the
// stored bricks of every grid of the batch, concatenated, one 512-thread block per brick (thread =
// cell) with an XCD-aware block-to-brick remap.  Stencil neighbours in the same brick are read at
// +-1/8/64, the others through the brick's neighbour table.  Reductions are per grid and
// deterministic (per-brick partials, combined in brick order).
#pragma once
#include "shkz_device.hpp"
#include "shkz_geometry.hpp"

// No floating-point contraction in any solver kernel: every a*b+c rounds twice, exactly as
// written.  The same sweep, residual and prolongation are computed by different kernels depending
// on a level's size (one launch per sweep, or several sweeps in LDS), and the size of a level
// depends on the batch a grid is in; with the operations fixed by the source, every form gives the
// same bits, so a grid's result does not depend on its batch.
#pragma clang fp contract(off)

namespace shkz {

// ------------------------------------------------------------------------------ helpers
constexpr int UNIFORM_COUNT_BIT = 1 << 20;  // brick counts: the brick is BM_UNIFORM (counts <= 512)

struct Nbrs {
    long base;
    int n[6];
};

__device__ __forceinline__ Nbrs nbrs_of(const BrickMeta &m, int b) {
    Nbrs N;
    N.base = (long)b * BRICK_CELLS;
#pragma unroll
    for (int d = 0; d < 6; ++d) N.n[d] = m.nbr[d];
    return N;
}

__device__ __forceinline__ Nbrs load_nbrs(const LevelDesc &L, int b) { return nbrs_of(L.meta[b], b); }

// Storage index of the six face neighbours of local cell t, -1 where no brick is stored.
__device__ __forceinline__ void nb_index(const Nbrs &N, int t, long idx[6]) {
    const int li = t >> 6, lj = (t >> 3) & 7, lk = t & 7;
    idx[NB_XM] = li > 0 ? N.base + t - 64 : (N.n[NB_XM] >= 0 ? (long)N.n[NB_XM] * BRICK_CELLS + t + 448 : -1);
    idx[NB_XP] = li < 7 ? N.base + t + 64 : (N.n[NB_XP] >= 0 ? (long)N.n[NB_XP] * BRICK_CELLS + t - 448 : -1);
    idx[NB_YM] = lj > 0 ? N.base + t - 8 : (N.n[NB_YM] >= 0 ? (long)N.n[NB_YM] * BRICK_CELLS + t + 56 : -1);
    idx[NB_YP] = lj < 7 ? N.base + t + 8 : (N.n[NB_YP] >= 0 ? (long)N.n[NB_YP] * BRICK_CELLS + t - 56 : -1);
    idx[NB_ZM] = lk > 0 ? N.base + t - 1 : (N.n[NB_ZM] >= 0 ? (long)N.n[NB_ZM] * BRICK_CELLS + t + 7 : -1);
    idx[NB_ZP] = lk < 7 ? N.base + t + 1 : (N.n[NB_ZP] >= 0 ? (long)N.n[NB_ZP] * BRICK_CELLS + t - 7 : -1);
}

template <class T>
__device__ __forceinline__ T ld(const T *a, long i) {
    return i >= 0 ? a[i] : T(0);
}

// (A p)_c for an unknown c; also returns the diagonal.
template <class T>
__device__ __forceinline__ T apply_row(const OpDesc<T> &A, const T *__restrict__ p, long c, const long idx[6], T dirc,
                                       T pc, T &diag) {
    const T gxm = A.gx[c], gym = A.gy[c], gzm = A.gz[c];
    const T gxp = ld(A.gx, idx[NB_XP]), gyp = ld(A.gy, idx[NB_YP]), gzp = ld(A.gz, idx[NB_ZP]);
    const T off = gxm * ld(p, idx[NB_XM]) + gxp * ld(p, idx[NB_XP]) + gym * ld(p, idx[NB_YM]) +
                  gyp * ld(p, idx[NB_YP]) + gzm * ld(p, idx[NB_ZM]) + gzp * ld(p, idx[NB_ZP]);
    diag = dirc + ((gxm + gxp) + (gym + gyp) + (gzm + gzp));
    return diag * pc - off;
}

// Sum of g_f * v_q over the six faces of cell c.
template <class T>
__device__ __forceinline__ T offdiag_sum(const OpDesc<T> &A, const T *__restrict__ v, long c, const long idx[6]) {
    const T gxp = ld(A.gx, idx[NB_XP]), gyp = ld(A.gy, idx[NB_YP]), gzp = ld(A.gz, idx[NB_ZP]);
    return A.gx[c] * ld(v, idx[NB_XM]) + gxp * ld(v, idx[NB_XP]) + A.gy[c] * ld(v, idx[NB_YM]) +
           gyp * ld(v, idx[NB_YP]) + A.gz[c] * ld(v, idx[NB_ZM]) + gzp * ld(v, idx[NB_ZP]);
}

// apply_row and offdiag_sum on a BM_UNIFORM brick: every coupling is g and the Dirichlet sum 0
// (the same operations in the same order, so the same values).
template <class T>
__device__ __forceinline__ T offdiag_uniform(T g, const T *__restrict__ v, const long idx[6]) {
    return g * ld(v, idx[NB_XM]) + g * ld(v, idx[NB_XP]) + g * ld(v, idx[NB_YM]) + g * ld(v, idx[NB_YP]) +
           g * ld(v, idx[NB_ZM]) + g * ld(v, idx[NB_ZP]);
}
template <class T>
__device__ __forceinline__ T apply_row_uniform(T g, const T *__restrict__ p, long c, const long idx[6], T pc) {
    (void)c;
    const T off = offdiag_uniform(g, p, idx);
    const T diag = T(0) + ((g + g) + (g + g) + (g + g));
    return diag * pc - off;
}

__device__ __forceinline__ int brick_or_idle(const LevelDesc &L) {
    const int b = xcd_brick(blockIdx.x, gridDim.x);
    return b < L.nbricks ? b : -1;
}

__device__ __forceinline__ bool all_done(const Gate &Q) { return Q.ctl && Q.ctl->all_done; }

// The brick's grid is done (in a batch of one, all_done says so already: no load).
__device__ __forceinline__ bool grid_done(const Gate &Q, const LevelDesc &L, const BrickMeta &m) {
    return L.ngrids > 1 && Q.S && Q.S[m.grid].done;
}

// Smoothing-side V-cycle work on a brick is skipped for a grid that is done, or where another kernel
// does it: on the grid's last level (the coarse solve), or on any level of its bottom (k_bottom).
__device__ __forceinline__ bool skip_smooth(const Gate &Q, const LevelDesc &L, const BrickMeta &m) {
    return (m.flags & Q.skip) || grid_done(Q, L, m);
}

// Value of level vector v at cell (i,j,k) of the grid described by G (0 outside or unstored).
template <class T>
__device__ __forceinline__ T level_value(const LevelDesc &L, const GridLevel &G, const T *__restrict__ v, int i, int j,
                                         int k) {
    if (i < 0 || j < 0 || k < 0 || i >= G.ni || j >= G.nj || k >= G.nk) return T(0);
    const int b = L.bmap[G.bmap_off + ((i >> 3) * G.nby + (j >> 3)) * G.nbz + (k >> 3)];
    if (b < 0) return T(0);
    return v[(long)b * BRICK_CELLS + (((i & 7) * 8 + (j & 7)) * 8 + (k & 7))];
}

// ------------------------------------------------------------------------------ build (one grid)
__global__ void k_reset_ints(int *a, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = 0;
}

// flag |= 1 when any of the n values is negative.  A 16-byte aligned array is read 16 bytes per
// load, four loads in flight per thread.
constexpr int NEGATIVE_THREADS = 256;
template <class T>
__device__ __forceinline__ bool any_negative(const T *a, size_t n, size_t tid, size_t nt) {
    constexpr int PER = 16 / sizeof(T);  // values per 16 bytes
    typedef T Vec __attribute__((ext_vector_type(PER)));
    bool found = false;
    size_t done = 0;
    if (((uintptr_t)a & 15) == 0) {
        const Vec *v = (const Vec *)a;
        const size_t nv = n / PER;
        auto negative = [](const Vec x) {
            bool neg = false;
#pragma unroll
            for (int j = 0; j < PER; ++j) neg |= x[j] < T(0);
            return neg;
        };
        size_t i = tid;
        for (; i + 3 * nt < nv; i += 4 * nt) {
            const Vec x0 = v[i], x1 = v[i + nt], x2 = v[i + 2 * nt], x3 = v[i + 3 * nt];
            found |= negative(x0) | negative(x1) | negative(x2) | negative(x3);  // (no short cut: the loads go out together)
        }
        for (; i < nv; i += nt) found |= negative(v[i]);
        done = nv * PER;
    }
    for (size_t i = done + tid; i < n; i += nt) found |= a[i] < T(0);
    return found;
}
__global__ __launch_bounds__(NEGATIVE_THREADS) void k_any_negative(const void *a, int is64, size_t n, int *flag) {
    const size_t tid = (size_t)blockIdx.x * NEGATIVE_THREADS + threadIdx.x, nt = (size_t)gridDim.x * NEGATIVE_THREADS;
    const bool found = is64 ? any_negative((const double *)a, n, tid, nt) : any_negative((const float *)a, n, tid, nt);
    // (a vote through LDS: __syncthreads_or, like an array that the compiler moves to LDS, reads the dispatch
    // packet, from host memory, 3 us of a short launch)
    __shared__ int votes[NEGATIVE_THREADS / 64];
    const bool wave = __ballot(found) != 0;
    if ((threadIdx.x & 63) == 0) votes[threadIdx.x >> 6] = wave;
    __syncthreads();
    if (threadIdx.x != 0) return;
    int any = 0;
#pragma unroll
    for (int w = 0; w < NEGATIVE_THREADS / 64; ++w) any |= votes[w];
    // the flag only ever goes from 0 to 1: a plain store, skipped once it is seen set; even the look at it costs 6 ns
    // per workgroup, one after another, so that a launch has few of them (any_negative_blocks)
    if (any && __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
        __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// 7-point Laplacian of the level set with clamped neighbours (macpressuresolver3.cpp:92-100);
// float level sets are summed in float as the reference sums Real values.
__global__ void k_curvature(GridDesc G, float *curv) {
    const size_t M = (size_t)G.w * G.h * G.d;
    const size_t c = (size_t)xcd_brick(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (c >= M) return;
    int i, j, k;
    unflatten((unsigned)c, (unsigned)G.h, (unsigned)G.d, i, j, k);
    const int im = clampi(i - 1, 0, G.w - 1), ip = clampi(i + 1, 0, G.w - 1);
    const int jm = clampi(j - 1, 0, G.h - 1), jp = clampi(j + 1, 0, G.h - 1);
    const int km = clampi(k - 1, 0, G.d - 1), kp = clampi(k + 1, 0, G.d - 1);
    double value;
    if (G.flat) {
        // 5-point Laplacian of the 2D module (macpressuresolver2.cpp:82-89), summed in the level
        // set's precision
        if (G.phi64) {
            const double s = +phi_at(G, im, j, k) + phi_at(G, ip, j, k) + phi_at(G, i, jm, k) + phi_at(G, i, jp, k);
            value = (s - 4.0 * phi_at(G, i, j, k)) / (G.dx * G.dx);
        } else {
            const float *f = (const float *)G.phi;
            const float s = +f[cell_index(G, im, j, k)] + f[cell_index(G, ip, j, k)] + f[cell_index(G, i, jm, k)] +
                            f[cell_index(G, i, jp, k)];
            value = (s - 4.0 * f[c]) / (G.dx * G.dx);
        }
    } else if (G.phi64) {
        const double s = +phi_at(G, im, j, k) + phi_at(G, ip, j, k) + phi_at(G, i, jm, k) + phi_at(G, i, jp, k) +
                         phi_at(G, i, j, km) + phi_at(G, i, j, kp);
        value = (s - 6.0 * phi_at(G, i, j, k)) / (G.dx * G.dx);
    } else {
        const float *f = (const float *)G.phi;
        const float s = +f[cell_index(G, im, j, k)] + f[cell_index(G, ip, j, k)] + f[cell_index(G, i, jm, k)] +
                        f[cell_index(G, i, jp, k)] + f[cell_index(G, i, j, km)] + f[cell_index(G, i, j, kp)];
        value = (s - 6.0 * f[c]) / (G.dx * G.dx);
    }
    curv[c] = (float)value;
}

// Surface-tension impulse on faces with 0 < rho < 1 (macpressuresolver3.cpp:102-113).
__global__ void k_surface_tension(GridDesc G, int dim, const float *curv, double kappa) {
    const int W = G.w + (dim == 0), H = G.h + (dim == 1), D = G.d + (dim == 2);
    const size_t n = (size_t)W * H * D;
    const size_t f = (size_t)xcd_brick(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (f >= n) return;
    if (G.active[dim] && !G.active[dim][f]) return;
    int i, j, k;
    unflatten((unsigned)f, (unsigned)H, (unsigned)D, i, j, k);
    const double rho = face_rho(G, exist_of(G), dim, i, j, k);
    if (rho && rho < 1.0) {
        const int i0 = clampi(i, 0, G.w - 1), j0 = clampi(j, 0, G.h - 1), k0 = clampi(k, 0, G.d - 1);
        const int i1 = clampi(i - (dim == 0), 0, G.w - 1), j1 = clampi(j - (dim == 1), 0, G.h - 1),
                  k1 = clampi(k - (dim == 2), 0, G.d - 1);
        const double sgn = phi_at(G, i0, j0, k0) < 0.0 ? -1.0 : 1.0;
        const double theta = sgn < 0 ? 1.0 - rho : rho;
        const double face_c = theta * curv[cell_index(G, i0, j0, k0)] + (1.0 - theta) * curv[cell_index(G, i1, j1, k1)];
        G.vel[dim][f] += (float)(-sgn * G.dt / (G.dx * rho) * kappa * face_c);
    }
}

// The kernels that run once per grid of a batch (labelling, assembly, output) take up to
// GRIDS_PER_LAUNCH grids in one launch: their descriptors travel in the kernel's arguments (which hold 4 KB),
// and workgroup b works for the grid whose range [first[g], first[g + 1]) holds b.  A launch of its own costs a
// small grid more than its work (64 cubes of 32 to 160 cells: 5 launches per grid).
constexpr int GRIDS_PER_LAUNCH = 12;
template <class D>
struct GridTable {
    int n;
    int first[GRIDS_PER_LAUNCH + 1];
    D g[GRIDS_PER_LAUNCH];
};
// The grid of this workgroup and its workgroup index within it (-1: a workgroup beyond the last grid).
// Each XCD takes a contiguous range of the launch.
template <class D>
__device__ __forceinline__ int table_grid(const GridTable<D> &T, int &local) {
    const int blk = xcd_brick(blockIdx.x, gridDim.x);
    int g = 0;
    while (g < T.n && blk >= T.first[g + 1]) ++g;
    if (g == T.n) return -1;
    local = blk - T.first[g];
    return g;
}

// Marks the bricks beside brick br (BM_LOOSE) if one of this wavefront's cells in it is coupled and no unknown.
__device__ __forceinline__ void mark_loose(BrickMeta *meta, int br, bool coupled_out) {
    if (__ballot(coupled_out) == 0) return;
    const int lane = threadIdx.x & 63;
    const int nb = lane < 6 ? meta[br].nbr[lane] : -1;
    if (nb >= 0) atomicOr(&meta[nb].flags, BM_LOOSE);
}

// Unknown labelling (macpressuresolver3.cpp:121-156): a liquid cell is an unknown when an
// in-bounds liquid neighbour shares a face with nonzero area (rho is nonzero between two liquid
// cells).  Writes cell flags (bit0 liquid, bit1 unknown) and per brick bit0 = holds an unknown, bit1 =
// holds a liquid cell (so the host learns levelset_exist() of the liquid, array_utility3.h:112-122, on
// the way).
//
// Without a solid only signs matter, and the kernel is a pass over the level set.  A thread takes a column
// of 8 cells along x, a workgroup the columns of FLAGS_SPAN bricks along z (FLAGS_SPAN_FLAT along y in a 2D
// grid), so that a sample is read 1.25 times instead of up to 7: the signs of a column are the bits of one
// byte, which neighbours take from LDS.  256^3 of FP64 samples: 116 us with one cell per thread and a
// chain of neighbour tests, 102 us with columns that load their neighbours, 67 us
// with 32 columns a workgroup along z, 60 with the 64 here (a border cell costs its whole cache line); 120x168x89
// within a solid's reach 40 to 17 us.
struct FlagsGrid {
    GridDesc G;
    int nbx, nby, nbz;
    uint8_t *cflag, *bflag;
};
constexpr int FLAGS_THREADS = 512;
constexpr int FLAGS_SPAN = FLAGS_THREADS / BRICK / BRICK, FLAGS_SPAN_FLAT = FLAGS_THREADS / BRICK;  // bricks
// Signs of `ni` cells at stride HD from c0 on: bit p = cell p is liquid.
template <class Tp>
__device__ __forceinline__ unsigned column_bits(const void *a, size_t c0, int ni, size_t HD) {
    const Tp *phi = (const Tp *)a;
    Tp v[BRICK];
#pragma unroll
    for (int p = 0; p < BRICK; ++p) v[p] = phi[c0 + (p < ni ? p : 0) * HD];
    unsigned m = 0;
#pragma unroll
    for (int p = 0; p < BRICK; ++p) m |= (unsigned)(v[p] < Tp(0)) << p;
    return m & ((1u << ni) - 1);
}
// The same of the ni + 1 solid nodes of a column (bit p = node p lies in the solid).
template <class Ts, int N = BRICK>
__device__ __forceinline__ unsigned node_bits(const void *a, size_t n0, int ni, size_t stride) {
    const Ts *solid = (const Ts *)a;
    Ts v[N + 1];
#pragma unroll
    for (int p = 0; p <= N; ++p) v[p] = solid[n0 + (p <= ni ? p : 0) * stride];
    unsigned m = 0;
#pragma unroll
    for (int p = 0; p <= N; ++p) m |= (unsigned)(v[p] < Ts(0)) << p;
    return m & ((2u << ni) - 1);
}
static inline int flags_blocks(const FlagsGrid &F) {
    if (F.G.flat) return F.nbx * ((F.nby + FLAGS_SPAN_FLAT - 1) / FLAGS_SPAN_FLAT);
    return F.nbx * F.nby * ((F.nbz + FLAGS_SPAN - 1) / FLAGS_SPAN);
}
__global__ __launch_bounds__(FLAGS_THREADS) void k_flags(GridTable<FlagsGrid> T) {
    // columns of the workgroup with one more on each side: rows along y (one in a 2D grid), contiguous axis
    constexpr int COLS = FLAGS_SPAN * BRICK, WIDE = COLS + 2;
    __shared__ uint8_t around[FLAGS_THREADS + 2 > (BRICK + 2) * WIDE ? FLAGS_THREADS + 2 : (BRICK + 2) * WIDE];
    __shared__ uint16_t nodes[FLAGS_THREADS + 1 > (BRICK + 1) * (COLS + 1) ? FLAGS_THREADS + 1 : (BRICK + 1) * (COLS + 1)];
    __shared__ int bits[FLAGS_SPAN_FLAT];
    int local;
    const int entry = table_grid(T, local);
    if (entry < 0) return;
    const FlagsGrid &F = T.g[entry];
    const GridDesc &G = F.G;
    const int t = threadIdx.x;
    // the workgroup's bricks: (bx, by, bz) on, along z (along y in a 2D grid); its thread's column (j, k), its
    // place in `around` and the column of the border that it also reads (at hat, -1: none)
    int bx, by, bz, j, k, slot, at, row = 0, hj = 0, hk = 0, hat = -1;
    if (G.flat) {
        const int nspan = (F.nby + FLAGS_SPAN_FLAT - 1) / FLAGS_SPAN_FLAT;
        bx = local / nspan, by = (local - bx * nspan) * FLAGS_SPAN_FLAT, bz = 0;
        j = by * BRICK + t, k = 0, slot = t / BRICK, at = t + 1;
        if (t < 2) hj = by * BRICK + (t ? FLAGS_THREADS : -1), hat = t ? FLAGS_THREADS + 1 : 0;
    } else {
        const int nspan = (F.nbz + FLAGS_SPAN - 1) / FLAGS_SPAN, r = local / nspan;
        bx = r / F.nby, by = r - bx * F.nby, bz = (local - r * nspan) * FLAGS_SPAN;
        const int jj = t / COLS, kk = t % COLS;
        j = by * BRICK + jj, k = bz * BRICK + kk, slot = kk / BRICK, row = WIDE;
        at = (jj + 1) * WIDE + kk + 1;
        int a = 0, b = 0;
        if (t < 2 * COLS) {
            a = t < COLS ? 0 : BRICK + 1, b = t % COLS + 1;
        } else if (t < 2 * (COLS + BRICK)) {
            a = t % BRICK + 1, b = t < 2 * COLS + BRICK ? 0 : COLS + 1;
        }
        if (t < 2 * (COLS + BRICK)) hj = by * BRICK + a - 1, hk = bz * BRICK + b - 1, hat = a * WIDE + b;
    }
    const size_t HD = (size_t)((unsigned)G.h * (unsigned)G.d);
    const int i0 = bx * BRICK, ni = min(BRICK, G.w - i0);
    const bool in = j < G.h && k < G.d, hin = hj >= 0 && hj < G.h && hk >= 0 && hk < G.d;
    const size_t c0 = in ? cell_index(G, i0, j, k) : 0;
    unsigned liquid = 0, beyond = 0, border = 0, known = 0;
    if (in) {
        // the column's own cells, and those before and after it along x (bits 0 and 1 of beyond)
        const size_t before = i0 > 0 ? HD : 0, after = i0 + BRICK < G.w ? BRICK * HD : 0;
        if (G.phi64) {
            const double *phi = (const double *)G.phi;
            const double b = phi[c0 - before], a = phi[c0 + after];
            liquid = column_bits<double>(phi, c0, ni, HD);
            beyond = (before && b < 0.0 ? 1 : 0) | (after && a < 0.0 ? 2 : 0);
        } else {
            const float *phi = (const float *)G.phi;
            const float b = phi[c0 - before], a = phi[c0 + after];
            liquid = column_bits<float>(phi, c0, ni, HD);
            beyond = (before && b < 0.0f ? 1 : 0) | (after && a < 0.0f ? 2 : 0);
        }
    }
    if (hat >= 0 && hin) {
        const size_t h0 = cell_index(G, i0, hj, hk);
        border = G.phi64 ? column_bits<double>(G.phi, h0, ni, HD) : column_bits<float>(G.phi, h0, ni, HD);
    }
    around[at] = (uint8_t)liquid;
    if (hat >= 0) around[hat] = (uint8_t)border;
    // solid nodes of the workgroup's columns: its (j, k) and one more on the high sides
    int nat = 0;
    if (G.solid) {
        const int cols = G.flat ? FLAGS_THREADS : COLS, rows = G.flat ? 1 : BRICK + 1;
        for (int q = t; q < rows * (cols + 1); q += FLAGS_THREADS) {
            const int a = G.flat ? 0 : q / (COLS + 1), b = q - a * (COLS + 1);
            const int nj = min(by * BRICK + (G.flat ? b : a), G.h), nk = G.flat ? 0 : min(bz * BRICK + b, G.d);
            const size_t n0 = G.flat ? (size_t)((unsigned)i0 * (unsigned)(G.h + 1) + (unsigned)nj) : node_index(G, i0, nj, nk);
            const size_t stride = G.flat ? (size_t)(G.h + 1) : (size_t)((unsigned)(G.h + 1) * (unsigned)(G.d + 1));
            nodes[q] = (uint16_t)(G.solid64 ? node_bits<double>(G.solid, n0, ni, stride)
                                            : node_bits<float>(G.solid, n0, ni, stride));
        }
        nat = G.flat ? t : t / COLS * (COLS + 1) + t % COLS;
    }
    if (t < FLAGS_SPAN_FLAT) bits[t] = 0;
    __syncthreads();
    if (liquid) {
        const Exist E{true, true};
        const unsigned xm = ((liquid << 1) | (beyond & 1)) & liquid, xp = ((liquid >> 1) | (beyond >> 1) << (BRICK - 1)) & liquid;
        const unsigned am = around[at - 1] & liquid, ap = around[at + 1] & liquid;  // along the contiguous axis
        const unsigned ym = G.flat ? am : around[at - row] & liquid, yp = G.flat ? ap : around[at + row] & liquid;
        const unsigned zm = G.flat ? 0 : am, zp = G.flat ? 0 : ap;
        unsigned unknown = xm | xp | ym | yp | zm | zp;
        if (G.solid) {
            // per face of a cell, from the signs of its corners: whole with none in the solid, shut with all;
            // only the others' areas are formed, until one is open
            const unsigned n00 = nodes[nat], n01 = G.flat ? n00 : nodes[nat + 1];
            const unsigned n10 = G.flat ? nodes[nat + 1] : nodes[nat + COLS + 1], n11 = G.flat ? n10 : nodes[nat + COLS + 2];
            unsigned part[6];
            unknown = 0;
            auto face = [&](int nq, unsigned both, unsigned any, unsigned all) {
                unknown |= both & ~any;
                part[nq] = both & any & ~all;
            };
            auto pair = [](unsigned m) { return m | m >> 1; };
            auto both = [](unsigned m) { return m & m >> 1; };
            face(0, xp, (n00 | n01 | n10 | n11) >> 1, (n00 & n01 & n10 & n11) >> 1);
            face(1, xm, n00 | n01 | n10 | n11, n00 & n01 & n10 & n11);
            face(2, yp, pair(n10 | n11), both(n10 & n11));
            face(3, ym, pair(n00 | n01), both(n00 & n01));
            face(4, zp, pair(n01 | n11), both(n01 & n11));
            face(5, zm, pair(n00 | n10), both(n00 & n10));
            unsigned left = (part[0] | part[1] | part[2] | part[3] | part[4] | part[5]) & ~unknown;
            while (left) {
                const int p = __ffs((int)left) - 1;
                left &= left - 1;
                unsigned faces = 0;
#pragma unroll
                for (int nq = 0; nq < 6; ++nq) faces |= (part[nq] >> p & 1) << nq;
                while (faces) {
                    const int nq = __ffs((int)faces) - 1, dim = nq >> 1, o = (nq & 1) ? 0 : 1;
                    faces &= faces - 1;
                    if (face_area(G, E, dim, i0 + p + (dim == 0) * o, j + (dim == 1) * o, k + (dim == 2) * o) != 0.0f) {
                        unknown |= 1u << p;
                        break;
                    }
                }
            }
        }
        known = unknown;
        atomicOr(&bits[slot], (unknown ? 1 : 0) | 2);
    }
    if (in) {
#pragma unroll
        for (int p = 0; p < BRICK; ++p)
            if (p < ni) F.cflag[c0 + p * HD] = (uint8_t)((liquid >> p & 1) | (known >> p & 1) << 1);
    }
    __syncthreads();
    const int nb = G.flat ? min(FLAGS_SPAN_FLAT, F.nby - by) : min(FLAGS_SPAN, F.nbz - bz);
    if (t < nb) {
        const int y = G.flat ? by + t : by, z = G.flat ? 0 : bz + t;
        F.bflag[((size_t)bx * F.nby + y) * F.nbz + z] = (uint8_t)bits[t];
    }
}

// Matrix-free assembly on the stored bricks of one grid at level 0 (macpressuresolver3.cpp:159-199).
// For an unknown c and each in-bounds neighbour q (+x,-x,+y,-y,+z,-z): with area>0 and rho>0
// the conductance w = dt*area/(dx*dx*rho) joins the diagonal, and couples c to q when q is
// liquid (then q is an unknown too); with area>0 the rhs gains -sgn*area*u/dx.  Stored: the
// low-face couplings gx/gy/gz and dir = the sum of conductances to non-unknown neighbours
// (so diag = dir + sum of the six couplings); dir = -1 marks a non-unknown.
//
// The same block also finishes the brick for the solver: the inverse diagonal the smoothers use
// (k_idiag's arithmetic on the stored FP32 (id32) or FP64 (id64) values, each coupling of a high
// face being the neighbour's low one, formed here from the same samples), the brick's unknown count
// (the count k_idiag forms on the coarse levels), and whether its operator is one
// constant: every cell an unknown, dir = 0, all six couplings and the inverse diagonal equal to the
// brick's first cell's (then BM_UNIFORM and its UniCoef record).
struct OperatorFinish {
    float *id32;      // FP32 inverse diagonal (the mixed V-cycle) or nullptr
    double *id64;     // FP64 inverse diagonal (FP64 V-cycle) or nullptr
    BrickMeta *meta;  // level-0 brick records (BM_UNIFORM is or-ed in)
    UniCoef *uni;
    int *counts;      // unknowns per brick (| UNIFORM_COUNT_BIT)
};
struct OperatorGrid {
    GridDesc G;
    GridLevel GL;
    const uint8_t *cflag;
    const double *warm;
    double rhs_correct;
};
__global__ __launch_bounds__(BLOCK) void k_operator(GridTable<OperatorGrid> T, LevelDesc L, double *dir64, double *gx64,
                                                    double *gy64, double *gz64, float *dir32, float *gx32, float *gy32,
                                                    float *gz32, double *b, double *x, OperatorFinish FIN) {
#pragma clang fp contract(off)
    int local;
    const int entry = table_grid(T, local);
    if (entry < 0) return;
    const OperatorGrid &F = T.g[entry];
    const GridDesc &G = F.G;
    const int br = F.GL.brick_start + local;
    const int t = threadIdx.x;
    const int bx = L.bxyz[3 * br], by = L.bxyz[3 * br + 1], bz = L.bxyz[3 * br + 2];
    const int i = bx * BRICK + (t >> 6), j = by * BRICK + ((t >> 3) & 7), k = bz * BRICK + (t & 7);
    const long c = (long)br * BRICK_CELLS + t;
    const bool inside = i < G.w && j < G.h && k < G.d;
    const bool unknown = inside && (F.cflag[cell_index(G, i, j, k)] & 2);
    double dir = -1.0, g[3] = {0.0, 0.0, 0.0}, rhs = 0.0, x0 = 0.0;
    double gp[3] = {0.0, 0.0, 0.0};  // couplings of the high faces (the neighbours' low ones)
    if (unknown) {
        // the cell's 8 solid corners (4 in a 2D grid), 7 level-set samples and 6 face velocities are loaded at
        // once; each face's area and liquid fraction then use the face functions' arithmetic
        const Exist E = exist_of(G);
        const double dt = G.dt, dx = G.dx;
        const int di[6] = {1, -1, 0, 0, 0, 0}, dj[6] = {0, 0, 1, -1, 0, 0}, dk[6] = {0, 0, 0, 0, 1, -1};
        const int sgn[6] = {1, -1, 1, -1, 1, -1};
        double sc[8];  // solid at node (i + a, j + b, k + c), index (a * 2 + b) * 2 + c
        if (G.solid) {
            size_t nidx[8];
#pragma unroll
            for (int n = 0; n < 8; ++n) {
                const int a = i + (n >> 2), b = j + ((n >> 1) & 1);
                nidx[n] = G.flat ? (size_t)((unsigned)a * (unsigned)(G.h + 1) + (unsigned)b) : node_index(G, a, b, k + (n & 1));
            }
            load_samples<8>(G.solid, G.solid64, nidx, sc);
        }
        // level set at the six neighbours (clamped into the grid: out-of-grid ones go unused) and
        // at the cell (last)
        size_t pidx[7];
        float uf[6];  // velocity at the six faces
#pragma unroll
        for (int nq = 0; nq < 6; ++nq) {
            pidx[nq] = cell_index(G, clampi(i + di[nq], 0, G.w - 1), clampi(j + dj[nq], 0, G.h - 1),
                                  clampi(k + dk[nq], 0, G.d - 1));
            const int dim = nq >> 1, o = (nq & 1) ? 0 : 1;
            uf[nq] = G.flat && dim == 2 ? 0.0f : G.vel[dim][face_index(G, dim, i + (dim == 0) * o, j + (dim == 1) * o, k + (dim == 2) * o)];
        }
        pidx[6] = cell_index(G, i, j, k);
        double ph[7];
        load_samples<7>(G.phi, G.phi64, pidx, ph);
        const double pc = ph[6];
        double dsum = 0.0;
        // the conductance of a whole face between two liquid cells (most of them): dt * 1 / (dx * dx * 1),
        // the same bits without a division per face
        const double whole = dt / (dx * dx);
        bool deep = E.liquid && rho_from_samples(G, E, -1.0, -1.0) == 1.0f;  // liquid all around
#pragma unroll
        for (int n = 0; n < 7; ++n) deep = deep && ph[n] < 0.0;
#pragma unroll
        for (int nq = 0; nq < 6; ++nq) {
            const int qi = i + di[nq], qj = j + dj[nq], qk = k + dk[nq];
            if (qi < 0 || qi >= G.w || qj < 0 || qj >= G.h || qk < 0 || qk >= G.d) continue;
            const int dim = nq >> 1, o = (nq & 1) ? 0 : 1;  // the face lies at offset o along dim
            float area = 1.0f;  // an interior face without solid (face_area's no-solid branch)
            if (G.solid) {
                // face_area's corner order for the face of axis dim at offset o
                double v[4];
                auto n = [&](int a, int b, int c) { return sc[(a * 2 + b) * 2 + c]; };
                if (dim == 0) {
                    v[0] = n(o, 0, 0); v[1] = n(o, 1, 0); v[2] = n(o, 1, 1); v[3] = n(o, 0, 1);
                } else if (dim == 1) {
                    v[0] = n(0, o, 0); v[1] = n(1, o, 0); v[2] = n(1, o, 1); v[3] = n(0, o, 1);
                } else {
                    v[0] = n(0, 0, o); v[1] = n(1, 0, o); v[2] = n(1, 1, o); v[3] = n(0, 1, o);
                }
                area = G.flat ? area_from_ends(G, v[0], v[1]) : area_from_corners(G, v);
            }
            if (area) {
                if (deep && area == 1.0f) {
                    if (nq & 1) g[dim] = whole;
                    else gp[dim] = whole;
                } else {
                    // face_rho: the sample at the face's index cell first, then the one below it
                    const double rho = o ? rho_from_samples(G, E, ph[nq], pc) : rho_from_samples(G, E, pc, ph[nq]);
                    if (rho) {
                        const double value = dt * (double)area / (dx * dx * rho);
                        if (ph[nq] < 0.0) {
                            if (nq & 1) g[dim] = value;
                            else gp[dim] = value;
                        } else {
                            dsum += value;
                        }
                    }
                }
                if (!G.flat) rhs += -sgn[nq] * (double)area * (double)uf[nq] / dx;
            }
            // the 2D module adds the term for every in-bounds neighbour (macpressuresolver2.cpp:176)
            if (G.flat) rhs += -sgn[nq] * (double)area * (double)uf[nq] / dx;
        }
        dir = dsum;
        rhs += F.rhs_correct;
        if (F.warm) x0 = F.warm[cell_index(G, i, j, k)];
    }
    mark_loose(FIN.meta, br, dir != dir);
    dir64[c] = dir;
    gx64[c] = g[0];
    gy64[c] = g[1];
    gz64[c] = g[2];
    b[c] = unknown ? rhs : 0.0;
    x[c] = x0;
    if (dir32) {
        dir32[c] = (float)dir;
        gx32[c] = (float)g[0];
        gy32[c] = (float)g[1];
        gz32[c] = (float)g[2];
    }
    // k_idiag: diag = dir + the six couplings, in the stored type
    float i32 = 0.0f;
    double i64 = 0.0;
    if (dir >= 0) {
        if (FIN.id32) {
            const float d = (float)dir + (((float)g[0] + (float)gp[0]) + ((float)g[1] + (float)gp[1]) +
                                          ((float)g[2] + (float)gp[2]));
            if (d > 0) i32 = 1.0f / d;
        }
        if (FIN.id64) {
            const double d = dir + ((g[0] + gp[0]) + (g[1] + gp[1]) + (g[2] + gp[2]));
            if (d > 0) i64 = 1.0 / d;
        }
    }
    if (FIN.id32) FIN.id32[c] = i32;
    if (FIN.id64) FIN.id64[c] = i64;
    // unknown count and the uniformity vote (the brick's first cell gives the reference values), by ballots
    __shared__ double gref, iref64;
    __shared__ float iref32;
    __shared__ int counted[BLOCK / 64], agreed[BLOCK / 64];
    if (t == 0) {
        gref = g[0];
        iref64 = i64;
        iref32 = i32;
    }
    __syncthreads();
    const double Gu = gref;
    const bool ok = Gu > 0.0 && dir == 0.0 && g[0] == Gu && g[1] == Gu && g[2] == Gu && gp[0] == Gu && gp[1] == Gu &&
                    gp[2] == Gu && (!FIN.id64 || i64 == iref64) && (!FIN.id32 || i32 == iref32);
    const unsigned long long unk = __ballot(dir >= 0), agree = __ballot(ok);
    if ((t & 63) == 0) {
        counted[t >> 6] = __popcll(unk);
        agreed[t >> 6] = agree == ~0ull;
    }
    __syncthreads();
    if (t != 0) return;
    int n = 0, uniform = 1;
#pragma unroll
    for (int w = 0; w < BLOCK / 64; ++w) {
        n += counted[w];
        uniform &= agreed[w];
    }
    {
        if (uniform) {
            atomicOr(&FIN.meta[br].flags, BM_UNIFORM);  // (the bricks beside may mark this one)
            UniCoef u;
            u.g64 = Gu;
            u.id64 = iref64;
            u.g32 = (float)Gu;
            u.id32 = iref32;
            u.pad[0] = u.pad[1] = 0.0f;
            FIN.uni[br] = u;
        }
        FIN.counts[br] = n | (uniform ? UNIFORM_COUNT_BIT : 0);
    }
}

// ------------------------------------------------------------------------------ hierarchy (batch)
// Coarse operator from the piecewise-constant aggregation P0 of the 2x2x2 children: the couplings
// are 1/2 of the Galerkin product (g_H = 1/2 sum of the four fine couplings across the coarse
// face, the usual rediscretisation factor for a 2h grid), the Dirichlet (air) part is kept whole
// (dir_H = sum of the children's dir), which keeps the free-surface condition as strong on the
// coarse grids as on the fine one.  Every child of a coarse cell and every fine face it needs lie
// in one fine brick.
template <class Ti, class To>
__global__ __launch_bounds__(BLOCK) void k_coarsen(LevelDesc Lf, OpDesc<Ti> Af, LevelDesc Lc, To *dir, To *gx, To *gy,
                                                   To *gz) {
    const int br = brick_or_idle(Lc);
    if (br < 0) return;
    const int t = threadIdx.x;
    const GridLevel F = Lf.gl[Lc.meta[br].grid];
    const int I = Lc.bxyz[3 * br] * BRICK + (t >> 6), J = Lc.bxyz[3 * br + 1] * BRICK + ((t >> 3) & 7),
              K = Lc.bxyz[3 * br + 2] * BRICK + (t & 7);
    const long c = (long)br * BRICK_CELLS + t;
    double sdir = 0.0, sg[3] = {0.0, 0.0, 0.0};
    bool any = false, coupled = false;
    const int fi0 = 2 * I, fj0 = 2 * J, fk0 = 2 * K;
    if (fi0 < F.ni && fj0 < F.nj && fk0 < F.nk) {
        const int fb = Lf.bmap[F.bmap_off + ((fi0 >> 3) * F.nby + (fj0 >> 3)) * F.nbz + (fk0 >> 3)];
        if (fb >= 0) {
            for (int a = 0; a < 2; ++a)
                for (int bb = 0; bb < 2; ++bb)
                    for (int cc = 0; cc < 2; ++cc) {
                        const int li = (fi0 + a) & 7, lj = (fj0 + bb) & 7, lk = (fk0 + cc) & 7;
                        const long f = (long)fb * BRICK_CELLS + (li * 8 + lj) * 8 + lk;
                        const double d = (double)Af.dir[f];
                        if (d >= 0.0) {
                            any = true;
                            sdir += d;
                        }
                        coupled = coupled | !(d >= -1.0);
                        if (a == 0) sg[0] += (double)Af.gx[f];
                        if (bb == 0) sg[1] += (double)Af.gy[f];
                        if (cc == 0) sg[2] += (double)Af.gz[f];
                    }
        }
    }
    mark_loose(const_cast<BrickMeta *>(Lc.meta), br, coupled && !any);
    dir[c] = any ? (To)sdir : (To)(coupled ? COUPLED_OUT : -1);
    gx[c] = any ? (To)(0.5 * sg[0]) : (To)0;
    gy[c] = any ? (To)(0.5 * sg[1]) : (To)0;
    gz[c] = any ? (To)(0.5 * sg[2]) : (To)0;
}

// Brick (x, y, z) of grid g on a level, -1 outside the grid or where none is stored.
__device__ __forceinline__ int brick_at(const LevelDesc &L, int g, int x, int y, int z) {
    const GridLevel &gl = L.gl[g];
    if (x < 0 || y < 0 || z < 0 || x >= gl.nbx || y >= gl.nby || z >= gl.nbz) return -1;
    return L.bmap[gl.bmap_off + (x * gl.nby + y) * gl.nbz + z];
}

// Transfer and neighbourhood tables of one level L from the base tables of L and its neighbours
// in the hierarchy (Lf one level finer, Lc one coarser; a table is skipped where its pointer is
// null).  One thread per (brick, slot), 99 slots: 64 of child64 (the finer bricks 2B-1 .. 2B+2
// per axis), 8 of parent8 (the coarser bricks (B+1)/2 - 1 + {0,1} per axis; left at -1 for a grid
// that ends on this level) and 27 of nb27 (B-1 .. B+1 per axis, in k_smooth_k's order).
constexpr int LINK_SLOTS = 64 + 8 + 27;
__global__ __launch_bounds__(256) void k_links(LevelDesc L, LevelDesc Lf, LevelDesc Lc, int *child64, int *parent8,
                                               int *nb27) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int br = t / LINK_SLOTS, q = t - br * LINK_SLOTS;
    if (br >= L.nbricks) return;
    const int g = L.meta[br].grid;
    const int X = L.bxyz[3 * br], Y = L.bxyz[3 * br + 1], Z = L.bxyz[3 * br + 2];
    if (q < 64) {
        if (child64)
            child64[64 * (size_t)br + q] = brick_at(Lf, g, 2 * X - 1 + (q >> 4), 2 * Y - 1 + ((q >> 2) & 3), 2 * Z - 1 + (q & 3));
    } else if (q < 72) {
        if (parent8) {
            const int c = q - 64;
            parent8[8 * (size_t)br + c] =
                L.gl[g].coarsest ? -1
                                 : brick_at(Lc, g, (X + 1) / 2 - 1 + (c >> 2), (Y + 1) / 2 - 1 + ((c >> 1) & 1),
                                            (Z + 1) / 2 - 1 + (c & 1));
        }
    } else if (nb27) {
        const int c = q - 72;
        nb27[27 * (size_t)br + c] = brick_at(L, g, X + c / 9 - 1, Y + (c / 3) % 3 - 1, Z + c % 3 - 1);
    }
}

// The smoothers use a stored inverse diagonal: damped Jacobi is
//   z' = (1 - omega) z + omega * idiag * (rhs + sum_f g_f z_q),
// and idiag = 0 marks a non-unknown (or a cell whose diagonal vanished).
// With counts, the same block also counts the brick's unknowns (dir >= 0), plus UNIFORM_COUNT_BIT
// on BM_UNIFORM bricks.
template <class T>
__global__ __launch_bounds__(BLOCK) void k_idiag(LevelDesc L, OpDesc<T> A, T *__restrict__ idiag, int *counts) {
    const int br = brick_or_idle(L);
    if (br < 0) return;
    const int t = threadIdx.x;
    const long c = (long)br * BRICK_CELLS + t;
    const T dirc = A.dir[c];
    T out = 0;
    if (dirc >= 0) {
        const Nbrs N = load_nbrs(L, br);
        long idx[6];
        nb_index(N, t, idx);
        const T diag = dirc + ((A.gx[c] + ld(A.gx, idx[NB_XP])) + (A.gy[c] + ld(A.gy, idx[NB_YP])) +
                               (A.gz[c] + ld(A.gz, idx[NB_ZP])));
        if (diag > 0) out = T(1) / diag;
    }
    idiag[c] = out;
    if (counts) {
        const int n = __syncthreads_count(dirc >= 0);
        if (t == 0) counts[br] = n | ((L.meta[br].flags & BM_UNIFORM) ? UNIFORM_COUNT_BIT : 0);
    }
}

// ------------------------------------------------------------------------------ Krylov (batch)
// Grid of brick br (no load in a batch of one).
__device__ __forceinline__ int grid_of(const LevelDesc &L, int br) { return L.ngrids > 1 ? L.meta[br].grid : 0; }

// q = A p and p.q partials (FIN_PQ forms alpha = (r.z) / (p.q)).
template <class T>
__global__ __launch_bounds__(BLOCK) void k_apply_dot(LevelDesc L, OpDesc<T> A, const T *__restrict__ p,
                                                     T *__restrict__ q, const SolveScalars *S, const BatchCtl *ctl,
                                                     RedBuf R) {
    __shared__ double lds[32];
    const int br = brick_or_idle(L);
    if (br < 0) return;
    const BrickMeta m = L.meta[br];
    const int t = threadIdx.x;
    const long c = (long)br * BRICK_CELLS + t;
    // single grid: p is loaded before the gate resolves; batch: finished grids load nothing
    if (L.ngrids > 1 && (ctl->all_done || S[m.grid].done)) return;
    const T pc = p[c];
    if (ctl->all_done) return;
    T out = 0;
    double part = 0.0;
    if (m.flags & BM_UNIFORM) {
        const UniT<T> u = uni_load<T>(L, br);
        long idx[6];
        nb_index(nbrs_of(m, br), t, idx);
        out = apply_row_uniform(u.g, p, c, idx, pc);
        part = (double)pc * (double)out;
    } else {
        // every load is issued before the unknown test (the values of other cells are discarded)
        const Nbrs N = nbrs_of(m, br);
        long idx[6];
        nb_index(N, t, idx);
        const T dirc = A.dir[c];
        T diag;
        const T v = apply_row(A, p, c, idx, dirc, pc, diag);
        out = dirc >= 0 ? v : T(0);
        part = dirc >= 0 ? (double)pc * (double)v : 0.0;
    }
    q[c] = out;
    part = block_sum(part, lds);
    store_partials(R, br, part, 0.0);
}

// x += alpha p, r -= alpha q with ||r||_inf and r.r partials (FIN_UPDATE runs the convergence
// test of pcg_solver.h:278-285).
// ZFIRST (preconditioned): also the V-cycle's first sweep from zero, z = omega * idiag * r (k_smooth_first's, which
// read r again in a launch of its own: 7.1 + 4.7 us at 128^3 in FP64, 8.6 here).
template <class T, int ZFIRST>
__global__ __launch_bounds__(BLOCK) void k_cg_update(LevelDesc L, T *__restrict__ x, T *__restrict__ r,
                                                     const T *__restrict__ p, const T *__restrict__ q,
                                                     const SolveScalars *S, const BatchCtl *ctl, RedBuf R,
                                                     const T *__restrict__ idiag, T *__restrict__ z, T omega) {
    __shared__ double lds[32];
    const int br = brick_or_idle(L);
    if (br < 0) return;
    const long c = (long)br * BRICK_CELLS + threadIdx.x;
    // A single grid issues the vectors' loads before the gate's loads resolve (they are wasted
    // only on an iteration past convergence); in a batch, bricks of finished grids load nothing.
    if (L.ngrids > 1 && (ctl->all_done || S[grid_of(L, br)].done)) return;
    const T xv = x[c], pv = p[c], r0 = r[c], qv = q[c];
    T id = T(0);
    bool first = false;
    if (ZFIRST) {
        const BrickMeta m = L.meta[br];
        first = !(m.flags & BM_COARSEST);  // (a grid's last level is its coarse solve's)
        id = (m.flags & BM_UNIFORM) ? uni_load<T>(L, br).id : idiag[c];
    }
    const SolveScalars &Sg = S[grid_of(L, br)];
    if (ctl->all_done || Sg.done) return;
    const T alpha = (T)Sg.alpha;
    x[c] = xv + alpha * pv;
    const T rv = r0 - alpha * qv;
    r[c] = rv;
    if (ZFIRST && first) z[c] = omega * id * rv;
    double mx = fabs((double)rv), sq = (double)rv * (double)rv;
    block_reduce2<true>(mx, sq, lds);
    store_partials(R, br, mx, sq);
}

// r.z partials for the next direction (FIN_RZ forms beta).
template <class T>
__global__ __launch_bounds__(BLOCK) void k_dot_rz(LevelDesc L, const T *__restrict__ r, const T *__restrict__ z,
                                                  const SolveScalars *S, const BatchCtl *ctl, RedBuf R) {
    __shared__ double lds[32];
    const int br = brick_or_idle(L);
    if (br < 0) return;
    if (ctl->all_done || S[grid_of(L, br)].done) return;
    const long c = (long)br * BRICK_CELLS + threadIdx.x;
    const double part = block_sum((double)r[c] * (double)z[c], lds);
    store_partials(R, br, part, 0.0);
}

// p = z + beta p (first: p = z).
template <class T>
__global__ __launch_bounds__(BLOCK) void k_update_p(LevelDesc L, const T *__restrict__ z, T *__restrict__ p,
                                                    const SolveScalars *S, const BatchCtl *ctl, int first) {
    const int br = brick_or_idle(L);
    if (br < 0) return;
    const long c = (long)br * BRICK_CELLS + threadIdx.x;
    // single grid: loads before the gate resolves; batch: finished grids load nothing
    if (L.ngrids > 1 && (ctl->all_done || S[grid_of(L, br)].done)) return;
    const T zv = z[c], pv = first ? T(0) : p[c];
    const SolveScalars &Sg = S[grid_of(L, br)];
    if (ctl->all_done || Sg.done) return;
    p[c] = first ? zv : zv + (T)Sg.beta * pv;
}

constexpr int ROW4_GROUP = BRICK_CELLS / 4;  // threads of a row-4 workgroup of one brick

enum FinOp {
    FIN_PQ = 0,           // alpha = rz / pq
    FIN_UPDATE = 1,       // rinf, rl2, iteration count, convergence test
    FIN_UPDATE_CG = 2,    // FIN_UPDATE plus beta = r.r / rz (unpreconditioned CG)
    FIN_RZ_FIRST = 3,     // rz of the first direction
    FIN_RZ = 4,           // beta = rz_new / rz
    FIN_DEFECT_FIRST = 5, // ||r0|| and the absolute tolerance  (param = relative residual)
    FIN_DEFECT = 6,       // ||r|| only
    FIN_INNER_INIT = 7,   // inner solve: ||r0||, tol = max(param, tol_outer/||r_outer||) * ||r0||,
                          // maxit = the grid's iterations left (0 when its defect correction is done)
    FIN_OUTER = 8         // defect correction: ||r||, iterations += the inner solve's; done when the
                          // defect converged, the iterations ran out or the defect fell by < 10 %
};

// Fresh per-grid scalars (norm, iteration limit; everything else 0) for n grids.
// Iterations without a new minimum of the residual after which an inner FP32 solve of the defect
// correction stops (and the FP64 defect is recomputed).
constexpr int INNER_STALL_LIMIT = 12;

__global__ void k_init_scalars(SolveScalars *S, int n, int norm, int maxit) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n) return;
    SolveScalars v{};
    v.norm = norm;
    v.maxit = maxit;
    S[g] = v;
}

// Resets a control block for a new Krylov solve over ngrids grids (a kernel, so that it orders
// with the work around it and needs no host buffer).
__global__ void k_init_ctl(BatchCtl *ctl, int ngrids) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        ctl->ngrids = ngrids;
        ctl->ndone = 0;
        ctl->all_done = 0;
        ctl->pad = 0;
    }
}

__device__ __forceinline__ void mark_done(SolveScalars &S, BatchCtl *ctl) {
    S.done = 1;
    if (ctl) {
        const int n = atomicAdd(&ctl->ndone, 1) + 1;
        if (n >= ctl->ngrids) ctl->all_done = 1;
    }
}

// The convergence test of pcg_solver.h:278-285 on a grid's updated residual: a = ||r||_inf, b = r.r;
// s0: the scalars before the update.
__device__ __forceinline__ void finish_update(SolveScalars &S, const SolveScalars &s0, double a, double b, BatchCtl *ctl,
                                              bool cg) {
    const double rl2 = sqrt(b);
    S.rinf = a;
    S.rl2 = rl2;
    const int it = s0.iter + 1;
    S.iter = it;
    const double cur = s0.norm == 0 ? a : rl2;
    if (cg) {
        S.beta = b / s0.rz[0];
        S.rz[0] = b;
    }
    // an inner solve whose FP32 residual stops reaching new minima hands back to the FP64
    // defect correction (a consistent singular system, for one, keeps a null-space component
    // of the FP32 rounding that no iteration removes)
    bool stalled = false;
    if (s0.stall_limit > 0) {
        if (cur < s0.rmin) {
            S.rmin = cur;
            S.stall = 0;
        } else {
            const int st = s0.stall + 1;
            S.stall = st;
            stalled = st >= s0.stall_limit;
        }
    }
    if (!(b == b)) {
        S.status = 1;
        mark_done(S, ctl);
    } else if (cur <= s0.tol) {
        S.converged = 1;
        mark_done(S, ctl);
    } else if (it >= s0.maxit || stalled) {
        mark_done(S, ctl);
    }
}

// The sums of a grid's partials are those of 1024 threads (k_finalize): thread t adds the partials t,
// t + 1024, ... of the grid, 64 threads a wavefront's butterfly, and the 16 wavefronts' sums are added
// in order.  The kernels below take them in smaller workgroups, with the same bits.
constexpr int FIN_THREADS = 1024;

// k_finalize's FIN_UPDATE of grid g in a 512-thread workgroup: each thread stands for two.
struct FinUpdate {
    const double *partials;  // nullptr: nothing to do
    SolveScalars *S;
    BatchCtl *ctl;
};
__device__ __forceinline__ void finalize_update(const FinUpdate &F, const LevelDesc &L0, int g) {
    __shared__ double lds[2][FIN_THREADS / 64];
    SolveScalars &S = F.S[g];
    const SolveScalars s0 = S;
    const bool stop = s0.done || F.ctl->all_done;
    int bs = 0, be = L0.nbricks;
    if (L0.ngrids > 1) {
        bs = L0.gl[g].brick_start;
        be = L0.gl[g].brick_end;
    }
    const double2 *pp = reinterpret_cast<const double2 *>(F.partials);
    double a[2] = {0.0, 0.0}, b[2] = {0.0, 0.0};
    constexpr int U = 6;  // 12 loads in flight per thread (a 256^3 grid of 10,000 bricks takes 20)
    for (int i = bs + (int)threadIdx.x; i < be; i += U * FIN_THREADS) {
        double2 v[2][U];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int j = i + u * FIN_THREADS + k * (FIN_THREADS / 2);
                v[k][u] = j < be ? pp[j] : make_double2(0.0, 0.0);
            }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                a[k] = fmax(a[k], v[k][u].x);
                b[k] += v[k][u].y;
            }
    }
    if (stop) return;
    const int w = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const double wa = wave_max(a[k]), wb = wave_sum(b[k]);
        if ((threadIdx.x & 63) == 0) {
            lds[0][w + k * (FIN_THREADS / 128)] = wa;
            lds[1][w + k * (FIN_THREADS / 128)] = wb;
        }
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    double sa = 0.0, sb = 0.0;
    for (int i = 0; i < FIN_THREADS / 64; ++i) {
        sa = fmax(sa, lds[0][i]);
        sb += lds[1][i];
    }
    finish_update(S, s0, sa, sb, F.ctl, false);
}

// The first partials of the n <= FOLD_BRICKS bricks of a single grid, summed by every 128-thread
// workgroup of the kernel that uses the sum, so that no finalize launch (3 to 4 us, most of it its
// boundary and one trip to memory) stands between the producer and it.  load() issues the loads,
// sum() adds; all threads call both.  What all workgroups read together grows with the square of the
// bricks, 8 MB from the L2s at 1024, and the loads of a larger limit cost registers at every size.  Projections to 1e-6
// with k_finalize / with the limit at 1024 / at 4096 (us): 95 bricks 901 / 848 / 856, 774 bricks 1368 / 1319 / 1336,
// 1439 bricks 1593 / 1597 / 1579, 2152 bricks 2162 / 2163 / 2228.
//
// A breakdown that such a kernel finds is recorded in the flags that it tests on entry, by the workgroup of
// brick 0 while others still enter.  So the two wavefronts of a workgroup don't go by flags of their own: sum()
// hands all of them the reading of the first thread (stop), behind its barrier, and a workgroup that
// reads the flags too early forms the same sum and leaves on it.
constexpr int FOLD_BRICKS = 1024;
struct FoldPartials {
    static constexpr int ROUNDS = FOLD_BRICKS / ROW4_GROUP, LDS = 2 * ROUNDS + 1;  // (in doubles)
    double v[ROUNDS];
    int n;
    __device__ __forceinline__ void load(const double *__restrict__ partials, int nb) {
        n = nb;
#pragma unroll
        for (int k = 0; k < ROUNDS; ++k) {
            const int i = k * ROW4_GROUP + (int)threadIdx.x;
            v[k] = i < nb ? partials[2 * i] : 0.0;
        }
    }
    __device__ __forceinline__ double sum(double *lds, bool &stop) const {
        const int w = threadIdx.x >> 6;
        if (threadIdx.x == 0) lds[2 * ROUNDS] = stop ? 1.0 : 0.0;
#pragma unroll
        for (int k = 0; k < ROUNDS; ++k) {
            if (k * ROW4_GROUP >= n) break;
            const double s = wave_sum(v[k]);
            if ((threadIdx.x & 63) == 0) lds[2 * k + w] = s;
        }
        __syncthreads();
        stop = lds[2 * ROUNDS] != 0.0;
        double total = 0.0;
        const int waves = 2 * ((n + ROW4_GROUP - 1) / ROW4_GROUP);
        for (int i = 0; i < waves; ++i) total += lds[i];
        return total;
    }
};

// One block per grid combines the partials of the grid's bricks in brick order and updates the
// grid's scalars.  Grids that finished are left alone (their kernels stored no partials).
// Every load is issued before the done test resolves: a single grid's brick range is the level's
// (no dependent load of its GridLevel), and the grid's scalars are copied in the same round trip,
// so the update after the reduction reads no memory (a chain of four dependent round trips became
// one).  The summation order is the brick order as before.
__global__ __launch_bounds__(1024) void k_finalize(const double *__restrict__ partials, LevelDesc L0,
                                                   SolveScalars *Sarr, BatchCtl *ctl, int op, double param, int iparam,
                                                   const SolveScalars *outer) {
    __shared__ double lds[32];
    const int g = blockIdx.x;
    SolveScalars &S = Sarr[g];
    const SolveScalars s0 = S;
    const bool stop = s0.done || (ctl && ctl->all_done);
    int bs = 0, be = L0.nbricks;
    if (L0.ngrids > 1) {
        const GridLevel G = L0.gl[g];
        bs = G.brick_start;
        be = G.brick_end;
    }
    const bool always = (op == FIN_DEFECT_FIRST || op == FIN_DEFECT || op == FIN_INNER_INIT);
    const bool a_is_max = (op == FIN_UPDATE || op == FIN_UPDATE_CG || op == FIN_DEFECT_FIRST || op == FIN_DEFECT ||
                           op == FIN_INNER_INIT || op == FIN_OUTER);
    double a = 0.0, b = 0.0;
    const double2 *pp = reinterpret_cast<const double2 *>(partials);
    // up to 16 loads in flight per thread (16K bricks per pass), in groups of four that a grid too small for
    // them skips; past the grid's end a thread adds zeros, which change neither the sums nor the maxima (of
    // norms).  A finished grid's partials are stale but in bounds, and its result is dropped below.
    //
    // One workgroup, four wavefronts to a SIMD: bound by their issue.  With all sixteen rounds whatever the size, both
    // values reduced for every operation and the last sum formed by every thread, 9248 bricks took 5.5 us and 1408
    // 4.5 us, here 4.7 and 3.9.
    constexpr int U = 4, GROUPS = 4;
    const int step = (int)blockDim.x;
    for (int i0 = bs; i0 < be; i0 += GROUPS * U * step) {
        double2 v[GROUPS][U];
#pragma unroll
        for (int q = 0; q < GROUPS; ++q) {
            if (i0 + q * U * step >= be) break;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int j = i0 + (q * U + u) * step + (int)threadIdx.x;
                v[q][u] = j < be ? pp[j] : make_double2(0.0, 0.0);
            }
        }
#pragma unroll
        for (int q = 0; q < GROUPS; ++q) {
            if (i0 + q * U * step >= be) break;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                a = a_is_max ? fmax(a, v[q][u].x) : a + v[q][u].x;
                b += v[q][u].y;
            }
        }
    }
    if (!always && stop) return;
    // block_reduce2 for the one thread that needs the result (b: the sums of squares, with the maxima only)
    a = a_is_max ? wave_max(a) : wave_sum(a);
    if (a_is_max) b = wave_sum(b);
    if ((threadIdx.x & 63) == 0) {
        lds[threadIdx.x >> 6] = a;
        lds[16 + (threadIdx.x >> 6)] = b;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    a = b = 0.0;
    const int nw = step >> 6;
    for (int w = 0; w < nw; ++w) {
        a = a_is_max ? fmax(a, lds[w]) : a + lds[w];
        b += lds[16 + w];
    }
    switch (op) {
    case FIN_PQ: {
        S.pq = a;
        const double al = s0.rz[0] / a;
        S.alpha = al;
        if (!(al == al) || al - al != 0.0) {
            S.status = 1;
            mark_done(S, ctl);
        }
        break;
    }
    case FIN_UPDATE:
    case FIN_UPDATE_CG:
        finish_update(S, s0, a, b, ctl, op == FIN_UPDATE_CG);
        break;
    case FIN_RZ_FIRST:
    case FIN_RZ: {
        S.beta = op == FIN_RZ_FIRST ? 0.0 : a / s0.rz[0];
        S.rz[0] = a;
        if (!(a == a)) {
            S.status = 1;
            mark_done(S, ctl);
        } else if (op == FIN_RZ_FIRST && a == 0.0) {
            mark_done(S, ctl);
        }
        break;
    }
    case FIN_DEFECT_FIRST:
    case FIN_DEFECT:
    case FIN_INNER_INIT: {
        const double rl2 = sqrt(b);
        S.rinf = a;
        S.rl2 = rl2;
        if (op != FIN_DEFECT) {
            S.r0inf = a;
            S.r0l2 = rl2;
            const double r0 = s0.norm == 0 ? a : rl2;
            double rel = param;
            int maxit = s0.maxit;
            if (op == FIN_INNER_INIT) {
                const SolveScalars &O = outer[g];
                const double ocur = O.norm == 0 ? O.rinf : O.rl2;
                rel = ocur > 0.0 ? fmax(param, O.tol / ocur) : param;
                maxit = (O.done || ocur <= O.tol || O.status) ? 0 : max(1, O.maxit - O.iter);
                S.maxit = maxit;
                S.rmin = r0;
                S.stall = 0;
                S.stall_limit = INNER_STALL_LIMIT;
            }
            S.tol = rel * r0;
            S.iter = 0;
            S.done = 0;
            const bool bad = !(b == b);
            S.status = bad ? 1 : 0;
            S.converged = (r0 == 0.0) ? 1 : 0;
            if (r0 == 0.0 || bad || maxit <= 0) mark_done(S, ctl);
        }
        break;
    }
    case FIN_OUTER: {
        const SolveScalars &I = outer[g];
        const double prev = s0.norm == 0 ? s0.rinf : s0.rl2;
        const double rl2 = sqrt(b);
        S.rinf = a;
        S.rl2 = rl2;
        const int it = s0.iter + I.iter;
        S.iter = it;
        const double cur = s0.norm == 0 ? a : rl2;
        if (!(b == b) || I.status) {
            S.status = 1;
            mark_done(S, ctl);
        } else if (cur <= s0.tol) {
            S.converged = 1;
            mark_done(S, ctl);
        } else if (it >= s0.maxit || cur > 0.9 * prev) {
            mark_done(S, ctl);
        }
        break;
    }
    default:
        break;
    }
}

// ------------------------------------------------------------------------------ V-cycle (batch)
// z = omega * idiag * rhs (one damped-Jacobi sweep from a zero guess).
// FINEST: 1 on the finest level (a distinct symbol for profiling), 0 on coarse levels.
template <class T, int FINEST>
__global__ __launch_bounds__(BLOCK) void k_smooth_first(LevelDesc L, const T *__restrict__ idiag,
                                                        const T *__restrict__ rhs, T *__restrict__ z, T omega,
                                                        Gate Q) {
    const int br = brick_or_idle(L);
    if (br < 0) return;
    const BrickMeta m = L.meta[br];
    if (all_done(Q) || skip_smooth(Q, L, m)) return;
    const long c = (long)br * BRICK_CELLS + threadIdx.x;
    const T id = (m.flags & BM_UNIFORM) ? uni_load<T>(L, br).id : idiag[c];
    z[c] = omega * id * rhs[c];
}

// Two damped-Jacobi sweeps from a zero guess in one pass: the first sweep's values at the
// neighbours, omega * idiag_q * rhs_q, are formed on the fly.
template <class T, int FINEST>
__global__ __launch_bounds__(BLOCK) void k_smooth2(LevelDesc L, OpDesc<T> A, const T *__restrict__ idiag,
                                                   const T *__restrict__ rhs, T *__restrict__ z, T omega,
                                                   Gate Q) {
    const int br = brick_or_idle(L);
    if (br < 0) return;
    const BrickMeta m = L.meta[br];
    if (all_done(Q) || skip_smooth(Q, L, m)) return;
    const int t = threadIdx.x;
    const long c = (long)br * BRICK_CELLS + t;
    if (m.flags & BM_UNIFORM) {
        const UniT<T> u = uni_load<T>(L, br);
        const Nbrs N = nbrs_of(m, br);
        long idx[6];
        nb_index(N, t, idx);
        // neighbours in the brick share its inverse diagonal; the others are read
        auto z1 = [&](long i) {
            return i >= 0 ? omega * ((i >= N.base && i < N.base + BRICK_CELLS) ? u.id : idiag[i]) * rhs[i] : T(0);
        };
        const T off = u.g * z1(idx[NB_XM]) + u.g * z1(idx[NB_XP]) + u.g * z1(idx[NB_YM]) + u.g * z1(idx[NB_YP]) +
                      u.g * z1(idx[NB_ZM]) + u.g * z1(idx[NB_ZP]);
        const T r = rhs[c];
        z[c] = (T(1) - omega) * (omega * u.id * r) + omega * u.id * (r + off);
        return;
    }
    const T id = idiag[c];
    T out = 0;
    if (id > 0) {
        const Nbrs N = nbrs_of(m, br);
        long idx[6];
        nb_index(N, t, idx);
        auto z1 = [&](long i) { return i >= 0 ? omega * idiag[i] * rhs[i] : T(0); };
        const T gxp = ld(A.gx, idx[NB_XP]), gyp = ld(A.gy, idx[NB_YP]), gzp = ld(A.gz, idx[NB_ZP]);
        const T off = A.gx[c] * z1(idx[NB_XM]) + gxp * z1(idx[NB_XP]) + A.gy[c] * z1(idx[NB_YM]) +
                      gyp * z1(idx[NB_YP]) + A.gz[c] * z1(idx[NB_ZM]) + gzp * z1(idx[NB_ZP]);
        const T r = rhs[c];
        out = (T(1) - omega) * (omega * id * r) + omega * id * (r + off);
    }
    z[c] = out;
}

// zout = (1 - omega) zin + omega idiag (rhs + offdiag(zin)) with the rhs.zout partial of each brick: the
// finest level's last post-smoothing sweep of an FP64 cycle yields r.z of the preconditioned CG for free.
// One brick per workgroup (its reduction costs two barriers per brick), one cell per thread: the
// partial keeps the order of the sum over the brick.
template <class T>
__global__ __launch_bounds__(BLOCK) void k_jacobi_dot(LevelDesc L, OpDesc<T> A, const T *__restrict__ idiag,
                                                      const T *__restrict__ rhs, const T *__restrict__ zin,
                                                      T *__restrict__ zout, T omega, Gate Q, RedBuf R) {
    __shared__ double lds[32];
    const int br = brick_or_idle(L);
    if (br < 0) return;
    const BrickMeta m = L.meta[br];
    if (all_done(Q) || skip_smooth(Q, L, m)) return;
    const int t = threadIdx.x;
    const long c = (long)br * BRICK_CELLS + t;
    long idx[6];
    nb_index(nbrs_of(m, br), t, idx);
    const T r = rhs[c];
    T out;
    double part;
    if (m.flags & BM_UNIFORM) {
        const UniT<T> u = uni_load<T>(L, br);
        out = (T(1) - omega) * zin[c] + omega * u.id * (r + offdiag_uniform(u.g, zin, idx));
        part = (double)r * (double)out;
    } else {
        // every load is issued before the unknown test (the values of other cells are discarded)
        const T id = idiag[c];
        const T v = (T(1) - omega) * zin[c] + omega * id * (r + offdiag_sum(A, zin, c, idx));
        out = id > 0 ? v : T(0);
        part = id > 0 ? (double)r * (double)v : 0.0;
    }
    zout[c] = out;
    part = block_sum(part, lds);
    store_partials(R, br, part, 0.0);
}

// ---- Sweeps on cell rows: four consecutive cells (one float4 along z) per thread, 128
// threads per brick.  Lane q of a brick holds the cells (q >> 4, (q >> 1) & 7, 4h .. 4h + 3) with
// h = q & 1; the two lanes of a row are neighbours in the wavefront and swap their edge values, so
// only the row's two end cells read a value across the brick's z faces.  A quarter of the load
// instructions of the one-cell form, and 16-byte accesses.
constexpr int ROW4_THREADS = ROW4_GROUP;

__device__ __forceinline__ float4 ld4(const float *__restrict__ a, long i) {
    return *reinterpret_cast<const float4 *>(a + i);
}
__device__ __forceinline__ void unpack4(const float4 v, float o[4]) {
    o[0] = v.x;
    o[1] = v.y;
    o[2] = v.z;
    o[3] = v.w;
}
// Four consecutive values (16-byte loads: one float4 or two double2).
__device__ __forceinline__ void load4(const float *__restrict__ a, long i, float o[4]) { unpack4(ld4(a, i), o); }
__device__ __forceinline__ void load4(const double *__restrict__ a, long i, double o[4]) {
    const double2 u = *reinterpret_cast<const double2 *>(a + i), w = *reinterpret_cast<const double2 *>(a + i + 2);
    o[0] = u.x;
    o[1] = u.y;
    o[2] = w.x;
    o[3] = w.y;
}
__device__ __forceinline__ void store4(float *__restrict__ a, long i, const float v[4]) {
    *reinterpret_cast<float4 *>(a + i) = make_float4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ void store4(double *__restrict__ a, long i, const double v[4]) {
    *reinterpret_cast<double2 *>(a + i) = make_double2(v[0], v[1]);
    *reinterpret_cast<double2 *>(a + i + 2) = make_double2(v[2], v[3]);
}

// The value of the pair's other lane (q ^ 1), a register move.
__device__ __forceinline__ float swap_pairs(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), DPP_QUAD_1032, 0xF, 0xF, true));
}
__device__ __forceinline__ double swap_pairs(double v) { return dpp_move<DPP_QUAD_1032>(v); }

// The six neighbour rows of lane q's cells: x and y neighbours as whole rows (index of their first
// cell), z neighbours as the row shifted by one cell.
//
// On the coarse levels a wavefront has its SIMD nearly to itself, and a kernel's time is its longest
// chain of instructions and round trips: the indices are formed by selects and always in range, so that no load
// waits behind a branch; where no brick is stored (out*) the value is set to 0 afterwards.
struct Row4Nbrs {
    long c, ixm, ixp, iym, iyp, iz;  // iz: the end cell across the z face (k = -1 for h = 0, 8 for h = 1)
    bool outxm, outxp, outym, outyp, outz;
    bool edge;  // any of them, on any lane of the brick
    int h;
};
__device__ __forceinline__ Row4Nbrs row4_nbrs(const BrickMeta &m, int br, int q) {
    Row4Nbrs N;
    const int li = q >> 4, lj = (q >> 1) & 7, h = q & 1;
    const int o = li * 64 + lj * 8 + 4 * h;
    const long own = (long)br * BRICK_CELLS;
    auto base = [&](int d) { return m.nbr[d] >= 0 ? (long)m.nbr[d] * BRICK_CELLS : own; };
    // (both sides formed before the choice: a select, not a branch)
    const long xm = base(NB_XM) + 448, xp = base(NB_XP) - 448, ym = base(NB_YM) + 56, yp = base(NB_YP) - 56;
    const long zm = base(NB_ZM) + 7, zp = base(NB_ZP) - 4;
    const long xl = own - 64, xh = own + 64, yl = own - 8, yh = own + 8;
    const int nzm = m.nbr[NB_ZM], nzp = m.nbr[NB_ZP];
    N.h = h;
    N.c = own + o;
    N.ixm = (li > 0 ? xl : xm) + o;
    N.ixp = (li < 7 ? xh : xp) + o;
    N.iym = (lj > 0 ? yl : ym) + o;
    N.iyp = (lj < 7 ? yh : yp) + o;
    N.iz = (h ? zp : zm) + o;
    N.outxm = li == 0 && m.nbr[NB_XM] < 0;
    N.outxp = li == 7 && m.nbr[NB_XP] < 0;
    N.outym = lj == 0 && m.nbr[NB_YM] < 0;
    N.outyp = lj == 7 && m.nbr[NB_YP] < 0;
    N.outz = (h ? nzp : nzm) < 0;
    N.edge = (m.nbr[NB_XM] | m.nbr[NB_XP] | m.nbr[NB_YM] | m.nbr[NB_YP] | m.nbr[NB_ZM] | m.nbr[NB_ZP]) < 0;
    return N;
}
template <class T>
__device__ __forceinline__ void zero4(bool out, T v[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = out ? T(0) : v[j];
}

// The values of v at the six neighbours of the lane's four cells (0 where no brick is stored): the loads,
// and what follows once they are there (row4_join), apart so that other loads can be issued in between.
template <class T>
struct Row4Raw {
    T c[4], xm[4], xp[4], ym[4], yp[4], end;
};
template <class T>
struct Row4Vals {
    T c[4], xm[4], xp[4], ym[4], yp[4], zm[4], zp[4];
};
template <class T>
__device__ __forceinline__ Row4Raw<T> row4_load(const T *__restrict__ v, const Row4Nbrs &N) {
    Row4Raw<T> o;
    load4(v, N.c, o.c);
    load4(v, N.ixm, o.xm);
    load4(v, N.ixp, o.xp);
    load4(v, N.iym, o.ym);
    load4(v, N.iyp, o.yp);
    o.end = v[N.iz];
    return o;
}
template <class T>
__device__ __forceinline__ Row4Vals<T> row4_join(Row4Raw<T> r, const Row4Nbrs &N) {
    if (N.edge) {
        zero4(N.outxm, r.xm);
        zero4(N.outxp, r.xp);
        zero4(N.outym, r.ym);
        zero4(N.outyp, r.yp);
        r.end = N.outz ? T(0) : r.end;
    }
    Row4Vals<T> o;
    // lane swap: h = 0 receives the cell k = 4 of its partner, h = 1 the cell k = 3
    const T swap = swap_pairs(N.h ? r.c[0] : r.c[3]);
    o.zm[0] = N.h ? swap : r.end;
    o.zp[3] = N.h ? r.end : swap;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        o.c[j] = r.c[j];
        o.xm[j] = r.xm[j];
        o.xp[j] = r.xp[j];
        o.ym[j] = r.ym[j];
        o.yp[j] = r.yp[j];
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        o.zm[j + 1] = r.c[j];
        o.zp[j] = r.c[j + 1];
    }
    return o;
}
template <class T>
__device__ __forceinline__ Row4Vals<T> row4_vals(const T *__restrict__ v, const Row4Nbrs &N) {
    return row4_join(row4_load(v, N), N);
}

// The couplings of the lane's cells: low faces from the cell itself, high faces from the next cell
// along each axis (0 where no brick is stored).
template <class T>
struct Row4Coef {
    T gxm[4], gym[4], gzm[4], gxp[4], gyp[4], gzp[4];
};
template <class T>
struct Row4CoefRaw {
    T gxm[4], gym[4], gzm[4], gxp[4], gyp[4], end;
};
template <class T>
__device__ __forceinline__ Row4CoefRaw<T> row4_coef_load(const OpDesc<T> &A, const Row4Nbrs &N) {
    Row4CoefRaw<T> o;
    load4(A.gx, N.c, o.gxm);
    load4(A.gy, N.c, o.gym);
    load4(A.gz, N.c, o.gzm);
    load4(A.gx, N.ixp, o.gxp);
    load4(A.gy, N.iyp, o.gyp);
    o.end = A.gz[N.iz];  // (h = 1: the coupling across k = 8)
    return o;
}
template <class T>
__device__ __forceinline__ Row4Coef<T> row4_coef_join(Row4CoefRaw<T> r, const Row4Nbrs &N) {
    if (N.edge) {
        zero4(N.outxp, r.gxp);
        zero4(N.outyp, r.gyp);
        r.end = N.outz ? T(0) : r.end;
    }
    Row4Coef<T> o;
    const T swap = swap_pairs(r.gzm[0]);  // h = 0: the partner's k = 4
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        o.gxm[j] = r.gxm[j];
        o.gym[j] = r.gym[j];
        o.gzm[j] = r.gzm[j];
        o.gxp[j] = r.gxp[j];
        o.gyp[j] = r.gyp[j];
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) o.gzp[j] = r.gzm[j + 1];
    o.gzp[3] = N.h ? r.end : swap;
    return o;
}
template <class T>
__device__ __forceinline__ Row4Coef<T> row4_coef(const OpDesc<T> &A, const Row4Nbrs &N) {
    return row4_coef_join(row4_coef_load(A, N), N);
}

// One sweep of the lane's four cells (k_jacobi_dot's arithmetic per cell); DOT adds rhs.zout of the
// unknowns, in cell order, to part.
template <int DOT, class T>
__device__ __forceinline__ void jacobi_row4(const LevelDesc &L, const OpDesc<T> &A, const T *__restrict__ idiag,
                                            const T *__restrict__ rhs, const T *__restrict__ zin,
                                            T *__restrict__ zout, T omega, int br, const BrickMeta &m, int q,
                                            double &part) {
    const Row4Nbrs N = row4_nbrs(m, br, q);
    const Row4Raw<T> raw = row4_load(zin, N);
    T r[4], out[4];
    load4(rhs, N.c, r);
    if (m.flags & BM_UNIFORM) {
        const UniT<T> u = uni_load<T>(L, br);
        const Row4Vals<T> z = row4_join(raw, N);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const T off = u.g * z.xm[j] + u.g * z.xp[j] + u.g * z.ym[j] + u.g * z.yp[j] + u.g * z.zm[j] +
                              u.g * z.zp[j];
            out[j] = (T(1) - omega) * z.c[j] + omega * u.id * (r[j] + off);
            if (DOT) part += (double)r[j] * (double)out[j];
        }
    } else {
        const Row4CoefRaw<T> graw = row4_coef_load(A, N);
        T id[4];
        load4(idiag, N.c, id);
        const Row4Vals<T> z = row4_join(raw, N);
        const Row4Coef<T> g = row4_coef_join(graw, N);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const T off = g.gxm[j] * z.xm[j] + g.gxp[j] * z.xp[j] + g.gym[j] * z.ym[j] + g.gyp[j] * z.yp[j] +
                              g.gzm[j] * z.zm[j] + g.gzp[j] * z.zp[j];
            const T v = (T(1) - omega) * z.c[j] + omega * id[j] * (r[j] + off);
            out[j] = id[j] > 0 ? v : T(0);
            if (DOT) part += id[j] > 0 ? (double)r[j] * (double)v : 0.0;
        }
    }
    store4(zout, N.c, out);
}

// Sweep: workgroups take 4 (coarse levels: 1) consecutive bricks per virtual block (virtual blocks
// vb = blockIdx.x + k * gridDim.x < nvirt, nvirt a multiple of 8, XCD-preserving); each wavefront
// works alone on half a brick (no barrier).  Bound by the latency of its loads: four cells per lane keep
// the brick's seven reads of z in 16-byte loads with a quarter of the index work.  FP64 at 128^3: 8.5 us
// with one cell per lane, 7.8 us here (residual 7.9 to 7.4, coarse levels 4.2 to 4.0).
template <int FINEST, class T>
__global__ __launch_bounds__(BLOCK) void k_jacobi4(LevelDesc L, OpDesc<T> A, const T *__restrict__ idiag,
                                                   const T *__restrict__ rhs, const T *__restrict__ zin,
                                                   T *__restrict__ zout, T omega, Gate Q, int nvirt) {
    if (all_done(Q)) return;
    constexpr int BPB = FINEST ? BLOCK / ROW4_THREADS : 1;
    const int slot = FINEST ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x / ROW4_THREADS)) : 0;
    const int q = threadIdx.x % ROW4_THREADS;
    for (int vb = blockIdx.x; vb < nvirt; vb += gridDim.x) {
        const int br = BPB * xcd_brick(vb, nvirt) + slot;
        if (br >= L.nbricks) continue;
        const BrickMeta m = L.meta[br];
        if (skip_smooth(Q, L, m)) continue;
        double part = 0.0;
        jacobi_row4<0, T>(L, A, idiag, rhs, zin, zout, omega, br, m, q, part);
    }
}

// The finest level's last post-smoothing sweep with the rhs.z partial of each brick: one brick
// per 128-thread workgroup.
__global__ __launch_bounds__(ROW4_THREADS) void k_jacobi4_dot(LevelDesc L, OpDesc<float> A,
                                                              const float *__restrict__ idiag,
                                                              const float *__restrict__ rhs,
                                                              const float *__restrict__ zin, float *__restrict__ zout,
                                                              float omega, Gate Q, RedBuf R) {
    __shared__ double lds[ROW4_THREADS / 64];
    const int br = brick_or_idle(L);
    if (br < 0) return;
    const BrickMeta m = L.meta[br];
    if (all_done(Q) || skip_smooth(Q, L, m)) return;
    double part = 0.0;
    jacobi_row4<1, float>(L, A, idiag, rhs, zin, zout, omega, br, m, threadIdx.x, part);
    part = wave_sum(part);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = part;
    __syncthreads();
    if (threadIdx.x == 0) {
        double sum = 0.0;
#pragma unroll
        for (int w = 0; w < ROW4_THREADS / 64; ++w) sum += lds[w];
        R.partials[2 * br + 0] = sum;
        R.partials[2 * br + 1] = 0.0;
    }
}

// ---- Brick-local smoother (finest level, FP32): z += M_b (rhs - A z), where M_b applies
// LOCAL_SGS_SWEEPS symmetric red-black Gauss-Seidel sweeps from zero to the brick's own operator
// (its couplings to cells in other bricks dropped, the diagonal whole), i.e. the half-sweeps red,
// black, red, ..., red.  Across bricks it is block Jacobi; inside a brick, Gauss-Seidel.  M_b is
// symmetric, so the V-cycle built on it is a symmetric preconditioner.  One pass over the level's
// arrays per application, like one Jacobi sweep, smoothing about as much as three.  The coarse
// levels use it too (three sweeps per application): there the pre-smoothing from zero runs inside
// the restriction that forms the level's right-hand side (k_restrict_pre).
constexpr int LOCAL_SGS_SWEEPS = 2;         // finest level: the default (2 or 3, a tuned control)
constexpr int LOCAL_SGS_SWEEPS_COARSE = 3;  // coarse levels (one application per smoothing step)

// Row4Coef of a BM_UNIFORM brick.
__device__ __forceinline__ Row4Coef<float> row4_uniform(float g) {
    Row4Coef<float> u;
#pragma unroll
    for (int j = 0; j < 4; ++j) u.gxm[j] = u.gxp[j] = u.gym[j] = u.gyp[j] = u.gzm[j] = u.gzp[j] = g;
    return u;
}

// One cell of a lane in the brick-local sweep: its couplings to the x and y neighbours, the weights of
// the z terms (the two own cells of the other group and the partner
// lane's swapped value, see sgs_cells) and its inverse diagonal.
struct SgsCell {
    float ax_m, ax_p, ay_m, ay_p;
    float za, zb, zs;
    float id;
};

// The brick-local sweep on the brick of a 128-thread group (lane q: cells 4q .. 4q+3 of the brick, the
// storage order).
//
// Cell j of the lane has colour col0 ^ (j & 1) (col0 = (li + lj) & 1), so each half-sweep updates
// two cells of every lane: group P (j = col0, col0 + 2) in the even half-sweeps (the first one, from
// zero, included), group Q (j = 1 - col0, 3 - col0) in the odd ones.  Held by group, the update has
// no divergent branch (adjacent lanes have opposite col0, so a branch on the colour would run both
// sides in every wavefront), and the neighbours of an updated cell are fixed registers:
//  - y: the lane two below / above in the same 16-lane row has the opposite col0, so the same cell
//    there belongs to the other group at the same position: one DPP row shift per value (0 outside
//    the row: lj = 0 / 7, outside the brick);
//  - z: the lane's own cells of the other group, and at the row's ends the partner lane's
//    (q ^ 1, same col0) by a DPP lane swap; the weights za, zb, zs place the two couplings;
//  - x: lanes q -+ 16 (other wavefront at li = 3 / 4), through LDS.  Their col0 is opposite too, so the
//    neighbours of a group's two cells are the other group's two of that lane: LDS holds each group as
//    one pair of floats per lane, and a half-sweep writes one pair and reads two (8-byte accesses; one
//    slot per cell took twice the LDS instructions and a select for every address).
// The sweeps take 0 for the cells across the brick's faces: along y from the DPP shift, along x from a
// slot of zeros past the group's pairs, along z by a zero weight.  So the couplings need no selects.
// The sums use fused multiply-adds in a fixed order.
constexpr int DPP_ROW_SHR2 = 0x112, DPP_ROW_SHL2 = 0x102, DPP_SWAP_PAIRS = 0xB1;  // quad_perm [1,0,3,2]
template <int CTRL>
__device__ __forceinline__ float sgs_dpp(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}

// A lane's four cells by group: p0, p1 (group P), q0, q1 (group Q); from the row and back.
struct SgsRow {
    float p0, p1, q0, q1;
};
__device__ __forceinline__ SgsRow sgs_group(const float v[4], bool c1) {
    return SgsRow{c1 ? v[1] : v[0], c1 ? v[3] : v[2], c1 ? v[0] : v[1], c1 ? v[2] : v[3]};
}
__device__ __forceinline__ void sgs_ungroup(const SgsRow &g, bool c1, float v[4]) {
    v[0] = c1 ? g.q0 : g.p0;
    v[1] = c1 ? g.p0 : g.q0;
    v[2] = c1 ? g.q1 : g.p1;
    v[3] = c1 ? g.p1 : g.q1;
}
__device__ __forceinline__ bool sgs_col1(int q) { return (((q >> 4) + (q >> 1)) & 1) != 0; }

struct SgsCells {
    SgsCell P0, P1, Q0, Q1;
};

// Adds the couplings times the neighbours of a group's cells a, b, the other group being (v0, v1), in
// the sweep's order: x, y, z.  The terms of other lanes (y: rows -+2; z: the pair's swap) use the
// multiply-add's own DPP operand.  The compiler moves a DPP
// value to a register first, 6 of 28 instructions of a half-sweep, and these kernels are bound by
// their issue.  The wait states cover a value written just before.
__device__ __forceinline__ void sgs_pair(const SgsCell &a, const SgsCell &b, float &accA, float &accB, float2 xm,
                                         float2 xp, float v0, float v1) {
    accA = __builtin_fmaf(a.ax_m, xm.x, accA);
    accB = __builtin_fmaf(b.ax_m, xm.y, accB);
    accA = __builtin_fmaf(a.ax_p, xp.x, accA);
    accB = __builtin_fmaf(b.ax_p, xp.y, accB);
    asm volatile("s_nop 1\n\t"
        "v_fmac_f32_dpp %0, %2, %4 row_shr:2 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
        "v_fmac_f32_dpp %1, %3, %6 row_shr:2 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
        "v_fmac_f32_dpp %0, %2, %5 row_shl:2 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
        "v_fmac_f32_dpp %1, %3, %7 row_shl:2 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
        "v_fmac_f32 %0, %2, %8\n\t"
        "v_fmac_f32 %1, %2, %11\n\t"
        "v_fmac_f32 %0, %3, %9\n\t"
        "v_fmac_f32 %1, %3, %12\n\t"
        "v_fmac_f32_dpp %0, %3, %10 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
        "v_fmac_f32_dpp %1, %2, %13 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf bound_ctrl:0"
        : "+&v"(accA), "+&v"(accB)
        : "v"(v0), "v"(v1), "v"(a.ay_m), "v"(a.ay_p), "v"(b.ay_m), "v"(b.ay_p), "v"(a.za), "v"(a.zb), "v"(a.zs),
          "v"(b.za), "v"(b.zb), "v"(b.zs));
}

// The lane's cells by group from its couplings and inverse diagonals.
// The lane's choice between its cells is made on loaded values (one select per field), never on an
// array index: an index chosen per lane would keep the arrays in memory (LDS, addressed through the
// dispatch packet), on the critical path of every launch.
__device__ __forceinline__ SgsCells sgs_cells(const Row4Coef<float> &c, const float id[4], int q) {
    const bool c1 = sgs_col1(q);
    float gxm[4], gxp[4], gym[4], gyp[4], gzm[4], gzp[4], idv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        gxm[j] = c.gxm[j];
        gxp[j] = c.gxp[j];
        gym[j] = c.gym[j];
        gyp[j] = c.gyp[j];
        gzm[j] = c.gzm[j];
        gzp[j] = c.gzp[j];
        idv[j] = id[j];
    }
    if (q & 1) gzp[3] = 0.0f;
    else gzm[0] = 0.0f;
    // cell ja when col0 = 0, jb when col0 = 1, with the z weights of each case
    auto cell_of = [&](int ja, float za_a, float zb_a, float zs_a, int jb, float za_b, float zb_b, float zs_b) {
        SgsCell o;
        o.ax_m = c1 ? gxm[jb] : gxm[ja];
        o.ax_p = c1 ? gxp[jb] : gxp[ja];
        o.ay_m = c1 ? gym[jb] : gym[ja];
        o.ay_p = c1 ? gyp[jb] : gyp[ja];
        o.za = c1 ? za_b : za_a;
        o.zb = c1 ? zb_b : zb_a;
        o.zs = c1 ? zs_b : zs_a;
        o.id = c1 ? idv[jb] : idv[ja];
        return o;
    };
    // group P: cells 0, 2 (col0 = 0) or 1, 3 (col0 = 1); group Q: the others.  For col0 = 0:
    //   P0 = cell 0: z- partner's cell 3 (= its Q1), z+ cell 1 (Q0)
    //   P1 = cell 2: z- cell 1 (Q0), z+ cell 3 (Q1)
    //   Q0 = cell 1: z- cell 0 (P0), z+ cell 2 (P1)
    //   Q1 = cell 3: z- cell 2 (P1), z+ partner's cell 0 (= its P0)
    // and for col0 = 1:
    //   P0 = cell 1: z- cell 0 (Q0), z+ cell 2 (Q1)
    //   P1 = cell 3: z- cell 2 (Q1), z+ partner's cell 0 (= its Q0)
    //   Q0 = cell 0: z- partner's cell 3 (= its P1), z+ cell 1 (P0)
    //   Q1 = cell 2: z- cell 1 (P0), z+ cell 3 (P1)
    // P0 and P1 take the swap of Q1 and Q0, Q0 and Q1 the swap of P1 and P0.
    return SgsCells{cell_of(0, gzp[0], 0.0f, gzm[0], 1, gzm[1], gzp[1], 0.0f),
                    cell_of(2, gzm[2], gzp[2], 0.0f, 3, 0.0f, gzm[3], gzp[3]),
                    cell_of(1, gzm[1], gzp[1], 0.0f, 0, gzp[0], 0.0f, gzm[0]),
                    cell_of(3, 0.0f, gzm[3], gzp[3], 2, gzm[2], gzp[2], 0.0f)};
}

// M_b r (K sweeps from zero).  lds: SGS_PAIRS pairs per group.  Every lane of the workgroup must call it
// (barriers, DPP).
constexpr int SGS_PAIRS = ROW4_THREADS + 1, SGS_LDS = 4 * SGS_PAIRS;  // (in floats)
template <int K>
__device__ __forceinline__ SgsRow sgs_sweeps(const SgsCells &C, const SgsRow &r, float2 *lds, int q) {
    const int qm = q >= 16 ? q - 16 : ROW4_THREADS, qp = q < ROW4_THREADS - 16 ? q + 16 : ROW4_THREADS;
    float2 *const lp = lds, *const lq = lds + SGS_PAIRS;
    // the first half-sweep, from zero: no neighbour values yet
    SgsRow e{C.P0.id * r.p0, C.P1.id * r.p1, 0.0f, 0.0f};
    lp[q] = make_float2(e.p0, e.p1);
    if (q == 0) lp[ROW4_THREADS] = lq[ROW4_THREADS] = make_float2(0.0f, 0.0f);
    __syncthreads();
#pragma unroll
    for (int s = 1; s <= 2 * K; ++s) {
        if (s & 1) {
            float a = r.q0, b = r.q1;
            sgs_pair(C.Q0, C.Q1, a, b, lp[qm], lp[qp], e.p0, e.p1);
            e.q0 = C.Q0.id * a;
            e.q1 = C.Q1.id * b;
            if (s < 2 * K) lq[q] = make_float2(e.q0, e.q1);
        } else {
            float a = r.p0, b = r.p1;
            sgs_pair(C.P0, C.P1, a, b, lq[qm], lq[qp], e.q0, e.q1);
            e.p0 = C.P0.id * a;
            e.p1 = C.P1.id * b;
            if (s < 2 * K) lp[q] = make_float2(e.p0, e.p1);
        }
        if (s < 2 * K) __syncthreads();
    }
    return e;
}

// The sum of a cell's couplings times its neighbours in the order x-, x+, y-, y+, z-, z+ of the
// residual (offdiag_sum) and of local_sgs1.  Which of the z weights is the lower and which the upper
// coupling depends on the cell and col0 (sgs_cells): v0, v1 are the other group's cells of the lane,
// end the cell across the row's end (of the pair's lane or of the next brick) and ce its coupling.
enum SgsPlace { AT_P0, AT_P1, AT_Q0, AT_Q1 };
template <SgsPlace AT>
__device__ __forceinline__ float sgs_ordered(const SgsCell &c, bool c1, float xm, float xp, float ym, float yp, float v0,
                                             float v1, float end, float ce) {
    float cm, cp, zm, zp;
    if (AT == AT_P0 || AT == AT_Q0) {
        const bool inner = AT == AT_P0 ? c1 : !c1;  // cell 1, else cell 0 (the row's lower end)
        cm = inner ? c.za : ce;
        zm = inner ? v0 : end;
        cp = inner ? c.zb : c.za;
        zp = inner ? v1 : v0;
    } else {
        const bool inner = AT == AT_P1 ? !c1 : c1;  // cell 2, else cell 3 (the row's upper end)
        cm = inner ? c.za : c.zb;
        zm = inner ? v0 : v1;
        cp = inner ? c.zb : ce;
        zp = inner ? v1 : end;
    }
    return c.ax_m * xm + c.ax_p * xp + c.ay_m * ym + c.ay_p * yp + cm * zm + cp * zp;
}

// local_sgs1's sweeps (its operations in its order) on a lane's row by group.
template <int K>
__device__ __forceinline__ SgsRow sgs_sweeps_ordered(const SgsCells &C, const SgsRow &r, float2 *lds, int q, bool c1) {
    const int qm = q >= 16 ? q - 16 : ROW4_THREADS, qp = q < ROW4_THREADS - 16 ? q + 16 : ROW4_THREADS;
    float2 *const lp = lds, *const lq = lds + SGS_PAIRS;
    SgsRow e{C.P0.id * r.p0, C.P1.id * r.p1, 0.0f, 0.0f};
    lp[q] = make_float2(e.p0, e.p1);
    if (q == 0) lp[ROW4_THREADS] = lq[ROW4_THREADS] = make_float2(0.0f, 0.0f);
    __syncthreads();
#pragma unroll 1
    for (int s = 0; s < K; ++s) {
        {
            const float2 xm = lp[qm], xp = lp[qp];
            const float n0 = sgs_ordered<AT_Q0>(C.Q0, c1, xm.x, xp.x, sgs_dpp<DPP_ROW_SHR2>(e.p0), sgs_dpp<DPP_ROW_SHL2>(e.p0),
                                                e.p0, e.p1, sgs_dpp<DPP_SWAP_PAIRS>(e.p1), C.Q0.zs);
            const float n1 = sgs_ordered<AT_Q1>(C.Q1, c1, xm.y, xp.y, sgs_dpp<DPP_ROW_SHR2>(e.p1), sgs_dpp<DPP_ROW_SHL2>(e.p1),
                                                e.p0, e.p1, sgs_dpp<DPP_SWAP_PAIRS>(e.p0), C.Q1.zs);
            e.q0 = C.Q0.id * (r.q0 + n0);
            e.q1 = C.Q1.id * (r.q1 + n1);
            lq[q] = make_float2(e.q0, e.q1);
        }
        __syncthreads();
        {
            const float2 xm = lq[qm], xp = lq[qp];
            const float n0 = sgs_ordered<AT_P0>(C.P0, c1, xm.x, xp.x, sgs_dpp<DPP_ROW_SHR2>(e.q0), sgs_dpp<DPP_ROW_SHL2>(e.q0),
                                                e.q0, e.q1, sgs_dpp<DPP_SWAP_PAIRS>(e.q1), C.P0.zs);
            const float n1 = sgs_ordered<AT_P1>(C.P1, c1, xm.y, xp.y, sgs_dpp<DPP_ROW_SHR2>(e.q1), sgs_dpp<DPP_ROW_SHL2>(e.q1),
                                                e.q0, e.q1, sgs_dpp<DPP_SWAP_PAIRS>(e.q0), C.P1.zs);
            e.p0 = C.P0.id * (r.p0 + n0);
            e.p1 = C.P1.id * (r.p1 + n1);
            lp[q] = make_float2(e.p0, e.p1);
        }
        __syncthreads();
    }
    return e;
}

// e = M_b r on rows.  lds: SGS_LDS floats (8-byte aligned).
template <int K>
__device__ __forceinline__ void local_sgs4(const Row4Coef<float> &c, const float id[4], const float r[4], float e[4],
                                           float *lds, int q) {
    const SgsCells C = sgs_cells(c, id, q);
    const bool c1 = sgs_col1(q);
    sgs_ungroup(sgs_sweeps<K>(C, sgs_group(r, c1), reinterpret_cast<float2 *>(lds), q), c1, e);
}

// Pre-smoothing from zero on the finest level: z = M_b rhs (one brick per 128-thread workgroup), K
// sweeps.
template <int K>
__global__ __launch_bounds__(ROW4_THREADS) void k_pre_local4(LevelDesc L, OpDesc<float> A,
                                                             const float *__restrict__ idiag,
                                                             const float *__restrict__ rhs, float *__restrict__ z,
                                                             Gate Q) {
    __shared__ __align__(16) float lds[SGS_LDS];
    const int br = brick_or_idle(L);
    if (br < 0) return;
    const BrickMeta m = L.meta[br];
    if (all_done(Q) || skip_smooth(Q, L, m)) return;
    const int q = threadIdx.x;
    const Row4Nbrs N = row4_nbrs(m, br, q);
    float r[4], id[4], e[4];
    unpack4(ld4(rhs, N.c), r);
    Row4Coef<float> c;
    if (m.flags & BM_UNIFORM) {
        const UniT<float> u = uni_load<float>(L, br);
        c = row4_uniform(u.g);
#pragma unroll
        for (int j = 0; j < 4; ++j) id[j] = u.id;
    } else {
        c = row4_coef(A, N);
        unpack4(ld4(idiag, N.c), id);
    }
    local_sgs4<K>(c, id, r, e, lds, q);
    *reinterpret_cast<float4 *>(z + N.c) = make_float4(e[0], e[1], e[2], e[3]);
}

// Post-smoothing on a level: z += M_b (rhs - A z), K sweeps (one brick per 128-thread workgroup).  Reads zin,
// writes zout (other bricks read this one's zin).  DOT (finest level's last application): also the rhs.z
// partial of each brick.
//
// PRO: zin first receives the coarse level's correction, trilinear as k_prolong4's (which wrote the
// corrected z out for this kernel to read again: 12 us of a 256^3 V-cycle's finest level, and a launch
// on each coarse level).  The coarse cells that the brick and the cells across its faces interpolate from are the
// same 6^3, interpolated axis by axis through LDS (12 operations per row at the end where eight
// corners per cell take 84); the rows beside a cell's own come from the
// lanes that hold them (through LDS) or, across a face, are loaded and corrected here as well.  A cell
// across a face that is no unknown is corrected too, where its coupling is 0 (else BM_LOOSE; reading every such cell's
// dir instead took 25.6 us on 256^3's finest level, 22.6 without).  Two launches took 29.5 us on the
// finest level of 256^3 (9248 bricks) and 9 us on a level of 40, this one 21.7 and 5.6.
constexpr int PRO_EDGE = 6, PRO_FINE = 10;  // coarse and fine rows per axis, those across the faces included
constexpr float PRO_NEAR = 0.75f, PRO_FAR = 0.25f;
__device__ __forceinline__ float pro_mix(float near, float far) { return PRO_NEAR * near + PRO_FAR * far; }
// The two coarse rows that fine row f (-1 .. 8) lies between, the nearer one first.
__device__ __forceinline__ int pro_near(int f) { return (f >> 1) + 1; }
__device__ __forceinline__ int pro_far(int f) { return (f & 1) ? pro_near(f) + 1 : pro_near(f) - 1; }
// Half a row: cells 4h .. 4h + 3, and the one across the row's end (k = -1 for h = 0, 8 for h = 1).
struct ProLds {
    float4 z[PRO_EDGE * PRO_EDGE * 2];  // interpolated along z: coarse row (a, b), half h
    float4 y[PRO_EDGE * PRO_FINE * 2];  // then along y: coarse a, fine j
    float ze[PRO_EDGE * PRO_EDGE * 2], ye[PRO_EDGE * PRO_FINE * 2];
};

template <int DOT, int K = LOCAL_SGS_SWEEPS, int FINEST = 1, int PRO = 0>
__global__ __launch_bounds__(ROW4_THREADS) void k_post_local4(LevelDesc L, OpDesc<float> A,
                                                              const float *__restrict__ idiag,
                                                              const float *__restrict__ rhs,
                                                              const float *__restrict__ zin, float *__restrict__ zout,
                                                              Gate Q, RedBuf R, const float *__restrict__ zcoarse) {
    __shared__ __align__(16) float lds[SGS_LDS];
    __shared__ __align__(16) unsigned char pro_lds[PRO ? sizeof(ProLds) : 1];
    ProLds &P = *reinterpret_cast<ProLds *>(pro_lds);
    __shared__ double red[2];
    const int br = brick_or_idle(L);
    if (br < 0) return;
    const BrickMeta m = L.meta[br];
    if (all_done(Q) || skip_smooth(Q, L, m)) return;
    const int q = threadIdx.x, li = q >> 4, lj = (q >> 1) & 7, h = q & 1;
    const Row4Nbrs N = row4_nbrs(m, br, q);
    const bool uniform = FINEST && (m.flags & BM_UNIFORM);
    Row4Raw<float> raw;
    float w[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (PRO) {
        // coarse row (a, b) with B = 2M + p is coarse cell row 8M + 4p - 1 + a ..: coarse brick M - 1 + p +
        // slot with slot = ((4p + 7 + a) >> 3) - p, local (4p + 7 + a) & 7; the four cells of half h
        const int px = L.bxyz[3 * br] & 1, py = L.bxyz[3 * br + 1] & 1, pz = L.bxyz[3 * br + 2] & 1;
        if (q < PRO_EDGE * PRO_EDGE * 2) {
            const int row = q >> 1, a = row / PRO_EDGE, b = row - a * PRO_EDGE;
            const int ia = 4 * px + 7 + a, ib = 4 * py + 7 + b, ic = 4 * pz + 7 + 2 * h;
            const int2 id = *reinterpret_cast<const int2 *>(
                L.parent8 + 8 * br + (((ia >> 3) - px) * 2 + ((ib >> 3) - py)) * 2);
            const int cell = ((ia & 7) * 8 + (ib & 7)) * 8;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int brick = ((ic + u) >> 3) - pz ? id.y : id.x;
                if (brick >= 0) w[u] = zcoarse[(long)brick * BRICK_CELLS + cell + ((ic + u) & 7)];
            }
        }
        load4(zin, N.c, raw.c);
        // the row across the x face and the one across the y face (a lane has at most one of each)
        load4(zin, li == 0 ? N.ixm : N.ixp, raw.xm);
        load4(zin, lj == 0 ? N.iym : N.iyp, raw.ym);
        raw.end = zin[N.iz];
    } else {
        raw = row4_load(zin, N);
    }
    float r[4], id[4], dir[4];
    load4(rhs, N.c, r);
    // the operator: on a coarse level in flight with the rest (latency), on the finest where it is used
    // (registers, so wavefronts)
    Row4CoefRaw<float> graw;
    if (!FINEST) {
        graw = row4_coef_load(A, N);
        load4(idiag, N.c, id);
    }
    if ((!FINEST || PRO) && !uniform) load4(A.dir, N.c, dir);
    if (PRO) {
        // a flat (2D) level has one cell layer: weight 1 on it, none on the empty neighbour layer
        const float nk = L.flat ? 1.0f : PRO_NEAR, fk = L.flat ? 0.0f : PRO_FAR;
        if (q < PRO_EDGE * PRO_EDGE * 2) {
            P.z[q] = make_float4(nk * w[1] + fk * w[0], nk * w[1] + fk * w[2], nk * w[2] + fk * w[1], nk * w[2] + fk * w[3]);
            P.ze[q] = h ? nk * w[3] + fk * w[2] : nk * w[0] + fk * w[1];
        }
        __syncthreads();
        auto mix4 = [](const float4 n, const float4 f) {
            return make_float4(pro_mix(n.x, f.x), pro_mix(n.y, f.y), pro_mix(n.z, f.z), pro_mix(n.w, f.w));
        };
        if (q < PRO_EDGE * PRO_FINE * 2) {
            const int a = q / (2 * PRO_FINE), j = (q >> 1) - a * PRO_FINE - 1;
            const int n = (a * PRO_EDGE + pro_near(j)) * 2 + h, f = (a * PRO_EDGE + pro_far(j)) * 2 + h;
            P.y[q] = mix4(P.z[n], P.z[f]);
            P.ye[q] = pro_mix(P.ze[n], P.ze[f]);
        }
        __syncthreads();
        auto at = [&](int a, int j) { return (a * PRO_FINE + j + 1) * 2 + h; };
        const int gi = li == 0 ? -1 : 8, gj = lj == 0 ? -1 : 8;
        float own[4], gx[4], gy[4];
        unpack4(mix4(P.y[at(pro_near(li), lj)], P.y[at(pro_far(li), lj)]), own);
        unpack4(mix4(P.y[at(pro_near(gi), lj)], P.y[at(pro_far(gi), lj)]), gx);
        unpack4(mix4(P.y[at(pro_near(li), gj)], P.y[at(pro_far(li), gj)]), gy);
        float end = pro_mix(P.ye[at(pro_near(li), lj)], P.ye[at(pro_far(li), lj)]);
        if (m.flags & BM_LOOSE) {
            float d[4];
            load4(A.dir, li == 0 ? N.ixm : N.ixp, d);
#pragma unroll
            for (int j = 0; j < 4; ++j) gx[j] = d[j] >= 0 ? gx[j] : 0.0f;
            load4(A.dir, lj == 0 ? N.iym : N.iyp, d);
#pragma unroll
            for (int j = 0; j < 4; ++j) gy[j] = d[j] >= 0 ? gy[j] : 0.0f;
            end = A.dir[N.iz] >= 0 ? end : 0.0f;
        }
        raw.end += end;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            raw.c[j] = (uniform || dir[j] >= 0) ? raw.c[j] + own[j] : raw.c[j];
            gx[j] += raw.xm[j];
            gy[j] += raw.ym[j];
        }
        float4 *const rows = reinterpret_cast<float4 *>(lds);
        rows[q] = make_float4(raw.c[0], raw.c[1], raw.c[2], raw.c[3]);
        __syncthreads();
        float nb[4];
        unpack4(rows[li > 0 ? q - 16 : q], nb);
#pragma unroll
        for (int j = 0; j < 4; ++j) raw.xm[j] = li > 0 ? nb[j] : gx[j];
        unpack4(rows[li < 7 ? q + 16 : q], nb);
#pragma unroll
        for (int j = 0; j < 4; ++j) raw.xp[j] = li < 7 ? nb[j] : gx[j];
        unpack4(rows[lj > 0 ? q - 2 : q], nb);
#pragma unroll
        for (int j = 0; j < 4; ++j) raw.ym[j] = lj > 0 ? nb[j] : gy[j];
        unpack4(rows[lj < 7 ? q + 2 : q], nb);
#pragma unroll
        for (int j = 0; j < 4; ++j) raw.yp[j] = lj < 7 ? nb[j] : gy[j];
        __syncthreads();  // the sweeps use lds again
    }
    float e[4], res[4];
    Row4Vals<float> v;
    Row4Coef<float> c;
    bool unk[4];
    if (uniform) {
        v = row4_join(raw, N);
        const UniT<float> u = uni_load<float>(L, br);
        const float diag = 0.0f + ((u.g + u.g) + (u.g + u.g) + (u.g + u.g));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float off = u.g * v.xm[j] + u.g * v.xp[j] + u.g * v.ym[j] + u.g * v.yp[j] + u.g * v.zm[j] +
                              u.g * v.zp[j];
            res[j] = r[j] - (diag * v.c[j] - off);
            id[j] = u.id;
            unk[j] = true;
        }
        c = row4_uniform(u.g);
    } else {
        if (FINEST) {
            graw = row4_coef_load(A, N);
            if (!PRO) load4(A.dir, N.c, dir);
            load4(idiag, N.c, id);
        }
        v = row4_join(raw, N);
        const Row4Coef<float> g = row4_coef_join(graw, N);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float off = g.gxm[j] * v.xm[j] + g.gxp[j] * v.xp[j] + g.gym[j] * v.ym[j] + g.gyp[j] * v.yp[j] +
                              g.gzm[j] * v.zm[j] + g.gzp[j] * v.zp[j];
            const float diag = dir[j] + ((g.gxm[j] + g.gxp[j]) + (g.gym[j] + g.gyp[j]) + (g.gzm[j] + g.gzp[j]));
            unk[j] = dir[j] >= 0;
            res[j] = unk[j] ? r[j] - (diag * v.c[j] - off) : 0.0f;
        }
        c = g;
    }
    local_sgs4<K>(c, id, res, e, lds, q);
    float out[4];
    double part = 0.0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        out[j] = unk[j] ? v.c[j] + e[j] : 0.0f;
        if (DOT) part += unk[j] ? (double)r[j] * (double)out[j] : 0.0;
    }
    *reinterpret_cast<float4 *>(zout + N.c) = make_float4(out[0], out[1], out[2], out[3]);
    if (DOT) {
        part = wave_sum(part);
        if ((q & 63) == 0) red[q >> 6] = part;
        __syncthreads();
        if (q == 0) {
            R.partials[2 * br + 0] = red[0] + red[1];
            R.partials[2 * br + 1] = 0.0;
        }
    }
}

// (A v) on the lane's four cells, with the unknown mask: apply_row / apply_row_uniform per cell.
template <int FINEST, class T>
__device__ __forceinline__ void apply_row4(const LevelDesc &L, const OpDesc<T> &A, int br, const BrickMeta &m,
                                           const Row4Nbrs &N, const Row4Raw<T> &raw, T av[4], bool unk[4]) {
    if (FINEST && (m.flags & BM_UNIFORM)) {
        const UniT<T> u = uni_load<T>(L, br);
        const Row4Vals<T> v = row4_join(raw, N);
        const T diag = T(0) + ((u.g + u.g) + (u.g + u.g) + (u.g + u.g));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const T off = u.g * v.xm[j] + u.g * v.xp[j] + u.g * v.ym[j] + u.g * v.yp[j] + u.g * v.zm[j] + u.g * v.zp[j];
            av[j] = diag * v.c[j] - off;
            unk[j] = true;
        }
    } else {
        const Row4CoefRaw<T> graw = row4_coef_load(A, N);
        T dir[4];
        load4(A.dir, N.c, dir);
        const Row4Vals<T> v = row4_join(raw, N);
        const Row4Coef<T> g = row4_coef_join(graw, N);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const T off = g.gxm[j] * v.xm[j] + g.gxp[j] * v.xp[j] + g.gym[j] * v.ym[j] + g.gyp[j] * v.yp[j] +
                          g.gzm[j] * v.zm[j] + g.gzp[j] * v.zp[j];
            const T diag = dir[j] + ((g.gxm[j] + g.gxp[j]) + (g.gym[j] + g.gyp[j]) + (g.gzm[j] + g.gzp[j]));
            av[j] = diag * v.c[j] - off;
            unk[j] = dir[j] >= 0;
        }
    }
}

// Brick and lane of a workgroup that takes BPB consecutive bricks (block ids remapped XCD-aware;
// gridDim.x a multiple of 8); br >= L.nbricks for an idle slot.  Row-4 launches give the finest
// level BLOCK threads (four bricks) and coarse levels ROW4_THREADS (one brick): the kernels' FINEST
// flag fixes BPB at compile time (blockDim.x is a 16-bit hidden kernel argument that hipcc reads
// with a vector load, one more memory round trip at the start of every wave).
template <int FINEST>
__device__ __forceinline__ void row4_slot(const LevelDesc &L, int &br, int &q, int skip = 0) {
    constexpr int BPB = FINEST ? BLOCK / ROW4_THREADS : 1;
    br = BPB * xcd_brick(blockIdx.x - skip, gridDim.x - skip);
    // a wavefront works on one brick (whose record is then a scalar load)
    if (FINEST) br += __builtin_amdgcn_readfirstlane((int)(threadIdx.x / ROW4_THREADS));
    q = threadIdx.x % ROW4_THREADS;
}

// Sum / max over the two wavefronts of a 128-thread workgroup (result valid in every thread).
template <bool AMAX>
__device__ __forceinline__ void row4_reduce2(double &a, double &b, double *lds) {
    a = AMAX ? wave_max(a) : wave_sum(a);
    b = wave_sum(b);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        lds[w] = a;
        lds[2 + w] = b;
    }
    __syncthreads();
    a = AMAX ? fmax(lds[0], lds[1]) : lds[0] + lds[1];
    b = lds[2] + lds[3];
}

// res = rhs - A z.  FIN (finest level): the first workgroups, one per grid (rounded
// up to 8, which keeps the bricks' XCDs), run the convergence test of the residual update before this
// kernel instead of a launch of their own (3 to 6 us).  Nothing in the V-cycle waits for its outcome: a
// grid that it finds done only loses what this kernel and its neighbours do for it.
template <class T, int FINEST, int FIN = 0>
__global__ __launch_bounds__(BLOCK) void k_residual4(LevelDesc L, OpDesc<T> A, const T *__restrict__ rhs,
                                                     const T *__restrict__ z, T *__restrict__ res, Gate Q,
                                                     FinUpdate F) {
    int br, q;
    if (FIN) {
        const int front = (L.ngrids + 7) & ~7;
        if ((int)blockIdx.x < front) {
            if ((int)blockIdx.x < L.ngrids) finalize_update(F, L, blockIdx.x);
            return;
        }
        row4_slot<FINEST>(L, br, q, front);
    } else {
        row4_slot<FINEST>(L, br, q);
    }
    if (br >= L.nbricks) return;
    const BrickMeta m = L.meta[br];
    if (all_done(Q) || skip_smooth(Q, L, m)) return;
    const Row4Nbrs N = row4_nbrs(m, br, q);
    const Row4Raw<T> v = row4_load(z, N);
    T r[4], av[4], out[4];
    bool unk[4];
    load4(rhs, N.c, r);
    apply_row4<FINEST>(L, A, br, m, N, v, av, unk);
#pragma unroll
    for (int j = 0; j < 4; ++j) out[j] = unk[j] ? r[j] - av[j] : T(0);
    store4(res, N.c, out);
}

// z = omega * idiag * rhs (k_smooth_first on rows).
template <int FINEST>
__global__ __launch_bounds__(BLOCK) void k_smooth_first4(LevelDesc L, const float *__restrict__ idiag,
                                                         const float *__restrict__ rhs, float *__restrict__ z,
                                                         float omega, Gate Q) {
    int br, q;
    row4_slot<FINEST>(L, br, q);
    if (br >= L.nbricks) return;
    const BrickMeta m = L.meta[br];
    if (all_done(Q) || skip_smooth(Q, L, m)) return;
    const long c = (long)br * BRICK_CELLS + 4 * q;
    float r[4], id[4], out[4];
    unpack4(ld4(rhs, c), r);
    if (m.flags & BM_UNIFORM) {
        const float u = uni_load<float>(L, br).id;
#pragma unroll
        for (int j = 0; j < 4; ++j) id[j] = u;
    } else {
        unpack4(ld4(idiag, c), id);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) out[j] = omega * id[j] * r[j];
    *reinterpret_cast<float4 *>(z + c) = make_float4(out[0], out[1], out[2], out[3]);
}

// ---- The FP32 Krylov iteration of the mixed-precision solve.  Its vectors r, p, q, z are stored in
// FP32, but the iterate is the FP64 pressure itself (x64 += alpha p in FP64) and q = A p is formed
// from the FP64 operator in FP64 arithmetic, rounded once when stored.  Then the recursive
// residual follows b - A x64 to FP32 storage accuracy of r and q: neither the rounding of an FP32
// iterate nor an FP32 operator apply (whose cancellation amplifies the rounding by about the
// condition number, 1e4 and more at 256^3) enters it, so one pass reaches the final tolerance.

// (A v) in FP64 on the lane's four cells from FP32 values v and the FP64 operator (k_apply_dot's
// arithmetic in FP64); unk: the unknown mask.
__device__ __forceinline__ void apply_row4_64(const LevelDesc &L, const OpDesc<double> &A, int br, const BrickMeta &m,
                                              const Row4Nbrs &N, const Row4Vals<float> &v, double av[4],
                                              bool unk[4]) {
    if (m.flags & BM_UNIFORM) {
        const double g = L.uni[br].g64;
        const double diag = 0.0 + ((g + g) + (g + g) + (g + g));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const double off = g * (double)v.xm[j] + g * (double)v.xp[j] + g * (double)v.ym[j] + g * (double)v.yp[j] +
                               g * (double)v.zm[j] + g * (double)v.zp[j];
            av[j] = diag * (double)v.c[j] - off;
            unk[j] = true;
        }
    } else {
        const Row4Coef<double> g = row4_coef(A, N);
        double dir[4];
        load4(A.dir, N.c, dir);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const double off = g.gxm[j] * (double)v.xm[j] + g.gxp[j] * (double)v.xp[j] + g.gym[j] * (double)v.ym[j] +
                               g.gyp[j] * (double)v.yp[j] + g.gzm[j] * (double)v.zm[j] + g.gzp[j] * (double)v.zp[j];
            const double diag = dir[j] + ((g.gxm[j] + g.gxp[j]) + (g.gym[j] + g.gyp[j]) + (g.gzm[j] + g.gzp[j]));
            av[j] = diag * (double)v.c[j] - off;
            unk[j] = dir[j] >= 0;
        }
    }
}

// q = A p (FP64 operator and arithmetic, q stored in FP32) with the p.q partials (FP64 q): one
// brick per 128-thread workgroup.
__global__ __launch_bounds__(ROW4_THREADS) void k_apply_dot4(LevelDesc L, OpDesc<double> A, const float *__restrict__ p,
                                                             float *__restrict__ qv, const SolveScalars *S,
                                                             const BatchCtl *ctl, RedBuf R) {
    __shared__ double lds[4];
    const int br = brick_or_idle(L);
    if (br < 0) return;
    const BrickMeta m = L.meta[br];
    // a batch skips finished grids before loading anything; a single grid loads first
    if (L.ngrids > 1 && (ctl->all_done || S[m.grid].done)) return;
    const Row4Nbrs N = row4_nbrs(m, br, threadIdx.x);
    const Row4Vals<float> v = row4_vals(p, N);
    if (ctl->all_done) return;
    double av[4];
    float out[4];
    bool unk[4];
    apply_row4_64(L, A, br, m, N, v, av, unk);
    double part = 0.0, unused = 0.0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        out[j] = unk[j] ? (float)av[j] : 0.0f;
        part += unk[j] ? (double)v.c[j] * av[j] : 0.0;
    }
    *reinterpret_cast<float4 *>(qv + N.c) = make_float4(out[0], out[1], out[2], out[3]);
    row4_reduce2<false>(part, unused, lds);
    store_partials(R, br, part, 0.0);
}

// k_update_p4 (p = z + beta p, FP32) fused into k_apply_dot4: the new direction of the lane's cells
// and of their neighbours is formed on the fly from z and the previous direction (the same FP32
// arithmetic), written to pnew (a different buffer than pold: other workgroups still read pold),
// and q = A pnew with the pnew.q partials.
// FOLD (a single grid of at most FOLD_BRICKS bricks): beta = r.z / (the r.z before, S->rz[slot]) is
// formed here from the partials of r.z (rz), as FIN_RZ does; the workgroup of brick 0 records it, r.z in
// S->rz[slot ^ 1].
template <int FOLD>
__global__ __launch_bounds__(ROW4_THREADS) void k_apply_dot4p(LevelDesc L, OpDesc<double> A,
                                                              const float *__restrict__ z,
                                                              const float *__restrict__ pold,
                                                              float *__restrict__ pnew, float *__restrict__ qv,
                                                              SolveScalars *S, BatchCtl *ctl, RedBuf R,
                                                              const double *__restrict__ rz, int slot) {
    __shared__ double lds[FOLD ? FoldPartials::LDS : 4];
    const int br = brick_or_idle(L);
    if (br < 0) return;
    const BrickMeta m = L.meta[br];
    const int g = L.ngrids > 1 ? m.grid : 0;
    if (L.ngrids > 1 && (ctl->all_done || S[g].done)) return;
    const Row4Nbrs N = row4_nbrs(m, br, threadIdx.x);
    FoldPartials P;
    if (FOLD) P.load(rz, L.nbricks);
    const Row4Vals<float> zv = row4_vals(z, N);
    const Row4Vals<float> po = row4_vals(pold, N);
    bool stop = ctl->all_done != 0;
    if (!FOLD && stop) return;
    float beta;
    if (FOLD) {
        const double now = P.sum(lds, stop), b64 = now / S->rz[slot];
        if (stop) return;
        if (br == 0 && threadIdx.x == 0) {
            S->beta = b64;
            S->rz[slot ^ 1] = now;
            if (!(now == now)) {
                S->status = 1;
                mark_done(*S, ctl);
            }
        }
        if (!(now == now)) return;
        beta = (float)b64;
        __syncthreads();  // lds is used again
    } else {
        beta = (float)S[g].beta;
    }
    Row4Vals<float> v;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v.c[j] = zv.c[j] + beta * po.c[j];
        v.xm[j] = zv.xm[j] + beta * po.xm[j];
        v.xp[j] = zv.xp[j] + beta * po.xp[j];
        v.ym[j] = zv.ym[j] + beta * po.ym[j];
        v.yp[j] = zv.yp[j] + beta * po.yp[j];
        v.zm[j] = zv.zm[j] + beta * po.zm[j];
        v.zp[j] = zv.zp[j] + beta * po.zp[j];
    }
    double av[4];
    float out[4];
    bool unk[4];
    apply_row4_64(L, A, br, m, N, v, av, unk);
    double part = 0.0, unused = 0.0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        out[j] = unk[j] ? (float)av[j] : 0.0f;
        part += unk[j] ? (double)v.c[j] * av[j] : 0.0;
    }
    *reinterpret_cast<float4 *>(pnew + N.c) = make_float4(v.c[0], v.c[1], v.c[2], v.c[3]);
    *reinterpret_cast<float4 *>(qv + N.c) = make_float4(out[0], out[1], out[2], out[3]);
    row4_reduce2<false>(part, unused, lds);
    store_partials(R, br, part, 0.0);
}

// x64 += alpha p (FP64), r -= alpha q (FP32) with ||r||_inf and r.r partials; ZFIRST: also the first
// pre-smoothing step of the next V-cycle from zero on the finest level, on the bricks it covers
// (not those of grids ending on this level), with the same arithmetic: 1 = a damped Jacobi sweep
// (k_smooth_first4<1>), z = omega * idiag * r; 2 = the brick-local smoother (k_pre_local4<K>),
// whose brick is the workgroup's.  A grid that this update finds converged gets a z it never uses.
// FOLD (a single grid of at most FOLD_BRICKS bricks): alpha = S->rz[slot] / (p.q) is formed here from the
// partials of p.q (pq), as FIN_PQ does; the workgroup of brick 0 records it.
template <int ZFIRST, int K = LOCAL_SGS_SWEEPS, int FOLD = 0>
__global__ __launch_bounds__(ROW4_THREADS) void k_cg_update4(LevelDesc L, double *__restrict__ x,
                                                             float *__restrict__ r, const float *__restrict__ p,
                                                             const float *__restrict__ qv, SolveScalars *S,
                                                             BatchCtl *ctl, RedBuf R,
                                                             const float *__restrict__ idiag, float *__restrict__ z,
                                                             float omega, OpDesc<float> A32,
                                                             const double *__restrict__ pq, int slot) {
    __shared__ double lds[FOLD ? FoldPartials::LDS : 4];
    const int br = brick_or_idle(L);
    if (br < 0) return;
    const long c = (long)br * BRICK_CELLS + 4 * threadIdx.x;
    const BrickMeta m = L.meta[br];
    const int g = L.ngrids > 1 ? m.grid : 0;
    if (L.ngrids > 1 && (ctl->all_done || S[g].done)) return;
    FoldPartials P;
    if (FOLD) P.load(pq, L.nbricks);
    double xv[4];
    float pv[4], rv[4], qq[4], id[4];
    load4(x, c, xv);
    unpack4(ld4(p, c), pv);
    unpack4(ld4(r, c), rv);
    unpack4(ld4(qv, c), qq);
    Row4Coef<float> cf;  // ZFIRST == 2: the brick's own couplings
    if (ZFIRST) {
        if (m.flags & BM_UNIFORM) {
            const UniT<float> u = uni_load<float>(L, br);
#pragma unroll
            for (int j = 0; j < 4; ++j) id[j] = u.id;
            if (ZFIRST == 2) cf = row4_uniform(u.g);
        } else {
            unpack4(ld4(idiag, c), id);
            if (ZFIRST == 2) cf = row4_coef(A32, row4_nbrs(m, br, threadIdx.x));
        }
    }
    const SolveScalars &Sg = S[g];
    bool stop = ctl->all_done || Sg.done;
    if (!FOLD && stop) return;
    double alpha;
    if (FOLD) {
        const double now = P.sum(lds, stop);
        if (stop) return;
        alpha = S->rz[slot] / now;
        const bool bad = !(alpha == alpha) || alpha - alpha != 0.0;
        if (br == 0 && threadIdx.x == 0) {
            S->pq = now;
            S->alpha = alpha;
            if (bad) {
                S->status = 1;
                mark_done(*S, ctl);
            }
        }
        if (bad) return;
        __syncthreads();  // lds is used again
    } else {
        alpha = Sg.alpha;
    }
    const float alpha32 = (float)alpha;
    double mx = 0.0, sq = 0.0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        xv[j] = xv[j] + alpha * (double)pv[j];
        rv[j] = rv[j] - alpha32 * qq[j];
        mx = fmax(mx, fabs((double)rv[j]));
        sq += (double)rv[j] * (double)rv[j];
    }
    store4(x, c, xv);
    *reinterpret_cast<float4 *>(r + c) = make_float4(rv[0], rv[1], rv[2], rv[3]);
    if (ZFIRST == 1 && !(m.flags & BM_COARSEST)) {
        float out[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) out[j] = omega * id[j] * rv[j];
        *reinterpret_cast<float4 *>(z + c) = make_float4(out[0], out[1], out[2], out[3]);
    }
    if (ZFIRST == 2 && !(m.flags & BM_COARSEST)) {
        // the brick-local smoother's pre-smoothing from zero (k_pre_local4) on the updated residual
        __shared__ __align__(16) float zl[SGS_LDS];
        float e[4];
        local_sgs4<K>(cf, id, rv, e, zl, threadIdx.x);
        *reinterpret_cast<float4 *>(z + c) = make_float4(e[0], e[1], e[2], e[3]);
    }
    row4_reduce2<true>(mx, sq, lds);
    store_partials(R, br, mx, sq);
}

// p = z + beta p (first: p = z), k_update_p on rows.
__global__ __launch_bounds__(BLOCK) void k_update_p4(LevelDesc L, const float *__restrict__ z, float *__restrict__ p,
                                                     const SolveScalars *S, const BatchCtl *ctl, int first) {
    int br, q;
    row4_slot<1>(L, br, q);  // the finest level only (row-4 launch of BLOCK threads)
    if (br >= L.nbricks) return;
    const long c = (long)br * BRICK_CELLS + 4 * q;
    if (L.ngrids > 1 && (ctl->all_done || S[grid_of(L, br)].done)) return;
    float zv[4], pv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    unpack4(ld4(z, c), zv);
    if (!first) unpack4(ld4(p, c), pv);
    const SolveScalars &Sg = S[grid_of(L, br)];
    if (ctl->all_done || Sg.done) return;
    const float beta = (float)Sg.beta;
#pragma unroll
    for (int j = 0; j < 4; ++j) pv[j] = first ? zv[j] : zv[j] + beta * pv[j];
    *reinterpret_cast<float4 *>(p + c) = make_float4(pv[0], pv[1], pv[2], pv[3]);
}

// r = b - A x in FP64 with per-brick ||r||_inf and ||r||^2 partials (finalized by FIN_DEFECT*):
// one brick per 128-thread workgroup, four cells per thread (two 16-byte loads per array).
__global__ __launch_bounds__(ROW4_THREADS) void k_defect4(LevelDesc L, OpDesc<double> A, const double *__restrict__ b,
                                                          const double *__restrict__ x, double *__restrict__ r,
                                                          RedBuf R) {
    __shared__ double lds[4];
    const int br = brick_or_idle(L);
    if (br < 0) return;
    const BrickMeta m = L.meta[br];
    const Row4Nbrs N = row4_nbrs(m, br, threadIdx.x);
    const Row4Raw<double> v = row4_load(x, N);
    double bv[4], av[4], out[4];
    bool unk[4];
    load4(b, N.c, bv);
    apply_row4<1>(L, A, br, m, N, v, av, unk);
    double mx = 0.0, sq = 0.0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        out[j] = unk[j] ? bv[j] - av[j] : 0.0;
        mx = fmax(mx, fabs(out[j]));
        sq += out[j] * out[j];
    }
    store4(r, N.c, out);
    row4_reduce2<true>(mx, sq, lds);
    store_partials(R, br, mx, sq);
}

// Inner (FP32) solve set-up of the defect correction: r32 = (float) r64 with ||r32|| partials
// (finalized by FIN_INNER_INIT); four cells per thread.  The inner solve adds its correction to the
// FP64 iterate directly (k_cg_update4).
__global__ __launch_bounds__(ROW4_THREADS) void k_inner_init4(LevelDesc L, const double *__restrict__ r64,
                                                              float *__restrict__ r32, RedBuf R) {
    __shared__ double lds[4];
    const int br = brick_or_idle(L);
    if (br < 0) return;
    const long c = (long)br * BRICK_CELLS + 4 * threadIdx.x;
    double rv[4];
    float v[4];
    load4(r64, c, rv);
    double mx = 0.0, sq = 0.0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v[j] = (float)rv[j];
        mx = fmax(mx, fabs((double)v[j]));
        sq += (double)v[j] * (double)v[j];
    }
    store4(r32, c, v);
    row4_reduce2<true>(mx, sq, lds);
    store_partials(R, br, mx, sq);
}

// Restriction = transpose of trilinear prolongation: coarse cell I gathers fine cells
// 2I-1..2I+2 per axis with weights 1/4, 3/4, 3/4, 1/4.  One block per coarse brick B stages the
// 18^3 fine residuals it needs (fine cells 16B-1 .. 16B+16 per axis, in the fine bricks 2B-1 ..
// 2B+2 that the brick's child table lists) in LDS.
// M_b r for one cell per thread of a 512-thread workgroup holding one brick (cell t, storage
// order): K symmetric red-black Gauss-Seidel sweeps from zero on the brick's own operator (c: the
// cell's couplings to cells of the brick, 0 across its faces), as local_sgs4.  lds: 512 floats.
template <int K>
__device__ __forceinline__ float local_sgs1(const float c[6], float id, float r, float *lds, int t) {
    const int li = t >> 6, lj = (t >> 3) & 7, lk = t & 7;
    const int colour = (li + lj + lk) & 1;
    float e = colour == 0 ? id * r : 0.0f;
    if (colour == 0) lds[t] = e;
    __syncthreads();
#pragma unroll
    for (int s = 1; s <= 2 * K; ++s) {
        if (colour == (s & 1)) {
            const float xm = li > 0 ? lds[t - 64] : 0.0f, xp = li < 7 ? lds[t + 64] : 0.0f;
            const float ym = lj > 0 ? lds[t - 8] : 0.0f, yp = lj < 7 ? lds[t + 8] : 0.0f;
            const float zm = lk > 0 ? lds[t - 1] : 0.0f, zp = lk < 7 ? lds[t + 1] : 0.0f;
            const float nb = c[0] * xm + c[1] * xp + c[2] * ym + c[3] * yp + c[4] * zm + c[5] * zp;
            e = id * (r + nb);
            lds[t] = e;
        }
        __syncthreads();
    }
    return e;
}

// k_restrict (FP32) that also runs the coarse level's pre-smoothing from zero with the brick-local
// smoother: zc = M_b rhs_c on the coarse brick (skipped on bricks of grids that end on the coarse
// level: their coarse solve starts from the right-hand side).
template <int FINEST>
__global__ __launch_bounds__(BLOCK) void k_restrict_pre(LevelDesc Lc, OpDesc<float> Ac, const float *__restrict__ idc,
                                                        const float *__restrict__ res, float *__restrict__ rhs_c,
                                                        float *__restrict__ zc, Gate Q) {
    constexpr int E = 18;
    __shared__ float tile[E * E * E];
    __shared__ int bid[64];
    const int br = brick_or_idle(Lc);
    if (br < 0) return;
    const int t = threadIdx.x;
    const long c = (long)br * BRICK_CELLS + t;
    const float dirc = Ac.dir[c];
    const int cid = t < 64 ? Lc.child64[64 * br + t] : -1;
    const BrickMeta m = Lc.meta[br];
    if (all_done(Q) || grid_done(Q, Lc, m) || (m.flags & Q.skip & BM_BELOW)) return;
    if (t < 64) bid[t] = cid;
    __syncthreads();
    constexpr int NQ = (E * E * E + BLOCK - 1) / BLOCK;
    float v[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int e = t + q * BLOCK;
        v[q] = 0.0f;
        if (e < E * E * E) {
            const int c3 = e % E, b = (e / E) % E, a = e / (E * E);
            const int slot = (((a + 7) >> 3) * 4 + ((b + 7) >> 3)) * 4 + ((c3 + 7) >> 3);
            const int id = bid[slot];
            if (id >= 0) v[q] = res[(long)id * BRICK_CELLS + ((((a + 7) & 7) * 8 + ((b + 7) & 7)) * 8 + ((c3 + 7) & 7))];
        }
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int e = t + q * BLOCK;
        if (e < E * E * E) tile[e] = v[q];
    }
    __syncthreads();
    const int li = t >> 6, lj = (t >> 3) & 7, lk = t & 7;
    float out = 0.0f;
    if (dirc >= 0) {
        const float w[4] = {0.25f, 0.75f, 0.75f, 0.25f};
        const float wk[4] = {Lc.flat ? 0.0f : w[0], Lc.flat ? 1.0f : w[1], Lc.flat ? 0.0f : w[2],
                             Lc.flat ? 0.0f : w[3]};
        float acc = 0.0f;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            float acc_a = 0.0f;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const float *row = &tile[((2 * li + a) * E + (2 * lj + b)) * E + 2 * lk];
                const float acc_b = wk[0] * row[0] + wk[1] * row[1] + wk[2] * row[2] + wk[3] * row[3];
                acc_a += w[b] * acc_b;
            }
            acc += w[a] * acc_a;
        }
        out = acc;
    }
    rhs_c[c] = out;
    if (m.flags & BM_COARSEST) return;  // the whole block: the flag is the brick's
    __syncthreads();                     // the tile becomes the smoother's scratch
    float cf[6];
    cf[0] = li > 0 ? Ac.gx[c] : 0.0f;
    cf[1] = li < 7 ? Ac.gx[c + 64] : 0.0f;
    cf[2] = lj > 0 ? Ac.gy[c] : 0.0f;
    cf[3] = lj < 7 ? Ac.gy[c + 8] : 0.0f;
    cf[4] = lk > 0 ? Ac.gz[c] : 0.0f;
    cf[5] = lk < 7 ? Ac.gz[c + 1] : 0.0f;
    const float e = local_sgs1<LOCAL_SGS_SWEEPS_COARSE>(cf, idc[c], out, tile, t);
    zc[c] = e;
}

template <class T, int FINEST>
__global__ __launch_bounds__(BLOCK) void k_restrict(LevelDesc Lc, OpDesc<T> Ac, const T *__restrict__ res,
                                                    T *__restrict__ rhs_c, Gate Q) {
    constexpr int E = 18;
    __shared__ T tile[E * E * E];
    __shared__ int bid[64];
    const int br = brick_or_idle(Lc);
    if (br < 0) return;
    const int t = threadIdx.x;
    const long c = (long)br * BRICK_CELLS + t;
    // loads that depend on the brick only, issued before the gate's loads resolve
    const T dirc = Ac.dir[c];
    const int cid = t < 64 ? Lc.child64[64 * br + t] : -1;
    const BrickMeta m = Lc.meta[br];
    if (all_done(Q) || grid_done(Q, Lc, m)) return;
    if (t < 64) bid[t] = cid;
    __syncthreads();
    // all NQ loads of a thread are issued before the first LDS store (one memory latency, not NQ)
    constexpr int NQ = (E * E * E + BLOCK - 1) / BLOCK;
    T v[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int e = t + q * BLOCK;
        v[q] = T(0);
        if (e < E * E * E) {
            const int c3 = e % E, b = (e / E) % E, a = e / (E * E);
            // tile offset a is fine cell 16B - 1 + a: fine brick 2B - 1 + ((a + 7) >> 3), local (a + 7) & 7
            const int slot = (((a + 7) >> 3) * 4 + ((b + 7) >> 3)) * 4 + ((c3 + 7) >> 3);
            const int id = bid[slot];
            if (id >= 0) v[q] = res[(long)id * BRICK_CELLS + ((((a + 7) & 7) * 8 + ((b + 7) & 7)) * 8 + ((c3 + 7) & 7))];
        }
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int e = t + q * BLOCK;
        if (e < E * E * E) tile[e] = v[q];
    }
    __syncthreads();
    T out = 0;
    if (dirc >= 0) {
        const int li = t >> 6, lj = (t >> 3) & 7, lk = t & 7;
        const T w[4] = {T(0.25), T(0.75), T(0.75), T(0.25)};
        // a flat (2D) level has one cell layer: the transfer is bilinear, weight 1 on that layer
        const T wk[4] = {Lc.flat ? T(0) : w[0], Lc.flat ? T(1) : w[1], Lc.flat ? T(0) : w[2], Lc.flat ? T(0) : w[3]};
        T acc = 0;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            T acc_a = 0;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const T *row = &tile[((2 * li + a) * E + (2 * lj + b)) * E + 2 * lk];
                const T acc_b = wk[0] * row[0] + wk[1] * row[1] + wk[2] * row[2] + wk[3] * row[3];
                acc_a += w[b] * acc_b;
            }
            acc += w[a] * acc_a;
        }
        out = acc;
    }
    rhs_c[c] = out;
}

// z_f += trilinear interpolation of the coarse correction (fine unknowns only).  One block per
// fine brick B stages the 6^3 coarse values it needs (coarse cells 4B-1 .. 4B+4 per axis, in the
// coarse bricks its parent table lists) in LDS.  Coarse cells outside the coarse grid read 0: they
// lie in unstored bricks or are non-unknowns, whose correction every V-cycle kernel keeps at 0.
template <class T, int FINEST>
__global__ __launch_bounds__(BLOCK) void k_prolong(LevelDesc Lf, OpDesc<T> Af, const T *__restrict__ zc,
                                                   T *__restrict__ zf, Gate Q) {
    constexpr int E = 6;
    __shared__ T tile[E * E * E];
    __shared__ int bid[8];
    const int br = brick_or_idle(Lf);
    if (br < 0) return;
    const int t = threadIdx.x;
    const long c = (long)br * BRICK_CELLS + t;
    // loads that depend on the brick only, issued before the gate's loads resolve
    const T zf0 = zf[c];
    const int pid = t < 8 ? Lf.parent8[8 * br + t] : -1;
    // with B = 2M + p, tile offset a is coarse cell 8M + 4p - 1 + a: coarse brick
    // M - 1 + p + slot with slot = ((4p + 7 + a) >> 3) - p, local (4p + 7 + a) & 7
    const int px = Lf.bxyz[3 * br] & 1, py = Lf.bxyz[3 * br + 1] & 1, pz = Lf.bxyz[3 * br + 2] & 1;
    const BrickMeta m = Lf.meta[br];
    if (all_done(Q) || skip_smooth(Q, Lf, m)) return;
    const bool upd = (m.flags & BM_UNIFORM) || Af.dir[c] >= 0;
    if (t < 8) bid[t] = pid;
    __syncthreads();
    if (t < E * E * E) {
        const int c = t % E, b = (t / E) % E, a = t / (E * E);
        const int ia = 4 * px + 7 + a, ib = 4 * py + 7 + b, ic = 4 * pz + 7 + c;
        const int slot = (((ia >> 3) - px) * 2 + ((ib >> 3) - py)) * 2 + ((ic >> 3) - pz);
        const int id = bid[slot];
        tile[t] = id >= 0 ? zc[(long)id * BRICK_CELLS + (((ia & 7) * 8 + (ib & 7)) * 8 + (ic & 7))] : T(0);
    }
    __syncthreads();
    if (!upd) return;
    const int li = t >> 6, lj = (t >> 3) & 7, lk = t & 7;
    const int a0 = (li >> 1) + 1, b0 = (lj >> 1) + 1, c0 = (lk >> 1) + 1;
    const int a1 = (li & 1) ? a0 + 1 : a0 - 1, b1 = (lj & 1) ? b0 + 1 : b0 - 1, c1 = (lk & 1) ? c0 + 1 : c0 - 1;
    auto at = [&](int a, int b, int cc) { return tile[(a * E + b) * E + cc]; };
    const T n = T(0.75), f = T(0.25);
    // a flat (2D) level has one cell layer: weight 1 on it, none on the empty neighbour layer
    const T nk = Lf.flat ? T(1) : n, fk = Lf.flat ? T(0) : f;
    const T v = n * (n * (nk * at(a0, b0, c0) + fk * at(a0, b0, c1)) + f * (nk * at(a0, b1, c0) + fk * at(a0, b1, c1))) +
                f * (n * (nk * at(a1, b0, c0) + fk * at(a1, b0, c1)) + f * (nk * at(a1, b1, c0) + fk * at(a1, b1, c1)));
    zf[c] = zf0 + v;
}

// k_prolong on cell rows (FP32): 512-thread workgroups take four fine bricks, each staging its own
// 6^3 coarse tile; lane q adds the correction to its four cells with k_prolong's arithmetic (cells
// that are not unknowns are written back unchanged).
template <int FINEST>
__global__ __launch_bounds__(BLOCK) void k_prolong4(LevelDesc Lf, OpDesc<float> Af, const float *__restrict__ zc,
                                                    float *__restrict__ zf, Gate Q) {
    constexpr int E = 6, NT = E * E * E;
    __shared__ float tile[BLOCK / ROW4_THREADS][NT];
    __shared__ int bid[BLOCK / ROW4_THREADS][8];
    if (all_done(Q)) return;
    int br, q;
    row4_slot<FINEST>(Lf, br, q);
    const int slot = threadIdx.x / ROW4_THREADS;
    // every thread reaches the barriers; a slot past the end or of a skipped brick only idles
    bool work = br < Lf.nbricks;
    BrickMeta m{};
    if (work) {
        m = Lf.meta[br];
        work = !skip_smooth(Q, Lf, m);
    }
    const long c = (long)br * BRICK_CELLS + 4 * q;
    float z0[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    int px = 0, py = 0, pz = 0;
    if (work) {
        unpack4(ld4(zf, c), z0);
        px = Lf.bxyz[3 * br] & 1;
        py = Lf.bxyz[3 * br + 1] & 1;
        pz = Lf.bxyz[3 * br + 2] & 1;
        if (q < 8) bid[slot][q] = Lf.parent8[8 * br + q];
    }
    __syncthreads();
    // with B = 2M + p, tile offset a is coarse cell 8M + 4p - 1 + a: coarse brick
    // M - 1 + p + slot with slot = ((4p + 7 + a) >> 3) - p, local (4p + 7 + a) & 7
    if (work) {
        float v[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int e = q + u * ROW4_THREADS;
            v[u] = 0.0f;
            if (e < NT) {
                const int cc = e % E, b = (e / E) % E, a = e / (E * E);
                const int ia = 4 * px + 7 + a, ib = 4 * py + 7 + b, ic = 4 * pz + 7 + cc;
                const int s8 = (((ia >> 3) - px) * 2 + ((ib >> 3) - py)) * 2 + ((ic >> 3) - pz);
                const int id = bid[slot][s8];
                if (id >= 0) v[u] = zc[(long)id * BRICK_CELLS + (((ia & 7) * 8 + (ib & 7)) * 8 + (ic & 7))];
            }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int e = q + u * ROW4_THREADS;
            if (e < NT) tile[slot][e] = v[u];
        }
    }
    __syncthreads();
    if (!work) return;
    float dir[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const bool uni = m.flags & BM_UNIFORM;
    if (!uni) unpack4(ld4(Af.dir, c), dir);
    const int li = q >> 4, lj = (q >> 1) & 7, h = q & 1;
    const int a0 = (li >> 1) + 1, b0 = (lj >> 1) + 1;
    const int a1 = (li & 1) ? a0 + 1 : a0 - 1, b1 = (lj & 1) ? b0 + 1 : b0 - 1;
    auto at = [&](int a, int b, int cc) { return tile[slot][(a * E + b) * E + cc]; };
    const float n = 0.75f, f = 0.25f;
    // a flat (2D) level has one cell layer: weight 1 on it, none on the empty neighbour layer
    const float nk = Lf.flat ? 1.0f : n, fk = Lf.flat ? 0.0f : f;
    float out[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int lk = 4 * h + j;
        const int c0 = (lk >> 1) + 1, c1 = (lk & 1) ? c0 + 1 : c0 - 1;
        const float v = n * (n * (nk * at(a0, b0, c0) + fk * at(a0, b0, c1)) + f * (nk * at(a0, b1, c0) + fk * at(a0, b1, c1))) +
                        f * (n * (nk * at(a1, b0, c0) + fk * at(a1, b0, c1)) + f * (nk * at(a1, b1, c0) + fk * at(a1, b1, c1)));
        out[j] = (uni || dir[j] >= 0) ? z0[j] + v : z0[j];
    }
    *reinterpret_cast<float4 *>(zf + c) = make_float4(out[0], out[1], out[2], out[3]);
}

// K damped-Jacobi sweeps in one launch (coarse levels, where every launch is latency-bound).  The
// block of brick B stages the cube of cells within distance K of B (bricks B-1 .. B+1 per axis,
// found through the grid's brick map) and runs all K sweeps on it in LDS; values near the cube's
// faces go stale by one cell per sweep, which after K sweeps has not reached B, so B's cells are
// exactly K sweeps of k_jacobi (same arithmetic).  FROM_ZERO: the first sweep starts from z = 0
// (pre-smoothing), else from zin.  1024 threads; the couplings sit in LDS, idiag and rhs in
// registers.
template <class T, int K>
struct SmoothK {
    static constexpr int R = BRICK + 2 * K;          // cube side
    static constexpr int NR = R * R * R;
    static constexpr int THREADS = 1024;
    static constexpr int CPT = (NR + THREADS - 1) / THREADS;  // cube cells per thread
};

//
// RES: the cube carries one more ghost layer, so that after the K sweeps the brick's neighbours are
// exact too, and the kernel also writes the residual rhs - A z of the brick (what k_residual4
// computes next, in the same arithmetic): one launch fewer per V-cycle on the level.
//
// PRO (post-smoothing, with zin): the level's z first receives the trilinear prolongation of the
// next coarser level's correction zcoarse, as k_prolong adds it (same arithmetic), on every cell
// of the cube: one launch fewer per V-cycle on the level.  The block stages the coarse cells the
// cube needs, in the (up to) 2x2x2 coarse bricks of its parent table.
template <class T, int K>
struct ProTile {
    static constexpr int R = BRICK + 2 * K;
    static constexpr int CT = R / 2 + 2;  // coarse cells per axis
    static constexpr int N = CT * CT * CT;
};

template <class T, int K, int FROM_ZERO, int RES = 0, int PRO = 0>
__global__ __launch_bounds__(1024) void k_smooth_k(LevelDesc L, OpDesc<T> A, const T *__restrict__ idiag,
                                                   const T *__restrict__ rhs, const T *__restrict__ zin,
                                                   T *__restrict__ zout, T omega, Gate Q, T *__restrict__ res,
                                                   const T *__restrict__ zcoarse) {
    static_assert(!(PRO && (FROM_ZERO || RES)), "the prolongation joins post-smoothing only");
    constexpr int GH = K + RES;  // ghost cells per side
    using C = SmoothK<T, GH>;
    constexpr int R = C::R, NR = C::NR, CPT = C::CPT;
    using PT = ProTile<T, GH>;
    // The cells' high couplings are other cells' low ones: exchanged through LDS, in arrays of their own
    // (the residual reads them again) or, where those would not fit (FP64 at K = 4: 160 KB), one axis after
    // another through the second z buffer.
    constexpr bool STAGED = sizeof(T) * 5 * NR > 128 * 1024;
    static_assert(!(STAGED && RES), "the residual reads the couplings from LDS");
    __shared__ T zs[2][NR];
    __shared__ T gxs[STAGED ? 1 : NR], gys[STAGED ? 1 : NR], gzs[STAGED ? 1 : NR];
    __shared__ T ctile[PRO ? PT::N : 1];
    __shared__ int nb27[27];
    __shared__ int pb[8];
    const int br = brick_or_idle(L);
    if (br < 0) return;
    const int t = threadIdx.x;
    // loads that depend on the brick only, issued before the gate's loads resolve
    const int nid = t < 27 ? L.nb27[27 * br + t] : -1;
    const int pid = (PRO && t < 8) ? L.parent8[8 * br + t] : -1;
    int px = 0, py = 0, pz = 0;
    if (PRO) {
        px = L.bxyz[3 * br] & 1;
        py = L.bxyz[3 * br + 1] & 1;
        pz = L.bxyz[3 * br + 2] & 1;
    }
    const BrickMeta m = L.meta[br];
    if (all_done(Q) || skip_smooth(Q, L, m)) return;
    if (t < 27) nb27[t] = nid;
    if (PRO && t < 8) pb[t] = pid;
    __syncthreads();
    // Coarse cells are indexed relative to coarse cell 8M - 8 of the brick B = 2M + p (per axis):
    // cube offset a is fine cell 16M + 8p + a - GH, i.e. fi = 16 + 8p + a - GH relative to fine
    // cell 16M - 16; its coarse cells are fi >> 1 (weight 3/4) and the one beside it toward fi's
    // parity side (1/4).  The tile starts at coarse index cmin = ((16 + 8p - GH) >> 1) - 1; coarse
    // index I lies in parent slot (I >> 3) - p, local cell I & 7.
    const int cmx = ((16 + 8 * px - GH) >> 1) - 1, cmy = ((16 + 8 * py - GH) >> 1) - 1,
              cmz = ((16 + 8 * pz - GH) >> 1) - 1;
    if (PRO) {
        constexpr int CT = PT::CT, NQ = (PT::N + C::THREADS - 1) / C::THREADS;
        T cv[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int e = t + q * C::THREADS;
            cv[q] = T(0);
            if (e < PT::N) {
                const int tc = e % CT, tb = (e / CT) % CT, ta = e / (CT * CT);
                const int Ia = cmx + ta, Ib = cmy + tb, Ic = cmz + tc;
                const int slot = (((Ia >> 3) - px) * 2 + ((Ib >> 3) - py)) * 2 + ((Ic >> 3) - pz);
                const int id = pb[slot];
                if (id >= 0) cv[q] = zcoarse[(long)id * BRICK_CELLS + (((Ia & 7) * 8 + (Ib & 7)) * 8 + (Ic & 7))];
            }
        }
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int e = t + q * C::THREADS;
            if (e < PT::N) ctile[e] = cv[q];
        }
        __syncthreads();
    }
    T rid[CPT], rr[CPT];
    T gxm[CPT], gxp[CPT], gym[CPT], gyp[CPT], gzm[CPT], gzp[CPT], zr[CPT];
#pragma unroll
    for (int q = 0; q < CPT; ++q) {
        const int e = t + q * C::THREADS;
        rid[q] = 0;
        rr[q] = 0;
        gxm[q] = gxp[q] = gym[q] = gyp[q] = gzm[q] = gzp[q] = zr[q] = T(0);
        if (e >= NR) continue;
        const int a = e / (R * R), b = (e / R) % R, c = e % R;
        // cube offset a is brick-local cell a - GH, in brick (-1, 0 or +1) + local (0..7)
        const int xa = a - GH + BRICK, xb = b - GH + BRICK, xc = c - GH + BRICK;  // 0 .. 23
        const int bi = xa >> 3, bj = xb >> 3, bk = xc >> 3;
        const int id = nb27[(bi * 3 + bj) * 3 + bk];
        T g0 = 0, g1 = 0, g2 = 0, z0 = 0;
        if (id >= 0) {
            const long cell = (long)id * BRICK_CELLS + (((xa & 7) * 8 + (xb & 7)) * 8 + (xc & 7));
            rid[q] = idiag[cell];
            rr[q] = rhs[cell];
            g0 = A.gx[cell];
            g1 = A.gy[cell];
            g2 = A.gz[cell];
            if (!FROM_ZERO) z0 = zin[cell];
            if (PRO && A.dir[cell] >= 0) {
                // k_prolong's correction of this cell
                constexpr int CT = PT::CT;
                const int fa = 16 + 8 * px + a - GH, fb = 16 + 8 * py + b - GH, fc = 16 + 8 * pz + c - GH;
                const int a0 = (fa >> 1) - cmx, b0 = (fb >> 1) - cmy, c0 = (fc >> 1) - cmz;
                const int a1 = (fa & 1) ? a0 + 1 : a0 - 1, b1 = (fb & 1) ? b0 + 1 : b0 - 1,
                          c1 = (fc & 1) ? c0 + 1 : c0 - 1;
                auto at = [&](int i, int j, int k) { return ctile[(i * CT + j) * CT + k]; };
                const T n = T(0.75), f = T(0.25);
                const T nk = L.flat ? T(1) : n, fk = L.flat ? T(0) : f;
                const T v = n * (n * (nk * at(a0, b0, c0) + fk * at(a0, b0, c1)) +
                                 f * (nk * at(a0, b1, c0) + fk * at(a0, b1, c1))) +
                            f * (n * (nk * at(a1, b0, c0) + fk * at(a1, b0, c1)) +
                                 f * (nk * at(a1, b1, c0) + fk * at(a1, b1, c1)));
                z0 = z0 + v;
            }
        }
        gxm[q] = g0;
        gym[q] = g1;
        gzm[q] = g2;
        zr[q] = z0;
        zs[0][e] = z0;
        if constexpr (!STAGED) {
            gxs[e] = g0;
            gys[e] = g1;
            gzs[e] = g2;
        }
    }
    // each thread keeps its cells' six couplings and own value in registers: a sweep reads only
    // the six neighbour values from LDS
    auto high = [&](const T *low, T *own, int axis) {
#pragma unroll
        for (int q = 0; q < CPT; ++q) {
            const int e = t + q * C::THREADS;
            if (e >= NR) continue;
            const int a = e / (R * R), b = (e / R) % R, c = e % R;
            if (axis == 0) own[q] = a < R - 1 ? low[e + R * R] : T(0);
            if (axis == 1) own[q] = b < R - 1 ? low[e + R] : T(0);
            if (axis == 2) own[q] = c < R - 1 ? low[e + 1] : T(0);
        }
    };
    if constexpr (STAGED) {
        auto stage = [&](const T *low, T *own, int axis) {
#pragma unroll
            for (int q = 0; q < CPT; ++q) {
                const int e = t + q * C::THREADS;
                if (e < NR) zs[1][e] = low[q];
            }
            __syncthreads();
            high(zs[1], own, axis);
            __syncthreads();
        };
        stage(gxm, gxp, 0);
        stage(gym, gyp, 1);
        stage(gzm, gzp, 2);
    } else {
        __syncthreads();
        high(gxs, gxp, 0);
        high(gys, gyp, 1);
        high(gzs, gzp, 2);
    }
#pragma unroll 1
    for (int s = 0; s < K; ++s) {
        const T *zc = zs[s & 1];
        T *zn = zs[(s & 1) ^ 1];
#pragma unroll
        for (int q = 0; q < CPT; ++q) {
            const int e = t + q * C::THREADS;
            if (e >= NR) continue;
            const int a = e / (R * R), b = (e / R) % R, c = e % R;
            T out = 0;
            if (rid[q] > T(0)) {
                const T zxm = a > 0 ? zc[e - R * R] : T(0), zxp = a < R - 1 ? zc[e + R * R] : T(0);
                const T zym = b > 0 ? zc[e - R] : T(0), zyp = b < R - 1 ? zc[e + R] : T(0);
                const T zzm = c > 0 ? zc[e - 1] : T(0), zzp = c < R - 1 ? zc[e + 1] : T(0);
                const T off = gxm[q] * zxm + gxp[q] * zxp + gym[q] * zym + gyp[q] * zyp + gzm[q] * zzm + gzp[q] * zzp;
                out = (T(1) - omega) * zr[q] + omega * rid[q] * (rr[q] + off);
            }
            zn[e] = out;
            zr[q] = out;
        }
        __syncthreads();
    }
    if (t < BRICK_CELLS) {
        const int li = t >> 6, lj = (t >> 3) & 7, lk = t & 7;
        const T *zz = zs[K & 1];
        const int e = ((li + GH) * R + (lj + GH)) * R + (lk + GH);
        const long c = (long)br * BRICK_CELLS + t;
        zout[c] = zz[e];
        if (RES) {
            // apply_row on the cube (the neighbours of the brick are exact after the K sweeps)
            const T dirc = A.dir[c];
            T out = 0;
            if (dirc >= 0) {
                const T gxm = gxs[e], gym = gys[e], gzm = gzs[e];
                const T gxp = gxs[e + R * R], gyp = gys[e + R], gzp = gzs[e + 1];
                const T off = gxm * zz[e - R * R] + gxp * zz[e + R * R] + gym * zz[e - R] + gyp * zz[e + R] +
                              gzm * zz[e - 1] + gzp * zz[e + 1];
                const T diag = dirc + ((gxm + gxp) + (gym + gyp) + (gzm + gzp));
                out = rhs[c] - (diag * zz[e] - off);
            }
            res[c] = out;
        }
    }
}

// Connected components of the coarsest brick of every grid ending on level L (block g: grid g):
// unknowns joined by a nonzero coupling, labelled by min-label propagation in LDS.  code[cell] =
// -1 off the unknowns, -2 in a component with a Dirichlet term (a nonsingular block), else the
// smallest cell index of its component: a pure-Neumann component, singular with the constants of
// the component as its null space (an all-fluid box, a pocket enclosed by solid).  Built once per
// projection; k_coarse_solve makes the right-hand side of such a component consistent.
template <class T>
__global__ __launch_bounds__(BRICK_CELLS) void k_coarse_components(LevelDesc L, OpDesc<T> A, int16_t *code) {
    __shared__ int lab[BRICK_CELLS];
    __shared__ int hasd[BRICK_CELLS];
    const int g = blockIdx.x;
    const GridLevel G = L.gl[g];
    if (!G.coarsest || G.brick_end <= G.brick_start) return;
    const int e = threadIdx.x;
    const long base = (long)G.brick_start * BRICK_CELLS;
    const long c = base + e;
    const int li = e >> 6, lj = (e >> 3) & 7, lk = e & 7;
    const T dirc = A.dir[c];
    const bool unk = dirc >= 0;
    // couplings to the six neighbours (the brick is the whole grid here: nothing outside it)
    const bool cxm = li > 0 && A.gx[c] > T(0), cxp = li < 7 && A.gx[c + 64] > T(0);
    const bool cym = lj > 0 && A.gy[c] > T(0), cyp = lj < 7 && A.gy[c + 8] > T(0);
    const bool czm = lk > 0 && A.gz[c] > T(0), czp = lk < 7 && A.gz[c + 1] > T(0);
    lab[e] = unk ? e : BRICK_CELLS;
    __syncthreads();
    // labels only decrease and always name a cell of the same component, so the propagation (with
    // pointer jumping) reaches the unique fixpoint, the smallest index of each component; at most
    // 512 rounds
    for (int it = 0; it < BRICK_CELLS; ++it) {
        int m = lab[e];
        if (unk) {
            m = min(m, lab[m]);  // pointer jumping: the label of the cell this one points to
            if (cxm) m = min(m, lab[e - 64]);
            if (cxp) m = min(m, lab[e + 64]);
            if (cym) m = min(m, lab[e - 8]);
            if (cyp) m = min(m, lab[e + 8]);
            if (czm) m = min(m, lab[e - 1]);
            if (czp) m = min(m, lab[e + 1]);
        }
        const bool changed = m < lab[e];
        __syncthreads();
        if (changed) lab[e] = m;
        if (!__syncthreads_or(changed)) break;
    }
    // whether each component has a Dirichlet term: dir of an unknown is a sum of conductances
    // (non-negative), so the component's sum of dir is positive exactly when one of its cells has
    // dir > 0 (a sum of non-negative numbers rounds to 0 only when every term is 0); each such cell
    // marks its root (concurrent stores of the same value)
    hasd[e] = 0;
    __syncthreads();
    if (unk && dirc > T(0)) hasd[lab[e]] = 1;
    __syncthreads();
    code[c] = !unk ? (int16_t)-1 : (hasd[lab[e]] ? (int16_t)-2 : (int16_t)lab[e]);
}

// Sums and sizes of the components of one brick in LDS, one entry per root cell.  The values are added
// as integers, scaled so that the component's largest has 53 bits: integer sums do not depend on the order of the
// atomic adds, 512 of them fit 64 bits, and the scaling loses at most 2^-54 of that value per
// term, no more than a sum in FP64 does.  Each component has a scale of its own: its values may be any
// number of orders of magnitude below those of another one in the brick.  (One thread adding a component
// of the whole brick in cell order took 35 us of the 47 us coarse solve of an all-fluid box; this takes
// about 1 us.)
//
// A barrier of the workgroup follows clear(), bound() and add() each.
struct ComponentSums {
    unsigned long long s[BRICK_CELLS];
    int n[BRICK_CELLS];
    unsigned top[BRICK_CELLS];  // upper half of the largest |value|
    __device__ __forceinline__ void clear(int e) {
        s[e] = 0;
        n[e] = 0;
        top[e] = 0;
    }
    __device__ __forceinline__ void bound(int root, double v) {
        if (root >= 0) atomicMax(&top[root], (unsigned)(__builtin_bit_cast(unsigned long long, fabs(v)) >> 32));
    }
    // (biased exponent b: the largest is below 2^(b - 1022))
    __device__ __forceinline__ int shift(int root) const { return 1075 - max((int)(top[root] >> 20), 1); }
    __device__ __forceinline__ void add(int root, double v) {
        if (root < 0) return;
        atomicAdd(&s[root], (unsigned long long)(long long)rint(ldexp(v, shift(root))));
        atomicAdd(&n[root], 1);
    }
    __device__ __forceinline__ double mean(int root) const {
        if (top[root] >= 0x7ff00000u) return __builtin_nan("");  // an infinity or NaN among the values
        return ldexp((double)(long long)s[root], -shift(root)) / n[root];
    }
};

// Coarse solve of every grid whose last level L is (one brick): block g handles grid g with
// `sweeps` damped-Jacobi sweeps from zero, in LDS.  DOT (finest level only): also the r.z partial
// of the grid's brick, as k_jacobi_dot stores it for grids with coarser levels.  CPT cells per
// thread (512 / CPT threads): fewer wavefronts make each sweep's barrier cheaper; every thread keeps
// its cells' couplings and own values in registers.
template <class T, int DOT, int CPT = 1>
__global__ __launch_bounds__(BRICK_CELLS / CPT) void k_coarse_solve(LevelDesc L, OpDesc<T> A,
                                                                    const T *__restrict__ rhs, T *__restrict__ z,
                                                                    int sweeps, T omega, Gate Q, RedBuf R,
                                                                    const int16_t *__restrict__ code) {
    constexpr int NT = BRICK_CELLS / CPT;
    __shared__ T zs[2][BRICK_CELLS];
    __shared__ double lds[32];
    __shared__ int16_t cc[BRICK_CELLS];
    __shared__ ComponentSums sums;
    if (all_done(Q)) return;
    const int g = blockIdx.x;
    const GridLevel G = L.gl[g];
    if (!G.coarsest || G.brick_end <= G.brick_start || (Q.S && Q.S[g].done)) return;
    const int t = threadIdx.x;
    const long base = (long)G.brick_start * BRICK_CELLS;
    T gxm[CPT], gym[CPT], gzm[CPT], gxp[CPT], gyp[CPT], gzp[CPT], diag[CPT], inv[CPT], r[CPT], zr[CPT];
    bool unk[CPT];
#pragma unroll
    for (int u = 0; u < CPT; ++u) {
        const int e = t + u * NT;
        const int li = e >> 6, lj = (e >> 3) & 7, lk = e & 7;
        const long c = base + e;
        const T dirc = A.dir[c];
        gxm[u] = A.gx[c];
        gym[u] = A.gy[c];
        gzm[u] = A.gz[c];
        gxp[u] = li < 7 ? A.gx[c + 64] : T(0);
        gyp[u] = lj < 7 ? A.gy[c + 8] : T(0);
        gzp[u] = lk < 7 ? A.gz[c + 1] : T(0);
        diag[u] = dirc + ((gxm[u] + gxp[u]) + (gym[u] + gyp[u]) + (gzm[u] + gzp[u]));
        unk[u] = dirc >= 0 && diag[u] > 0;
        r[u] = rhs[c];
        inv[u] = unk[u] ? omega / diag[u] : T(0);
        cc[e] = code[c];
    }
    // A pure-Neumann component (k_coarse_components) is singular: its right-hand side is made
    // consistent (its mean over the component removed) so that the sweeps do not grow the
    // component's constant mode, which the Krylov iteration would carry into the pressure.
    bool sing = false;
#pragma unroll
    for (int u = 0; u < CPT; ++u) sing = sing || cc[t + u * NT] >= 0;
    T rs[CPT];  // the right-hand side the sweeps solve (r itself, or made consistent)
#pragma unroll
    for (int u = 0; u < CPT; ++u) rs[u] = r[u];
    if (__syncthreads_or(sing)) {
#pragma unroll
        for (int u = 0; u < CPT; ++u) sums.clear(t + u * NT);
        __syncthreads();
#pragma unroll
        for (int u = 0; u < CPT; ++u) sums.bound(cc[t + u * NT], (double)r[u]);
        __syncthreads();
#pragma unroll
        for (int u = 0; u < CPT; ++u) sums.add(cc[t + u * NT], (double)r[u]);
        __syncthreads();
#pragma unroll
        for (int u = 0; u < CPT; ++u)
            if (cc[t + u * NT] >= 0) rs[u] = r[u] - (T)sums.mean(cc[t + u * NT]);
    }
#pragma unroll
    for (int u = 0; u < CPT; ++u) {
        zr[u] = unk[u] ? inv[u] * rs[u] : T(0);
        zs[0][t + u * NT] = zr[u];
    }
    __syncthreads();
    int cur = 0;
    for (int s = 1; s < sweeps; ++s) {
        const T *zz = zs[cur];
        T out[CPT];
#pragma unroll
        for (int u = 0; u < CPT; ++u) {
            const int e = t + u * NT;
            const int li = e >> 6, lj = (e >> 3) & 7, lk = e & 7;
            out[u] = T(0);
            if (unk[u]) {
                const T off = gxm[u] * (li > 0 ? zz[e - 64] : T(0)) + gxp[u] * (li < 7 ? zz[e + 64] : T(0)) +
                              gym[u] * (lj > 0 ? zz[e - 8] : T(0)) + gyp[u] * (lj < 7 ? zz[e + 8] : T(0)) +
                              gzm[u] * (lk > 0 ? zz[e - 1] : T(0)) + gzp[u] * (lk < 7 ? zz[e + 1] : T(0));
                out[u] = zr[u] + inv[u] * (rs[u] - (diag[u] * zr[u] - off));
            }
        }
#pragma unroll
        for (int u = 0; u < CPT; ++u) {
            zs[cur ^ 1][t + u * NT] = out[u];
            zr[u] = out[u];
        }
        __syncthreads();
        cur ^= 1;
    }
    double part = 0.0;
#pragma unroll
    for (int u = 0; u < CPT; ++u) {
        z[base + t + u * NT] = zr[u];
        part += (double)r[u] * (double)zr[u];
    }
    if (DOT) {
        part = block_sum(part, lds);
        store_partials(R, G.brick_start, part, 0.0);
    }
}

// The bottom of the V-cycle (BottomGrid) of one grid in one 1024-thread workgroup: from the first
// level of at most 8 stored bricks, whose right-hand side and pre-smoothing from zero the restriction
// has written, down to the coarsest brick and back up.  128 threads per brick hold its cells as rows of
// four (Row4), with the operator in registers and the vectors that neighbours read in LDS.
//
// These levels are a few thousand cells: each launch on them costs its boundary and two to three
// dependent trips to memory (another XCD wrote the data), 3 to 5 us for well under 1 us of work, and
// the coarsest brick's sweeps a barrier of eight wavefronts each.  In one workgroup only the first
// loads go to memory.  Measured per V-cycle on the last two levels of a 32^3 grid (V(1,1), 48 sweeps on
// the coarsest brick): 26 us in five launches, 17 us here, of which 8 us are those sweeps; of a 256^3
// grid (V(2,2), 4 sweeps): 35 us in eight launches, 17 us here.  Eight bricks fill the 1024 threads with one brick each; a level of 16 or more
// would make the one CU's issue the bound (about 2 us of it per smoothing step and 8 bricks, as long
// as the launch it saves).
// Every value is formed by the operations of the kernels for larger levels in their order
// (k_post_local4, k_residual4, k_restrict_pre, k_prolong4, k_coarse_solve; the restriction's nested
// sums one axis at a time), so both forms give the same bits.
constexpr int BOTTOM_THREADS = BOTTOM_BRICKS * ROW4_THREADS;

// Damped-Jacobi sweeps from zero on the coarsest brick (k_coarse_solve's operations in its order), two
// cells (z[0], z[1]) per lane of the first four wavefronts; every thread of the workgroup calls it
// (barriers).  A 16-lane DPP row holds the eight y rows of one x and one half of z: lane bits kqlo, lj
// (3), kqhi, li (3), cells 4 kqhi + 2 kqlo and the next.  So the y neighbours are two lanes away in the
// DPP row, one z neighbour is the lane's other cell, the other the pair's or, across the halves, through
// LDS (zb: 2 x 512 floats), as the x neighbours are.  One wavefront per SIMD: with four cells per lane of
// two wavefronts a sweep took 500 cycles, its 76 instructions issued one after the other.
struct BottomCells {
    float xm, xp, ym, yp, zm, zp;  // couplings
    float diag, inv, rs;
};
__device__ __forceinline__ void bottom_solve(const BottomCells (&c)[2], float z[2], float *zb, int sweeps, bool mine,
                                             int base, int kqlo) {
    if (mine) {
        z[0] = c[0].inv * c[0].rs;
        z[1] = c[1].inv * c[1].rs;
        *reinterpret_cast<float2 *>(zb + base) = make_float2(z[0], z[1]);
    }
    __syncthreads();
    if (!mine) {  // the other wavefronts only keep the barriers
        for (int s = 1; s < sweeps; ++s) __syncthreads();
        return;
    }
    // (a coupling is 0 across the brick's faces; its value is then the cell's own)
    const int ixm = base >= 64 ? base - 64 : base, ixp = base < 448 ? base + 64 : base;
    const int iz = kqlo ? ((base & 7) < 6 ? base + 2 : base) : ((base & 7) ? base - 1 : base);
    for (int s = 1; s < sweeps; ++s) {
        const float *zc = zb + ((s & 1) ? 0 : BRICK_CELLS);
        float *zn = zb + ((s & 1) ? BRICK_CELLS : 0);
        const float2 xm = *reinterpret_cast<const float2 *>(zc + ixm), xp = *reinterpret_cast<const float2 *>(zc + ixp);
        const float far = zc[iz];
        const float sw0 = sgs_dpp<DPP_SWAP_PAIRS>(z[0]), sw1 = sgs_dpp<DPP_SWAP_PAIRS>(z[1]);
        float ym[2], yp[2], d[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            ym[j] = c[j].ym * sgs_dpp<DPP_ROW_SHR2>(z[j]);
            yp[j] = c[j].yp * sgs_dpp<DPP_ROW_SHL2>(z[j]);
            d[j] = c[j].diag * z[j];
        }
        const float zp0 = c[0].zp * z[1], zm1 = c[1].zm * z[0];
        __builtin_amdgcn_sched_barrier(0);  // the products of registers cover the LDS reads
        const float zm0 = c[0].zm * (kqlo ? sw1 : far), zp1 = c[1].zp * (kqlo ? far : sw0);
        const float off0 = c[0].xm * xm.x + c[0].xp * xp.x + ym[0] + yp[0] + zm0 + zp0;
        const float off1 = c[1].xm * xm.y + c[1].xp * xp.y + ym[1] + yp[1] + zm1 + zp1;
        z[0] = z[0] + c[0].inv * (c[0].rs - (d[0] - off0));
        z[1] = z[1] + c[1].inv * (c[1].rs - (d[1] - off1));
        *reinterpret_cast<float2 *>(zn + base) = make_float2(z[0], z[1]);
        __syncthreads();
    }
}

__global__ __launch_bounds__(BOTTOM_THREADS) void k_bottom(const BottomGrid *__restrict__ grids, int pre, int post,
                                                           int sweeps, float omega, int slot, Gate Q) {
    constexpr int E = 18, NC = BOTTOM_BRICKS * BRICK_CELLS;
    __shared__ __align__(16) float zl[NC];  // z of the level in hand
    __shared__ __align__(16) float ex[BOTTOM_BRICKS * SGS_LDS];  // the smoother's exchange; the residual that is restricted
    __shared__ __align__(16) float rc[NC];  // the next level's right-hand side, then its z
    __shared__ __align__(16) float t1[E * E * 8];  // the restriction's partial sums along z (and the coarse sweeps'
    __shared__ float t2[E * 8 * 8];    // buffers), then along y
    __shared__ __align__(16) float cop[4][BRICK_CELLS];  // the coarsest brick's gx, gy, gz, dir
    __shared__ __align__(16) int cid[64 * BOTTOM_BRICKS];  // child64 and parent8 of the level in hand
    __shared__ __align__(16) int pb[BOTTOM_BRICKS][8];
    __shared__ int16_t code[BRICK_CELLS];
    __shared__ int any[4];
    __shared__ ComponentSums sums;
    const BottomGrid &G = grids[blockIdx.x];
    const int n = G.n;
    if (n == 0 || all_done(Q) || (Q.S && Q.S[blockIdx.x].done)) return;
    const int t = threadIdx.x, q = t % ROW4_THREADS;
    const int own = __builtin_amdgcn_readfirstlane(t / ROW4_THREADS);  // (a wavefront works on one brick)
    const int li = q >> 4, lj = (q >> 1) & 7, h = q & 1;

    // the coarsest brick's operator, kept in LDS
    if (own < 4) {
        const BottomLevel &L = G.lev[n - 1];
        const float *const from[4] = {L.gx, L.gy, L.gz, L.dir};
        *reinterpret_cast<float4 *>(&cop[own][4 * q]) = ld4(from[own], 4 * q);
    }
    if (t >= BOTTOM_THREADS - BRICK_CELLS) code[t - (BOTTOM_THREADS - BRICK_CELLS)] = G.code[t - (BOTTOM_THREADS - BRICK_CELLS)];

    // The level in hand: the thread's four cells by colour group (SgsRow) with all of their couplings, so
    // that neither the sweeps nor the residual select or reload anything.  Neighbour bricks count from
    // the grid's first brick of the level.  The wavefronts of bricks the level does not have keep zeros
    // and the barriers.
    const bool c1 = sgs_col1(q);
    const int me = own * ROW4_THREADS + q;
    SgsCells A{};
    SgsRow diag{}, ez{};  // diagonal; couplings across the brick's z faces
    SgsRow r{}, z{};
    int ixm = me, ixp = me, iym = me, iyp = me, iz = 4 * me;  // the rows beside the thread's, the cell across z
    int unk = 0;                        // bit j: the row's cell j is an unknown
    bool work = false;
    int parity = 0;  // of the brick's position (x, y, z)
    auto load = [&](const BottomLevel &L, const BottomLevel &C) {
        work = own < L.nb;
        A = SgsCells{};
        diag = ez = r = z = SgsRow{};
        ixm = ixp = iym = iyp = me;
        iz = 4 * me;
        // every load of the level at once, its tables included; the operator's rows to LDS
        const int nc = C.nb;
        const int id64 = t < 64 * nc ? C.child64[t] : -1, id8 = t < 8 * L.nb ? L.parent8[t] : -1;
        BrickMeta m{};
        float own_gz[4] = {0.0f, 0.0f, 0.0f, 0.0f}, own_dir[4] = {0.0f, 0.0f, 0.0f, 0.0f}, own_id[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (work) {
            m = L.meta[own];
            parity = (L.bxyz[3 * own] & 1) << 2 | (L.bxyz[3 * own + 1] & 1) << 1 | (L.bxyz[3 * own + 2] & 1);
            const float4 gx0 = ld4(L.gx, 4 * me), gy0 = ld4(L.gy, 4 * me);
            load4(L.gz, 4 * me, own_gz);
            load4(L.dir, 4 * me, own_dir);
            load4(L.idiag, 4 * me, own_id);
            reinterpret_cast<float4 *>(zl)[me] = gx0;
            reinterpret_cast<float4 *>(ex)[me] = gy0;
            t1[me] = own_gz[0];
        }
        if (t < 64 * nc) cid[t] = id64 >= 0 ? id64 - L.brick_start : -1;
        if (t < 8 * L.nb) pb[t >> 3][t & 7] = id8 >= 0 ? id8 - C.brick_start : -1;
        __syncthreads();
        if (!work) return;
#pragma unroll
        for (int d = 0; d < 6; ++d) m.nbr[d] = m.nbr[d] >= 0 ? m.nbr[d] - L.brick_start : -1;
        float dg[4], gz[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        // the high couplings are the next cells' low ones, in rows of other threads
        Row4Coef<float> g;
        const float4 *lx = reinterpret_cast<const float4 *>(zl), *ly = reinterpret_cast<const float4 *>(ex);
        unpack4(lx[me], g.gxm);
        unpack4(ly[me], g.gym);
#pragma unroll
        for (int j = 0; j < 4; ++j) g.gzm[j] = own_gz[j];
        // the rows beside the thread's, in the brick or across its faces; where no brick is stored the
        // coupling is 0, and the row the thread's own
        const int jxp = li < 7 ? me + 16 : m.nbr[NB_XP] >= 0 ? m.nbr[NB_XP] * ROW4_THREADS + q - 112 : -1;
        const int jyp = lj < 7 ? me + 2 : m.nbr[NB_YP] >= 0 ? m.nbr[NB_YP] * ROW4_THREADS + q - 14 : -1;
        const int jz = !h ? me + 1 : m.nbr[NB_ZP] >= 0 ? m.nbr[NB_ZP] * ROW4_THREADS + q - 1 : -1;
        unpack4(jxp >= 0 ? lx[jxp] : make_float4(0.0f, 0.0f, 0.0f, 0.0f), g.gxp);
        unpack4(jyp >= 0 ? ly[jyp] : make_float4(0.0f, 0.0f, 0.0f, 0.0f), g.gyp);
        if (jxp >= 0) ixp = jxp;
        if (jyp >= 0) iyp = jyp;
        if (li > 0) ixm = me - 16;
        else if (m.nbr[NB_XM] >= 0) ixm = m.nbr[NB_XM] * ROW4_THREADS + q + 112;
        if (lj > 0) iym = me - 2;
        else if (m.nbr[NB_YM] >= 0) iym = m.nbr[NB_YM] * ROW4_THREADS + q + 14;
        g.gzp[0] = g.gzm[1];
        g.gzp[1] = g.gzm[2];
        g.gzp[2] = g.gzm[3];
        g.gzp[3] = jz >= 0 ? t1[jz] : 0.0f;
        unk = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            dg[j] = own_dir[j] >= 0 ? own_dir[j] + ((g.gxm[j] + g.gxp[j]) + (g.gym[j] + g.gyp[j]) + (g.gzm[j] + g.gzp[j]))
                                    : 0.0f;
            unk |= own_dir[j] >= 0 ? 1 << j : 0;
        }
        A = sgs_cells(g, own_id, q);
        diag = sgs_group(dg, c1);
        // across z the row's col0 is the same (across x and y the other one)
        const int nz = h ? m.nbr[NB_ZP] : m.nbr[NB_ZM];
        if (h) gz[3] = g.gzp[3];
        else gz[0] = g.gzm[0];
        ez = sgs_group(gz, c1);
        if (nz >= 0) iz = 4 * (nz * ROW4_THREADS + (q ^ 1)) + (h ? (c1 ? 2 : 0) : (c1 ? 1 : 3));
    };
    // rhs - A z of the thread's cells; zl: z by row and group
    auto residual = [&]() {
        const float4 *zr = reinterpret_cast<const float4 *>(zl);
        const float4 xm = zr[ixm], xp = zr[ixp], ym = zr[iym], yp = zr[iyp];
        const float fz = zl[iz];
        const float sp0 = sgs_dpp<DPP_SWAP_PAIRS>(z.p0), sp1 = sgs_dpp<DPP_SWAP_PAIRS>(z.p1);
        const float sq0 = sgs_dpp<DPP_SWAP_PAIRS>(z.q0), sq1 = sgs_dpp<DPP_SWAP_PAIRS>(z.q1);
        // across the row's lower end (h = 0) or upper end (h = 1) lies the next brick, else the pair's lane
        const float lo0 = h ? sp1 : fz, hi0 = h ? fz : sp0, lo1 = h ? sq1 : fz, hi1 = h ? fz : sq0;
        SgsRow o;
        o.p0 = r.p0 - (diag.p0 * z.p0 - sgs_ordered<AT_P0>(A.P0, c1, xm.z, xp.z, ym.z, yp.z, z.q0, z.q1, lo1, A.P0.zs + ez.p0));
        o.p1 = r.p1 - (diag.p1 * z.p1 - sgs_ordered<AT_P1>(A.P1, c1, xm.w, xp.w, ym.w, yp.w, z.q0, z.q1, hi1, A.P1.zs + ez.p1));
        o.q0 = r.q0 - (diag.q0 * z.q0 - sgs_ordered<AT_Q0>(A.Q0, c1, xm.x, xp.x, ym.x, yp.x, z.p0, z.p1, lo0, A.Q0.zs + ez.q0));
        o.q1 = r.q1 - (diag.q1 * z.q1 - sgs_ordered<AT_Q1>(A.Q1, c1, xm.y, xp.y, ym.y, yp.y, z.p0, z.p1, hi0, A.Q1.zs + ez.q1));
        return o;
    };
    auto publish = [&]() {
        reinterpret_cast<float4 *>(zl)[me] = make_float4(z.p0, z.p1, z.q0, z.q1);
        __syncthreads();
    };
    float2 *const exq = reinterpret_cast<float2 *>(ex) + own * 2 * SGS_PAIRS;
    // z += M_b (rhs - A z)
    auto smooth = [&]() {
        const SgsRow e = sgs_sweeps<LOCAL_SGS_SWEEPS_COARSE>(A, residual(), exq, q);
        z = SgsRow{z.p0 + e.p0, z.p1 + e.p1, z.q0 + e.q0, z.q1 + e.q1};
        publish();  // (every read of zl lies before the sweeps' barriers)
    };
    auto take = [&](const float *from) {  // the thread's row, by group
        float v[4];
        load4(from, (long)4 * me, v);
        return sgs_group(v, c1);
    };
    auto give = [&](float *to, const SgsRow &g) {
        float v[4];
        sgs_ungroup(g, c1, v);
        store4(to, (long)4 * me, v);
    };

    for (int d = 0; d + 1 < n; ++d) {
        const BottomLevel &L = G.lev[d], &C = G.lev[d + 1];
        load(L, C);
        if (work) {
            if (d == 0) {
                r = take(L.rhs);
                z = take(L.z);
            } else {
                float v[4];
                load4((const float *)rc, (long)4 * me, v);
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = (unk >> j) & 1 ? v[j] : 0.0f;
                r = sgs_group(v, c1);
            }
        }
        __syncthreads();  // the operator's rows in zl and ex have been read
        if (d > 0) z = sgs_sweeps_ordered<LOCAL_SGS_SWEEPS_COARSE>(A, r, exq, q, c1);  // from zero, as k_restrict_pre
        publish();
        for (int s = 1; s < pre; ++s) smooth();
        give(ex, residual());
        if (work && d + 2 < n) {  // for the way up (this thread reads them back)
            give(L.z, z);
            if (d > 0) give(L.rhs, r);
        }
        __syncthreads();
        // k_restrict_pre's sums, one coarse brick after another.  Along z first: thread e forms the eight
        // sums of the tile's row (a, b), from the two whole rows of fine bricks in it and a cell at each end.
        const bool flat = L.flat;
        const float w0 = 0.25f, w1 = 0.75f;
        for (int B = 0; B < C.nb; ++B) {
            if (t < E * E) {
                const int b = t % E, a = t / E;
                const int rowcell = (((a + 7) & 7) * 8 + ((b + 7) & 7)) * 8;
                const int4 id = reinterpret_cast<const int4 *>(cid + 64 * B)[((a + 7) >> 3) * 4 + ((b + 7) >> 3)];
                const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                auto row = [&](int brick, int half) {
                    return brick >= 0 ? *reinterpret_cast<const float4 *>(&ex[brick * BRICK_CELLS + rowcell + 4 * half]) : zero;
                };
                float v[E];
                v[0] = id.x >= 0 ? ex[id.x * BRICK_CELLS + rowcell + 7] : 0.0f;
                unpack4(row(id.y, 0), v + 1);
                unpack4(row(id.y, 1), v + 5);
                unpack4(row(id.z, 0), v + 9);
                unpack4(row(id.z, 1), v + 13);
                v[17] = id.w >= 0 ? ex[id.w * BRICK_CELLS + rowcell] : 0.0f;
                float o[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const float *u = v + 2 * k;
                    o[k] = flat ? 0.0f * u[0] + 1.0f * u[1] + 0.0f * u[2] + 0.0f * u[3]
                                : w0 * u[0] + w1 * u[1] + w1 * u[2] + w0 * u[3];
                }
                store4(t1, 8 * t, o);
                store4(t1, 8 * t + 4, o + 4);
            }
            __syncthreads();
            for (int e = t; e < E * 64; e += BOTTOM_THREADS) {
                const int k = e & 7, j = (e >> 3) & 7, a = e >> 6;
                const float *row = &t1[(a * E + 2 * j) * 8 + k];
                float acc = 0.0f;
                acc += w0 * row[0];
                acc += w1 * row[8];
                acc += w1 * row[16];
                acc += w0 * row[24];
                t2[e] = acc;
            }
            __syncthreads();
            if (t < BRICK_CELLS) {
                const float *row = &t2[(2 * (t >> 6)) * 64 + (t & 63)];
                float acc = 0.0f;
                acc += w0 * row[0];
                acc += w1 * row[64];
                acc += w1 * row[128];
                acc += w0 * row[192];
                rc[B * BRICK_CELLS + t] = acc;
            }
        }
        __syncthreads();
    }

    // the coarsest brick: k_coarse_solve
    {
        const BottomLevel &L = G.lev[n - 1];
        const bool mine = own < 2;
        const int kqlo = t & 1, base = ((t >> 5) & 7) * 64 + ((t >> 1) & 7) * 8 + ((t >> 4) & 1) * 4 + 2 * kqlo;
        BottomCells c[2]{};
        int cc[2] = {-1, -1};
        float cz[2] = {0.0f, 0.0f};
        __syncthreads();
        if (mine) {
            const float *gx = cop[0], *gy = cop[1], *gz = cop[2], *dir = cop[3];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int e = base + j, ei = e >> 6, ej = (e >> 3) & 7, ek = e & 7;
                BottomCells &o = c[j];
                o.xm = gx[e];
                o.ym = gy[e];
                o.zm = gz[e];
                o.xp = ei < 7 ? gx[e + 64] : 0.0f;
                o.yp = ej < 7 ? gy[e + 8] : 0.0f;
                o.zp = ek < 7 ? gz[e + 1] : 0.0f;
                o.diag = dir[e] + ((o.xm + o.xp) + (o.ym + o.yp) + (o.zm + o.zp));
                o.inv = dir[e] >= 0 && o.diag > 0 ? omega / o.diag : 0.0f;
                o.rs = n == 1 ? L.rhs[e] : dir[e] >= 0 ? rc[e] : 0.0f;
                cc[j] = code[e];
            }
        }
        const unsigned long long vote = __ballot(cc[0] >= 0 || cc[1] >= 0);
        if (mine && (t & 63) == 0) any[t >> 6] = vote != 0;
        __syncthreads();
        if (any[0] | any[1] | any[2] | any[3]) {
            if (t < BRICK_CELLS) sums.clear(t);
            __syncthreads();
#pragma unroll
            for (int j = 0; j < 2; ++j) sums.bound(cc[j], (double)c[j].rs);
            __syncthreads();
#pragma unroll
            for (int j = 0; j < 2; ++j) sums.add(cc[j], (double)c[j].rs);
            __syncthreads();
#pragma unroll
            for (int j = 0; j < 2; ++j)
                if (cc[j] >= 0) c[j].rs = c[j].rs - (float)sums.mean(cc[j]);
        }
        bottom_solve(c, cz, t1, sweeps, mine, base, kqlo);
        if (mine) {
            float *to = n > 1 ? rc : slot && !L.deepest ? L.tmp : L.z;
            to[base] = cz[0];
            to[base + 1] = cz[1];
        }
        __syncthreads();
    }

    for (int d = n - 2; d >= 0; --d) {
        const BottomLevel &L = G.lev[d], &C = G.lev[d + 1];
        if (d + 2 < n) {
            load(L, C);
            if (work) {
                r = take(L.rhs);
                z = take(L.z);
            }
            __syncthreads();
        }
        // k_prolong4's correction from rc
        if (work) {
            const int px = parity >> 2, py = (parity >> 1) & 1, pz = parity & 1;
            const int a0 = (li >> 1) + 1, b0 = (lj >> 1) + 1;
            const int a1 = (li & 1) ? a0 + 1 : a0 - 1, b1 = (lj & 1) ? b0 + 1 : b0 - 1;
            // the four coarse values 2h .. 2h + 3 along z of tile row (a, b)
            auto row = [&](int a, int b, float o[4]) {
                const int ia = 4 * px + 7 + a, ib = 4 * py + 7 + b;
                const int rowslot = (((ia >> 3) - px) * 2 + ((ib >> 3) - py)) * 2, rowcell = ((ia & 7) * 8 + (ib & 7)) * 8;
                const int2 id = *reinterpret_cast<const int2 *>(&pb[own][rowslot]);  // both bricks of the row
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int ic = 4 * pz + 7 + 2 * h + u;
                    const int b = (ic >> 3) - pz ? id.y : id.x;
                    o[u] = b >= 0 ? rc[b * BRICK_CELLS + rowcell + (ic & 7)] : 0.0f;
                }
            };
            float c00[4], c01[4], c10[4], c11[4];
            row(a0, b0, c00);
            row(a0, b1, c01);
            row(a1, b0, c10);
            row(a1, b1, c11);
            const float nn = 0.75f, f = 0.25f;
            const float nk = L.flat ? 1.0f : nn, fk = L.flat ? 0.0f : f;
            float add[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int u0 = (j >> 1) + 1, u1 = (j & 1) ? u0 + 1 : u0 - 1;
                const float v = nn * (nn * (nk * c00[u0] + fk * c00[u1]) + f * (nk * c01[u0] + fk * c01[u1])) +
                                f * (nn * (nk * c10[u0] + fk * c10[u1]) + f * (nk * c11[u0] + fk * c11[u1]));
                add[j] = (unk >> j) & 1 ? v : 0.0f;
            }
            const SgsRow a = sgs_group(add, c1);
            z.p0 += a.p0;
            z.p1 += a.p1;
            z.q0 += a.q0;
            z.q1 += a.q1;
        }
        publish();
        for (int s = 0; s < post; ++s) smooth();
        if (work) {
            give(d > 0 ? rc : slot && !L.deepest ? L.tmp : L.z, z);
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------------------ output (one grid)
// Dense export of the level-0 system: diag (0 off the unknowns), the low-face couplings and the
// right-hand side, all cell-indexed.
__global__ void k_export_system(GridDesc G, LevelDesc L, GridLevel GL, OpDesc<double> A, const double *__restrict__ b,
                                double *diag, double *gx, double *gy, double *gz, double *rhs) {
    const size_t M = (size_t)G.w * G.h * G.d;
    const size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= M) return;
    int i, j, k;
    unflatten((unsigned)c, (unsigned)G.h, (unsigned)G.d, i, j, k);
    const bool stored = L.bmap[GL.bmap_off + ((i >> 3) * GL.nby + (j >> 3)) * GL.nbz + (k >> 3)] >= 0;
    const double dirc = stored ? level_value(L, GL, A.dir, i, j, k) : -1.0;
    const bool unk = dirc >= 0.0;
    const double gxm = level_value(L, GL, A.gx, i, j, k), gym = level_value(L, GL, A.gy, i, j, k),
                 gzm = level_value(L, GL, A.gz, i, j, k);
    const double gxp = level_value(L, GL, A.gx, i + 1, j, k), gyp = level_value(L, GL, A.gy, i, j + 1, k),
                 gzp = level_value(L, GL, A.gz, i, j, k + 1);
    diag[c] = unk ? dirc + ((gxm + gxp) + (gym + gyp) + (gzm + gzp)) : 0.0;
    gx[c] = gxm;
    gy[c] = gym;
    gz[c] = gzm;
    rhs[c] = unk ? level_value(L, GL, b, i, j, k) : 0.0;
}

// Output of a grid: m_pressure, the dense float (and optional FP64) pressure, 0 off the unknowns
// (macpressuresolver3.cpp:245-248), the unknown mask (the labelling's cell flag, bit 1), and the velocity
// update (:252-268): open interior faces lose dt*(P1-P0)/(rho*dx) with P stored in float and P1-P0
// taken in float; all other (active) faces are switched off (0), as the domain's boundary faces are (their
// area is 0), which stay active where the cell inside holds liquid.
//
// One pass for all of it, on columns of OUT_PLANES cells along x per thread and 64 consecutive cells of a
// plane per wavefront (whatever the row length), so that the index arithmetic is done once per column, a
// cell's low neighbour along x is in registers, and the pressure comes from the bricks instead of a dense
// copy.  A wavefront with only air around (most of a domain) reads the level set and writes zeros.
// Bound by its traffic: at 256^3 (28% liquid, FP64 samples) 176 us, 2.7 TB/s; a scatter and an update
// with one node per thread took 46 + 223 us.  120x168x89, all liquid with activity masks: 41 us.
struct OutputGrid {
    GridDesc G;
    GridLevel GL;
    float *P;         // dense outputs (or nullptr)
    double *P64, *scene;
    const uint8_t *cflag;
    uint8_t *unknown_out;
};
constexpr int OUT_THREADS = 256, OUT_PLANES = 4;
// A long grid of few cells per plane: a workgroup takes as many slabs of OUT_PLANES planes as its threads hold
// whole, in a kernel of its own (THIN), since the slab then differs between the lanes: 112 registers instead of 100, and
// 157 us instead of 147 for 256^3 without liquid.  60000x2x2 without liquid: 42 us with a slab per workgroup, 9 us here.
static inline bool output_thin(const GridDesc &G) { return G.h * G.d <= OUT_THREADS / 2; }
static inline int output_blocks(const GridDesc &G) {
    const unsigned HD = (unsigned)G.h * (unsigned)G.d, slabs = (unsigned)((G.w + OUT_PLANES - 1) / OUT_PLANES);
    if (output_thin(G)) {
        const unsigned per = OUT_THREADS / HD;
        return (int)((slabs + per - 1) / per);
    }
    return (int)((HD + OUT_THREADS - 1) / OUT_THREADS * slabs);
}

// A face's new velocity and activity; an inactive face keeps its velocity.
__device__ __forceinline__ void put_face(const GridDesc &G, int dim, size_t f, float u, bool keep) {
    const bool inactive = G.active[dim] && !G.active[dim][f];
    if (!inactive) G.vel[dim][f] = u;
    if (G.active_out[dim]) G.active_out[dim][f] = keep && !inactive;
}

// Level set of a column from plane i0 - 1 on and of the low neighbours along y and z (clamped).
struct OutputPhi {
    double c[OUT_PLANES + 1], j[OUT_PLANES], k[OUT_PLANES];
};
template <class Tp>
__device__ __forceinline__ void output_phi(const void *a, size_t c0, int n, size_t di, size_t dj, size_t dk, size_t HD,
                                           OutputPhi &o) {
    const Tp *__restrict__ phi = (const Tp *)a;
    o.c[0] = (double)phi[c0 - di];
#pragma unroll
    for (int p = 0; p < OUT_PLANES; ++p) {
        const size_t c = c0 + (size_t)(p < n ? p : 0) * HD;
        o.c[p + 1] = (double)phi[c];
        o.j[p] = (double)phi[c - dj];
        o.k[p] = (double)phi[c - dk];
    }
}

template <int THIN>
__global__ __launch_bounds__(OUT_THREADS) void k_output(GridTable<OutputGrid> T, LevelDesc L,
                                                        const double *__restrict__ x) {
#pragma clang fp contract(off)
    int local;
    const int entry = table_grid(T, local);
    if (entry < 0) return;
    const OutputGrid &F = T.g[entry];
    const GridDesc &G = F.G;
    const unsigned HD = (unsigned)G.h * (unsigned)G.d, ne = (HD + OUT_THREADS - 1) / OUT_THREADS;
    unsigned slab = (unsigned)local / ne, e = ((unsigned)local - slab * ne) * OUT_THREADS + threadIdx.x;
    if (THIN) {
        const unsigned per = OUT_THREADS / HD, q = threadIdx.x / HD;
        slab = (unsigned)local * per + q;
        e = q < per && slab * OUT_PLANES < (unsigned)G.w ? threadIdx.x - q * HD : HD;
    }
    if (e >= HD) return;
    const int j = (int)(e / (unsigned)G.d), k = (int)(e - (unsigned)j * (unsigned)G.d);
    const int i0 = (int)slab * OUT_PLANES, n = min(OUT_PLANES, G.w - i0);
    const Exist E = exist_of(G);
    const size_t c0 = cell_index(G, i0, j, k);
    // the bricks of the column and of its low neighbours: the planes lie in one brick layer
    const int *bm = L.bmap + F.GL.bmap_off;
    const int layer = F.GL.nby * F.GL.nbz, at = (i0 >> 3) * layer + (j >> 3) * F.GL.nbz + (k >> 3);
    const int b = bm[at];
    const int bi = i0 == 0 ? -1 : (i0 & 7) ? b : bm[at - layer];
    const int bj = j == 0 ? -1 : (j & 7) ? b : bm[at - F.GL.nbz];
    const int bk = k == 0 ? -1 : (k & 7) ? b : bm[at - 1];
    OutputPhi ph;
    const size_t dj = j > 0 ? G.d : 0, dk = k > 0;
    if (G.phi64) output_phi<double>(G.phi, c0, n, i0 > 0 ? HD : 0, dj, dk, HD, ph);
    else output_phi<float>(G.phi, c0, n, i0 > 0 ? HD : 0, dj, dk, HD, ph);
    // pressures of the column and of the low neighbours
    double v[OUT_PLANES] = {};
    float lx = 0.0f, ly[OUT_PLANES] = {}, lz[OUT_PLANES] = {};
    const int cell = ((i0 & 7) * 8 + (j & 7)) * 8 + (k & 7);
    if (b >= 0) {
#pragma unroll
        for (int p = 0; p < OUT_PLANES; ++p) v[p] = x[(long)b * BRICK_CELLS + cell + 64 * p];
    }
    if (bi >= 0) lx = (float)x[(long)bi * BRICK_CELLS + ((cell - 64) & 511)];
    const int cj = (cell & ~56) | ((cell - 8) & 56), ck = (cell & ~7) | ((cell - 1) & 7);
    if (bj >= 0) {
#pragma unroll
        for (int p = 0; p < OUT_PLANES; ++p) ly[p] = (float)x[(long)bj * BRICK_CELLS + cj + 64 * p];
    }
    if (bk >= 0) {
#pragma unroll
        for (int p = 0; p < OUT_PLANES; ++p) lz[p] = (float)x[(long)bk * BRICK_CELLS + ck + 64 * p];
    }
    bool air = ph.c[0] >= 0.0;
#pragma unroll
    for (int p = 0; p < OUT_PLANES; ++p) air = air && ph.c[p + 1] >= 0.0 && ph.j[p] >= 0.0 && ph.k[p] >= 0.0;
    const bool quiet = E.liquid && __ballot(!air) == 0;  // every face around is closed
#pragma unroll
    for (int p = 0; p < OUT_PLANES; ++p) {
        if (p >= n) break;
        const size_t c = c0 + (size_t)p * HD;
        if (F.P) F.P[c] = (float)v[p];
        if (F.P64) F.P64[c] = v[p];
        if (F.scene) F.scene[c] = v[p];
        if (F.unknown_out) F.unknown_out[c] = (F.cflag[c] >> 1) & 1;
    }
    const bool last_j = j == G.h - 1, last_k = k == G.d - 1 && !G.flat;
    const size_t f0[3] = {c0, c0 + (size_t)i0 * G.d, c0 + (size_t)((unsigned)i0 * G.h + j)};
    const size_t df[3] = {HD, HD + G.d, HD + G.h};
    // no activity in or out: plain stores
    const bool plain = !(G.active[0] || G.active[1] || G.active[2] || G.active_out[0] || G.active_out[1] || G.active_out[2]);
    if (quiet) {
#pragma unroll
        for (int p = 0; p < OUT_PLANES; ++p) {
            if (p >= n) break;
            if (plain) {
                G.vel[0][f0[0] + p * df[0]] = 0.0f;
                G.vel[1][f0[1] + p * df[1]] = 0.0f;
                if (!G.flat) G.vel[2][f0[2] + p * df[2]] = 0.0f;
            } else {
                put_face(G, 0, f0[0] + p * df[0], 0.0f, false);
                put_face(G, 1, f0[1] + p * df[1], 0.0f, false);
                if (!G.flat) put_face(G, 2, f0[2] + p * df[2], 0.0f, false);
            }
            if (i0 + p == G.w - 1) put_face(G, 0, f0[0] + (p + 1) * HD, 0.0f, false);
            if (last_j) put_face(G, 1, f0[1] + p * df[1] + G.d, 0.0f, false);
            if (last_k) put_face(G, 2, f0[2] + p * df[2] + 1, 0.0f, false);
        }
        return;
    }
    // interior low faces (bit 3 p + dim) that are not shut by the solid; the area only matters where the
    // liquid fraction is nonzero
    unsigned open = 0;
#pragma unroll
    for (int p = 0; p < OUT_PLANES; ++p) {
        const bool dry = E.liquid && ph.c[p + 1] >= 0.0;
        if (p < n) {
            if (i0 + p > 0 && !(dry && ph.c[p] >= 0.0)) open |= 1u << (3 * p);
            if (j > 0 && !(dry && ph.j[p] >= 0.0)) open |= 2u << (3 * p);
            if (k > 0 && !(dry && ph.k[p] >= 0.0)) open |= 4u << (3 * p);
        }
    }
    if (G.solid && __ballot(open != 0)) {
        // signs of the column's nodes at its four corners: a face with no corner in the solid is whole, one
        // with all four has none; only the others' areas are formed
        unsigned s00, s01, s10, s11;
        const size_t stride = G.flat ? (size_t)(G.h + 1) : (size_t)((unsigned)(G.h + 1) * (unsigned)(G.d + 1));
        const size_t n00 = G.flat ? (size_t)((unsigned)i0 * (unsigned)(G.h + 1) + (unsigned)j) : node_index(G, i0, j, k);
        const size_t up = G.flat ? 1 : (size_t)(G.d + 1), right = G.flat ? 0 : 1;
        if (G.solid64) {
            s00 = node_bits<double, OUT_PLANES>(G.solid, n00, n, stride), s01 = node_bits<double, OUT_PLANES>(G.solid, n00 + right, n, stride);
            s10 = node_bits<double, OUT_PLANES>(G.solid, n00 + up, n, stride);
            s11 = node_bits<double, OUT_PLANES>(G.solid, n00 + up + right, n, stride);
        } else {
            s00 = node_bits<float, OUT_PLANES>(G.solid, n00, n, stride), s01 = node_bits<float, OUT_PLANES>(G.solid, n00 + right, n, stride);
            s10 = node_bits<float, OUT_PLANES>(G.solid, n00 + up, n, stride);
            s11 = node_bits<float, OUT_PLANES>(G.solid, n00 + up + right, n, stride);
        }
        unsigned part = 0;
#pragma unroll
        for (int p = 0; p < OUT_PLANES; ++p) {
            auto face = [&](int dim, unsigned any, unsigned all) {
                const unsigned bit = 1u << (3 * p + dim);
                if (all & 1) open &= ~bit;
                else if (any & 1) part |= bit;
            };
            const unsigned a = s00 >> p, b = s01 >> p, c = s10 >> p, d = s11 >> p;
            face(0, a | b | c | d, a & b & c & d);
            face(1, a | b | (a | b) >> 1, a & b & (a & b) >> 1);
            if (!G.flat) face(2, a | c | (a | c) >> 1, a & c & (a & c) >> 1);
        }
        for (unsigned left = open & part; left; left &= left - 1) {
            const int bit = __ffs((int)left) - 1, p = bit / 3;
            if (face_area(G, E, bit - 3 * p, i0 + p, j, k) == 0.0f) open &= ~(1u << bit);
        }
    }
    // the velocities of the open faces, loaded together
    float *const U[3] = {G.vel[0], G.vel[1], G.vel[2]};
    float u[OUT_PLANES][3];
#pragma unroll
    for (int p = 0; p < OUT_PLANES; ++p) {
#pragma unroll
        for (int dim = 0; dim < 3; ++dim) {
            u[p][dim] = 0.0f;
            if (open >> (3 * p + dim) & 1) u[p][dim] = U[dim][f0[dim] + p * df[dim]];
        }
    }
#pragma unroll
    for (int p = 0; p < OUT_PLANES; ++p) {
        const double c = ph.c[p + 1], low[3] = {ph.c[p], ph.j[p], ph.k[p]};
        const float p1 = (float)v[p], p0[3] = {p ? (float)v[p ? p - 1 : 0] : lx, ly[p], lz[p]};
#pragma unroll
        for (int dim = 0; dim < 3; ++dim) {
            if (!(open >> (3 * p + dim) & 1)) continue;
            const double rho = rho_from_samples(G, E, c, low[dim]);
            if (rho != 0.0) {
                const float diff = p1 - p0[dim];
                const float delta = (float)(G.dt * (double)diff / (rho * G.dx));
                u[p][dim] = u[p][dim] - delta;
            } else {
                u[p][dim] = 0.0f;
                open &= ~(1u << (3 * p + dim));
            }
        }
    }
#pragma unroll
    for (int p = 0; p < OUT_PLANES; ++p) {
        if (p >= n) break;
        const int i = i0 + p;
        const bool liquid = ph.c[p + 1] < 0.0;
        const int edge[3] = {i, j, k};
#pragma unroll
        for (int dim = 0; dim < 3; ++dim) {
            if (dim == 2 && G.flat) continue;
            const size_t f = f0[dim] + p * df[dim];
            if (plain) U[dim][f] = u[p][dim];
            else put_face(G, dim, f, u[p][dim], (open >> (3 * p + dim) & 1) || (edge[dim] == 0 && liquid));
        }
        // the domain's high faces
        if (i == G.w - 1) put_face(G, 0, f0[0] + (p + 1) * HD, 0.0f, liquid);
        if (last_j) put_face(G, 1, f0[1] + p * df[1] + G.d, 0.0f, liquid);
        if (last_k) put_face(G, 2, f0[2] + p * df[2] + 1, 0.0f, liquid);
    }
}

}  // namespace shkz
