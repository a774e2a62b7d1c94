// shkz_device.hpp -- device-side data structures shared by the kernels and the host runtime.
//
// Storage model.  Every grid (and every multigrid level of it) is cut into 8x8x8 bricks.  Only
// bricks that hold at least one unknown are stored, brick-major, 512 cells each, with the cell
// order (li*8 + lj)*8 + lk (z fastest).  A dense brick map (one int per brick position) gives
// the compact id of a stored brick or -1.  Vectors are zero on every stored cell that is not an
// unknown, so the operator needs no separate mask: dir < 0 marks a non-unknown.
//
// The operator of one level is four arrays over the stored cells:
//   dir      sum of the conductances of the open faces towards non-unknown (air) neighbours,
//            -1 on a stored cell that is not an unknown,
//   gx,gy,gz conductance of the cell's low x/y/z face when both cells are unknowns, else 0,
// so that diag_c = dir_c + the six couplings and (A p)_c = diag_c p_c - sum_f g_f p_q with
// p = 0 off the unknowns.  On the
// finest level the conductance is dt*area/(dx*dx*rho), the reference's matrix entry
// (src/projection/macpressuresolver3.cpp:185).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace shkz {

constexpr int BRICK = 8;
constexpr int BRICK_CELLS = 512;
constexpr int BLOCK = 512;  // brick kernels: one thread per cell
constexpr int MAX_LEVELS = 32;  // a grid side of 8 * 2^31 cells would need more

// Neighbour slots of a brick in its neighbour table.
enum { NB_XM = 0, NB_XP = 1, NB_YM = 2, NB_YP = 3, NB_ZM = 4, NB_ZP = 5 };

// Per grid and level: the grid's cell and brick extents, where its dense brick map starts in the
// level's combined map, and its range of stored bricks in the level's combined brick list.
struct GridLevel {
    int ni, nj, nk;     // cells
    int nbx, nby, nbz;  // bricks per axis
    int bmap_off;       // offset of this grid's dense brick map
    int brick_start;    // first stored brick of this grid
    int brick_end;      // one past the last
    int coarsest;       // 1: the grid fits one brick here, so this is its last level (coarse solve)
    int pad[2];
};

// Per stored brick: its six neighbour bricks (NB_*, -1 = none), its grid and flags, in one
// 32-byte record (one scalar load per workgroup).
enum {
    BM_COARSEST = 1,  // the brick's grid ends on this level (its coarse solve handles it)
    BM_UNIFORM = 2,   // level 0: the operator is one constant on the brick (UniCoef)
    BM_BOTTOM = 4,    // a level of the grid's bottom (BottomGrid): k_bottom works on it
    BM_BELOW = 8,     // ... and not the bottom's first level, whose right-hand side the restriction forms
    BM_LOOSE = 16     // a cell across one of its faces may be coupled to it and yet be no unknown (COUPLED_OUT)
};
// A NaN in the level set leaves the liquid cells beside it with a NaN for their diagonal, so that no kernel takes them
// as unknowns (dir >= 0), but with their couplings.  A coarse cell over such cells and no unknown has this dir instead of -1.
constexpr int COUPLED_OUT = -2;
struct __align__(32) BrickMeta {
    int nbr[6];
    int grid;
    int flags;
};

// A level-0 brick on which every cell is an unknown without a Dirichlet term and every face of
// every cell (the high faces of its last layers included) has the same conductance g -- the
// interior of the liquid away from surfaces and solids, most of the domain.  The smoothing and
// operator kernels take g and the inverse diagonal from this record instead of streaming the
// four operator arrays and idiag: the same values, so the same results, with 5 fewer arrays read.
struct __align__(32) UniCoef {
    double g64, id64;  // FP64 conductance and inverse diagonal (FP64 smoothers)
    float g32, id32;   // the FP32 copies of the mixed-precision V-cycle
    float pad[2];
};

template <class T>
struct UniT {
    T g, id;
};
__device__ __forceinline__ void uni_pick(const UniCoef &u, UniT<double> &o) {
    o.g = u.g64;
    o.id = u.id64;
}
__device__ __forceinline__ void uni_pick(const UniCoef &u, UniT<float> &o) {
    o.g = u.g32;
    o.id = u.id32;
}

// One multigrid level of a batch of grids: the stored bricks of every grid, concatenated
// (grid-major, Morton order inside a grid).  A single grid is a batch of one.
struct LevelDesc {
    int nbricks;             // stored bricks, all grids
    int ngrids;
    int flat;                // 2D grids (one cell layer): bilinear transfers
    int pad;
    const int *bmap;         // per grid g: bmap[gl[g].bmap_off + (bx*nby + by)*nbz + bz] -> brick or -1
    const int *bxyz;         // brick -> bx, by, bz (in its grid)
    const BrickMeta *meta;   // brick -> neighbours, grid, flags
    const GridLevel *gl;
    const int *child64;      // brick -> the 4x4x4 finer-level bricks 2B-1 .. 2B+2 per axis (-1 = none)
    const int *parent8;      // brick -> the 2x2x2 coarser-level bricks (B+1)/2 - 1 + {0,1} per axis
    const UniCoef *uni;      // level 0: constants of the BM_UNIFORM bricks (nullptr elsewhere)
    const int *nb27;         // coarse levels: brick -> the 3x3x3 bricks B-1 .. B+1 per axis (-1 = none)
};

template <class T>
__device__ __forceinline__ UniT<T> uni_load(const LevelDesc &L, int br) {
    UniT<T> o;
    uni_pick(L.uni[br], o);
    return o;
}

template <class T>
struct OpDesc {
    const T *dir;  // sum of conductances to non-unknown neighbours; -1 marks a non-unknown
    const T *gx;
    const T *gy;
    const T *gz;
};

// Scalars of one grid's Krylov solve, resident on the device so that no iteration waits on the
// host.
struct SolveScalars {
    double rz[2];     // r.z of the current iteration: [0], or, where the kernels that use r.z form it
                      // themselves (fold_partials), alternately [0] and [1]
    double pq;        // p.Ap
    double alpha, beta;
    double rinf;      // ||r||_inf after the last update
    double rl2;       // ||r||_2 after the last update
    double r0inf;     // ||r0||_inf
    double r0l2;
    double tol;       // absolute tolerance in the chosen norm
    double rmin;      // smallest residual norm reached (stagnation test)
    int32_t iter;     // iterations done
    int32_t maxit;
    int32_t done;     // 1 = stop (converged or out of iterations)
    int32_t converged;
    int32_t norm;     // shkz_norm
    int32_t status;   // 0 ok, 1 = NaN met
    int32_t stall;        // iterations since the residual last reached a new minimum
    int32_t stall_limit;  // > 0: stop after that many (inner solves of the defect correction)
};

// Batch-wide state of one Krylov solve: how many grids are done; every kernel returns at once when
// all are.
struct BatchCtl {
    int32_t ngrids;
    int32_t ndone;
    int32_t all_done;
    int32_t pad;
};

// What a V-cycle launch may skip: everything once all grids are done, and the bricks of a grid
// that is done.  S may be NULL (no per-grid test).
// skip: the brick flags (BM_*) whose bricks the smoothing kernels leave to another kernel.
struct Gate {
    const BatchCtl *ctl;
    const SolveScalars *S;
    int skip;
};

// The bottom of one grid's hierarchy: its last levels, each of at most BOTTOM_BRICKS stored bricks,
// down to the single brick of the coarsest one.  One workgroup runs that whole part of the V-cycle
// (k_bottom), whose arrays and tables these records name.
constexpr int BOTTOM_BRICKS = 8;
constexpr int BOTTOM_LEVELS = 4;
struct BottomLevel {
    const float *dir, *gx, *gy, *gz, *idiag;  // from the grid's first brick of the level on
    float *rhs, *z, *tmp;
    const BrickMeta *meta;
    const int *bxyz, *child64, *parent8;
    int brick_start, nb;
    int deepest;  // the batch's last level (its result is always in z)
    int flat;
};
struct BottomGrid {
    int n;  // levels (0: the grid has no level below the finest)
    int pad[3];
    const int16_t *code;  // component codes of the coarsest brick (k_coarse_components)
    BottomLevel lev[BOTTOM_LEVELS];
};

// Deterministic two-pass reduction: every brick of a reducing kernel stores two partials (plain
// stores, no atomics); a finalize kernel with one block per grid combines the partials of that
// grid's bricks in brick order and updates the grid's scalars.
struct RedBuf {
    double *partials;  // 2 per brick
};

// Remaps a linear block id so that each of the 8 XCDs (which receive blocks round-robin) gets a
// contiguous range of bricks: neighbouring bricks then share that XCD's L2.
__device__ __forceinline__ int xcd_brick(int block, int nblocks) {
    const int per = (nblocks + 7) >> 3;
    return (block & 7) * per + (block >> 3);
}

// Sum / max over a wavefront: the xor butterfly 32, 16, 8, 4, 2, 1, so every lane ends with the same
// bits.  The exchanges are register moves (gfx950's half and row swaps, DPP) instead of a shuffle
// through LDS, about 130 cycles for each of twelve 32-bit halves: most of what a small reducing
// kernel takes.  After the steps 32, 16 and 8 a value depends on its lane modulo 8 only, so that a
// rotation by 4 within 16 lanes is the exchange with lane ^ 4.
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)u, CTRL, 0xF, 0xF, true);
    const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), CTRL, 0xF, 0xF, true);
    return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
}
// v of this lane's half (HALF) or even/odd row pair and of the other one, in a fixed order.
template <bool HALF>
__device__ __forceinline__ double2 swap_pair(double v) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)u, hi = (unsigned)(u >> 32);
    const auto l = HALF ? __builtin_amdgcn_permlane32_swap(lo, lo, false, false)
                        : __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
    const auto h = HALF ? __builtin_amdgcn_permlane32_swap(hi, hi, false, false)
                        : __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    return make_double2(__builtin_bit_cast(double, (unsigned long long)h[0] << 32 | l[0]),
                        __builtin_bit_cast(double, (unsigned long long)h[1] << 32 | l[1]));
}
constexpr int DPP_ROR8 = 0x128, DPP_ROR4 = 0x124, DPP_QUAD_2301 = 0x4E, DPP_QUAD_1032 = 0xB1;
__device__ __forceinline__ double wave_sum(double v) {
    const double2 a = swap_pair<true>(v);
    v = a.x + a.y;
    const double2 b = swap_pair<false>(v);
    v = b.x + b.y;
    v += dpp_move<DPP_ROR8>(v);
    v += dpp_move<DPP_ROR4>(v);
    v += dpp_move<DPP_QUAD_2301>(v);
    v += dpp_move<DPP_QUAD_1032>(v);
    return v;
}
__device__ __forceinline__ double wave_max(double v) {
    const double2 a = swap_pair<true>(v);
    v = fmax(a.x, a.y);
    const double2 b = swap_pair<false>(v);
    v = fmax(b.x, b.y);
    v = fmax(v, dpp_move<DPP_ROR8>(v));
    v = fmax(v, dpp_move<DPP_ROR4>(v));
    v = fmax(v, dpp_move<DPP_QUAD_2301>(v));
    v = fmax(v, dpp_move<DPP_QUAD_1032>(v));
    return v;
}

// Block-wide sum of one value per thread (BLOCK threads).  Result valid in every thread.
__device__ __forceinline__ double block_sum(double v, double *lds) {
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) lds[wid] = v;
    __syncthreads();
    double s = 0.0;
    const int nw = blockDim.x >> 6;
    for (int i = 0; i < nw; ++i) s += lds[i];
    return s;
}

// Two block-wide reductions in one LDS round: a by max (AMAX) or sum, b by sum.  The sum's
// operations and their order are block_sum's.  lds holds 32 doubles.
template <bool AMAX>
__device__ __forceinline__ void block_reduce2(double &a, double &b, double *lds) {
    a = AMAX ? wave_max(a) : wave_sum(a);
    b = wave_sum(b);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) {
        lds[wid] = a;
        lds[16 + wid] = b;
    }
    __syncthreads();
    double sa = 0.0, sb = 0.0;
    const int nw = blockDim.x >> 6;
    for (int i = 0; i < nw; ++i) {
        sa = AMAX ? fmax(sa, lds[i]) : sa + lds[i];
        sb += lds[16 + i];
    }
    a = sa;
    b = sb;
}

__device__ __forceinline__ void store_partials(const RedBuf &R, int brick, double a, double b) {
    if (threadIdx.x == 0) {
        R.partials[2 * brick + 0] = a;
        R.partials[2 * brick + 1] = b;
    }
}

}  // namespace shkz
