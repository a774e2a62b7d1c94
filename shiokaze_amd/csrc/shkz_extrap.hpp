// shkz_extrap.hpp -- the step after a projection in Shiokaze's time steppers, on the device:
// velocity extrapolation and the solid constraint, macutility3::extrapolate_and_constrain_velocity
// (src/utility/macutility3.cpp:89-93), which macliquid3::extend_both (macliquid3.cpp:309-319) and
// macsmoke3 (macsmoke3.cpp:294) call on the velocity the projection left.
//
//   k_pack_activity,
//   k_extrap_pass,
//   k_unpack_activity  array_extrapolator3::extrapolate (array_extrapolator3.h:47-80, over
//                   dilate3.h:43-101) on all three face arrays, on bit-packed activity
//   k_constrain,
//   k_constrain_apply  macutility3::constrain_velocity (macutility3.cpp:61-88) with the
//                   interpolation of array_interpolator3.h:40-97, array_derivative3.h:40-103 and
//                   macarray_interpolator3.h:43-50; the first kernel writes constrained values to
//                   a side buffer, the second applies them and the boundary rule, so the velocity
//                   needs no full copy (the reference samples a copy, velocity_save)
//
// Layout: the dense face arrays of the projection (u (w+1,h,d), v (w,h+1,d), w (w,h,d+1), z
// fastest) with one activity byte per face.  One launch covers the three arrays (blockIdx.y
// selects the array).  The extrapolation passes ping-pong two bit-packed copies of the activity
// and write the values of the faces they activate in place (no thread of a pass reads them).
//
// Arithmetic matches the reference's types operation by operation (no contraction): float sums
// of float velocities, interpolation into the array's element type after a double product, vec3d
// normals and dot products, the result rounded to float.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "shkz_device.hpp"
#include "shkz_geometry.hpp"

namespace shkz {

struct VelField {
    int w, h, d;
    int solid64;          // solid level set in double (else float, the reference's Real)
    double dx;
    const void *solid;    // nodal (w+1,h+1,d+1) or nullptr
    float *vel[3];
    uint8_t *act[3];
    size_t n[3];          // faces per array
    // dx a power of two (1/256 for a unit box of 256 cells): x / dx then equals x * inv_dx bit for
    // bit (both round the same exact value once; the inverse is a power of two), and the kernels
    // multiply instead of dividing (an FP64 division is about eleven instructions here)
    int dx_pow2;
    double inv_dx;
    FastDiv by1[3], by2[3];  // by the extents s[1], s[2] of each face array
    FastDiv cell1, cell2;    // by h, d
};
inline void vf_set_divisors(VelField &F) {
    for (int a = 0; a < 3; ++a) {
        F.by1[a] = fast_div((unsigned)(F.h + (a == 1)));
        F.by2[a] = fast_div((unsigned)(F.d + (a == 2)));
    }
    F.cell1 = fast_div((unsigned)F.h);
    F.cell2 = fast_div((unsigned)F.d);
}

// x / F.dx, exactly as the division rounds.
__device__ __forceinline__ double vf_div_dx(const VelField &F, double x) { return F.dx_pow2 ? x * F.inv_dx : x / F.dx; }

__device__ __forceinline__ void vf_shape(const VelField &F, int a, int s[3]) {
    s[0] = F.w + (a == 0);
    s[1] = F.h + (a == 1);
    s[2] = F.d + (a == 2);
}

// Face kernels launch a (ceil(max n / 256), 3) grid: blockIdx.y is the face array, so the array
// index is uniform across a wavefront and every per-array field (extent, pointers) is a scalar
// load.  (A flat index over the three arrays made it vary inside the wavefront that straddles two
// arrays, and hipcc then lowered a dynamically indexed kernel-argument read with v_readfirstlane,
// as if it were uniform: that wavefront's lanes read the first lane's array extent.)
// Threads per block of every face, cell and activity-word kernel here.  The kernels index with
// this constant, not blockDim.x: the workgroup size is a 16-bit field of the hidden kernel
// arguments, which hipcc reads with a vector load, one more memory round trip before a wave can
// form its index.
constexpr int VF_BLOCK = 256;
// A wavefront takes G groups of 64 consecutive faces, all of their activity bytes loaded at once.  Most
// groups of a domain are inactive, and with one group per wavefront the launch is bound by how many wavefronts
// are resident over the round trip of one byte load (256^3, 50 million faces: k_constrain 223 us against 157,
// k_constrain_apply 67 against 33, k_adv_face_bwd 273 against 237).  G = 8 where the launch keeps VF_MANY wavefronts
// all the same (twice what the chip holds); a smaller field takes one group per wavefront, all of them resident
// at once.  The step's three calls with eight groups / by the rule / with one (us): 96^3 279 / 249 / 251, 128^3
// 376 / 352 / 350, 140^3 434 / 425 / 426, 160^3 541 / 536 / 546, 200^3 866 / 869 / 905.
constexpr int VF_GROUPS = 8;
constexpr size_t VF_MANY = 16384;
inline bool vf_many(const size_t n[3]) { return (n[0] + n[1] + n[2]) / (64 * VF_GROUPS) >= VF_MANY; }
inline dim3 vf_grid(const size_t n[3], int groups = 1) {
    const size_t m = n[0] > n[1] ? (n[0] > n[2] ? n[0] : n[2]) : (n[1] > n[2] ? n[1] : n[2]);
    const size_t per = (size_t)VF_BLOCK * groups;
    return dim3((unsigned)(((m + per - 1) / per + 7) / 8 * 8), 3);
}

// This thread's faces f0 + 64 g (g < G) of array a and their activity codes, 8 bits each (0 past the end).
template <int G>
struct VfFaces {
    int a;
    size_t f0;
    unsigned long long codes;
    __device__ __forceinline__ size_t face(int g) const { return f0 + 64 * (size_t)g; }
    __device__ __forceinline__ int code(int g) const { return (int)(codes >> (8 * g)) & 255; }
};
template <int G>
__device__ __forceinline__ VfFaces<G> vf_faces(const VelField &F) {
    static_assert(G <= 8, "a byte each");
    VfFaces<G> V;
    V.a = (int)blockIdx.y;
    const unsigned block = (unsigned)xcd_brick(blockIdx.x, gridDim.x);  // XCD-contiguous slabs
    V.f0 = ((size_t)block * (VF_BLOCK / 64) + (threadIdx.x >> 6)) * (64 * G) + (threadIdx.x & 63);
    uint8_t t[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const size_t f = V.f0 + 64 * (size_t)g;
        t[g] = F.act[V.a][f < F.n[V.a] ? f : F.n[V.a] - 1];
        if (f >= F.n[V.a]) t[g] = 0;
    }
    V.codes = 0;
#pragma unroll
    for (int g = 0; g < G; ++g) V.codes |= (unsigned long long)t[g] << (8 * g);
    return V;
}
// 32-bit decode (each face array holds fewer than 2^32 faces, checked at entry)
__device__ __forceinline__ void vf_decode(const VelField &F, int a, size_t f, int &i, int &j, int &k) {
    int s[3];
    vf_shape(F, a, s);
    const unsigned u = (unsigned)f, t = divide(u, F.by2[a]), ii = divide(t, F.by1[a]);
    k = (int)(u - t * (unsigned)s[2]);
    j = (int)(t - ii * (unsigned)s[1]);
    i = (int)ii;
}

// The extrapolation works on bit-packed activity: each row (i, j) of a face array is a run of
// 32-bit words along k, bit b of word kw = face k = 32 kw + b.  A pass is then one thread per word:
// it forms the six neighbour masks from the word, its two neighbours along k and the words of the
// rows +-1 in j and i, and activates the inactive faces with an active neighbour.
struct BitField {
    uint32_t *bits[3];
    int W[3];  // words per row
    FastDiv by[3];
};

__device__ __forceinline__ int vf_rows(const VelField &F, int a) { return (F.w + (a == 0)) * (F.h + (a == 1)); }

// activity bytes -> bits, a word per thread: its 32 bytes (consecutive along the row, at any alignment) in two
// loads, each byte reduced to one bit.  With a lane per face and a ballot per two words, most of the time went
// into index arithmetic (256^3: 64 us, 13 us here).
__device__ __forceinline__ uint32_t nonzero_bytes(uint32_t x) {
    const uint32_t y = ((((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x) >> 7) & 0x01010101u;
    return (y | y >> 7 | y >> 14 | y >> 21) & 15u;
}
__global__ __launch_bounds__(VF_BLOCK) void k_pack_activity(VelField F, BitField B) {
    const int a = (int)blockIdx.y;
    int s[3];
    vf_shape(F, a, s);
    const int W = B.W[a];
    const size_t w = (size_t)blockIdx.x * VF_BLOCK + threadIdx.x;
    if (w >= (size_t)vf_rows(F, a) * W) return;
    const unsigned r = divide((unsigned)w, B.by[a]), kw = (unsigned)w - r * (unsigned)W;  // 32-bit: fewer than 2^32 words
    const size_t f0 = (size_t)r * s[2] + (size_t)kw * 32;
    const int nbits = min(32, s[2] - (int)kw * 32);
    const uint8_t *act = F.act[a] + f0;
    uint32_t m = 0;
    if (f0 + 32 <= F.n[a]) {
        // (beyond the row's end these are the next row's bytes, masked out below)
        uint32_t x[8];
        __builtin_memcpy(x, act, 32);
#pragma unroll
        for (int q = 0; q < 8; ++q) m |= nonzero_bytes(x[q]) << (4 * q);
        if (nbits < 32) m &= (1u << nbits) - 1u;
    } else {
        for (int b = 0; b < nbits; ++b) m |= (act[b] ? 1u : 0u) << b;
    }
    B.bits[a][w] = m;
}

// One extrapolation pass: Bo = Bi plus every inactive face with an in-bounds neighbour active in
// Bi, which takes the mean of those neighbours, summed in float in the order +x, -x, +y, -y, -z,
// +z (array_extrapolator3.h:57-72).  The faces a pass activates are inactive in Bi, so no thread
// of the pass reads their values (but its own face's, where a neighbour is missing, to no effect).
//
// One thread per word forms the masks; a wavefront then lists the faces of its 64 words in LDS
// and takes them 64 at a time, six loads in flight for each.  With each thread walking the faces of its own
// word, up to 32 in a row, a pass took 15.0 us at 61x90x77 and 31.6 us at 256^3, here 5.7 and 24.
struct ExtrapWave {
    uint32_t ip[64], im[64], jp[64], jm[64], km[64], kp[64], f0[64];
    uint16_t list[64 * 32];
};
__global__ __launch_bounds__(VF_BLOCK) void k_extrap_pass(VelField F, BitField Bi, BitField Bo) {
#pragma clang fp contract(off)
    __shared__ ExtrapWave waves[VF_BLOCK / 64];
    ExtrapWave &V = waves[threadIdx.x >> 6];
    const int lane = threadIdx.x & 63;
    const int a = (int)blockIdx.y;
    int s[3];
    vf_shape(F, a, s);
    const int W = Bi.W[a];
    const size_t w = (size_t)blockIdx.x * VF_BLOCK + threadIdx.x;
    const size_t nw = (size_t)vf_rows(F, a) * W;
    uint32_t cand = 0;
    if (w < nw) {
        const unsigned r = divide((unsigned)w, Bi.by[a]), kw = (unsigned)w - r * (unsigned)W;  // 32-bit: fewer than 2^32 words
        const int i = (int)divide(r, F.by1[a]), j = (int)(r - (unsigned)i * s[1]);
        const uint32_t *B = Bi.bits[a];
        const uint32_t A = B[w];
        const uint32_t nxt = kw + 1 < (unsigned)W ? B[w + 1] : 0u, prv = kw > 0 ? B[w - 1] : 0u;
        const uint32_t kp = (A >> 1) | (nxt << 31);  // bit b: face k+1 active
        const uint32_t km = (A << 1) | (prv >> 31);  // bit b: face k-1 active
        const uint32_t jp = j + 1 < s[1] ? B[w + W] : 0u, jm = j > 0 ? B[w - W] : 0u;
        const size_t sxw = (size_t)s[1] * W;
        const uint32_t ip = i + 1 < s[0] ? B[w + sxw] : 0u, im = i > 0 ? B[w - sxw] : 0u;
        const int nbits = s[2] - (int)kw * 32;
        const uint32_t valid = nbits >= 32 ? 0xffffffffu : ((1u << nbits) - 1u);
        cand = (kp | km | jp | jm | ip | im) & ~A & valid;
        Bo.bits[a][w] = A | cand;
        if (cand) {
            V.ip[lane] = ip;
            V.im[lane] = im;
            V.jp[lane] = jp;
            V.jm[lane] = jm;
            V.km[lane] = km;
            V.kp[lane] = kp;
            V.f0[lane] = r * (unsigned)s[2] + kw * 32;
        }
    }
    // places in the list: a prefix sum of the words' counts over the wavefront
    const int mine = __popc(cand);
    int upto = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(upto, o, 64);
        if (lane >= o) upto += v;
    }
    const int total = __shfl(upto, 63, 64);
    int at = upto - mine;
    for (; cand; cand &= cand - 1) V.list[at++] = (uint16_t)(lane << 5 | __builtin_ctz(cand));
    __syncthreads();
    float *U = F.vel[a];
    const unsigned sx = (unsigned)s[1] * (unsigned)s[2], sy = (unsigned)s[2];
    for (int t = lane; t < total; t += 64) {
        const int e = V.list[t], l = e >> 5, b = e & 31;
        const unsigned f = V.f0[l] + (unsigned)b;
        // an absent neighbour's place is the face itself: six loads without a branch
        const bool on[6] = {((V.ip[l] >> b) & 1u) != 0, ((V.im[l] >> b) & 1u) != 0, ((V.jp[l] >> b) & 1u) != 0,
                            ((V.jm[l] >> b) & 1u) != 0, ((V.km[l] >> b) & 1u) != 0, ((V.kp[l] >> b) & 1u) != 0};
        const unsigned at6[6] = {f + sx, f - sx, f + sy, f - sy, f - 1, f + 1};
        float u[6];
#pragma unroll
        for (int n = 0; n < 6; ++n) u[n] = U[on[n] ? at6[n] : f];
        float sum = 0.0f;
        int weight = 0;
#pragma unroll
        for (int n = 0; n < 6; ++n) {
            sum = on[n] ? sum + u[n] : sum;
            weight += on[n];
        }
        // float / int in the reference; the double quotient rounded once to float is the
        // correctly rounded float quotient
        U[f] = (float)((double)sum / (double)weight);
    }
}

// bits -> activity bytes for the faces the passes activated (final & ~initial)
__global__ void k_unpack_activity(VelField F, BitField B0, BitField Bf) {
    const int a = (int)blockIdx.y;
    int s[3];
    vf_shape(F, a, s);
    const int W = Bf.W[a];
    const size_t w = (size_t)blockIdx.x * VF_BLOCK + threadIdx.x;
    if (w >= (size_t)vf_rows(F, a) * W) return;
    uint32_t fresh = Bf.bits[a][w] & ~B0.bits[a][w];
    if (!fresh) return;
    const unsigned r = divide((unsigned)w, Bf.by[a]), kw = (unsigned)w - r * (unsigned)W;  // 32-bit: fewer than 2^32 words
    const size_t f0 = (size_t)r * s[2] + (size_t)kw * 32;
    while (fresh) {
        const int b = __builtin_ctz(fresh);
        fresh &= fresh - 1;
        F.act[a][f0 + b] = 1;
    }
}

__device__ __forceinline__ double dmin_(double a, double b) { return b < a ? b : a; }  // std::min
__device__ __forceinline__ double dmax_(double a, double b) { return a < b ? b : a; }  // std::max

// Corner base index and clamped position of array_interpolator3::interpolate_coef (:40-62).
struct Corner {
    int i, j, k;
    double x, y, z;
};
__device__ __forceinline__ Corner corner_of(const int s[3], const double p[3]) {
#pragma clang fp contract(off)
    Corner c;
    c.x = dmax_(0.0, dmin_(s[0] - 1., p[0]));
    c.y = dmax_(0.0, dmin_(s[1] - 1., p[1]));
    c.z = dmax_(0.0, dmin_(s[2] - 1., p[2]));
    c.i = (int)dmin_(c.x, s[0] - 2.);
    c.j = (int)dmin_(c.y, s[1] - 2.);
    c.k = (int)dmin_(c.z, s[2] - 2.);
    return c;
}

// Trilinear weights in corner order (i,j,k), (i+1,j,k), (i,j+1,k), (i+1,j+1,k), then k+1.
__device__ __forceinline__ void interp_weights(const Corner &c, double w[8]) {
#pragma clang fp contract(off)
    const double zk1 = (c.k + 1) - c.z, zk = c.z - c.k, xi1 = (c.i + 1) - c.x, xi = c.x - c.i, yj1 = (c.j + 1) - c.y,
                 yj = c.y - c.j;
    w[0] = zk1 * xi1 * yj1;
    w[1] = zk1 * xi * yj1;
    w[2] = zk1 * xi1 * yj;
    w[3] = zk1 * xi * yj;
    w[4] = zk * xi1 * yj1;
    w[5] = zk * xi * yj1;
    w[6] = zk * xi1 * yj;
    w[7] = zk * xi * yj;
}

// Derivative weights of array_derivative3::derivative_interpolate_coef (:40-85), dw[8*dim+n].
__device__ __forceinline__ void deriv_weights(const Corner &c, double dw[24]) {
#pragma clang fp contract(off)
    const double zk1 = (c.k + 1) - c.z, zk = c.z - c.k, xi1 = (c.i + 1) - c.x, xi = c.x - c.i, yj1 = (c.j + 1) - c.y,
                 yj = c.y - c.j;
    dw[0] = -zk1 * yj1;
    dw[1] = zk1 * yj1;
    dw[2] = -zk1 * yj;
    dw[3] = zk1 * yj;
    dw[4] = -zk * yj1;
    dw[5] = zk * yj1;
    dw[6] = -zk * yj;
    dw[7] = zk * yj;
    dw[8] = -zk1 * xi1;
    dw[9] = -zk1 * xi;
    dw[10] = zk1 * xi1;
    dw[11] = zk1 * xi;
    dw[12] = -zk * xi1;
    dw[13] = -zk * xi;
    dw[14] = zk * xi1;
    dw[15] = zk * xi;
    dw[16] = -xi1 * yj1;
    dw[17] = -xi * yj1;
    dw[18] = -xi1 * yj;
    dw[19] = -xi * yj;
    dw[20] = xi1 * yj1;
    dw[21] = xi * yj1;
    dw[22] = xi1 * yj;
    dw[23] = xi * yj;
}

// Flat indices of the eight corners of c in an array of shape s.  32-bit arithmetic: the entry points that
// sample face, cell and node arrays reject grids with (w+1)(h+1)(d+1) >= 2^32.
__device__ __forceinline__ void corner_indices(const Corner &c, const int s[3], unsigned q[8]) {
    const unsigned sy = (unsigned)s[2], sx = (unsigned)s[1] * sy;
    const unsigned base = ((unsigned)c.i * (unsigned)s[1] + (unsigned)c.j) * sy + (unsigned)c.k;
#pragma unroll
    for (int n = 0; n < 8; ++n) q[n] = base + ((n & 1) ? sx : 0u) + ((n & 2) ? sy : 0u) + ((n & 4) ? 1u : 0u);
}

// Accumulation in the array's element type T after a double product (value += array(idx)*coef).
template <class T>
__device__ __forceinline__ T acc(T v, double term) {
#pragma clang fp contract(off)
    return (T)((double)v + term);
}

// The solid sample and its derivative at the centre p of a face (nodal array), in the level set's type T: der and
// true where the point is inside (negative).  The centre's corner (corner_of) is the face's own (i, j, k),
// the last but one node where that lies past it, so the corners are loaded and tested without FP64.
template <class T>
__device__ __forceinline__ bool inside_solid(const VelField &F, int i, int j, int k, const double p[3], double der[3]) {
#pragma clang fp contract(off)
    const int s[3] = {F.w + 1, F.h + 1, F.d + 1};
    Corner c;
    c.i = i < F.w - 1 ? i : F.w - 1;
    c.j = j < F.h - 1 ? j : F.h - 1;
    c.k = k < F.d - 1 ? k : F.d - 1;
    const T *S = (const T *)F.solid;
    T v[8];
    unsigned q[8];
    corner_indices(c, s, q);
#pragma unroll
    for (int n = 0; n < 8; ++n) v[n] = S[q[n]];
    // with no negative corner the interpolation is a sum of non-negative products (a NaN corner
    // makes it NaN): never below 0 whatever the rounding, so the point is outside and the weights
    // are not needed (most faces lie away from the solid)
    bool any_neg = false;
#pragma unroll
    for (int n = 0; n < 8; ++n) any_neg = any_neg || v[n] < T(0);
    if (!any_neg) return false;
    c = corner_of(s, p);
    double w[8];
    interp_weights(c, w);
    T val = T(0);
#pragma unroll
    for (int n = 0; n < 8; ++n)
        if (w[n] != 0.0) val = acc<T>(val, (double)v[n] * w[n]);
    if (!((double)val < 0.0)) return false;
    double dw[24];
    deriv_weights(c, dw);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        T r = T(0);
#pragma unroll
        for (int n = 0; n < 8; ++n) r = acc<T>(r, dw[8 * a + n] * (double)v[n]);
        der[a] = (double)r;
    }
    return true;
}

// Component b of the saved velocity at p (macarray_interpolator3.h:43-50): inactive faces read 0.
__device__ __forceinline__ double vel_sample(const VelField &F, const float *const Sv[3], int b, const double p[3]) {
#pragma clang fp contract(off)
    int s[3];
    vf_shape(F, b, s);
    const double pos[3] = {p[0] - 0.5 * (b != 0), p[1] - 0.5 * (b != 1), p[2] - 0.5 * (b != 2)};
    const Corner c = corner_of(s, pos);
    double w[8];
    interp_weights(c, w);
    // all eight corners are loaded at once (they lie in the array: the constraint asks for at
    // least 2 cells per axis); zero weights still skip the accumulation
    float u[8];
    unsigned q[8];
    corner_indices(c, s, q);
#pragma unroll
    for (int n = 0; n < 8; ++n) {
        const float sv = Sv[b][q[n]];
        u[n] = F.act[b][q[n]] ? sv : 0.0f;
    }
    float val = 0.0f;
#pragma unroll
    for (int n = 0; n < 8; ++n)
        if (w[n] != 0.0) val = acc<float>(val, (double)u[n] * w[n]);
    return (double)val;
}

// Activity code of a face whose constrained value waits in the side buffer (k_constrain_apply).
constexpr uint8_t ACT_CONSTRAINED = 255;

// macutility3::constrain_velocity, first half.  For every active face: the activity codes of the
// passes become 1; when `constrain` is set and the solid level set has a negative value (*exist),
// a face whose centre samples the solid below 0 and whose velocity points into the solid gets
// the velocity minus its normal component, written to X (not to the velocity, which neighbouring
// threads still sample, as the reference samples its velocity_save copy) and marked
// ACT_CONSTRAINED.  The velocity arrays are only read here.
//
// Bound by issue: most of the faces are inactive and most of the others away from the solid, so the decode
// divides by multiplying and the corner test needs no FP64 (256^3: 223 us before, 157 us).  The corners that the
// test loads serve the interpolation too: with loads of its own for each, 130x140x150 faces near a solid everywhere
// (random nodes) took 207 us a call, 179 here.
__device__ __forceinline__ void constrain_face(const VelField &F, int a, size_t f, int t, float *X0, float *X1, float *X2,
                                               bool with_solid) {
#pragma clang fp contract(off)
    int i, j, k;
    vf_decode(F, a, f, i, j, k);
    if (with_solid) {
        const float *const Sv[3] = {F.vel[0], F.vel[1], F.vel[2]};
        const double p[3] = {i + 0.5 * (a != 0), j + 0.5 * (a != 1), k + 0.5 * (a != 2)};
        double der[3] = {0.0, 0.0, 0.0};
        if (F.solid64 ? inside_solid<double>(F, i, j, k, p, der) : inside_solid<float>(F, i, j, k, p, der)) {
            double nrm[3];
#pragma unroll
            for (int b = 0; b < 3; ++b) nrm[b] = vf_div_dx(F, der[b]);
            double n2 = 0.0;
#pragma unroll
            for (int b = 0; b < 3; ++b) n2 += nrm[b] * nrm[b];
            if (n2 != 0.0) {
                double u[3];
#pragma unroll
                for (int b = 0; b < 3; ++b) u[b] = vel_sample(F, Sv, b, p);
                double un = 0.0;
#pragma unroll
                for (int b = 0; b < 3; ++b) un += u[b] * nrm[b];
                if (un < 0.0) {
                    float *const X[3] = {X0, X1, X2};
                    X[a][f] = (float)(u[a] - nrm[a] * un);
                    F.act[a][f] = ACT_CONSTRAINED;  // nonzero: neighbours still read the face as active
                    return;
                }
            }
        }
    }
    if (t > 1) F.act[a][f] = 1;
}
template <int G>
__global__ void k_constrain(VelField F, float *X0, float *X1, float *X2, const int *exist, int constrain) {
#pragma clang fp contract(off)
    const VfFaces<G> V = vf_faces<G>(F);
    const bool with_solid = constrain && F.solid && *exist;  // loaded with the activity bytes
    if (!V.codes) return;
#pragma unroll 1
    for (int g = 0; g < G; ++g)
        if (V.code(g)) constrain_face(F, V.a, V.face(g), V.code(g), X0, X1, X2, with_solid);
}

// Second half: constrained faces take their value from X, then (with the constraint on and a
// solid present) active faces on the domain boundary pointing out of the domain become 0.
template <int G>
__global__ void k_constrain_apply(VelField F, const float *X0, const float *X1, const float *X2, const int *exist,
                                  int constrain) {
    const VfFaces<G> V = vf_faces<G>(F);
    const bool with_solid = constrain && F.solid && *exist;  // loaded with the activity bytes
    if (!V.codes || !with_solid) return;
    const int a = V.a;
#pragma unroll 1
    for (int g = 0; g < G; ++g) {
        const int t = V.code(g);
        const size_t f = V.face(g);
        if (!t) continue;
        int i, j, k;
        vf_decode(F, a, f, i, j, k);
        const int at = a == 0 ? i : a == 1 ? j : k, end = a == 0 ? F.w : a == 1 ? F.h : F.d;
        if (t != ACT_CONSTRAINED && at != 0 && at != end) continue;
        float out = t == ACT_CONSTRAINED ? (a == 0 ? X0 : a == 1 ? X1 : X2)[f] : F.vel[a][f];
        if (at == 0 && out < 0.0f) out = 0.0f;
        if (at == end && out > 0.0f) out = 0.0f;
        F.vel[a][f] = out;
        if (t == ACT_CONSTRAINED) F.act[a][f] = 1;
    }
}

}  // namespace shkz
