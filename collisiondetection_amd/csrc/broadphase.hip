// Broadphase: the candidate stencil sets of KDOPBroadPhase::findCollisionCandidates
// (src/KDOPBroadPhase.cpp:34-185), built MI355X-first.
//
// The reference builds a top-down median-split tree of 13-axis swept k-DOPs and traverses it against
// itself.  Its output does not depend on the tree's shape (interior bounds are exact unions of child
// bounds, KDOPBroadPhase.cpp:85-98, so a leaf pair is visited iff its two leaf bounds overlap), so this
// file sorts the leaves along a Morton curve and searches 64-wide levels of boxes over that order:
//   1. leaf bounds: per face, 13 axes x (3 vertices x history entries), min/max of pos.axis -/+ eta in
//      FP64 exactly as KDOPBroadPhase.cpp:60-70 (bit-identical);
//   2. Morton codes of the leaf centres, radix-sorted (devprims.hip);
//   3. box records quantised to 16 bits per bound: one per leaf, one per 64 leaves (a cluster), one per
//      64 clusters, and so on: the width of a wavefront;
//   4. the pair search: one wavefront per cluster finds the clusters its box meets, 64 box tests at a
//      time, and tests each as a 64 x 64 tile of leaves.  The quantised test culls; the leaf-leaf
//      decision is the reference's FP64 13-axis test (touching overlaps) and the shared-vertex test
//      (Mesh.cpp:13-20), run on full wavefronts from a queue in LDS;
//      Its finds become one row per face, of clusters with a mask of the related faces in each;
//   5. the 6 vertex-face and 9 edge-edge stencils of each face pair (KDOPBroadPhase.cpp:150-184), each
//      once: a vertex's or an edge's stencils are the union of the rows of the faces around it, an OR of
//      masks, so the unique set comes out with no global sort.
// Meshes with degenerate faces (a repeated vertex) or duplicate faces break the rule's
// assumptions; for them the raw stencils are emitted and deduplicated by sorting.
#include <cstring>
#include <rocprim/device/device_merge_sort.hpp>
#include <rocprim/device/device_select.hpp>

#include "ccd_core.h"
#include "ccd_internal.h"
#include "grids.h"

namespace {

constexpr int KAX = 13;
constexpr int NB = 2 * KAX;   // bounds per node: 13 mins then 13 maxs

struct Axes {
    double a[KAX][3];
};

// KDOPBroadPhase.cpp:10-32: the 13 directions, each divided by its norm.
Axes make_axes()
{
    static const double raw[KAX][3] = {{1, 0, 0},  {0, 1, 0},  {0, 0, 1},  {1, 1, 0},  {1, -1, 0},
                                       {0, 1, 1},  {0, 1, -1}, {1, 0, 1},  {1, 0, -1}, {1, 1, 1},
                                       {1, 1, -1}, {1, -1, 1}, {1, -1, -1}};
    Axes ax;
    for (int i = 0; i < KAX; i++) {
        ccd::V3 v = ccd::mk(raw[i][0], raw[i][1], raw[i][2]);
        double n = ccd::norm(v);
        ax.a[i][0] = v.x / n;
        ax.a[i][1] = v.y / n;
        ax.a[i][2] = v.z / n;
    }
    return ax;
}

inline unsigned blocks_for(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// ------------------------------------------------------------------------------------------------
// 1. Leaf bounds
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ void dop_point(const Axes &ax, double x, double y, double z, double eta, double *mn,
                                          double *mx)
{
    ccd::V3 p = ccd::mk(x, y, z);
#pragma unroll
    for (int k = 0; k < KAX; k++) {
        double s = ccd::dot(p, ccd::mk(ax.a[k][0], ax.a[k][1], ax.a[k][2]));
        mn[k] = ccd::smin(s - eta, mn[k]);
        mx[k] = ccd::smax(s + eta, mx[k]);
    }
}

// AABBBroadPhase.cpp:31-36: per coordinate, min/max of pos[k] -/+ eta.
__device__ __forceinline__ void aabb_point(double x, double y, double z, double eta, double *mn, double *mx)
{
    double p[3] = {x, y, z};
#pragma unroll
    for (int k = 0; k < 3; k++) {
        mn[k] = ccd::smin(p[k] - eta, mn[k]);
        mx[k] = ccd::smax(p[k] + eta, mx[k]);
    }
}

// Two-entry histories (qs = entry at t=0, qe = entry at t=1) or CSR histories (hoff/hpos).
// aabb != 0 gives AABBBroadPhase's bounds (AABBBroadPhase.cpp:9-40): the three coordinates -/+ eta,
// with the other ten slabs unbounded so that the 13-axis overlap test reduces to the 3-axis one.
__global__ __launch_bounds__(256) void k_leaf_bounds(const int32_t *__restrict__ faces, int64_t F,
                                                     const double *__restrict__ qs, const double *__restrict__ qe,
                                                     const int64_t *__restrict__ hoff,
                                                     const double *__restrict__ hpos, double eta, Axes ax, int aabb,
                                                     double *__restrict__ dop64, double *__restrict__ centre)
{
    int64_t f = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (f >= F) return;
    double mn[KAX], mx[KAX];
#pragma unroll
    for (int k = 0; k < KAX; k++) {
        mn[k] = __builtin_inf();
        mx[k] = -__builtin_inf();
    }
    for (int j = 0; j < 3; j++) {
        int v = faces[3 * f + j];
        if (hoff) {
            for (int64_t e = hoff[v]; e < hoff[v + 1]; e++) {
                if (aabb)
                    aabb_point(hpos[3 * e], hpos[3 * e + 1], hpos[3 * e + 2], eta, mn, mx);
                else
                    dop_point(ax, hpos[3 * e], hpos[3 * e + 1], hpos[3 * e + 2], eta, mn, mx);
            }
        } else {
            const double *a = qs + 3 * (int64_t)v;
            const double *b = qe + 3 * (int64_t)v;
            if (aabb) {
                aabb_point(a[0], a[1], a[2], eta, mn, mx);
                aabb_point(b[0], b[1], b[2], eta, mn, mx);
            } else {
                dop_point(ax, a[0], a[1], a[2], eta, mn, mx);
                dop_point(ax, b[0], b[1], b[2], eta, mn, mx);
            }
        }
    }
    if (aabb) {
#pragma unroll
        for (int k = 3; k < KAX; k++) {
            mn[k] = -__builtin_inf();
            mx[k] = __builtin_inf();
        }
    }
    double *o = dop64 + NB * f;
#pragma unroll
    for (int k = 0; k < KAX; k++) {
        o[k] = mn[k];
        o[KAX + k] = mx[k];
    }
    centre[3 * f + 0] = 0.5 * (mn[0] + mx[0]);
    centre[3 * f + 1] = 0.5 * (mn[1] + mx[1]);
    centre[3 * f + 2] = 0.5 * (mn[2] + mx[2]);
}

// Scene bounds of the centres: per-block partial min/max, then one block folds the partials.
__global__ __launch_bounds__(256) void k_bounds_partial(const double *__restrict__ centre, int64_t F,
                                                        double *__restrict__ partial)
{
    __shared__ double s[6][256];
    double lo[3] = {__builtin_inf(), __builtin_inf(), __builtin_inf()};
    double hi[3] = {-__builtin_inf(), -__builtin_inf(), -__builtin_inf()};
    for (int64_t f = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; f < F; f += (int64_t)gridDim.x * blockDim.x) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
            double v = centre[3 * f + c];
            lo[c] = v < lo[c] ? v : lo[c];
            hi[c] = v > hi[c] ? v : hi[c];
        }
    }
#pragma unroll
    for (int c = 0; c < 3; c++) {
        s[c][threadIdx.x] = lo[c];
        s[3 + c][threadIdx.x] = hi[c];
    }
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
#pragma unroll
            for (int c = 0; c < 3; c++) {
                double a = s[c][threadIdx.x + w];
                if (a < s[c][threadIdx.x]) s[c][threadIdx.x] = a;
                double b = s[3 + c][threadIdx.x + w];
                if (b > s[3 + c][threadIdx.x]) s[3 + c][threadIdx.x] = b;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x < 6) partial[6 * blockIdx.x + threadIdx.x] = s[threadIdx.x][0];
}

__global__ __launch_bounds__(256) void k_bounds_final(double *__restrict__ partial, int nparts,
                                                      double *__restrict__ out)
{
    __shared__ double s[6][256];
    double v[6] = {__builtin_inf(), __builtin_inf(), __builtin_inf(), -__builtin_inf(), -__builtin_inf(),
                   -__builtin_inf()};
    for (int p = threadIdx.x; p < nparts; p += blockDim.x) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
            double a = partial[6 * p + c];
            double b = partial[6 * p + 3 + c];
            v[c] = a < v[c] ? a : v[c];
            v[3 + c] = b > v[3 + c] ? b : v[3 + c];
        }
    }
#pragma unroll
    for (int c = 0; c < 6; c++) s[c][threadIdx.x] = v[c];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
#pragma unroll
            for (int c = 0; c < 3; c++) {
                double a = s[c][threadIdx.x + w];
                if (a < s[c][threadIdx.x]) s[c][threadIdx.x] = a;
                double b = s[3 + c][threadIdx.x + w];
                if (b > s[3 + c][threadIdx.x]) s[3 + c][threadIdx.x] = b;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x < 6) out[threadIdx.x] = s[threadIdx.x][0];
}

// ------------------------------------------------------------------------------------------------
// 2. Morton codes (21 bits per axis)
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ uint64_t spread21(uint64_t x)
{
    x &= 0x1fffffull;
    x = (x | (x << 32)) & 0x1f00000000ffffull;
    x = (x | (x << 16)) & 0x1f0000ff0000ffull;
    x = (x | (x << 8)) & 0x100f00f00f00f00full;
    x = (x | (x << 4)) & 0x10c30c30c30c30c3ull;
    x = (x | (x << 2)) & 0x1249249249249249ull;
    return x;
}

// Keys are (instance id << 3 * axis_bits) | Morton code with axis_bits bits per axis: sorting groups each
// instance's faces, so every instance owns a contiguous range of the leaves.
__global__ __launch_bounds__(256) void k_morton(const double *__restrict__ centre, int64_t F,
                                                const double *__restrict__ box, const int32_t *__restrict__ face_inst,
                                                int axis_bits, uint64_t *__restrict__ keys, int32_t *__restrict__ vals)
{
    int64_t f = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (f >= F) return;
    const double scale = (double)((1u << axis_bits) - 1);
    uint64_t code = 0;
#pragma unroll
    for (int c = 0; c < 3; c++) {
        double lo = box[c], hi = box[3 + c];
        double ext = hi - lo;
        double u = ext > 0 ? (centre[3 * f + c] - lo) / ext : 0.0;
        u = u < 0 ? 0 : (u > 1 ? 1 : u);
        if (!(u == u)) u = 0;   // NaN positions sort first; bounds still decide every pair
        uint64_t q = (uint64_t)(u * scale);
        code |= spread21(q) << c;
    }
    if (face_inst) code |= (uint64_t)face_inst[f] << (3 * axis_bits);
    keys[f] = code;
    vals[f] = (int32_t)f;
}

// Instance of each face: the last instance whose first face is <= f.
__global__ __launch_bounds__(256) void k_face_instance(const int64_t *__restrict__ inst_off, int ninst, int64_t F,
                                                       int32_t *__restrict__ face_inst)
{
    int64_t f = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (f >= F) return;
    int lo = 0, hi = ninst - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (inst_off[mid] <= f)
            lo = mid;
        else
            hi = mid - 1;
    }
    face_inst[f] = lo;
}

// ------------------------------------------------------------------------------------------------
// 3. Leaf, cluster and group records
// ------------------------------------------------------------------------------------------------
// A record holds a box's 26 bounds quantised to 16 bits, two axes to a 32-bit word: lo[w] has the lower
// bounds of axes 2w (low half) and 2w + 1, hi[w] the upper ones; the 14th slot is a padding axis that
// separates nothing (lo 0, hi 65535).  Two boxes are disjoint on some axis exactly when a saturating
// subtraction a.lo - b.hi or b.lo - a.hi leaves a nonzero half, so a box test is 14 packed
// subtractions.  64 consecutive sorted leaves form a cluster (level 1), 64 clusters a group (level 2),
// 64 groups a level-3 record; each record is the union of its children.
//
// The quantisation (ccd::quant_lo, ccd::quant_hi) only ever keeps more pairs; the FP64 leaf test decides.
constexpr int NWORD = 7;   // 32-bit words per side of a box
struct __align__(16) BoxRec {
    uint32_t lo[NWORD];
    uint32_t hi[NWORD];
    uint32_t face;   // a leaf's face id (0 at the upper levels)
    uint32_t pad;
};
static_assert(sizeof(BoxRec) == 64, "box records are 64 bytes");
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u16x2 as_halves(uint32_t x) { return __builtin_bit_cast(u16x2, x); }
__device__ __forceinline__ uint32_t as_word(u16x2 x) { return __builtin_bit_cast(uint32_t, x); }
// The halves of a that exceed those of b, as a nonzero value.
__device__ __forceinline__ uint32_t exceeds(uint32_t a, uint32_t b)
{
    return as_word(__builtin_elementwise_sub_sat(as_halves(a), as_halves(b)));
}
__device__ __forceinline__ uint32_t halves_min(uint32_t a, uint32_t b)
{
    return as_word(__builtin_elementwise_min(as_halves(a), as_halves(b)));
}
__device__ __forceinline__ uint32_t halves_max(uint32_t a, uint32_t b)
{
    return as_word(__builtin_elementwise_max(as_halves(a), as_halves(b)));
}
struct Box16 {
    uint32_t lo[NWORD], hi[NWORD];
};
__device__ __forceinline__ void load_box(const BoxRec *__restrict__ recs, int64_t n, Box16 &b)
{
    const uint4 *p = reinterpret_cast<const uint4 *>(recs + n);
    const uint4 w0 = p[0], w1 = p[1], w2 = p[2], w3 = p[3];
    b.lo[0] = w0.x, b.lo[1] = w0.y, b.lo[2] = w0.z, b.lo[3] = w0.w, b.lo[4] = w1.x, b.lo[5] = w1.y, b.lo[6] = w1.z;
    b.hi[0] = w1.w, b.hi[1] = w2.x, b.hi[2] = w2.y, b.hi[3] = w2.z, b.hi[4] = w2.w, b.hi[5] = w3.x, b.hi[6] = w3.y;
}
__device__ __forceinline__ bool boxes_meet(const Box16 &a, const Box16 &b)
{
    uint32_t sep = 0;
#pragma unroll
    for (int w = 0; w < NWORD; w++) sep |= exceeds(a.lo[w], b.hi[w]) | exceeds(b.lo[w], a.hi[w]);
    return sep == 0;
}
// The union of the 64 lanes' boxes, in every lane.
__device__ __forceinline__ void wave_union(Box16 &b)
{
#pragma unroll
    for (int w = 0; w < NWORD; w++) {
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) {
            b.lo[w] = halves_min(b.lo[w], __shfl_xor(b.lo[w], d));
            b.hi[w] = halves_max(b.hi[w], __shfl_xor(b.hi[w], d));
        }
    }
}
__device__ __forceinline__ void store_box(BoxRec *__restrict__ recs, int64_t n, const Box16 &b, uint32_t face)
{
    uint4 *p = reinterpret_cast<uint4 *>(recs + n);
    p[0] = make_uint4(b.lo[0], b.lo[1], b.lo[2], b.lo[3]);
    p[1] = make_uint4(b.lo[4], b.lo[5], b.lo[6], b.hi[0]);
    p[2] = make_uint4(b.hi[1], b.hi[2], b.hi[3], b.hi[4]);
    p[3] = make_uint4(b.hi[5], b.hi[6], face, 0u);
}
// Quantisation parameters: per-block partial min of the finite lower and max of the finite upper
// bounds per axis (wavefront shuffles, then LDS), then one block folds the partials into origin[13]
// and inv[13] (qparam[0..12], qparam[13..25]).
__global__ __launch_bounds__(256) void k_qrange_partial(const double *__restrict__ dop64, int64_t F,
                                                        double *__restrict__ partial)
{
    __shared__ double s[4][NB];
    double lo[KAX], hi[KAX];
#pragma unroll
    for (int k = 0; k < KAX; k++) {
        lo[k] = __builtin_inf();
        hi[k] = -__builtin_inf();
    }
    for (int64_t f = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; f < F; f += (int64_t)gridDim.x * blockDim.x) {
#pragma unroll
        for (int k = 0; k < KAX; k++) {
            const double a = dop64[NB * f + k], b = dop64[NB * f + KAX + k];
            if (__builtin_isfinite(a) && a < lo[k]) lo[k] = a;
            if (__builtin_isfinite(b) && b > hi[k]) hi[k] = b;
        }
    }
#pragma unroll
    for (int k = 0; k < KAX; k++) {
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) {
            const double a = __shfl_xor(lo[k], d), b = __shfl_xor(hi[k], d);
            lo[k] = a < lo[k] ? a : lo[k];
            hi[k] = b > hi[k] ? b : hi[k];
        }
    }
    const int w = threadIdx.x >> 6;
    if (__lane_id() == 0) {
#pragma unroll
        for (int k = 0; k < KAX; k++) {
            s[w][k] = lo[k];
            s[w][KAX + k] = hi[k];
        }
    }
    __syncthreads();
    if (threadIdx.x < NB) {
        const int c = threadIdx.x;
        double v = s[0][c];
        for (int ww = 1; ww < 4; ww++) v = c < KAX ? (s[ww][c] < v ? s[ww][c] : v) : (s[ww][c] > v ? s[ww][c] : v);
        partial[NB * blockIdx.x + c] = v;
    }
}

__global__ __launch_bounds__(64) void k_qrange_final(const double *__restrict__ partial, int nparts,
                                                     double *__restrict__ qparam, unsigned long long *__restrict__ zero,
                                                     int nzero)
{
    const int k = blockIdx.x;   // one wavefront per axis
    for (int z = k * 64 + threadIdx.x; z < nzero; z += 64 * gridDim.x) zero[z] = 0;   // counters of later kernels
    double lo = __builtin_inf(), hi = -__builtin_inf();
    for (int p = threadIdx.x; p < nparts; p += 64) {
        const double a = partial[NB * p + k], b = partial[NB * p + KAX + k];
        lo = a < lo ? a : lo;
        hi = b > hi ? b : hi;
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
        const double a = __shfl_xor(lo, d), b = __shfl_xor(hi, d);
        lo = a < lo ? a : lo;
        hi = b > hi ? b : hi;
    }
    if (threadIdx.x != 0) return;
    qparam[k] = __builtin_isfinite(lo) ? lo : 0.0;
    qparam[KAX + k] = ccd::quant_scale(lo, hi);
}

// Leaf records in sorted order with the record of each wavefront's cluster, and the FP64 bounds and
// vertex triples in sorted order.
__global__ __launch_bounds__(256) void k_leaf_records(const int32_t *__restrict__ order,
                                                      const double *__restrict__ dop64,
                                                      const int32_t *__restrict__ faces, int64_t F,
                                                      const double *__restrict__ qparam, BoxRec *__restrict__ leaves,
                                                      BoxRec *__restrict__ clusters, double *__restrict__ sdop64,
                                                      int4 *__restrict__ sfaces, int32_t *__restrict__ rank)
{
    const int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int lane = __lane_id();
    const int64_t j0 = j - lane;   // the wavefront's first leaf
    if (j0 >= F) return;           // the whole wavefront is past the leaves
    const bool active = j < F;
    const int64_t f = active ? order[j] : 0;
    // The wavefront's 64 rows of sorted FP64 bounds are one contiguous block: written element by element
    // across the lanes (each store instruction covers consecutive doubles), not row by row per lane.
    const int nrow = F - j0 < 64 ? (int)(F - j0) : 64;
    for (int e = lane; e < 64 * NB; e += 64) {
        const int rr = e / NB, c = e - rr * NB;
        const int64_t fr = __shfl(f, rr);
        if (rr < nrow) sdop64[NB * j0 + e] = dop64[NB * fr + c];
    }
    Box16 r;
#pragma unroll
    for (int w = 0; w < NWORD; w++) {   // the empty box: neutral in the cluster's union
        r.lo[w] = 0xffffffffu;
        r.hi[w] = 0u;
    }
    if (active) {
        const double *src = dop64 + NB * f;
#pragma unroll
        for (int w = 0; w < NWORD; w++) {
            const int k = 2 * w;
            uint32_t lo = ccd::quant_lo(src[k], qparam[k], qparam[KAX + k]);
            uint32_t hi = ccd::quant_hi(src[KAX + k], qparam[k], qparam[KAX + k]);
            if (k + 1 < KAX) {
                lo |= (uint32_t)ccd::quant_lo(src[k + 1], qparam[k + 1], qparam[KAX + k + 1]) << 16;
                hi |= (uint32_t)ccd::quant_hi(src[KAX + k + 1], qparam[k + 1], qparam[KAX + k + 1]) << 16;
            } else {
                hi |= 0xffff0000u;   // the padding axis
            }
            r.lo[w] = lo;
            r.hi[w] = hi;
        }
        store_box(leaves, j, r, (uint32_t)f);
        rank[f] = (int32_t)j;
        sfaces[j] = make_int4(faces[3 * f], faces[3 * f + 1], faces[3 * f + 2], (int)f);
    }
    wave_union(r);
    if (lane == 0) store_box(clusters, j0 >> 6, r, 0u);
}

// The records one level up: each wavefront the union of 64 records.
__global__ __launch_bounds__(256) void k_group_records(const BoxRec *__restrict__ in, int64_t n,
                                                       BoxRec *__restrict__ out)
{
    const int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int lane = __lane_id();
    if (j - lane >= n) return;
    Box16 r;
    load_box(in, j < n ? j : n - 1, r);   // the last record again: the union does not change
    wave_union(r);
    if (lane == 0) store_box(out, j >> 6, r, 0u);
}

// ------------------------------------------------------------------------------------------------
// 4. Unordered overlapping non-neighbouring face pairs
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ bool neighbours(int4 a, int4 b)   // Mesh.cpp:13-20
{
    return a.x == b.x || a.x == b.y || a.x == b.z || a.y == b.x || a.y == b.y || a.y == b.z || a.z == b.x ||
           a.z == b.y || a.z == b.z;
}

// The related faces of every face, as rows (CSR) in sorted leaf order: row i describes the sorted leaves j
// that overlap leaf i without sharing a vertex with it (both directions of every pair), as tiles: a
// cluster's number and the 64-bit mask of its related leaves.  A tile holds several related faces, and
// the union of rows is an OR of masks.
//
// One wavefront finds the rows of one cluster's 64 sorted leaves (one per lane): it looks for the clusters
// its cluster's box meets, 64 records per step (one per lane), and tests each such cluster as a 64 x 64
// tile.  In a tile, each lane first tests its own leaf of the target cluster against the query cluster's
// box; the leaves that pass are broadcast one by one (readlane) and tested against all 64 queries at
// once.  So every step of the search decides 64 box tests from one load, and no step waits for the one
// before it but for the ballot: a tree walk by one wavefront is a chain of dependent record loads.
//
// The pairs that pass are queued in LDS and finished 64 at a time, so that the FP64 test runs with full
// wavefronts: the shared-vertex test (Mesh.cpp:13-20), then the reference's 13-axis test (touching
// counts).  Where every axis overlaps by two quanta or more the FP64 bounds are not read, since they then
// overlap as well (ccd::surely_reaches).
//
// The search keeps the tiles it finds in the order it finds them, and counts them by row; after a scan of
// the counts a second run puts them into their rows.  A row belongs to one wavefront, or to the `slices`
// wavefronts that share its cluster, each taking every slices-th of the target clusters with a count and a
// part of the row of its own: no counter in memory is shared.  Writing each pair once, from its lower leaf, and building the rows from the pairs afterwards
// took two atomics per pair and pass and a claim on one counter per wavefront (about 10 ns each, one after
// another): 76 ms on a 1024^2 sheet with 31M tiles, and 7.7 ms on 128 instances with 3.8M; here 14.3 and
// 1.75 ms, of which placing the tiles is 0.6 and 0.14 (searching a second time instead: 13.4 and 1.5).
// For batched instances a query pairs only with leaves of its instance (face_inst / inst_off; its faces
// are the sorted range [inst_off[k], inst_off[k + 1])).
constexpr int ROW_BLOCK = 256;
constexpr int ROW_QUEUE = 128;   // quantised hits waiting for the exact test (below 64 after a flush)
struct RowLds {
    unsigned long long mask[64];   // each query's related leaves of the tile
    ulonglong2 staged[128];        // records waiting to be written
    int count[64];                 // tiles placed so far, by query
    uint16_t queue[ROW_QUEUE];     // query lane + 64 * target lane
};

// Orders a wavefront's LDS accesses (its own region; one wavefront's LDS instructions execute in order,
// so this only stops the compiler from moving them across).
__device__ __forceinline__ void wave_lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int read_lane(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ int64_t read_lane(int64_t v, int l)
{
    return (int64_t)((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)v, l) |
                     (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), l) << 32);
}

__device__ __forceinline__ int64_t wave_sum(int64_t v)
{
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d);
    return v;
}

// Certainly overlapping: two quanta or more on every axis.
__device__ __forceinline__ bool boxes_meet_surely(const Box16 &a, const Box16 &b)
{
    bool ok = true;
#pragma unroll
    for (int k = 0; k < KAX; k++) {
        const int sh = (k & 1) * 16, w = k >> 1;
        const int al = (a.lo[w] >> sh) & 0xffff, ah = (a.hi[w] >> sh) & 0xffff;
        const int bl = (b.lo[w] >> sh) & 0xffff, bh = (b.hi[w] >> sh) & 0xffff;
        ok = ok & ccd::surely_reaches(ah, bl) & ccd::surely_reaches(bh, al);
    }
    return ok;
}
// Disjoint iff some axis separates them strictly (KDOPBroadPhase.cpp:132-137), with every comparison of a
// part evaluated (no early exit: the loads of a part issue together).  Two
// parts: all 52 doubles at once would take 159 registers, three wavefronts per SIMD.
__device__ __forceinline__ bool overlap64_all(const double *__restrict__ a, const double *__restrict__ b)
{
    bool ok = true;
#pragma nounroll
    for (int part = 0; part < KAX && ok; part += 7) {
        double al[7], ah[7], bl[7], bh[7];
#pragma unroll
        for (int u = 0; u < 7; u++) {
            const int k = part + u < KAX ? part + u : KAX - 1;
            al[u] = a[k];
            ah[u] = a[KAX + k];
            bl[u] = b[k];
            bh[u] = b[KAX + k];
        }
#pragma unroll
        for (int u = 0; u < 7; u++) ok = ok & !((ah[u] < bl[u]) | (bh[u] < al[u]));
    }
    return ok;
}

// The rows' tiles.
struct Rows {
    uint64_t *mask;
    int32_t *cluster;
    int64_t cap;
};
// What the first run finds, kept for the second one: segments of records, the last one of a wavefront known
// by its head and each holding the place of the one before it.  They lie in the edge-edge keys' buffer,
// which nothing writes before the rows are complete; each shard of it has a counter of its own (one counter:
// about 10 ns per claim, one after another).  A wavefront whose shard is used up keeps nothing and searches
// again.
constexpr int REC_SHARDS = 64, REC_STRIDE = 8;   // (a counter per 64 bytes)
constexpr unsigned long long REC_NONE = ~0ull, REC_LOST = ~1ull;
struct RowRecords {
    ulonglong2 *rec;               // mask, cluster | query lane << 32; first of a segment: the one before it
    ulonglong2 *head;              // [wavefronts] last segment: its place (or REC_NONE, REC_LOST), its records
    unsigned long long *claimed;   // [shards * REC_STRIDE]
    int64_t per_shard;
};
struct RowLevels {
    const BoxRec *rec[4];   // leaves, clusters, groups, level 3 (levels above `top` unused)
    int64_t n[4];
    int top;                // the level scanned from end to end
};

// off: [leaf * slices + slice], the tiles in the parts of the rows, or (FILL) their starts; pairs (may be
// null): the related faces in them that come after their row's own.
template <bool FILL>
__global__ __launch_bounds__(ROW_BLOCK, 4) void k_rows(RowLevels lv, int slices, const double *__restrict__ sdop64,
                                                    const int4 *__restrict__ sfaces,
                                                    const int32_t *__restrict__ face_inst,
                                                    const int64_t *__restrict__ inst_off, int64_t *__restrict__ off,
                                                    int32_t *__restrict__ pairs, Rows rows, RowRecords kept)
{
    __shared__ RowLds s_lds[ROW_BLOCK / 64];
    RowLds &L = s_lds[threadIdx.x >> 6];
    const int lane = __lane_id();
    const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    const int F = (int)lv.n[0];   // below 2^30
    // (consecutive blocks run on different XCDs: each gets a contiguous part of the clusters)
    const int64_t nb = gridDim.x >> 3;
    const int64_t block = blockIdx.x < 8 * nb ? (blockIdx.x & 7) * nb + (blockIdx.x >> 3) : blockIdx.x;
    const int64_t wave = block * (ROW_BLOCK / 64) + (threadIdx.x >> 6);
    const int c = __builtin_amdgcn_readfirstlane((int)(wave / slices));   // the query cluster
    const int slice = __builtin_amdgcn_readfirstlane((int)(wave % slices));
    if (c >= lv.n[1]) return;   // the whole wavefront
    const BoxRec *__restrict__ leaves = lv.rec[0];
    const int i0 = c * 64, i = i0 + lane;
    Box16 q, cb;
    load_box(leaves, i < F ? i : F - 1, q);
    load_box(lv.rec[1], c, cb);
    int ibeg = 0x7fffffff, iend = 0;   // lanes past the leaves accept none
    if (i < F) {
        ibeg = 0;
        iend = F;
        if (face_inst) {
            const int k = face_inst[sfaces[i].w];
            ibeg = (int)inst_off[k];
            iend = (int)inst_off[k + 1];
        }
    }
    int jmin = ibeg, jmax = iend;
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
        const int x = __shfl_xor(jmin, d), y = __shfl_xor(jmax, d);
        jmin = x < jmin ? x : jmin;
        jmax = y > jmax ? y : jmax;
    }
    jmin = __builtin_amdgcn_readfirstlane(jmin);
    jmax = __builtin_amdgcn_readfirstlane(jmax);
    const int tfirst = jmin >> 6, tlast = (jmax - 1) >> 6;   // the clusters any lane pairs with
    int64_t row = 0;   // FILL: where this lane's part of the row starts
    if (FILL && i < F) row = off[(int64_t)i * slices + slice];
    int ntiles = 0, npairs = 0, turn = 0;
    if (FILL) {
        ulonglong2 seg = kept.head[wave];
        if (seg.x != REC_LOST) {   // the tiles that the first run kept
            L.count[lane] = 0;
            wave_lds_order();
            while (seg.x != REC_NONE) {
                const ulonglong2 *r = kept.rec + seg.x;
                const int n = (int)seg.y;
                seg = r[0];
                for (int k = lane; k < n; k += 64) {
                    const ulonglong2 e = r[1 + k];
                    const int ql = (int)(e.y >> 32);
                    const int64_t at = off[(int64_t)(i0 + ql) * slices + slice] + atomicAdd(&L.count[ql], 1);
                    if (at < rows.cap) {
                        rows.mask[at] = e.x;
                        rows.cluster[at] = (int32_t)e.y;
                    }
                }
            }
            return;
        }
    }
    // !FILL: the last segment written, and the records waiting.
    unsigned long long last = REC_NONE;
    int last_n = 0, staged = 0;
    auto write_segment = [&]() {
        wave_lds_order();
        const int shard = (int)(wave & (REC_SHARDS - 1));
        unsigned long long got = 0;
        if (lane == 0) got = atomicAdd(&kept.claimed[shard * REC_STRIDE], (unsigned long long)staged + 1);
        got = (unsigned long long)read_lane((int64_t)got, 0);
        if ((int64_t)got + staged + 1 <= kept.per_shard) {
            ulonglong2 *r = kept.rec + shard * kept.per_shard + got;
            if (lane == 0) r[0] = make_ulonglong2(last, last_n);
            for (int k = lane; k < staged; k += 64) r[1 + k] = L.staged[k];
            last = shard * kept.per_shard + got;
            last_n = staged;
        } else {
            last = REC_LOST;
        }
        staged = 0;
        wave_lds_order();
    };
    L.mask[lane] = 0;

    // The exact test of queue[from .. from + n), n <= 64.
    auto test = [&](int t, int from, int n) {
        wave_lds_order();
        if (lane < n) {
            const int e = L.queue[from + lane], ql = e & 63, iq = i0 + ql, j = t * 64 + (e >> 6);
            bool ok = !neighbours(sfaces[iq], sfaces[j]);
            if (ok) {
                Box16 x, y;
                load_box(leaves, iq, x);
                load_box(leaves, j, y);
                if (!boxes_meet_surely(x, y)) ok = overlap64_all(sdop64 + NB * (int64_t)iq, sdop64 + NB * (int64_t)j);
            }
            if (ok) atomicOr(&L.mask[ql], 1ull << (e >> 6));
        }
        wave_lds_order();
    };
    auto tile = [&](int t) {
        const int j = t * 64 + lane;
        Box16 b;
        load_box(leaves, j < F ? j : F - 1, b);
        int nq = 0;
        for (uint64_t m = __ballot(j >= jmin && j < jmax && boxes_meet(b, cb)); m; m &= m - 1) {
            const int s = __ffsll((unsigned long long)m) - 1;
            const int js = t * 64 + s;
            uint32_t sep = 0;
#pragma unroll
            for (int w = 0; w < NWORD; w++) {
                const uint32_t tlo = __builtin_amdgcn_readlane(b.lo[w], s), thi = __builtin_amdgcn_readlane(b.hi[w], s);
                sep |= exceeds(tlo, q.hi[w]) | exceeds(q.lo[w], thi);
            }
            const bool hit = (sep == 0) & (js != i) & (js >= ibeg) & (js < iend);
            const uint64_t h = __ballot(hit);
            if (h == 0) continue;
            if (hit) L.queue[nq + __popcll(h & lt)] = (uint16_t)(lane | s << 6);
            nq += __popcll(h);
            if (nq >= 64) {
                test(t, nq - 64, 64);
                nq -= 64;
            }
        }
        if (nq) test(t, 0, nq);
        const uint64_t mine = L.mask[lane];
        if (!FILL && last != REC_LOST) {
            const uint64_t some = __ballot(mine != 0);
            if (mine) L.staged[staged + __popcll(some & lt)] = make_ulonglong2(mine, (uint32_t)t | (uint64_t)lane << 32);
            staged += __popcll(some);
            if (staged >= 64) write_segment();
        }
        if (mine) {
            L.mask[lane] = 0;
            if (FILL && row + ntiles < rows.cap) {
                rows.mask[row + ntiles] = mine;
                rows.cluster[row + ntiles] = t;
            }
            ntiles++;
            if (pairs) npairs += __popcll(t > c ? mine : (t == c ? mine & ~(lt << 1 | 1ull) : 0ull));   // j > i
        }
        wave_lds_order();
    };
    // The clusters of the 64 records [base, base + 64) of level 1 that the query cluster's box meets.
    auto scan1 = [&](int base) {
        const int t = base + lane;
        Box16 b;
        load_box(lv.rec[1], t < lv.n[1] ? t : lv.n[1] - 1, b);
        for (uint64_t m = __ballot(t >= tfirst && t <= tlast && boxes_meet(b, cb)); m; m &= m - 1) {
            const int tt = base + __ffsll((unsigned long long)m) - 1;
            if (turn == slice) tile(tt);
            turn = turn + 1 == slices ? 0 : turn + 1;
        }
    };
    // Level `lv.top` from end to end, then down to level 1 below the records that the box meets.
    const int up = 6 * (lv.top - 1);
    for (int base = (tfirst >> up) & ~63; base <= (tlast >> up); base += 64) {
        if (lv.top == 1) {
            scan1(base);
            continue;
        }
        const int t = base + lane;
        Box16 b;
        load_box(lv.rec[lv.top], t < lv.n[lv.top] ? t : lv.n[lv.top] - 1, b);
        for (uint64_t m = __ballot(t >= (tfirst >> up) && t <= (tlast >> up) && boxes_meet(b, cb)); m; m &= m - 1) {
            const int t2 = base + __ffsll((unsigned long long)m) - 1;
            if (lv.top == 2) {
                scan1(t2 << 6);
                continue;
            }
            const int u = (t2 << 6) + lane;
            Box16 b2;
            load_box(lv.rec[2], u < lv.n[2] ? u : lv.n[2] - 1, b2);
            for (uint64_t m2 = __ballot(u >= (tfirst >> 6) && u <= (tlast >> 6) && boxes_meet(b2, cb)); m2; m2 &= m2 - 1)
                scan1(((t2 << 6) + __ffsll((unsigned long long)m2) - 1) << 6);
        }
    }
    if (!FILL) {
        if (staged) write_segment();
        if (lane == 0) kept.head[wave] = make_ulonglong2(last, last_n);
    }
    if (!FILL && i < F) {
        off[(int64_t)i * slices + slice] = ntiles;
        if (pairs) pairs[(int64_t)i * slices + slice] = npairs;
    }
}

// ------------------------------------------------------------------------------------------------
// Vertex -> face table (CSR)
// ------------------------------------------------------------------------------------------------
__global__ void k_vf_count(const int32_t *__restrict__ faces, int64_t F, int32_t *__restrict__ cnt)
{
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= 3 * F) return;
    atomicAdd(&cnt[faces[i]], 1);
}
__global__ void k_vf_fill(const int32_t *__restrict__ faces, int64_t F, const int32_t *__restrict__ off,
                          int32_t *__restrict__ cursor, int32_t *__restrict__ list)
{
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= 3 * F) return;
    int v = faces[i];
    int pos = atomicAdd(&cursor[v], 1);
    list[off[v] + pos] = (int32_t)(i / 3);
}

// Mesh checks for the owner rule: a face with a repeated vertex, or two faces with the same vertex
// set (found as equal sorted triples among the faces of each triple's smallest vertex).
__global__ void k_mesh_check(const int32_t *__restrict__ faces, int64_t F, const int32_t *__restrict__ off,
                             const int32_t *__restrict__ list, unsigned long long *flag)
{
    int64_t f = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (f >= F) return;
    int a = faces[3 * f], b = faces[3 * f + 1], c = faces[3 * f + 2];
    bool bad = (a == b || b == c || a == c);
    if (!bad) {
        int lo = a < b ? (a < c ? a : c) : (b < c ? b : c);
        int hi = a > b ? (a > c ? a : c) : (b > c ? b : c);
        int md = a + b + c - lo - hi;
        for (int k = off[lo]; k < off[lo + 1]; k++) {
            int g = list[k];
            if (g == (int)f) continue;
            int x = faces[3 * g], y = faces[3 * g + 1], z = faces[3 * g + 2];
            int l2 = x < y ? (x < z ? x : z) : (y < z ? y : z);
            int h2 = x > y ? (x > z ? x : z) : (y > z ? y : z);
            int m2 = x + y + z - l2 - h2;
            if (l2 == lo && m2 == md && h2 == hi) bad = true;
        }
    }
    if (bad) atomicAdd(flag, 1ull);
}

// Edges of the mesh, faces by their rows (sorted leaves): half-edge 3i + s is edge (v[s], v[s+1]) of face i.
// edge: the edge's number, the smallest of its half-edges; other: the other face on it, -1 on a boundary
// edge, -2 where there are more.
struct FaceEdges {
    uint32_t edge[3];
    int32_t other[3];
    int32_t pad[2];
};
__global__ __launch_bounds__(256) void k_edges(const int4 *__restrict__ sfaces, int64_t F, const int32_t *__restrict__ faces,
                                               const int32_t *__restrict__ off, const int32_t *__restrict__ list,
                                               const int32_t *__restrict__ rank, FaceEdges *__restrict__ edges)
{
    const int64_t x = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (x >= 3 * F) return;
    const int i = (int)(x / 3), s = (int)(x - 3 * (int64_t)i);
    const int4 A = sfaces[i];
    const int a = s == 0 ? A.x : (s == 1 ? A.y : A.z), b = s == 0 ? A.y : (s == 1 ? A.z : A.x);
    int found = -1, n = 0;
    uint32_t c = (uint32_t)x;   // (half-edge numbers need 32 bits: 3 * 2^30)
    for (int k = off[a]; k < off[a + 1]; k++) {
        const int h = list[k];
        if (h == A.w) continue;
        const int32_t *v = faces + 3 * (int64_t)h;
#pragma unroll
        for (int e = 0; e < 3; e++) {
            const int p = v[e], q = v[(e + 1) % 3];
            if ((p == a && q == b) || (p == b && q == a)) {
                found = rank[h];
                n++;
                const uint32_t g = (uint32_t)(3 * (int64_t)found + e);
                c = g < c ? g : c;
            }
        }
    }
    edges[i].edge[s] = c;
    edges[i].other[s] = n > 1 ? -2 : found;
}

// ------------------------------------------------------------------------------------------------
// 5. Stencil expansion: unions of rows
// ------------------------------------------------------------------------------------------------
// The pair of faces {a, b} generates the six vertex-face stencils (a's vertices, b) and (b's vertices, a)
// and the nine edge-edge stencils (KDOPBroadPhase.cpp:150-184); different pairs generate the same ones.
// Gathered by feature instead, each comes out once:
//   * vertex p has the stencils (p, g) for the faces g in the union of the rows of the faces around p;
//   * edge u has the stencils (u, w) for the edges w of the faces in the union of the rows of the faces on
//     u; both u and w see each other, so the one with the smaller number has the stencil.  An edge w of two
//     faces of the union counts at the one that gives it its number.
// (Faces in a row share no vertex with its face, so g does not hold p, and w shares no vertex with u.)
// One wavefront takes a vertex or an edge and ORs its rows' tiles into a table in LDS, by cluster; the set
// bits, numbered across the table, are then shared out over the lanes.  Counts, a scan, and a second run
// that writes the keys: no shared counter.
//
// Deciding for each pair by itself which of its fifteen stencils no smaller pair generates takes up to 39
// membership tests in other faces' sorted rows: 99.5 ms on a 1024^2 sheet with 1.15G stencils, 4.5 ms on 128
// instances with 92M (and minutes where rows of more than 2,048 faces were searched linearly); here 29 ms
// and 3.9 ms.  Writing the keys is 18 GB at 1.2 TB/s on the sheet: the instructions around it bound it, about
// 300 a feature.
//
// A feature whose rows name more clusters than the table takes goes through it several times, each time
// with one class of the clusters, by the upper bits of a hash.  The edge rule may ask for a face of another
// class; whether that is related to the edge's faces is decided again from the bounds.  (Looking it up in
// their rows, which are as long as what they hold, took 1009 ms for a detection of a 256^2 cloth over a ground
// of two triangles, quadratic in the faces; here 26 ms, 20 of them the ground's features, about a microsecond for
// 64 faces.)
constexpr int UNION_BLOCK = 256;
constexpr int TABLE_SLOTS = 512;
struct UnionTable {
    unsigned long long mask[TABLE_SLOTS];
    uint32_t cluster[TABLE_SLOTS];   // ~0u: empty
    int list[128];                   // faces waiting to be written (below 64 after a batch)
};
struct MeshView {
    const int32_t *faces;
    const int32_t *vf_off;
    const int32_t *vf_list;
    const uint8_t *fixed;
    const FaceEdges *edges;   // by row
    const int32_t *rank;      // [F] face -> its row
    const int4 *sfaces;       // vertices and face id by row
    const double *sdop64;     // bounds by row
    const int64_t *off;       // [F * slices + 1] parts of the rows
    Rows rows;
    int slices;
};
__device__ __forceinline__ bool is_fixed(const MeshView &m, int v) { return m.fixed && m.fixed[v]; }

__device__ __forceinline__ int4 vf_key(int p, int a, int b, int c)   // Stencils.h:13-57
{
    int lo = a < b ? (a < c ? a : c) : (b < c ? b : c);
    int hi = a > b ? (a > c ? a : c) : (b > c ? b : c);
    int md = a + b + c - lo - hi;
    return make_int4(p, lo, md, hi);
}
__device__ __forceinline__ int4 ee_key(int a, int b, int c, int d)   // Stencils.h:86-117
{
    int p0 = a < b ? a : b, p1 = a < b ? b : a;
    int q0 = c < d ? c : d, q1 = c < d ? d : c;
    if (p0 > q0) return make_int4(q0, q1, p0, p1);
    return make_int4(p0, p1, q0, q1);
}

// A bijection of 32-bit words (xor-shifts and odd multipliers).
__device__ __forceinline__ uint32_t hash32(uint32_t x)
{
    x ^= x >> 16;
    x *= 0x9E3779B1u;
    x ^= x >> 15;
    x *= 0x85EBCA6Bu;
    return x ^ (x >> 16);
}
// ORs a tile into a table of `last` + 1 slots (a power of two); false when there is no room near its place (a full
// table searched from end to end by tile after tile took longer than the pass that fits).
constexpr uint32_t MOST_PROBES = 128;
__device__ __forceinline__ bool table_or(UnionTable &T, uint32_t last, uint32_t cluster, uint64_t mask)
{
    uint32_t h = hash32(cluster) & last;
    for (uint32_t probe = 0; probe <= last && probe < MOST_PROBES; probe++) {
        const uint32_t old = atomicCAS(&T.cluster[h], ~0u, cluster);
        if (old == ~0u || old == cluster) {
            atomicOr(&T.mask[h], (unsigned long long)mask);
            return true;
        }
        h = (h + 1) & last;
    }
    return false;
}
__device__ __forceinline__ bool table_has(const UnionTable &T, uint32_t last, int j)
{
    const uint32_t cluster = (uint32_t)j >> 6;
    uint32_t h = hash32(cluster) & last;
    for (uint32_t probe = 0; probe <= last; probe++) {
        const uint32_t at = T.cluster[h];
        if (at == ~0u) return false;
        if (at == cluster) return (T.mask[h] >> (j & 63)) & 1ull;
        h = (h + 1) & last;
    }
    return false;
}
// Inclusive sum over the wavefront's lanes (DPP row shifts and broadcasts: no LDS round trips).
__device__ __forceinline__ int wave_scan(int x)
{
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);   // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);   // row_bcast:15
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);   // row_bcast:31
    return x;
}
// Tiles [start, start + len) of row r.
__device__ __forceinline__ void row_range(const MeshView &m, int r, int64_t &start, int &len)
{
    int64_t z = m.off[(int64_t)(r + 1) * m.slices];
    start = m.off[(int64_t)r * m.slices];
    z = z < m.rows.cap ? z : m.rows.cap;
    len = start < z ? (int)(z - start) : 0;
}
// Whether the leaves r and j are related, as the search decides it.
__device__ __forceinline__ bool related(const MeshView &m, int r, int j)
{
    if (neighbours(m.sfaces[r], m.sfaces[j])) return false;
    const double *a = m.sdop64 + NB * (int64_t)r, *b = m.sdop64 + NB * (int64_t)j;
    bool apart = false;
#pragma unroll 3
    for (int k = 0; k < KAX; k++) apart = apart | (a[KAX + k] < b[k]) | (b[KAX + k] < a[k]);
    return !apart;
}
// j related to the leaf f0 or f1, or (f1 -2) to one of the faces around u0 that hold u1.
__device__ bool edge_related(const MeshView &m, int f0, int f1, int u0, int u1, int j)
{
    const int star = m.vf_off[u0], n = f1 == -2 ? m.vf_off[u0 + 1] - star : (f1 == -1 ? 1 : 2);
    for (int k = 0; k < n; k++) {
        int r = k == 0 ? f0 : f1;
        if (f1 == -2) {
            const int f = m.vf_list[star + k];
            const int32_t *v = m.faces + 3 * (int64_t)f;
            if (v[0] != u1 && v[1] != u1 && v[2] != u1) continue;
            r = m.rank[f];
        }
        if (related(m, r, j)) return true;
    }
    return false;
}

// Feature x < V is vertex x; V + h the edge of half-edge h (nothing for a half-edge that is not its edge's
// number).  counts[x]: its stencils (first run) or their offsets (WRITE): vertex-face ones from 0, edge-edge
// ones from counts[V].  Nothing for meshes with degenerate or duplicate faces (raw emission).
//
// A wavefront takes `chunk` features one after another; what leads to their rows (five dependent loads) is
// read for all of them at once, one feature or one face around a vertex per lane.
constexpr int UNION_CHUNK = 16;   // at most
template <bool WRITE>
__global__ __launch_bounds__(UNION_BLOCK) void k_union(MeshView m, int64_t F, int64_t V, int chunk,
                                                       const unsigned long long *__restrict__ raw_dev,
                                                       int64_t *__restrict__ counts, int4 *__restrict__ vf_out,
                                                       int64_t vf_cap, int4 *__restrict__ ee_out, int64_t ee_cap)
{
    __shared__ UnionTable s_table[UNION_BLOCK / 64];
    UnionTable &T = s_table[threadIdx.x >> 6];
    const int lane = __lane_id();
    const int64_t total = V + 3 * F;
    const int64_t nb = gridDim.x >> 3;   // (contiguous features per XCD, as in k_rows)
    const int64_t block = blockIdx.x < 8 * nb ? (blockIdx.x & 7) * nb + (blockIdx.x >> 3) : blockIdx.x;
    const int64_t x0 = (block * (UNION_BLOCK / 64) + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6))) * chunk;
    if (x0 >= total) return;   // the whole wavefront

    // One feature per lane: its end or ends; the faces around it as part [star, star + n) of the vertex ->
    // face table, or (an edge of up to two faces) as the tiles of their rows.
    const int64_t x = x0 + lane;
    int u0 = 0, u1 = -1, f0 = -1, f1 = -2, star = 0, n = 0, len0 = 0, len1 = 0;
    int64_t start0 = 0, start1 = 0, out = 0, result = 0;
    if (lane < chunk && x < total && *raw_dev == 0) {
        if (WRITE) out = counts[x];
        bool star_needed = true;
        if (x < V) {
            u0 = (int)x;
        } else {
            const int64_t h = x - V;
            f0 = (int)(h / 3);
            const int s = (int)(h - 3 * (int64_t)f0);
            star_needed = false;
            if ((int64_t)m.edges[f0].edge[s] == h) {
                const int4 A = m.sfaces[f0];
                u0 = s == 0 ? A.x : (s == 1 ? A.y : A.z);
                u1 = s == 0 ? A.y : (s == 1 ? A.z : A.x);
                f1 = m.edges[f0].other[s];
                if (f1 == -2) {
                    star_needed = true;
                } else {
                    row_range(m, f0, start0, len0);
                    if (f1 >= 0) row_range(m, f1, start1, len1);
                }
            }
        }
        if (star_needed) {
            star = m.vf_off[u0];
            n = m.vf_off[u0 + 1] - star;
        }
    }
    const bool fixed_end = m.fixed && lane < chunk && m.fixed[u0] && (u1 < 0 || m.fixed[u1]);
    const uint64_t fixed_features = __ballot(fixed_end);

    const int64_t ee_base = WRITE ? counts[V] : 0;

    // Entries [wbase, wbase + 64) of the vertex -> face table, with the faces' rows.
    int wbase = -128, wlen = 0;
    int64_t wstart = 0;

    for (uint64_t todo = __ballot(n > 0 || len0 + len1 > 0); todo; todo &= todo - 1) {
        const int s = __ffsll((unsigned long long)todo) - 1;
        const bool edge = x0 + s >= V, ufix = (fixed_features >> s) & 1ull;
        const uint32_t h = edge ? (uint32_t)(x0 + s - V) : 0;
        const int a0 = read_lane(u0, s), a1 = read_lane(u1, s), fn = read_lane(n, s), fstar = read_lane(star, s);
        const int l0 = read_lane(len0, s), l1 = read_lane(len1, s);
        const int64_t s0 = read_lane(start0, s), s1 = read_lane(start1, s);
        const int64_t first = WRITE ? read_lane(out, s) - (edge ? ee_base : 0) : 0;
        int64_t room = (edge ? ee_cap : vf_cap) - first;
        room = room > 0 ? room : 0;
        int4 *const keys = (edge ? ee_out : vf_out) + first;
        int64_t found = 0;   // stencils so far
        int bits = 0;        // classes of clusters: 2^bits, by the hash's upper bits
        uint32_t slots = TABLE_SLOTS;
        for (uint32_t cls = 0; cls < (1u << bits); cls++) {
            bool over = false;
            auto clear = [&](int entries) {
                slots = 64;
                while (slots < TABLE_SLOTS && slots < 2u * (uint32_t)entries) slots <<= 1;
                if (bits) slots = TABLE_SLOTS;
                for (uint32_t q = lane; q < slots; q += 64) {
                    T.cluster[q] = ~0u;
                    T.mask[q] = 0ull;
                }
                wave_lds_order();
            };
            auto add = [&](int64_t at) {
                const uint32_t t = (uint32_t)m.rows.cluster[at];
                const uint64_t mask = m.rows.mask[at];
                if (!over && (bits == 0 || hash32(t) >> (32 - bits) == cls)) over = !table_or(T, slots - 1, t, mask);
            };
            if (fn == 0) {
                clear(l0 + l1);
                for (int e0 = 0; e0 < l0 + l1; e0 += 64) {
                    const int e = e0 + lane;
                    if (e < l0 + l1) add(e < l0 ? s0 + e : s1 + (e - l0));
                }
            } else {
                if (fn > 64) clear(TABLE_SLOTS);
                for (int k0 = 0; k0 < fn; k0 += 64) {
                    const int at0 = fstar + k0, k = fn - k0 < 64 ? fn - k0 : 64;
                    if (at0 < wbase || at0 + k > wbase + 64) {
                        wbase = at0;
                        wlen = 0;
                        if ((int64_t)wbase + lane < 3 * F) row_range(m, m.rank[m.vf_list[wbase + lane]], wstart, wlen);
                    }
                    const int a = at0 - wbase;
                    int len = lane >= a && lane < a + k ? wlen : 0;
                    if (edge && len) {   // those around a0 that hold a1
                        const int32_t *v = m.faces + 3 * (int64_t)m.vf_list[wbase + lane];
                        if (v[0] != a1 && v[1] != a1 && v[2] != a1) len = 0;
                    }
                    const int incl = wave_scan(len);
                    const int all = read_lane(incl, 63);
                    if (fn <= 64) clear(all);
                    int steps = 1;
                    while (steps < k) steps <<= 1;
                    for (int e0 = 0; e0 < all; e0 += 64) {
                        const int e = e0 + lane;
                        int row = a;   // the row that holds entry e: the first whose inclusive sum exceeds it
                        for (int d = steps >> 1; d > 0; d >>= 1) {
                            const int probe = row + d - 1;
                            if (__shfl(incl, probe < 63 ? probe : 63) <= e) row += d;
                        }
                        row = row < 63 ? row : 63;
                        const int before = __shfl(incl - len, row);
                        const int64_t at = __shfl(wstart, row) + (e - before);
                        if (e < all) add(at);
                    }
                }
            }
            wave_lds_order();
            if (__ballot(over)) {   // start again with twice the classes (the clusters of one of 2^23 have a slot each)
                bits++;
                found = 0;
                cls = ~0u;
                continue;
            }
            // The faces of the table, 64 at a time.
            auto batch = [&](int from, int cnt) {
                const bool valid = lane < cnt;
                wave_lds_order();
                const int g = valid ? T.list[from + lane] : 0;
                const int4 G = m.sfaces[g];
                auto emit = [&](bool mine, int4 key) {
                    const uint64_t b = __ballot(mine);
                    if (WRITE && mine) {
                        const int64_t pos = found + __builtin_amdgcn_mbcnt_hi((int)(b >> 32), __builtin_amdgcn_mbcnt_lo((int)b, 0));
                        if (pos < room) keys[pos] = key;
                    }
                    found += __popcll(b);
                };
                if (!edge) {
                    emit(valid && !(ufix && m.fixed[G.x] && m.fixed[G.y] && m.fixed[G.z]), vf_key(a0, G.x, G.y, G.z));
                    return;
                }
                const FaceEdges E = m.edges[g];
#pragma unroll
                for (int w = 0; w < 3; w++) {
                    const int w0 = w == 0 ? G.x : (w == 1 ? G.y : G.z), w1 = w == 0 ? G.y : (w == 1 ? G.z : G.x);
                    bool mine = valid && E.edge[w] > h && !(ufix && m.fixed[w0] && m.fixed[w1]);
                    if (mine && E.edge[w] != (uint32_t)g * 3u + (uint32_t)w) {
                        // The number comes from another face: it has the edge if it is in the union.
                        const int owner = (int)(E.edge[w] / 3u);
                        auto has = [&](int j) {
                            if (bits == 0) return table_has(T, slots - 1, j);
                            return edge_related(m, (int)(h / 3u), m.edges[h / 3u].other[h % 3u], a0, a1, j);
                        };
                        bool in = has(owner);
                        if (!in && E.other[w] == -2) {
                            // Several faces: the first of them in the union, by row, has it.
                            for (int k = m.vf_off[w0]; k < m.vf_off[w0 + 1] && !in; k++) {
                                const int f = m.vf_list[k], r = m.rank[f];
                                const int32_t *v = m.faces + 3 * (int64_t)f;
                                if (r < g && (v[0] == w1 || v[1] == w1 || v[2] == w1)) in = has(r);
                            }
                        }
                        mine = !in;
                    }
                    emit(mine, ee_key(a0, a1, w0, w1));
                }
            };
            int waiting = 0;
            for (uint32_t q0 = 0; q0 < slots; q0 += 64) {
                const int t = (int)T.cluster[q0 + lane];
                const int64_t mask = (int64_t)T.mask[q0 + lane];
                for (uint64_t b = __ballot(mask != 0); b; b &= b - 1) {
                    const int q = __ffsll((unsigned long long)b) - 1;
                    const uint64_t mk = (uint64_t)read_lane(mask, q);
                    if (!WRITE && !edge && !ufix) {
                        found += __popcll(mk);
                        continue;
                    }
                    if ((mk >> lane) & 1ull)
                        T.list[waiting + __builtin_amdgcn_mbcnt_hi((int)(mk >> 32), __builtin_amdgcn_mbcnt_lo((int)mk, 0))] =
                            read_lane(t, q) * 64 + lane;
                    waiting += __popcll(mk);
                    if (waiting >= 64) {
                        batch(waiting - 64, 64);
                        waiting -= 64;
                    }
                }
            }
            if (waiting) batch(0, waiting);
            wave_lds_order();
        }
        if (!WRITE && lane == s) result = found;
    }
    if (!WRITE && lane < chunk && x < total) counts[x] = result;
}

// The counters after the scans: the rows' tiles and the stencils.
__global__ void k_expand_counts(const int64_t *__restrict__ row_total, const int64_t *__restrict__ counts, int64_t V,
                                const int64_t *__restrict__ total, unsigned long long *c)
{
    c[ccdi::C_ROWS] = (unsigned long long)*row_total;
    if (c[ccdi::C_BAD] == 0) {
        c[ccdi::C_VF] = (unsigned long long)counts[V];
        c[ccdi::C_EE] = (unsigned long long)(*total - counts[V]);
    }
}
// Face pairs, from what the parts of the rows hold of them.
__global__ __launch_bounds__(256) void k_pair_total(const int32_t *__restrict__ pairs, int64_t n, unsigned long long *c)
{
    __shared__ int64_t s[4];
    int64_t v = 0;
    for (int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) v += pairs[i];
    v = wave_sum(v);
    if (__lane_id() == 0) s[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(&c[ccdi::C_PAIRS], (unsigned long long)(s[0] + s[1] + s[2] + s[3]));
}

// Raw emission, for meshes with degenerate or duplicate faces: all fifteen stencils of every pair (but those
// of fixed vertices), deduplicated afterwards by sorting.  One wavefront per face over its row's later
// faces.  A wavefront counts what its faces give, claims their places with one atomic per stencil kind, and goes
// through them again to write: 0.56 ms for the expansion of a 256^2 cloth with a degenerate face.  (An atomic per
// stencil of the fifteen and tile, on two counters: 50.6 ms.)
__global__ __launch_bounds__(256) void k_expand_raw(MeshView m, int64_t F, const unsigned long long *__restrict__ raw_dev,
                                                    int4 *__restrict__ vf_out, int64_t vf_cap,
                                                    unsigned long long *vf_counter, int4 *__restrict__ ee_out,
                                                    int64_t ee_cap, unsigned long long *ee_counter)
{
    if (*raw_dev == 0) return;
    const int lane = __lane_id();
    const int64_t nwaves = (int64_t)gridDim.x * 4;
    // emit(vertex-face or not, whether the lane has the stencil, its key) for every stencil of the wavefront's faces
    auto walk = [&](auto &&emit) {
        for (int64_t i = blockIdx.x * (int64_t)4 + (threadIdx.x >> 6); i < F; i += nwaves) {
            const int64_t lo = m.off[i * m.slices];
            int64_t hi = m.off[(i + 1) * m.slices];
            hi = hi < m.rows.cap ? hi : m.rows.cap;
            const int4 A = m.sfaces[i];
            const int fv[3] = {A.x, A.y, A.z};
            const bool ffix = is_fixed(m, A.x) && is_fixed(m, A.y) && is_fixed(m, A.z);
            for (int64_t e = lo; e < hi; e++) {   // a tile: one of its leaves per lane
                const int64_t j = (int64_t)m.rows.cluster[e] * 64 + lane;
                const bool valid = j > i && ((m.rows.mask[e] >> lane) & 1ull);
                const int4 B = m.sfaces[valid ? j : 0];
                const int gv[3] = {B.x, B.y, B.z};
                const bool gfix = is_fixed(m, B.x) && is_fixed(m, B.y) && is_fixed(m, B.z);
#pragma unroll
                for (int s = 0; s < 3; s++) {
                    emit(true, valid && !(is_fixed(m, fv[s]) && gfix), vf_key(fv[s], gv[0], gv[1], gv[2]));
                    emit(true, valid && !(is_fixed(m, gv[s]) && ffix), vf_key(gv[s], fv[0], fv[1], fv[2]));
#pragma unroll
                    for (int t = 0; t < 3; t++) {
                        const int a0 = fv[s], a1 = fv[(s + 1) % 3], b0 = gv[t], b1 = gv[(t + 1) % 3];
                        emit(false, valid && !(is_fixed(m, a0) && is_fixed(m, a1) && is_fixed(m, b0) && is_fixed(m, b1)),
                             ee_key(a0, a1, b0, b1));
                    }
                }
            }
        }
    };
    unsigned long long nvf = 0, nee = 0;
    walk([&](bool vf, bool want, int4) { (vf ? nvf : nee) += __popcll(__ballot(want)); });
    unsigned long long vf_at = 0, ee_at = 0;
    if (lane == 0 && nvf) vf_at = atomicAdd(vf_counter, nvf);
    if (lane == 0 && nee) ee_at = atomicAdd(ee_counter, nee);
    vf_at = (unsigned long long)read_lane((int64_t)vf_at, 0);
    ee_at = (unsigned long long)read_lane((int64_t)ee_at, 0);
    walk([&](bool vf, bool want, int4 key) {
        const uint64_t b = __ballot(want);
        unsigned long long &at = vf ? vf_at : ee_at;
        const int64_t pos = (int64_t)at + __popcll(b & ((1ull << lane) - 1ull));
        if (want && pos < (vf ? vf_cap : ee_cap)) (vf ? vf_out : ee_out)[pos] = key;
        at += __popcll(b);
    });
}

// Stencil order of the reference's std::set (Stencils.h:59-77 and :119-137): lexicographic.
struct KeyLess {
    __host__ __device__ bool operator()(const int4 &a, const int4 &b) const
    {
        if (a.x != b.x) return a.x < b.x;
        if (a.y != b.y) return a.y < b.y;
        if (a.z != b.z) return a.z < b.z;
        return a.w < b.w;
    }
};
struct KeyEq {
    __host__ __device__ bool operator()(const int4 &a, const int4 &b) const
    {
        return a.x == b.x && a.y == b.y && a.z == b.z && a.w == b.w;
    }
};

}   // namespace

namespace ccdi {

// Sorts n stencil keys (device, 4*n int32) into the reference's set order.
int sort_stencils(ccd_ctx *ctx, int32_t *keys, int64_t n)
{
    if (n <= 1) return CCD_OK;
    size_t tmp = 0;
    int4 *sorted = (int4 *)buffer(ctx, "sort_out", (size_t)n * 16 + 16);
    if (!sorted) return CCD_E_OOM;
    CCD_HIP_CHECK(ctx, rocprim::merge_sort((void *)nullptr, tmp, (int4 *)keys, sorted, (size_t)n, KeyLess(),
                                           ctx->stream));
    void *t = buffer(ctx, "sort_tmp", tmp + 16);
    if (!t) return CCD_E_OOM;
    CCD_HIP_CHECK(ctx, rocprim::merge_sort(t, tmp, (int4 *)keys, sorted, (size_t)n, KeyLess(), ctx->stream));
    CCD_HIP_CHECK(ctx, hipMemcpyAsync(keys, sorted, (size_t)n * 16, hipMemcpyDeviceToDevice, ctx->stream));
    return CCD_OK;
}

// Sort + unique in place; the unique count goes to *count_dev.
static int sort_unique(ccd_ctx *ctx, int32_t *keys, int64_t n, const char *tag, int64_t *count_dev)
{
    int rc = sort_stencils(ctx, keys, n);
    if (rc) return rc;
    std::string name = std::string("uniq_out_") + tag;
    int4 *out = (int4 *)buffer(ctx, name.c_str(), (size_t)n * 16 + 16);
    if (!out) return CCD_E_OOM;
    size_t tmp = 0;
    CCD_HIP_CHECK(ctx, rocprim::unique((void *)nullptr, tmp, (int4 *)keys, out, (unsigned long long *)count_dev,
                                       (size_t)n, KeyEq(), ctx->stream));
    void *t = buffer(ctx, "uniq_tmp", tmp + 16);
    if (!t) return CCD_E_OOM;
    CCD_HIP_CHECK(ctx, rocprim::unique(t, tmp, (int4 *)keys, out, (unsigned long long *)count_dev, (size_t)n,
                                       KeyEq(), ctx->stream));
    CCD_HIP_CHECK(ctx, hipMemcpyAsync(keys, out, (size_t)n * 16, hipMemcpyDeviceToDevice, ctx->stream));
    return CCD_OK;
}

int build_vertex_face_table_buffers(ccd_ctx *ctx, int64_t F, int64_t V)
{
    if (!buffer(ctx, "vf_cnt", (size_t)(V + 1) * 4) || !buffer(ctx, "vf_off", (size_t)(V + 1) * 4) ||
        !buffer(ctx, "vf_list", (size_t)(3 * F + 1) * 4) || !buffer(ctx, "scan_tmp", scan_temp_bytes(V + 1)))
        return CCD_E_OOM;
    return CCD_OK;
}

int build_vertex_face_table(ccd_ctx *ctx, const int32_t *faces, int64_t F, int64_t V)
{
    hipStream_t st = ctx->stream;
    int rc = build_vertex_face_table_buffers(ctx, F, V);
    if (rc) return rc;
    int32_t *vcnt = (int32_t *)ctx->bufs["vf_cnt"].ptr;
    int32_t *voff = (int32_t *)ctx->bufs["vf_off"].ptr;
    int32_t *vlist = (int32_t *)ctx->bufs["vf_list"].ptr;
    void *scan_tmp = ctx->bufs["scan_tmp"].ptr;
    rc = fill_u32(ctx, (uint32_t *)vcnt, V + 1, 0);
    if (rc) return rc;
    if (F > 0) {
        hipLaunchKernelGGL(k_vf_count, dim3(blocks_for(3 * F, 256)), dim3(256), 0, st, faces, F, vcnt);
        CCD_LAUNCH_CHECK(ctx);
    }
    rc = exclusive_scan_i32(ctx, vcnt, voff, V + 1, scan_tmp, nullptr);
    if (rc) return rc;
    rc = fill_u32(ctx, (uint32_t *)vcnt, V + 1, 0);
    if (rc) return rc;
    if (F > 0) {
        hipLaunchKernelGGL(k_vf_fill, dim3(blocks_for(3 * F, 256)), dim3(256), 0, st, faces, F, voff, vcnt, vlist);
        CCD_LAUNCH_CHECK(ctx);
    }
    return CCD_OK;
}

void vertex_face_table(ccd_ctx *ctx, const int32_t **off, const int32_t **list)
{
    *off = (const int32_t *)ctx->bufs["vf_off"].ptr;
    *list = (const int32_t *)ctx->bufs["vf_list"].ptr;
}

// Device buffers of one broadphase, sized for F faces and V vertices and the capacities in caps.
struct BPBufs {
    double *dop64, *centre, *partial, *sdop64;
    double *qpartial, *qparam;   // node quantisation: per-block partial ranges, origin[13] + inv[13]
    uint64_t *keys, *keys2;
    int32_t *vals, *order, *face_inst;
    BoxRec *boxes;   // leaf records, then the levels above (level_offsets)
    int4 *sfaces;
    void *sort_tmp;
    int64_t *row_off;    // parts of the related-face rows: tiles, then starts
    Rows rows;           // their tiles
    RowRecords kept;     // the first run's finds
    int32_t *row_pairs;  // related faces in them (null unless the pairs are counted)
    int64_t *counts;     // stencils per vertex and half-edge: counts, then offsets
    int64_t *totals;     // their sum
    void *scan_tmp;
    int4 *vfk, *eek;
    FaceEdges *edges;   // by row (kept with the vertex -> face table for refits)
    int32_t *rank;   // face id -> Morton-sorted position
};
// Where each level's records start in BPBufs::boxes, and their number: level 0 the leaves, each level
// above a 64th of the one below (rounded up).
struct LevelOffsets {
    int64_t at[4], n[4], total;
};
static LevelOffsets level_offsets(int64_t F)
{
    LevelOffsets l;
    int64_t at = 0, n = F;
    for (int k = 0; k < 4; k++) {
        l.at[k] = at;
        l.n[k] = n;
        at += n;
        n = (n + 63) >> 6;
    }
    l.total = at;
    return l;
}
constexpr int NPARTS = 512;
constexpr int QPARTS = 4096;   // blocks of the quantisation range pass (enough to fill the GPU)

// Wavefronts that share a cluster in the row search: a power of two up to 16 (each of them scans the upper
// levels by itself), and up to 512 wavefronts per CU, since work per cluster is very uneven.  Measured with
// 64, 128, 512 and 1024 per CU: 436, 400, 366 and 355 us on 2,033 clusters, 4580, 2540, 1614 and 1970 us on
// 14,294, and 29, 29, 13.6 and 13.2 ms on 32,705; with up to 32 in a cluster 57 and 27 us on 288 and 3
// clusters become 61 and 27, and placing the tiles 6 and 4 become 8 and 23.
static int row_slices(const ccd_ctx *ctx, int64_t F)
{
    const int64_t clusters = (F + 63) / 64, want = (int64_t)ctx->num_cus * 512;
    int s = 1;
    while (s < 16 && 2 * s * clusters <= want) s *= 2;
    return s;
}

static int bp_buffers(ccd_ctx *ctx, int64_t F, int64_t V, bool batched, BPBufs &b)
{
    b.dop64 = (double *)buffer(ctx, "dop64", (size_t)F * NB * 8);
    b.centre = (double *)buffer(ctx, "centre", (size_t)F * 3 * 8);
    b.partial = (double *)buffer(ctx, "bpartial", (size_t)NPARTS * 6 * 8 + 64);
    b.qpartial = (double *)buffer(ctx, "qpartial", (size_t)QPARTS * NB * 8);
    b.qparam = (double *)buffer(ctx, "qparam", (size_t)NB * 8);
    b.keys = (uint64_t *)buffer(ctx, "mkeys", (size_t)F * 8);
    b.keys2 = (uint64_t *)buffer(ctx, "mkeys2", (size_t)F * 8);
    b.vals = (int32_t *)buffer(ctx, "mvals", (size_t)F * 4);
    b.order = (int32_t *)buffer(ctx, "order", (size_t)F * 4);
    b.face_inst = batched ? (int32_t *)buffer(ctx, "face_inst", (size_t)F * 4) : nullptr;
    b.boxes = (BoxRec *)buffer(ctx, "boxes", (size_t)level_offsets(F).total * sizeof(BoxRec));
    b.sdop64 = (double *)buffer(ctx, "sdop64", (size_t)F * NB * 8);
    b.sfaces = (int4 *)buffer(ctx, "sfaces", (size_t)F * 16);
    b.sort_tmp = buffer(ctx, "radix_tmp", radix_sort_temp_bytes(F));
    b.vfk = (int4 *)buffer(ctx, "vf_keys", (size_t)ctx->cap_vf * 16);
    b.eek = (int4 *)buffer(ctx, "ee_keys", (size_t)ctx->cap_ee * 16);
    b.edges = (FaceEdges *)buffer(ctx, "face_edges", (size_t)F * sizeof(FaceEdges));
    b.rank = (int32_t *)buffer(ctx, "face_rank", (size_t)F * 4);
    const int64_t parts = (F + 1) * row_slices(ctx, F), feats = V + 3 * F + 1;
    b.row_off = (int64_t *)buffer(ctx, "row_off", (size_t)parts * 8);
    b.rows.mask = (uint64_t *)buffer(ctx, "row_mask", (size_t)ctx->cap_rows * 8);
    b.rows.cluster = (int32_t *)buffer(ctx, "row_cluster", (size_t)ctx->cap_rows * 4);
    b.rows.cap = ctx->cap_rows;
    const int64_t waves = (F + 63) / 64 * row_slices(ctx, F);
    b.kept.head = (ulonglong2 *)buffer(ctx, "row_heads", (size_t)waves * 16 + REC_SHARDS * REC_STRIDE * 8);
    b.kept.claimed = (unsigned long long *)(b.kept.head + waves);
    b.kept.rec = (ulonglong2 *)b.eek;
    b.kept.per_shard = ctx->cap_ee / REC_SHARDS;
    b.row_pairs = ctx->count_pairs ? (int32_t *)buffer(ctx, "row_pairs", (size_t)parts * 4) : nullptr;
    b.counts = (int64_t *)buffer(ctx, "feature_counts", (size_t)feats * 8);
    b.totals = (int64_t *)buffer(ctx, "expand_totals", 16);
    b.scan_tmp = buffer(ctx, "expand_scan_tmp", scan_temp_bytes(std::max(parts, feats)));
    if (!b.dop64 || !b.centre || !b.partial || !b.qpartial || !b.qparam || !b.keys || !b.keys2 || !b.vals || !b.order ||
        (batched && !b.face_inst) || !b.boxes || !b.sdop64 || !b.sfaces || !b.sort_tmp || !b.vfk || !b.eek || !b.edges ||
        !b.rank || !b.row_off || !b.rows.mask || !b.rows.cluster || !b.kept.head || (ctx->count_pairs && !b.row_pairs) || !b.counts ||
        !b.totals || !b.scan_tmp)
        return CCD_E_OOM;
    return CCD_OK;
}

// The node quantisation's range from the leaves' FP64 bounds (before the leaf records are written).
static int launch_qrange(ccd_ctx *ctx, const BPBufs &b, int64_t F)
{
    const int nb = (int)std::min<int64_t>(QPARTS, blocks_for(F, 256));
    hipLaunchKernelGGL(k_qrange_partial, dim3(nb), dim3(256), 0, ctx->stream, b.dop64, F, b.qpartial);
    CCD_LAUNCH_CHECK(ctx);
    hipLaunchKernelGGL(k_qrange_final, dim3(KAX), dim3(64), 0, ctx->stream, b.qpartial, nb, b.qparam,
                       b.kept.claimed, REC_SHARDS * REC_STRIDE);
    CCD_LAUNCH_CHECK(ctx);
    return CCD_OK;
}

// The box records of every level, and the pair search over them.  The search scans the lowest level of at
// most SCAN_MAX records from end to end (64 records a step), and descends from there.
constexpr int64_t SCAN_MAX = 512;   // (2,048: 476 us instead of 397 on 2,033 clusters)
static int launch_boxes(ccd_ctx *ctx, const BPBufs &b, const int32_t *order, const int32_t *faces, int64_t F)
{
    const LevelOffsets l = level_offsets(F);
    hipLaunchKernelGGL(k_leaf_records, dim3(blocks_for(F, 256)), dim3(256), 0, ctx->stream, order, b.dop64, faces, F,
                       b.qparam, b.boxes, b.boxes + l.at[1], b.sdop64, b.sfaces, b.rank);
    CCD_LAUNCH_CHECK(ctx);
    for (int k = 1; k < 3 && l.n[k] > SCAN_MAX; k++) {
        hipLaunchKernelGGL(k_group_records, dim3(blocks_for(l.n[k], 256)), dim3(256), 0, ctx->stream, b.boxes + l.at[k],
                           l.n[k], b.boxes + l.at[k + 1]);
        CCD_LAUNCH_CHECK(ctx);
    }
    return CCD_OK;
}
// The related-face rows: count, scan, fill.  The rows' starts end up in b.row_off, (F + 1) * slices of them.
static int launch_rows(ccd_ctx *ctx, const BPBufs &b, int64_t F, const int64_t *inst_off)
{
    const LevelOffsets l = level_offsets(F);
    RowLevels lv;
    lv.top = 1;
    for (int k = 0; k < 4; k++) {
        lv.rec[k] = b.boxes + l.at[k];
        lv.n[k] = l.n[k];
    }
    while (lv.top < 3 && l.n[lv.top] > SCAN_MAX) lv.top++;
    const int slices = row_slices(ctx, F);
    const dim3 grid(blocks_for(l.n[1] * slices, ROW_BLOCK / 64));
    hipLaunchKernelGGL(k_rows<false>, grid, dim3(ROW_BLOCK), 0, ctx->stream, lv, slices, b.sdop64, b.sfaces, b.face_inst,
                       inst_off, b.row_off, b.row_pairs, b.rows, b.kept);
    CCD_LAUNCH_CHECK(ctx);
    // One scan over all parts; the entry past the last row's gets the total (what it held counts for nothing).
    int rc = exclusive_scan_i64(ctx, b.row_off, b.row_off, F * slices + 1, b.scan_tmp, nullptr);
    if (rc) return rc;
    hipLaunchKernelGGL(k_rows<true>, grid, dim3(ROW_BLOCK), 0, ctx->stream, lv, slices, b.sdop64, b.sfaces, b.face_inst,
                       inst_off, b.row_off, (int32_t *)nullptr, b.rows, b.kept);
    CCD_LAUNCH_CHECK(ctx);
    return CCD_OK;
}

// The stencils from the rows: count, scan, write (or raw emission, by the device's own decision).
static int launch_expand(ccd_ctx *ctx, const BPBufs &b, const int32_t *faces, int64_t F, int64_t V, const int32_t *voff,
                         const int32_t *vlist, const uint8_t *fixed)
{
    hipStream_t st = ctx->stream;
    unsigned long long *c = (unsigned long long *)ctx->d_counts;
    const MeshView mv{faces, voff, vlist, fixed, b.edges, b.rank, b.sfaces, b.sdop64, b.row_off, b.rows, row_slices(ctx, F)};
    const int64_t feats = V + 3 * F;
    // Fewer features to a wavefront where there are few: on 160 faces the two runs take 24 and 29 us with 16,
    // 8 and 7 with 1; on 18,432 faces 43 and 52 with 16, 37 and 44 with 4, 40 and 45 with 2.
    int chunk = UNION_CHUNK;
    while (chunk > 1 && feats / chunk < (int64_t)ctx->num_cus * 48) chunk /= 2;
    const dim3 grid(blocks_for(feats, chunk * (UNION_BLOCK / 64)));
    hipLaunchKernelGGL(k_union<false>, grid, dim3(UNION_BLOCK), 0, st, mv, F, V, chunk, c + C_BAD, b.counts, b.vfk,
                       (int64_t)0, b.eek, (int64_t)0);
    CCD_LAUNCH_CHECK(ctx);
    int rc = exclusive_scan_i64(ctx, b.counts, b.counts, feats, b.scan_tmp, b.totals);
    if (rc) return rc;
    hipLaunchKernelGGL(k_expand_counts, dim3(1), dim3(1), 0, st, b.row_off + F * mv.slices, b.counts, V, b.totals, c);
    CCD_LAUNCH_CHECK(ctx);
    if (b.row_pairs) {
        const int64_t parts = F * mv.slices;
        hipLaunchKernelGGL(k_pair_total, dim3((unsigned)std::min<int64_t>(blocks_for(parts, 1024), 256)), dim3(256), 0, st,
                           b.row_pairs, parts, c);
        CCD_LAUNCH_CHECK(ctx);
    }
    hipLaunchKernelGGL(k_union<true>, grid, dim3(UNION_BLOCK), 0, st, mv, F, V, chunk, c + C_BAD, b.counts, b.vfk, ctx->cap_vf,
                       b.eek, ctx->cap_ee);
    CCD_LAUNCH_CHECK(ctx);
    hipLaunchKernelGGL(k_expand_raw, dim3((unsigned)std::min<int64_t>(blocks_for(F, 4), 4096)), dim3(256), 0, st, mv, F,
                       c + C_BAD, b.vfk, ctx->cap_vf, c + C_VF, b.eek, ctx->cap_ee, c + C_EE);
    CCD_LAUNCH_CHECK(ctx);
    return CCD_OK;
}

int broadphase_prepare(ccd_ctx *ctx, int64_t F, int64_t V, bool batched)
{
    // Capacities: grow-only, first guesses from the face count (the 256^2 cloth has 3.7 row tiles, 21
    // vertex-face and 38 edge-edge stencils per face); an overflow is detected after the run.
    ctx->cap_rows = std::max<int64_t>(ctx->cap_rows, 8 * F + 1024);
    ctx->cap_vf = std::max<int64_t>(ctx->cap_vf, 24 * F + 1024);
    ctx->cap_ee = std::max<int64_t>(ctx->cap_ee, 40 * F + 1024);
    BPBufs b;
    int rc = bp_buffers(ctx, F, V, batched, b);
    if (rc) return rc;
    rc = build_vertex_face_table_buffers(ctx, F, V);
    return rc;
}

int broadphase_launch(ccd_ctx *ctx, const int32_t *faces, int64_t F, const double *qs, const double *qe,
                      const int64_t *hist_off, const double *hist_pos, int64_t V, double eta, const uint8_t *fixed,
                      bool aabb, const int64_t *inst_off, int ninst)
{
    hipStream_t st = ctx->stream;
    int64_t *cnt = ctx->d_counts;
    unsigned long long *c = (unsigned long long *)cnt;
    int rc = fill_u64(ctx, (uint64_t *)cnt, NCOUNTERS, 0);
    if (rc) return rc;
    if (F < 2) return CCD_OK;
    const bool batched = inst_off && ninst > 1;
    BPBufs b;
    rc = bp_buffers(ctx, F, V, batched, b);
    if (rc) return rc;
    static const Axes axes = make_axes();
    int inst_bits = 0;
    if (batched)
        while ((1ll << inst_bits) < ninst) inst_bits++;

    prof_begin(ctx, CCD_T_BOUNDS);
    hipLaunchKernelGGL(k_leaf_bounds, dim3(blocks_for(F, 256)), dim3(256), 0, st, faces, F, qs, qe, hist_off,
                       hist_pos, eta, axes, aabb ? 1 : 0, b.dop64, b.centre);
    CCD_LAUNCH_CHECK(ctx);
    int nb = (int)std::min<int64_t>(NPARTS, blocks_for(F, 256));
    hipLaunchKernelGGL(k_bounds_partial, dim3(nb), dim3(256), 0, st, b.centre, F, b.partial);
    CCD_LAUNCH_CHECK(ctx);
    double *box = b.partial + 6 * NPARTS;
    hipLaunchKernelGGL(k_bounds_final, dim3(1), dim3(256), 0, st, b.partial, nb, box);
    CCD_LAUNCH_CHECK(ctx);
    if (batched) {
        hipLaunchKernelGGL(k_face_instance, dim3(blocks_for(F, 256)), dim3(256), 0, st, inst_off, ninst, F,
                           b.face_inst);
        CCD_LAUNCH_CHECK(ctx);
    }
    const int axis_bits = ccd::morton_axis_bits(inst_bits), sort_bits = inst_bits + 3 * axis_bits;
    hipLaunchKernelGGL(k_morton, dim3(blocks_for(F, 256)), dim3(256), 0, st, b.centre, F, box,
                       batched ? b.face_inst : (const int32_t *)nullptr, axis_bits, b.keys, b.vals);
    CCD_LAUNCH_CHECK(ctx);
    prof_end(ctx, CCD_T_BOUNDS);

    prof_begin(ctx, CCD_T_SORT);
    bool in_alt = false;
    rc = radix_sort_pairs(ctx, b.keys, b.vals, b.keys2, b.order, F, sort_bits, b.sort_tmp, in_alt);
    if (rc) return rc;
    const int32_t *order = in_alt ? b.order : b.vals;
    ctx->tree_order = order;
    prof_end(ctx, CCD_T_SORT);

    prof_begin(ctx, CCD_T_BUILD);
    rc = launch_qrange(ctx, b, F);
    if (rc) return rc;
    rc = launch_boxes(ctx, b, order, faces, F);
    if (rc) return rc;
    prof_end(ctx, CCD_T_BUILD);

    prof_begin(ctx, CCD_T_TABLES);
    rc = build_vertex_face_table(ctx, faces, F, V);
    if (rc) return rc;
    const int32_t *voff = nullptr, *vlist = nullptr;
    vertex_face_table(ctx, &voff, &vlist);
    hipLaunchKernelGGL(k_mesh_check, dim3(blocks_for(F, 256)), dim3(256), 0, st, faces, F, voff, vlist, c + C_BAD);
    CCD_LAUNCH_CHECK(ctx);
    hipLaunchKernelGGL(k_edges, dim3(blocks_for(3 * F, 256)), dim3(256), 0, st, b.sfaces, F, faces, voff, vlist, b.rank,
                       b.edges);
    CCD_LAUNCH_CHECK(ctx);
    prof_end(ctx, CCD_T_TABLES);

    prof_begin(ctx, CCD_T_TRAVERSE);
    rc = launch_rows(ctx, b, F, inst_off);
    if (rc) return rc;
    prof_end(ctx, CCD_T_TRAVERSE);

    prof_begin(ctx, CCD_T_EXPAND);
    rc = launch_expand(ctx, b, faces, F, V, voff, vlist, fixed);
    if (rc) return rc;
    prof_end(ctx, CCD_T_EXPAND);
    return CCD_OK;
}

// Refit: the sorted order of the last full build on this context (same faces, same instance layout) with
// new positions -- new leaf bounds and records; the Morton order and the vertex->face table are kept.
// Candidate sets do not depend on the order, so this is exact; only culling efficiency depends on how
// far the mesh moved since the build.
int broadphase_refit_launch(ccd_ctx *ctx, const int32_t *faces, int64_t F, const double *qs, const double *qe,
                            int64_t V, double eta, const uint8_t *fixed, const int64_t *inst_off, int ninst)
{
    hipStream_t st = ctx->stream;
    int64_t *cnt = ctx->d_counts;
    int rc = fill_u64(ctx, (uint64_t *)cnt, NCOUNTERS, 0);
    if (rc) return rc;
    if (F < 2) return CCD_OK;
    const bool batched = inst_off && ninst > 1;
    BPBufs b;
    rc = bp_buffers(ctx, F, V, batched, b);
    if (rc) return rc;
    static const Axes axes = make_axes();
    prof_begin(ctx, CCD_T_BOUNDS);
    hipLaunchKernelGGL(k_leaf_bounds, dim3(blocks_for(F, 256)), dim3(256), 0, st, faces, F, qs, qe,
                       (const int64_t *)nullptr, (const double *)nullptr, eta, axes, 0, b.dop64, b.centre);
    CCD_LAUNCH_CHECK(ctx);
    prof_end(ctx, CCD_T_BOUNDS);
    prof_begin(ctx, CCD_T_BUILD);
    rc = launch_qrange(ctx, b, F);
    if (rc) return rc;
    rc = launch_boxes(ctx, b, ctx->tree_order, faces, F);
    if (rc) return rc;
    prof_end(ctx, CCD_T_BUILD);
    const int32_t *voff = nullptr, *vlist = nullptr;
    vertex_face_table(ctx, &voff, &vlist);
    prof_begin(ctx, CCD_T_TRAVERSE);
    rc = launch_rows(ctx, b, F, inst_off);
    if (rc) return rc;
    prof_end(ctx, CCD_T_TRAVERSE);
    prof_begin(ctx, CCD_T_EXPAND);
    rc = launch_expand(ctx, b, faces, F, V, voff, vlist, fixed);
    if (rc) return rc;
    prof_end(ctx, CCD_T_EXPAND);
    return CCD_OK;
}

int broadphase(ccd_ctx *ctx, const int32_t *faces, int64_t F, const double *qs, const double *qe,
               const int64_t *hist_off, const double *hist_pos, int64_t V, double eta, const uint8_t *fixed,
               Candidates &out, bool aabb, const int64_t *inst_off, int ninst)
{
    out = Candidates();
    hipStream_t st = ctx->stream;
    int rc = broadphase_prepare(ctx, F, V, inst_off && ninst > 1);
    if (rc) return rc;
    for (int attempt = 0; attempt < 3; attempt++) {
        rc = broadphase_launch(ctx, faces, F, qs, qe, hist_off, hist_pos, V, eta, fixed, aabb, inst_off, ninst);
        if (rc) return rc;
        CCD_HIP_CHECK(ctx, hipMemcpyAsync(ctx->h_counts, ctx->d_counts, sizeof(int64_t) * NCOUNTERS,
                                          hipMemcpyDeviceToHost, st));
        CCD_HIP_CHECK(ctx, hipStreamSynchronize(st));
        int64_t P = ctx->h_counts[C_ROWS], nv = ctx->h_counts[C_VF], ne = ctx->h_counts[C_EE];
        if (P <= ctx->cap_rows && nv <= ctx->cap_vf && ne <= ctx->cap_ee) break;
        // Too small: grow to the counts seen (the stencil counts are exact only once the rows fit).
        ctx->cap_rows = std::max(ctx->cap_rows, P + P / 8 + 1024);
        ctx->cap_vf = std::max(ctx->cap_vf, nv + nv / 8 + 1024);
        ctx->cap_ee = std::max(ctx->cap_ee, ne + ne / 8 + 1024);
        rc = broadphase_prepare(ctx, F, V, inst_off && ninst > 1);
        if (rc) return rc;
        if (attempt == 2) return set_error(ctx, CCD_E_CAPACITY, "broadphase buffers did not converge");
    }
    out.nvf = ctx->h_counts[C_VF];
    out.nee = ctx->h_counts[C_EE];
    out.vf = (int32_t *)ctx->bufs["vf_keys"].ptr;
    out.ee = (int32_t *)ctx->bufs["ee_keys"].ptr;
    out.vf_cap = ctx->cap_vf;
    out.ee_cap = ctx->cap_ee;
    if (F >= 2 && ctx->h_counts[C_BAD] != 0) {   // raw emission: deduplicate by sorting
        int64_t *cnt = ctx->d_counts;
        rc = sort_unique(ctx, out.vf, out.nvf, "vf", cnt + C_VF);
        if (rc) return rc;
        rc = sort_unique(ctx, out.ee, out.nee, "ee", cnt + C_EE);
        if (rc) return rc;
        CCD_HIP_CHECK(ctx, hipMemcpyAsync(ctx->h_counts, cnt, sizeof(int64_t) * NCOUNTERS, hipMemcpyDeviceToHost, st));
        CCD_HIP_CHECK(ctx, hipStreamSynchronize(st));
        out.nvf = ctx->h_counts[C_VF];
        out.nee = ctx->h_counts[C_EE];
    }
    return CCD_OK;
}

}   // namespace ccdi
