// Narrowphase kernels: one lane per stencil (or per primitive item), FP64, no fused multiply-add.
//
// Layout: positions are read straight from the caller's flat double[3V] arrays (24-byte vertex
// records); stencil keys are int4 (16 bytes, one dwordx4 load per lane).  Consecutive stencils share
// vertices (the broadphase emits them face pair by face pair), so the gathers hit L2 after the first
// touch.  The work per stencil is the reference's fixed sub-test order with early exit
// (CTCDNarrowPhase.cpp:43-69, :91-132), so lanes diverge; the kernel is FP64-VALU bound.
#include "ccd_core.h"
#include <algorithm>

#include "ccd_internal.h"
#include "narrow_common.h"

namespace {

using ccd::V3;

// Every kernel here that reaches the root finder asks for two wavefronts per SIMD.  The register
// allocator otherwise gives such kernels up to 512 registers and one wavefront per SIMD, which leaves the
// FP64 pipeline idle on dependent instructions.
#define CCD_TWO_WAVES __attribute__((amdgpu_waves_per_eu(2)))

template <class M>
__global__ __launch_bounds__(256) CCD_TWO_WAVES void k_primitives(int kind, const double *__restrict__ q,
                                                    const double *__restrict__ eta, double eta_s, int64_t n,
                                                    uint8_t *__restrict__ hit, double *__restrict__ tout)
{
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    double e = eta ? eta[i] : eta_s;
    double t = 0.0;
    bool r = false;
    if (kind == CCD_PRIM_VERTEX_FACE || kind == CCD_PRIM_EDGE_EDGE) {
        const double *p = q + 24 * i;
        V3 a[8];
#pragma unroll
        for (int k = 0; k < 8; k++) a[k] = ccd::mk(p[3 * k], p[3 * k + 1], p[3 * k + 2]);
        if (kind == CCD_PRIM_VERTEX_FACE)
            r = ccd::vertex_face(a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], e, t, M());
        else
            r = ccd::edge_edge(a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], e, t, M());
    } else if (kind == CCD_PRIM_VERTEX_EDGE) {
        const double *p = q + 18 * i;
        V3 a[6];
#pragma unroll
        for (int k = 0; k < 6; k++) a[k] = ccd::mk(p[3 * k], p[3 * k + 1], p[3 * k + 2]);
        r = ccd::vertex_edge(a[0], a[1], a[2], a[3], a[4], a[5], e, t, M());
    } else {
        const double *p = q + 12 * i;
        V3 a[4];
#pragma unroll
        for (int k = 0; k < 4; k++) a[k] = ccd::mk(p[3 * k], p[3 * k + 1], p[3 * k + 2]);
        r = ccd::vertex_vertex(a[0], a[1], a[2], a[3], e, t, M());
    }
    hit[i] = r ? 1 : 0;
    if (tout) tout[i] = r ? t : 0.0;
}

// Two-entry histories: window (stitch0(start), end), CTCDNarrowPhase.cpp:24-36 with History.cpp:127-133.
template <bool VF, class M>
__device__ __forceinline__ int stencil2(const double *__restrict__ qs, const double *__restrict__ qe, int4 k,
                                        double eta, double &t)
{
    int v[4] = {k.x, k.y, k.z, k.w};
    V3 s[4], e[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        V3 a = load3(qs, v[j]);
        V3 b = load3(qe, v[j]);
        s[j] = ccd::mk(ccd::stitch0(a.x, b.x), ccd::stitch0(a.y, b.y), ccd::stitch0(a.z, b.z));
        e[j] = b;
    }
    return VF ? ccd::check_vf_window(s, e, eta, t, M()) : ccd::check_ee_window(s, e, eta, t, M());
}

template <bool VF, class M>
__global__ __launch_bounds__(256) CCD_TWO_WAVES void k_narrow2(const double *__restrict__ qs, const double *__restrict__ qe,
                                                 const int4 *__restrict__ keys, const double *__restrict__ eta,
                                                 double eta_s, int64_t n, uint8_t *__restrict__ hit,
                                                 double *__restrict__ tout, uint8_t *__restrict__ sub)
{
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    double t = 0.0;
    int r = stencil2<VF, M>(qs, qe, keys[i], eta ? eta[i] : eta_s, t);
    hit[i] = r >= 0 ? 1 : 0;
    if (tout) tout[i] = r >= 0 ? t : 0.0;
    if (sub) sub[i] = r >= 0 ? (uint8_t)r : (uint8_t)255;
}

// The whole cascade on a persistent grid, for stencil lists that the screening form (screened.hip) does not
// take (2^31 stencils and more, or switched off): each wavefront repeatedly takes the next `tile` stencils with
// one atomic on *work and tests them 64 at a time.
template <bool VF, class M>
__global__ __launch_bounds__(256) CCD_TWO_WAVES void k_narrow2_queue(
    const double *__restrict__ qs, const double *__restrict__ qe, const int4 *__restrict__ keys,
    const int64_t *__restrict__ n_dev, int64_t n_max, double eta, int4 *__restrict__ out_keys,
    double *__restrict__ out_toi, int64_t cap, unsigned long long *counter, unsigned long long *work, int tile)
{
    // Clamp to the stored keys: an overflowing broadphase counts more stencils than it stores.
    const int64_t n = *n_dev < n_max ? *n_dev : n_max;
    const int lane = __lane_id();
    while (true) {
        unsigned long long start = 0;
        if (lane == 0) start = atomicAdd(work, (unsigned long long)tile);
        start = __shfl(start, 0);
        if ((int64_t)start >= n) break;
        const int64_t end = (int64_t)start + tile < n ? (int64_t)start + tile : n;
        for (int64_t j0 = (int64_t)start; j0 < end; j0 += 64) {
            const int64_t i = j0 + lane;
            bool hit = false;
            double t = 0.0;
            int4 k = make_int4(0, 0, 0, 0);
            if (i < end) {
                k = keys[i];
                hit = stencil2<VF, M>(qs, qe, k, eta, t) >= 0;
            }
            append_hits(hit, k, t, out_keys, out_toi, cap, counter);
        }
    }
}

__global__ void k_validate_keys(const int32_t *__restrict__ keys, int64_t n4, int64_t nverts,
                                unsigned long long *bad)
{
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    bool b = false;
    if (i < n4) {
        int32_t v = keys[i];
        b = v < 0 || v >= nverts;
    }
    uint64_t m = __ballot(b);
    if (m && __lane_id() == __ffsll((unsigned long long)m) - 1) atomicAdd(bad, (unsigned long long)__popcll(m));
}

// A history is valid when off[] is nondecreasing within [0, nentries], each vertex has at least
// one entry, its times start at 0, end at 1 and never decrease.
__global__ void k_validate_history(const int64_t *__restrict__ off, const double *__restrict__ ht, int64_t nverts,
                                   int64_t nentries, unsigned long long *bad)
{
    int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    bool b = false;
    if (v < nverts) {
        int64_t a = off[v], z = off[v + 1];
        if (a < 0 || z > nentries || z <= a) {
            b = true;
        } else {
            if (ht[a] != 0.0 || ht[z - 1] != 1.0) b = true;
            for (int64_t e = a + 1; e < z && !b; e++)
                if (!(ht[e] >= ht[e - 1])) b = true;
        }
    }
    uint64_t m = __ballot(b);
    if (m && __lane_id() == __ffsll((unsigned long long)m) - 1) atomicAdd(bad, (unsigned long long)__popcll(m));
}

// History::computeMinimumGap (History.cpp:78-93): min(1, every gap between consecutive entry times),
// reduced with an atomic min on the bit pattern (the gaps of a validated history are non-negative, so
// their bits order as the values do).  *gap_bits must hold the bits of 1.0 on entry.
__global__ __launch_bounds__(256) void k_min_gap(const int64_t *__restrict__ off, const double *__restrict__ ht,
                                                 int64_t nverts, unsigned long long *gap_bits)
{
    double g = 1.0;
    for (int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; v < nverts;
         v += (int64_t)gridDim.x * blockDim.x)
        for (int64_t j = off[v] + 1; j < off[v + 1]; j++) g = ccd::smin(ht[j] - ht[j - 1], g);
    for (int o = 32; o > 0; o >>= 1) g = ccd::smin(__shfl_xor(g, o), g);
    if (__lane_id() == 0) atomicMin(gap_bits, (unsigned long long)ccd::double_to_bits(g));
}
__global__ void k_set_bits(unsigned long long *p, unsigned long long v) { *p = v; }

inline unsigned blocks_for(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// One wavefront per block for the kernels that give each lane one stencil of very uneven cost: a wavefront's
// slot is refilled as soon as it finishes instead of when the slowest of its block's wavefronts does.
constexpr int LANE_BLOCK = 64;

}   // namespace

namespace ccdi {

// Every narrowphase launch instantiates its kernel with the product's counter type: no work
// accounting, cascades pruned once no interval combination can overlap.
#define CCD_PRODUCT_LAUNCH(LAUNCH)                                                                                  \
    do {                                                                                                            \
        using M = ccd::NoCount;                                                                                     \
        LAUNCH;                                                                                                     \
    } while (0)

int launch_primitives(ccd_ctx *ctx, int kind, const double *q, const double *eta, double eta_s, int64_t n,
                      uint8_t *hit, double *t)
{
    if (n == 0) return CCD_OK;
    CCD_PRODUCT_LAUNCH(hipLaunchKernelGGL(k_primitives<M>, dim3(blocks_for(n, LANE_BLOCK)), dim3(LANE_BLOCK), 0, ctx->stream,
                                              kind, q, eta, eta_s, n, hit, t));
    CCD_LAUNCH_CHECK(ctx);
    return CCD_OK;
}

// The per-stencil narrowphase is screened where its stencils are more than the lanes that k_narrow2 keeps resident
// (two wavefronts per SIMD: 131,072 on 256 compute units).  Below, all of them run at once, and the launch takes as long
// as its slowest lane, with or without a screen before it.  One launch against three, vertex-face / edge-edge, us:
//   256^2 cloth: 139 / 209 against 124 / 182 for 4,096 stencils, 152 / 228 against 171 / 246 for 65,536, 177 / 281 against
//     202 / 308 for 131,072, 317 / 483 against 254 / 424 for 262,144;
//   256^2 sheet: 24 / 95 against 39 / 104, 59 / 103 against 69 / 131, 67 / 132 against 95 / 181, 88 / 232 against 93 / 233.
constexpr int64_t RESIDENT_LANES_PER_CU = 4 * 2 * 64;

int launch_narrow2(ccd_ctx *ctx, bool vf, const double *qs, const double *qe, const int32_t *keys,
                   const double *eta, double eta_s, int64_t n, uint8_t *hit, double *t, uint8_t *sub, void *list)
{
    if (n == 0) return CCD_OK;
    if (n > RESIDENT_LANES_PER_CU * ctx->num_cus && n <= 0x7fffffffll) {   // (the screening form counts stencils in 31 bits)
        if (!list) list = open_list(ctx, n);
        if (!list) return CCD_E_OOM;
        NarrowOut o;
        o.eta = eta;
        o.hit = hit;
        o.t = t;
        o.sub = sub;
        return launch_screened(ctx, vf, true, qs, qe, keys, nullptr, n, eta_s, o,
                               (vf ? ctx->vf_shape : ctx->ee_shape).tile, list);
    }
    if (vf)
        CCD_PRODUCT_LAUNCH(hipLaunchKernelGGL((k_narrow2<true, M>), dim3(blocks_for(n, LANE_BLOCK)), dim3(LANE_BLOCK), 0,
                                                  ctx->stream, qs, qe, (const int4 *)keys, eta, eta_s, n, hit, t, sub));
    else
        CCD_PRODUCT_LAUNCH(hipLaunchKernelGGL((k_narrow2<false, M>), dim3(blocks_for(n, LANE_BLOCK)), dim3(LANE_BLOCK), 0,
                                                  ctx->stream, qs, qe, (const int4 *)keys, eta, eta_s, n, hit, t, sub));
    CCD_LAUNCH_CHECK(ctx);
    return CCD_OK;
}

int launch_narrow2_queue(ccd_ctx *ctx, bool vf, const double *qs, const double *qe, const int32_t *keys,
                         const int64_t *n_dev, int64_t n_max, double eta, int32_t *out_keys, double *out_toi,
                         int64_t cap, int64_t *counter, unsigned long long *work, const QueueShape &shape,
                         void *list)
{
    if (n_max == 0) return CCD_OK;
    if (list && n_max <= 0x7fffffffll) {
        NarrowOut o;
        o.out_keys = (int4 *)out_keys;
        o.out_toi = out_toi;
        o.cap = cap;
        o.counter = (unsigned long long *)counter;
        return launch_screened(ctx, vf, false, qs, qe, keys, n_dev, n_max, eta, o, shape.tile, list);
    }
    // Sixteen turns of the queue for each resident wavefront if there are so many chunks of 64: a wavefront's turns are
    // of very uneven length (87,000 edge-edge stencils by 1,024 at a time, 85 turns in all: 2.16 ms; by 64: 0.20).
    const int64_t resident = (int64_t)ctx->num_cus * shape.waves_per_cu;
    const int tile = (int)std::max<int64_t>(64, std::min<int64_t>(shape.tile, n_max / (16 * resident) / 64 * 64));
    const int64_t need = (n_max + tile - 1) / tile;
    const int64_t waves = std::max<int64_t>(1, std::min(resident, need));
    const unsigned grid = (unsigned)((waves * 64 + shape.block - 1) / shape.block);
    if (vf)
        CCD_PRODUCT_LAUNCH(hipLaunchKernelGGL((k_narrow2_queue<true, M>), dim3(grid), dim3(shape.block), 0, ctx->stream, qs,
                                              qe, (const int4 *)keys, n_dev, n_max, eta, (int4 *)out_keys, out_toi, cap,
                                              (unsigned long long *)counter, work, tile));
    else
        CCD_PRODUCT_LAUNCH(hipLaunchKernelGGL((k_narrow2_queue<false, M>), dim3(grid), dim3(shape.block), 0, ctx->stream, qs,
                                              qe, (const int4 *)keys, n_dev, n_max, eta, (int4 *)out_keys, out_toi, cap,
                                              (unsigned long long *)counter, work, tile));
    CCD_LAUNCH_CHECK(ctx);
    return CCD_OK;
}

int launch_min_gap(ccd_ctx *ctx, const int64_t *off, const double *ht, int64_t nverts, uint64_t *gap_bits)
{
    hipLaunchKernelGGL(k_set_bits, dim3(1), dim3(1), 0, ctx->stream, (unsigned long long *)gap_bits,
                       (unsigned long long)ccd::double_to_bits(1.0));
    CCD_LAUNCH_CHECK(ctx);
    if (nverts == 0) return CCD_OK;
    unsigned grid = (unsigned)std::min<int64_t>(blocks_for(nverts, 256), 4096);
    hipLaunchKernelGGL(k_min_gap, dim3(grid), dim3(256), 0, ctx->stream, off, ht, nverts,
                       (unsigned long long *)gap_bits);
    CCD_LAUNCH_CHECK(ctx);
    return CCD_OK;
}

int launch_validate_keys(ccd_ctx *ctx, const int32_t *keys, int64_t n4, int64_t nverts, int64_t *bad)
{
    if (n4 == 0) return CCD_OK;
    hipLaunchKernelGGL(k_validate_keys, dim3(blocks_for(n4, 256)), dim3(256), 0, ctx->stream, keys, n4, nverts,
                       (unsigned long long *)bad);
    CCD_LAUNCH_CHECK(ctx);
    return CCD_OK;
}

int launch_validate_history(ccd_ctx *ctx, const int64_t *off, const double *ht, int64_t nverts, int64_t nentries,
                            int64_t *bad)
{
    if (nverts == 0) return CCD_OK;
    hipLaunchKernelGGL(k_validate_history, dim3(blocks_for(nverts, 256)), dim3(256), 0, ctx->stream, off, ht,
                       nverts, nentries, (unsigned long long *)bad);
    CCD_LAUNCH_CHECK(ctx);
    return CCD_OK;
}

}   // namespace ccdi
