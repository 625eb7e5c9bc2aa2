// The screening narrowphase of two-entry histories: screen every stencil, refine what the screen left open, solve
// what the refinement left open.
#include "narrow_common.h"
#include <algorithm>

namespace {

using ccdi::NarrowOut;

// Three passes, each a launch:
//   1. k_screen: ccd::screen_vf_window / screen_ee_window on every stencil, straight-line FP64 without a
//      solver, a division or a branch, so all 64 lanes work all the time.
//   2. k_refine: ccd::refine_primary / refine_others (loops over parts of [0, 1], no solver) on the stencils
//      whose screen left sub-tests open.
//   3. k_solve: the sub-tests still open, by the cascade's own functions.
// The results are the cascade's own (ccd_core.h has the argument).  The cascade loops differently in every
// lane (23-53% of an issued instruction's lanes worked when it ran on all stencils, and that took 90% of
// the time), so what counts is to run it on few, gathered into full wavefronts.
//
// The stencils are split into regions of consecutive ones, one wavefront's work in each pass.  A region has
// its own two lists of open stencils, as long as the region: A those whose face or edge-edge test is open, B
// those with vertex-edge or vertex-vertex tests open (with a mask of them); a stencil may be in both.  So no
// counter is shared: with one list and one queue counter per pass, claims on the counters (about 10 ns each,
// one after another) were most of the time of small launches.  Lists A and B of a region are refined and
// solved by different wavefronts, whose lanes then run the same code.
// In B a hit counts only if the face or edge-edge test, which comes first, does not hit: where that was open
// too (the mask's bit says so) the lane runs it again, which happens only for the few stencils whose
// later tests hit.
//
// Region length: consecutive stencils share vertices, and a region's come from the L1 of one compute unit
// (54M edge-edge stencils of 128 instances are screened in 11.7 ms by 64-stencil pieces handed to whichever
// wavefront is free, in 2.4 ms by 1024-stencil ones), but small launches need all the wavefronts they can
// get; at most 65536 regions keep an offset within one below 2^16.
struct OpenLists {
    int32_t *count;       // [2 * regions]: entries of A, then of B
    uint16_t *a, *b;      // offsets within the region
    uint8_t *mask;        // of B's entries
    int regions;
};

// The regions' common length for n stencils, and this wavefront's region: block index modulo 8 is the XCD, so
// each XCD gets consecutive regions.
__device__ __forceinline__ int region_length(int64_t n, int regions)
{
    return (int)(((n + regions - 1) / regions + 63) & ~(int64_t)63);
}
__device__ __forceinline__ int region_of(int block, int regions) { return (block & 7) * (regions >> 3) + (block >> 3); }

// Where the stencils' windows come from.  at(i) gives the i-th stencil's vertices by their place in it, a
// runtime index: read again, since selecting from arrays of positions would keep those in scratch memory.
// extent: a region's first stencil and its length.
struct KeyedWindows {   // two-entry histories, by the vertices' numbers
    const double *__restrict__ qs, *__restrict__ qe;
    const int4 *__restrict__ keys;
    const int64_t *__restrict__ n_dev;   // may exceed n_max: an overflowing broadphase counts every stencil
    int64_t n_max;
    struct At {
        const double *qs, *qe;
        int4 k;
        __device__ __forceinline__ void operator()(int w, V3 &x, V3 &y) const
        {
            window_pos(qs, qe, w == 0 ? k.x : (w == 1 ? k.y : (w == 2 ? k.z : k.w)), x, y);
        }
    };
    __device__ __forceinline__ At at(int64_t i) const { return At{qs, qe, keys[i]}; }
    __device__ __forceinline__ int4 key(int64_t i) const { return keys[i]; }
    __device__ __forceinline__ int extent(int r, int regions, int64_t &begin) const
    {
        const int64_t n = n_dev && *n_dev < n_max ? *n_dev : n_max;
        const int len = region_length(n, regions);
        begin = (int64_t)r * len;
        return (int)(begin < n ? (n - begin < len ? n - begin : len) : 0);
    }
};
struct PooledWindows {   // a pool of windows with their positions: eight vertices each, four at the start, four at the end
    ccdi::WindowPool pool;
    struct At {
        const double *p;
        __device__ __forceinline__ void operator()(int w, V3 &x, V3 &y) const
        {
            x = ccd::mk(p[3 * w], p[3 * w + 1], p[3 * w + 2]);
            y = ccd::mk(p[12 + 3 * w], p[13 + 3 * w], p[14 + 3 * w]);
        }
    };
    __device__ __forceinline__ At at(int64_t i) const { return At{pool.pos + 24 * i}; }
    __device__ __forceinline__ int4 key(int64_t) const { return make_int4(0, 0, 0, 0); }
    __device__ __forceinline__ int extent(int r, int, int64_t &begin) const
    {
        begin = (int64_t)r * 64;
        const int64_t shard = begin / pool.per_shard, left = pool.filled(shard) - (begin - shard * pool.per_shard);
        return (int)(left < 0 ? 0 : (left < 64 ? left : 64));
    }
};
template <class At>
__device__ __forceinline__ void load_window(const At &at, V3 *s, V3 *e)
{
#pragma unroll
    for (int q = 0; q < 4; q++) at(q, s[q], e[q]);
}
template <bool PER_STENCIL>
__device__ __forceinline__ void store_result(const NarrowOut &o, int64_t i, int r, double t)
{
    if (PER_STENCIL) {
        o.hit[i] = r >= 0 ? 1 : 0;
        if (o.t) o.t[i] = r >= 0 ? t : 0.0;
        if (o.sub) o.sub[i] = r >= 0 ? (uint8_t)r : (uint8_t)255;
    }
}
__device__ __forceinline__ int rank_in(uint64_t mask) { return __popcll(mask & ((1ull << __lane_id()) - 1ull)); }

// Without a solver the registers would allow three wavefronts per SIMD as well as two; the kernel is bound by
// its FP64 instructions (about 1,270 for an edge-edge stencil).
template <bool VF, bool PER_STENCIL, class Windows>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3))) void k_screen(
    Windows windows, double eta, NarrowOut o, OpenLists l)
{
    const int lane = __lane_id();
    const int r = region_of(blockIdx.x, l.regions);
    int64_t begin;
    const int cnt = windows.extent(r, l.regions, begin);
    int na = 0, nb = 0;
    for (int j0 = 0; j0 < cnt; j0 += 64) {
        const int j = j0 + lane;
        unsigned m = 0;
        if (j < cnt) {
            const int64_t i = begin + j;
            V3 s[4], e[4];
            load_window(windows.at(i), s, e);
            const double et = PER_STENCIL && o.eta ? o.eta[i] : eta;
            m = VF ? ccd::screen_vf_window(s, e, et) : ccd::screen_ee_window(s, e, et);
            store_result<PER_STENCIL>(o, i, -1, 0.0);   // a hit found later replaces it
        }
        const bool in_a = (m & ccd::SCREEN_PRIMARY) != 0, in_b = (m & ~ccd::SCREEN_PRIMARY) != 0;
        const uint64_t ba = __ballot(in_a), bb = __ballot(in_b);
        if (in_a) l.a[begin + na + rank_in(ba)] = (uint16_t)j;
        if (in_b) {
            l.b[begin + nb + rank_in(bb)] = (uint16_t)j;
            l.mask[begin + nb + rank_in(bb)] = (uint8_t)m;
        }
        na += __popcll(ba);
        nb += __popcll(bb);
    }
    if (lane == 0) {
        l.count[r] = na;
        l.count[l.regions + r] = nb;
    }
}

// A list of more than two chunks is refined with few parts first, since many stencils need no more (of 200^2
// cloth stencils 4 parts clear 40-48%, 16 clear 66-86%; the rest costs 16 parts besides): edge-edge and
// vertex-face 1240 + 490 -> 1034 + 385 us on a 256^2 cloth, 78.6 + 26.6 -> 64.3 + 19.8 ms on a 1024^2 sheet.
// More than 16 would clear 6-14% of what is left of the edge-edge stencils at a fifth of a solve's cost each.
constexpr int COARSE_FROM = 128, COARSE_LEAVES = 4;
// One wavefront per region and list; a list is compacted in place (an entry moves only to where entries
// were read before).
template <bool VF, bool PER_STENCIL, class Windows>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void k_refine(
    Windows windows, double eta, NarrowOut o, OpenLists l)
{
    const int lane = __lane_id();
    const bool list_b = (int)blockIdx.x >= l.regions;
    const int r = region_of(list_b ? blockIdx.x - l.regions : blockIdx.x, l.regions);
    int64_t begin;
    windows.extent(r, l.regions, begin);
    int32_t *count = l.count + (list_b ? l.regions : 0) + r;
    int cnt = *count;
    if (cnt == 0) return;
    uint16_t *list = list_b ? l.b : l.a;
    int kept = 0;
    for (int leaves = cnt > COARSE_FROM ? COARSE_LEAVES : ccd::REFINE_LEAVES;; leaves = ccd::REFINE_LEAVES) {
        kept = 0;
        for (int j0 = 0; j0 < cnt; j0 += 64) {
            const int j = j0 + lane;
            bool open = false;
            uint16_t off = 0;
            unsigned m = 0;
            if (j < cnt) {
                off = list[begin + j];
                const int64_t i = begin + off;
                const auto at = windows.at(i);
                const double et = PER_STENCIL && o.eta ? o.eta[i] : eta;
                V3 s[4], e[4];
                load_window(at, s, e);
                if (list_b) {
                    m = l.mask[begin + j];
                    m = ccd::refine_others<VF>(s, e, et, m, at, leaves);
                    open = (m & ~ccd::SCREEN_PRIMARY) != 0;
                } else {
                    open = ccd::refine_primary<VF>(s, e, et, ccd::SCREEN_PRIMARY, leaves) != 0;
                }
            }
            const uint64_t b = __ballot(open);
            if (open) {
                list[begin + kept + rank_in(b)] = off;
                if (list_b) l.mask[begin + kept + rank_in(b)] = (uint8_t)m;
            }
            kept += __popcll(b);
        }
        if (leaves == ccd::REFINE_LEAVES) break;
        cnt = kept;
        __threadfence_block();   // other lanes read what these wrote
    }
    if (lane == 0) *count = kept;
}

// Three wavefronts per SIMD: 168 registers, 20 to 256 bytes a lane spilled (two: up to 231 registers, up to 48
// bytes).  The root solves are chains of dependent FP64 operations, and a third wavefront hides more of their latency
// than the spills cost: edge-edge 1.61 ms against 1.82 on 128 instances, 1.61 against 1.71 on a 256^2 cloth, 78 against
// 91 on a 1024^2 sheet; lists too short to fill the chip take up to 10 us longer (12 small instances 88 against 80 us).
template <bool VF, bool PER_STENCIL, class Windows>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3))) void k_solve(
    Windows windows, double eta, NarrowOut o, OpenLists l)
{
    const int lane = __lane_id();
    const bool list_b = (int)blockIdx.x >= l.regions;
    const int r = region_of(list_b ? blockIdx.x - l.regions : blockIdx.x, l.regions);
    int64_t begin;
    windows.extent(r, l.regions, begin);
    const int cnt = l.count[(list_b ? l.regions : 0) + r];
    for (int j0 = 0; j0 < cnt; j0 += 64) {
        const int j = j0 + lane;
        int4 k = make_int4(0, 0, 0, 0);
        double t = 0.0;
        int sub = -1;
        if (j < cnt) {
            const int64_t i = begin + (list_b ? l.b : l.a)[begin + j];
            k = windows.key(i);
            const auto at = windows.at(i);
            const double et = PER_STENCIL && o.eta ? o.eta[i] : eta;
            unsigned m = list_b ? l.mask[begin + j] : ccd::SCREEN_PRIMARY;
            const bool also_a = list_b && (m & ccd::SCREEN_PRIMARY);
            bool again = false;
            // List B's hits with an open first test come round a second time for that test.
            do {
                double tt = 0.0;
                int found = -1;
                if (again || !list_b) {
                    V3 s[4], e[4];
                    load_window(at, s, e);
                    found = ccd::check_masked<VF>(s, e, et, tt, ccd::SCREEN_PRIMARY, at, ccd::NoCount());
                } else {
                    found = ccd::check_others<VF>(et, tt, m, at, ccd::NoCount());
                }
                if (again) {
                    if (found >= 0) sub = -1;   // list A reports it
                    break;
                }
                sub = found;
                t = tt;
                again = also_a && sub >= 0;
            } while (again);
            if (sub >= 0) store_result<PER_STENCIL>(o, i, sub, t);
        }
        if (!PER_STENCIL) append_hits(sub >= 0, k, t, o.out_keys, o.out_toi, o.cap, o.counter);
    }
}

// Regions for up to n stencils (n < 2^31): see above.  A multiple of 8, for the XCDs.
constexpr int64_t MAX_REGIONS = 65536, MAX_REGION_TILE = 4096;
int64_t region_max_length(int64_t n, int64_t tile)
{
    tile = std::min(tile, MAX_REGION_TILE);
    const int64_t len = std::max((n + MAX_REGIONS - 1) / MAX_REGIONS, std::min(tile, n / 4096));
    return std::max<int64_t>(64, (len + 63) / 64 * 64);
}

}   // namespace

namespace ccdi {

int64_t open_list_bytes(int64_t n)
{
    // Two counts per region; per slot two offsets and a mask; the slots of the last region and of up to
    // seven empty ones.
    return 8 * (MAX_REGIONS + 8) + 5 * (n + 9 * region_max_length(n, MAX_REGION_TILE)) + 64;
}

void *open_list(ccd_ctx *ctx, int64_t n)
{
    if (n <= 0 || n > 0x7fffffffll) return nullptr;   // one pass instead (the same results)
    return buffer(ctx, "open_list", (size_t)open_list_bytes(n));
}

template <bool VF, bool PER_STENCIL, class Windows>
static int launch_passes(ccd_ctx *ctx, const Windows &w, double eta, const NarrowOut &o, int64_t len, int regions, void *list)
{
    OpenLists l;
    l.regions = regions;
    const int64_t cap = regions * len;
    l.count = (int32_t *)list;
    l.a = (uint16_t *)(l.count + 2 * (MAX_REGIONS + 8));
    l.b = l.a + cap;
    l.mask = (uint8_t *)(l.b + cap);
    const dim3 one((unsigned)regions), both((unsigned)(2 * regions)), wave(64);
    hipLaunchKernelGGL((k_screen<VF, PER_STENCIL, Windows>), one, wave, 0, ctx->stream, w, eta, o, l);
    CCD_LAUNCH_CHECK(ctx);
    hipLaunchKernelGGL((k_refine<VF, PER_STENCIL, Windows>), both, wave, 0, ctx->stream, w, eta, o, l);
    CCD_LAUNCH_CHECK(ctx);
    hipLaunchKernelGGL((k_solve<VF, PER_STENCIL, Windows>), both, wave, 0, ctx->stream, w, eta, o, l);
    CCD_LAUNCH_CHECK(ctx);
    return CCD_OK;
}

int launch_screened(ccd_ctx *ctx, bool vf, bool per_stencil, const double *qs, const double *qe, const int32_t *keys,
                    const int64_t *n_dev, int64_t n, double eta, const NarrowOut &o, int tile, void *list)
{
    const KeyedWindows w{qs, qe, (const int4 *)keys, n_dev, n};
    const int64_t len = region_max_length(n, tile);
    const int regions = (int)(((n + len - 1) / len + 7) / 8 * 8);
    auto f = vf ? (per_stencil ? launch_passes<true, true, KeyedWindows> : launch_passes<true, false, KeyedWindows>)
                : (per_stencil ? launch_passes<false, true, KeyedWindows> : launch_passes<false, false, KeyedWindows>);
    return f(ctx, w, eta, o, len, regions, list);
}

// One chunk of 64 windows to a region: their positions lie side by side, so longer regions would gain nothing.
int launch_screened_pool(ccd_ctx *ctx, bool vf, const WindowPool &pool, void *list)
{
    NarrowOut o;
    o.eta = pool.eta;
    o.hit = pool.hit;
    o.t = pool.t;
    o.sub = pool.sub;
    auto f = vf ? launch_passes<true, true, PooledWindows> : launch_passes<false, true, PooledWindows>;
    return f(ctx, PooledWindows{pool}, 0.0, o, 64, (int)(WindowPool::SHARDS * pool.per_shard / 64), list);
}

}   // namespace ccdi
