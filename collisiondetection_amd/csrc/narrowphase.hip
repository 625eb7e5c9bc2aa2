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

// Multi-entry histories: stitch on the fly (History.cpp:98-140) and test window by window.
template <bool VF, class M>
__global__ __launch_bounds__(256) CCD_TWO_WAVES void k_narrow_hist(const int64_t *__restrict__ off, const double *__restrict__ ht,
                                                     const double *__restrict__ hp, const int4 *__restrict__ keys,
                                                     const double *__restrict__ eta, double eta_s, int64_t n,
                                                     uint8_t *__restrict__ hit, double *__restrict__ tout,
                                                     uint8_t *__restrict__ sub, int32_t *__restrict__ win)
{
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    int4 k = keys[i];
    int v[4] = {k.x, k.y, k.z, k.w};
    double e = eta ? eta[i] : eta_s;
    int64_t its[4], ends[4];
    int64_t total = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        its[j] = off[v[j]];
        ends[j] = off[v[j] + 1];
        total += ends[j] - its[j];
    }
    V3 prev[4], cur[4];
    double curtime = 0.0;
    int w = -1;
    int r = -1;
    double t = 0.0;
    // Each pass advances curtime strictly (entries at or before it are consumed), so the number of
    // stitched entries is at most the total entry count; the bound also guards malformed input.
    for (int64_t guard = 0; guard <= total && curtime <= 1.0; guard++) {
        double newtime = __builtin_inf();
#pragma unroll
        for (int j = 0; j < 4; j++) {
            int64_t next = its[j] + 1;
            while (next != ends[j] && ht[next] <= curtime) {
                ++next;
                ++its[j];
            }
            V3 oldp = ccd::mk(hp[3 * its[j]], hp[3 * its[j] + 1], hp[3 * its[j] + 2]);
            if (next == ends[j]) {
                cur[j] = oldp;
            } else {
                V3 newp = ccd::mk(hp[3 * next], hp[3 * next + 1], hp[3 * next + 2]);
                double dt = ht[next] - ht[its[j]];
                double a = curtime - ht[its[j]];
                double b = ht[next] - curtime;
                cur[j] = ccd::mk((b * oldp.x + a * newp.x) / dt, (b * oldp.y + a * newp.y) / dt,
                                 (b * oldp.z + a * newp.z) / dt);
                newtime = ccd::smin(newtime, ht[next]);
            }
        }
        if (w >= 0) {
            r = VF ? ccd::check_vf_window(prev, cur, e, t, M()) : ccd::check_ee_window(prev, cur, e, t, M());
            if (r >= 0) break;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) prev[j] = cur[j];
        w++;
        curtime = newtime;
    }
    hit[i] = r >= 0 ? 1 : 0;
    if (tout) tout[i] = r >= 0 ? t : 0.0;
    if (sub) sub[i] = r >= 0 ? (uint8_t)r : (uint8_t)255;
    if (win) win[i] = r >= 0 ? w : -1;
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

// SeparatingPlaneNarrowPhase (SeparatingPlaneNarrowPhase.cpp:9-278): one lane per stencil, status 1
// (collision), 0 (none) or 2 (undecided: the reference's recursion would not end; counted in *undecided).
template <bool VF, class M>
__global__ __launch_bounds__(256) CCD_TWO_WAVES void k_separating_plane(
    const int64_t *__restrict__ off, const double *__restrict__ ht, const double *__restrict__ hp,
    const int4 *__restrict__ keys, const double *__restrict__ eta, double eta_s, int64_t n,
    const unsigned long long *__restrict__ gap_bits, uint8_t *__restrict__ status, unsigned long long *undecided,
    const int32_t *__restrict__ order)
{
    const int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    int r = 0;
    if (j < n) {
        const int64_t i = order ? (int64_t)order[j] : j;   // lane j runs stencil order[j]
        const double eps = ccd::bits_to_double((long long)*gap_bits) / 4.0;
        int4 k = keys[i];
        int v[4] = {k.x, k.y, k.z, k.w};
        ccd::HistCSR h{off, ht, hp};
        r = ccd::separating_plane_check<VF>(h, v, eta ? eta[i] : eta_s, eps, M());
        status[i] = (uint8_t)r;
    }
    uint64_t m = __ballot(r == 2);
    if (m && __lane_id() == __ffsll((unsigned long long)m) - 1) atomicAdd(undecided, (unsigned long long)__popcll(m));
}

// Sort key for the separating-plane narrowphase: 1 if a stencil's root interval [0, 1] does not decide
// it (its recursion goes on; with two-entry histories that means one or two CTCD window tests), else 0.
// Most stencils are decided at the root; grouping the others keeps a wavefront's lanes on the same path.
template <bool VF>
__global__ __launch_bounds__(256) void k_sp_order_key(const int64_t *__restrict__ off, const double *__restrict__ ht,
                                                      const double *__restrict__ hp, const int4 *__restrict__ keys,
                                                      const double *__restrict__ eta, double eta_s, int64_t n,
                                                      const unsigned long long *__restrict__ gap_bits,
                                                      uint64_t *__restrict__ key, int32_t *__restrict__ idx)
{
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double eps = ccd::bits_to_double((long long)*gap_bits) / 4.0;
    const int4 k = keys[i];
    const int v[4] = {k.x, k.y, k.z, k.w};
    ccd::HistCSR h{off, ht, hp};
    const int r = ccd::separating_plane_check<VF>(h, v, eta ? eta[i] : eta_s, eps, ccd::FullCascade(), ccd::SeqScan(), 1);
    key[i] = r == 3 ? 1u : 0u;
    idx[i] = (int32_t)i;
}

// The narrowphase over stitched history windows (k_narrow_hist) with one wavefront per stencil, for
// long histories.  The stitching (History.cpp:98-140) is a merge of the four vertices' timelines; every
// lane runs the same merge (uniform control flow, identical values) 65 steps at a time and keeps the
// stitched positions of two consecutive steps, so lane l holds window W0 + l of a 64-window chunk and
// tests it.  The first window in order that collides (the lowest set bit of a ballot, in the first
// chunk with any) gives the answer, as the sequential loop's early exit does.
template <bool VF, class M>
__global__ __launch_bounds__(64) CCD_TWO_WAVES void k_narrow_hist_wave(
    const int64_t *__restrict__ off, const double *__restrict__ ht, const double *__restrict__ hp,
    const int4 *__restrict__ keys, const double *__restrict__ eta, double eta_s, int64_t n, uint8_t *__restrict__ hit,
    double *__restrict__ tout, uint8_t *__restrict__ sub, int32_t *__restrict__ win)
{
    using ccd::V3;
    const int64_t i = blockIdx.x;
    if (i >= n) return;
    const int lane = (int)__lane_id();
    const int4 k = keys[i];
    const int v[4] = {k.x, k.y, k.z, k.w};
    const double e = eta ? eta[i] : eta_s;
    int64_t its[4], ends[4];
    int64_t total = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        its[j] = off[v[j]];
        ends[j] = off[v[j] + 1];
        total += ends[j] - its[j];
    }
    double curtime = 0.0;
    int64_t g = 0;   // step index of the sequential loop (its guard); cur is evaluated at curtime
    int r = -1, w = -1;
    double t = 0.0;
    bool alive = true;
    while (alive) {
        const int64_t w0 = g;   // this chunk: windows w0 .. w0 + 63, window w = (step w, step w + 1)
        V3 pa[4], pb[4];
        bool va = false, vb = false;
        for (int s = 0; s <= 64; s++) {
            alive = g <= total && curtime <= 1.0;
            if (!alive) break;
            V3 cur[4];
            double newtime = __builtin_inf();
#pragma unroll
            for (int j = 0; j < 4; j++) {
                int64_t next = its[j] + 1;
                while (next != ends[j] && ht[next] <= curtime) {
                    ++next;
                    ++its[j];
                }
                V3 oldp = ccd::mk(hp[3 * its[j]], hp[3 * its[j] + 1], hp[3 * its[j] + 2]);
                if (next == ends[j]) {
                    cur[j] = oldp;
                } else {
                    V3 newp = ccd::mk(hp[3 * next], hp[3 * next + 1], hp[3 * next + 2]);
                    double dt = ht[next] - ht[its[j]];
                    double a = curtime - ht[its[j]];
                    double b = ht[next] - curtime;
                    cur[j] = ccd::mk((b * oldp.x + a * newp.x) / dt, (b * oldp.y + a * newp.y) / dt,
                                     (b * oldp.z + a * newp.z) / dt);
                    newtime = ccd::smin(newtime, ht[next]);
                }
            }
            if (s == lane) {
#pragma unroll
                for (int j = 0; j < 4; j++) pa[j] = cur[j];
                va = true;
            }
            if (s == lane + 1) {
#pragma unroll
                for (int j = 0; j < 4; j++) pb[j] = cur[j];
                vb = true;
            }
            if (s == 64) break;   // the next chunk starts by evaluating this step again (idempotent)
            curtime = newtime;
            g++;
        }
        bool h = false;
        int rl = -1;
        double tl = 0.0;
        if (va && vb) {
            rl = VF ? ccd::check_vf_window(pa, pb, e, tl, M()) : ccd::check_ee_window(pa, pb, e, tl, M());
            h = rl >= 0;
        }
        const unsigned long long m = __ballot(h);
        if (m) {
            const int f = __ffsll(m) - 1;
            r = __shfl(rl, f);
            t = __shfl(tl, f);
            w = (int)(w0 + f);
            break;
        }
    }
    if (lane == 0) {
        hit[i] = r >= 0 ? 1 : 0;
        if (tout) tout[i] = r >= 0 ? t : 0.0;
        if (sub) sub[i] = r >= 0 ? (uint8_t)r : (uint8_t)255;
        if (win) win[i] = r >= 0 ? w : -1;
    }
}

// The trajectory scan of planeTrajectoryIntersect (SeparatingPlaneNarrowPhase.cpp:216-265) split over
// the 64 lanes of a wavefront that all run the same stencil: each lane tests one history segment of a
// 64-segment chunk, and the first segment in scan order that meets the plane (the lowest lane whose
// test passes, in the first chunk with any) gives the result, computed by that lane with the
// sequential scan's own expressions.  Needs the whole wavefront active and on the same call.
struct WaveScan {
    __device__ double operator()(const ccd::HistCSR &h, int v, int start, bool forward, ccd::V3 ppos, ccd::V3 pvel,
                                 ccd::V3 nrm, ccd::V3 ptstart, double tstart, double eta) const
    {
        using ccd::V3;
        const double inf = ccd::bits_to_double(0x7ff0000000000000ll);
        const int64_t b = h.off[v];
        const int n = (int)(h.off[v + 1] - b);
        const double dt = forward ? h.t[b + start] - tstart : tstart - h.t[b + start];
        const double t = ccd::plane_intersect(ppos, (forward ? 1.0 : -1.0) * pvel, nrm, ptstart,
                                              ccd::hist_pos(h, b + start), dt, eta);
        if (t >= 0 && t <= dt) return t;
        const int lane = (int)__lane_id();
        if (forward) {
            // segments (i, i + 1) for i = start .. n - 2, in increasing i
            for (int base = start; base < n - 1; base += 64) {
                const int i = base + lane;
                bool hit = false;
                double r = 0.0;
                if (i < n - 1) {
                    V3 npp = ppos + (h.t[b + i] - tstart) * pvel;
                    double d = h.t[b + i + 1] - h.t[b + i];
                    double u = ccd::plane_intersect(npp, pvel, nrm, ccd::hist_pos(h, b + i), ccd::hist_pos(h, b + i + 1),
                                                    d, eta);
                    hit = u >= 0 && u <= d;
                    r = h.t[b + i] + u - tstart;
                }
                const unsigned long long m = __ballot(hit);
                if (m) return __shfl(r, __ffsll(m) - 1);
            }
        } else {
            // segments (i, i - 1) for i = start .. 1, in decreasing i
            for (int base = start; base >= 1; base -= 64) {
                const int i = base - lane;
                bool hit = false;
                double r = 0.0;
                if (i >= 1) {
                    V3 npp = ppos - (tstart - h.t[b + i]) * pvel;
                    double d = h.t[b + i] - h.t[b + i - 1];
                    double u = ccd::plane_intersect(npp, -1.0 * pvel, nrm, ccd::hist_pos(h, b + i),
                                                    ccd::hist_pos(h, b + i - 1), d, eta);
                    hit = u >= 0 && u <= d;
                    r = tstart - (h.t[b + i] - u);
                }
                const unsigned long long m = __ballot(hit);
                if (m) return __shfl(r, __ffsll(m) - 1);
            }
        }
        return inf;
    }
};

// SeparatingPlaneNarrowPhase with one wavefront per stencil, for long histories: the lanes share the
// trajectory scans (WaveScan) and otherwise compute the same values, so control flow stays uniform.
template <bool VF, class M>
__global__ __launch_bounds__(64) CCD_TWO_WAVES void k_separating_plane_wave(
    const int64_t *__restrict__ off, const double *__restrict__ ht, const double *__restrict__ hp,
    const int4 *__restrict__ keys, const double *__restrict__ eta, double eta_s, int64_t n,
    const unsigned long long *__restrict__ gap_bits, uint8_t *__restrict__ status, unsigned long long *undecided)
{
    const int64_t i = blockIdx.x;
    if (i >= n) return;
    const double eps = ccd::bits_to_double((long long)*gap_bits) / 4.0;
    const int4 k = keys[i];
    const int v[4] = {k.x, k.y, k.z, k.w};
    ccd::HistCSR h{off, ht, hp};
    const int r = ccd::separating_plane_check<VF>(h, v, eta ? eta[i] : eta_s, eps, M(), WaveScan());
    if (__lane_id() == 0) {
        status[i] = (uint8_t)r;
        if (r == 2) atomicAdd(undecided, 1ull);
    }
}

inline unsigned blocks_for(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// One wavefront per block for the kernels that give each lane one stencil of very uneven cost (the
// separating-plane recursion, the plain narrowphases): a wavefront's slot is refilled as soon as it
// finishes instead of when the slowest of its block's wavefronts does.  Separating plane on the 256^2
// cloth candidates: 92 ms with 256-thread blocks, 73 ms with 64.
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

// Stencils from which the per-stencil narrowphase is screened: below, one lane per stencil in one launch.
constexpr int64_t SCREEN_MIN = 4096;

int launch_narrow2(ccd_ctx *ctx, bool vf, const double *qs, const double *qe, const int32_t *keys,
                   const double *eta, double eta_s, int64_t n, uint8_t *hit, double *t, uint8_t *sub, void *list)
{
    if (n == 0) return CCD_OK;
    if (n >= SCREEN_MIN && n <= 0x7fffffffll) {   // (the screening form counts stencils in 31 bits)
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
    const int64_t need = (n_max + shape.tile - 1) / shape.tile;
    const int64_t waves = std::max<int64_t>(1, std::min((int64_t)ctx->num_cus * shape.waves_per_cu, need));
    const unsigned grid = (unsigned)((waves * 64 + shape.block - 1) / shape.block);
    if (vf)
        CCD_PRODUCT_LAUNCH(hipLaunchKernelGGL((k_narrow2_queue<true, M>), dim3(grid), dim3(shape.block), 0, ctx->stream, qs,
                                              qe, (const int4 *)keys, n_dev, n_max, eta, (int4 *)out_keys, out_toi, cap,
                                              (unsigned long long *)counter, work, shape.tile));
    else
        CCD_PRODUCT_LAUNCH(hipLaunchKernelGGL((k_narrow2_queue<false, M>), dim3(grid), dim3(shape.block), 0, ctx->stream, qs,
                                              qe, (const int4 *)keys, n_dev, n_max, eta, (int4 *)out_keys, out_toi, cap,
                                              (unsigned long long *)counter, work, shape.tile));
    CCD_LAUNCH_CHECK(ctx);
    return CCD_OK;
}

int launch_narrow_hist(ccd_ctx *ctx, bool vf, const int64_t *off, const double *ht, const double *hp,
                       const int32_t *keys, const double *eta, double eta_s, int64_t n, uint8_t *hit, double *t,
                       uint8_t *sub, int32_t *win, bool wave)
{
    if (n == 0) return CCD_OK;
    if (wave) {
        if (n > 0x7fffffffll) return set_error(ctx, CCD_E_INVALID, "too many stencils for one launch");
        if (vf)
            CCD_PRODUCT_LAUNCH(hipLaunchKernelGGL((k_narrow_hist_wave<true, M>), dim3((unsigned)n), dim3(64), 0,
                                                      ctx->stream, off, ht, hp, (const int4 *)keys, eta, eta_s, n, hit,
                                                      t, sub, win));
        else
            CCD_PRODUCT_LAUNCH(hipLaunchKernelGGL((k_narrow_hist_wave<false, M>), dim3((unsigned)n), dim3(64), 0,
                                                      ctx->stream, off, ht, hp, (const int4 *)keys, eta, eta_s, n, hit,
                                                      t, sub, win));
        CCD_LAUNCH_CHECK(ctx);
        return CCD_OK;
    }
    if (vf)
        CCD_PRODUCT_LAUNCH(hipLaunchKernelGGL((k_narrow_hist<true, M>), dim3(blocks_for(n, LANE_BLOCK)), dim3(LANE_BLOCK), 0,
                                                  ctx->stream, off, ht, hp, (const int4 *)keys, eta, eta_s, n, hit, t,
                                                  sub, win));
    else
        CCD_PRODUCT_LAUNCH(hipLaunchKernelGGL((k_narrow_hist<false, M>), dim3(blocks_for(n, LANE_BLOCK)), dim3(LANE_BLOCK), 0,
                                                  ctx->stream, off, ht, hp, (const int4 *)keys, eta, eta_s, n, hit, t,
                                                  sub, win));
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

int launch_separating_plane(ccd_ctx *ctx, bool vf, const int64_t *off, const double *ht, const double *hp,
                            const int32_t *keys, const double *eta, double eta_s, int64_t n, const uint64_t *gap_bits,
                            uint8_t *status, int64_t *undecided, bool wave)
{
    if (n == 0) return CCD_OK;
    auto gb = (const unsigned long long *)gap_bits;
    auto und = (unsigned long long *)undecided;
    if (wave) {
        if (n > 0x7fffffffll) return set_error(ctx, CCD_E_INVALID, "too many stencils for one launch");
        if (vf)
            CCD_PRODUCT_LAUNCH(hipLaunchKernelGGL((k_separating_plane_wave<true, M>), dim3((unsigned)n), dim3(64),
                                                      0, ctx->stream, off, ht, hp, (const int4 *)keys, eta, eta_s, n,
                                                      gb, status, und));
        else
            CCD_PRODUCT_LAUNCH(hipLaunchKernelGGL((k_separating_plane_wave<false, M>), dim3((unsigned)n),
                                                      dim3(64), 0, ctx->stream, off, ht, hp, (const int4 *)keys, eta,
                                                      eta_s, n, gb, status, und));
        CCD_LAUNCH_CHECK(ctx);
        return CCD_OK;
    }
    // Order the stencils so that those decided at the root run together (results are per stencil and
    // land at the stencil's own index, so the order changes nothing else).
    const int32_t *order = nullptr;
    if (n >= 4096 && n <= 0x7fffffffll) {   // int32 order indices
        uint64_t *key = (uint64_t *)buffer(ctx, "spo_key", (size_t)n * 8);
        uint64_t *key2 = (uint64_t *)buffer(ctx, "spo_key2", (size_t)n * 8);
        int32_t *idx = (int32_t *)buffer(ctx, "spo_idx", (size_t)n * 4);
        int32_t *idx2 = (int32_t *)buffer(ctx, "spo_idx2", (size_t)n * 4);
        void *tmp = buffer(ctx, "spo_tmp", radix_sort_temp_bytes(n));
        if (!key || !key2 || !idx || !idx2 || !tmp) return CCD_E_OOM;
        if (vf)
            hipLaunchKernelGGL(k_sp_order_key<true>, dim3(blocks_for(n, 256)), dim3(256), 0, ctx->stream, off, ht, hp,
                               (const int4 *)keys, eta, eta_s, n, gb, key, idx);
        else
            hipLaunchKernelGGL(k_sp_order_key<false>, dim3(blocks_for(n, 256)), dim3(256), 0, ctx->stream, off, ht, hp,
                               (const int4 *)keys, eta, eta_s, n, gb, key, idx);
        CCD_LAUNCH_CHECK(ctx);
        bool in_alt = false;
        int rc = radix_sort_pairs(ctx, key, idx, key2, idx2, n, 1, tmp, in_alt);   // one stable pass
        if (rc) return rc;
        order = in_alt ? idx2 : idx;
    }
    if (vf)
        CCD_PRODUCT_LAUNCH(hipLaunchKernelGGL((k_separating_plane<true, M>), dim3(blocks_for(n, LANE_BLOCK)), dim3(LANE_BLOCK),
                                                  0, ctx->stream, off, ht, hp, (const int4 *)keys, eta, eta_s, n, gb,
                                                  status, und, order));
    else
        CCD_PRODUCT_LAUNCH(hipLaunchKernelGGL((k_separating_plane<false, M>), dim3(blocks_for(n, LANE_BLOCK)), dim3(LANE_BLOCK),
                                                  0, ctx->stream, off, ht, hp, (const int4 *)keys, eta, eta_s, n, gb,
                                                  status, und, order));
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
