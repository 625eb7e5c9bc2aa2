// The narrowphases over multi-entry histories: stitched windows (History.cpp:98-140) and separating planes
// (SeparatingPlaneNarrowPhase.cpp:9-278).
//
// Both come down to the two-entry cascade on windows that depend on the stencil.  The cascade's root solver
// loops differently in every lane, and a kernel that holds it gets two wavefronts per SIMD, so no kernel here
// runs it (but for the rare stencils named below): windows that the screen (ccd::screen_vf_window /
// screen_ee_window) does not clear go with their positions to a pool, and the screening passes refine and
// solve them in full wavefronts; a last kernel puts the answers together.
// Times for 0.27M vertex-face and 0.47M edge-edge stencils over 4 entries per vertex, and for 15,000 and 26,000
// over 48, vertex-face + edge-edge:
//   stitched windows, the cascade in the lane: 0.59 + 1.59 ms, 1.00 + 1.96 ms (a wavefront a stencil); here
//     0.34 + 0.59 ms, 0.21 + 0.34 ms;
//   separating plane, the cascade in the lane: 1.38 + 1.96 ms, 2.71 + 3.23 ms (a wavefront a stencil); here
//     0.81 + 0.98 ms, 0.89 + 1.04 ms.
// A pool that is too small costs time only: the last kernel runs the stencils without room from the start, a
// wavefront each.
#include "narrow_common.h"
#include <algorithm>

namespace {

using ccdi::WindowPool;

// Room for `need` windows of each lane in the wavefront's shard: the lane's first place, or -1.  All lanes
// that are active take part.
__device__ __forceinline__ int64_t claim(const WindowPool &pool, int shard, int need)
{
    const uint64_t active = __ballot(true);
    const int lane = __lane_id(), leader = __ffsll((unsigned long long)active) - 1;
    int before = 0, all = 0;
    for (uint64_t b = active; b; b &= b - 1) {
        const int l = __ffsll((unsigned long long)b) - 1;
        const int x = __builtin_amdgcn_readlane(need, l);
        before += l < lane ? x : 0;
        all += x;
    }
    if (all == 0) return -1;
    unsigned long long base = 0;
    if (lane == leader) base = atomicAdd(&pool.claimed[shard * WindowPool::STRIDE], (unsigned long long)all);
    base = __shfl(base, leader);
    const int64_t at = (int64_t)base + before;
    if (at + need <= pool.per_shard) return shard * pool.per_shard + at;
    for (int64_t k = at; k < at + need && k < pool.per_shard; k++) pool.owner[shard * pool.per_shard + k] = -1;
    return -1;
}
__device__ __forceinline__ void store_window(const WindowPool &pool, int64_t at, int64_t owner, uint32_t place, double eta,
                                             const V3 (&s)[4], const V3 (&e)[4])
{
    double *p = pool.pos + 24 * at;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        p[3 * j] = s[j].x;
        p[3 * j + 1] = s[j].y;
        p[3 * j + 2] = s[j].z;
        p[12 + 3 * j] = e[j].x;
        p[13 + 3 * j] = e[j].y;
        p[14 + 3 * j] = e[j].z;
    }
    pool.eta[at] = eta;
    pool.owner[at] = (int32_t)owner;
    pool.place[at] = place;
}

// ------------------------------------------------------------------------------------------------
// Stitched windows
// ------------------------------------------------------------------------------------------------
// The merge of a stencil's four timelines.  at(now) gives the positions at a stitched time and the next one
// (infinity after the last); the state depends on `now` alone, so a walk may start at any stitched time.
struct Stitch {
    const double *__restrict__ ht, *__restrict__ hp;
    int64_t its[4], ends[4];
    __device__ __forceinline__ Stitch(const int64_t *__restrict__ off, const double *t, const double *p, int4 k) : ht(t), hp(p)
    {
        const int v[4] = {k.x, k.y, k.z, k.w};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            its[j] = off[v[j]];
            ends[j] = off[v[j] + 1];
        }
    }
    // The first stitched time at or after `from`; the walk starts there.
    __device__ __forceinline__ double start(double from)
    {
        double now = __builtin_inf();
#pragma unroll
        for (int j = 0; j < 4; j++) {
            int64_t lo = its[j], hi = ends[j];   // first entry at or after `from`
            while (lo < hi) {
                const int64_t mid = lo + (hi - lo) / 2;
                if (ht[mid] < from) lo = mid + 1;
                else hi = mid;
            }
            if (lo < ends[j]) now = ccd::smin(now, ht[lo]);
            if (lo > its[j]) its[j] = lo - 1;
        }
        return now;
    }
    __device__ __forceinline__ double at(double now, V3 (&cur)[4])
    {
        double newtime = __builtin_inf();
#pragma unroll
        for (int j = 0; j < 4; j++) {
            int64_t next = its[j] + 1;
            while (next != ends[j] && ht[next] <= now) {
                ++next;
                ++its[j];
            }
            V3 oldp = ccd::mk(hp[3 * its[j]], hp[3 * its[j] + 1], hp[3 * its[j] + 2]);
            if (next == ends[j]) {
                cur[j] = oldp;
            } else {
                V3 newp = ccd::mk(hp[3 * next], hp[3 * next + 1], hp[3 * next + 2]);
                double dt = ht[next] - ht[its[j]];
                double a = now - ht[its[j]];
                double b = ht[next] - now;
                cur[j] = ccd::mk((b * oldp.x + a * newp.x) / dt, (b * oldp.y + a * newp.y) / dt,
                                 (b * oldp.z + a * newp.z) / dt);
                newtime = ccd::smin(newtime, ht[next]);
            }
        }
        return newtime;
    }
};

// A stencil's windows are walked through by 2^log_parts lanes, each those that start in one of as many equal spans
// of time, 64 windows between two visits to the pool.  A lane stops after a window at whose end the features are
// closer than the thickness: that window should collide, and later ones do not matter then.  (Walking on took
// 24.8 ms, and testing the windows at once 2.2 ms, for 8,600 stencils of each kind over 60 entries that nearly all
// collide; here 1.7.)
// count[part]: its windows; best[stencil]: the least of ~0 and, where a part stopped or the pool had no room, the
// place after which its windows are not known, with 0 for the place in the pool.
constexpr int PLACE_BITS = 20;   // a window's place: part << PLACE_BITS | number in the part
constexpr uint32_t LAST_PLACE = (1u << PLACE_BITS) - 1;
template <bool VF>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void k_hist_open(
    const int64_t *__restrict__ off, const double *__restrict__ ht, const double *__restrict__ hp,
    const int4 *__restrict__ keys, const double *__restrict__ eta, double eta_s, int64_t n, int log_parts,
    int32_t *__restrict__ count, unsigned long long *__restrict__ best, WindowPool pool)
{
    const int64_t x = blockIdx.x * (int64_t)64 + threadIdx.x;
    const int64_t i = x >> log_parts;
    const int g = (int)(x & ((1 << log_parts) - 1));
    const double until = g == (1 << log_parts) - 1 ? __builtin_inf() : ldexp((double)(g + 1), -log_parts);
    const bool mine = i < n;
    const int4 k = mine ? keys[i] : make_int4(0, 0, 0, 0);
    const double et = mine ? (eta ? eta[i] : eta_s) : 0.0;
    Stitch s(off, ht, hp, k);
    V3 prev[4], cur[4];
    double now = __builtin_inf(), next = __builtin_inf();
    if (mine) {
        now = g == 0 ? 0.0 : s.start(ldexp((double)g, -log_parts));
        if (now < until && now <= 1.0) next = s.at(now, prev);
    }
    int w = 0;
    bool stopped = false;
    uint32_t unknown = 0;   // where `stopped`: the place from which the part's windows are not known
    while (__ballot(!stopped && now < until && next <= 1.0)) {
        const double first = now;
        const int w0 = w;
        uint64_t open = 0;
        for (; !stopped && now < until && next <= 1.0 && w < w0 + 64; w++) {
            const double after = s.at(next, cur);
            if (VF ? ccd::screen_vf_window(prev, cur, et) : ccd::screen_ee_window(prev, cur, et)) {
                open |= 1ull << (w - w0);
                stopped = ccd::touching<VF>(cur, et);
                unknown = LAST_PLACE;
            }
#pragma unroll
            for (int j = 0; j < 4; j++) prev[j] = cur[j];
            now = next;
            next = after;
        }
        const bool room = w <= 1 << PLACE_BITS;
        const int need = room ? __popcll(open) : 0;
        int64_t at = claim(pool, (int)(blockIdx.x & (WindowPool::SHARDS - 1)), need);
        if (open == 0) continue;
        if (at < 0 || !room) {
            stopped = true;
            unknown = (uint32_t)w0 < LAST_PLACE ? (uint32_t)w0 : LAST_PLACE;
            continue;
        }
        // Once more, to the windows to be kept.
        Stitch again(off, ht, hp, k);
        V3 a[4], b[4];
        double t = again.at(again.start(first), a);
        uint32_t place = (uint32_t)g << PLACE_BITS | (uint32_t)w0;
        for (; open; open >>= 1, place++) {
            const double after = again.at(t, b);
            if (open & 1) store_window(pool, at++, i, place, et, a, b);
#pragma unroll
            for (int j = 0; j < 4; j++) a[j] = b[j];
            t = after;
        }
    }
    if (!mine) return;
    count[x] = w;
    if (stopped) atomicMin(&best[i], (unsigned long long)((uint32_t)g << PLACE_BITS | unknown) << 32);
}
// The first window, in time, that collides: its place and where it lies in the pool.
__global__ __launch_bounds__(64) void k_hist_hits(WindowPool pool, unsigned long long *__restrict__ best)
{
    const int64_t at = blockIdx.x * (int64_t)64 + threadIdx.x, shard = at / pool.per_shard;
    if (at - shard * pool.per_shard < pool.filled(shard) && pool.owner[at] >= 0 && pool.hit[at])
        atomicMin(&best[pool.owner[at]], (unsigned long long)pool.place[at] << 32 | (unsigned long long)(at + 1));
}
// The windows of one stencil by a whole wavefront, from the start: every lane runs the same merge 65 steps at a
// time and keeps the positions of two consecutive ones, so lane l holds window l of 64 and tests it; the first
// that collides gives the answer.
template <bool VF>
__device__ void hist_wave(const int64_t *__restrict__ off, const double *__restrict__ ht, const double *__restrict__ hp, int4 k,
                          double e, int &r, double &t, int &w)
{
    const int lane = __lane_id();
    Stitch s(off, ht, hp, k);
    V3 cur[4];
    double now = 0.0, next = s.at(0.0, cur);
    r = -1;
    for (int w0 = 0; next <= 1.0; w0 += 64) {
        V3 pa[4], pb[4];
        bool window = false;
        for (int q = 0; q < 64 && next <= 1.0; q++) {
            if (q == lane) {
#pragma unroll
                for (int j = 0; j < 4; j++) pa[j] = cur[j];
            }
            now = next;
            next = s.at(now, cur);
            if (q == lane) {
#pragma unroll
                for (int j = 0; j < 4; j++) pb[j] = cur[j];
                window = true;
            }
        }
        int rl = -1;
        double tl = 0.0;
        if (window)
            rl = VF ? ccd::check_vf_window(pa, pb, e, tl, ccd::NoCount()) : ccd::check_ee_window(pa, pb, e, tl, ccd::NoCount());
        const uint64_t m = __ballot(rl >= 0);
        if (m) {
            const int f = __ffsll((unsigned long long)m) - 1;
            r = __shfl(rl, f);
            t = __shfl(tl, f);
            w = w0 + f;
            return;
        }
    }
}
template <bool VF>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void k_hist_result(
    const int64_t *__restrict__ off, const double *__restrict__ ht, const double *__restrict__ hp,
    const int4 *__restrict__ keys, const double *__restrict__ eta, double eta_s, int64_t n, int log_parts,
    const int32_t *__restrict__ count, const unsigned long long *__restrict__ best, WindowPool pool, int share,
    uint8_t *__restrict__ hit, double *__restrict__ tout, uint8_t *__restrict__ sub, int32_t *__restrict__ win)
{
    const int lane = __lane_id();
    const int64_t i0 = (int64_t)(blockIdx.x / share) * 64, i = i0 + lane;
    const bool mine = i < n && lane % share == (int)(blockIdx.x % share);
    const unsigned long long found = mine ? best[i] : ~0ull;
    int r = -1, w = 0;
    double t = 0.0;
    const bool again = (uint32_t)found == 0;   // (a place in the pool is above 0, no window at all ~0)
    if (found != ~0ull && !again) {
        const int64_t at = (int64_t)(uint32_t)found - 1;
        const uint32_t place = (uint32_t)(found >> 32);
        r = pool.sub[at];
        t = pool.t[at];
        w = (int)(place & ((1u << PLACE_BITS) - 1));
        if (win)
            for (uint32_t g = 0; g < place >> PLACE_BITS; g++) w += count[(i << log_parts) + g];
    }
    for (uint64_t lost = __ballot(again); lost; lost &= lost - 1) {
        const int l = __ffsll((unsigned long long)lost) - 1;
        int rr, ww = 0;
        double tt = 0.0;
        hist_wave<VF>(off, ht, hp, keys[i0 + l], eta ? eta[i0 + l] : eta_s, rr, tt, ww);
        if (lane == l) {
            r = rr;
            t = tt;
            w = ww;
        }
    }
    if (!mine) return;
    hit[i] = r >= 0 ? 1 : 0;
    if (tout) tout[i] = r >= 0 ? t : 0.0;
    if (sub) sub[i] = r >= 0 ? (uint8_t)r : (uint8_t)255;
    if (win) win[i] = r >= 0 ? w : -1;
}

// ------------------------------------------------------------------------------------------------
// Separating planes
// ------------------------------------------------------------------------------------------------
// Status 1 (collision), 0 (none) or 2 (undecided: the reference's recursion would not end); SP_LOST and
// SP_RUN_AGAIN between the passes.

// W lanes that all run the same stencil.
template <int W>
struct Group {
    int sub, base;
    __device__ __forceinline__ Group() : sub(__lane_id() & (W - 1)), base(__lane_id() & ~(W - 1)) {}
    __device__ __forceinline__ double from(double x, int s) const   // lane s of the group's (s the same in all of them)
    {
        if constexpr (W == 64) {
            const int l = __builtin_amdgcn_readfirstlane(s);
            const unsigned long long u = (unsigned long long)ccd::double_to_bits(x);
            return ccd::bits_to_double((long long)((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)u, l) |
                                                   (unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(u >> 32), l) << 32));
        } else {
            return __shfl(x, base + s);
        }
    }
    __device__ __forceinline__ V3 from(V3 x, int s) const { return ccd::mk(from(x.x, s), from(x.y, s), from(x.z, s)); }
    __device__ __forceinline__ uint64_t votes(bool b) const
    {
        const uint64_t m = __ballot(b);
        return W == 64 ? m : (m >> base) & ((1ull << (W & 63)) - 1);
    }
};

// Histories of any length, in memory: the lanes share a trajectory scan (planeTrajectoryIntersect,
// SeparatingPlaneNarrowPhase.cpp:216-265), W segments at a time; the first in scan order that meets the plane
// gives the result.
template <int W>
struct SharedHistory : Group<W> {
    const ccd::CsrHistory &csr;
    __device__ __forceinline__ explicit SharedHistory(const ccd::CsrHistory &c) : csr(c) {}
    __device__ __forceinline__ V3 pos(int j, double time, int &idx) const { return csr.pos(j, time, idx); }
    __device__ __forceinline__ void step(int j, int idx, V3 &d, double &dt) const { csr.step(j, idx, d, dt); }
    template <bool VF>
    __device__ __forceinline__ void scan(const int (&mi)[4], V3 ppos, V3 pvel, V3 closest, const V3 (&mp)[4], double midt,
                                         double eta, double &t_lo, double &t_hi) const
    {
        const ccd::HistCSR &h = csr.h;
        for (int q = 0; q < 8; q++) {
            const int j = q & 3;
            const bool fwd = q >= 4;
            const int vj = j == 0 ? csr.v[0] : (j == 1 ? csr.v[1] : (j == 2 ? csr.v[2] : csr.v[3]));
            const int start = (j == 0 ? mi[0] : (j == 1 ? mi[1] : (j == 2 ? mi[2] : mi[3]))) + (fwd ? 1 : 0);
            const V3 mid = j == 0 ? mp[0] : (j == 1 ? mp[1] : (j == 2 ? mp[2] : mp[3]));
            const V3 nrm = ((j == 0 || (j == 1 && !VF)) ? -1.0 : 1.0) * closest;
            const V3 vel = (fwd ? 1.0 : -1.0) * pvel;
            const int64_t b = h.off[vj];
            const int n = (int)(h.off[vj + 1] - b);
            double &least = fwd ? t_hi : t_lo;
            const double dt = fwd ? h.t[b + start] - midt : midt - h.t[b + start];
            const double t = ccd::plane_intersect(ppos, vel, nrm, mid, ccd::hist_pos(h, b + start), dt, eta);
            if (t >= 0 && t <= dt) {
                least = ccd::smin(least, t);
                continue;
            }
            // Segments (i, i + 1) for i = start .. n - 2, or (i, i - 1) for i = start .. 1.
            for (int i0 = start; fwd ? i0 < n - 1 : i0 >= 1; i0 += fwd ? W : -W) {
                const int i = fwd ? i0 + this->sub : i0 - this->sub;
                bool hit = false;
                double r = 0.0;
                if (fwd ? i < n - 1 : i >= 1) {
                    const double ti = h.t[b + i], tn = h.t[b + i + (fwd ? 1 : -1)];
                    const V3 npp = fwd ? ppos + (ti - midt) * pvel : ppos - (midt - ti) * pvel;
                    const double d = fwd ? tn - ti : ti - tn;
                    const double u = ccd::plane_intersect(npp, vel, nrm, ccd::hist_pos(h, b + i),
                                                          ccd::hist_pos(h, b + i + (fwd ? 1 : -1)), d, eta);
                    hit = u >= 0 && u <= d;
                    r = fwd ? ti + u - midt : midt - (ti - u);
                }
                const uint64_t m = this->votes(hit);
                if (m) {
                    least = ccd::smin(least, this->from(r, __ffsll((unsigned long long)m) - 1));
                    break;
                }
            }
        }
    }
};

// Histories of at most W entries in the lanes' registers: lane s holds entry s of each vertex and the one after
// it, so a time is looked up by a ballot, an entry comes from its lane, and one evaluation tests all segments
// of a vertex, in both directions.  The chain of nodes of one stencil is what bounds the kernel: a node's
// searches and scans in memory are some 50 dependent loads.
template <int W>
struct LaneHistory : Group<W> {
    using Group<W>::sub;
    using Group<W>::from;
    using Group<W>::votes;
    double t[4], tn[4];
    V3 p[4], pn[4];
    int n[4];
    const ccd::CsrHistory &csr;
    __device__ __forceinline__ explicit LaneHistory(const ccd::CsrHistory &c) : csr(c)
    {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int64_t b = c.h.off[c.v[j]];
            n[j] = (int)(c.h.off[c.v[j] + 1] - b);
            const int64_t e = b + (sub < n[j] ? sub : n[j] - 1), next = b + (sub + 1 < n[j] ? sub + 1 : n[j] - 1);
            t[j] = sub < n[j] ? c.h.t[e] : __builtin_inf();   // past the last: later than every time
            p[j] = ccd::hist_pos(c.h, e);
            tn[j] = c.h.t[next];
            pn[j] = ccd::hist_pos(c.h, next);
        }
    }
    __device__ __forceinline__ V3 pos(int j, double time, int &idx) const   // ccd::pos_at_time
    {
        const int lo = __popcll(votes(t[j] <= time));   // the first entry after `time`
        if (lo == n[j]) {
            idx = lo - 1;
            return from(p[j], idx);
        }
        const int prev = lo > 0 ? lo - 1 : 0;
        idx = prev;
        const double t0 = from(t[j], prev), t1 = lo > 0 ? from(tn[j], prev) : t0;
        const V3 a = from(p[j], prev), c = lo > 0 ? from(pn[j], prev) : a;
        const double alpha = (time - t0) / (t1 - t0);
        return (1.0 - alpha) * a + alpha * c;
    }
    __device__ __forceinline__ void step(int j, int idx, V3 &d, double &dt) const
    {
        if (idx == n[j] - 1) return csr.step(j, idx, d, dt);   // (a time of exactly 1, where histories repeat a time)
        d = from(pn[j], idx) - from(p[j], idx);
        dt = from(tn[j], idx) - from(t[j], idx);
    }
    template <bool VF>
    __device__ __forceinline__ void scan(const int (&mi)[4], V3 ppos, V3 pvel, V3 closest, const V3 (&mp)[4], double midt,
                                         double eta, double &t_lo, double &t_hi) const
    {
        if (mi[0] == n[0] - 1 || mi[1] == n[1] - 1 || mi[2] == n[2] - 1 || mi[3] == n[3] - 1)
            return csr.scan<VF>(mi, ppos, pvel, closest, mp, midt, eta, t_lo, t_hi);
        // planeTrajectoryIntersect (SeparatingPlaneNarrowPhase.cpp:216-265), by lane s: the segment (s, s + 1),
        // backward before the entry mi and forward after it; lane mi the first piece backward, from the middle.
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const V3 nrm = ((j == 0 || (j == 1 && !VF)) ? -1.0 : 1.0) * closest;
            const bool back = sub < mi[j], start = sub == mi[j];
            const V3 npp = start ? ppos : (back ? ppos - (midt - tn[j]) * pvel : ppos + (t[j] - midt) * pvel);
            const V3 vel = back || start ? -1.0 * pvel : pvel;
            const V3 a = start ? mp[j] : (back ? pn[j] : p[j]), b = back || start ? p[j] : pn[j];
            const double d = start ? midt - t[j] : tn[j] - t[j];
            const double u = ccd::plane_intersect(npp, vel, nrm, a, b, d, eta);
            const bool hit = u >= 0 && u <= d && sub < n[j] - 1;   // (the last entry starts no segment)
            const double r = start ? u : (back ? midt - (tn[j] - u) : t[j] + u - midt);
            const uint64_t m = votes(hit), earlier = m & ((2ull << mi[j]) - 1ull), later = m & ~((2ull << mi[j]) - 1ull);
            if (earlier) t_lo = ccd::smin(t_lo, from(r, 63 - __clzll((long long)earlier)));
            // The first piece forward, from the middle to entry mi + 1.
            const double t1 = from(tn[j], mi[j]), d1 = t1 - midt;
            const double u1 = ccd::plane_intersect(ppos, pvel, nrm, mp[j], from(pn[j], mi[j]), d1, eta);
            if (u1 >= 0 && u1 <= d1) t_hi = ccd::smin(t_hi, u1);
            else if (later) t_hi = ccd::smin(t_hi, from(r, __ffsll((unsigned long long)later) - 1));
        }
    }
};

// Most stencils are decided at the root interval [0, 1], one lane each: status, and sort key 0.  Key 1: the
// recursion goes on; sorted together, those fill wavefronts.
template <bool VF>
__global__ __launch_bounds__(256) void k_sp_order_key(const int64_t *__restrict__ off, const double *__restrict__ ht,
                                                      const double *__restrict__ hp, const int4 *__restrict__ keys,
                                                      const double *__restrict__ eta, double eta_s, int64_t n,
                                                      const unsigned long long *__restrict__ gap_bits,
                                                      uint64_t *__restrict__ key, int32_t *__restrict__ idx,
                                                      uint8_t *__restrict__ status)
{
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double eps = ccd::bits_to_double((long long)*gap_bits) / 4.0;
    const int4 k = keys[i];
    const int v[4] = {k.x, k.y, k.z, k.w};
    ccd::HistCSR h{off, ht, hp};
    // (eps is at most 1/4, so the root is never short enough for a window test)
    const int r = ccd::separating_plane_nodes<VF>(ccd::CsrHistory{h, v}, eta ? eta[i] : eta_s, eps, 1,
                                                  [](const V3 (&)[4], const V3 (&)[4]) { return false; });
    key[i] = r == 3 ? 1u : 0u;
    idx[i] = (int32_t)i;
    if (r != 3) status[i] = (uint8_t)r;
}

// The recursions, their windows left to the pool, their statuses as DeferredWindows gives them.  W lanes to a
// stencil; with an order, group j runs stencil order[j] if open[j] is not 0.
template <bool VF, int W>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void k_sp_nodes(
    const int64_t *__restrict__ off, const double *__restrict__ ht, const double *__restrict__ hp,
    const int4 *__restrict__ keys, const double *__restrict__ eta, double eta_s, int64_t n,
    const unsigned long long *__restrict__ gap_bits, const int32_t *__restrict__ order,
    const uint64_t *__restrict__ open, uint8_t *__restrict__ status, WindowPool pool)
{
    const int64_t x = (blockIdx.x * (int64_t)64 + threadIdx.x) / W;
    if (x >= n || (order && open[x] == 0)) return;   // (whole groups)
    const int64_t i = order ? (int64_t)order[x] : x;
    const double eps = ccd::bits_to_double((long long)*gap_bits) / 4.0, et = eta ? eta[i] : eta_s;
    const int4 k = keys[i];
    const int v[4] = {k.x, k.y, k.z, k.w};
    ccd::HistCSR h{off, ht, hp};
    const ccd::CsrHistory csr{h, v};
    const bool writes = (__lane_id() & (W - 1)) == 0;
    auto store = [&](const V3 (&s)[4], const V3 (&e)[4]) {
        int64_t at = claim(pool, (int)(blockIdx.x & (WindowPool::SHARDS - 1)), writes ? 1 : 0);
        at = __shfl(at, __lane_id() & ~(W - 1));
        if (at >= 0 && writes) store_window(pool, at, i, 0, et, s, e);
        return at >= 0;
    };
    ccd::DeferredWindows<VF, decltype(store) &> window(et, store);
    int r;
    if constexpr (W == 1) {
        r = ccd::separating_plane_nodes<VF>(csr, et, eps, 0x7fffffff, window);
    } else {
        bool fits = true;
#pragma unroll
        for (int j = 0; j < 4; j++) fits = fits && off[v[j] + 1] - off[v[j]] <= W;
        if (fits) {
            const LaneHistory<W> lanes(csr);
            r = ccd::separating_plane_nodes<VF>(lanes, et, eps, 0x7fffffff, window);
        } else {
            const SharedHistory<W> shared(csr);
            r = ccd::separating_plane_nodes<VF>(shared, et, eps, 0x7fffffff, window);
        }
    }
    if (writes) status[i] = (uint8_t)window.status(r);
}
// A window that collides decides its stencil.
__global__ __launch_bounds__(64) void k_sp_hits(WindowPool pool, uint8_t *__restrict__ status)
{
    const int64_t at = blockIdx.x * (int64_t)64 + threadIdx.x, shard = at / pool.per_shard;
    if (at - shard * pool.per_shard < pool.filled(shard) && pool.owner[at] >= 0 && pool.hit[at]) status[pool.owner[at]] = 1;
}
template <bool VF>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void k_sp_result(
    const int64_t *__restrict__ off, const double *__restrict__ ht, const double *__restrict__ hp,
    const int4 *__restrict__ keys, const double *__restrict__ eta, double eta_s, int64_t n,
    const unsigned long long *__restrict__ gap_bits, int share, uint8_t *__restrict__ status, unsigned long long *undecided)
{
    const int lane = __lane_id();
    const int64_t i0 = (int64_t)(blockIdx.x / share) * 64, i = i0 + lane;
    int r = i < n && lane % share == (int)(blockIdx.x % share) ? status[i] : 0;
    const double eps = ccd::bits_to_double((long long)*gap_bits) / 4.0;
    for (uint64_t lost = __ballot(r == ccd::SP_LOST || r == ccd::SP_RUN_AGAIN); lost; lost &= lost - 1) {   // by the whole wavefront
        const int l = __ffsll((unsigned long long)lost) - 1;
        const int4 k = keys[i0 + l];
        const int v[4] = {k.x, k.y, k.z, k.w};
        const double et = eta ? eta[i0 + l] : eta_s;
        ccd::HistCSR h{off, ht, hp};
        const ccd::CsrHistory csr{h, v};
        const SharedHistory<64> shared(csr);
        const int rr = ccd::separating_plane_nodes<VF>(shared, et, eps, 0x7fffffff, [&](const V3 (&s)[4], const V3 (&e)[4]) {
            double t = 0.0;
            return (VF ? ccd::check_vf_window(s, e, et, t, ccd::NoCount()) : ccd::check_ee_window(s, e, et, t, ccd::NoCount())) >= 0;
        });
        if (lane == l) {
            r = rr;
            status[i] = (uint8_t)rr;
        }
    }
    const uint64_t m = __ballot(r == 2);
    if (m && __lane_id() == __ffsll((unsigned long long)m) - 1) atomicAdd(undecided, (unsigned long long)__popcll(m));
}

inline unsigned blocks_for(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

}   // namespace

namespace ccdi {

// A pool for the windows of n stencils, and its lists (223 bytes a window, and half a megabyte).  All the windows
// of the stencils on short lists, one per stencil on long ones: most stencils need none.  Without memory for that,
// half as many, and so on: the pool's size changes no result.
static int window_pool(ccd_ctx *ctx, int64_t n, int64_t windows, WindowPool &p, void *&list)
{
    constexpr int64_t FEW = 1 << 14, ENOUGH = 1 << 19, MOST = 1 << 22, STEP = 4096;
    int64_t cap = std::max(std::min(std::max(windows * n, FEW), ENOUGH), std::min(n, MOST));
    char *b = nullptr;
    for (;; cap /= 2) {
        cap = (cap + STEP - 1) / STEP * STEP;
        b = (char *)buffer(ctx, "window_pool", (size_t)cap * (192 + 8 + 8 + 4 + 4 + 1 + 1) + WindowPool::SHARDS * WindowPool::STRIDE * 8);
        list = b ? open_list(ctx, cap) : nullptr;
        if (list) break;
        if (cap == STEP) return CCD_E_OOM;
    }
    p.pos = (double *)b;
    p.eta = p.pos + 24 * cap;
    p.t = p.eta + cap;
    p.claimed = (unsigned long long *)(p.t + cap);
    p.owner = (int32_t *)(p.claimed + WindowPool::SHARDS * WindowPool::STRIDE);
    p.place = (uint32_t *)(p.owner + cap);
    p.hit = (uint8_t *)(p.place + cap);
    p.sub = p.hit + cap;
    p.per_shard = cap / WindowPool::SHARDS;
    return fill_u64(ctx, (uint64_t *)p.claimed, WindowPool::SHARDS * WindowPool::STRIDE, 0);
}

// Wavefronts that share 64 stencils in the last kernels, each its part of those to be run again: as many as there
// are places for on the chip, since nearly all of a call's stencils may be such.
static int result_share(int64_t n)
{
    int share = 64;
    while (share > 1 && n * share > 1 << 18) share /= 2;
    return share;
}

// Stencils to a set of launches: bounds the scratch memory and the grids.
constexpr int64_t PIECE = 1 << 22;

static int narrow_hist_piece(ccd_ctx *ctx, bool vf, const int64_t *off, const double *ht, const double *hp,
                             const int32_t *keys, const double *eta, double eta_s, int64_t n, uint8_t *hit, double *t,
                             uint8_t *sub, int32_t *win, int64_t entries)
{
    // A stencil has up to four times a vertex's entries of windows.  A lane to about sixteen of them, since it
    // walks through them one after another, but not more lanes than fill the chip.
    int log_parts = 0;
    while (log_parts < 12 && (4 * entries) >> log_parts > 16 && n << log_parts <= 1 << 22) log_parts++;
    const int64_t nparts = n << log_parts;
    WindowPool pool;
    void *list;
    int rc = window_pool(ctx, n, 4 * entries, pool, list);
    if (rc) return rc;
    unsigned long long *best = (unsigned long long *)buffer(ctx, "hist_best", (size_t)n * 8);
    int32_t *count = (int32_t *)buffer(ctx, "hist_count", (size_t)nparts * 4);
    if (!best || !count) return CCD_E_OOM;
    rc = fill_u64(ctx, (uint64_t *)best, n, ~0ull);
    if (rc) return rc;
    auto k_open = vf ? k_hist_open<true> : k_hist_open<false>;
    hipLaunchKernelGGL(k_open, dim3(blocks_for(nparts, 64)), dim3(64), 0, ctx->stream, off, ht, hp, (const int4 *)keys, eta,
                       eta_s, n, log_parts, count, best, pool);
    CCD_LAUNCH_CHECK(ctx);
    rc = launch_screened_pool(ctx, vf, pool, list);
    if (rc) return rc;
    hipLaunchKernelGGL(k_hist_hits, dim3((unsigned)(WindowPool::SHARDS * pool.per_shard / 64)), dim3(64), 0, ctx->stream, pool,
                       best);
    CCD_LAUNCH_CHECK(ctx);
    auto k_result = vf ? k_hist_result<true> : k_hist_result<false>;
    const int share = result_share(n);
    hipLaunchKernelGGL(k_result, dim3(blocks_for(n, 64) * share), dim3(64), 0, ctx->stream, off, ht, hp, (const int4 *)keys, eta,
                       eta_s, n, log_parts, count, best, pool, share, hit, t, sub, win);
    CCD_LAUNCH_CHECK(ctx);
    return CCD_OK;
}

int launch_narrow_hist(ccd_ctx *ctx, bool vf, const int64_t *off, const double *ht, const double *hp,
                       const int32_t *keys, const double *eta, double eta_s, int64_t n, uint8_t *hit, double *t,
                       uint8_t *sub, int32_t *win, int64_t entries)
{
    for (int64_t i = 0; i < n; i += PIECE) {
        const int rc = narrow_hist_piece(ctx, vf, off, ht, hp, keys + 4 * i, eta ? eta + i : nullptr, eta_s,
                                         std::min(PIECE, n - i), hit + i, t ? t + i : nullptr, sub ? sub + i : nullptr,
                                         win ? win + i : nullptr, entries);
        if (rc) return rc;
    }
    return CCD_OK;
}

static int separating_plane_piece(ccd_ctx *ctx, bool vf, const int64_t *off, const double *ht, const double *hp,
                                  const int32_t *keys, const double *eta, double eta_s, int64_t n,
                                  const uint64_t *gap_bits, uint8_t *status, int64_t *undecided, int64_t entries)
{
    auto gb = (const unsigned long long *)gap_bits;
    // Lanes to a stencil: as many as its histories have entries, of the forms there are; one for histories of
    // two entries, whose recursions end after a window test or two, so that all stencils together bound the
    // launch and not the longest one (7.67M stencils of a 256^2 cloth, a call and
    // its copies: 6.9 ms with the cascade in the lane, 8.0 with eight lanes, 5.2 with one).
    const int lanes = entries <= 2 ? 1 : (entries <= 8 ? 8 : 64);
    WindowPool pool;
    void *list;
    int rc = window_pool(ctx, n, 16, pool, list);   // (a recursion ends after a window or two)
    if (rc) return rc;
    const int32_t *order = nullptr;
    const uint64_t *open = nullptr;
    if (lanes < 64 && n >= 4096) {
        uint64_t *key = (uint64_t *)buffer(ctx, "spo_key", (size_t)n * 8);
        uint64_t *key2 = (uint64_t *)buffer(ctx, "spo_key2", (size_t)n * 8);
        int32_t *idx = (int32_t *)buffer(ctx, "spo_idx", (size_t)n * 4);
        int32_t *idx2 = (int32_t *)buffer(ctx, "spo_idx2", (size_t)n * 4);
        void *tmp = buffer(ctx, "spo_tmp", radix_sort_temp_bytes(n));
        if (!key || !key2 || !idx || !idx2 || !tmp) return CCD_E_OOM;
        auto k_key = vf ? k_sp_order_key<true> : k_sp_order_key<false>;
        hipLaunchKernelGGL(k_key, dim3(blocks_for(n, 256)), dim3(256), 0, ctx->stream, off, ht, hp, (const int4 *)keys, eta,
                           eta_s, n, gb, key, idx, status);
        CCD_LAUNCH_CHECK(ctx);
        bool in_alt = false;
        rc = radix_sort_pairs(ctx, key, idx, key2, idx2, n, 1, tmp, in_alt);   // one stable pass
        if (rc) return rc;
        order = in_alt ? idx2 : idx;
        open = in_alt ? key2 : key;
    }
    auto k_nodes = vf ? (lanes == 1 ? k_sp_nodes<true, 1> : lanes == 8 ? k_sp_nodes<true, 8> : k_sp_nodes<true, 64>)
                      : (lanes == 1 ? k_sp_nodes<false, 1> : lanes == 8 ? k_sp_nodes<false, 8> : k_sp_nodes<false, 64>);
    hipLaunchKernelGGL(k_nodes, dim3(blocks_for(n * lanes, 64)), dim3(64), 0, ctx->stream, off, ht, hp,
                       (const int4 *)keys, eta, eta_s, n, gb, order, open, status, pool);
    CCD_LAUNCH_CHECK(ctx);
    rc = launch_screened_pool(ctx, vf, pool, list);
    if (rc) return rc;
    hipLaunchKernelGGL(k_sp_hits, dim3((unsigned)(WindowPool::SHARDS * pool.per_shard / 64)), dim3(64), 0, ctx->stream, pool,
                       status);
    CCD_LAUNCH_CHECK(ctx);
    auto k_result = vf ? k_sp_result<true> : k_sp_result<false>;
    const int share = result_share(n);
    hipLaunchKernelGGL(k_result, dim3(blocks_for(n, 64) * share), dim3(64), 0, ctx->stream, off, ht, hp, (const int4 *)keys, eta,
                       eta_s, n, gb, share, status, (unsigned long long *)undecided);
    CCD_LAUNCH_CHECK(ctx);
    return CCD_OK;
}

int launch_separating_plane(ccd_ctx *ctx, bool vf, const int64_t *off, const double *ht, const double *hp,
                            const int32_t *keys, const double *eta, double eta_s, int64_t n, const uint64_t *gap_bits,
                            uint8_t *status, int64_t *undecided, int64_t entries)
{
    for (int64_t i = 0; i < n; i += PIECE) {
        const int rc = separating_plane_piece(ctx, vf, off, ht, hp, keys + 4 * i, eta ? eta + i : nullptr, eta_s,
                                              std::min(PIECE, n - i), gap_bits, status + i, undecided, entries);
        if (rc) return rc;
    }
    return CCD_OK;
}

}   // namespace ccdi
