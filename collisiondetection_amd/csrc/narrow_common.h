// What the narrowphase translation units share: vertex loads and the hit list.
#pragma once

#include "ccd_core.h"

#include "ccd_internal.h"

namespace {

using ccd::V3;

__device__ __forceinline__ V3 load3(const double *__restrict__ p, int v)
{
    const double *q = p + 3 * (int64_t)v;
    return ccd::mk(q[0], q[1], q[2]);
}

// A vertex's positions at the start and the end of a two-entry history's window.
__device__ __forceinline__ void window_pos(const double *__restrict__ qs, const double *__restrict__ qe, int v, V3 &s,
                                           V3 &e)
{
    const V3 a = load3(qs, v), b = load3(qe, v);
    s = ccd::mk(ccd::stitch0(a.x, b.x), ccd::stitch0(a.y, b.y), ccd::stitch0(a.z, b.z));
    e = b;
}

// Appends the colliding stencils of a wavefront to the output: one atomic per wavefront with a hit.
__device__ __forceinline__ void append_hits(bool hit, int4 k, double t, int4 *__restrict__ out_keys,
                                            double *__restrict__ out_toi, int64_t cap, unsigned long long *counter)
{
    const uint64_t mask = __ballot(hit);
    if (mask == 0) return;
    const int lane = __lane_id();
    const int leader = __ffsll((unsigned long long)mask) - 1;
    unsigned long long base = 0;
    if (lane == leader) base = atomicAdd(counter, (unsigned long long)__popcll(mask));
    base = __shfl(base, leader);
    if (hit) {
        const uint64_t below = mask & ((lane == 0) ? 0ull : (~0ull >> (64 - lane)));
        const int64_t pos = (int64_t)base + __popcll(below);
        if (pos < cap) {
            out_keys[pos] = k;
            if (out_toi) out_toi[pos] = t;
        }
    }
}

}   // namespace
