// Integer grids that the broadphase puts boxes on: the rounding rules, for the device and for tests on the host.
#pragma once

#include "ccd_core.h"

namespace ccd {

// ------------------------------------------------------------------------------------------------
// Bounds quantised to 16 bits
// ------------------------------------------------------------------------------------------------
// Per axis, a bound v maps to x = (v - origin) * inv, with origin the smallest finite lower bound of all leaves
// and inv = 65535 / (largest finite upper bound - origin), or 0 where that is no finite positive number; lower
// bounds take floor(x), upper bounds ceil(x), both clamped to [0, 65535].  Correctly rounded subtraction and
// multiplication are monotone, and so are floor, ceil and the clamps, so overlapping boxes keep overlapping
// (a.hi >= b.lo gives q(a.hi) >= q(b.lo)): the quantised test only ever keeps more.
constexpr double QUANT_MAX = 65535.0;
CCD_FHD double quant_scale(double lo, double hi)
{
    const double ext = hi - lo;
    const bool ok = __builtin_isfinite(lo) && __builtin_isfinite(hi) && ext > 0.0 && __builtin_isfinite(QUANT_MAX / ext);
    return ok ? QUANT_MAX / ext : 0.0;
}
CCD_FHD uint16_t quant_lo(double v, double o, double inv)
{
    const double x = (v - o) * inv;
    if (!(x >= 0.0)) return 0;   // below the range, -inf, NaN: the smallest
    if (x >= QUANT_MAX) return (uint16_t)QUANT_MAX;
    return (uint16_t)__builtin_floor(x);
}
CCD_FHD uint16_t quant_hi(double v, double o, double inv)
{
    const double x = (v - o) * inv;
    // No number: a bound that separates nothing (NaN, +inf) is the largest.  Any other comes from an axis without
    // a scale (0 times a difference that overflows, or -inf): the smallest, where every lower bound is too, so
    // that the quantised values decide nothing.
    if (x != x) return v != v || v == __builtin_inf() ? (uint16_t)QUANT_MAX : 0;
    if (x <= 0.0) return 0;
    if (x >= QUANT_MAX) return (uint16_t)QUANT_MAX;
    return (uint16_t)__builtin_ceil(x);
}

// The bounds a.hi >= b.lo hold for certain if their quantised values differ by two quanta or more: with
// qhi = ceil(x) and so x > qhi - 1, qlo = floor(y) and so y < qlo + 1, qhi - 1 >= qlo + 1 gives x > y, and the
// map to x is monotone.  (The clamps keep this: a clamped qhi = 65535 has x >= 65535 or is a bound that
// separates nothing, a clamped qlo = 0 has y < 1 or is NaN, and the other clamps fail the test.  On an axis
// without a scale only bounds that separate nothing differ from 0.)
CCD_FHD bool surely_reaches(int qhi, int qlo) { return qhi - qlo >= 2; }


// ------------------------------------------------------------------------------------------------
// Cells of the Morton order
// ------------------------------------------------------------------------------------------------
// Bits per axis of a Morton code below inst_bits bits of an instance's number: all that a 63-bit key holds,
// since a body far away makes the rest of the scene small.  (Only as many as 32 times what a surface of the mesh's
// faces takes saved three of eight passes of the sort on 18,432 faces, 55 us of a 1.24 ms call; but with a
// triangle 10^5 mesh sizes away the order of a shuffled sheet of 522,242 faces was its input order: a detection
// took 673 ms, against 62 with all bits and 24 without the triangle.)
CCD_FHD int morton_axis_bits(int inst_bits) { return (63 - inst_bits) / 3; }

// ------------------------------------------------------------------------------------------------
// Cells of the closest-vertex search
// ------------------------------------------------------------------------------------------------
// Bits for the cell coordinates 0 .. extent * inv of an axis and the neighbour after the last.  An extent that is
// no number (a NaN coordinate in the box, or all of them the same infinity) puts every vertex into cell 0.
constexpr int CELL_BITS = 21;   // at most: three axes to a 64-bit key
CCD_FHD int cell_bits(double extent, double inv)
{
    const double last = extent * inv;
    if (!(last >= 1.0)) return 1;
    int bits = 2;
    while (bits < CELL_BITS && last + 1.0 >= (double)(1ll << bits)) bits++;
    return bits;
}

}   // namespace ccd
