// Test-only: the broadphase's integer grids (collisiondetection_amd/csrc/grids.h) on the host.
#include "../../collisiondetection_amd/csrc/grids.h"

// One axis of n boxes: the quantised bounds, with the range that the broadphase takes from all of them.
extern "C" void quantise_axis(const double *lo, const double *hi, int64_t n, uint16_t *qlo, uint16_t *qhi)
{
    double least = __builtin_inf(), most = -__builtin_inf();
    for (int64_t i = 0; i < n; i++) {
        if (__builtin_isfinite(lo[i]) && lo[i] < least) least = lo[i];
        if (__builtin_isfinite(hi[i]) && hi[i] > most) most = hi[i];
    }
    const double inv = ccd::quant_scale(least, most), o = __builtin_isfinite(least) ? least : 0.0;
    for (int64_t i = 0; i < n; i++) {
        qlo[i] = ccd::quant_lo(lo[i], o, inv);
        qhi[i] = ccd::quant_hi(hi[i], o, inv);
    }
}
extern "C" int surely_reaches(int qhi, int qlo) { return ccd::surely_reaches(qhi, qlo); }
extern "C" int cell_bits(double extent, double inv) { return ccd::cell_bits(extent, inv); }
