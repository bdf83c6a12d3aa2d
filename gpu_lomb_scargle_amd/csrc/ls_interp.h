// Modes of the coarse-grid sweep (ls_sweep_interp.hip), shared with the
// statistics and record kernels that choose a mode per object (ls_sweep.hip).
//
// A mode has a coarse step of h bins and result rows of m coarse steps (h m
// <= 32 bins, one lane each).  Two uses:
//   sums   (FP32 periodograms) W = 8 taps, the window for an oversampling of
//     2.25, used from kIpSigma = 2.32 on: aliasing of at most 6e-8 of an
//     observation (those at the ends of the span), 2e-8 in the mean, so that
//     the rounding is what is left.  Error against 64 bits, coarse over direct
//     sums, rms over bins of at least 1e-3 of the peak, at 2.32 to 3: 33 to 50
//     observations 0.99 to 1.05, 64 0.97 to 1.00, 100 to 500 0.77 to 0.96,
//     2,000 to 65,000 0.82 to 1.00 (worst bins alike, 8.1e-6).  Used at its own
//     oversampling a window aliases ten times more: the one for 1.95, at
//     1.95 (7.6e-7 at the ends), had 1.5 to 1.7 at 100 observations, 2.5 to 3.4
//     at 30.  The generalized power, from four interpolated sums, takes 2.4: 33
//     to 50 observations 0.98 to 1.05, 64 to 8,000 0.77 to 0.99; its direct sums
//     fold y's in FP64, the coarse ones in FP32, which shows from there: 12,000
//     1.06, 65,000 1.26.
//   screen (peaks without a periodogram) FP16 heads alone, W = 6 taps at an
//     oversampling of at least 1.3: aliasing 1.2e-4, powers near the peak
//     good to ~1e-3, which only decide which chunks the direct tile sweeps.
#pragma once

#include "ls_device.h"

namespace lsamd {

namespace {

constexpr int kIpModes = 7;           // h = 3 in the screen only
constexpr double kIpSigma = 2.32, kIpSigmaGen = 2.4, kIpSigmaScreen = 1.3, kIpSigmaWindow = 2.25;
__host__ __device__ constexpr int ip_frags(bool screen) { return screen ? 4 : 8; }  // column-factor fragments per 16 observations
// Relative margin of the marked chunks below the top_k-th best power: ten
// times the sums' error bound; the screen's: see k_sweep_interp.
constexpr float kIpMargin = 1e-4f, kIpMarginScreen = 0.125f;
__host__ __device__ constexpr int ip_step(int mode) {
    return mode == 1 ? 3 : mode == 2 ? 4 : mode == 3 ? 5 : mode == 4 ? 6 : mode == 5 ? 8 : mode == 6 ? 10 : 16;
}
__host__ __device__ constexpr int ip_per_row(int mode) { return 32 / ip_step(mode); }
// rows of a workgroup: m rows + W - 1 <= 2048 points, a multiple of 32 where that loses less than a tile
__host__ __device__ constexpr int ip_rows(int mode) {
    return mode == 1 ? 192 : mode == 2 ? 255 : mode == 3 ? 320 : mode == 4 ? 408 : mode == 5 ? 510 : mode == 6 ? 672 : 1020;
}
__host__ __device__ constexpr int ip_taps(bool screen) { return screen ? 6 : 8; }
// Points in LDS of a sum at f and of the sum at 2 f, the zeros behind the last ones included.
constexpr uint32_t kIpPoints = 2048 + 32, kIpPoints2 = 4096 + 32;
// Result row whose points lane row rc of tile t reads: its own, or the last one
// (rows are no multiple of 32 in every mode; the results of those past it are dropped).
__host__ __device__ constexpr uint32_t ip_operand_row(uint32_t rows, uint32_t t, uint32_t rc) {
    const uint32_t s = 32u * t + rc;
    return s < rows ? s : rows - 1u;
}
// A row's window at 2 f reaches past 16 points.
__host__ __device__ constexpr bool ip_wide(bool screen, int mode) { return 2 * ip_per_row(mode) - 1 + ip_taps(screen) > 16; }
constexpr bool ip_reads_fit() {
    for (int screen = 0; screen < 2; ++screen)
        for (int mode = 1; mode <= kIpModes; ++mode) {
            const uint32_t m = (uint32_t)ip_per_row(mode), rows = (uint32_t)ip_rows(mode);
            const uint32_t last = ip_operand_row(rows, (rows - 1) / 32, 31);
            if (m * last + 16u > kIpPoints || 2u * m * last + (ip_wide(screen, mode) ? 32u : 16u) > kIpPoints2) return false;
        }
    return true;
}
static_assert(ip_reads_fit(), "operand reads stay within the points");
__host__ __device__ constexpr double ip_beta(bool screen) {
    return 3.14159265358979323846 * ip_taps(screen) * (1.0 - 1.0 / (2.0 * (screen ? kIpSigmaScreen : kIpSigmaWindow)));
}
// Largest 1/Phi at the ends of the span (ip_inv_window), rounded up: 2.08 and 9.94.
__host__ __device__ constexpr double ip_window_most(bool screen) { return screen ? 10.0 : 3.0; }
// The points' scale is 2^ip_point_shift / 2^bits, n < 2^bits: with the factors'
// 2^10 and n observations in phase, at most 1 each, they end below FP16's 65504.
__host__ __device__ constexpr int ip_point_shift(bool screen) { return screen ? 2 : 3; }
static_assert(ip_window_most(false) * (1024 << ip_point_shift(false)) < 65504.0 &&
                  ip_window_most(true) * (1024 << ip_point_shift(true)) < 65504.0,
              "points within FP16's range");
constexpr uint32_t kIpLeastBins = 255 * 32, kIpLeastBinsScreen = 192 * 30;  // bins per workgroup, smallest mode
constexpr uint32_t kIpGroup = 4;  // consecutive items of an object per workgroup, at most
// The generalized sums' workgroups take one (the loop costs them 4%).
__host__ __device__ constexpr bool ip_grouped(bool screen, bool gen) { return screen || !gen; }
// Objects up to here (generalized ones also from kIpMostObsGen on) keep the
// direct sums, those of at most 16 observations their FP64 ones: with 18
// observations and weights over a factor of 400 the worst bin reached 1.4e-5
// (direct 1.0e-5).  Peaks alone, generalized: with
// few observations most chunks hold bins that either sweep computes again in
// FP64, or powers near 1 (400 objects x 400,000 bins, direct / coarse, us: 20
// observations 8420 / 13400, 30 2295 / 2517, 35 2004 / 930, 50 1939 / 405).
constexpr uint32_t kIpLeastObs = 32, kIpLeastObsScreen = 16, kIpLeastObsScreenGen = 32, kIpMostObsGen = 8192;
// The screen computes a tile's ill-conditioned bins again when no more lanes
// than this have one (1, 4, 16 lanes: 1394, 1227, 937 us at 35 observations,
// 2485, 2517, 2654 at 30).
constexpr int kIpScreenIll = 16;
// Below these the direct sums are sooner done (FP32, top-1, ten bins per
// resolution element; direct / coarse, us): 400 objects x 20,000 bins, 1.4e9
// terms, 152 / 170 standard and 288 / 260 generalized; 100 x 80,000, 1.4e9:
// 131 / 130; 100 x 200,000, 3.4e9: 252 / 177 and 440 / 235; 4 x 500,000, 0.3e9:
// 56 / 75.  A call that may not look at how many objects it sweeps takes the
// coarse grid from 2^18 bins on, where a few objects lose ~25 us by it.
constexpr uint32_t kIpMinFreqs = 8192;  // about the bins that a workgroup takes (5760 screen, 8160 sums, or more)
constexpr double kIpMinTerms = 1.5e9;
// Peaks alone (FP64, top-3, direct / coarse): 10 objects x 300,000 bins, 0.5e9
// terms, 82 / 76 standard and 127 / 110 generalized; 40 x 100,000, 0.7e9: 87 / 99
// and 135 / 139; 200 x 20,000, 0.7e9: 104 / 137 and 166 / 205; 200 x 50,000,
// 1.7e9: 160 / 149 and 240 / 212.
constexpr double kIpMinTermsScreen = 1e9;
constexpr uint32_t kIpAloneFreqs = 1u << 18;
constexpr uint32_t kIpMaxFreqs = 1u << 29;   // byte offsets of an object's row in 32 bits

// 1 / Phi(xi) of the window, Phi(0) = 1, at xi = h df t' cycles per coarse
// step, |xi| <= 1 / (2 sigma): s = sqrt(beta^2 - (pi W xi)^2) >= 17 (screen 9),
// where sinh s = e^s / 2 to FP64 (screen: 2e-8).
__device__ __forceinline__ double ip_inv_window(bool screen, double xi) {
    const double beta = ip_beta(screen), u = 3.14159265358979323846 * ip_taps(screen) * xi;
    const double s = sqrt(beta * beta - u * u);
    return s / beta * exp(beta - s);
}

// Scale of the points of an object of n observations.
__device__ __forceinline__ float ip_point_scale(bool screen, uint32_t n) {
    return ldexpf(1.0f, ip_point_shift(screen) - (32 - __clz((int)n)));
}
// Unit of the screen's standard powers before the object's scale: the screen
// only ranks an object's bins, and powers in this unit are of one order for
// every unit of y (in FP32 the powers themselves leave the range for |y| below
// 1e-20 or above 1e18).  A power of two.
__device__ __forceinline__ double ip_rank_unit(double ys, double ws, uint32_t n) {
    const double un = 1.0 / (1024.0 * 1024.0 * (double)ip_point_scale(true, n));
    return un / ys * (ws / ys);
}

}  // namespace

// Kernels of the coarse-grid sweep, [screen][variant][dtype] (sums: FP32 only).
struct InterpEntry {
    SweepFn fac, sweep;
    int threads;
};
extern const InterpEntry kInterp[2][2][2];

}  // namespace lsamd
