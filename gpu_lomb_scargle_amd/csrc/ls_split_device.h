// Device code shared by the split-form sweep kernels (ls_sweep_split.hip,
// ls_sweep_interp.hip): FP64 phasors and powers, the FP64 recomputation of
// single bins, FP16 head/tail splits and the matrix-core operand helpers.
#pragma once

#include "ls_device.h"

namespace lsamd {

namespace {

// ---------------------------------------------------------------------------
// FP64 recomputation of ill-conditioned bins.  Every split-form power comes
// from a 2x2 (standard) or centred 2x2 (generalized) least-squares system; its
// relative error is the sums' relative error times a condition number that
// the sums themselves give:
//   standard:    k = (CC + SS)^2 / (4 D)                 (1 for balanced phases)
//   generalized: k = (1 + C^2 + S^2) (CC + SS) / D      (centred CC, SS, CS;
//                the 1 + C^2 + S^2 covers the centring CC = CCw - C^2)
// with D = CC SS - CS^2.  The FP32 sums (split32) leave ~2.4e-7 k relative
// (measured on the 1000-object generalized batch at the 1 cycle/day alias,
// k ~ 110-230), the FP32-seeded FP64 sums (split) less.  Bins with
// k > kCondMax (a few per 10^6 for nightly-sampled objects) and every bin of
// objects of at most kSmallObs observations (5 points against the
// generalized 3-parameter model can give k ~ 10^5) are computed again from
// the caller's FP64 t, y, dy with FP64 phasors.
// ---------------------------------------------------------------------------
constexpr double kCondMax = 16.0;
constexpr uint32_t kSmallObs = 16;

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Lane src's v, in every lane (src the same in all lanes).
__device__ __forceinline__ double lane_value(double v, int src) {
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, src);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), src);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// sin and cos of 2 pi r for |r| <= 1/2 revolution: the octant q = rint(4 r)
// is taken off exactly, and x = 2 pi (r - q/4), |x| <= pi/4, goes through the
// Taylor series of sin to x^17 and of cos to x^16 (the first omitted terms
// are below 5e-17 and 2e-18), in Horner form.
__device__ __forceinline__ void sincos_rev64(double r, double &s, double &c) {
    const double q = __builtin_rint(4.0 * r);
    const double x = (r - 0.25 * q) * kTwoPi, x2 = x * x;
    double ps = -1.0 / 355687428096000.0;  // -1/17!
    ps = fma(ps, x2, 1.0 / 1307674368000.0);
    ps = fma(ps, x2, -1.0 / 6227020800.0);
    ps = fma(ps, x2, 1.0 / 39916800.0);
    ps = fma(ps, x2, -1.0 / 362880.0);
    ps = fma(ps, x2, 1.0 / 5040.0);
    ps = fma(ps, x2, -1.0 / 120.0);
    ps = fma(ps, x2, 1.0 / 6.0);
    const double sx = fma(-ps * x2, x, x);  // x - x^3/3! + ... - x^17/17!... with alternating signs
    double pc = 1.0 / 20922789888000.0;     // 1/16!
    pc = fma(pc, x2, -1.0 / 87178291200.0);
    pc = fma(pc, x2, 1.0 / 479001600.0);
    pc = fma(pc, x2, -1.0 / 3628800.0);
    pc = fma(pc, x2, 1.0 / 40320.0);
    pc = fma(pc, x2, -1.0 / 720.0);
    pc = fma(pc, x2, 1.0 / 24.0);
    pc = fma(pc, x2, -0.5);
    const double cx = fma(pc, x2, 1.0);
    const int o = (int)q & 3;  // sin/cos of q pi/2 + x
    s = o == 0 ? sx : o == 1 ? cx : o == 2 ? -sx : -cx;
    c = o == 0 ? cx : o == 1 ? -sx : o == 2 ? -cx : sx;
}

// e^{2 pi i f t} in FP64: the phase reduced to [-1/2, 1/2] revolutions with
// the product f t fused (exact before the subtraction).
__device__ __forceinline__ void phasor64(double f, double t, double &c, double &s) {
    const double n = __builtin_rint(f * t);
    sincos_rev64(fma(f, t, -n), s, c);
}

// n / d for d > 0 (normal): the hardware reciprocal refined by two Newton
// steps, then one correction of the quotient (within an ulp or two; the
// IEEE division sequence is twice as long).
__device__ __forceinline__ double fdiv(double n, double d) {
    double r = __builtin_amdgcn_rcp(d);
    r = fma(fma(-d, r, 1.0), r, r);
    r = fma(fma(-d, r, 1.0), r, r);
    const double q = n * r;
    return fma(fma(-d, q, n), r, q);
}

// Power of the standard variant from its uncentred sums (SS = N - CC);
// `ill` when its condition number exceeds kCondMax (or D <= 0, or NaN).
__device__ __forceinline__ double std_power(double XC, double XS, double CC, double CS, double N, bool &ill) {
    const double SS = N - CC, D = CC * SS - CS * CS;
    ill = !((CC + SS) * (CC + SS) <= 4.0 * kCondMax * D) || !(D > 0.0);
    return fdiv(0.5 * (SS * XC * XC - 2.0 * CS * XC * XS + CC * XS * XS), D);
}

// Power of the generalized variant from sums over weights normalised to
// sum 1 (C, S, CCw, SSw, CSw, YCw, YSw; Yb = weighted mean of the y in them,
// YY the centred weighted sum of squares); `ill` as for std_power.
__device__ __forceinline__ double gen_power(double C, double S, double CCw, double SSw, double CSw,
                                            double YCw, double YSw, double Yb, double YY, bool &ill) {
    const double YC = YCw - Yb * C, YS = YSw - Yb * S;
    const double CC = CCw - C * C, SS = SSw - S * S, CS = CSw - C * S;
    const double D = CC * SS - CS * CS;
    ill = !((1.0 + C * C + S * S) * (CC + SS) <= kCondMax * D) || !(D > 0.0);
    return fdiv(SS * YC * YC - 2.0 * CS * YC * YS + CC * YS * YS, D * YY);
}

// FP64 power of bin kf of object obj (before the object's scale); every lane
// of the wavefront calls it with the same (obj, kf) and gets the result.
// Standard: raw y, unit weights.  Generalized: w = dy^-2 / W and y - ybar with
// W and ybar from the statistics kernel (the power does not depend on them
// beyond rounding: the weights are normalised and the mean floats).
template <bool GEN, typename IN>
__device__ double exact_power(const SweepArgs &a, uint32_t obj, uint32_t kf) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t b = a.offsets[obj], e = a.offsets[obj + 1];
    const double f = a.fmin_rev + (double)kf * a.df_rev;
    const IN *y = static_cast<const IN *>(a.y);
    const IN *dy = static_cast<const IN *>(a.dy);
    double iW = 1.0, ybar = 0.0;
    if constexpr (GEN) {
        iW = 1.0 / a.obj_gen[kGen * obj + 4];
        ybar = a.obj_gen[kGen * obj + 3];
    }
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0, s4 = 0.0, s5 = 0.0, s6 = 0.0, s7 = 0.0, s8 = 0.0;
    for (uint64_t j = b + lane; j < e; j += 64) {
        double c, sn;
        phasor64(f, a.rec_t[j], c, sn);
        if constexpr (GEN) {
            const double dj = (double)dy[j], w = iW / (dj * dj), yc = (double)y[j] - ybar;
            const double wc = w * c, wy = w * yc;
            s0 += wc;
            s1 = fma(w, sn, s1);
            s2 = fma(wc, c, s2);
            s3 = fma(wc, sn, s3);
            s4 = fma(wy, c, s4);
            s5 = fma(wy, sn, s5);
            s6 += w;
            s7 += wy;
            s8 = fma(wy, yc, s8);
        } else {
            const double yj = (double)y[j];
            s0 = fma(yj, c, s0);
            s1 = fma(yj, sn, s1);
            s2 = fma(c, c, s2);
            s3 = fma(c, sn, s3);
        }
    }
    bool ill;
    if constexpr (GEN) {
        const double W = wave_sum(s6), iWn = 1.0 / W;
        const double C = wave_sum(s0) * iWn, S = wave_sum(s1) * iWn, CCw = wave_sum(s2) * iWn;
        const double CSw = wave_sum(s3) * iWn, YCw = wave_sum(s4) * iWn, YSw = wave_sum(s5) * iWn;
        const double Yb = wave_sum(s7) * iWn, YY = wave_sum(s8) * iWn - Yb * Yb;
        return gen_power(C, S, CCw, 1.0 - CCw, CSw, YCw, YSw, Yb, YY, ill);
    } else {
        return std_power(wave_sum(s0), wave_sum(s1), wave_sum(s2), wave_sum(s3), (double)(e - b), ill);
    }
}

// Bin of result entry v of lane (rc, kh) in a matrix-core work item.
__device__ __forceinline__ uint32_t mfma_bin(uint32_t kbase, uint32_t rc, uint32_t kh, int v) {
    return kbase + 32u * (8u * (uint32_t)(v / 4) + 4u * kh + (uint32_t)(v % 4)) + rc;
}

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr float kFacScale = 1024.0f;  // 2^10 on the column factors

// Heads and tails of two factors x: h = fp16(x), l = fp16(x - h) (x - h is
// exact in FP32).  The head must be one value.  When x is a product a b, the compiler may
// round the exact product to FP16 in one step for the tail's head
// (v_fma_mixlo_f16 h, a, b, 0) yet convert the FP32-rounded x for the packed
// MFMA operand (v_cvt_pk_f16_f32); the two roundings differ by one FP16 ulp
// in ~1 of 2^13 factors, which are then wrong by 2^-11 (seen as 4e-3 power
// errors).  Here the two heads of a pair of factors come from one packed
// conversion of their FP32 values (v_cvt_pk_f16_f32), and the tails are
// taken against those very heads (the compiler may form x - h from the exact
// product; that only makes h + l closer to it).  tests/test_split_rounding.py
// checks the built kernels for the one-step product-to-FP16 form.
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef float float2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ void split16x2(float x0, float x1, half2_t &h, half2_t &l) {
    h = __builtin_convertvector((float2_t){x0, x1}, half2_t);
    const float2_t hf = __builtin_convertvector(h, float2_t);
    l = __builtin_convertvector((float2_t){x0 - hf.x, x1 - hf.y}, half2_t);
}

// First column-factor slot of an object: the slots of object k are
// [floor(beg/16) + k, floor(beg/16) + k + ceil(N/16)), which never reach the
// next object's floor((beg + N)/16) + k + 1.
__device__ __forceinline__ uint64_t colfac_slot(uint64_t beg, uint32_t obj) { return (beg >> 4) + obj; }

// The tables are made by a wavefront per slot, whatever object it is of (the
// statistics kernel writes that down), so that a long object's blocks are made
// side by side: with wavefronts (object, one of the mean object's blocks) the
// longest object's took its several blocks, ~5 us each, one after another: 499
// objects of up to 1500 observations 50 -> 24 us, 8000 of up to 5000, coarse and
// direct tables with the marks, 480 -> 345.  Slots count from the first
// object's; false: past the last object, or between two.
__device__ __forceinline__ bool slot_block(const SweepArgs &a, uint64_t slot, uint32_t &obj, uint32_t &block) {
    const uint64_t first = a.offsets[0], last = a.offsets[a.K];
    slot += colfac_slot(first, 0u);
    if (slot >= colfac_slot(last, a.K)) return false;
    obj = a.slot_obj[slot];
    const uint64_t beg = a.offsets[obj];
    block = (uint32_t)(slot - colfac_slot(beg, obj));
    return (uint64_t)block * 16u < a.offsets[obj + 1] - beg;
}

// Heads and tails of two FP64 factors: h = fp16(fp32(x)), l = fp16(x - h),
// the remainder x - h exact in FP64 (~22 bits of x in h + l).
__device__ __forceinline__ void split64x2(double x0, double x1, half2_t &h, half2_t &l) {
    h = __builtin_convertvector((float2_t){(float)x0, (float)x1}, half2_t);
    l = __builtin_convertvector((float2_t){(float)(x0 - (double)h.x), (float)(x1 - (double)h.y)}, half2_t);
}

// The direct tile's tables of object k: wavefront y0 of gy writes the
// column-factor fragments of 16-observation blocks y0, y0 + gy, ... of the object, each factor
// as head and tail of the real and imaginary parts (a product that needs -f_i
// takes the row factor's negated fragment instead):
//   standard:    y v (4 fragments), w (4)
//   generalized: (w/W) v (4), (w/W) y_c v (4), (w/W) w (4)
// with v = e^{2 pi i b df t} (b < 32 the column) and w = v^2, from the
// caller's FP64 (or FP32) t, y, dy in FP64 arithmetic: FP64 phase and
// sin/cos, w/W = 1 / (dy^2 W) the normalised weight, y_c = y - ybar; y (or
// (w/W) y_c) scaled per object by a power of two ys, and w/W by a power of
// two ws, to a maximum in [0.5, 1) (from the statistics), then all by 2^10
// (FP16 range; the scales are undone exactly in the power); and the
// row-step fragments (e^{2 pi i 32 a df t}, row a = l % 32).  Observations
// past the object's end have zero factors.
template <bool GEN, typename IN>
__device__ __forceinline__ void direct_table(const SweepArgs &a, uint32_t k, uint32_t q) {
    constexpr int NF = GEN ? kColfacFragsGen : kColfacFragsStd;
    const uint32_t l = threadIdx.x;
    const uint64_t beg = a.offsets[k], end = a.offsets[k + 1];
    const uint32_t n = (uint32_t)(end - beg);
    const IN *y = static_cast<const IN *>(a.y);
    const IN *dy = static_cast<const IN *>(a.dy);
    double iW = 1.0, ybar = 0.0;
    if constexpr (GEN) {
        iW = 1.0 / a.obj_gen[kGen * k + 4];
        ybar = a.obj_gen[kGen * k + 3];
    }
    auto weight = [&](uint64_t i) -> double {  // w / W (1 for the standard variant)
        if constexpr (GEN) {
            const double d = (double)dy[i];
            return iW / (d * d);
        } else {
            return 1.0;
        }
    };
    auto yfac = [&](uint64_t i) -> double {  // y, or (w / W) (y - ybar)
        if constexpr (GEN) return weight(i) * ((double)y[i] - ybar);
        else return (double)y[i];
    };
    const double ys = (double)a.obj_ys[2 * k], ws = (double)a.obj_ys[2 * k + 1];
    const double sy = ys * (double)kFacScale, sw = ws * (double)kFacScale;  // exact: powers of two
    const double fb = (double)(l & 31u) * a.df_rev;
    const double fr = (double)(32u * (l & 31u)) * a.df_rev;  // row step of row l % 32
    uint4 *dst = a.colfac + colfac_slot(beg, k) * (uint64_t)(NF * 64) + l;
    uint4 *rdst = a.rowfac + colfac_slot(beg, k) * (uint64_t)(kRowfacFrags * 64) + l;
    // row-step phasors R = e^{2 pi i 32 (l % 32) df t} of observations
    // 8 (l / 32) .. + 7, in FP64 rounded to FP32 (zero past the end)
#pragma unroll
    for (int p = 0; p < kRowfacFrags; ++p) {
        float r4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const uint32_t j = q * 16u + 8u * (l >> 5) + (uint32_t)(2 * p + e);
            if (j < n) {
                double c, sn;
                phasor64(fr, a.rec_t[beg + j], c, sn);
                r4[2 * e] = (float)c;
                r4[2 * e + 1] = (float)sn;
            }
        }
        uint4 u;
        __builtin_memcpy(&u, r4, sizeof(u));
        rdst[(uint64_t)(q * kRowfacFrags + p) * 64] = u;
    }
    half8_t f[NF];
#pragma unroll
    for (int v = 0; v < 8; v += 2) {
        double x[NF / 2][2];  // the factors of observations v, v + 1: real, imaginary per sum
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const uint32_t j = q * 16u + 8u * (l >> 5) + (uint32_t)(v + e);
            double cb = 0.0, sb = 0.0, yv = 0.0, wv = 0.0;
            if (j < n) {
                phasor64(fb, a.rec_t[beg + j], cb, sb);
                yv = yfac(beg + j) * sy;
                wv = weight(beg + j) * sw;
            }
            const double wr = cb * cb - sb * sb, wi = 2.0 * cb * sb;  // v^2
            if constexpr (GEN) {
                x[0][e] = wv * cb;
                x[1][e] = wv * sb;
                x[2][e] = yv * cb;
                x[3][e] = yv * sb;
                x[4][e] = wv * wr;
                x[5][e] = wv * wi;
            } else {
                x[0][e] = yv * cb;
                x[1][e] = yv * sb;
                x[2][e] = wv * wr;
                x[3][e] = wv * wi;
            }
        }
#pragma unroll
        for (int p = 0; p < NF / 4; ++p) {  // each complex factor: r (h, l), i (h, l)
            half2_t h, t;
            split64x2(x[2 * p][0], x[2 * p][1], h, t);
            f[4 * p + 0][v] = h.x; f[4 * p + 0][v + 1] = h.y;
            f[4 * p + 1][v] = t.x; f[4 * p + 1][v + 1] = t.y;
            split64x2(x[2 * p + 1][0], x[2 * p + 1][1], h, t);
            f[4 * p + 2][v] = h.x; f[4 * p + 2][v + 1] = h.y;
            f[4 * p + 3][v] = t.x; f[4 * p + 3][v + 1] = t.y;
        }
    }
#pragma unroll
    for (int i = 0; i < NF; ++i) {
        uint4 u;
        __builtin_memcpy(&u, &f[i], sizeof(u));
        dst[(uint64_t)(q * NF + i) * 64] = u;
    }
}

__device__ __forceinline__ half8_t neg8(half8_t x) {
    uint4 u;
    __builtin_memcpy(&u, &x, sizeof(u));
    u.x ^= 0x80008000u;
    u.y ^= 0x80008000u;
    u.z ^= 0x80008000u;
    u.w ^= 0x80008000u;
    __builtin_memcpy(&x, &u, sizeof(u));
    return x;
}

// Loads the row-step fragments of one 16-observation block.
__device__ __forceinline__ void load_rows(const uint4 *rf, uint4 (&rr)[kRowfacFrags]) {
#pragma unroll
    for (int i = 0; i < kRowfacFrags; ++i) rr[i] = rf[i * 64];
}

// Loads the column-factor fragments of one 16-observation block.
template <int NF>
__device__ __forceinline__ void load_cols(const uint4 *cf, half8_t (&col)[NF]) {
#pragma unroll
    for (int i = 0; i < NF; ++i) {
        const uint4 u = cf[i * 64];
        __builtin_memcpy(&col[i], &u, sizeof(u));
    }
}

// Work items of the direct matrix-core tiles: the sweep's; or, beside the
// coarse-grid sweep, two kinds of workgroups.  The first a.marked_groups take
// the marked chunks of the objects in coarse mode, workgroup r of an object
// every cand_split-th, an object's workgroups on one XCD (its tables are then
// fetched once and found in the L2: 0.46 -> 0.15 ms for 1000 generalized
// objects).  The others take the groups of the objects in direct mode, in the
// grid schedule's order; the launch has a workgroup for every group that there
// could be, and those past the list's end, which only the device knows, leave
// at once; or, with a queue, as many workgroups as fill the chip drain it.  (In
// the grid's place, where all objects are direct, standard, 4000 x 100,000 bins,
// 4.53 ms with the plain grid: workgroups that stay on the chip and stride over
// the groups 5.9, the persistent queues 4.9, groups of eight items 4.8.)
__device__ __forceinline__ uint64_t cand_item(const SweepArgs &a, uint32_t obj, uint32_t from, uint32_t skip) {
    const uint64_t *bits = a.cand + (uint64_t)obj * a.cand_words;
    for (uint32_t w = from >> 6; w < a.cand_words; ++w) {
        uint64_t b = bits[w];
        if (w == from >> 6) b &= ~0ull << (from & 63u);
        for (; b; b &= b - 1u, --skip)
            if (skip == 0u) return (uint64_t)obj * a.chunks + 64u * w + (uint32_t)__builtin_ctzll(b);
    }
    return ~0ull;
}
__device__ __forceinline__ uint64_t direct_first(SweepArgs &a, uint64_t *s_item) {
    if (!a.obj_ip) return first_item(a, s_item);
    if (blockIdx.x >= a.marked_groups) {
        a.cand = nullptr;
        a.order = a.direct_list;
        a.total_items = (uint64_t)*a.direct_count * a.chunks;
        if (a.queue) return fetch_item(a, s_item, true);
        const uint64_t groups = (a.total_items + a.group - 1u) / a.group, w = a.item_base + blockIdx.x - a.marked_groups;
        if (w >= groups) return ~0ull;
        a.item_base = 0;
        return xcd_group(w, groups, a.xcd_run) * a.group;
    }
    const uint32_t g = (uint32_t)xcd_group(blockIdx.x, a.marked_groups, a.cand_split);
    const uint32_t pos = g / a.cand_split, r = g - pos * a.cand_split;
    if (pos >= a.K) return ~0ull;
    const uint32_t obj = a.order ? a.order[pos] : pos;
    a.order = nullptr;  // the items name the object itself
    a.queue = nullptr;
    return a.obj_ip[obj].mode ? cand_item(a, obj, 0u, r) : ~0ull;
}
__device__ __forceinline__ uint64_t direct_next(const SweepArgs &a, uint64_t *s_item, uint64_t item) {
    if (!a.cand) return next_item(a, s_item, item);
    const uint32_t obj = (uint32_t)(item / a.chunks);
    return cand_item(a, obj, (uint32_t)(item - (uint64_t)obj * a.chunks) + 1u, a.cand_split - 1u);
}

#define LS_MFMA(ACC, A, B) ACC = __builtin_amdgcn_mfma_f32_32x32x16_f16(A, B, ACC, 0, 0, 0)
}  // namespace

}  // namespace lsamd
