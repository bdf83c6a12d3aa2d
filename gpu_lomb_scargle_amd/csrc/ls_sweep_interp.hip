// Coarse-grid form of the split32 sweep (matrix cores), its per-object tables
// and the selection of the chunks that can hold an object's best bins.
//
// A frequency grid finer than an object's resolution 1/T (T its time span)
// holds no more information than a coarse one: Z(f) = sum_j a_j e^{2 pi i f t_j}
// with |t_j| <= T/2 is band-limited.  The sums are therefore formed directly
// only on a grid of step h bins, and every bin follows by interpolation,
//   Z(f_b) = sum_m phi(b/h - m) G_m,  G_m = sum_j a_j / Phi(h df t_j) e^{2 pi i f_m t_j},
// phi the Kaiser-Bessel window of W taps (Kaiser & Kuo 1966; the standard
// window of nonuniform FFTs) and Phi its Fourier transform, so that the only
// error is the window's aliasing, e^{-pi W sqrt(1 - 1/sigma)} at an
// oversampling sigma = 1/(h df T).  Per bin and observation this leaves 3/h
// complex products (standard: Z1 at f, and the weights' sum X at 2 f, which
// has twice the coarse points) or 4/h (generalized: X at f too) instead of 2
// or 3; the interpolation itself is a matrix product with a constant 16-point
// (or 32-point) operand, on the matrix cores as well.
//
// FP32 periodograms, measured (top-1, ms of the whole sweep, direct -> coarse):
// 1000 objects (164,000 observations) x 10^6 bins, standard, 23 bins per
// resolution element, h = 10: 10.5 -> 2.75; 250 objects (42,700) x 429,119,
// generalized, ten bins, h = 4: 2.0 -> 0.68.  k_sweep_interp takes 2.55 ms of
// the first: a third the coarse points, the rest the interpolation and the
// FP64 powers (22 FP64 instructions per bin; VALU 58% and matrix cores 16% of
// the SIMD cycles at 2.0 GHz), the stores 0.2 and the bins past the condition
// bound 0.04.  Tried on the way: points of one sign per row factor (3.47 ms:
// twice the MFMAs and row factors), three wavefronts per standard workgroup
// (2.99: six wavefronts fit a CU instead of eight), a branch per bin around
// the store (its FP64 chains then run one after another: 5.1 against 4.5).
//
// Peaks without a periodogram (SCREEN): the powers only choose which chunks of
// 1024 bins the direct tile sweeps, so FP16 heads alone, six taps, larger
// steps and FP32 powers do: the powers near the peak are good to 7e-3 at worst
// (17 observations of uneven weight), 1e-3 typically, against a margin of
// 1/8; where an object's peak does not stand clear of the sums' rounding, all its
// chunks are marked (mark_chunks).  The results are the direct sums', bit for bit.  Measured: 8000 uneven
// objects x 200,000 bins, top-3, standard FP64, 4.7 bins per resolution
// element, h = 3: 13.1 -> 4.8 ms (screen 3.0, the marked chunks and the objects
// of at most 16 observations 1.45, tables 0.35); 1000 objects x 500,000,
// generalized, 10.5 bins, h = 8: 11.2 -> 1.2 ms.
#include <type_traits>

#include "ls_split_device.h"

#include "ls_interp.h"

namespace lsamd {

namespace {

// ---------------------------------------------------------------------------
// Interpolation operands: fragment f of mode q at [(6 q + f) 64 + lane], the
// MFMA B operand phi[k][b] (lane: column b = lane % 32, rows k = 8 (lane / 32)
// .. +7) times 2^10, as FP16 head and tail: f = 0, 1 for sums at f (position
// b/h), 2, 3 and 4, 5 for rows 0..15 and 16..31 at 2 f (position 2b/h).  Row k
// of a result row whose window starts at coarse point m0 multiplies G[m0 + k]:
// phi((position) - (k - W/2 + 1)), zero outside the window.
// ---------------------------------------------------------------------------
__device__ double bessel_i0(double x) {  // power series, 0 <= x < 20
    const double q = 0.25 * x * x;
    double term = 1.0, sum = 1.0;
#pragma unroll
    for (int k = 1; k < 48; ++k) {
        term *= q * (1.0 / (double)(k * k));
        sum += term;
    }
    return sum;
}

template <bool SCREEN>
__device__ void interp_table(uint4 *tab, int mode, int f) {  // f: sums at f; at 2 f, rows 0..15; 16..31
    const int lane = (int)threadIdx.x;
    const int h = ip_step(mode), W = ip_taps(SCREEN);
    const double beta = ip_beta(SCREEN);
    // phi(x) = I0(beta sqrt(1 - (2x/W)^2)) / Phi(0), Phi(0) = W sinh(beta) / beta
    const double norm = 1024.0 * beta / ((double)W * sinh(beta));
    const double pos = (f == 0 ? 1.0 : 2.0) * (double)(lane & 31) / (double)h;
    half8_t hd = {}, tl = {};
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
        double x[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int k = 8 * (lane >> 5) + i + e + (f == 2 ? 16 : 0);
            const double u = 2.0 * (pos - (double)(k - W / 2 + 1)) / (double)W, r = 1.0 - u * u;
            x[e] = r >= 0.0 ? norm * bessel_i0(beta * sqrt(r)) : 0.0;
        }
        half2_t a, b;
        split64x2(x[0], x[1], a, b);
        hd[i] = a.x; hd[i + 1] = a.y;
        tl[i] = b.x; tl[i + 1] = b.y;
    }
    uint4 u;
    uint4 *dst = tab + ((mode - 1) * 6 + 2 * f) * 64 + lane;
    __builtin_memcpy(&u, &hd, sizeof(u));
    dst[0] = u;
    __builtin_memcpy(&u, &tl, sizeof(u));
    dst[64] = u;
}

// e^{2 pi i f t} from the FP64 phase: in FP64, or (screen) by the hardware FP32
// sine and cosine (1e-7, below the FP16 heads' 5e-4).
template <bool SCREEN>
__device__ __forceinline__ void ip_phasor(double f, double t, double &c, double &s) {
    if constexpr (SCREEN) {
        const double n = __builtin_rint(f * t);
        const float r = (float)fma(f, t, -n);
        c = (double)__builtin_amdgcn_cosf(r);
        s = (double)__builtin_amdgcn_sinf(r);
    } else {
        phasor64(f, t, c, s);
    }
}

// The objects in direct mode, in processing order, and their number (one
// wavefront; 512 objects' modes in flight).
__device__ void list_direct(const SweepArgs &a) {
    const uint32_t lane = threadIdx.x;
    uint32_t count = 0;
    for (uint32_t base = 0; base < a.K; base += 512u) {
        uint32_t obj[8], mode[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const uint32_t pos = base + 64u * (uint32_t)q + lane;
            obj[q] = pos < a.K ? (a.order ? a.order[pos] : pos) : 0u;
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) mode[q] = base + 64u * (uint32_t)q + lane < a.K ? a.obj_ip[obj[q]].mode : 1u;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const uint64_t direct = __ballot(mode[q] == 0u);
            if (mode[q] == 0u) a.direct_list[count + (uint32_t)__popcll(direct & ((1ull << lane) - 1ull))] = obj[q];
            count += (uint32_t)__popcll(direct);
        }
    }
    if (lane == 0) *a.direct_count = count;
    if (lane < kQueues) a.queue[lane * kQueueStride] = 0ull;
}

// The first workgroups list the objects in direct mode (blockIdx.x = 0) and
// write the interpolation operands (1 + 3 (mode - 1) + which third).  The others
// write the tables of a slot's 16 observations, as k_colfac does for the direct
// tile, into the same slots (objects in direct mode: the direct tile's
// themselves): column factors e^{2 pi i (b + 1/2) h df t'} a / Phi (b < 32) of the
// two weights a = y (generalized: (w/W) (y - ybar)) and a = 1 (w/W), four head
// and tail fragments each, and the row steps e^{2 pi i 64 a h df t'} (a < 32),
// with t' = t - tc and 1/Phi from the records.
template <bool GEN, typename IN, bool SCREEN>
__global__ __launch_bounds__(64) void k_interp_fac(SweepArgs a) {
    constexpr int FR = ip_frags(SCREEN), NC = SCREEN ? 1 : 2;  // fragments; heads alone or with tails
    const uint32_t l = threadIdx.x;
    if (blockIdx.x == 0) return list_direct(a);
    if (blockIdx.x <= 3u * kIpModes)
        return interp_table<SCREEN>(a.ip_tab, (int)(blockIdx.x - 1u) / 3 + 1, (int)(blockIdx.x - 1u) % 3);
    uint32_t k, q;
    if (!slot_block(a, blockIdx.x - 1u - 3u * kIpModes, k, q)) return;
    const int mode = (int)a.obj_ip[k].mode;
    if (mode == 0) return direct_table<GEN, IN>(a, k, q);
    const uint64_t beg = a.offsets[k], end = a.offsets[k + 1];
    const uint32_t n = (uint32_t)(end - beg);
    const IN *y = static_cast<const IN *>(a.y);
    const IN *dy = static_cast<const IN *>(a.dy);
    double iW = 1.0, ybar = 0.0;
    if constexpr (GEN) {
        iW = 1.0 / a.obj_gen[kGen * k + 4];
        ybar = a.obj_gen[kGen * k + 3];
    }
    const double sy = (double)a.obj_ys[2 * k] * (double)kFacScale, sw = (double)a.obj_ys[2 * k + 1] * (double)kFacScale;
    const double step = (double)ip_step(mode) * a.df_rev;
    const double fb = ((double)(l & 31u) + 0.5) * step, fr = (double)(64u * (l & 31u)) * step;
    constexpr int NF = GEN ? kColfacFragsGen : kColfacFragsStd;
    uint4 *dst = a.colfac + colfac_slot(beg, k) * (uint64_t)(NF * 64) + l;
    uint4 *rdst = a.rowfac + colfac_slot(beg, k) * (uint64_t)(kRowfacFrags * 64) + l;
    half8_t f[FR];
#pragma unroll
    for (int v = 0; v < 8; v += 2) {
        double x[4][2];
        float r4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const uint32_t j = q * 16u + 8u * (l >> 5) + (uint32_t)(v + e);
            double cb = 0.0, sb = 0.0, yv = 0.0, wv = 0.0;
            if (j < n) {
                const double2 tp = a.rec_r[beg + j];  // t', 1/Phi
                double c, sn;
                ip_phasor<SCREEN>(fr, tp.x, c, sn);
                r4[2 * e] = (float)c;
                r4[2 * e + 1] = (float)sn;
                ip_phasor<SCREEN>(fb, tp.x, cb, sb);
                double w = 1.0, yj = (double)y[beg + j];
                if constexpr (GEN) {
                    const double d = (double)dy[beg + j];
                    w = iW / (d * d);
                    yj = w * (yj - ybar);
                }
                yv = yj * sy * tp.y;
                wv = w * sw * tp.y;
            }
            x[0][e] = yv * cb;
            x[1][e] = yv * sb;
            x[2][e] = wv * cb;
            x[3][e] = wv * sb;
        }
        uint4 u;
        __builtin_memcpy(&u, r4, sizeof(u));
        rdst[(uint64_t)(q * kRowfacFrags + (uint32_t)(v >> 1)) * 64] = u;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            half2_t hd, tl;
            split64x2(x[p][0], x[p][1], hd, tl);
            f[NC * p][v] = hd.x; f[NC * p][v + 1] = hd.y;
            if constexpr (!SCREEN) {
                f[2 * p + 1][v] = tl.x; f[2 * p + 1][v + 1] = tl.y;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < FR; ++i) {
        uint4 u;
        __builtin_memcpy(&u, &f[i], sizeof(u));
        dst[(uint64_t)(q * FR + i) * 64] = u;
    }
}

// Row factors u = u0 R of a 16-observation block (as row_factors, without u^2).
struct UnitFrags {
    half8_t r_h, r_l, i_h, i_l;
};
template <bool SCREEN>
__device__ __forceinline__ void unit_factors(const float2 *s_u0, uint32_t j0, uint32_t kh,
                                             const uint4 (&rr)[kRowfacFrags], UnitFrags &R) {
#pragma unroll
    for (int v = 0; v < 8; v += 2) {
        const uint4 r = rr[v >> 1];
        const float rx[2] = {__uint_as_float(r.x), __uint_as_float(r.z)};
        const float ry[2] = {__uint_as_float(r.y), __uint_as_float(r.w)};
        float ur[2], ui[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float2 b = s_u0[j0 + 8u * kh + (uint32_t)(v + e)];
            ur[e] = fmaf(b.x, rx[e], -(b.y * ry[e]));
            ui[e] = fmaf(b.x, ry[e], b.y * rx[e]);
        }
        half2_t h, t;
        if constexpr (SCREEN) {
            h = __builtin_convertvector((float2_t){ur[0], ur[1]}, half2_t);
            R.r_h[v] = h.x; R.r_h[v + 1] = h.y;
            h = __builtin_convertvector((float2_t){ui[0], ui[1]}, half2_t);
            R.i_h[v] = h.x; R.i_h[v + 1] = h.y;
            continue;
        }
        split16x2(ur[0], ur[1], h, t);
        R.r_h[v] = h.x; R.r_h[v + 1] = h.y;
        R.r_l[v] = t.x; R.r_l[v + 1] = t.y;
        split16x2(ui[0], ui[1], h, t);
        R.i_h[v] = h.x; R.i_h[v + 1] = h.y;
        R.i_l[v] = t.x; R.i_l[v + 1] = t.y;
    }
}

// A value that is the same in all lanes, held in scalar registers.
__device__ __forceinline__ double uniform(double v) { return lane_value(v, 0); }
__device__ __forceinline__ float uniform(float v) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// Orders a wavefront's LDS writes before its own later reads (LDS operations
// of one wavefront complete in order; this only holds the compiler).
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Maximum over the wavefront's lanes (each >= 0), the same in all: DPP row
// shifts and broadcasts, lane 63's result.
__device__ __forceinline__ float wave_fmax(float x) {
    auto step = [&](auto ctrl, int rows) {
        const int o = rows == 0xf ? __builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(ctrl)::value, 0xf, 0xf, true)
                    : rows == 0xa ? __builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(ctrl)::value, 0xa, 0xf, true)
                                  : __builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(ctrl)::value, 0xc, 0xf, true);
        x = fmaxf(x, __int_as_float(o));
    };
    step(std::integral_constant<int, 0x111>{}, 0xf);  // row_shr 1, 2, 4, 8
    step(std::integral_constant<int, 0x112>{}, 0xf);
    step(std::integral_constant<int, 0x114>{}, 0xf);
    step(std::integral_constant<int, 0x118>{}, 0xf);
    step(std::integral_constant<int, 0x142>{}, 0xa);  // row_bcast 15, 31
    step(std::integral_constant<int, 0x143>{}, 0xc);
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}

// ---------------------------------------------------------------------------
// The sweep of the objects in coarse mode.  A workgroup takes rows x rb bins
// of one object (8160 to 32640), rb = h m bins per result row.  Its wavefronts
// form 2048 consecutive coarse points each: wavefront 0 of the y sum at f,
// (generalized: 1 of the weights' sum at f,) the last two of the weights' sum
// at 2 f, which spans twice as many.  The points are 32 rows of 64, at
// f_a -+ (b + 1/2) h df, b < 32: the weights are real, so the columns of the
// two signs are conjugates, and with row factor u and column factor c the four
// real sums
//   A = sum u_r c_r,  B = sum u_i c_i,  C = sum u_r c_i,  D = sum u_i c_r
// give both points, (A - B) + i (C + D) at +b and (A + B) + i (D - C) at -b: 12
// MFMAs and one set of row factors per 16 observations and 2048 points, where
// a direct block takes 12 per 1024.  The points go to LDS as FP16 heads and tails; then
// the wavefronts share the result tiles of 32 rows x 32 columns (row s, bin
// rb s + b): A = the points m s .. m s + 15 (of the sums at 2 f 2 m s .. + 31
// when a row spans more than 16), B = the table, three products each.  The
// power, the condition bound and its FP64 recomputation are the direct tile's.
// ---------------------------------------------------------------------------
template <bool GEN, typename IN, bool SCREEN>
__global__ __launch_bounds__(256, SCREEN ? 3 : 2) void k_sweep_interp(SweepArgs a) {
    static_assert(SCREEN || sizeof(IN) == 4, "periodograms: FP32");
    constexpr int NC = SCREEN ? 1 : 2, FR = ip_frags(SCREEN);
    constexpr int NW = 4, NZ = GEN ? 2 : 1;
    constexpr uint32_t kFoldObs = 256;
    constexpr int kZ = (int)kIpPoints, kX = (int)kIpPoints2;
    __shared__ float2 s_u0[NW][64];
    __shared__ __align__(16) _Float16 s_z[NZ][2][NC][kZ];  // [sum][re, im][head, tail]
    __shared__ __align__(16) _Float16 s_x[2][NC][kX];
    const uint32_t l = threadIdx.x & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint64_t g = a.item_base + grid_group(a);
    const uint32_t per_obj = (a.ip_items + a.group - 1u) / a.group;  // workgroups
    const uint32_t pos = (uint32_t)(g / per_obj), it0 = (uint32_t)(g - (uint64_t)pos * per_obj) * a.group;
    if (pos >= a.K) return;
    const uint32_t obj = a.order ? a.order[pos] : pos;
    const int mode = (int)a.obj_ip[obj].mode;
    if (mode == 0) return;
    const uint32_t h = (uint32_t)ip_step(mode), m = (uint32_t)ip_per_row(mode), rb = h * m;
    const uint32_t rows = (uint32_t)ip_rows(mode);
    if ((uint64_t)it0 * (rows * rb) >= a.nf) return;
    constexpr int W = ip_taps(SCREEN);

    const uint64_t obeg = a.offsets[obj], oend = a.offsets[obj + 1];
    const uint32_t n = (uint32_t)(oend - obeg);
    const float ys = a.obj_ys[2 * obj], ws = a.obj_ys[2 * obj + 1];
    // |G| <= n max(1/Phi) 2^10 into FP16's range
    const float gs = ip_point_scale(SCREEN, n);
    const bool at2f = wave >= (uint32_t)NZ;
    const bool wide = ip_wide(SCREEN, mode);
    const double un = 1.0 / ((double)kFacScale * 1024.0 * (double)gs);  // power of two
    const double uy = un / (double)ys, uw = un / (double)ws;
    const double scale = a.obj_scale[obj];
    // The powers from the unscaled results.  Standard, with c + i s = X / 2 and
    // CC = N/2 + c, SS = N/2 - c, CS = s:
    //   P = (N/2 |Z|^2 - c Re Z^2 - s Im Z^2) / (2 (N^2/4 - c^2 - s^2)),
    // all in units of X's result (u = uw / 2): N/2 = hn u, P scaled by kp (the
    // screen's ranks: in units of ip_rank_unit = uy^2 / (2 u)).
    const double nobs = (double)n, u = 0.5 * uw, hn = 0.5 * nobs / u, hn2 = hn * hn;
    const double dmin = nobs * nobs / (4.0 * kCondMax) / (u * u), kp = SCREEN ? 1.0 : 0.5 * uy * uy / u * scale;
    const double ke = SCREEN && !GEN ? 1.0 / ip_rank_unit((double)ys, (double)ws, n) : scale;  // of the powers computed again
    double Wf = 1.0, Yb = 0.0, YY = 1.0;
    if constexpr (GEN) {
        Wf = a.obj_gen[kGen * obj + 5];
        Yb = a.obj_gen[kGen * obj + 6];
        YY = a.obj_gen[kGen * obj + 7];
    }
    // generalized: gen_power with y in units of its result
    const double iW = 1.0 / Wf, sw = uw * iW, sy = uy * iW, hsw = 0.5 * sw, ybu = Yb / sy, kg = sy * sy / YY * scale;
    typedef std::conditional_t<SCREEN, float, double> R;
    const R rsw = uniform((R)sw), rhsw = uniform((R)hsw), rybu = uniform((R)ybu), rkg = uniform((R)kg);
    const R rhn = uniform((R)hn), rhn2 = uniform((R)hn2), rdmin = uniform((R)dmin), rkp = uniform((R)kp);
    const R rcond = (R)kCondMax;
    // a.group workgroups' worths of bins in turn (ip_grouped), the object's
    // constants and addresses stay
    auto sweep_item = [&](const uint32_t it, const uint32_t l) {
    const uint32_t rc = l & 31u, kh = l >> 5;
    const uint32_t kbase = it * (rows * rb);
    if (GEN || wave < 3u) {
        const double step = (double)h * a.df_rev;
        double f0 = a.fmin_rev + (double)kbase * a.df_rev;
        if (at2f) f0 = 2.0 * f0 + (wave > (uint32_t)NZ ? 2048.0 * step : 0.0);
        f0 += (31.5 - (double)(W / 2 - 1)) * step;  // the first row's middle
        constexpr int NF = GEN ? kColfacFragsGen : kColfacFragsStd;
        const uint64_t slot = colfac_slot(obeg, obj);
        const uint4 *cf = a.colfac + slot * (uint64_t)(NF * 64) + (wave == 0 ? 0 : FR / 2 * 64) + l;
        const uint4 *rf = a.rowfac + slot * (uint64_t)(kRowfacFrags * 64) + l;
        f32x16_t sum[4] = {}, cross[SCREEN ? 1 : 4] = {};  // A, B, C, D: head x head, cross products
        // sums of whole 256-observation runs, in the room of this wavefront's
        // points: entry i of lane l, each lane its own
        _Float16 *const base = at2f ? &s_x[0][0][0] + 2048u * (wave - NZ) : &s_z[wave < NZ ? wave : 0][0][0][0];
        const uint32_t len = at2f ? kX : kZ;
        auto run_sum = [&](int q, int v) { return reinterpret_cast<float *>(base + (uint32_t)q * len) + 64 * v + l; };
        constexpr bool kRuns = !SCREEN;  // the screen's sums stay in the accumulators
        bool folded = false;
        uint4 rr[kRowfacFrags];
        load_rows(rf, rr);
        half8_t next[FR / 2];
        if constexpr (SCREEN) load_cols<FR / 2>(cf, next);
        for (uint32_t g0 = 0; g0 < n; g0 += kRuns ? kFoldObs : n) {
            const uint32_t gend = !kRuns || n - g0 < kFoldObs ? n : g0 + kFoldObs;
            for (uint32_t b0 = g0; b0 < gend; b0 += 64) {
                const uint32_t cnt = gend - b0 < 64u ? gend - b0 : 64u;
                float2 u0 = make_float2(0.0f, 0.0f);
                if (l < cnt) {
                    double c, sn;
                    ip_phasor<SCREEN>(f0, a.rec_r[obeg + b0 + l].x, c, sn);
                    u0 = make_float2((float)c, (float)sn);
                }
                wave_lds_fence();
                s_u0[wave][l] = u0;
                wave_lds_fence();
                for (uint32_t j0 = 0; j0 < cnt; j0 += 16, cf += FR * 64, rf += kRowfacFrags * 64) {
                    half8_t col[FR / 2];
                    if constexpr (SCREEN) {  // one block ahead, as the rows
#pragma unroll
                        for (int i = 0; i < FR / 2; ++i) col[i] = next[i];
                        load_cols<FR / 2>(cf + FR * 64, next);
                    } else {
                        load_cols<FR / 2>(cf, col);
                    }
                    UnitFrags R;
                    unit_factors<SCREEN>(s_u0[wave], j0, kh, rr, R);
                    load_rows(rf + kRowfacFrags * 64, rr);  // the next block's (one slot past the end is allocated)
                    if constexpr (SCREEN) {
                        LS_MFMA(sum[0], R.r_h, col[0]);
                        LS_MFMA(sum[1], R.i_h, col[1]);
                        LS_MFMA(sum[2], R.r_h, col[1]);
                        LS_MFMA(sum[3], R.i_h, col[0]);
                    } else {
                        LS_MFMA(sum[0], R.r_h, col[0]);
                        LS_MFMA(cross[0], R.r_h, col[1]);
                        LS_MFMA(cross[0], R.r_l, col[0]);
                        LS_MFMA(sum[2], R.r_h, col[2]);
                        LS_MFMA(cross[2], R.r_h, col[3]);
                        LS_MFMA(cross[2], R.r_l, col[2]);
                        LS_MFMA(sum[1], R.i_h, col[2]);
                        LS_MFMA(cross[1], R.i_h, col[3]);
                        LS_MFMA(cross[1], R.i_l, col[2]);
                        LS_MFMA(sum[3], R.i_h, col[0]);
                        LS_MFMA(cross[3], R.i_h, col[1]);
                        LS_MFMA(cross[3], R.i_l, col[0]);
                    }
                }
            }
            if constexpr (kRuns) {
                if (gend < n) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            float *r = run_sum(q, v);
                            *r = (folded ? *r : 0.0f) + (sum[q][v] + cross[q][v]);
                        }
                        sum[q] = f32x16_t{};
                        cross[q] = f32x16_t{};
                    }
                    folded = true;
                }
            }
        }
        if constexpr (kRuns) {
#pragma unroll
            for (int q = 0; q < 4; ++q) sum[q] += cross[q];
            if (folded) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int v = 0; v < 16; ++v) sum[q][v] += *run_sum(q, v);
                wave_lds_fence();  // all read before the points overwrite them
            }
        }
        if (SCREEN && it != it0) __syncthreads();  // the last tiles' points are read
#pragma unroll
        for (int v = 0; v < 16; v += 2) {
            // row 8 (v / 4) + 4 kh + v % 4, point 64 row + 32 + b and 64 row + 31 - b; v + 1: 64 on
            const uint32_t ip = 64u * (8u * (uint32_t)(v / 4) + 4u * kh + (uint32_t)(v % 4)) + 32u + rc, im = ip - 1u - 2u * rc;
            half2_t hd, tl;
            auto put = [&](int c, uint32_t at, float x0, float x1) {
                if constexpr (SCREEN) hd = __builtin_convertvector((float2_t){x0 * gs, x1 * gs}, half2_t);
                else split16x2(x0 * gs, x1 * gs, hd, tl);
                base[NC * c * len + at] = hd.x; base[NC * c * len + at + 64] = hd.y;
                if constexpr (!SCREEN) {
                    base[(2 * c + 1) * len + at] = tl.x; base[(2 * c + 1) * len + at + 64] = tl.y;
                }
            };
            put(0, ip, sum[0][v] - sum[1][v], sum[0][v + 1] - sum[1][v + 1]);
            put(1, ip, sum[2][v] + sum[3][v], sum[2][v + 1] + sum[3][v + 1]);
            put(0, im, sum[0][v] + sum[1][v], sum[0][v + 1] + sum[1][v + 1]);
            put(1, im, sum[3][v] - sum[2][v], sum[3][v + 1] - sum[2][v + 1]);
        }
        if (l < 32) {  // zeros past the last point (a window's unused rows meet them with weight 0)
            if (wave < (uint32_t)NZ) {
#pragma unroll
                for (int c = 0; c < 2 * NC; ++c) base[c * kZ + 2048 + l] = (_Float16)0.0f;
            } else if (wave == (uint32_t)NZ) {
#pragma unroll
                for (int c = 0; c < 2 * NC; ++c) base[c * kX + 4096 + l] = (_Float16)0.0f;
            }
        }
    } else if (SCREEN && it != it0) {
        __syncthreads();  // as the other wavefronts, before their points
    }
    // the table's operands (fragments 4, 5: rows 16..31 of the sums at 2 f)
    half8_t tb[6];
#pragma unroll
    for (int i = 0; i < 6; i += SCREEN ? 2 : 1) {  // (the screen uses the heads)
        const uint4 u = a.ip_tab[((mode - 1) * 6 + i) * 64 + (int)l];
        __builtin_memcpy(&tb[i], &u, sizeof(u));
    }
    __syncthreads();
    float *tmax = reinterpret_cast<float *>(a.part_pow + (uint64_t)obj * a.chunks * kPeaks) + 3u * it * ((rows + 31u) / 32u);
    const uint32_t left = a.nf - kbase;
    const uint32_t rows_here = left < rows * rb ? (left + rb - 1u) / rb : rows;
    // Stores past the workgroup's bins (rows of the next one, the grid's end,
    // lanes beyond rb) are dropped by the buffer's range: no branch per bin, so
    // that the bins' FP64 chains overlap.
    const uint32_t bin_end = left < rows * rb ? a.nf : kbase + rows * rb;
    float *pg = SCREEN ? nullptr : static_cast<float *>(a.pgram) + (uint64_t)obj * a.nf;
    const auto out = __builtin_amdgcn_make_buffer_rsrc(pg, 0, (int)(bin_end * 4u), 0x00027000);

    for (uint32_t tile = wave; 32u * tile < rows_here; tile += NW) {
        const uint32_t s = ip_operand_row(rows, tile, rc);  // this lane's row of the A operand
        f32x16_t z[2 * NZ], x[2];
        auto product = [&](const _Float16 *gh, const _Float16 *gt, const half8_t &th, const half8_t &tt, f32x16_t &acc) {
            half8_t ah, at;
            __builtin_memcpy(&ah, __builtin_assume_aligned(gh, 2), 16);
            if constexpr (!SCREEN) {
                __builtin_memcpy(&at, __builtin_assume_aligned(gt, 2), 16);
                LS_MFMA(acc, at, th);
                LS_MFMA(acc, ah, tt);
            }
            LS_MFMA(acc, ah, th);
        };
        const uint32_t zo = m * s + 8u * kh, xo = 2u * m * s + 8u * kh;
#pragma unroll
        for (int q = 0; q < NZ; ++q)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                z[2 * q + c] = f32x16_t{};
                product(&s_z[q][c][0][zo], &s_z[q][c][NC - 1][zo], tb[0], tb[1], z[2 * q + c]);
            }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            x[c] = f32x16_t{};
            product(&s_x[c][0][xo], &s_x[c][NC - 1][xo], tb[2], tb[3], x[c]);
            if (wide) product(&s_x[c][0][xo + 16], &s_x[c][NC - 1][xo + 16], tb[4], tb[5], x[c]);
        }
        // result entry v: row 8 (v / 4) + 4 kh + v % 4 of the tile, bin rb row + rc
        const uint32_t bin0 = kbase + rb * (32u * tile + 4u * kh) + rc;
        const uint32_t off0 = rc < rb ? bin0 : 0x3FFF0000u;  // past any bin_end (nf < kIpMaxFreqs)
        // power of entry v, and whether its condition number exceeds the bound
        // (the screen's in FP32: a few 1e-6 beside the heads' ~1e-3)
        auto fm = [](R p, R q, R r) {
            if constexpr (SCREEN) return fmaf(p, q, r);
            else return fma(p, q, r);
        };
        auto power = [&](int v, bool &ill) -> float {
            R num, D;
            if constexpr (GEN) {
                const R C = (R)z[2][v] * rsw, S = (R)z[3][v] * rsw;
                const R half = fm((R)x[0][v], rhsw, (R)0.5);
                const R CC = fm(-C, C, half), SS = fm(-S, S, (R)1.0 - half);
                const R CS = fm(-C, S, (R)x[1][v] * rhsw);
                const R yc = fm(-rybu, C, (R)z[0][v]), ysn = fm(-rybu, S, (R)z[1][v]);
                D = fm(CC, SS, -(CS * CS));
                const R t = fm(C, C, S * S);  // (1 + t) (CC + SS) = 1 - t^2
                ill = !(fm(-t, t, (R)1.0) <= rcond * D) | !(D > (R)0.0);
                num = rkg * fm(SS, yc * yc, fm(CC, ysn * ysn, (R)-2.0 * CS * (yc * ysn)));
            } else {
                const R XC = (R)z[0][v], XS = (R)z[1][v], c = (R)x[0][v], sn = (R)x[1][v];
                D = fm(-c, c, fm(-sn, sn, rhn2));
                ill = !(D >= rdmin);
                const R q = XC * XC;
                num = fm(rhn, fm(XS, XS, q), -fm(c, fm(-XS, XS, q), (sn + sn) * (XC * XS)));
                if constexpr (!SCREEN) num *= rkp;
            }
            if constexpr (SCREEN) return num * __builtin_amdgcn_rcpf(D);
            else {
                // num / D, the hardware reciprocal's error e taken off to third order
                const double r = __builtin_amdgcn_rcp(D), e = fma(-D, r, 1.0);
                return (float)(num * fma(r, fma(e, e, e), r));
            }
        };
        float best = 0.0f, pw[16];
        uint64_t any_ill = 0u, ills[16];  // lanes of entry v past the condition bound (scalar registers)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const uint32_t kf = off0 + rb * (8u * (uint32_t)(v / 4) + (uint32_t)(v % 4));
            bool ill;
            pw[v] = power(v, ill);
            if constexpr (!SCREEN) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(pw[v]), out, kf * 4u, 0, 0);
            best = fmaxf(best, pw[v]);
            ills[v] = __ballot(ill);
            any_ill |= ills[v];
        }
        best = rc < rb ? best : 0.0f;
        // rarely: bins past the condition bound, or a tile that the workgroup's
        // last row or the grid's end cuts (whose other entries count for nothing)
        uint32_t flags = 0u;
        if (kbase + rb * (32u * tile + 32u) > bin_end || any_ill != 0u) {
            best = 0.0f;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const uint32_t kf = off0 + rb * (8u * (uint32_t)(v / 4) + (uint32_t)(v % 4));
                if (kf < bin_end) {
                    if ((ills[v] >> l) & 1u) flags |= 1u << v;
                    else best = fmaxf(best, pw[v]);
                }
            }
        }
        uint64_t lanes = __ballot(flags != 0u);
        // The screen leaves a tile with many of them to the direct sums, which
        // compute them again anyway: all its chunks are marked by the sign.
        const bool unread = SCREEN && __popcll(lanes) > kIpScreenIll;
        if (unread) lanes = 0u;
        while (lanes) {
            const uint32_t src = (uint32_t)__builtin_ctzll(lanes);
            const uint32_t f = (uint32_t)__shfl((int)flags, (int)src, 64), v = (uint32_t)__builtin_ctz(f);
            const uint32_t kf = kbase + rb * (32u * tile + 4u * (src >> 5) + 8u * (v / 4u) + v % 4u) + (src & 31u);
            const double pe = exact_power<GEN, IN>(a, obj, kf);
            if (l == src) {
                const float pw = (float)(pe * ke);
                if constexpr (!SCREEN) pg[kf] = pw;
                best = fmaxf(best, pw);
                flags &= flags - 1u;
            }
            lanes = __ballot(flags != 0u);
        }
        if (a.top_k) {
            // the best lane's value (top-3: the best three lanes')
            const float t0 = wave_fmax(best);
            float t1 = 0.0f, t2 = 0.0f;
            if (a.top_k > 1) {
                if (l == (uint32_t)__builtin_ctzll(__ballot(best == t0))) best = 0.0f;
                t1 = wave_fmax(best);
                if (l == (uint32_t)__builtin_ctzll(__ballot(best == t1))) best = 0.0f;
                t2 = wave_fmax(best);
            }
            const float tv = l == 0 ? t0 : l == 1 ? t1 : t2;
            if (l < 3) tmax[3u * tile + l] = unread ? -tv : tv;
        }
    }
    };
    if constexpr (ip_grouped(SCREEN, GEN)) {
        for (uint32_t it = it0; it < it0 + a.group && (uint64_t)it * (rows * rb) < a.nf; ++it) {
            if (!SCREEN && it != it0) __syncthreads();  // the last tiles' points are read
            uint32_t lane = l;  // opaque: nothing derived from it is worth registers across items
            asm volatile("" : "+v"(lane));
            sweep_item(it, lane);
        }
    } else {
        sweep_item(it0, l);
    }
}

}  // namespace

#define LS_IP(GEN, IN, SCREEN) {k_interp_fac<GEN, IN, SCREEN>, k_sweep_interp<GEN, IN, SCREEN>, 256}

const InterpEntry kInterp[2][2][2] = {
    {{LS_IP(false, float, false), {nullptr, nullptr, 0}}, {LS_IP(true, float, false), {nullptr, nullptr, 0}}},
    {{LS_IP(false, float, true), LS_IP(false, double, true)}, {LS_IP(true, float, true), LS_IP(true, double, true)}},
};

}  // namespace lsamd
