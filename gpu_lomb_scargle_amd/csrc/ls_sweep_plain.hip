// Plain-form sweep kernels: the reference's own arithmetic, standard and
// generalized (source/main.cu:1566-1599, 1701-1777), for the FP32 and FP64
// builds, and their tile registry entries.

#include <type_traits>

#include "ls_device.h"

namespace lsamd {

namespace {

// Both kernels are bound by FP64 vector issue: sine and cosine, then the sums.
// With sincos_near in place of the library's sincos: standard FP64, 100
// objects (17,200 observations) x 100,003 bins 7.47 -> 3.38 ms (5.1e11
// terms/s); generalized (two sines and cosines per term) FP64, 3555
// observations x 200,000 bins 9.0 -> 5.7 ms, FP32, 136 objects (7,200
// observations) x 100,000 bins 7.1 -> 3.5 ms.  The stepped FP64 sweeps below
// form most of them from their neighbours'.
//
// A bound of |omega| over the bins below k_end, and whether omega t may leave
// the range of sincos_near (2^30, half the range its reduction holds for, so
// that the roundings of omega and t - tau do not matter): a workgroup whose
// staged observations have such a time runs the block with the library's
// sincos.  NaN times count as near (both give NaN).
__device__ __forceinline__ double chunk_omega_most(const SweepArgs &a, uint32_t k_end) {
    return fmax(fabs(a.fmin_r), fabs(a.fmin_r + a.fstep_r * (double)k_end));
}
__device__ __forceinline__ bool far_phase(double om_most, double t) { return om_most * fabs(t) >= kTrigFar; }

// Power of a bin from its sums (the reference's tau form).
template <typename R>
__device__ __forceinline__ R plain_std_power(R omega, R xc, R xs, R cc, R ss, R cs, double scale) {
#pragma clang fp contract(off)
    const R tau = (R)(atan2(2.0 * (double)cs, (double)(cc - ss)) / (2.0 * (double)omega));
    R s_tau, c_tau;
    sincos_r<true, false>(omega * tau, &s_tau, &c_tau);  // |omega tau| <= pi/2, or not finite
    const R c_tau2 = c_tau * c_tau, s_tau2 = s_tau * s_tau;
    const R cs_tau = (R)(2.0 * (double)c_tau * (double)s_tau);
    const R p1 = c_tau * xc + s_tau * xs;
    const R p2 = c_tau * xs - s_tau * xc;
    const R q = (p1 * p1) / (c_tau2 * cc + cs_tau * cs + s_tau2 * ss) +
                (p2 * p2) / (c_tau2 * ss - cs_tau * cs + s_tau2 * cc);
    const R pw = (R)(0.5 * (double)q);
    return (R)((double)pw * scale);  // main.cu:1335 / 1350
}

// ---------------------------------------------------------------------------
// Plain form: the reference's arithmetic, standard variant
// (lombscarglecpuinnerloop, main.cu:1566-1599).
// ---------------------------------------------------------------------------
template <typename R, int T, int M>
__global__ __launch_bounds__(T) void k_sweep_plain_std(SweepArgs a) {
#pragma clang fp contract(off)
    __shared__ R s_t[T], s_y[T];
    __shared__ double s_pp[T / 64][kPeaks];
    __shared__ uint32_t s_pi[T / 64][kPeaks];
    __shared__ uint64_t s_item;
    for (uint64_t item = first_item(a, &s_item); item < a.total_items;
         item = next_item(a, &s_item, item)) {
        uint32_t obj, chunk;
        item_coords(a, item, obj, chunk);
        const uint64_t beg = a.offsets[obj], end = a.offsets[obj + 1];
        const R *gt = static_cast<const R *>(a.t);
        const R *gy = static_cast<const R *>(a.y);
        const uint32_t tid = threadIdx.x;
        const uint32_t kbase = chunk * (uint32_t)(T * M);
        const R fmin = (R)a.fmin_r, fstep = (R)a.fstep_r;
        R om[M], xc[M], xs[M], cc[M], ss[M], cs[M];
    #pragma unroll
        for (int m = 0; m < M; ++m) {
            om[m] = fmin + (fstep * (R)(kbase + m * T + tid));  // main.cu:1611
            xc[m] = xs[m] = cc[m] = ss[m] = cs[m] = (R)0;
        }
        const double om_most = chunk_omega_most(a, kbase + (uint32_t)(T * M));
        for (uint64_t b0 = beg; b0 < end; b0 += T) {
            const uint32_t cnt = (uint32_t)((end - b0) < (uint64_t)T ? (end - b0) : (uint64_t)T);
            __syncthreads();
            bool far = false;
            if (tid < cnt) {
                const R t = gt[b0 + tid];
                s_t[tid] = t;
                s_y[tid] = gy[b0 + tid];
                far = far_phase(om_most, (double)t);
            }
            auto sums = [&](auto near) {
                for (uint32_t j = 0; j < cnt; ++j) {
                    const R tj = s_t[j], yj = s_y[j];
    #pragma unroll
                    for (int m = 0; m < M; ++m) {
                        R s, c;
                        sincos_r<decltype(near)::value, false>(om[m] * tj, &s, &c);
                        xc[m] = xc[m] + yj * c;
                        xs[m] = xs[m] + yj * s;
                        cc[m] = cc[m] + c * c;
                        ss[m] = ss[m] + s * s;
                        cs[m] = cs[m] + c * s;
                    }
                }
            };
            if (__syncthreads_or(far)) sums(std::false_type{});
            else sums(std::true_type{});
        }
        const double scale = a.obj_scale[obj];
        R *pg = static_cast<R *>(a.pgram);
        Peaks L;
        peaks_init(L);
    #pragma unroll
        for (int m = 0; m < M; ++m) {
            const uint32_t kf = kbase + m * T + tid;
            const R pw = plain_std_power(om[m], xc[m], xs[m], cc[m], ss[m], cs[m], scale);
            if (kf < a.nf) {
                if (pg) pg[(uint64_t)obj * a.nf + kf] = pw;
                peaks_add(L, a.top_k, (double)pw, kf);
            }
        }
        if (a.top_k) write_partial<R, T>(a, L, obj, chunk, s_pp, s_pi);
    }
}

// ---------------------------------------------------------------------------
// Standard FP64 variant, 16 bins from one sine and cosine.  A sine
// and cosine of every phase is 59 of the 70 instructions per term above, though
// the phases of a thread's bins, x_m = fl(om_m t), lie one common step
// D = 64 df t apart up to their roundings.  So the phasor of the middle bin is
// (the ninth of 16) is evaluated and the others follow from it,
//   e^{i x_m} = e^{i x_{m-1}} e^{i D} (1 + i r),  r = (x_m - x_{m-1}) - D,
// where r holds the roundings of om_m and of the products: both differences
// are exact (|x_{m-1}| >= D, see `low`), so each phase is the reference's own,
// rounding included.  |r| <= 2 ulp of a phase, so that the 1 + r^2/2 of the last
// factor stays within 2e-14 for phases below kStepFar (typically 1e-15).
// 13 instructions per term and 59 / 16 for the middle bin; the eight
// steps each way add 2e-16 to 3e-16 to a phasor.  M = 16: a thread forms all 16
// bins.  M = 8: the upper or the lower eight of them (by wavefront), from the same middle bin
// in the same steps, so both give the same bits; twice the wavefronts, for
// calls that would leave SIMDs idle.  Against the CPU path over the test light
// curves (14 to 3555 observations) 2.3e-13 on bins of at least 1e-6 of the
// peak, with a stride of 256 bins instead of 64 1.1e-11 at the lowest bins
// (the differences are not exact there).  Against powers of the exact phases in
// 80 bits (40 to 3555 observations, times from 0, 51,075 and 2,458,652 days) the
// errors are those of a sine and cosine per bin to three digits, 1e-11 to 3e-8:
// the roundings of the phases, which both have.
// The sums above serve, bin by bin, what this does not: bins whose 2x2 system
// amplifies the phasors' error (condition number above kStepCond), frequencies
// below the step (or of both signs in a thread), phases past kStepFar, objects of fewer than
// kStepLeastObs observations, most of whose bins are ill-conditioned.
// 100 objects (17,200 observations) x 100,003 bins: 3.38 -> 0.96 ms (M = 16, two wavefronts per SIMD by 18 spilled registers, mostly outside
// the loop; 1.06 with one and none).  Chains of 8, 10, 12 and 14 bins: 1.31, 1.03, 1.14 and
// 1.07 where 16 has 0.98; four wavefronts of 8 spill to 2.8 ms.
// ---------------------------------------------------------------------------
constexpr double kStepFar = 268435456.0;  // 2^28
constexpr double kStepCond = 16.0;
constexpr uint32_t kStepLeastObs = 16;
constexpr int kStepRun = 16, kStepMid = 8;  // bins of a chain, its middle bin

// Power at omega from a sine and cosine per observation, as k_sweep_plain_std
// gives it (256 observations at a time near or far); the observations'
// addresses are the same in all lanes.
__device__ __forceinline__ double direct_std_power(const SweepArgs &a, uint64_t beg, uint64_t end, double omega,
                                                   double om_most, double scale) {
#pragma clang fp contract(off)
    const double *t = static_cast<const double *>(a.t), *y = static_cast<const double *>(a.y);
    double xc = 0.0, xs = 0.0, cc = 0.0, ss = 0.0, cs = 0.0;
    for (uint64_t b0 = beg; b0 < end; b0 += 256) {
        const uint64_t e0 = end - b0 < 256u ? end : b0 + 256;
        bool far = false;
        for (uint64_t i = b0 + (threadIdx.x & 63u); i < e0; i += 64) far |= far_phase(om_most, t[i]);
        auto sums = [&](auto near) {
            for (uint64_t i = b0; i < e0; ++i) {
                const double ti = t[i], yi = y[i];
                double s, c;
                sincos_r<decltype(near)::value, false>(omega * ti, &s, &c);
                xc = xc + yi * c;
                xs = xs + yi * s;
                cc = cc + c * c;
                ss = ss + s * s;
                cs = cs + c * s;
            }
        };
        if (__ballot(far) != 0u) sums(std::false_type{});
        else sums(std::true_type{});
    }
    return plain_std_power(omega, xc, xs, cc, ss, cs, scale);
}

// (c, s) turned by (ec, es), corrected by the rotation r.
__device__ __forceinline__ void turn_step(double &c, double &s, double ec, double es, double r) {
    const double rc = fma(-r, es, ec), rs = fma(r, ec, es), c0 = c;
    c = fma(c, rc, -(s * rs));
    s = fma(c0, rs, s * rc);
}

template <int T, int M>
__global__ __launch_bounds__(T, 2) void k_sweep_plain_step(SweepArgs a) {
#pragma clang fp contract(off)
    __shared__ double2 s_ty[T], s_step[T];  // t, y; cos D, sin D
    __shared__ double s_d[T];               // D
    __shared__ double s_pp[T / 64][kPeaks];
    __shared__ uint32_t s_pi[T / 64][kPeaks];
    __shared__ uint64_t s_item;
    static_assert(T == 256 && (M == kStepRun || M == kStepMid), "chains of whole wavefronts, or halves");
    constexpr bool kHalf = M != kStepRun;
    for (uint64_t item = first_item(a, &s_item); item < a.total_items;
         item = next_item(a, &s_item, item)) {
        uint32_t obj, chunk;
        item_coords(a, item, obj, chunk);
        const uint64_t beg = a.offsets[obj], end = a.offsets[obj + 1];
        const double *gt = static_cast<const double *>(a.t);
        const double *gy = static_cast<const double *>(a.y);
        const uint32_t tid = threadIdx.x;
        const uint32_t kbase = chunk * (uint32_t)(T * M);
        // The bins of a wavefront's chains are consecutive: bin b of a lane's chain
        // is k0 + 64 b.  Entry m of a thread is bin m, or with half chains bin 8 + m
        // (upper) or 7 - m: the steps lead away from the middle.
        const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
        const uint32_t k0 = kbase + (kHalf ? wave >> 1 : wave) * (uint32_t)(64 * kStepRun) + (tid & 63u);
        const bool upper = (wave & 1u) != 0u;
        auto chain_bin = [&](int m) { return (uint32_t)(!kHalf ? m : upper ? kStepMid + m : kStepMid - 1 - m); };
        auto bin_omega = [&](uint32_t b) { return a.fmin_r + (a.fstep_r * (double)(k0 + 64u * b)); };
        const double step = 64.0 * a.fstep_r;
        double om[M], xc[M], xs[M], cc[M], cs[M];
#pragma unroll
        for (int m = 0; m < M; ++m) {
            om[m] = bin_omega(chain_bin(m));
            xc[m] = xs[m] = cc[m] = cs[m] = 0.0;
        }
        const double om_mid = bin_omega((uint32_t)kStepMid);
        // over the 4096 bins that whole chains of the workgroup would have
        const double om_a = a.fmin_r + a.fstep_r * (double)(kbase & ~(uint32_t)(T * kStepRun - 1));
        const double om_b = om_a + a.fstep_r * (double)(T * kStepRun);
        const double om_most = fmax(fabs(om_a), fabs(om_b));
        const bool crosses = (bin_omega(0u) < 0.0) != (bin_omega((uint32_t)(kStepRun - 1)) < 0.0);
        bool direct = end - beg < (uint64_t)kStepLeastObs;
        for (uint64_t b0 = beg; b0 < end && !direct; b0 += T) {
            const uint32_t cnt = (uint32_t)((end - b0) < (uint64_t)T ? (end - b0) : (uint64_t)T);
            __syncthreads();
            bool far = false;
            if (tid < cnt) {
                const double t = gt[b0 + tid], d = step * t;
                double s, c;
                far = om_most * fabs(t) >= kStepFar;
                sincos_near<false>(far ? 0.0 : d, &s, &c);
                s_ty[tid] = make_double2(t, gy[b0 + tid]);
                s_step[tid] = make_double2(c, s);
                s_d[tid] = d;
            }
            direct = __syncthreads_or(far) != 0;
            if (direct) break;
            for (uint32_t j = 0; j < cnt; ++j) {
                const double2 ty = s_ty[j], e = s_step[j];
                const double d = s_d[j];
                auto add = [&](int m, double c, double s) {
                    xc[m] = fma(ty.y, c, xc[m]);
                    xs[m] = fma(ty.y, s, xs[m]);
                    cc[m] = fma(c, c, cc[m]);
                    cs[m] = fma(c, s, cs[m]);
                };
                const double xm = om_mid * ty.x;
                double cm, sm;
                sincos_near<false>(xm, &sm, &cm);
                double c = cm, s = sm, x = xm;
                if constexpr (kHalf) {
                    const double es = upper ? e.y : -e.y, ds = upper ? d : -d;
#pragma unroll
                    for (int m = 0; m < M; ++m) {
                        if (m > 0 || !upper) {  // (the middle bin itself is the first upper one)
                            const double xn = om[m] * ty.x;
                            turn_step(c, s, e.x, es, (xn - x) - ds);
                            x = xn;
                        }
                        add(m, c, s);
                    }
                    continue;
                }
                add(kStepMid, cm, sm);
#pragma unroll
                for (int m = kStepMid + 1; m < M; ++m) {
                    const double xn = om[m] * ty.x;
                    turn_step(c, s, e.x, e.y, (xn - x) - d);
                    x = xn;
                    add(m, c, s);
                }
                c = cm;
                s = sm;
                x = xm;
#pragma unroll
                for (int m = kStepMid - 1; m >= 0; --m) {
                    const double xn = om[m] * ty.x;
                    turn_step(c, s, e.x, -e.y, (xn - x) + d);
                    x = xn;
                    add(m, c, s);
                }
            }
        }
        const double scale = a.obj_scale[obj], nobs = (double)(end - beg);
        const double least = nobs * nobs / (4.0 * kStepCond);
        double P[M];
        uint32_t flags = 0u;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const double ss = nobs - cc[m];
            const bool ill = !(fma(cc[m], ss, -(cs[m] * cs[m])) >= least);
            const bool low = crosses || !(fabs(om[m]) >= step);
            if ((direct || ill || low) && k0 + 64u * chain_bin(m) < a.nf) flags |= 1u << m;
            P[m] = direct ? 0.0 : plain_std_power(om[m], xc[m], xs[m], cc[m], ss, cs[m], scale);
            __builtin_amdgcn_sched_barrier(0);  // one bin's temporaries at a time
        }
        // bin m of all lanes at once, where a lane needs it
        for (int m = 0; m < M; ++m) {
            const bool mine = ((flags >> m) & 1u) != 0u;
            if (__ballot(mine) == 0u) continue;
            const double omega = bin_omega(chain_bin(m));
            const double most = chunk_omega_most(a, k0 - (tid & 63u) + 512u * (chain_bin(m) / 8u + 1u));
            const double p = direct_std_power(a, beg, end, omega, most, scale);
#pragma unroll
            for (int q = 0; q < M; ++q) P[q] = mine && q == m ? p : P[q];
        }
        double *pg = static_cast<double *>(a.pgram);
        Peaks L;
        peaks_init(L);
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const uint32_t kf = k0 + 64u * chain_bin(m);
            if (kf < a.nf) {
                if (pg) pg[(uint64_t)obj * a.nf + kf] = P[m];
                if constexpr (kHalf) peaks_merge(L, a.top_k, P[m], kf);  // (not in ascending order)
                else peaks_add(L, a.top_k, P[m], kf);
            }
        }
        if (a.top_k) write_partial<double, T>(a, L, obj, chunk, s_pp, s_pi);
    }
}

// ---------------------------------------------------------------------------
// The generalized FP64 second pass, stepped.  Its phases fl(om_m fl(t - tau_m))
// differ from bin to bin by D - (T_m - T_{m-1}), T_m = om_m tau_m, and by their
// roundings, so with u_m = e^{i (x_m + T_m - T_mid)}
//   u_m = u_{m-1} e^{i D} (1 + i r),  r = (x_m - x_{m-1}) - D + (T_m - T_{m-1}),
// as in the standard sweep, every phase the reference's own; the sums are turned
// back by T_m - T_mid at the end.  (The first pass keeps a sine and cosine per
// phase: the roundings of t - tau hang on the last bit of tau.)  A wavefront
// takes a quarter of the observations and all 256 bins of the workgroup, four per
// lane: ~33 instructions per term instead of ~105.  The quarters' sums meet in
// LDS, and thread tid ends with those of its bin.  3555 observations x 200,000
// bins 5.61 -> 3.41 ms, 100 objects of 165 x 100,003 8.84 -> 5.53 (two wavefronts per SIMD;
// unbounded it takes 266 registers and one, 4.3 and 8.1 ms, three spill, 3.6 and
// 6.2).
// ---------------------------------------------------------------------------
template <typename R>
struct TauSums {  // weighted sums of y, y y, c, s, y c, y s, c c, and s s
    R Y, YY, C, S, YC, YS, CC, SS;
};
constexpr uint32_t kStepGenLeastObs = 32;

// The sums at thread tid's bin, with c s in the place of s s, turned by T - T_mid;
// false, and no sums, if a phase is past kStepFar.  tau: of that bin, finite.  All
// threads of the workgroup call it.
template <int T>
__device__ __forceinline__ bool stepped_tau_sums(const double *gt, const double *gy, const double *gw, uint64_t beg,
                                                 uint64_t end, double fmin_r, double fstep_r, uint32_t kbase,
                                                 double tau, TauSums<double> &out) {
#pragma clang fp contract(off)
    static_assert(T == 256, "four wavefronts");
    constexpr int M = T / 64, kMid = M / 2, NS = 6;
    // the staged observations, and when they are done with a sum of every
    // wavefront and bin, [M][T]
    __shared__ double2 s_obs[3][T];
    double2 *const s_t = s_obs[0], *const s_w = s_obs[1], *const s_e = s_obs[2];  // t, D; w, w y; cos D, sin D
    double *const s_sum = reinterpret_cast<double *>(s_obs);
    static_assert(sizeof(s_obs) >= M * T * sizeof(double), "s_sum lies within s_obs");
    __shared__ double s_yy[T];  // w y y
    __shared__ double s_tau[T], s_y[M][2];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const double step = 64.0 * fstep_r;
    const double om_most = fmax(fabs(fmin_r + fstep_r * (double)kbase),
                                fabs(fmin_r + fstep_r * ((double)kbase + (double)T)));
    s_tau[tid] = tau;
    __syncthreads();
    double om[M], tm[M], dT[M], acc[NS][M], Y = 0.0, YY = 0.0;
#pragma unroll
    for (int m = 0; m < M; ++m) {
        om[m] = fmin_r + (fstep_r * (double)(kbase + 64u * (uint32_t)m + lane));
        tm[m] = s_tau[64 * m + (int)lane];
        dT[m] = m == 0 ? 0.0 : om[m] * tm[m] - om[m - 1] * tm[m - 1];
#pragma unroll
        for (int q = 0; q < NS; ++q) acc[q][m] = 0.0;
    }
    for (uint64_t b0 = beg; b0 < end; b0 += T) {
        const uint32_t cnt = (uint32_t)((end - b0) < (uint64_t)T ? (end - b0) : (uint64_t)T);
        __syncthreads();
        bool far = false;
        if (tid < cnt) {
            const double t = gt[b0 + tid], w = gw[b0 + tid], d = step * t;
            double s, c;
            far = om_most * fabs(t) >= kStepFar;
            sincos_near<false>(far ? 0.0 : d, &s, &c);
            s_t[tid] = make_double2(t, d);
            const double y = gy[b0 + tid], wy = w * y;
            s_w[tid] = make_double2(w, wy);
            s_yy[tid] = wy * y;
            s_e[tid] = make_double2(c, s);
        }
        if (__syncthreads_or(far)) return false;
        for (uint32_t j = wave; j < cnt; j += M) {
            const double2 td = s_t[j], ww = s_w[j], e = s_e[j];
            Y += ww.y;
            YY += s_yy[j];
            auto add = [&](int m, double c, double s) {
                const double wc = ww.x * c;
                acc[0][m] += wc;
                acc[1][m] = fma(ww.x, s, acc[1][m]);
                acc[2][m] = fma(ww.y, c, acc[2][m]);
                acc[3][m] = fma(ww.y, s, acc[3][m]);
                acc[4][m] = fma(wc, c, acc[4][m]);
                acc[5][m] = fma(wc, s, acc[5][m]);
            };
            const double xm = om[kMid] * (td.x - tm[kMid]);
            double cm, sm;
            sincos_near<false>(xm, &sm, &cm);
            add(kMid, cm, sm);
            double c = cm, s = sm, x = xm;
#pragma unroll
            for (int m = kMid + 1; m < M; ++m) {
                const double xn = om[m] * (td.x - tm[m]);
                turn_step(c, s, e.x, e.y, ((xn - x) - td.y) + dT[m]);
                x = xn;
                add(m, c, s);
            }
            c = cm;
            s = sm;
            x = xm;
#pragma unroll
            for (int m = kMid - 1; m >= 0; --m) {
                const double xn = om[m] * (td.x - tm[m]);
                turn_step(c, s, e.x, -e.y, ((xn - x) + td.y) - dT[m + 1]);
                x = xn;
                add(m, c, s);
            }
        }
    }
    double sum[NS];
    if (lane == 0) {
        s_y[wave][0] = Y;
        s_y[wave][1] = YY;
    }
#pragma unroll
    for (int q = 0; q < NS; ++q) {
        __syncthreads();
#pragma unroll
        for (int m = 0; m < M; ++m) s_sum[wave * T + 64u * (uint32_t)m + lane] = acc[q][m];
        __syncthreads();
        sum[q] = 0.0;
#pragma unroll
        for (int w = 0; w < M; ++w) sum[q] += s_sum[(uint32_t)w * T + tid];
    }
    out.Y = out.YY = 0.0;
#pragma unroll
    for (int w = 0; w < M; ++w) {
        out.Y += s_y[w][0];
        out.YY += s_y[w][1];
    }
    out.C = sum[0];
    out.S = sum[1];
    out.YC = sum[2];
    out.YS = sum[3];
    out.CC = sum[4];
    out.SS = sum[5];
    return true;
}

// ---------------------------------------------------------------------------
// Plain form, generalized variant: two passes, tau then the tau-shifted sums
// (lombscarglecpuinnerloopAstroPy, main.cu:1701-1777).
// ---------------------------------------------------------------------------
template <typename R, int T, int M>
__global__ __launch_bounds__(T, 2) void k_sweep_plain_gen(SweepArgs a) {
#pragma clang fp contract(off)
    __shared__ R s_t[T], s_y[T], s_w[T];
    __shared__ double s_pp[T / 64][kPeaks];
    __shared__ uint32_t s_pi[T / 64][kPeaks];
    __shared__ uint64_t s_item;
    for (uint64_t item = first_item(a, &s_item); item < a.total_items;
         item = next_item(a, &s_item, item)) {
        uint32_t obj, chunk;
        item_coords(a, item, obj, chunk);
        const uint64_t beg = a.offsets[obj], end = a.offsets[obj + 1];
        const R *gt = static_cast<const R *>(a.t);
        const R *gy = static_cast<const R *>(a.y);
        const R *gw = static_cast<const R *>(a.w);
        const uint32_t tid = threadIdx.x;
        const uint32_t kbase = chunk * (uint32_t)(T * M);
        const R fmin = (R)a.fmin_r, fstep = (R)a.fstep_r;
        R om[M], wsum[M], S[M], C[M], S2[M], C2[M], tau[M];
    #pragma unroll
        for (int m = 0; m < M; ++m) {
            om[m] = fmin + (fstep * (R)(kbase + m * T + tid));
            wsum[m] = S[m] = C[m] = S2[m] = C2[m] = (R)0;
        }
        // pass 1: tau
        const double om_most = chunk_omega_most(a, kbase + (uint32_t)(T * M));
        for (uint64_t b0 = beg; b0 < end; b0 += T) {
            const uint32_t cnt = (uint32_t)((end - b0) < (uint64_t)T ? (end - b0) : (uint64_t)T);
            __syncthreads();
            bool far = false;
            if (tid < cnt) {
                const R t = gt[b0 + tid];
                s_t[tid] = t;
                s_w[tid] = gw[b0 + tid];
                far = far_phase(om_most, (double)t);
            }
            auto sums = [&](auto near) {
                for (uint32_t j = 0; j < cnt; ++j) {
                    const R tj = s_t[j], w = s_w[j];
    #pragma unroll
                    for (int m = 0; m < M; ++m) {
                        R s, c;
                        wsum[m] += w;
                        sincos_r<decltype(near)::value, true>(om[m] * tj, &s, &c);
                        S[m] += w * s;
                        C[m] += w * c;
                        S2[m] = (R)((double)S2[m] + 2.0 * (double)w * (double)s * (double)c);
                        C2[m] = (R)((double)C2[m] + ((double)w - 2.0 * (double)w * (double)s * (double)s));
                    }
                }
            };
            if (__syncthreads_or(far)) sums(std::false_type{});
            else sums(std::true_type{});
        }
    #pragma unroll
        for (int m = 0; m < M; ++m) {
            S2[m] /= wsum[m];
            C2[m] /= wsum[m];
            S[m] /= wsum[m];
            C[m] /= wsum[m];
            S2[m] = (R)((double)S2[m] - 2.0 * (double)S[m] * (double)C[m]);
            C2[m] -= (C[m] * C[m] - S[m] * S[m]);
            tau[m] = (R)(0.5 * (double)atan2_r(S2[m], C2[m]) / (double)om[m]);
        }
        // pass 2: the tau-shifted sums.  FP64: stepped, but for objects of few
        // observations, chunks that reach below the step (see
        // k_sweep_plain_step), bins that amplify the steps' error (ccv ssv below
        // 1 / (4 kStepCond)) and a tau that is not finite.
        TauSums<R> q[M];
        bool again = true;  // this thread's sums are still to be formed, phase by phase
        if constexpr (std::is_same_v<R, double>) {
            static_assert(M == 1, "a bin per thread");
            const double tf = __builtin_isfinite(tau[0]) ? tau[0] : 0.0;
            TauSums<double> u;
            const double least = 64.0 * fstep, lo = fmin + fstep * (double)kbase, hi = lo + fstep * (double)(T - 1);
            const bool apart = ::fmin(fabs(lo), fabs(hi)) >= least && (lo < 0.0) == (hi < 0.0);
            if (apart && end - beg >= (uint64_t)kStepGenLeastObs &&
                stepped_tau_sums<T>(gt, gy, gw, beg, end, fmin, fstep, kbase, tf, u)) {
                s_t[tid] = om[0] * tf;
                __syncthreads();
                double sa, ca;
                sincos_near<true>(s_t[tid] - s_t[128u + (tid & 63u)], &sa, &ca);
                const double ss = wsum[0] - u.CC, w2 = 2.0 * ca * sa;
                q[0].Y = u.Y;
                q[0].YY = u.YY;
                q[0].C = fma(u.C, ca, u.S * sa);
                q[0].S = fma(u.S, ca, -(u.C * sa));
                q[0].YC = fma(u.YC, ca, u.YS * sa);
                q[0].YS = fma(u.YS, ca, -(u.YC * sa));
                q[0].CC = fma(ca * ca, u.CC, fma(w2, u.SS, sa * sa * ss));  // (u.SS: the sum of c s)
                q[0].SS = fma(ca * ca, ss, fma(-w2, u.SS, sa * sa * u.CC));
                const double ct = q[0].C / wsum[0], st = q[0].S / wsum[0];
                const double ccv = q[0].CC / wsum[0] - ct * ct, ssv = q[0].SS / wsum[0] - st * st;
                again = tf != tau[0] || !(ccv * ssv * (4.0 * kStepCond) >= 1.0);
            }
        }
        if (__syncthreads_or(again)) {
            TauSums<R> d[M];
    #pragma unroll
            for (int m = 0; m < M; ++m) d[m] = TauSums<R>{};
            const bool wave_any = __ballot(again) != 0u;
            for (uint64_t b0 = beg; b0 < end; b0 += T) {
                const uint32_t cnt = (uint32_t)((end - b0) < (uint64_t)T ? (end - b0) : (uint64_t)T);
                __syncthreads();
                bool far = false;
                if (tid < cnt) {
                    const R t = gt[b0 + tid];
                    s_t[tid] = t;
                    s_y[tid] = gy[b0 + tid];
                    s_w[tid] = gw[b0 + tid];
                    far = far_phase(om_most, (double)t);
                }
                auto sums = [&](auto near) {
                    for (uint32_t j = 0; j < cnt; ++j) {
                        const R tj = s_t[j], yj = s_y[j], w = s_w[j];
    #pragma unroll
                        for (int m = 0; m < M; ++m) {
                            R s, c;  // |omega tau| <= pi/4 beside omega t
                            sincos_r<decltype(near)::value, true>(om[m] * (tj - tau[m]), &s, &c);
                            d[m].Y += w * yj;
                            d[m].YY += w * yj * yj;
                            d[m].C += w * c;
                            d[m].S += w * s;
                            d[m].YC += w * yj * c;
                            d[m].YS += w * yj * s;
                            d[m].CC += w * c * c;
                            d[m].SS += w * s * s;
                        }
                    }
                };
                const bool some_far = __syncthreads_or(far) != 0;
                if (!wave_any) continue;
                if (some_far) sums(std::false_type{});
                else sums(std::true_type{});
            }
    #pragma unroll
            for (int m = 0; m < M; ++m)
                if (again) q[m] = d[m];
        }
        R *pg = static_cast<R *>(a.pgram);
        Peaks L;
        peaks_init(L);
    #pragma unroll
        for (int m = 0; m < M; ++m) {
            const uint32_t kf = kbase + m * T + tid;
            const R ws = wsum[m];
            R y_ = q[m].Y / ws, yy = q[m].YY / ws, ct = q[m].C / ws, st = q[m].S / ws;
            R yc = q[m].YC / ws, ys = q[m].YS / ws, ccv = q[m].CC / ws, ssv = q[m].SS / ws;
            yc -= y_ * ct;
            ys -= y_ * st;
            ccv -= ct * ct;
            ssv -= st * st;
            yy -= y_ * y_;
            const R pw = (yc * yc / ccv + ys * ys / ssv) / yy;
            if (kf < a.nf) {
                if (pg) pg[(uint64_t)obj * a.nf + kf] = pw;
                peaks_add(L, a.top_k, (double)pw, kf);
            }
        }
        if (a.top_k) write_partial<R, T>(a, L, obj, chunk, s_pp, s_pi);
    }
}

}  // namespace

#define LS_PLAIN_STD(R, DT, TT, MM) \
    {LSAMD_FORM_PLAIN, 0, DT, TT, MM, k_sweep_plain_std<R, TT, MM>, nullptr}
#define LS_PLAIN_GEN(R, DT, TT, MM) \
    {LSAMD_FORM_PLAIN, 1, DT, TT, MM, k_sweep_plain_gen<R, TT, MM>, nullptr}

const TileEntry kPlainTiles[] = {
    LS_PLAIN_STD(float, LSAMD_F32, 256, 1), LS_PLAIN_STD(double, LSAMD_F64, 256, 1),
    LS_PLAIN_STD(float, LSAMD_F32, 256, 2), LS_PLAIN_STD(double, LSAMD_F64, 256, 2),
    LS_PLAIN_GEN(float, LSAMD_F32, 256, 1), LS_PLAIN_GEN(double, LSAMD_F64, 256, 1),
    {LSAMD_FORM_PLAIN, 0, LSAMD_F64, 256, 8, k_sweep_plain_step<256, 8>, nullptr},
    {LSAMD_FORM_PLAIN, 0, LSAMD_F64, 256, 16, k_sweep_plain_step<256, 16>, nullptr},
};
const int kPlainTileCount = (int)(sizeof(kPlainTiles) / sizeof(kPlainTiles[0]));

}  // namespace lsamd
