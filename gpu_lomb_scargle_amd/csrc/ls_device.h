// Device-side pieces shared by the sweep kernels (ls_sweep_plain.hip,
// ls_sweep_split.hip) and the host side of the sweep (ls_sweep.hip): the
// sweep's launch arguments, the work-item schedule, per-chunk peak lists and
// the tile registry entry.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "ls_internal.h"

namespace lsamd {

// Coarse-grid sweep, per object: the mode (0: direct), the centre of its time
// span, and the sum of the squares of its y (generalized: of (w/W) (y - ybar)),
// times its y scale.
struct InterpObj {
    double tc;
    uint32_t mode;
    float energy;
};

struct SweepArgs {
    const uint64_t *offsets;
    const uint32_t *order;
    uint32_t K, nf, chunks;
    uint64_t item_base;        // first item of this launch
    uint64_t total_items;      // K * chunks
    uint32_t group;            // consecutive items per workgroup fetch (a power of two)
    uint32_t xcd_run;          // grid schedule: groups kept together on one XCD (0: blockIdx order)
    uint32_t slices;           // split forms: observation slices per (object, chunk), >= 1
    double *part_sums;         // slices > 1: per-slice FP64 sums [K*chunks][slices][NS][M][T]
    unsigned long long *queue; // persistent schedule: kQueues group counters (one per XCD), else null
    // plain (t, y, w); split forms: the caller's y and dy (DTYPE), read by
    // the FP64 recomputation of ill-conditioned bins and small objects
    const void *t, *y, *w, *dy;
    double fmin_r, fstep_r;    // DTYPE values stored in double
    // split
    const double *rec_t;
    const float4 *rec_a;
    const float *rec_n;
    const double2 *rec_r;
    double fmin_rev, df_rev;   // revolutions/day
    const double *obj_gen;
    // common
    const double *obj_scale;
    void *pgram;
    double *part_pow;
    uint32_t *part_idx;
    int top_k;                 // peaks kept per chunk: 0, 1 or 3
    // matrix-core tile: per-object column- and row-factor fragments, y scale
    uint4 *colfac;
    uint4 *rowfac;
    uint32_t *slot_obj;  // the object of each 16-observation slot
    float *obj_ys;  // per object: y scale, weight scale
    // coarse-grid sweep (null: every object direct): the objects' modes, the
    // interpolation operands, workgroups per object, and the chunks to sweep
    // again directly (bit c % 64 of word c / 64; null: the main pass)
    const InterpObj *obj_ip;
    uint4 *ip_tab;
    uint32_t ip_items;
    float ip_margin;  // of the marked chunks' powers
    uint32_t cand_words, cand_split;  // words per object; workgroups per object that sweep them,
    uint32_t marked_groups;           // and of all objects (a multiple of 8)
    uint64_t *cand;
    // the objects in direct mode, about in processing order, and their number
    uint32_t *direct_list, *direct_count;
};

typedef void (*SweepFn)(SweepArgs);

// One compiled sweep kernel: form, variant, output type and tile shape.
struct TileEntry {
    int form, variant, dtype, T, M;
    SweepFn fn;
    SweepFn combine;  // split forms: sums the observation slices (null: plain)
    SweepFn prep;     // per-object set-up launched before the sweep (K x G workgroups of 64), or null
};
extern const TileEntry kPlainTiles[];  // ls_sweep_plain.hip
extern const int kPlainTileCount;
extern const TileEntry kSplitTiles[];  // ls_sweep_split.hip
extern const int kSplitTileCount;

namespace {

// Observations per FP32 partial sum of the split32 sweep before it is folded
// into FP64.  Standard 32: on the 1000-object batch the worst relative power
// error drops from 9.4e-6 (64) to 7.0e-6 for ~1% of the time.  Generalized
// 64: even 16 stays above 1e-5 there (1.2e-5), at ~7% of the time.
constexpr uint32_t kFlushStd = 32, kFlushGen = 64;
constexpr uint32_t kGroup = 4;  // work items per workgroup fetch, split forms (a power of two)
constexpr uint64_t kGroupMinItems = 65536;  // fewer items: one per fetch (e.g. a single object)
// Split forms: below this many (object, chunk) items, long objects are also
// split by observations (at least T observations per slice), up to about
// this many items.
constexpr uint64_t kSliceTargetItems = 2048;
// Matrix-core tile: column-factor fragments per 16 observations (standard:
// y v and w; generalized: (w/W) v, (w/W) y_c v and (w/W) w; real and
// imaginary head and tail of each).
constexpr int kColfacFragsStd = 8, kColfacFragsGen = 12;
// Matrix-core tile: row-step phasors e^{2 pi i 32 a df t} per 16 observations
// (lane a + 32 h: observations 8 h .. 8 h + 7 as 4 x two complex FP32).
constexpr int kRowfacFrags = 4;
// Groups of T threads that share the M bins per thread of a tile when its
// observation slices are added up: the largest divisor of M that fits a
// workgroup of 1024 threads.
constexpr int combine_groups(int T, int M) {
    int g = 1;
    for (int d = 2; d <= M && d * T <= 1024; ++d)
        if (M % d == 0) g = d;
    return g;
}
constexpr int kPeaks = 3;      // peaks tracked per object (top-1 and top-3)
// doubles per object of split-generalized constants: [0..2] Wf, Yb, YY over
// the FP32-rounded weights the VALU split sweeps apply; [3] ybar, [4] W (sum
// of 1/dy^2); [5..7] Wf, Yb, YY over the FP64 weights w / W (matrix-core tile)
constexpr int kGen = 8;
constexpr double kInv2Pi = 0.159154943091895335768883763372514362;  // 1/(2 pi)
constexpr double kTwoPi = 6.283185307179586476925286766559005768;   // 2 pi

// ---------------------------------------------------------------------------
// Peak lists: best kPeaks (power, bin) pairs, ordered by power descending and
// bin ascending.  Initialised to (0, 0): a bin enters only with power > 0,
// and an equal power never displaces an earlier bin -- the reference's
// "first index of the strict maximum, starting from 0" (main.cu:1140-1149,
// 1545-1556) and its three-scan top-3 (main.cu:1165-1219).  NaN never enters.
// ---------------------------------------------------------------------------
struct Peaks {
    double p[kPeaks];
    uint32_t i[kPeaks];
};

__device__ __forceinline__ bool better(double p1, uint32_t i1, double p2, uint32_t i2) {
    return p1 > p2 || (p1 == p2 && i1 < i2);
}

__device__ __forceinline__ void peaks_init(Peaks &L) {
#pragma unroll
    for (int r = 0; r < kPeaks; ++r) {
        L.p[r] = 0.0;
        L.i[r] = 0u;
    }
}

// Insertion by compare-and-swap down the list (static indices only).
__device__ __forceinline__ void peaks_insert(Peaks &L, double p, uint32_t i) {
#pragma unroll
    for (int r = 0; r < kPeaks; ++r) {
        if (better(p, i, L.p[r], L.i[r])) {
            const double tp = L.p[r];
            const uint32_t ti = L.i[r];
            L.p[r] = p;
            L.i[r] = i;
            p = tp;
            i = ti;
        }
    }
}

// Adds bin i to the list kept for top_k = 1 (the best bin only) or 3;
// nothing for top_k = 0.  Each thread adds its bins in ascending order, so an
// equal power never displaces an earlier bin and a strict comparison of the
// powers decides.
// Out-of-order insertion (bins that are not the lane's next in index order):
// the index breaks ties, as the in-order strict comparison of peaks_add does.
__device__ __forceinline__ void peaks_merge(Peaks &L, int top_k, double p, uint32_t i) {
    if (top_k == 1) {
        if (better(p, i, L.p[0], L.i[0])) {
            L.p[0] = p;
            L.i[0] = i;
        }
    } else if (top_k) {
        peaks_insert(L, p, i);
    }
}

__device__ __forceinline__ void peaks_add(Peaks &L, int top_k, double p, uint32_t i) {
    if (top_k == 1) {
        if (p > L.p[0]) {
            L.p[0] = p;
            L.i[0] = i;
        }
    } else if (top_k) {
        const bool c0 = p > L.p[0], c1 = p > L.p[1], c2 = p > L.p[2];
        const double p2 = c1 ? L.p[1] : (c2 ? p : L.p[2]);
        const uint32_t i2 = c1 ? L.i[1] : (c2 ? i : L.i[2]);
        const double p1 = c0 ? L.p[0] : (c1 ? p : L.p[1]);
        const uint32_t i1 = c0 ? L.i[0] : (c1 ? i : L.i[1]);
        L.p[0] = c0 ? p : L.p[0];
        L.i[0] = c0 ? i : L.i[0];
        L.p[1] = p1;
        L.i[1] = i1;
        L.p[2] = p2;
        L.i[2] = i2;
    }
}

// Best (power, bin) of a whole workgroup; the result is valid in thread 0.
template <int T>
__device__ __forceinline__ void block_best(double &p, uint32_t &i, double (*s_p)[kPeaks],
                                           uint32_t (*s_i)[kPeaks]) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const double op = __shfl_xor(p, off, 64);
        const uint32_t oi = __shfl_xor(i, off, 64);
        if (better(op, oi, p, i)) {
            p = op;
            i = oi;
        }
    }
    if constexpr (T > 64) {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        if (lane == 0) {
            s_p[wave][0] = p;
            s_i[wave][0] = i;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int w = 1; w < T / 64; ++w)
                if (better(s_p[w][0], s_i[w][0], p, i)) {
                    p = s_p[w][0];
                    i = s_i[w][0];
                }
        }
    }
}

// Best (power, bin) of a whole workgroup, valid in every thread; `slot`
// selects the LDS entries used, so that consecutive calls need no barrier
// between them.
template <int T>
__device__ __forceinline__ void block_best_all(double &p, uint32_t &i, double (*s_p)[kPeaks],
                                               uint32_t (*s_i)[kPeaks], int slot) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const double op = __shfl_xor(p, off, 64);
        const uint32_t oi = __shfl_xor(i, off, 64);
        if (better(op, oi, p, i)) {
            p = op;
            i = oi;
        }
    }
    if constexpr (T > 64) {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        if (lane == 0) {
            s_p[wave][slot] = p;
            s_i[wave][slot] = i;
        }
        __syncthreads();
        p = s_p[0][slot];
        i = s_i[0][slot];
#pragma unroll
        for (int w = 1; w < T / 64; ++w)
            if (better(s_p[w][slot], s_i[w][slot], p, i)) {
                p = s_p[w][slot];
                i = s_i[w][slot];
            }
    }
}

// Top three (power, bin) of a whole workgroup from every thread's own
// sorted top three: three rounds of "best head, then its owner drops it",
// i.e. three scans that exclude the bins already taken.  The result is
// returned in every thread.
template <int T>
__device__ __forceinline__ void block_top3(Peaks &L, double (*s_p)[kPeaks],
                                           uint32_t (*s_i)[kPeaks], Peaks &W) {
#pragma unroll
    for (int r = 0; r < kPeaks; ++r) {
        double p = L.p[0];
        uint32_t i = L.i[0];
        block_best_all<T>(p, i, s_p, s_i, r);
        W.p[r] = p;
        W.i[r] = i;
        if (L.p[0] == p && L.i[0] == i) {  // the owner (or an empty (0, 0) head)
            L.p[0] = L.p[1];
            L.i[0] = L.i[1];
            L.p[1] = L.p[2];
            L.i[1] = L.i[2];
            L.p[2] = 0.0;
            L.i[2] = 0u;
        }
    }
}

// ---------------------------------------------------------------------------
// Reference-arithmetic helpers (plain form)
// ---------------------------------------------------------------------------
// The FP32 plain form evaluates sin, cos and atan2 of its float arguments in
// FP64 and rounds once: correctly rounded float results (double rounding is
// possible only within 2^-29 of a float midpoint).  The reference's float CPU
// build calls glibc's sinf/cosf/atan2f, which are correctly rounded on most
// but not all inputs, so this is the closest reproducible target.
// FP64 sine and cosine for |x| < kTrigFar: Cody-Waite reduction by pi/2 in
// three parts (the first FMA is exact, the second leaves its remainder in l),
// then minimax polynomials of sin (h + h^3 p(h^2)) and cos (1 - h^2/2 +
// h^4 q(h^2)) on |h| <= pi/4 (own Remez fits).  NaN and infinities give NaN.
// Results off the correctly rounded one, over 10^6 arguments each up to 10,
// 10^3, 2.7e5 and 4e8 (the device library's sincos, ~130 instructions for
// arguments of any size: 3.1%, at most 0.78 ulp):
//   CARRIED false (45 instructions): 1.7%, at most 0.74 ulp; the terms of l
//     and of the rounding of h^2 in cos are carried.
//   CARRIED true (69 instructions): 0.07%, at most 0.51 ulp; one term more per
//     polynomial, whose leading products carry their rounding too.  The
//     generalized FP64 power amplifies a last-bit difference 10^4-10^5 times
//     where its sums cancel; with 1.7% its distance from the CPU path reached
//     1.3e-12 on a 3555-observation object.
constexpr double kTrigFar = 1073741824.0;  // 2^30: the quadrant number fits the low word of n
template <bool CARRIED>
__device__ __forceinline__ void sincos_near(double x, double *so, double *co) {
#pragma clang fp contract(off)
    const double kMagic = 6755399441055744.0;  // 1.5 2^52: adding it rounds to an integer
    const double tn = fma(x, 0x1.45f306dc9c883p-1, kMagic), n = tn - kMagic;
    const double r = fma(-n, 0x1.921fb54442d18p+0, x);
    const double h = fma(-n, 0x1.1a62633145c07p-54, r);
    const double l = fma(-n, -0x1.f1976b7ed8fbcp-110, fma(-n, 0x1.1a62633145c07p-54, r - h));
    const double z = h * h, hz = 0.5 * z, w = 1.0 - hz, e = (1.0 - w) - hz;  // w + e = 1 - z/2
    double sv, cv;
    if constexpr (CARRIED) {
        const double zl = fma(h + h, l, fma(h, h, -z));  // (h + l)^2 = z + zl
        double p = fma(-0x1.aaa14a1d5a48ep-41, z, 0x1.61208a50e477cp-33);
        p = fma(p, z, -0x1.ae64528a74aa9p-26);
        p = fma(p, z, 0x1.71de3a532e3f9p-19);
        p = fma(p, z, -0x1.a01a01a018a51p-13);
        p = fma(p, z, 0x1.111111111110bp-7);
        p = fma(p, z, -0x1.5555555555555p-57);  // -1/6 = kS + this
        const double kS = -0x1.5555555555555p-3;
        const double ua = z * kS, ub = fma(z, p, fma(zl, kS, fma(z, kS, -ua)));
        const double t = h * ua, ts = fma(h, ub, fma(h, ua, -t)) + fma(l, ua, l);
        const double a = h + t;
        sv = a + (((h - a) + t) + ts);
        double q = fma(0x1.aabc209d313b5p-45, z, -0x1.939321f9f61e1p-37);
        q = fma(q, z, 0x1.1eed8c8ee7d5fp-29);
        q = fma(q, z, -0x1.27e4fb75e9defp-22);
        q = fma(q, z, 0x1.a01a01a018cb1p-16);
        q = fma(q, z, -0x1.6c16c16c16c0fp-10);
        q = fma(q, z, 0x1.5555555555555p-59);  // 1/24 = kC + this
        const double kC = 0x1.5555555555555p-5;
        const double z2 = z * z, y = z2 * kC;
        double yl = fma(z2, q, fma(fma(z, z, -z2), kC, fma(z2, kC, -y)));
        yl = fma(zl, fma(z, 2.0 * kC, -0.5), yl);
        const double b = w + y;
        cv = b + (((w - b) + y) + (e + yl));
    } else {
        double p = fma(0x1.5d8ee79a66441p-33, z, -0x1.ae5e57812b6fep-26);
        p = fma(p, z, 0x1.71de356408b31p-19);
        p = fma(p, z, -0x1.a01a019bf9b61p-13);
        p = fma(p, z, 0x1.111111110f7b0p-7);
        p = fma(p, z, -0x1.5555555555548p-3);
        sv = h + fma(z * h, p, fma(-hz, l, l));
        double q = fma(-0x1.8fa395845a07fp-37, z, 0x1.1ee9d5c9140e1p-29);
        q = fma(q, z, -0x1.27e4f7e802715p-22);
        q = fma(q, z, 0x1.a01a019c80967p-16);
        q = fma(q, z, -0x1.6c16c16c14f6cp-10);
        q = fma(q, z, 0x1.555555555554bp-5);
        cv = w + (e + fma(z * z, q, fma(-0.5, fma(h, h, -z), -(h * l))));
    }
    const uint32_t k = (uint32_t)__double_as_longlong(tn);  // quadrant
    const bool odd = (k & 1u) != 0u;
    const double s0 = odd ? cv : sv, c0 = odd ? sv : cv;
    const long long ss = (long long)((uint64_t)((k & 2u) << 30) << 32);
    const long long cs = (long long)((uint64_t)(((k + 1u) & 2u) << 30) << 32);
    *so = __longlong_as_double(__double_as_longlong(s0) ^ ss);
    *co = __longlong_as_double(__double_as_longlong(c0) ^ cs);
}

// NEAR: |x| < kTrigFar (or not finite) is known.  The device library's sincos
// is called, not inlined: its reduction of large arguments holds ~100 registers,
// which would cost every sweep its second and third wavefront per SIMD.
struct SinCos {
    double s, c;
};
__device__ __attribute__((noinline)) SinCos sincos_far(double x) {
    SinCos r;
    sincos(x, &r.s, &r.c);
    return r;
}
template <bool NEAR, bool CARRIED>
__device__ __forceinline__ void sincos_r(double x, double *s, double *c) {
    if constexpr (NEAR) {
        sincos_near<CARRIED>(x, s, c);
    } else {
        const SinCos r = sincos_far(x);
        *s = r.s;
        *c = r.c;
    }
}
template <bool NEAR, bool CARRIED>
__device__ __forceinline__ void sincos_r(float x, float *s, float *c) {
    double sd, cd;
    sincos_r<NEAR, false>((double)x, &sd, &cd);
    *s = (float)sd;
    *c = (float)cd;
}
__device__ __forceinline__ double atan2_r(double y, double x) { return atan2(y, x); }
__device__ __forceinline__ float atan2_r(float y, float x) { return (float)atan2((double)y, (double)x); }
__device__ __forceinline__ double sqrt_r(double x) { return sqrt(x); }
__device__ __forceinline__ float sqrt_r(float x) { return sqrtf(x); }

__device__ __forceinline__ void item_coords(const SweepArgs &a, uint64_t item, uint32_t &obj,
                                            uint32_t &chunk) {
    const uint32_t pos = (uint32_t)(item / a.chunks);
    chunk = (uint32_t)(item - (uint64_t)pos * a.chunks);
    obj = a.order ? a.order[pos] : pos;
}

// Split forms: item = (object position, chunk, observation slice), slice
// minor.  With one slice an item is the whole object; with S slices it is
// observations [beg + s L, beg + (s + 1) L) of the object, L = ceil(N / S).
__device__ __forceinline__ void item_coords_sliced(const SweepArgs &a, uint64_t item, uint32_t &obj,
                                                   uint32_t &chunk, uint32_t &slice, uint64_t &beg,
                                                   uint64_t &end) {
    uint64_t oc = item;
    slice = 0;
    if (a.slices > 1) {
        oc = item / a.slices;
        slice = (uint32_t)(item - oc * a.slices);
    }
    item_coords(a, oc, obj, chunk);
    beg = a.offsets[obj];
    end = a.offsets[obj + 1];
    if (a.slices > 1) {
        const uint64_t len = (end - beg + a.slices - 1) / a.slices;
        const uint64_t b = beg + (uint64_t)slice * len;
        beg = b < end ? b : end;
        end = (beg + len) < end ? beg + len : end;
    }
}

// Work items are numbered in processing order (longest object first),
// chunk-minor, and taken in aligned groups of a.group consecutive items (the
// next chunks of the same object, mostly): either one group per workgroup
// (item_base + grid_group * group, below), or, with queues, persistent
// workgroups that take groups until the items run out.
//
// Persistent schedule: kQueues counters, one per XCD.  Groups form runs of
// L = xcd_run (about one object's chunks); queue q holds runs q, 15 - q,
// 16 + q, 31 - q, ... (the grid schedule's XCD assignment), so its i-th group
// is run 8 rho + (rho odd ? 7 - q : q), rho = i / L, offset i % L: every group
// belongs to exactly one queue, and a queue's groups ascend with i.  A
// workgroup starts on the queue of its own XCD (blockIdx.x % 8, the dispatch
// order) and, once that queue is exhausted, takes groups from the next ones in
// turn, so that an object's tables stay in one XCD's L2 while its work lasts
// and no XCD idles while another has work.
// Each counter has a cache line of its own (one line for all eight serialised
// the ~16,000 fetches that find the queues dry, 0.25 ms), and a queue that
// reads as exhausted, which it then stays, is passed by without an atomic.
constexpr uint32_t kQueues = 8, kQueueStride = 16;  // 64-bit counters, words apart
__device__ __forceinline__ uint64_t queue_group(const SweepArgs &a, uint32_t q, uint64_t i) {
    const uint64_t L = a.xcd_run ? a.xcd_run : 1u;
    const uint64_t rho = i / L, x = (rho & 1u) ? 7u - q : q;
    return (8u * rho + x) * L + (i - rho * L);
}
__device__ __forceinline__ uint64_t fetch_item(const SweepArgs &a, uint64_t *s_item, bool first) {
    __shared__ uint32_t s_queue, s_tried;  // this workgroup's current queue, queues found empty
    __syncthreads();  // every thread is done with the previous item and its s_item read
    if (threadIdx.x == 0) {
        if (first) {
            s_queue = blockIdx.x & (kQueues - 1u);
            s_tried = 0u;
        }
        const uint64_t groups = (a.total_items - a.item_base + a.group - 1u) / a.group;
        uint64_t item = ~0ull;
        while (s_tried < kQueues) {
            unsigned long long *const c = &a.queue[s_queue * kQueueStride];
            uint64_t g = queue_group(a, s_queue, __hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
            if (g < groups) g = queue_group(a, s_queue, atomicAdd(c, 1ull));
            if (g < groups) {
                item = a.item_base + g * a.group;
                break;
            }
            s_queue = (s_queue + 1u) & (kQueues - 1u);  // exhausted for good: groups ascend with i
            ++s_tried;
        }
        *s_item = item;
    }
    __syncthreads();
    return *s_item;
}
// Grid schedule: the 8 XCDs receive workgroups round-robin (workgroup w goes
// to XCD w % 8), each with its own L2.  Runs of L = xcd_run consecutive
// groups (about one object's chunks) go to one XCD, and consecutive runs to
// consecutive XCDs, in alternating direction per round of 8 runs (objects
// come longest first): workgroup w = 8 i + x takes run 8 r + x' (r = i / L,
// x' = x, or 7 - x for odd r), group i % L of it; a bijection on the whole
// rounds of 8 L groups (the rest in blockIdx order).  An object's tables are
// then fetched into one L2, and the XCDs get equal shares of the work.
__device__ __forceinline__ uint64_t xcd_group(uint64_t w, uint64_t groups, uint64_t L) {
    if (L == 0) return w;
    const uint64_t round = 8u * L, full = (groups / round) * round;
    if (w >= full) return w;
    const uint64_t i = w >> 3, r = i / L, x = (r & 1u) ? 7u - (w & 7u) : (w & 7u);
    return r * round + x * L + i % L;
}
__device__ __forceinline__ uint64_t grid_group(const SweepArgs &a) { return xcd_group(blockIdx.x, gridDim.x, a.xcd_run); }
__device__ __forceinline__ uint64_t first_item(const SweepArgs &a, uint64_t *s_item) {
    return a.queue ? fetch_item(a, s_item, true) : a.item_base + grid_group(a) * a.group;
}
__device__ __forceinline__ uint64_t next_item(const SweepArgs &a, uint64_t *s_item, uint64_t item) {
    const uint64_t n = item + 1;
    if (((n - a.item_base) & (uint64_t)(a.group - 1)) != 0) return n;  // same group
    return a.queue ? fetch_item(a, s_item, false) : ~0ull;
}

template <typename OUT, int T>
__device__ __forceinline__ void write_partial(const SweepArgs &a, Peaks &L, uint32_t obj,
                                              uint32_t chunk, double (*s_p)[kPeaks],
                                              uint32_t (*s_i)[kPeaks]) {
    const uint64_t o = ((uint64_t)obj * a.chunks + chunk) * kPeaks;
    if (a.top_k == 1) {  // entries 1 and 2 of the chunk's slot stay unused
        block_best<T>(L.p[0], L.i[0], s_p, s_i);
        if (threadIdx.x == 0) {
            a.part_pow[o] = L.p[0];
            a.part_idx[o] = L.i[0];
        }
        return;
    }
    Peaks W;
    block_top3<T>(L, s_p, s_i, W);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int r = 0; r < kPeaks; ++r) {
            a.part_pow[o + r] = W.p[r];
            a.part_idx[o + r] = W.i[r];
        }
    }
}

}  // namespace

}  // namespace lsamd
