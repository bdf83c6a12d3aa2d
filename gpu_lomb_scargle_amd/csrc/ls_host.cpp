// Host orchestration of the MI355X-native Lomb-Scargle library: error state,
// segmentation of the observation stream into objects, reference-faithful
// pre-centring, device buffers, memory-budget batching and the pinned,
// double-buffered copy of the periodogram back into the caller's memory.
//
// A drop-in call on a few stars is all latency, a catalogue's mostly the way of
// its periodogram into fresh host memory.  So small inputs travel packed, in one
// copy; outputs of up to 256 MiB are written by the sweep itself into pinned
// memory, a slice of objects at a time, and copied from there, page faults
// included, while the next slices are swept.  No copy queue takes part: copies
// are kernels here, and two streams of a process with several libraries may
// share a hardware queue, where a copy waits for every sweep enqueued before it.
// Larger outputs go through device memory and staging buffers as before.
// Whole call, us: one star of 29 observations, 1188 bins, 204 -> 99; 136 stars
// x 100,000 bins, generalized FP32 (54 MB), 7678 -> 4770 (the sweep alone 2750 into device
// memory, ~3800 into pinned memory, coherent or not, where a copy kernel after it
// would take the difference; with slices copied on a second stream 5400, or 8700
// beside another library).
//
// Replaces the reference's GPU host path: computeObjectRanges
// (source/main.cu:468-510), computeNumBatches (main.cu:423-466),
// batchGPULSWrapper / batchGPULS (main.cu:742-1280), GPULSOneObject
// (main.cu:570-720) and pinnedMemoryCopyDtoH (main.cu:513-559).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <numeric>
#include <string>
#include <vector>

#include "ls_internal.h"

namespace lsamd {

// ---------------------------------------------------------------------------
// error state
// ---------------------------------------------------------------------------
namespace {
thread_local int t_err_code = LSAMD_OK;
thread_local std::string t_err_msg;
}  // namespace

int set_error(int code, const std::string &msg) {
    t_err_code = code;
    t_err_msg = msg;
    return code;
}

void clear_error() {
    t_err_code = LSAMD_OK;
    t_err_msg.clear();
}

// ---------------------------------------------------------------------------
// segmentation: objects are runs of equal ids (main.cu:468-510)
// ---------------------------------------------------------------------------
uint32_t count_runs(const uint32_t *id, uint64_t n) {
    if (n == 0) return 0;
    uint32_t k = 1;
    for (uint64_t i = 1; i < n; ++i) k += id[i] != id[i - 1];
    return k;
}

uint32_t run_offsets(const uint32_t *id, uint64_t n, uint64_t *off, uint32_t *ids) {
    if (n == 0) return 0;
    uint32_t k = 0;
    off[0] = 0;
    for (uint64_t i = 1; i < n; ++i) {
        if (id[i] != id[i - 1]) {
            if (ids) ids[k] = id[i - 1];
            off[++k] = i;
        }
    }
    if (ids) ids[k] = id[n - 1];
    off[++k] = n;
    return k;
}

// updateYerrorfactor (main.cu:1631-1662) with the reductions summed in index
// order; w = 1/sqrt(dy) is the reference's weight for this step.
template <typename R>
void precenter_host(R *y, const R *dy, uint64_t n) {
    R sumw = 0, dot = 0;
    for (uint64_t i = 0; i < n; ++i) sumw += (R)(1.0 / (double)std::sqrt(dy[i]));
    for (uint64_t i = 0; i < n; ++i) dot += (R)(1.0 / (double)std::sqrt(dy[i])) * y[i];
    const R shift = dot / sumw;
    for (uint64_t i = 0; i < n; ++i) y[i] = y[i] - shift;
}
template void precenter_host<float>(float *, const float *, uint64_t);
template void precenter_host<double>(double *, const double *, uint64_t);

// ---------------------------------------------------------------------------
// device contexts: per device, one stream and grow-only buffers, reused
// across calls
// ---------------------------------------------------------------------------
namespace {

struct DevBuf {
    void *p = nullptr;
    size_t cap = 0;
};

// Slices whose sweeps are enqueued, each with pinned memory of its own, before the
// first of them is copied on, at most.
constexpr size_t kAhead = 4;

struct Ctx {
    std::mutex mu;
    bool ready = false;
    int device = -1;
    hipStream_t stream = nullptr;       // uploads and sweeps
    hipStream_t copy_stream = nullptr;  // periodogram copy-back
    DevBuf in, ws, pgram, peaks;
    char *io = nullptr;                 // pinned: packed inputs, then small outputs
    bool busy = false;                  // a call is enqueued (or failed half-way)
    char *pinned = nullptr;             // staging buffers, or the slices under way (ring)
    size_t pinned_cap = 0;
    hipEvent_t ev[2] = {nullptr, nullptr};     // staging chunks (copy stream)
    hipEvent_t slice[kAhead] = {};             // sweep of a slice done (sweep stream)
};

// One context per device, for the device current on the calling thread.
// Calls on one device serialise on its context; calls on different devices
// (one host thread each) run side by side.  Contexts are never destroyed:
// HIP may be torn down first at exit.
Ctx *ctx_for_current_device(int *err) {
    static std::mutex mu;
    static std::map<int, Ctx *> *table = new std::map<int, Ctx *>();
    int dev = 0;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) {
        *err = set_error(LSAMD_ERR_NODEVICE, "no HIP device visible");
        return nullptr;
    }
    const hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        *err = set_error(LSAMD_ERR_HIP, std::string("hipGetDevice: ") + hipGetErrorString(e));
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(mu);
    Ctx *&c = (*table)[dev];
    if (!c) {
        c = new Ctx();
        c->device = dev;
    }
    return c;
}

#define HIP_OK(call)                                                                          \
    do {                                                                                      \
        hipError_t e_ = (call);                                                               \
        if (e_ != hipSuccess)                                                                 \
            return set_error(e_ == hipErrorOutOfMemory ? LSAMD_ERR_NOMEM : LSAMD_ERR_HIP,     \
                             std::string(#call) + ": " + hipGetErrorString(e_));              \
    } while (0)

// Pinned room of a context: packed inputs (larger ones are copied from the
// caller's arrays), and outputs (larger ones go through the staging buffers).
constexpr size_t kIoIn = size_t(1) << 20, kIoOut = size_t(8) << 20;
// Periodograms up to here are written into pinned memory in slices of at most
// kRingSlice.
constexpr size_t kRingTotal = size_t(256) << 20, kRingSlice = size_t(32) << 20;

int ctx_init(Ctx &c) {
    if (c.ready) return LSAMD_OK;
    HIP_OK(hipStreamCreateWithFlags(&c.stream, hipStreamNonBlocking));
    HIP_OK(hipStreamCreateWithFlags(&c.copy_stream, hipStreamNonBlocking));
    for (hipEvent_t &e : c.ev) HIP_OK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    for (hipEvent_t &e : c.slice) HIP_OK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    HIP_OK(hipHostMalloc(reinterpret_cast<void **>(&c.io), kIoIn + kIoOut, hipHostMallocCoherent));
    c.ready = true;
    return LSAMD_OK;
}

int ensure(DevBuf &b, size_t bytes) {
    if (bytes == 0) bytes = 256;
    if (b.cap >= bytes) return LSAMD_OK;
    if (b.p) {
        HIP_OK(hipFree(b.p));
        b.p = nullptr;
        b.cap = 0;
    }
    HIP_OK(hipMalloc(&b.p, bytes));
    b.cap = bytes;
    return LSAMD_OK;
}

constexpr size_t kPinnedChunk = size_t(64) << 20;  // a staging buffer, at most

// Pinned memory of a context: two staging buffers or kAhead slices, never both in
// one call (128 MiB at most either way, kept for the next call).
int ensure_pinned(Ctx &c, size_t bytes) {
    if (c.pinned_cap >= bytes) return LSAMD_OK;
    c.pinned_cap = 0;
    if (c.pinned) HIP_OK(hipHostFree(c.pinned));
    c.pinned = nullptr;
    HIP_OK(hipHostMalloc(reinterpret_cast<void **>(&c.pinned), bytes, hipHostMallocCoherent));
    c.pinned_cap = bytes;
    return LSAMD_OK;
}

// Pinned to pageable memory: first touches of fresh pages dominate, which
// threads share.
void host_copy(char *to, const char *from, size_t len) {
    if (len <= (size_t(1) << 20)) {
        std::memcpy(to, from, len);
        return;
    }
    const size_t parts = 8, step = (len + parts - 1) / parts;
#pragma omp parallel for num_threads(8) schedule(static)
    for (long long p = 0; p < (long long)parts; ++p) {
        const size_t a = (size_t)p * step;
        if (a < len) std::memcpy(to + a, from + a, std::min(step, len - a));
    }
}

// Device -> pageable host copy on the copy stream through two pinned staging
// buffers, so the DMA of one chunk overlaps the host copy of the previous one:
// four chunks or more, of 2 to 64 MiB.  Returns when the data is in dst.
int copy_to_host(Ctx &c, void *dst, const void *src, size_t bytes) {
    if (bytes == 0) return LSAMD_OK;
    const size_t chunk = std::min(kPinnedChunk, std::max(size_t(2) << 20, (bytes / 4 + 4095) & ~size_t(4095)));
    const int rc = ensure_pinned(c, 2 * chunk);
    if (rc) return rc;
    char *const stage[2] = {c.pinned, c.pinned + chunk};
    const size_t nch = (bytes + chunk - 1) / chunk;
    auto chunk_len = [&](size_t i) { return std::min(chunk, bytes - i * chunk); };
    const char *s = static_cast<const char *>(src);
    char *d = static_cast<char *>(dst);
    HIP_OK(hipMemcpyAsync(stage[0], s, chunk_len(0), hipMemcpyDeviceToHost, c.copy_stream));
    HIP_OK(hipEventRecord(c.ev[0], c.copy_stream));
    for (size_t i = 1; i <= nch; ++i) {
        if (i < nch) {
            HIP_OK(hipMemcpyAsync(stage[i & 1], s + i * chunk, chunk_len(i), hipMemcpyDeviceToHost,
                                  c.copy_stream));
            HIP_OK(hipEventRecord(c.ev[i & 1], c.copy_stream));
        }
        HIP_OK(hipEventSynchronize(c.ev[(i - 1) & 1]));
        host_copy(d + (i - 1) * chunk, stage[(i - 1) & 1], chunk_len(i - 1));
    }
    return LSAMD_OK;
}

// numpy.argmax of a row: the first NaN, else the first maximum.
template <typename R>
uint64_t row_argmax(const R *x, uint64_t n) {
    constexpr uint64_t kBlock = 512, kLanes = 16;
    R best = x[0];
    uint64_t at = 0;
    for (uint64_t b = 0; b < n; b += kBlock) {
        const uint64_t len = std::min(kBlock, n - b);
        const R *p = x + b;
        R m[kLanes];
        int odd[kLanes] = {};
        uint64_t i = 0;
        if (len >= kLanes) {
            for (uint64_t l = 0; l < kLanes; ++l) m[l] = p[l];
            for (; i + kLanes <= len; i += kLanes)
                for (uint64_t l = 0; l < kLanes; ++l) {
                    const R v = p[i + l];
                    m[l] = v > m[l] ? v : m[l];
                    odd[l] |= v != v;
                }
        }
        bool some = false;  // a NaN, or more than the best so far
        if (len >= kLanes)
            for (uint64_t l = 0; l < kLanes; ++l) some |= odd[l] != 0 || m[l] > best;
        for (; i < len; ++i) some |= p[i] != p[i] || p[i] > best;
        if (!some && !(b == 0 && best != best)) continue;
        for (i = 0; i < len; ++i) {
            if (p[i] != p[i]) return b + i;
            if (p[i] > best) {
                best = p[i];
                at = b + i;
            }
        }
    }
    return at;
}

double env_double(const char *name, double dflt) {
    const char *v = std::getenv(name);
    if (!v || !*v) return dflt;
    char *end = nullptr;
    const double x = std::strtod(v, &end);
    return (end && end != v) ? x : dflt;
}

}  // namespace
}  // namespace lsamd

using namespace lsamd;

extern "C" {

int lsamd_version(void) { return 10000; }  // 1.0.0

int lsamd_last_error_code(void) { return t_err_code; }
const char *lsamd_last_error(void) { return t_err_msg.c_str(); }
void lsamd_clear_error(void) { clear_error(); }

int lsamd_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

uint32_t lsamd_count_objects(const uint32_t *objectId, uint64_t n) {
    return objectId ? count_runs(objectId, n) : (n ? 1u : 0u);
}

uint32_t lsamd_object_offsets(const uint32_t *objectId, uint64_t n, uint64_t *offsets,
                              uint32_t *ids) {
    if (!objectId || !offsets) return 0;
    return run_offsets(objectId, n, offsets, ids);
}

int lsamd_batch_host(int variant, int dtype, int form, int normalize, int precenter,
                     const uint32_t *objectId, const void *t, void *y, const void *dy, uint64_t n,
                     double fmin, double fmax, uint32_t nf, void *pgram, uint32_t top_k,
                     uint32_t *peak_index, void *peak_power, void *peak_period,
                     uint32_t *num_objects_out) {
    clear_error();
    if (n == 0 || nf == 0) return set_error(LSAMD_ERR_INVALID, "lsamd_batch_host: empty input");
    if (!t || !y || (variant == LSAMD_GENERALIZED && !dy))
        return set_error(LSAMD_ERR_INVALID, "lsamd_batch_host: null input array");
    if (dtype != LSAMD_F32 && dtype != LSAMD_F64)
        return set_error(LSAMD_ERR_INVALID, "lsamd_batch_host: bad dtype");
    if (top_k != 0 && top_k != 1 && top_k != 3)
        return set_error(LSAMD_ERR_INVALID, "lsamd_batch_host: top_k must be 0, 1 or 3");
    if (!(fmax > fmin))
        return set_error(LSAMD_ERR_INVALID, "lsamd_batch_host: max_freq must exceed min_freq");
    const size_t rsz = dtype == LSAMD_F64 ? 8 : 4;

    // segmentation (a NULL id array means one object: reference MODE 2)
    std::vector<uint64_t> off;
    uint32_t K;
    if (objectId) {
        K = count_runs(objectId, n);
        off.resize((size_t)K + 1);
        run_offsets(objectId, n, off.data(), nullptr);
    } else {
        K = 1;
        off = {0, n};
    }
    if (num_objects_out) *num_objects_out = K;

    // reference side effect: the generalized variant pre-centres magY in place
    if (variant == LSAMD_GENERALIZED && precenter) {
        for (uint32_t k = 0; k < K; ++k) {
            if (dtype == LSAMD_F64)
                precenter_host(static_cast<double *>(y) + off[k],
                               static_cast<const double *>(dy) + off[k], off[k + 1] - off[k]);
            else
                precenter_host(static_cast<float *>(y) + off[k],
                               static_cast<const float *>(dy) + off[k], off[k + 1] - off[k]);
        }
    }

    int rc = LSAMD_OK;
    Ctx *cp = ctx_for_current_device(&rc);
    if (!cp) return rc;
    Ctx &c = *cp;
    std::lock_guard<std::mutex> lock(c.mu);
    rc = ctx_init(c);
    if (rc) return rc;

    // an earlier call that failed half-way may still use the pinned memory
    if (c.busy) {
        HIP_OK(hipStreamSynchronize(c.stream));
        HIP_OK(hipStreamSynchronize(c.copy_stream));
    }
    c.busy = true;

    // memory budget for the periodogram (computeNumBatches, main.cu:423-466):
    // a fraction of the free device memory, LSAMD_MEM_FRACTION (default 0.5),
    // or an absolute LSAMD_PGRAM_BUDGET_BYTES.  What an earlier call's buffer
    // holds needs no look at the free memory.
    const size_t per_obj = pgram ? (size_t)nf * rsz : 0;
    const double abs_budget = env_double("LSAMD_PGRAM_BUDGET_BYTES", 0.0);
    const double fraction = env_double("LSAMD_MEM_FRACTION", -1.0);
    uint32_t objs_per_batch = K;
    const bool ring_call = pgram && (size_t)K * per_obj <= kRingTotal && per_obj <= kRingSlice && !(abs_budget > 0) &&
                           fraction < 0;
    if (per_obj > 0 && !ring_call && (abs_budget > 0 || fraction >= 0 || c.pgram.cap / per_obj < K)) {
        size_t budget = (size_t)abs_budget;
        if (!(abs_budget > 0)) {
            size_t freeb = 0, totalb = 0;
            HIP_OK(hipMemGetInfo(&freeb, &totalb));
            budget = (size_t)((fraction >= 0 ? fraction : 0.5) * (double)freeb);
        }
        const size_t fit = std::max<size_t>(1, budget / per_obj);
        objs_per_batch = (uint32_t)std::min<size_t>(K, fit);
    }

    // Each memory-budget batch is swept in slices of objects: while the
    // periodogram of slice s is copied back, slice s+1 is swept, so the
    // end-to-end time approaches the longer of the two.  A slice in pinned memory
    // holds an eighth of the periodogram, 8 to 32 MiB, one in device memory 2 GiB
    // (at least 1 object; LSAMD_SLICE_BYTES overrides): each slice's copy through
    // the staging buffers restarts their pipeline.
    const size_t eighth = std::min(kRingSlice, std::max(size_t(8) << 20, (size_t)K * per_obj / 8));
    size_t kSliceBytes = (size_t)env_double("LSAMD_SLICE_BYTES", ring_call ? (double)eighth : (double)(size_t(2) << 30));
    if (ring_call) kSliceBytes = std::min(kRingSlice, kSliceBytes);
    const uint32_t objs_per_slice =
        per_obj > 0 ? (uint32_t)std::max<size_t>(1, std::min<size_t>(objs_per_batch, kSliceBytes / per_obj))
                    : objs_per_batch;
    std::vector<uint32_t> slice_start;
    for (uint32_t b0 = 0; b0 < K; b0 += objs_per_batch) {
        const uint32_t b1 = std::min(K, b0 + objs_per_batch);
        for (uint32_t s0 = b0; s0 < b1; s0 += objs_per_slice) slice_start.push_back(s0);
    }
    // longest objects first inside every slice (slice-local indices)
    std::vector<uint32_t> order(K);
    for (size_t i = 0; i < slice_start.size(); ++i) {
        const uint32_t s0 = slice_start[i];
        const uint32_t s1 = i + 1 < slice_start.size() ? std::min(slice_start[i + 1], K) : K;
        for (uint32_t k = s0; k < s1; ++k) order[k] = k - s0;
        std::stable_sort(order.begin() + s0, order.begin() + s1, [&](uint32_t a, uint32_t b) {
            return off[s0 + a + 1] - off[s0 + a] > off[s0 + b + 1] - off[s0 + b];
        });
    }

    // inputs, once: one device buffer, each part on a 256-byte boundary
    size_t in_bytes = 0;
    auto part = [](size_t &at, size_t bytes) {
        const size_t o = at;
        at += (bytes + 255) & ~size_t(255);
        return o;
    };
    const size_t in_t = part(in_bytes, n * rsz), in_y = part(in_bytes, n * rsz);
    const size_t in_dy = part(in_bytes, variant == LSAMD_GENERALIZED ? n * rsz : 0);
    const size_t in_off = part(in_bytes, ((size_t)K + 1) * 8), in_order = part(in_bytes, (size_t)K * 4);
    rc = ensure(c.in, in_bytes);
    if (rc) return rc;
    char *const in = static_cast<char *>(c.in.p);
    const bool packed = in_bytes <= kIoIn;
    auto upload = [&](size_t at, const void *from, size_t bytes) -> int {
        if (packed) std::memcpy(c.io + at, from, bytes);
        else HIP_OK(hipMemcpyAsync(in + at, from, bytes, hipMemcpyHostToDevice, c.stream));
        return LSAMD_OK;
    };
    rc = upload(in_t, t, n * rsz);
    if (!rc) rc = upload(in_y, y, n * rsz);
    if (!rc && variant == LSAMD_GENERALIZED) rc = upload(in_dy, dy, n * rsz);
    if (!rc) rc = upload(in_off, off.data(), ((size_t)K + 1) * 8);
    if (!rc) rc = upload(in_order, order.data(), (size_t)K * 4);
    if (rc) return rc;
    if (packed) HIP_OK(hipMemcpyAsync(in, c.io, in_bytes, hipMemcpyHostToDevice, c.stream));

    // outputs: the peaks, and behind them the periodogram of a small call, in one
    // run of pinned memory; a larger periodogram in the ring or a device buffer
    const uint32_t tk = top_k;
    size_t out_bytes = 0;
    const size_t out_idx = part(out_bytes, (size_t)K * tk * 4), out_pow = part(out_bytes, (size_t)K * tk * rsz);
    const size_t out_per = part(out_bytes, (size_t)K * tk * rsz), peak_bytes = out_bytes;
    const size_t out_pg = part(out_bytes, (size_t)K * per_obj);
    const bool small = out_bytes <= kIoOut && slice_start.size() == 1;
    const bool ring = ring_call && !small;
    const bool peaks_pinned = peak_bytes <= kIoOut;
    char *const io_out = c.io + kIoIn;
    if (!peaks_pinned) rc = ensure(c.peaks, peak_bytes);
    // (slices of the ring start on page boundaries)
    const size_t ring_step = ((size_t)objs_per_slice * per_obj + 4095) & ~size_t(4095);
    if (!rc && ring) rc = ensure_pinned(c, kAhead * ring_step);
    if (!rc && pgram && !ring && !small) rc = ensure(c.pgram, (size_t)objs_per_batch * per_obj);
    if (rc) return rc;
    char *const peaks = peaks_pinned ? io_out : static_cast<char *>(c.peaks.p);

    // slice i covers objects [s0, s1) and, inside its batch, periodogram rows
    // from (s0 - batch start); a slice never spans two batches
    auto slice_end = [&](size_t i) {
        const uint32_t s0 = slice_start[i];
        const uint32_t batch_end = std::min(K, (s0 / objs_per_batch) * objs_per_batch + objs_per_batch);
        return std::min(batch_end, s0 + objs_per_slice);
    };
    auto batch_row = [&](uint32_t k) { return (size_t)(k % objs_per_batch); };
    auto sweep_slice = [&](size_t i) -> int {
        const uint32_t s0 = slice_start[i], s1 = slice_end(i);
        lsamd_sweep_args a{};
        a.variant = variant;
        a.dtype = dtype;
        a.form = form;
        a.normalize = normalize;
        a.precenter = 0;  // already done on the host, in place
        a.num_objects = s1 - s0;
        a.num_freqs = nf;
        a.top_k = tk;
        a.num_obs = n;
        a.min_freq = fmin;
        a.max_freq = fmax;
        a.offsets = reinterpret_cast<const uint64_t *>(in + in_off) + s0;
        a.order = reinterpret_cast<const uint32_t *>(in + in_order) + s0;
        a.t = in + in_t;
        a.y = in + in_y;
        a.dy = variant == LSAMD_GENERALIZED ? in + in_dy : nullptr;
        a.pgram = !pgram  ? nullptr
                  : small ? io_out + out_pg
                  : ring  ? c.pinned + i % kAhead * ring_step
                          : static_cast<char *>(c.pgram.p) + batch_row(s0) * per_obj;
        // a call of one object may slice its observations; sub-sweeps of a
        // larger call never do, so batching cannot change any result
        a.obs_slices = K == 1 ? 0 : 1;
        if (tk) {
            a.peak_index = reinterpret_cast<uint32_t *>(peaks + out_idx) + (size_t)s0 * tk;
            a.peak_power = peaks + out_pow + (size_t)s0 * tk * rsz;
            a.peak_period = peaks + out_per + (size_t)s0 * tk * rsz;
        }
        const size_t wsb = lsamd_sweep_workspace_size(&a);
        int r = LSAMD_OK;
        if (c.ws.cap < wsb) {
            // growing the workspace frees it: wait for the sweeps using it
            HIP_OK(hipStreamSynchronize(c.stream));
            r = ensure(c.ws, wsb);
            if (r) return r;
        }
        r = lsamd_sweep(&a, c.ws.p, c.ws.cap, c.stream);
        if (r) return r;
        if (!small) HIP_OK(hipEventRecord(c.slice[i % kAhead], c.stream));
        return LSAMD_OK;
    };
    auto copy_slice = [&](size_t i) -> int {
        const uint32_t s0 = slice_start[i], s1 = slice_end(i);
        char *const to = static_cast<char *>(pgram) + (size_t)s0 * per_obj;
        const size_t bytes = (size_t)(s1 - s0) * per_obj;
        if (ring) {
            HIP_OK(hipEventSynchronize(c.slice[i % kAhead]));
            host_copy(to, c.pinned + i % kAhead * ring_step, bytes);
            return LSAMD_OK;
        }
        HIP_OK(hipStreamWaitEvent(c.copy_stream, c.slice[i % kAhead], 0));
        return copy_to_host(c, to, static_cast<char *>(c.pgram.p) + batch_row(s0) * per_obj, bytes);
    };
    // Within a batch the slices' rows are apart: the next sweeps are enqueued (as
    // many as the ring holds, else one) while a slice is copied back.  A new
    // batch reuses the rows, and is enqueued when the last slice before it is in
    // host memory (copy_slice returns then).
    const size_t ns = slice_start.size(), ahead = ring ? kAhead : 2;
    for (size_t i = 0, queued = 0; i < ns; ++i) {
        for (; queued < ns && queued < i + ahead &&
               slice_start[queued] / objs_per_batch == slice_start[i] / objs_per_batch;
             ++queued) {
            rc = sweep_slice(queued);
            if (rc) return rc;
        }
        if (pgram && !small) {
            rc = copy_slice(i);
            if (rc) return rc;
        }
    }
    // the peaks (and a small call's periodogram), then into the caller's arrays
    auto fetch = [&](void *to, size_t at, size_t bytes) -> int {
        if (to && !peaks_pinned) HIP_OK(hipMemcpyAsync(to, peaks + at, bytes, hipMemcpyDeviceToHost, c.stream));
        return LSAMD_OK;
    };
    if (tk) {
        rc = fetch(peak_index, out_idx, (size_t)K * tk * 4);
        if (!rc) rc = fetch(peak_power, out_pow, (size_t)K * tk * rsz);
        if (!rc) rc = fetch(peak_period, out_per, (size_t)K * tk * rsz);
        if (rc) return rc;
    }
    HIP_OK(hipStreamSynchronize(c.stream));
    if (tk && peaks_pinned) {
        if (peak_index) host_copy(reinterpret_cast<char *>(peak_index), io_out + out_idx, (size_t)K * tk * 4);
        if (peak_power) host_copy(static_cast<char *>(peak_power), io_out + out_pow, (size_t)K * tk * rsz);
        if (peak_period) host_copy(static_cast<char *>(peak_period), io_out + out_per, (size_t)K * tk * rsz);
    }
    if (pgram && small) host_copy(static_cast<char *>(pgram), io_out + out_pg, (size_t)K * per_obj);
    c.busy = false;
    return LSAMD_OK;
}

// numpy.argmax along the rows of a rows x cols array.
int lsamd_row_argmax(int dtype, const void *data, uint64_t rows, uint64_t cols, uint64_t *index) {
    if (!data || !index || cols == 0 || (dtype != LSAMD_F32 && dtype != LSAMD_F64))
        return set_error(LSAMD_ERR_INVALID, "lsamd_row_argmax: bad arguments");
#pragma omp parallel for num_threads(8) schedule(static) if (rows > 1 && rows * cols > 100000)
    for (long long r = 0; r < (long long)rows; ++r)
        index[r] = dtype == LSAMD_F64 ? row_argmax(static_cast<const double *>(data) + (uint64_t)r * cols, cols)
                                      : row_argmax(static_cast<const float *>(data) + (uint64_t)r * cols, cols);
    return LSAMD_OK;
}

int lsamd_cpu_batch(int variant, int dtype, int normalize, const uint32_t *objectId, const void *t,
                    void *y, const void *dy, uint64_t n, double fmin, double fmax, uint32_t nf,
                    void *pgram, int nthreads) {
    clear_error();
    return cpu_batch(variant, dtype, normalize, objectId, t, y, dy, n, fmin, fmax, nf, pgram,
                     nthreads);
}

int lsamd_cpu_single(int variant, int dtype, int normalize, const void *t, void *y, const void *dy,
                     uint64_t n, double fmin, double fmax, uint32_t nf, void *pgram, int nthreads) {
    clear_error();
    return cpu_single(variant, dtype, normalize, t, y, dy, n, fmin, fmax, nf, pgram, nthreads);
}

}  // extern "C"
