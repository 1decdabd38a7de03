// C-ABI layer of libwtsurf (declared in include/wtsurf.h): argument checks,
// device buffers owned by the context, launches on the context stream.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <numeric>
#include <string>
#include <vector>

#include "../../include/wtsurf.h"
#include "wtsurf_internal.h"

using namespace wtsurf;

namespace {

// Decimation stop rule of src/surfgreen.f90:39,42 (1e-16 as a real(4) literal).
constexpr int kRefItermax = 100;
constexpr double kRefAccuracy = (double)1e-16f;

template <typename T>
struct DevBuf {
    T *p = nullptr;
    size_t n = 0;
    int ensure(size_t want) {
        if (want <= n && p) return 0;
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
        if (want == 0) return 0;
        if (hipMalloc(&p, want * sizeof(T)) != hipSuccess) {
            (void)hipGetLastError();  // not to be taken for a later launch's
            p = nullptr;
            return -1;
        }
        n = want;
        return 0;
    }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
};

// Pinned host memory, grown on demand.
struct PinnedBuf {
    unsigned char *p = nullptr;
    size_t n = 0;
    int ensure(size_t want) {
        if (want <= n) return 0;
        release();
        if (hipHostMalloc((void **)&p, want, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            p = nullptr;
            return -1;
        }
        n = want;
        return 0;
    }
    void release() {
        if (p) (void)hipHostFree(p);
        p = nullptr;
        n = 0;
    }
};

}  // namespace

// ---------------------------------------------------------------------------
// Device scratch of wtsurf_surfgreen_1985_noalloc: one instance of order up to
// kNoallocMaxN (the orders of the persistent schedule), so the call needs no
// device allocation.  The array lives on every device the library
// runs on until the process ends; each device has its own copy at its own
// address, taken once per device with hipGetSymbolAddress.  Calls on one
// device share it, so calls that
// overlap on one device race.  The address is taken on the entry point's
// first call on a device, with that device current.  Layout (256-byte aligned
// pieces):
//   hk    padded H00, H01              2 NP^2 complex double
//   work  two decimation slots         2 slot_bytes_lds_fp64(Q), or one of mid.hip
//   state two SlotState or MidState, queue [2]
//   gfull GLL, GRR, GB                 3 n^2 complex double
//   outs  dos_l, dos_r, dos_bulk; iters, status, an empty orbital list
namespace {
constexpr int kNoallocMaxN = 80;
constexpr int kNoallocNP = 80;
constexpr size_t kAlign = 256;
constexpr size_t align_up(size_t x) { return (x + kAlign - 1) / kAlign * kAlign; }
constexpr size_t kOffHk = 0;
constexpr size_t kOffWork = kOffHk + align_up((size_t)2 * kNoallocNP * kNoallocNP * sizeof(double2));
constexpr size_t kOffState =
    kOffWork + align_up(std::max((size_t)kSlotSets * slot_bytes_lds_fp64(kNoallocNP / 16), kMidNoallocSlotBytes));
constexpr size_t kOffQueue =
    kOffState + align_up((size_t)kSlotSets * std::max(sizeof(SlotState), sizeof(MidState)));
constexpr size_t kOffG = kOffQueue + kAlign;
constexpr size_t kOffOut = kOffG + align_up((size_t)3 * kNoallocMaxN * kNoallocMaxN * sizeof(double2));
constexpr size_t kNoallocScratchBytes = kOffOut + kAlign;
static_assert(kNoallocScratchBytes <= ((size_t)2 << 20), "scratch kept under 2 MiB");
constexpr int kMaxDevices = 64;

std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices] = {};  // device address of `scratch` per device
int g_scratch_err[kMaxDevices] = {};    // hipGetSymbolAddress's error per device (0: none yet)
}  // namespace

// Referenced from host code (HIP_SYMBOL below), so the compiler gives it a
// global symbol in the device code object, which the runtime looks up by name.
// (An __attribute__((used)) would keep it a local symbol that the lookup does
// not find.)
static __device__ __align__(256) unsigned char scratch[kNoallocScratchBytes];

// Take this device's address of `scratch` (the device must be current).
static void scratch_setup(int device) {
    if (device < 0 || device >= kMaxDevices) return;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[device]) return;
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
        g_scratch_err[device] = e != hipSuccess ? (int)e : -1;
        (void)hipGetLastError();
        return;
    }
    g_scratch_ptr[device] = ptr;
}

static void *scratch_ptr(int device) {
    if (device < 0 || device >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    return g_scratch_ptr[device];
}

struct wtsurf_ctx {
    int device = 0;
    int num_cu = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev[3] = {nullptr, nullptr, nullptr};
    // round driver of the decimation: the other sets' work streams, the
    // counter stream, their events and a pinned progress counter
    hipStream_t aux[kSlotSets - 1] = {}, cnt = nullptr;
    hipEvent_t drv[kRoundEvents] = {};
    unsigned *pinned = nullptr;
    std::string err;

    // model
    bool has_model = false;
    int nw = 0, np = 0, nr = 0, ijmax = 0, n = 0;
    int nslot = 0, d_lo = 0;
    DevBuf<double2> hr;
    DevBuf<int> irvec, slot_begin;
    // stop rule and orbitals
    int itermax = kRefItermax;
    double accuracy = kRefAccuracy;
    int schedule = WTSURF_SCHEDULE_AUTO;
    std::vector<int> top, bot;
    bool orbitals_set = false;
    DevBuf<int> d_top, d_bot;
    // grid
    int nk = 0, nomega = 0;
    DevBuf<double> kpts, omega;
    DevBuf<double2> phase, hk, hpack;
    PinnedBuf hpin;  // pieces of H00 and H01 on their way to the caller
    DevBuf<double> qpi;  // fields, scratch and result of the QPI sums
    DevBuf<double> dos_l, dos_r, dos_b;
    DevBuf<int> iters, status;
    // per-instance batch (wtsurf_spectral_batch)
    DevBuf<int> inst_k;
    DevBuf<double> inst_w, inst_eta;
    // spin-resolved traces: mode for the next runs, the last run's outputs
    int spin_mode = WTSURF_SPIN_OFF;
    DevBuf<double> spin;
    size_t spin_ninst = 0;  // instances of the last run that took spin traces (0: none)
    // per-instance path (wtsurf_surfgreen_1985): padded H00/H01, full G out,
    // [dos_l, dos_r, dos_bulk, omega] and [iters, status, empty list]
    DevBuf<double2> hk1, gfull;
    DevBuf<double> one_d;
    DevBuf<int> one_i;
    // decimation workspace
    DevBuf<unsigned char> work, state;
    DevBuf<unsigned> queue;
    int per_set = 0;
    MidPlan plan;        // slots of the last ensure_work for mid.hip's rounds
    bool ran = false;    // a grid run is queued or done (wtsurf_grid_download)
    bool timed = false;  // ev[0..2] bracket the last grid or batch run

    int fail(const std::string &m) {
        err = m;
        return -1;
    }
    int hipfail(hipError_t e, const char *what) {
        err = std::string(what) + ": " + hipGetErrorString(e);
        return -2;
    }
};

#define WT_HIP(ctx, call)                                   \
    do {                                                    \
        hipError_t e_ = (call);                             \
        if (e_ != hipSuccess) return (ctx)->hipfail(e_, #call); \
    } while (0)

static int use_device(wtsurf_ctx *c) {
    WT_HIP(c, hipSetDevice(c->device));
    return 0;
}

// Upload the orbital lists (default 1..Num_wann for both, as
// src/readinput.f90:2857,2920-2935 for SOC = 0 single-cell defaults).
static int sync_orbitals(wtsurf_ctx *c) {
    if (!c->orbitals_set) {
        c->top.resize(c->nw);
        c->bot.resize(c->nw);
        std::iota(c->top.begin(), c->top.end(), 1);
        std::iota(c->bot.begin(), c->bot.end(), 1);
    }
    for (int v : c->top)
        if (v < 1 || v > c->n) return c->fail("top orbital index outside 1..Ndim");
    for (int v : c->bot)
        if (v < 1 || v > c->nw) return c->fail("bottom orbital index outside 1..Num_wann");
    if (c->d_top.ensure(std::max<size_t>(c->top.size(), 1)) ||
        c->d_bot.ensure(std::max<size_t>(c->bot.size(), 1)))
        return c->fail("out of device memory (orbital lists)");
    if (!c->top.empty())
        WT_HIP(c, hipMemcpy(c->d_top.p, c->top.data(), c->top.size() * sizeof(int),
                            hipMemcpyHostToDevice));
    if (!c->bot.empty())
        WT_HIP(c, hipMemcpy(c->d_bot.p, c->bot.data(), c->bot.size() * sizeof(int),
                            hipMemcpyHostToDevice));
    return 0;
}

// FP64 rounds of mid.hip's orders: the schedule asked for is the rounds, or
// automatic above the small kernel's orders, or has no kernel for the order.
static bool use_mid(int schedule, int n, int precision) {
    if (precision != WTSURF_FP64 || n > decimate_mid_max_n()) return false;
    if (schedule == WTSURF_SCHEDULE_PERSISTENT && padded_q(n) <= decimate_persistent_max_q())
        return false;
    return schedule == WTSURF_SCHEDULE_ROUNDS || n > decimate_small_max_n();
}

static int ensure_work(wtsurf_ctx *c, int schedule, int n, int precision, int ninst) {
    if (use_mid(schedule, n, precision)) {
        c->plan = decimate_mid_plan(ninst, c->num_cu);
        const size_t slot = decimate_mid_slot_bytes(n);
        auto want = [&] { return (size_t)c->plan.sets * c->plan.per_set * slot; };
        size_t free = 0, total = 0;
        if (want() > c->work.n && hipMemGetInfo(&free, &total) == hipSuccess)
            decimate_mid_limit(c->plan, c->num_cu, (free + c->work.n) / 4 / slot);
        while (want() > c->work.n) {
            c->work.release();
            if (!c->work.ensure(want())) break;
            // the rounds run with any number of slots
            if (!decimate_mid_halve(c->plan))
                return c->fail("out of device memory (decimation workspace)");
        }
        if (c->state.ensure(2 * (size_t)c->plan.sets * c->plan.per_set * sizeof(MidState)) ||
            c->queue.ensure(2))
            return c->fail("out of device memory (slot state)");
        return 0;
    }
    const int q = padded_q(n);
    const size_t per_slot = decimate_slot_bytes(q, precision);
    if (per_slot == 0) return c->fail("no decimation kernel for this order");
    const int per_set = decimate_slots_per_set(ninst, c->num_cu);
    const size_t want = (size_t)kSlotSets * per_set * per_slot;
    if (want > c->work.n) {
        c->work.release();
        if (c->work.ensure(want)) return c->fail("out of device memory (decimation workspace)");
    }
    if (c->state.ensure((size_t)kSlotSets * per_set * sizeof(SlotState)) || c->queue.ensure(2))
        return c->fail("out of device memory (slot state)");
    c->per_set = per_set;
    return 0;
}

extern "C" {

int wtsurf_ctx_create(int device, wtsurf_ctx **out) {
    if (!out) return -1;
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev) return -1;
    auto *c = new wtsurf_ctx();
    c->device = device;
    if (hipSetDevice(device) != hipSuccess) { delete c; return -2; }
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) { delete c; return -2; }
    c->num_cu = prop.multiProcessorCount;
    bool aux_ok = true;
    for (auto &a : c->aux) aux_ok = aux_ok && hipStreamCreateWithFlags(&a, hipStreamNonBlocking) == hipSuccess;
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess || !aux_ok ||
        hipStreamCreateWithFlags(&c->cnt, hipStreamNonBlocking) != hipSuccess ||
        hipHostMalloc((void **)&c->pinned, 2 * sizeof(unsigned), hipHostMallocDefault) != hipSuccess) {
        wtsurf_ctx_destroy(c);
        return -2;
    }
    for (auto &e : c->ev)
        if (hipEventCreate(&e) != hipSuccess) { wtsurf_ctx_destroy(c); return -2; }
    for (auto &e : c->drv)
        if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
            wtsurf_ctx_destroy(c);
            return -2;
        }
    *out = c;
    return 0;
}

void wtsurf_ctx_destroy(wtsurf_ctx *c) {
    if (!c) return;
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    for (auto a : c->aux)
        if (a) (void)hipStreamSynchronize(a);
    if (c->cnt) (void)hipStreamSynchronize(c->cnt);
    c->hr.release(); c->irvec.release(); c->slot_begin.release();
    c->d_top.release(); c->d_bot.release();
    c->kpts.release(); c->omega.release(); c->phase.release(); c->hk.release();
    c->hpack.release(); c->hpin.release(); c->qpi.release();
    c->dos_l.release(); c->dos_r.release(); c->dos_b.release();
    c->inst_k.release(); c->inst_w.release(); c->inst_eta.release(); c->spin.release();
    c->iters.release(); c->status.release(); c->work.release(); c->state.release();
    c->hk1.release(); c->gfull.release(); c->one_d.release(); c->one_i.release();
    c->queue.release();
    for (auto &e : c->ev)
        if (e) (void)hipEventDestroy(e);
    for (auto &e : c->drv)
        if (e) (void)hipEventDestroy(e);
    if (c->pinned) (void)hipHostFree(c->pinned);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    for (auto a : c->aux)
        if (a) (void)hipStreamDestroy(a);
    if (c->cnt) (void)hipStreamDestroy(c->cnt);
    delete c;
}

const char *wtsurf_last_error(const wtsurf_ctx *c) { return c ? c->err.c_str() : "null context"; }

int wtsurf_max_ndim(void) { return 16 * decimate_max_q(); }

int wtsurf_set_model(wtsurf_ctx *c, int nw, int np, int nr, int ijmax, const int *irvec,
                     const double *hr) {
    if (!c) return -1;
    if (nw <= 0 || np <= 0 || nr < 0 || ijmax < 0) return c->fail("invalid model sizes");
    if (nr > 0 && (!irvec || !hr)) return c->fail("null model arrays");
    if (int r = use_device(c)) return r;
    // a run in flight still reads the model, the orbital lists and hk
    if (int r = wtsurf_sync(c)) return r;
    // Slots d = R3 that H00/H01 can use: [-(np-1), 2np-1], clipped by ijmax.
    const int d_lo = std::max(-(np - 1), -ijmax), d_hi = std::min(2 * np - 1, ijmax);
    const int nslot = d_hi >= d_lo ? d_hi - d_lo + 1 : 0;
    std::vector<int> order;
    order.reserve(nr);
    for (int s = 0; s < nslot; ++s)
        for (int ir = 0; ir < nr; ++ir)
            if (irvec[3 * ir + 2] == d_lo + s) order.push_back(ir);
    std::vector<int> begin(nslot + 1, 0);
    {
        int pos = 0;
        for (int s = 0; s < nslot; ++s) {
            begin[s] = pos;
            for (int ir = 0; ir < nr; ++ir)
                if (irvec[3 * ir + 2] == d_lo + s) ++pos;
        }
        begin[nslot] = pos;
    }
    const int nsel = (int)order.size();
    const size_t nw2 = (size_t)nw * nw;
    std::vector<double2> hsel(std::max<size_t>((size_t)nsel * nw2, 1));
    std::vector<int> rsel(std::max(3 * nsel, 3));
    for (int q = 0; q < nsel; ++q) {
        const int ir = order[q];
        std::memcpy(&hsel[(size_t)q * nw2], hr + 2 * (size_t)ir * nw2, nw2 * sizeof(double2));
        for (int x = 0; x < 3; ++x) rsel[3 * q + x] = irvec[3 * ir + x];
    }
    if (c->hr.ensure(hsel.size()) || c->irvec.ensure(rsel.size()) ||
        c->slot_begin.ensure(begin.size()))
        return c->fail("out of device memory (model)");
    WT_HIP(c, hipMemcpy(c->hr.p, hsel.data(), hsel.size() * sizeof(double2), hipMemcpyHostToDevice));
    WT_HIP(c, hipMemcpy(c->irvec.p, rsel.data(), rsel.size() * sizeof(int), hipMemcpyHostToDevice));
    WT_HIP(c, hipMemcpy(c->slot_begin.p, begin.data(), begin.size() * sizeof(int),
                        hipMemcpyHostToDevice));
    c->nw = nw; c->np = np; c->nr = nsel; c->ijmax = ijmax; c->n = nw * np;
    c->nslot = nslot; c->d_lo = d_lo;
    c->has_model = true;
    c->nk = 0;  // grid must be re-uploaded for the new model
    c->ran = false;
    c->orbitals_set = false;  // orbital lists belong to a model: back to the defaults
    return sync_orbitals(c);
}

int wtsurf_set_stop_rule(wtsurf_ctx *c, int itermax, double accuracy) {
    if (!c) return -1;
    if (itermax < 1) return c->fail("itermax must be >= 1");
    if (!(accuracy >= 0.0)) return c->fail("accuracy must be >= 0");
    c->itermax = itermax;
    c->accuracy = accuracy;
    return 0;
}

int wtsurf_set_schedule(wtsurf_ctx *c, int schedule) {
    if (!c) return -1;
    if (schedule < WTSURF_SCHEDULE_ROUNDS || schedule > WTSURF_SCHEDULE_AUTO)
        return c->fail("unknown decimation schedule");
    if (int r = use_device(c)) return r;
    if (int r = wtsurf_sync(c)) return r;  // a run in flight owns the workspace
    c->schedule = schedule;
    return 0;
}

int wtsurf_set_orbitals(wtsurf_ctx *c, int ntop, const int *top, int nbot, const int *bot) {
    if (!c) return -1;
    if (ntop < 0 || nbot < 0 || (ntop && !top) || (nbot && !bot)) return c->fail("invalid orbital lists");
    if (c->has_model) {
        for (int i = 0; i < ntop; ++i)
            if (top[i] < 1 || top[i] > c->n) return c->fail("top orbital index outside 1..Ndim");
        for (int i = 0; i < nbot; ++i)
            if (bot[i] < 1 || bot[i] > c->nw) return c->fail("bottom orbital index outside 1..Num_wann");
    }
    c->top.assign(top, top + ntop);
    c->bot.assign(bot, bot + nbot);
    c->orbitals_set = true;
    if (!c->has_model) return 0;
    if (int r = use_device(c)) return r;
    if (int r = wtsurf_sync(c)) return r;  // a run in flight reads the lists
    return sync_orbitals(c);
}

static int run_fourier(wtsurf_ctx *c) {
    const int NP = 16 * padded_q(c->n);
    if (c->phase.ensure(std::max<size_t>((size_t)c->nk * std::max(c->nr, 1), 1)) ||
        c->hk.ensure((size_t)c->nk * 2 * NP * NP))
        return c->fail("out of device memory (Fourier)");
    FourierArgs fa{};
    fa.hr = c->hr.p; fa.irvec = c->irvec.p; fa.slot_begin = c->slot_begin.p;
    fa.nslot = c->nslot; fa.d_lo = c->d_lo; fa.nr = c->nr; fa.nw = c->nw; fa.np = c->np;
    fa.ijmax = c->ijmax; fa.kpts = c->kpts.p; fa.nk = c->nk; fa.phase = c->phase.p;
    fa.hk = c->hk.p; fa.NP = NP;
    if (fourier_launch(fa, c->stream)) return c->fail("Fourier kernel launch failed");
    return 0;
}

int wtsurf_ham_qlayer2qlayer(wtsurf_ctx *c, int nk, const double *kpts, double *h00, double *h01) {
    if (!c) return -1;
    if (!c->has_model) return c->fail("no model (wtsurf_set_model)");
    if (nk < 0 || (nk > 0 && (!kpts || !h00 || !h01))) return c->fail("invalid arguments");
    if (nk == 0) return 0;
    if (int r = use_device(c)) return r;
    if (int r = wtsurf_sync(c)) return r;  // a run in flight may still read kpts and hk
    c->ran = false;
    if (c->kpts.ensure(2 * (size_t)nk)) return c->fail("out of device memory");
    WT_HIP(c, hipMemcpy(c->kpts.p, kpts, 2 * (size_t)nk * sizeof(double), hipMemcpyHostToDevice));
    c->nk = nk;
    c->nomega = 0;
    if (int r = run_fourier(c)) return r;
    const int n = c->n, NP = 16 * padded_q(n);
    // The pads come off on the device, and pieces of 1 MiB (one k point's pair
    // at least) go through pinned memory: one is copied out while the next is
    // on its way.  (Copies straight to the caller's pageable arrays: 257 points
    // at Ndim 72 4.7 ms for 3.7, 100 at Ndim 48 1.7 for 1.3, one at Ndim 8 62
    // us for 41; pieces of 4 MiB 3.9, 1.7 ms and 41 us, of 256 KiB 8.0, 1.5 ms
    // and 41 us.)
    const size_t nn = (size_t)n * n, pair = 2 * nn * sizeof(double2);
    const int step = (int)std::min<size_t>(nk, std::max<size_t>(1, ((size_t)1 << 20) / pair));
    const int pieces = (nk + step - 1) / step;
    if (c->hpack.ensure(2 * step * 2 * nn)) return c->fail("out of device memory (H00, H01)");
    if (c->hpin.ensure(2 * step * pair)) return c->fail("out of pinned host memory (H00, H01)");
    int rc = 0;
    hipError_t e = hipSuccess;
    for (int i = 0; i <= pieces && !rc; ++i) {
        if (i < pieces) {
            const int ik = i * step, m = std::min(step, nk - ik);
            double2 *p0 = c->hpack.p + (size_t)(i & 1) * step * 2 * nn;
            if (unpad_launch(c->hk.p + (size_t)ik * 2 * NP * NP, m, n, NP, p0, p0 + m * nn, c->stream))
                rc = c->fail("H00/H01 unpadding launch failed");
            else if ((e = hipMemcpyAsync(c->hpin.p + (size_t)(i & 1) * step * pair, p0, m * pair,
                                         hipMemcpyDeviceToHost, c->stream)) != hipSuccess ||
                     (e = hipEventRecord(c->drv[i & 1], c->stream)) != hipSuccess)
                rc = c->hipfail(e, "download");
        }
        if (i > 0 && !rc) {
            const int h = (i - 1) & 1, ik = (i - 1) * step;
            const size_t b = std::min(step, nk - ik) * nn * sizeof(double2);
            if ((e = hipEventSynchronize(c->drv[h])) != hipSuccess) {
                rc = c->hipfail(e, "download");
                break;
            }
            const unsigned char *src = c->hpin.p + (size_t)h * step * pair;
            std::memcpy(h00 + 2 * (size_t)ik * nn, src, b);
            std::memcpy(h01 + 2 * (size_t)ik * nn, src + b, b);
        }
    }
    if (rc) (void)hipStreamSynchronize(c->stream);
    c->nk = 0;  // hk no longer matches an uploaded grid
    return rc;
}

// Per-instance (k index, omega, eta) device arrays for a batch run, or all null
// for the k x omega grid with one eta.
struct InstanceLists {
    const int *k = nullptr;
    const double *w = nullptr, *eta = nullptr;
};

// Device buffers one decimation run reads and writes: padded H00/H01, the
// outputs, the slot workspace and its state and queue.
struct RunBufs {
    const double2 *hk = nullptr;
    double *dos_l = nullptr, *dos_r = nullptr, *dos_b = nullptr;
    int *iters = nullptr, *status = nullptr;
    void *work = nullptr;
    void *state = nullptr;  // SlotState or MidState records
    unsigned *queue = nullptr;
    int per_set = 0;
    MidPlan plan;
    int schedule = WTSURF_SCHEDULE_AUTO;
};

// Enqueue the rounds of one decimation run on the context streams.
static int run_decimation(wtsurf_ctx *c, const RunBufs &b, int ninst, int nk, int nomega,
                          const double *d_omega, double eta, double divisor, double2 *gfull,
                          int n, int nw, const int *d_top, int ntop, const int *d_bot, int nbot,
                          int precision, InstanceLists inst, double *spin, double omega0 = 0.0) {
    DecimateArgs a{};
    a.omega0 = omega0;
    a.hk = b.hk; a.omega = d_omega; a.eta = inst.eta; a.inst_k = inst.k; a.inst_w = inst.w;
    a.eta0 = eta; a.nk = nk; a.nomega = nomega; a.ninst = ninst; a.n = n; a.nw = nw;
    a.itermax = c->itermax; a.accuracy = c->accuracy;
    a.top = d_top; a.ntop = ntop; a.bot = d_bot; a.nbot = nbot; a.divisor = divisor;
    a.work = b.work; a.state = static_cast<SlotState *>(b.state); a.queue = b.queue;
    a.dos_l = b.dos_l; a.dos_r = b.dos_r; a.dos_bulk = b.dos_b;
    a.iters = b.iters; a.status = b.status; a.gfull = gfull;
    if (spin) {
        a.spin_mode = c->spin_mode;
        a.spin = spin;
    }
    const int q = padded_q(n);
    if (precision == WTSURF_FP64 && n <= decimate_small_max_n() &&
        (b.schedule == WTSURF_SCHEDULE_SMALL || b.schedule == WTSURF_SCHEDULE_AUTO)) {
        if (decimate_small_run(a, c->num_cu, c->stream)) {
            const hipError_t e = hipGetLastError();
            return e != hipSuccess ? c->hipfail(e, "small-order decimation")
                                   : c->fail("small-order decimation launch failed");
        }
        return 0;
    }
    if (b.schedule == WTSURF_SCHEDULE_PERSISTENT && q <= decimate_persistent_max_q()) {
        // one workgroup per CU (at most one per instance), slots 0.. of the workspace
        const int nblocks = std::min(c->num_cu, ninst);
        if (nblocks > kSlotSets * b.per_set) return c->fail("decimation workspace too small");
        if (decimate_persistent_run(a, q, precision, nblocks, c->stream)) {
            const hipError_t e = hipGetLastError();
            return e != hipSuccess ? c->hipfail(e, "persistent decimation")
                                   : c->fail("persistent decimation launch failed");
        }
        return 0;
    }
    RoundCtl ctl{};
    ctl.s[0] = c->stream;
    for (int k = 1; k < kSlotSets; ++k) ctl.s[k] = c->aux[k - 1];
    ctl.s[kSlotSets] = c->cnt;
    for (int i = 0; i < kRoundEvents; ++i) ctl.ev[i] = c->drv[i];
    ctl.pinned = c->pinned;
    ctl.num_cu = c->num_cu;
    const bool mid = use_mid(b.schedule, n, precision);
    if (int r = mid ? decimate_mid_run(a, b.plan, static_cast<MidState *>(b.state), c->num_cu, ctl)
                    : decimate_run(a, q, precision, b.per_set, ctl)) {
        for (auto s : c->aux) (void)hipStreamSynchronize(s);  // rounds already queued there
        (void)hipStreamSynchronize(c->cnt);
        if (r == -2) return c->fail("decimation made no progress within its round bound");
        const hipError_t e = hipGetLastError();
        return e != hipSuccess ? c->hipfail(e, "decimation rounds") : c->fail("decimation rounds failed");
    }
    return 0;
}

static int check_order(wtsurf_ctx *c, int n, int precision) {
    const int q = padded_q(n);
    if (q > decimate_max_q()) return c->fail("Ndim exceeds the largest built decimation kernel");
    if (precision == WTSURF_FP32 && q > 5)
        return c->fail("WTSURF_FP32 is limited to Ndim <= 80: beyond that the doubling "
                       "recursion in FP32 diverges on some instances (use WTSURF_FP64)");
    // (the orders that mode has always taken)
    if (precision == WTSURF_MIXED && q > decimate_persistent_max_q())
        return c->fail("WTSURF_MIXED is built for Ndim <= 80 (use WTSURF_FP64)");
    return 0;
}

static bool known_precision(int p) {
    return p == WTSURF_FP64 || p == WTSURF_FP32 || p == WTSURF_MIXED;
}

// A grid or batch run into the context's own output buffers.
static int launch_decimation(wtsurf_ctx *c, int ninst, int nk, int nomega, const double *d_omega,
                             double eta, double divisor, int n, int nw, const int *d_top, int ntop,
                             const int *d_bot, int nbot, int precision,
                             InstanceLists inst = InstanceLists()) {
    if (int r = check_order(c, n, precision)) return r;
    // The mixed precision was FP64 but for the last sixth of the iterations, on
    // kernels of its own whatever the schedule; FP64 on the automatic schedule
    // takes two thirds of the time those took.
    RunBufs b;
    b.schedule = precision == WTSURF_MIXED ? (int)WTSURF_SCHEDULE_AUTO : c->schedule;
    if (precision == WTSURF_MIXED) precision = WTSURF_FP64;
    // the outputs first: the workspace takes what is left
    c->spin_ninst = 0;
    if (c->dos_l.ensure(ninst) || c->dos_r.ensure(ninst) || c->dos_b.ensure(ninst) ||
        c->iters.ensure(ninst) || c->status.ensure(ninst))
        return c->fail("out of device memory (outputs)");
    if (c->spin_mode != WTSURF_SPIN_OFF && c->spin.ensure((size_t)6 * ninst))
        return c->fail("out of device memory (spin traces)");
    if (int r = ensure_work(c, b.schedule, n, precision, ninst)) return r;
    b.hk = c->hk.p;
    b.dos_l = c->dos_l.p; b.dos_r = c->dos_r.p; b.dos_b = c->dos_b.p;
    b.iters = c->iters.p; b.status = c->status.p;
    b.work = c->work.p; b.state = c->state.p; b.queue = c->queue.p;
    b.per_set = c->per_set;
    b.plan = c->plan;
    double *spin = c->spin_mode != WTSURF_SPIN_OFF ? c->spin.p : nullptr;
    if (int r = run_decimation(c, b, ninst, nk, nomega, d_omega, eta, divisor, nullptr, n, nw, d_top,
                               ntop, d_bot, nbot, precision, inst, spin))
        return r;
    if (spin) c->spin_ninst = (size_t)ninst;
    return 0;
}

// Pad an n x n column-major complex matrix to NP x NP (zeros outside).
static void pad_matrix(const double *src, int n, int NP, double2 *dst) {
    for (int j = 0; j < NP; ++j)
        for (int i = 0; i < NP; ++i)
            dst[(size_t)j * NP + i] = (i < n && j < n)
                                          ? make_double2(src[2 * ((size_t)j * n + i)],
                                                         src[2 * ((size_t)j * n + i) + 1])
                                          : make_double2(0.0, 0.0);
}

int wtsurf_surfgreen_1985(wtsurf_ctx *c, int n, double omega, double eta, const double *h00,
                          const double *h01, double *gll, double *grr, double *gb, int *iters) {
    if (!c) return -1;
    if (n <= 0 || !h00 || !h01 || !gll || !grr || !gb) return c->fail("invalid arguments");
    if (int r = check_order(c, n, WTSURF_FP64)) return r;
    if (int r = use_device(c)) return r;
    // a grid run still in flight shares the slot workspace with this call
    if (int r = wtsurf_sync(c)) return r;
    const int NP = 16 * padded_q(n);
    std::vector<double2> pad((size_t)2 * NP * NP);
    pad_matrix(h00, n, NP, pad.data());
    pad_matrix(h01, n, NP, pad.data() + (size_t)NP * NP);
    // buffers of their own (grown on demand, kept for the next call), so that
    // the grid's H00/H01, energies and outputs stay as the last grid run left them
    if (c->hk1.ensure(pad.size()) || c->one_d.ensure(4) || c->one_i.ensure(3) ||
        c->gfull.ensure((size_t)3 * n * n) || ensure_work(c, c->schedule, n, WTSURF_FP64, 1))
        return c->fail("out of device memory");
    WT_HIP(c, hipMemcpy(c->hk1.p, pad.data(), pad.size() * sizeof(double2), hipMemcpyHostToDevice));
    WT_HIP(c, hipMemcpy(c->one_d.p + 3, &omega, sizeof(double), hipMemcpyHostToDevice));
    RunBufs b;
    b.schedule = c->schedule;
    b.hk = c->hk1.p;
    b.dos_l = c->one_d.p; b.dos_r = c->one_d.p + 1; b.dos_b = c->one_d.p + 2;
    b.iters = c->one_i.p; b.status = c->one_i.p + 1;
    b.work = c->work.p; b.state = c->state.p; b.queue = c->queue.p;
    b.per_set = c->per_set;
    b.plan = c->plan;
    // traces are not needed here: empty orbital lists (pointing at a valid int)
    if (int r = run_decimation(c, b, 1, 1, 1, c->one_d.p + 3, eta, 1.0, c->gfull.p, n, n,
                               c->one_i.p + 2, 0, c->one_i.p + 2, 0, WTSURF_FP64, InstanceLists(),
                               nullptr))
        return r;
    WT_HIP(c, hipStreamSynchronize(c->stream));
    std::vector<double2> g((size_t)3 * n * n);
    WT_HIP(c, hipMemcpy(g.data(), c->gfull.p, g.size() * sizeof(double2), hipMemcpyDeviceToHost));
    std::memcpy(gll, &g[0], (size_t)n * n * sizeof(double2));
    std::memcpy(grr, &g[(size_t)n * n], (size_t)n * n * sizeof(double2));
    std::memcpy(gb, &g[(size_t)2 * n * n], (size_t)n * n * sizeof(double2));
    if (iters) WT_HIP(c, hipMemcpy(iters, c->one_i.p, sizeof(int), hipMemcpyDeviceToHost));
    return 0;
}

int wtsurf_surfgreen_1985_noalloc(wtsurf_ctx *c, int n, double omega, double eta,
                                  const double *d_h00, const double *d_h01, double *d_gll,
                                  double *d_grr, double *d_gb, int *d_iters) {
    if (!c) return -1;
    if (n <= 0 || !d_h00 || !d_h01 || !d_gll || !d_grr || !d_gb) return c->fail("invalid arguments");
    if (n > kNoallocMaxN)
        return c->fail("wtsurf_surfgreen_1985_noalloc takes Ndim <= 80 (its device scratch is "
                       "sized for one instance of that order); use wtsurf_surfgreen_1985");
    if (int r = use_device(c)) return r;
    scratch_setup(c->device);  // once per device, on the first call there
    unsigned char *base = static_cast<unsigned char *>(scratch_ptr(c->device));
    if (!base) {
        const int e = c->device >= 0 && c->device < kMaxDevices ? g_scratch_err[c->device] : -1;
        return c->fail("no device scratch on this device (hipGetSymbolAddress failed: " +
                       std::to_string(e) + ")");
    }
    // rounds of a grid run still in flight use the context's streams and counter
    if (int r = wtsurf_sync(c)) return r;
    const int NP = 16 * padded_q(n);
    const size_t row = (size_t)n * sizeof(double2), prow = (size_t)NP * sizeof(double2);
    double2 *hk = reinterpret_cast<double2 *>(base + kOffHk);
    double2 *gfull = reinterpret_cast<double2 *>(base + kOffG);
    double *outs = reinterpret_cast<double *>(base + kOffOut);
    int *iouts = reinterpret_cast<int *>(base + kOffOut + 4 * sizeof(double));
    // the scratch keeps the last call's contents: pads and state start at zero
    WT_HIP(c, hipMemsetAsync(hk, 0, (size_t)2 * NP * prow, c->stream));
    WT_HIP(c, hipMemcpy2DAsync(hk, prow, d_h00, row, row, n, hipMemcpyDeviceToDevice, c->stream));
    WT_HIP(c, hipMemcpy2DAsync(hk + (size_t)NP * NP, prow, d_h01, row, row, n,
                               hipMemcpyDeviceToDevice, c->stream));
    RunBufs b;
    b.schedule = c->schedule;
    b.hk = hk;
    b.dos_l = outs; b.dos_r = outs + 1; b.dos_b = outs + 2;
    b.iters = iouts; b.status = iouts + 1;
    b.work = base + kOffWork;
    b.state = base + kOffState;
    b.queue = reinterpret_cast<unsigned *>(base + kOffQueue);
    b.per_set = 1;
    if (int r = run_decimation(c, b, 1, 1, 1, nullptr, eta, 1.0, gfull, n, n, iouts + 2, 0,
                               iouts + 2, 0, WTSURF_FP64, InstanceLists(), nullptr, omega))
        return r;
    const size_t nn = (size_t)n * n;
    WT_HIP(c, hipMemcpyAsync(d_gll, gfull, nn * sizeof(double2), hipMemcpyDeviceToDevice, c->stream));
    WT_HIP(c, hipMemcpyAsync(d_grr, gfull + nn, nn * sizeof(double2), hipMemcpyDeviceToDevice,
                             c->stream));
    WT_HIP(c, hipMemcpyAsync(d_gb, gfull + 2 * nn, nn * sizeof(double2), hipMemcpyDeviceToDevice,
                             c->stream));
    if (d_iters)
        WT_HIP(c, hipMemcpyAsync(d_iters, iouts, sizeof(int), hipMemcpyDeviceToDevice, c->stream));
    WT_HIP(c, hipStreamSynchronize(c->stream));
    return 0;
}

int wtsurf_grid_upload(wtsurf_ctx *c, int nk, const double *kpts, int nomega, const double *omega) {
    if (!c) return -1;
    if (!c->has_model) return c->fail("no model (wtsurf_set_model)");
    if (nk <= 0 || nomega <= 0 || !kpts || !omega) return c->fail("invalid grid");
    if ((long)nk * nomega > 0x7fffffffL) return c->fail("grid too large");
    if (int r = use_device(c)) return r;
    WT_HIP(c, hipStreamSynchronize(c->stream));  // a run in flight may still read the grid
    if (c->kpts.ensure(2 * (size_t)nk) || c->omega.ensure(nomega)) return c->fail("out of device memory");
    WT_HIP(c, hipMemcpy(c->kpts.p, kpts, 2 * (size_t)nk * sizeof(double), hipMemcpyHostToDevice));
    WT_HIP(c, hipMemcpy(c->omega.p, omega, (size_t)nomega * sizeof(double), hipMemcpyHostToDevice));
    c->nk = nk;
    c->nomega = nomega;
    c->ran = false;
    return 0;
}

int wtsurf_grid_run_async(wtsurf_ctx *c, double eta, double divisor, int precision) {
    if (!c) return -1;
    if (!c->has_model || c->nk <= 0 || c->nomega <= 0) return c->fail("no grid (wtsurf_grid_upload)");
    if (!known_precision(precision)) return c->fail("unknown precision mode");
    if (!(divisor != 0.0)) return c->fail("divisor must be non-zero");
    if (int r = use_device(c)) return r;
    WT_HIP(c, hipEventRecord(c->ev[0], c->stream));
    if (int r = run_fourier(c)) return r;
    WT_HIP(c, hipEventRecord(c->ev[1], c->stream));
    if (int r = launch_decimation(c, c->nk * c->nomega, c->nk, c->nomega, c->omega.p, eta, divisor,
                                  c->n, c->nw, c->d_top.p, (int)c->top.size(), c->d_bot.p,
                                  (int)c->bot.size(), precision))
        return r;
    WT_HIP(c, hipEventRecord(c->ev[2], c->stream));
    c->ran = true;
    c->timed = true;
    return 0;
}

int wtsurf_sync(wtsurf_ctx *c) {
    if (!c) return -1;
    if (int r = use_device(c)) return r;
    WT_HIP(c, hipStreamSynchronize(c->stream));
    for (auto a : c->aux) WT_HIP(c, hipStreamSynchronize(a));
    return 0;
}

int wtsurf_grid_timing(wtsurf_ctx *c, float *ms_fourier, float *ms_decimate) {
    if (!c) return -1;
    if (!c->timed) return c->fail("no completed run");
    float a = 0.f, b = 0.f;
    WT_HIP(c, hipEventSynchronize(c->ev[2]));
    WT_HIP(c, hipEventElapsedTime(&a, c->ev[0], c->ev[1]));
    WT_HIP(c, hipEventElapsedTime(&b, c->ev[1], c->ev[2]));
    if (ms_fourier) *ms_fourier = a;
    if (ms_decimate) *ms_decimate = b;
    return 0;
}

int wtsurf_grid_download(wtsurf_ctx *c, double *dos_l, double *dos_r, double *dos_bulk, int *iters,
                         int *status) {
    if (!c) return -1;
    if (!c->ran) return c->fail("no completed run");
    if (int r = use_device(c)) return r;
    WT_HIP(c, hipStreamSynchronize(c->stream));
    const size_t ni = (size_t)c->nk * c->nomega;
    if (dos_l) WT_HIP(c, hipMemcpy(dos_l, c->dos_l.p, ni * sizeof(double), hipMemcpyDeviceToHost));
    if (dos_r) WT_HIP(c, hipMemcpy(dos_r, c->dos_r.p, ni * sizeof(double), hipMemcpyDeviceToHost));
    if (dos_bulk) WT_HIP(c, hipMemcpy(dos_bulk, c->dos_b.p, ni * sizeof(double), hipMemcpyDeviceToHost));
    if (iters) WT_HIP(c, hipMemcpy(iters, c->iters.p, ni * sizeof(int), hipMemcpyDeviceToHost));
    if (status) WT_HIP(c, hipMemcpy(status, c->status.p, ni * sizeof(int), hipMemcpyDeviceToHost));
    return 0;
}

int wtsurf_spectral_batch(wtsurf_ctx *c, int nk, const double *kpts, int ninst, const int *k_index,
                          const double *omega, const double *eta, double divisor, int precision,
                          double *dos_l, double *dos_r, double *dos_bulk, int *iters, int *status) {
    if (!c) return -1;
    if (!c->has_model) return c->fail("no model (wtsurf_set_model)");
    if (nk <= 0 || ninst <= 0 || !kpts || !k_index || !omega || !eta || !dos_l || !dos_r || !dos_bulk)
        return c->fail("invalid arguments");
    if (!known_precision(precision)) return c->fail("unknown precision mode");
    if (!(divisor != 0.0)) return c->fail("divisor must be non-zero");
    for (int i = 0; i < ninst; ++i)
        if (k_index[i] < 0 || k_index[i] >= nk) return c->fail("k index outside 0..nk-1");
    if (int r = use_device(c)) return r;
    WT_HIP(c, hipStreamSynchronize(c->stream));  // a run in flight may still read the buffers
    if (c->kpts.ensure(2 * (size_t)nk) || c->inst_k.ensure(ninst) || c->inst_w.ensure(ninst) ||
        c->inst_eta.ensure(ninst))
        return c->fail("out of device memory");
    WT_HIP(c, hipMemcpy(c->kpts.p, kpts, 2 * (size_t)nk * sizeof(double), hipMemcpyHostToDevice));
    WT_HIP(c, hipMemcpy(c->inst_k.p, k_index, (size_t)ninst * sizeof(int), hipMemcpyHostToDevice));
    WT_HIP(c, hipMemcpy(c->inst_w.p, omega, (size_t)ninst * sizeof(double), hipMemcpyHostToDevice));
    WT_HIP(c, hipMemcpy(c->inst_eta.p, eta, (size_t)ninst * sizeof(double), hipMemcpyHostToDevice));
    c->nk = nk;
    c->nomega = 0;  // the grid no longer matches; wtsurf_grid_upload again for a grid run
    c->ran = false;
    c->timed = false;
    WT_HIP(c, hipEventRecord(c->ev[0], c->stream));
    if (int r = run_fourier(c)) return r;
    WT_HIP(c, hipEventRecord(c->ev[1], c->stream));
    InstanceLists inst;
    inst.k = c->inst_k.p;
    inst.w = c->inst_w.p;
    inst.eta = c->inst_eta.p;
    if (int r = launch_decimation(c, ninst, nk, 1, nullptr, 0.0, divisor, c->n, c->nw,
                                  c->d_top.p, (int)c->top.size(), c->d_bot.p, (int)c->bot.size(),
                                  precision, inst))
        return r;
    WT_HIP(c, hipEventRecord(c->ev[2], c->stream));
    c->timed = true;
    WT_HIP(c, hipStreamSynchronize(c->stream));
    const size_t ni = (size_t)ninst;
    WT_HIP(c, hipMemcpy(dos_l, c->dos_l.p, ni * sizeof(double), hipMemcpyDeviceToHost));
    WT_HIP(c, hipMemcpy(dos_r, c->dos_r.p, ni * sizeof(double), hipMemcpyDeviceToHost));
    WT_HIP(c, hipMemcpy(dos_bulk, c->dos_b.p, ni * sizeof(double), hipMemcpyDeviceToHost));
    if (iters) WT_HIP(c, hipMemcpy(iters, c->iters.p, ni * sizeof(int), hipMemcpyDeviceToHost));
    if (status) WT_HIP(c, hipMemcpy(status, c->status.p, ni * sizeof(int), hipMemcpyDeviceToHost));
    return 0;
}

int wtsurf_set_spin_traces(wtsurf_ctx *c, int mode) {
    if (!c) return -1;
    if (mode != WTSURF_SPIN_OFF && mode != WTSURF_SPIN_SURFSTAT && mode != WTSURF_SPIN_ARC)
        return c->fail("unknown spin trace mode");
    c->spin_mode = mode;
    return 0;
}

int wtsurf_spin_download(wtsurf_ctx *c, double *spin_l, double *spin_r) {
    if (!c) return -1;
    if (c->spin_ninst == 0) return c->fail("the last run took no spin traces");
    if (int r = use_device(c)) return r;
    WT_HIP(c, hipStreamSynchronize(c->stream));
    const size_t m = 3 * c->spin_ninst;
    if (spin_l) WT_HIP(c, hipMemcpy(spin_l, c->spin.p, m * sizeof(double), hipMemcpyDeviceToHost));
    if (spin_r) WT_HIP(c, hipMemcpy(spin_r, c->spin.p + m, m * sizeof(double), hipMemcpyDeviceToHost));
    return 0;
}

// The QPI sums' buffer grows on demand and is kept for the next call up to a
// bound (257 x 257 points and four fields take 8 MB, 512 x 512 on a path 34 MB).
static void trim_qpi(wtsurf_ctx *c) {
    constexpr size_t kKeepBytes = (size_t)256 << 20;
    if (c->qpi.n * sizeof(double) > kKeepBytes) c->qpi.release();
}

int wtsurf_kplane_autocorrelation(wtsurf_ctx *c, int nkx, int nky, int m1, int m2, int nfield,
                                  const double *fields, double *out) {
    if (!c) return -1;
    if (nkx < 1 || nky < 1 || nfield < 1 || !fields || !out) return c->fail("invalid arguments");
    if (m1 < 1 || m2 < 1 || m1 > nkx || m2 > nky)
        return c->fail("moduli must lie in 1..nkx and 1..nky");
    if (m1 > kplane_corr_max_m()) return c->fail("k-plane too large for the autocorrelation kernel");
    if (int r = use_device(c)) return r;
    const size_t plane = (size_t)nkx * nky;
    DevBuf<double> &buf = c->qpi;
    const size_t corr = kplane_corr_doubles(m1, m2, nfield);
    if (buf.ensure((size_t)nfield * plane + (size_t)nfield * m1 * m2 + corr + plane))
        return c->fail("out of device memory (k-plane autocorrelation)");
    KplaneCorrArgs k{};
    k.fields = buf.p;
    k.nkx = nkx; k.nky = nky; k.m1 = m1; k.m2 = m2; k.nfield = nfield;
    k.folded = buf.p + (size_t)nfield * plane;
    k.corr = k.folded + (size_t)nfield * m1 * m2;
    k.out = k.corr + corr;
    int rc = 0;
    hipError_t e;
    if ((e = hipMemcpyAsync(buf.p, fields, (size_t)nfield * plane * sizeof(double),
                            hipMemcpyHostToDevice, c->stream)) != hipSuccess)
        rc = c->hipfail(e, "upload");
    else if (kplane_corr_launch(k, c->stream))
        rc = c->fail("k-plane autocorrelation launch failed");
    else if ((e = hipMemcpyAsync(out, k.out, plane * sizeof(double), hipMemcpyDeviceToHost,
                                 c->stream)) != hipSuccess ||
             (e = hipStreamSynchronize(c->stream)) != hipSuccess)
        rc = c->hipfail(e, "download");
    if (rc) (void)hipStreamSynchronize(c->stream);
    trim_qpi(c);
    return rc;
}

static int kpath_jdos(wtsurf_ctx *c, int nk, int nomega, int nfield, bool k_fastest,
                      const double *fields, double *out) {
    if (!c) return -1;
    if (nk < 1 || nomega < 1 || nfield < 1 || !fields || !out) return c->fail("invalid arguments");
    if (int r = use_device(c)) return r;
    const size_t n = (size_t)nfield * nomega * nk;
    DevBuf<double> &buf = c->qpi;
    if (buf.ensure(2 * n)) return c->fail("out of device memory (k-path jdos)");
    int rc = 0;
    hipError_t e;
    // a long path with the energy fastest: the two halves take turns
    const bool turn = !k_fastest && nk > kJdosStagedMaxNk;
    double *in = turn ? buf.p + n : buf.p, *res = turn ? buf.p : buf.p + n;
    if ((e = hipMemcpyAsync(in, fields, n * sizeof(double), hipMemcpyHostToDevice, c->stream)) !=
        hipSuccess)
        rc = c->hipfail(e, "upload");
    else if ((turn && transpose_launch(in, nk, nomega, nfield, buf.p, c->stream)) ||
             kpath_jdos_launch(buf.p, nk, nomega, nfield, k_fastest || turn, buf.p + n, c->stream) ||
             (turn && transpose_launch(buf.p + n, nomega, nk, nfield, res, c->stream)))
        rc = c->fail("k-path jdos launch failed");
    else if ((e = hipMemcpyAsync(out, res, n * sizeof(double), hipMemcpyDeviceToHost,
                                 c->stream)) != hipSuccess ||
             (e = hipStreamSynchronize(c->stream)) != hipSuccess)
        rc = c->hipfail(e, "download");
    if (rc) (void)hipStreamSynchronize(c->stream);
    trim_qpi(c);
    return rc;
}

int wtsurf_kpath_jdos(wtsurf_ctx *c, int nk, int nomega, int nfield, const double *fields,
                      double *out) {
    return kpath_jdos(c, nk, nomega, nfield, true, fields, out);
}

int wtsurf_kpath_jdos_energy_fastest(wtsurf_ctx *c, int nk, int nomega, int nfield,
                                     const double *fields, double *out) {
    return kpath_jdos(c, nk, nomega, nfield, false, fields, out);
}

int wtsurf_spectral_grid(wtsurf_ctx *c, int nk, const double *kpts, int nomega, const double *omega,
                         double eta, double divisor, int precision, double *dos_l, double *dos_r,
                         double *dos_bulk, int *iters, int *status) {
    if (int r = wtsurf_grid_upload(c, nk, kpts, nomega, omega)) return r;
    if (int r = wtsurf_grid_run_async(c, eta, divisor, precision)) return r;
    if (int r = wtsurf_sync(c)) return r;
    return wtsurf_grid_download(c, dos_l, dos_r, dos_bulk, iters, status);
}

}  // extern "C"
