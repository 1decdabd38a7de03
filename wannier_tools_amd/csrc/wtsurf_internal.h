// Host-side declarations shared between the C-ABI layer and the kernel
// launchers.  Not part of the public interface (include/wtsurf.h is).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace wtsurf {

// Whether a ticket of the instance queue is past its end.  Tickets go on counting
// there (every wave or slot takes one before it stops), beyond what an int
// holds for the largest runs.
constexpr bool queue_empty(unsigned ticket, int ninst) { return ticket >= (unsigned)ninst; }
static_assert(queue_empty(0x80000003u, 0x7fffffff) && !queue_empty(0x7ffffffeu, 0x7fffffff),
              "tickets past 2^31");

// Workgroups that share one slot's GEMM round beyond order 112 at most.
constexpr int kMaxSplit = 6;
// Decimation state of one instance slot between rounds (device memory).
struct SlotState {
    int phase;              // empty, inverse next, GEMMs next, final inverse 0..2, done
    int t;                  // instance id
    int it;                 // current iteration (1-based)
    int status;             // bit0 singular solve, bit1 not converged
    double dl, dr;          // traces of the final inverses done so far
    double part[kMaxSplit]; // sum |alpha'| by share of a split GEMM round
    unsigned arrived;       // shares of the round that are done
};

// Arguments of one batched decimation launch (surfgreen_1985 over many
// (k, omega) instances, src/surfgreen.f90:7-137, with the trace epilogue of
// src/surfstat.f90:150-160 / src/fermiarc.f90:238-248).
struct DecimateArgs {
    const double2 *hk;      // [nk][2][NP*NP] padded H00(k), H01(k)
    const double *omega;    // [nomega], or null -> omega0 (grid mode, nomega = 1)
    const double *eta;      // [ninst] per-instance broadening, or null -> eta0
    const int *inst_k;      // [ninst] k index per instance, or null -> grid order
    const double *inst_w;   // [ninst] omega per instance (with inst_k), or null
    double eta0;
    double omega0;
    int nk, nomega, ninst;  // grid mode: ninst = nk*nomega, ik = t / nomega
    int n, nw;              // Ndim and Num_wann
    int itermax;
    double accuracy;
    const int *top;         // 1-based orbital lists (TopOrbitals / BottomOrbitals)
    int ntop;
    const int *bot;
    int nbot;
    double divisor;         // 1 (surfstat) or pi (SurfaceDOSkk)
    void *work;             // [kSlotSets*per_set][decimate_slot_bytes]
    SlotState *state;       // [kSlotSets*per_set], zeroed by decimate_run
    unsigned *queue;        // [2]: next instance ticket, finished instances
    double *dos_l, *dos_r, *dos_bulk;  // [ninst] in (ik + nk*iw) order
    int *iters;             // [ninst]
    int *status;            // [ninst] bit0 singular solve, bit1 not converged
    double2 *gfull;         // [ninst][3][n*n] GLL, GRR, GB or null
    // spin-resolved traces (src/surfstat.f90:163-192, src/fermiarc.f90:250-328):
    // 0 none; 1 GRR's sums over the top list (surfstat); 2 over the bottom
    // list in the last principal layer (SurfaceDOSkk)
    int spin_mode;
    double *spin;           // [2][3][ninst]: (left, right) x (sx, sy, sz), output order
    __host__ __device__ double *spin_out(size_t o, int side) const {
        return spin + (size_t)3 * side * ninst + o;
    }
};

// Slot sets of the decimation, one work stream each: the sets' rounds
// interleave on every CU (one Gauss-Jordan and one GEMM workgroup at a time).
constexpr int kSlotSets = 2;

// Streams and host-visible progress counter of the round driver: kSlotSets
// work streams and a counter-copy stream, all at default priority; events
// (two per set for the batch marks, two for the counter copies, one start
// mark); two pinned unsigneds.
constexpr int kRoundEvents = 2 * kSlotSets + 3;
struct RoundCtl {
    hipStream_t s[kSlotSets + 1];
    hipEvent_t ev[kRoundEvents];
    unsigned *pinned;
    int num_cu;
};

int padded_q(int n);        // NP/16 for order n
// Bytes of one FP64 slot of the orders whose matrix fits in LDS (Q <= 5):
// alpha, beta, m1, m2, g, eps_s, eps_t, each NP x NP complex double.
constexpr size_t slot_bytes_lds_fp64(int q) { return (size_t)7 * (16 * q) * (16 * q) * 16; }
int decimate_max_q();       // largest Q the decimation kernels are built for
// Slots per stream set for ninst instances on num_cu CUs (one of each kernel per CU).
int decimate_slots_per_set(int ninst, int num_cu);
// precision: 0 = FP64, 1 = FP32 inverse/GEMMs with FP64 accumulation and finals
size_t decimate_slot_bytes(int q, int precision);
// Enqueues the decimation of a.ninst instances on the work streams
// ctl.s[0..kSlotSets) and returns once every instance is counted finished
// (the work is complete when ctl.s[0] reaches the end of what was enqueued;
// ctl.s[0] waits for the others).
// Returns -2 when the count stops short of a.ninst within the round bound.
int decimate_run(const DecimateArgs &a, int q, int precision, int per_set, const RoundCtl &ctl);
// The persistent schedule (orders up to 16 * decimate_persistent_max_q()): one
// launch of nblocks workgroups on stream s, each running whole instances from
// the queue; slots 0..nblocks-1 of a.work.  Returns once the launch is queued.
int decimate_persistent_max_q();
int decimate_persistent_run(const DecimateArgs &a, int q, int precision, int nblocks,
                            hipStream_t s);
// Orders up to decimate_small_max_n() in FP64 on the vector ALUs: one
// workgroup per instance for its whole decimation, matrices in LDS, as many
// workgroups per CU as the LDS holds, instances from the queue (a.work and
// a.state unused).  Returns once the launch is queued on s.
int decimate_small_max_n();
int decimate_small_run(const DecimateArgs &a, int num_cu, hipStream_t s);
// The same up to decimate_tiny_max_n(), in the registers of one wave (tiny.hip).
int decimate_tiny_max_n();
int decimate_tiny_run(const DecimateArgs &a, int num_cu, hipStream_t s);

// FP64 orders up to decimate_mid_max_n() as rounds of two kernels with the
// inverse in registers (mid.hip).  State of one slot between rounds; two per
// slot (a round reads one and writes the other).
struct MidState {
    int phase;   // empty, in an iteration, done
    int t;       // instance id
    int it;      // current iteration (1-based)
    int status;  // bit0 singular solve, bit1 not converged
    int buf;     // which of the slot's two states the iteration reads
};
struct MidPlan {
    int sets = 1, per_set = 1;  // slot sets (one stream each) and slots per set
};
constexpr size_t kMidNoallocSlotBytes = (size_t)922112;  // slot of order 80
int decimate_mid_max_n();
size_t decimate_mid_slot_bytes(int n);
MidPlan decimate_mid_plan(int ninst, int num_cu);
// The plan cut to `most` slots, but to no fewer than two a CU (one launch of each
// set then still fills the chip).
void decimate_mid_limit(MidPlan &p, int num_cu, size_t most);
// Half as many slots; false if there is only one.
bool decimate_mid_halve(MidPlan &p);
// a.work: sets * per_set slots of decimate_mid_slot_bytes(a.n); state: 2 * sets
// * per_set records.  As decimate_run otherwise (-2: no progress).
int decimate_mid_run(const DecimateArgs &a, const MidPlan &plan, MidState *state, int num_cu,
                     const RoundCtl &ctl);

// Fourier sum H00(k), H01(k) (src/ham_qlayer2qlayer.f90:45-97).
struct FourierArgs {
    const double2 *hr;      // [nr][nw*nw] col-major per R, Hartree, /ndegen
    const int *irvec;       // [nr][3]
    const int *slot_begin;  // [nslot+1] R ranges sorted by R3 (device)
    int nslot;              // slots for R3 = d_lo .. d_lo+nslot-1
    int d_lo;
    int nr, nw, np, ijmax;
    const double *kpts;     // [nk][2]
    int nk;
    double2 *phase;         // [nk][nr] scratch
    double2 *hk;            // [nk][2][NP*NP] out (pad zero)
    int NP;
};
int fourier_launch(const FourierArgs &a, hipStream_t s);
// hk [nk][2][NP*NP] without its pads: h00 and h01 [nk][n*n].
int unpad_launch(const double2 *hk, int nk, int n, int NP, double2 *h00, double2 *h01, hipStream_t s);

// QPI autocorrelation over a k-plane (src/fermiarc.f90:496-560), device buffers.
constexpr int kKplaneMaxM = 2048;  // largest m1 (rows in LDS)
struct KplaneCorrArgs {
    const double *fields;   // [nfield][nky][nkx]
    int nkx, nky, m1, m2, nfield;
    double *folded;         // [nfield][m2][m1] scratch
    double *corr;           // kplane_corr_doubles() scratch: [slices][m2][m1]
    double *out;            // [nky][nkx]
};
int kplane_corr_max_m();
size_t kplane_corr_doubles(int m1, int m2, int nfield);
int kplane_corr_launch(const KplaneCorrArgs &k, hipStream_t s);
// dst [nfield][cols][rows] = src [nfield][rows][cols], device buffers.
int transpose_launch(const double *src, int rows, int cols, int nfield, double *dst, hipStream_t s);
// Longest path that kpath_jdos_launch stages in LDS (160 KB, two doubles a
// point): 9000 points, 50 rows 4.1 ms from global memory, 1.3 staged; 5121
// points, four rows 0.47 and 0.50.
constexpr int kJdosStagedMaxNk = 160 * 1024 / 16;
// k-path joint density of states (src/surfstat.f90:891-907); device buffers
// [nfield][nomega][nk] (k_fastest) or [nfield][nk][nomega].
int kpath_jdos_launch(const double *fields, int nk, int nomega, int nfield, bool k_fastest,
                      double *out, hipStream_t s);

}  // namespace wtsurf
