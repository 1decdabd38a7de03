// FP64 decimation for orders up to 112 as rounds of two kernels
// (src/surfgreen.f90:74-134 over many instances).  An iteration is
//
//   g = (z - eps_i)^-1                                       mid_inverse_kernel
//   [m1; m2] = [alpha; beta] g                               mid_gemm_kernel
//   [m1; m2] [alpha beta] = [alpha'  d_eps_s; d_eps_t  beta'] mid_gemm_kernel
//
// with eps_s += m1 beta, eps_t += m2 alpha and eps_i = eps_s + eps_t - H00
// (every iteration adds both products to eps_i, starting from H00 for all
// three).  The orders are padded to nb = 8 KT (pad rows and columns zero).
// The second product is one product of the stacked [m1; m2] with [alpha
// beta], cut into strips of 16 rows of the 2 nb (KT of them) and tiles of 16
// of the 2 nb columns (KT of them): no order is padded further to the MFMA
// tile.  A slot holds its state twice (one read, one written).
//
// Slots come in up to two sets, one per stream, so that the tail of one
// set's launch is filled by the other's.  A slot keeps its state in global
// memory between rounds and takes the next (k, omega) instance from a device
// counter once its previous one has converged.
#include <algorithm>
#include <utility>

#include "decimate_common.h"

namespace wtsurf {

namespace {

// Per-slot workspace: two states (read one, write the other), g, and the
// partial sums of |alpha'_ij| by tile.  Complex elements, nb = 8 KT:
//   ab  [alpha beta] (nb x 2 nb) in fragments: element (k, c) at
//       ((c / 16) KS + k / 4) 64 + c % 16 + 16 (k % 4), KS = nb / 4, so that
//       lane i + 16 q of fragment (t, s) is element (4 s + q, 16 t + i): the
//       1 KB a wave's MFMA step takes from it is contiguous
//   eps eps_s then eps_t, column-major
//   g   in fragments as ab (MT tiles; the half tile of an odd KT is padding)
template <int KT>
struct MidLay {
    static constexpr int NB = 8 * KT;
    static constexpr int KS = 2 * KT;
    static constexpr int MT = (KT + 1) / 2;  // 16-wide tiles of an nb-wide matrix
    static constexpr int AB = 2 * NB * NB;
    static constexpr int ST = 2 * AB;        // one state: ab, eps
    static constexpr int G = 16 * MT * NB;
    static constexpr size_t bytes =
        (size_t)(2 * ST + G) * sizeof(double2) + (size_t)MT * MT * sizeof(double);
    static constexpr size_t stride = (bytes + 255) / 256 * 256;
    // place of element (k, c) of ab or g
    __device__ static __forceinline__ int frag(int k, int c) {
        return ((c >> 4) * KS + (k >> 2)) * 64 + (c & 15) + 16 * (k & 3);
    }
};
static_assert(MidLay<10>::stride <= kMidNoallocSlotBytes, "slot larger than its host-side bound");

template <int KT>
struct MidSlot {
    using L = MidLay<KT>;
    double2 *z, *g;
    double *part;
    __device__ MidSlot(void *work, int slot) {
        unsigned char *base = reinterpret_cast<unsigned char *>(work) + (size_t)slot * L::stride;
        z = reinterpret_cast<double2 *>(base);
        g = z + 2 * L::ST;
        part = reinterpret_cast<double *>(g + L::G);
    }
    __device__ double2 *ab(int b) const { return z + b * L::ST; }
    __device__ double2 *eps(int b) const { return z + b * L::ST + L::AB; }
};

enum : int { kMidEmpty = 0, kMidLoop = 1, kMidDone = 2 };

// The element at a byte offset from a uniform base: base in scalar registers,
// offset in one vector register.
__device__ __forceinline__ double2 frag_at(const double2 *base, unsigned off) {
    return *reinterpret_cast<const double2 *>(reinterpret_cast<const char *>(base) + off);
}

// ---------------------------------------------------------------------------
// Both products of one iteration, one wave per strip of 16 rows of [alpha;
// beta] (and per share of the output columns when csplit > 1).
//
// An FP64 16x16x4 MFMA holds its SIMD for 64 cycles and a complex step is
// four of them, so one 1 KB operand fragment feeds 256 cycles: the fragments
// come straight from L2 with no LDS stage, no barrier and no wave waiting for
// another.  Bound by the matrix cores (busy 75% of the launches' time at
// order 72 alone on the chip, the rest their starts and ends; 576 us for 2048
// instances, where the LDS-staged kernel it replaces took 132 us for 256).  The
// fragments are contiguous in memory for the cache's sake: as 64 B pieces of
// column-major matrices they kept its lookups busy all the time, and 1024
// instances took 393 us where they then took 313 contiguous (288 now).  The
// MFMAs are issued transposed (the shared matrix as the A
// operand, the strip as the B operand): the accumulators of the first
// product, m^T, are then laid out exactly as the B operand of the second, and
// m1, m2 never leave the registers.
template <int KT>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(KT <= 10 ? 3 : 2)))
mid_gemm_kernel(void *work, const MidState *__restrict__ state, int slots, int csplit) {
    using L = MidLay<KT>;
    using P = Prec<double>;
    constexpr int NB = L::NB, MT = L::MT, KS = L::KS;
    // tasks of one slot on one XCD (blocks go round robin over the eight), so
    // that its matrices are fetched into one L2
    const int b = blockIdx.x;
    const int per = KT * csplit;
    const int qd = b >> 3;
    const int slot = (qd / per) * 8 + (b & 7);
    if (slot >= slots) return;
    const MidState *st = state + slot;
    if (uniform(st->phase) != kMidLoop) return;
    const int rem = qd % per;
    const int strip = rem % KT, share = rem / KT;
    const int t0 = KT * share / csplit, t1 = KT * (share + 1) / csplit;
    const MidSlot<KT> w(work, slot);
    const int buf = uniform(st->buf);
    const double2 *__restrict__ AB = w.ab(buf), *__restrict__ E = w.eps(buf);
    const double2 *__restrict__ G = w.g;
    double2 *__restrict__ ABo = w.ab(buf ^ 1), *__restrict__ Eo = w.eps(buf ^ 1);
    const int lane = threadIdx.x;
    const int j = lane & 15, q = lane >> 4;
    const int R = 16 * strip + j;            // row of [alpha; beta]
    const bool top = R < NB;
    const int k = top ? R : R - NB;          // its row in alpha or beta

    // m^T tiles: register v of tile t is m[R][16 t + 4 v + q]
    v4d mR[MT], mI[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) mR[t] = mI[t] = v4d{0, 0, 0, 0};
    // One k step: the strip's fragment (64 B segments of ab) and the MT
    // fragments of g.  Two in flight by turns; the barriers keep the
    // scheduler from pulling a load down to its use.
    struct Step {
        double2 a, g[MT];
    };
    constexpr unsigned kFrag = 64 * sizeof(double2);
    const unsigned lo = (unsigned)lane * sizeof(double2);
    // element (k, c + q) of ab, c = 4 s for a row of alpha, nb + 4 s for one of
    // beta
    const unsigned ro = ((k >> 2) * 64 + 16 * (k & 3) + q) * sizeof(double2);
    auto load_step = [&](Step &f, int s) {
        auto at = [&](int c) { return (unsigned)((c >> 4) * (KS * 64) + (c & 15)) * (unsigned)sizeof(double2); };
        f.a = frag_at(AB, ro + (top ? at(4 * s) : at(NB + 4 * s)));
#pragma unroll
        for (int t = 0; t < MT; ++t) f.g[t] = frag_at(G + (t * KS + s) * 64, lo);
    };
    auto multiply = [&](const Step &f) {
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            mR[t] = P::mfma(f.g[t].x, f.a.x, mR[t]);
            mI[t] = P::mfma(f.g[t].x, f.a.y, mI[t]);
            mR[t] = mfma_neg(f.g[t].y, f.a.y, mR[t]);
            mI[t] = P::mfma(f.g[t].y, f.a.x, mI[t]);
        }
    };
    {
        Step f0, f1;
        load_step(f0, 0);
#pragma unroll 1
        for (int s = 0; s < KS; s += 2) {  // KS is even
            load_step(f1, s + 1);
            __builtin_amdgcn_sched_barrier(0);
            multiply(f0);
            __builtin_amdgcn_sched_barrier(0);
            load_step(f0, s + 2 < KS ? s + 2 : s);
            __builtin_amdgcn_sched_barrier(0);
            multiply(f1);
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // the second product, one 16-column tile of [alpha beta] at a time; a
    // fragment register is loaded again right after its use, GS steps ahead
    constexpr int GS = KT % 3 == 0 ? 6 : KT % 5 == 0 ? 5 : KT % 7 == 0 ? 7
                     : KT == 11 || KT == 13 ? KT : KT % 2 == 0 ? 4 : 2;
    constexpr int NG = KS / GS;
    static_assert(NG * GS == KS, "whole groups");
    const double2 *col = AB + t0 * (KS * 64);
    double2 fr[GS];
#pragma unroll
    for (int i = 0; i < GS; ++i) fr[i] = frag_at(col, lo + i * kFrag);
    // eps quadrants accumulate: element (R, c) where exactly one of R, c is
    // below nb
    const int eb = top ? k - NB * NB : NB * NB + k;
    const int ob = (k >> 2) * 64 + 16 * (k & 3) + q;
    for (int t = t0; t < t1; ++t) {
        const double2 *nxt = t + 1 < t1 ? col + KS * 64 : col;
        double2 old[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int c = 16 * t + 4 * v + q;
            old[v] = make_double2(0.0, 0.0);
            if (top != (c < NB)) old[v] = E[eb + c * NB];
        }
        v4d pR = {0, 0, 0, 0}, pI = {0, 0, 0, 0};
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int i = 0; i < GS; ++i) {
                const int s = g * GS + i;
                const double mx = mR[s / 4][s % 4], my = mI[s / 4][s % 4];
                const double2 f = fr[i];
                pR = P::mfma(f.x, mx, pR);
                pI = P::mfma(f.x, my, pI);
                pR = mfma_neg(f.y, my, pR);
                pI = P::mfma(f.y, mx, pI);
                fr[i] = g + 1 < NG ? frag_at(col + 64 * (s + GS), lo) : frag_at(nxt + 64 * i, lo);
                __builtin_amdgcn_sched_barrier(0);
            }
        col = nxt;
        double asum = 0.0;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int c = 16 * t + 4 * v + q;
            const double2 o = make_double2(pR[v], pI[v]);
            if (top != (c < NB))
                Eo[eb + c * NB] = cadd(old[v], o);
            else
                ABo[t * (KS * 64) + 4 * v + ob] = o;
            if (16 * strip < NB && 16 * t < NB) {
                const double m = cabs_scaled(o.x, o.y);
                if (top && c < NB) asum += m;
            }
        }
        if (16 * strip < NB && 16 * t < NB) {
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) asum += __shfl_xor(asum, off, 64);
            if (lane == 0) w.part[strip * MT + t] = asum;
        }
    }
}

// ---------------------------------------------------------------------------
// Gauss-Jordan inverses, one workgroup each, the matrix in the registers of
// W waves (3 up to order 80, 7 beyond): lane (a = lane % 8, b = lane / 8) of wave w holds rows a + 8 s
// (s < KT) of columns 8 (w + W t) + b (t < CL).  Partial pivoting on
// |re| + |im| over the rows not yet used (the izamax rule of zgesv, the lowest
// row on ties), rows never swapped: step c's pivot row p keeps its
// values unscaled, standing for 1/pivot times itself, takes every later step
// like any other row and is scaled once at the end; element (row r, column c)
// is then X^-1[step of r][pivot row of step c].
//
// Columns are eliminated in panels of 8, one register group t of one wave, by
// one more wave: it takes the panel from LDS, runs its steps by itself and
// publishes the panel's columns M.  The others then take the pivot rows T of their own columns out of their
// registers and add M T, on the vector ALUs, whose FP64 rate is that of the
// matrix cores: the group of the next panel first, which that wave then
// eliminates while they update the rest.
//
// What it is bound by: an inverse alone is a chain of n pivot searches and
// reciprocals (2048 of order 72 alone on the chip 459 us, its vector ALUs busy 40%
// of it).  In registers two to three instances fit a CU (in LDS one
// does), and the updates of the others fill the waits of one's panels.
template <int KT>
struct MidGj {
    // Four waves a workgroup: those of three or five leave SIMDs idle (the
    // dispatcher refills them badly: 2048 workgroups of three waves take 1141
    // us where 1024 of four take 760 us).
    // Eight where the matrix needs the registers of two waves a SIMD.
    static constexpr int W = KT <= 10 ? 3 : 7;
    static constexpr int CL = (KT + W - 1) / W;  // column groups of the first waves
    static constexpr int NT = 64 * (W + 1);
    static constexpr int LDM = 8 * KT + (KT % 2 ? 0 : 8);  // columns on alternate halves of the banks
    // waves per SIMD that the registers are capped for
    static constexpr int OCC = W == 7 ? 2 : KT * CL <= 16 ? 4 : KT * CL <= 30 ? 3 : 2;
};

template <int KT>
struct MidGjShared {
    using C = MidGj<KT>;
    static constexpr int NB = 8 * KT;
    double2 m[2][8][C::LDM];      // a panel's columns after its elimination, by panel parity
    double2 pan[8][C::LDM];       // the next panel's columns before it
    double2 t[C::W][8][C::CL][8]; // a panel's pivot rows, each wave's own columns
    double2 rpiv[NB];             // 1 / pivot of step c
    int pivrow[NB];               // pivot row of step c
    int pivstep[NB];              // step at which row i was the pivot
    int sing;                     // a column without a pivot
    int tk;                       // instance taken from the queue
    double2 diag[NB], part[NB];   // final inverses: G(i, i), G(i, spin partner)
};

// A wave's role (0 .. W - 1: columns, W: panels), another one for the same
// SIMD in every other workgroup.
template <int KT>
__device__ __forceinline__ int mid_wave(int tid) {
    return (uniform(tid >> 6) + (int)blockIdx.x) % (MidGj<KT>::W + 1);
}

// d of lane 8 a + k to every lane 8 a + b (two DPP row broadcasts, one for each
// half of a row of 16 lanes).
template <int K>
__device__ __forceinline__ double group_bcast(double d) {
    const long long v = __double_as_longlong(d);
    long long r = __builtin_amdgcn_mov_dpp(v, 0x150 + K, 0xf, 0x3, false);
    r = __builtin_amdgcn_update_dpp(r, v, 0x158 + K, 0xf, 0xc, false);
    return __longlong_as_double(r);
}

// The pivot of column k by whole values, as the search's key; the sign bit is
// set where no value is positive.
template <int KT>
__device__ __forceinline__ int mid_pivot(const double2 (&x)[KT], int used, int a, int k) {
    double best = 0.0;
    int row = a;
#pragma unroll
    for (int s = 0; s < KT; ++s) {
        const double v = fabs(x[s].x) + fabs(x[s].y);
        if (!(used >> s & 1) && v > best) {
            best = v;
            row = a + 8 * s;
        }
    }
#pragma unroll
    for (int off = 8; off < 64; off *= 2) {
        const double ob = __shfl_xor(best, off, 64);
        const int orow = __shfl_xor(row, off, 64);
        if (ob > best || (ob == best && orow < row)) {
            best = ob;
            row = orow;
        }
    }
    best = readlane_f64(best, k);
    row = __builtin_amdgcn_readlane(row, k);
    return (__double2hiint(best) & ~127) | (8 * (KT - 1 - (row >> 3)) | (7 - (row & 7))) |
           (best > 0.0 ? 0 : 1 << 31);
}

// The panel wave: every panel's elimination.  Lane 8 a + b holds rows a + 8 s
// of the panel's column b; a step's exchanges stay in the registers (DPP,
// lane reads and one permute), since its latency is what an inverse's time is
// made of.
template <int KT>
__device__ __forceinline__ void mid_panels(int n, MidGjShared<KT> &sh) {
    const int lane = opaque_tid() & 63;
    const int a = lane >> 3, b = lane & 7;
    int used = 0;  // bit s: row a + 8 s has been a pivot, or is padding
#pragma unroll
    for (int s = 0; s < KT; ++s) used |= a + 8 * s < n ? 0 : 1 << s;
    int sing = 0;
#pragma unroll 1
    for (int jp = 0; jp < KT; ++jp) {
        const int c0 = 8 * jp, kk = std::min(8, n - c0);
        __syncthreads();  // the panel is in sh.pan
        double2 x[KT];
#pragma unroll
        for (int s = 0; s < KT; ++s) x[s] = sh.pan[b][a + 8 * s];
        int myrow = 0;  // pivot row and reciprocal of step c0 + lane
        double2 myr = make_double2(0.0, 0.0);
        auto step = [&](auto kc) {
            constexpr int k = kc;
            if (k >= kk) return;
            // pivot search: the row (first s, then a, the lower the better)
            // in the low 7 bits of the high word of |re| + |im|, so that one
            // integer maximum finds value and row; used rows count as zero,
            // and so does NaN.  Where a second row has the same upper bits
            // (seldom; all rows of a column without a pivot do), mid_pivot()
            // looks at whole values.
            int key = 0, key2 = 0;  // the largest of the lane's rows, the next
#pragma unroll
            for (int s = 0; s < KT; ++s) {
                const double v = fmax_nocanon(fabs(x[s].x) + fabs(x[s].y), 0.0);
                const int free = ~(used << (31 - s) >> 31);
                const int ks = (__double2hiint(v) & free & ~127) | (8 * (KT - 1 - s));
                key2 = imed3(key, key2, ks);
                key = std::max(key, ks);
            }
            key |= 7 - a;
            const int top = key;
            key = std::max(key, __builtin_amdgcn_mov_dpp(key, 0x118, 0xf, 0xf, true));  // row_shr:8
            int kh = std::max(std::max(__builtin_amdgcn_readlane(key, 8 + k),
                                       __builtin_amdgcn_readlane(key, 24 + k)),
                              std::max(__builtin_amdgcn_readlane(key, 40 + k),
                                       __builtin_amdgcn_readlane(key, 56 + k)));
            constexpr unsigned long long kCol = 0x0101010101010101ull << k;  // lanes of column k
            const int other = top == kh ? key2 : top;  // the largest of the lane's rows but the pivot
            if (__ballot(other >= (kh & ~127)) & kCol) {
                kh = mid_pivot<KT>(x, used, a, k);
                // (without a pivot -- the column is zero, or NaN -- the steps
                // go on with row 0, and the result is dropped)
                sing |= kh < 0;
                kh &= 0x7fffffff;
            }
            const int sp = KT - 1 - ((kh & 127) >> 3), ap = 7 - (kh & 7);
            // the pivot row's entry of this lane's column: bitwise selects (an
            // indexed read would put x in scratch)
            int u0 = 0, u1 = 0, u2 = 0, u3 = 0;
#pragma unroll
            for (int s = 0; s < KT; ++s) {
                const int m = sp == s ? -1 : 0;
                u0 = (u0 & ~m) | (__double2loint(x[s].x) & m);
                u1 = (u1 & ~m) | (__double2hiint(x[s].x) & m);
                u2 = (u2 & ~m) | (__double2loint(x[s].y) & m);
                u3 = (u3 & ~m) | (__double2hiint(x[s].y) & m);
            }
            const int src = (8 * ap | b) << 2, pl = 8 * ap + k;
            const double2 y =
                make_double2(__hiloint2double(__builtin_amdgcn_ds_bpermute(src, u1),
                                              __builtin_amdgcn_ds_bpermute(src, u0)),
                             __hiloint2double(__builtin_amdgcn_ds_bpermute(src, u3),
                                              __builtin_amdgcn_ds_bpermute(src, u2)));
            const double2 pv = make_double2(__hiloint2double(__builtin_amdgcn_readlane(u1, pl),
                                                             __builtin_amdgcn_readlane(u0, pl)),
                                            __hiloint2double(__builtin_amdgcn_readlane(u3, pl),
                                                             __builtin_amdgcn_readlane(u2, pl)));
            // (|re| + |im| < 2^e: the search key has the exponent)
            const double2 r = crecip_scaled(pv, (kh >> 20) - 1022);
            // the multipliers, 0 at the pivot row (up to a denormal number:
            // the low word stays)
            double2 f[KT];
            const bool prow = a == ap;
#pragma unroll
            for (int s = 0; s < KT; ++s) {
                const bool piv = prow && sp == s;
                const double fx = __hiloint2double(piv ? 0 : __double2hiint(x[s].x), __double2loint(x[s].x));
                const double fy = __hiloint2double(piv ? 0 : __double2hiint(x[s].y), __double2loint(x[s].y));
                f[s] = make_double2(group_bcast<k>(fx), group_bcast<k>(fy));
            }
            // the step leaves -f r in its own column, and 0 in the pivot row:
            // there the panel keeps the distance from 1
            const bool mine = b == k;
            double2 u = cmul(y, r);
            if (mine) {
                u = r;
#pragma unroll
                for (int s = 0; s < KT; ++s) x[s] = make_double2(0.0, 0.0);
            }
            if (prow) used |= 1 << sp;
            if (lane == k) {
                myrow = 8 * sp + ap;
                myr = r;
            }
#pragma unroll
            for (int s = 0; s < KT; ++s) {
                x[s].x = fma(-f[s].x, u.x, fma(f[s].y, u.y, x[s].x));
                x[s].y = fma(-f[s].x, u.y, fma(-f[s].y, u.x, x[s].y));
            }
        };
        each_of(std::make_integer_sequence<int, 8>(), step);
        double2 *mp = &sh.m[jp & 1][b][a];
#pragma unroll
        for (int s = 0; s < KT; ++s) mp[8 * s] = x[s];
        if (lane < kk) {
            sh.pivrow[c0 + lane] = myrow;
            sh.pivstep[myrow] = c0 + lane;
            sh.rpiv[c0 + lane] = myr;
        }
        if (sing && lane == 0) sh.sing = 1;
        __syncthreads();  // M and the pivots are there
    }
}

// A column wave's part: x -> its inverse in the permuted places described
// above (of no use when sh.sing is set).
template <int KT>
__device__ __forceinline__ void mid_columns(double2 (&x)[KT][MidGj<KT>::CL], int n, int wave,
                                            MidGjShared<KT> &sh) {
    using C = MidGj<KT>;
    using std::integral_constant;
    constexpr int W = C::W, CL = C::CL;
    constexpr bool kEven = KT % W == 0;
    const int lane = opaque_tid() & 63;
    const int a = lane & 7, b = lane >> 3;
    // the last column group exists only in the first waves of an uneven split
    const bool whole = kEven || wave < KT % W;

    // x += M T of panel jp for the register groups in the mask (the panel's
    // own columns left alone).  Software-pipelined by hand: a ring of
    // multipliers on their way from LDS, each register loaded again right
    // after its use.
    auto update = [&](int jp, auto groups) {
        constexpr int kMask = groups;
        if constexpr (kMask != 0) {
            constexpr int D = KT % 5 == 0 ? 5 : KT % 4 == 0 ? 4 : KT % 3 == 0 ? 3 : KT;
            const int kk = std::min(8, n - 8 * jp);
            const int skip = wave == jp % W ? jp / W : -1;
            const double2 *mp = &sh.m[jp & 1][0][a];
            const double2 *tp = &sh.t[wave][0][0][b];
            double2 u[CL], un[CL], f[D];
            auto load_u = [&](int k) {
#pragma unroll
                for (int v = 0; v < CL; ++v)
                    if (kMask >> v & 1) un[v] = tp[(k * CL + v) * 8];
            };
            load_u(0);
#pragma unroll
            for (int s = 0; s < D; ++s) f[s] = mp[8 * s];
#pragma unroll 1
            for (int k = 0; k < kk; ++k) {
                const int kn = k + 1 < kk ? k + 1 : k;
#pragma unroll
                for (int v = 0; v < CL; ++v)
                    if (kMask >> v & 1) u[v] = v == skip ? make_double2(0.0, 0.0) : un[v];
#pragma unroll
                for (int s = 0; s < KT; ++s) {
                    const double2 g = f[s % D];
#pragma unroll
                    for (int v = 0; v < CL; ++v)
                        if (kMask >> v & 1) {
                            x[s][v].x = fma(g.x, u[v].x, fma(-g.y, u[v].y, x[s][v].x));
                            x[s][v].y = fma(g.x, u[v].y, fma(g.y, u[v].x, x[s][v].y));
                        }
                    f[s % D] = s + D < KT ? mp[k * C::LDM + 8 * (s + D)]
                                          : mp[kn * C::LDM + 8 * (s + D - KT)];
                    if (s == KT - D) load_u(kn);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    };
    constexpr int kAll = (1 << CL) - 1, kBase = kEven ? kAll : kAll >> 1, kEnd = kAll & ~kBase;
    auto update_of = [&](int jp, auto groups) {
        constexpr int kMask = groups;
        update(jp, integral_constant<int, kMask & kBase>());
        if (kMask & kEnd)
            if (whole) update(jp, integral_constant<int, kMask & kEnd>());
    };
    auto publish = [&](int jp, auto group) {  // panel jp's columns, by the wave that holds them
        if (wave == jp % W) {
#pragma unroll
            for (int s = 0; s < KT; ++s) sh.pan[b][a + 8 * s] = x[s][group];
        }
    };
    // Panel jp, in group t; the next one in group tn.
    auto step = [&](auto panel) {
        constexpr int jp = panel, t = jp / W, tn = (jp + 1) / W;
        const int c0 = 8 * jp, kk = std::min(8, n - c0);
        __syncthreads();  // M and the pivots of panel jp are there
        if (wave == jp % W) {
            // the panel's columns are M, with 1 where a pivot row meets its
            // own column
            const double2 *mp = &sh.m[jp & 1][b][a];
            const int pb = b < kk ? sh.pivrow[c0 + b] : -1;
#pragma unroll
            for (int s = 0; s < KT; ++s) {
                x[s][t] = mp[8 * s];
                x[s][t].x += pb == a + 8 * s ? 1.0 : 0.0;
            }
        }
        // T: the pivot rows of the wave's columns.  M holds the distance from
        // 1 where a pivot row meets its own column, so that x + M T is right
        // for the pivot rows too (their new value is M T).
#pragma unroll
        for (int s = 0; s < KT; ++s) {
            const int k = sh.pivstep[a + 8 * s] - c0;
            if (k >= 0 && k < kk) {
#pragma unroll
                for (int v = 0; v < CL; ++v) sh.t[wave][k][v][b] = x[s][v];
            }
        }
        wave_order();
        if constexpr (jp + 1 < KT) {
            update_of(jp, integral_constant<int, 1 << tn>());
            publish(jp + 1, integral_constant<int, tn>());
            __syncthreads();
            update_of(jp, integral_constant<int, kAll & ~(1 << tn)>());
        } else {
            update_of(jp, integral_constant<int, kAll>());
        }
    };
    publish(0, integral_constant<int, 0>());
    __syncthreads();
    // KT panels, each its own code: which registers a step takes is known then
    each_of(std::make_integer_sequence<int, KT>(), step);
#pragma unroll
    for (int s = 0; s < KT; ++s) {
        const double2 r = sh.rpiv[std::max(sh.pivstep[a + 8 * s], 0)];
#pragma unroll
        for (int v = 0; v < CL; ++v) x[s][v] = cmul(x[s][v], r);
    }
}

// Traces of final inverse q (0: GLL, 1: GRR, 2: GB) from its diagonal and
// spin-partner elements in shared memory, in the reference's summation order
// (src/surfstat.f90:150-192, src/fermiarc.f90:238-328): every term is formed
// by its own thread, thread 0 adds the trace and threads 1..3 the spin sums.
template <int KT>
__device__ __forceinline__ void mid_traces(const DecimateArgs &a, MidGjShared<KT> &sh, int q,
                                           int t, int ik, int extra) {
    const int n = a.n, tid = threadIdx.x;
    const int o = a.inst_k ? t : ik + a.nk * (t - ik * a.nomega);
    __syncthreads();
    // terms in place: diag -> (Im G/d, sz), part -> (sx, sy)
    for (int i = tid; i < n; i += MidGj<KT>::NT) {
        bool up;
        const int pr = spin_partner(i, a.nw, up);
        const double2 d = sh.diag[i], g = sh.part[i];
        sh.diag[i] = make_double2(d.y / a.divisor, pr < 0 ? 0.0 : (up ? d.y : -d.y) / a.divisor);
        if (a.spin_mode)
            sh.part[i] = pr < 0 ? make_double2(0.0, 0.0)
                                : make_double2(g.y / a.divisor, (up ? g.x : -g.x) / a.divisor);
    }
    __syncthreads();
    // the trace runs over the top orbitals of GLL, the bottom ones of GRR in
    // the last layer, every orbital of GB
    const int *list = q == 0 ? a.top : q == 1 ? a.bot : nullptr;
    int cnt = q == 0 ? a.ntop : q == 1 ? a.nbot : n;
    int off = q == 1 ? n - a.nw : 0;
    if (tid == 0) {
        double s = 0.0;
        for (int i = 0; i < cnt; ++i) s = s - sh.diag[list ? list[i] - 1 + off : i].x;
        (q == 0 ? a.dos_l : q == 1 ? a.dos_r : a.dos_bulk)[o] = s;
        if (extra && a.status) atomicOr(a.status + o, extra);
    } else if (tid < 4 && a.spin_mode && q < 2) {
        // surfstat sums GRR's spin traces over the top orbital indices,
        // SurfaceDOSkk over the bottom orbitals of the last layer
        if (q == 1 && a.spin_mode == 1) {
            list = a.top;
            cnt = a.ntop;
            off = 0;
        }
        double s = 0.0;
        for (int i = 0; i < cnt; ++i) {
            const int io = list[i] - 1 + off;
            bool up;
            if (spin_partner(io, a.nw, up) < 0) continue;
            s = s - (tid == 1 ? sh.part[io].x : tid == 2 ? sh.part[io].y : sh.diag[io].y);
        }
        a.spin_out(o, q)[(size_t)(tid - 1) * a.ninst] = s;
    }
}

// The inverse left in x by mid_invert: g in natural order for the iteration
// (fin false), or the diagonal, spin-partner elements and traces (and the
// full matrix when asked for) of final inverse q.
template <int KT>
__device__ __forceinline__ void store_inverse(const DecimateArgs &a,
                                              double2 (&x)[KT][MidGj<KT>::CL], bool sing, bool fin,
                                              int q, int t, int wave, double2 *g,
                                              MidGjShared<KT> &sh) {
    using C = MidGj<KT>;
    constexpr int NB = 8 * KT, W = C::W, CL = C::CL;
    const int lane = opaque_tid() & 63;
    const int ra = lane & 7, cb = lane >> 3;
    const int n = a.n;
    if (!fin) {
#pragma unroll
        for (int v = 0; v < CL; ++v) {
            const int c = 8 * (wave + W * v) + cb;
            if (c < NB) {
                const int j = sing ? c : sh.pivrow[c];
#pragma unroll
                for (int s = 0; s < KT; ++s) {
                    const int i = sing ? ra + 8 * s : sh.pivstep[ra + 8 * s];
                    g[MidLay<KT>::frag(i, j)] =
                        sing ? make_double2(i == j && i < n ? 1.0 : 0.0, 0.0) : x[s][v];
                }
            }
        }
        return;
    }
    double2 *full = a.gfull ? a.gfull + ((size_t)t * 3 + q) * n * n : nullptr;
#pragma unroll
    for (int v = 0; v < CL; ++v) {
        const int c = 8 * (wave + W * v) + cb;
        if (c < n) {
            const int j = sing ? c : sh.pivrow[c];
            // rows i that want G(i, j): j itself and the row whose spin
            // partner j is (j's own partner)
            bool up;
            const int jp = a.spin_mode ? spin_partner(j, a.nw, up) : -1;
#pragma unroll
            for (int s = 0; s < KT; ++s) {
                const int r = ra + 8 * s;
                if (r < n) {
                    const int i = sing ? r : sh.pivstep[r];
                    const double2 e = sing ? make_double2(i == j ? 1.0 : 0.0, 0.0) : x[s][v];
                    if (i == j) sh.diag[i] = e;
                    if (i == jp) sh.part[i] = e;
                    if (full) full[i + (size_t)j * n] = e;
                }
            }
        }
    }
}

// Blocks 0 .. 3 slots - 1: the final inverses of the slots whose instance the
// last GEMM round brought to its end; the others: one per slot, the inverse
// its next GEMM round needs, of the same instance or of the next one from the
// queue.  Both kinds read the slot's old state, the latter write the new one.
// A finished instance's Z stays as it is while the next instance starts in
// the slot's other Z.
template <int KT>
__global__ void __launch_bounds__(MidGj<KT>::NT) __attribute__((amdgpu_waves_per_eu(MidGj<KT>::OCC)))
mid_inverse_kernel(DecimateArgs a, const MidState *__restrict__ in, MidState *__restrict__ out,
                   int slots) {
    using C = MidGj<KT>;
    using L = MidLay<KT>;
    constexpr int NB = L::NB, MT = L::MT, W = C::W, CL = C::CL, NT = C::NT;
    __shared__ MidGjShared<KT> sh;
    const int fin = (int)blockIdx.x < 3 * slots;
    const int slot = fin ? blockIdx.x % slots : blockIdx.x - 3 * slots;
    const int q = fin ? blockIdx.x / slots : 3;
    const int tid = threadIdx.x;
    const int wave = mid_wave<KT>(tid), lane = tid & 63;
    const int ra = lane & 7, cb = lane >> 3;
    const int n = a.n;
    const MidSlot<KT> w(a.work, slot);
    MidState st;
    st.phase = uniform(in[slot].phase);
    st.t = uniform(in[slot].t);
    st.it = uniform(in[slot].it);
    st.status = uniform(in[slot].status);
    st.buf = uniform(in[slot].buf);
    if (st.phase == kMidDone || (fin && st.phase != kMidLoop)) {
        if (!fin && tid == 0) out[slot] = st;
        return;
    }
    bool ended = false;
    if (st.phase == kMidLoop) {
        double s = 0.0;
        for (int i = 0; i < MT * MT; ++i) s += w.part[i];
        const int conv = uniform(s <= a.accuracy ? 1 : 0);
        ended = conv || st.it >= a.itermax;
        if (!conv && ended) st.status |= 2;
        st.buf ^= 1;  // the GEMM round wrote the other Z
    }
    if (fin && !ended) return;
    int t = st.t, ik;
    double2 z;
    bool fresh = false;
    if (!fin && (ended || st.phase == kMidEmpty)) {
        if (ended && tid == 0) {
            // iterations and status of the finished instance; the final
            // inverses of this launch add their singular bits, and the host's
            // streams wait for whole launches
            int ik0;
            double2 z0;
            instance_of(a, t, ik0, z0);
            const int o = a.inst_k ? t : ik0 + a.nk * (t - ik0 * a.nomega);
            if (a.iters) a.iters[o] = st.it;
            if (a.status && st.status) atomicOr(a.status + o, st.status);
            atomicAdd(a.queue + 1, 1u);
        }
        if (tid == 0) sh.tk = (int)atomicAdd(a.queue, 1u);
        __syncthreads();
        t = uniform(sh.tk);
        if (queue_empty((unsigned)t, a.ninst)) {
            if (tid == 0) {
                st.phase = kMidDone;
                out[slot] = st;
            }
            return;
        }
        fresh = true;
        st.buf ^= 1;
        st.t = t;
        st.it = 1;
        st.status = 0;
    } else if (!fin) {
        st.it += 1;
    }
    instance_of(a, t, ik, z);
    const int NP = 16 * ((n + 15) / 16);
    const double2 *H00 = a.hk + (size_t)ik * 2 * NP * NP;
    double2 *eps = w.eps(st.buf);

    if (fresh) {
        // alpha = H01, beta = H01^dagger, eps_s = eps_t = H00
        // (src/surfgreen.f90:74-78), pads zero as in H00 and H01
        const double2 *__restrict__ h0 = H00;
        const double2 *__restrict__ h1 = H00 + NP * NP;
        double2 *__restrict__ ab = w.ab(st.buf);
        double2 *__restrict__ ep = eps;
#pragma unroll 4
        for (int e = tid; e < NB * NB; e += NT) {
            const int i = e % NB, j = e / NB;
            const double2 h = h0[i + j * NP], al = h1[i + j * NP], ht = h1[j + i * NP];
            ep[e] = ep[NB * NB + e] = h;
            ab[L::frag(i, j)] = al;
            ab[L::frag(i, NB + j)] = make_double2(ht.x, -ht.y);
        }
    }

    if (tid == 0) sh.sing = 0;
    for (int i = tid; i < NB; i += NT) {
        sh.pivrow[i] = i;
        sh.pivstep[i] = i < n ? -1 : i;
        sh.rpiv[i] = make_double2(1.0, 0.0);
    }
    if (wave == W) {
        __syncthreads();
        mid_panels<KT>(n, sh);
    } else {
        // X = z - E: eps_i = eps_s + eps_t - H00 (H00 itself in a first
        // iteration), or eps_s, eps_t, eps_i of the final inverses; every load
        // is in bounds of the padded arrays
        double2 x[KT][CL];
        const bool three = !fresh && q >= 2;
        const double2 *e1 = fresh ? H00 : q == 1 ? eps + NB * NB : eps;
        const int ld1 = fresh ? NP : NB;
        int jc[CL];
#pragma unroll
        for (int v = 0; v < CL; ++v) {
            jc[v] = std::min(8 * (wave + W * v) + cb, NB - 1);
#pragma unroll
            for (int s = 0; s < KT; ++s) x[s][v] = e1[ra + 8 * s + jc[v] * ld1];
        }
        if (three) {
            // (the empty asm keeps one column's loads behind the last's additions:
            // all of them at once would take more registers than there are)
            double2 y[KT];
#pragma unroll
            for (int v = 0; v < CL; ++v) {
                asm volatile("" ::: "memory");
#pragma unroll
                for (int s = 0; s < KT; ++s) y[s] = eps[NB * NB + ra + 8 * s + jc[v] * NB];
#pragma unroll
                for (int s = 0; s < KT; ++s) x[s][v] = cadd(x[s][v], y[s]);
            }
#pragma unroll
            for (int v = 0; v < CL; ++v) {
                asm volatile("" ::: "memory");
#pragma unroll
                for (int s = 0; s < KT; ++s) y[s] = H00[ra + 8 * s + jc[v] * NP];
#pragma unroll
                for (int s = 0; s < KT; ++s) {
                    x[s][v].x -= y[s].x;
                    x[s][v].y -= y[s].y;
                }
            }
        }
#pragma unroll
        for (int v = 0; v < CL; ++v) {
            const int j = 8 * (wave + W * v) + cb;
#pragma unroll
            for (int s = 0; s < KT; ++s) {
                const int i = ra + 8 * s;
                const bool in = i < n && j < n;
                x[s][v].x = in ? (i == j ? z.x : 0.0) - x[s][v].x : 0.0;
                x[s][v].y = in ? (i == j ? z.y : 0.0) - x[s][v].y : 0.0;
            }
        }
        __syncthreads();
        mid_columns<KT>(x, n, wave, sh);
        store_inverse<KT>(a, x, uniform(sh.sing) != 0, fin, q, t, wave, w.g, sh);
    }
    const int sing = uniform(sh.sing);
    if (fin) {
        mid_traces<KT>(a, sh, q, t, ik, sing);
    } else if (tid == 0) {
        st.status |= sing;
        st.phase = kMidLoop;
        out[slot] = st;
    }
}

__global__ void mid_clear_kernel(MidState *state, int nstate, unsigned *queue, int *status, int ninst) {
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < (unsigned)nstate) state[i] = MidState{kMidEmpty, 0, 0, 0, 0};
    if (i < 2) queue[i] = 0;
    if (status && i < (unsigned)ninst) status[i] = 0;
}

template <int KT>
int launch_mid(const DecimateArgs &a, MidState *in, MidState *out, void *work, int slots,
               int csplit, bool inverse, hipStream_t s) {
    if (inverse) {
        DecimateArgs b = a;
        b.work = work;
        hipLaunchKernelGGL((mid_inverse_kernel<KT>), dim3(4 * slots), dim3(MidGj<KT>::NT), 0, s, b,
                           in, out, slots);
    } else {
        const int grid = (slots + 7) / 8 * 8 * KT * csplit;
        hipLaunchKernelGGL((mid_gemm_kernel<KT>), dim3(grid), dim3(64), 0, s, work, out, slots, csplit);
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

#define WTSURF_FOR_EACH_KT(X) \
    X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14)

int dispatch_mid(int kt, const DecimateArgs &a, MidState *in, MidState *out, void *work, int slots,
                 int csplit, bool inverse, hipStream_t s) {
    switch (kt) {
#define WTSURF_CASE(K) \
    case K: return launch_mid<K>(a, in, out, work, slots, csplit, inverse, s);
        WTSURF_FOR_EACH_KT(WTSURF_CASE)
#undef WTSURF_CASE
        default: return -1;
    }
}

// Slots per CU and set: a launch ends with its slowest workgroups, so many
// slots a launch (8192 instances of order 72: 76.6 ms with 512 slots a set,
// 72.1 with 1024, 69.0 with 2048 and with 4096; one set of 2048: 75.9).  The
// workspace is 0.76 MB a slot at order 72 and 1.8 MB at order 112: 3.1 and 7.4
// GB for all of them, less where the card has less (decimate_mid_limit).
constexpr int kMidSlotsPerCu = 8;
constexpr int kMidRoundsPerBatch = 4;

}  // namespace

// Beyond 112 the inverse's registers (28 complex of a lane at two waves a SIMD)
// run out.  Between 81 and 112 the kernels with the matrix in global memory that
// took these orders before: 1500 instances of order 108 59.6 ms, 47.5 here;
// 400 of order 96 11.8 and 10.7, of order 81 11.3 and 8.7; one of order 108
// 9.6 and 4.6.
int decimate_mid_max_n() { return 112; }

size_t decimate_mid_slot_bytes(int n) {
    switch ((n + 7) / 8) {
#define WTSURF_CASE(K) \
    case K: return MidLay<K>::stride;
        WTSURF_FOR_EACH_KT(WTSURF_CASE)
#undef WTSURF_CASE
        default: return 0;
    }
}

MidPlan decimate_mid_plan(int ninst, int num_cu) {
    MidPlan p;
    p.sets = ninst > 1 ? 2 : 1;
    p.per_set = std::min((ninst + p.sets - 1) / p.sets, kMidSlotsPerCu * num_cu);
    return p;
}

void decimate_mid_limit(MidPlan &p, int num_cu, size_t most) {
    const size_t slots = std::max(most, (size_t)2 * num_cu);
    if ((size_t)p.sets * p.per_set > slots) p.per_set = (int)(slots / p.sets);
}

bool decimate_mid_halve(MidPlan &p) {
    if (p.per_set > 1)
        p.per_set = (p.per_set + 1) / 2;
    else if (p.sets > 1)
        p.sets = 1;
    else
        return false;
    return true;
}

int decimate_mid_run(const DecimateArgs &a, const MidPlan &plan, MidState *state, int num_cu,
                     const RoundCtl &ctl) {
    const int kt = (a.n + 7) / 8;
    const size_t stride = decimate_mid_slot_bytes(a.n);
    if (a.n < 1 || stride == 0 || plan.sets < 1 || plan.sets > kSlotSets || plan.per_set < 1) return -1;
    const int NS = plan.sets, per = plan.per_set;
    const hipStream_t s0 = ctl.s[0], sc = ctl.s[kSlotSets];
    const hipEvent_t start = ctl.ev[2 * kSlotSets + 2];
    // an idle part of the chip takes shares of the output columns, each of
    // which forms m1, m2 of its strip again
    const int csplit = std::max(1, std::min(kt, 4 * num_cu / (per * kt)));
    const int nstate = 2 * NS * per;
    const unsigned nclear = std::max(std::max(nstate, a.ninst), 2);
    hipLaunchKernelGGL(mid_clear_kernel, dim3((nclear + 255u) / 256u), dim3(256), 0, s0, state, nstate,
                       a.queue, a.status, a.ninst);
    if (hipGetLastError() != hipSuccess || hipEventRecord(start, s0) != hipSuccess) return -1;
    for (int k = 1; k < NS; ++k)
        if (hipStreamWaitEvent(ctl.s[k], start, 0) != hipSuccess) return -1;
    // An instance takes at most itermax rounds and the inverse of one more; a
    // slot runs ceil(ninst / slots) instances.  Past that bound (with slack)
    // the device has stopped making progress.
    const long per_slot = (a.ninst + (long)NS * per - 1) / ((long)NS * per) + 1;
    const long max_batches = per_slot * (a.itermax + 2) / kMidRoundsPerBatch + 4;
    const unsigned want = (unsigned)a.ninst;
    // Set k starts with an inverse round; the sets' rounds drift as their
    // launches interleave.  The counter stream copies the finished count to
    // pinned memory after every batch, and the host reads the previous
    // batch's while this one runs.
    long round = 0;
    for (long b = 0;; ++b) {
        if (b > max_batches) return -2;
        for (int r = 0; r < kMidRoundsPerBatch; ++r, ++round)
            for (int k = 0; k < NS; ++k) {
                MidState *s = state + (size_t)k * 2 * per;
                MidState *in = s + (round & 1 ? per : 0), *out = s + (round & 1 ? 0 : per);
                void *work = static_cast<unsigned char *>(a.work) + (size_t)k * per * stride;
                if (dispatch_mid(kt, a, in, out, work, per, csplit, true, ctl.s[k]) ||
                    dispatch_mid(kt, a, in, out, work, per, csplit, false, ctl.s[k]))
                    return -1;
            }
        const int h = (int)(b & 1);
        for (int k = 0; k < NS; ++k)
            if (hipEventRecord(ctl.ev[2 * k + h], ctl.s[k]) != hipSuccess ||
                hipStreamWaitEvent(sc, ctl.ev[2 * k + h], 0) != hipSuccess)
                return -1;
        if (hipMemcpyAsync(ctl.pinned + h, a.queue + 1, sizeof(unsigned), hipMemcpyDeviceToHost, sc) !=
                hipSuccess ||
            hipEventRecord(ctl.ev[2 * kSlotSets + h], sc) != hipSuccess)
            return -1;
        if (b > 0) {
            if (hipEventSynchronize(ctl.ev[2 * kSlotSets + (h ^ 1)]) != hipSuccess) return -1;
            if (ctl.pinned[h ^ 1] >= want) break;
        }
    }
    for (int k = 1; k < NS; ++k)
        if (hipEventRecord(ctl.ev[2 * k], ctl.s[k]) != hipSuccess ||
            hipStreamWaitEvent(s0, ctl.ev[2 * k], 0) != hipSuccess)
            return -1;
    return 0;
}

}  // namespace wtsurf
