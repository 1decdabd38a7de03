// Decimation for orders 17 to 32 on the vector ALUs, one workgroup per
// instance for its whole decimation (src/surfgreen.f90:74-134); smaller orders
// are tiny.hip's.
//
// At these orders the 16 x 16 matrix-core tiles are partly padding, and the
// round schedule's traffic of the slot state through HBM and its launches
// weigh on it.  MI355X's FP64 vector
// rate equals its FP64 matrix rate, so here every product is a plain FMA
// loop over the true order n.  Each instance lives in one workgroup of W
// waves from its set-up to its traces: its matrices in LDS, eps_s, eps_t and
// H00 in registers, and nothing passes through global memory but its inputs
// and outputs.  Workgroups take instances from a device queue until it runs
// dry, several per CU.
//
// Lane layout: thread L = i + NP jc (i < NP the row, jc < NC the column
// group, NC = 64 W / NP) holds row i at the columns j = jc + NC t, t < EPL
// (EPL = NP / NC).  The lanes of one column group lie in one wave (NP divides
// 64).  LDS matrices are NP x (NP + 1) column-major: the column groups' reads
// of one row then fall on different banks.
#include <algorithm>

#include "decimate_common.h"

namespace wtsurf {

namespace {

constexpr int NP = 32;  // order of the padded matrices (as H00 and H01 are stored)
constexpr int W = 8;    // waves per instance

struct SmallCfg {
    static constexpr int NT = 64 * W;
    static constexpr int NC = NT / NP;
    static constexpr int EPL = NP / NC;
    static constexpr int GPW = 64 / NP;  // column groups per wave
    static constexpr int LD = NP + 1;
    static constexpr int MAT = NP * LD;
    static_assert(64 % NP == 0 && W > 1 && NT % NP == 0 && NP % NC == 0, "layout must tile the workgroup");
};

// Pivot exchange of the Gauss-Jordan steps, double-buffered by step parity.
struct SmallPivot {
    double2 mcol[2][NP];  // multipliers X[i][c] / pivot (0 for the pivot row)
    double2 rr[2];        // 1 / pivot
    int piv[2];           // pivot row
    int sing[2];          // zero pivot column
};

struct SmallLay {
    using Cfg = SmallCfg;
    // alpha, beta, g (then m1), m2
    static constexpr size_t mats = (size_t)4 * Cfg::MAT * sizeof(double2);
    static constexpr size_t bytes = mats + sizeof(SmallPivot);
};

// Element (i, j) of a natural-order LDS matrix.
template <int LD>
struct SmallG {
    const double2 *g;
    __device__ double2 operator()(int i, int j) const { return g[i + j * LD]; }
};

// X^-1 of the n x n matrix X held in the lane layout (x: this thread's
// elements; pad rows and columns zero) written to G in natural order (pad
// zero).  Partial pivoting on |re| + |im| over the rows not yet used, the
// lowest row on ties (the izamax rule of zgesv).  Rows are never swapped: the
// step-c pivot row keeps its values unscaled and stands for 1/pivot times
// itself, takes every later step like any other row (its own multiplier is
// zero), and is scaled once at the end; the element then at (row r, column
// c) is X^-1[step(r)][pivot row of step c].  The wave that holds column c
// finds the pivot (DPP wave maximum and a ballot) and publishes the pivot
// row, 1/pivot and the multipliers in LDS; after one barrier every thread
// applies the step, reading the pivot row's entries of its own columns from
// the pivot lane of its column group.  Returns true on an exactly zero pivot
// column; G then holds the identity, as the reference's inv hands back
// (src/inverse.f90:44-55).
__device__ __forceinline__ bool small_gj(double2 (&x)[SmallCfg::EPL], int n,
                                         SmallPivot &sh, double2 *G) {
    using Cfg = SmallCfg;
    constexpr int NC = Cfg::NC, EPL = Cfg::EPL, GPW = Cfg::GPW, LD = Cfg::LD;
    const int tid = threadIdx.x;
    const int wave = uniform(tid >> 6), lane = tid & 63;
    const int i = tid % NP, jc = tid / NP;
    bool fr = i < n;       // row i not yet a pivot
    int srow = i;          // step at which row i was the pivot
    double2 myr = make_double2(1.0, 0.0);
    int pr[EPL];           // pivot row of the step of each own column
#pragma unroll
    for (int t = 0; t < EPL; ++t) pr[t] = jc + NC * t;
    bool singular = false;
#pragma unroll
    for (int t = 0; t < EPL; ++t) {
        if (singular) break;
        for (int jh = 0; jh < NC; ++jh) {
            const int c = jh + NC * t;
            if (c >= n) break;
            int p;
            double2 r, m;
            const int b = c & 1;
            if (wave == jh / GPW) {
                const double v = (jc == jh && fr) ? fabs(x[t].x) + fabs(x[t].y) : -1.0;
                const double best = wave_max_f64(v);
                if (!(best > 0.0)) {
                    if (lane == 0) sh.sing[b] = 1;
                } else {
                    const unsigned long long msk = __ballot(v == best);
                    const int pl = uniform(__ffsll((long long)msk) - 1);
                    const int ph = pl - NP * (jh % GPW);
                    const double2 piv = make_double2(readlane_f64(x[t].x, pl), readlane_f64(x[t].y, pl));
                    const double2 rh = crecip_fast(piv);
                    if (jc == jh) {
                        double2 mh = cmul(x[t], rh);
                        if (i == ph) mh = make_double2(0.0, 0.0);
                        sh.mcol[b][i] = mh;
                    }
                    if (lane == 0) {
                        sh.piv[b] = ph;
                        sh.rr[b] = rh;
                        sh.sing[b] = 0;
                    }
                }
            }
            __syncthreads();
            if (uniform(sh.sing[b])) {
                singular = true;
                break;
            }
            p = uniform(sh.piv[b]);
            r = sh.rr[b];
            m = sh.mcol[b][i];
            const int src = p + NP * (jc % GPW);  // lane of (p, jc) in this wave
#pragma unroll
            for (int u = 0; u < EPL; ++u) {
                const double2 pv = make_double2(__shfl(x[u].x, src), __shfl(x[u].y, src));
                if (jc + NC * u == c) {
                    x[u].x = (i == p ? 1.0 : 0.0) - m.x;
                    x[u].y = -m.y;
                } else {
                    x[u].x = fma(-m.x, pv.x, fma(m.y, pv.y, x[u].x));
                    x[u].y = fma(-m.x, pv.y, fma(-m.y, pv.x, x[u].y));
                }
            }
            if (i == p) {
                fr = false;
                srow = c;
                myr = r;
            }
            if (jc == jh) pr[t] = p;
        }
    }
#pragma unroll
    for (int u = 0; u < EPL; ++u) {
        const int C = jc + NC * u;
        double2 v = make_double2(0.0, 0.0);
        int ro = i, co = C;
        if (singular) {
            if (i == C && i < n) v.x = 1.0;
        } else if (i < n && C < n) {
            ro = srow;
            co = pr[u];
            v = cmul(x[u], myr);
        }
        G[ro + co * LD] = v;
    }
    __syncthreads();
    return singular;
}

// P0 = A0 B and P1 = A1 B over K = n, the thread's own elements of each.
__device__ __forceinline__ void small_dual(const double2 *__restrict__ A0,
                                           const double2 *__restrict__ A1,
                                           const double2 *__restrict__ B, int n,
                                           double2 (&p0)[SmallCfg::EPL],
                                           double2 (&p1)[SmallCfg::EPL]) {
    using Cfg = SmallCfg;
    constexpr int NC = Cfg::NC, EPL = Cfg::EPL, LD = Cfg::LD;
    const int tid = threadIdx.x;
    const int i = tid % NP, jc = tid / NP;
#pragma unroll
    for (int u = 0; u < EPL; ++u) p0[u] = p1[u] = make_double2(0.0, 0.0);
#pragma unroll 4
    for (int k = 0; k < n; ++k) {
        const double2 a0 = A0[i + k * LD], a1 = A1[i + k * LD];
#pragma unroll
        for (int u = 0; u < EPL; ++u) {
            const double2 b = B[k + (jc + NC * u) * LD];
            p0[u].x = fma(a0.x, b.x, fma(-a0.y, b.y, p0[u].x));
            p0[u].y = fma(a0.x, b.y, fma(a0.y, b.x, p0[u].y));
            p1[u].x = fma(a1.x, b.x, fma(-a1.y, b.y, p1[u].x));
            p1[u].y = fma(a1.x, b.y, fma(a1.y, b.x, p1[u].y));
        }
    }
}

__device__ __forceinline__ void small_store(double2 *M, const double2 (&p)[SmallCfg::EPL]) {
    using Cfg = SmallCfg;
    const int tid = threadIdx.x;
    const int i = tid % NP, jc = tid / NP;
#pragma unroll
    for (int u = 0; u < Cfg::EPL; ++u) M[i + (jc + Cfg::NC * u) * Cfg::LD] = p[u];
}

// Workgroups per CU: as many as the LDS holds (with the static part); and the
// waves per SIMD that gives, which caps the registers of the kernel (512 /
// waves per SIMD).
constexpr int small_per_cu() {
    constexpr size_t per = SmallLay::bytes + sizeof(Common<NP / 16>) + W * sizeof(double) + 256;
    return (int)((size_t)160 * 1024 / per);
}
constexpr int small_waves_per_simd() {
    constexpr int w = (small_per_cu() * W + 3) / 4;
    return w > 8 ? 8 : w;
}

__global__ void __launch_bounds__(64 * W)
    __attribute__((amdgpu_waves_per_eu(small_waves_per_simd())))
    small_kernel(DecimateArgs a) {
    using Cfg = SmallCfg;
    constexpr int NC = Cfg::NC, EPL = Cfg::EPL, LD = Cfg::LD, MAT = Cfg::MAT;
    constexpr int QC = NP / 16;
    extern __shared__ __align__(16) unsigned char lds[];
    double2 *AL = reinterpret_cast<double2 *>(lds);
    double2 *BE = AL + MAT, *GM = BE + MAT, *M2 = GM + MAT;
    SmallPivot &sh = *reinterpret_cast<SmallPivot *>(lds + SmallLay::mats);
    __shared__ Common<QC> cm;
    __shared__ double red[W];
    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const int i = tid % NP, jc = tid / NP;
    const int n = a.n;
    for (;;) {
        if (tid == 0) cm.s.t = (int)atomicAdd(a.queue, 1u);
        __syncthreads();
        const int t = uniform(cm.s.t);
        if (queue_empty((unsigned)t, a.ninst)) break;
        int ik;
        double2 z;
        instance_of(a, t, ik, z);
        const double2 *H00 = a.hk + (size_t)ik * 2 * NP * NP;
        const double2 *H01 = H00 + NP * NP;
        // eps_s = eps_t = H00, alpha = H01, beta = H01^dagger (src/surfgreen.f90:74-78)
        double2 es[EPL], et[EPL], h0[EPL];
#pragma unroll
        for (int u = 0; u < EPL; ++u) {
            const int j = jc + NC * u;
            double2 h = make_double2(0.0, 0.0), al = h, be = h;
            if (i < n && j < n) {
                h = H00[i + j * NP];
                al = H01[i + j * NP];
                const double2 ht = H01[j + i * NP];
                be = make_double2(ht.x, -ht.y);
            }
            es[u] = et[u] = h0[u] = h;
            AL[i + j * LD] = al;
            BE[i + j * LD] = be;
        }
        int it = 1, status = 0;
        for (;;) {
            // g = (z - eps_i)^-1, eps_i = eps_s + eps_t - H00 (src/surfgreen.f90:88-89)
            double2 x[EPL];
#pragma unroll
            for (int u = 0; u < EPL; ++u) {
                const int j = jc + NC * u;
                const double ex = (es[u].x + et[u].x) - h0[u].x, ey = (es[u].y + et[u].y) - h0[u].y;
                x[u].x = (i == j ? z.x : 0.0) - ex;
                x[u].y = (i == j ? z.y : 0.0) - ey;
                if (i >= n || j >= n) x[u] = make_double2(0.0, 0.0);
            }
            __syncthreads();  // the set-up or the last products are in LDS, GM is free
            if (small_gj(x, n, sh, GM)) status |= 1;
            double2 p0[EPL], p1[EPL];
            // m1 = alpha g, m2 = beta g (:92-95)
            small_dual(AL, BE, GM, n, p0, p1);
            __syncthreads();  // every read of g done: m1 takes its place
            small_store(GM, p0);
            small_store(M2, p1);
            __syncthreads();
            // eps_s += m1 beta, beta' = m2 beta (:98-102, 116-117)
            small_dual(GM, M2, BE, n, p0, p1);
#pragma unroll
            for (int u = 0; u < EPL; ++u) es[u] = cadd(es[u], p0[u]);
            __syncthreads();
            small_store(BE, p1);
            // eps_t += m2 alpha, alpha' = m1 alpha (:107-114)
            small_dual(M2, GM, AL, n, p0, p1);
            double asum = 0.0;
#pragma unroll
            for (int u = 0; u < EPL; ++u) {
                et[u] = cadd(et[u], p0[u]);
                asum += hypot(p1[u].x, p1[u].y);
            }
            __syncthreads();
            small_store(AL, p1);
            // stop when sum_ij |alpha'_ij| <= accuracy (:120-122)
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) asum += __shfl_xor(asum, off, 64);
            if (lane == 0) red[wave] = asum;
            __syncthreads();
            double tot = 0.0;
#pragma unroll
            for (int w = 0; w < W; ++w) tot += red[w];
            if (tot <= a.accuracy) break;
            if (it >= a.itermax) {
                status |= 2;
                break;
            }
            ++it;
        }
        // G_LL = (z - eps_s)^-1, G_RR = (z - eps_t)^-1, G_B = (z - eps_i)^-1 (:127-134)
        for (int q = 0; q < 3; ++q) {
            double2 x[EPL];
#pragma unroll
            for (int u = 0; u < EPL; ++u) {
                const int j = jc + NC * u;
                double ex = q == 1 ? et[u].x : es[u].x, ey = q == 1 ? et[u].y : es[u].y;
                if (q == 2) {
                    ex = (es[u].x + et[u].x) - h0[u].x;
                    ey = (es[u].y + et[u].y) - h0[u].y;
                }
                x[u].x = (i == j ? z.x : 0.0) - ex;
                x[u].y = (i == j ? z.y : 0.0) - ey;
                if (i >= n || j >= n) x[u] = make_double2(0.0, 0.0);
            }
            __syncthreads();  // the previous final's traces are done with GM
            if (small_gj(x, n, sh, GM)) status |= 1;
            for (int e = tid; e < n; e += Cfg::NT) cm.diag[e] = GM[e + e * LD];
            if (a.gfull) {
                double2 *full = a.gfull + ((size_t)t * 3 + q) * n * n;
                for (int e = tid; e < n * n; e += Cfg::NT) full[e] = GM[e % n + (e / n) * LD];
            }
            __syncthreads();
            if (tid == 0) {
                cm.s.it = it;
                cm.s.status = status;
                final_traces<QC>(a, cm, SmallG<LD>{GM}, q, ik);
            }
        }
        __syncthreads();  // cm.s is free for the next ticket
    }
}

static int launch_small(const DecimateArgs &a, int num_cu, hipStream_t s) {
    constexpr size_t lds = SmallLay::bytes;
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(&small_kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        (void)hipGetLastError();  // the launch reports whether the size is accepted
    const long want = (long)num_cu * small_per_cu();
    const int nblocks = (int)std::max<long>(1, std::min<long>(want, a.ninst));
    hipLaunchKernelGGL(small_kernel, dim3(nblocks), dim3(64 * W), lds, s, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace

int decimate_small_max_n() { return NP; }

int decimate_small_run(const DecimateArgs &a, int num_cu, hipStream_t s) {
    if (a.n < 1 || a.n > decimate_small_max_n() || num_cu < 1) return -1;
    if (hipMemsetAsync(a.queue, 0, 2 * sizeof(unsigned), s) != hipSuccess) return -1;
    if (a.n <= decimate_tiny_max_n()) return decimate_tiny_run(a, num_cu, s);
    return launch_small(a, num_cu, s);
}

}  // namespace wtsurf
