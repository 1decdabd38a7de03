// Decimation for orders up to 16, everything in the registers of one wave
// (src/surfgreen.f90:74-134).
//
// Orders 9 to 16 take one instance per wave, orders up to 8 four, each with
// the FP64 MFMA whose tile they fill: 16x16x4, or 4x4x4 on four blocks, of
// which each instance uses one.  Both instructions want, and give, the lanes
// of a matrix X in one of two ways; for a tile of edge B (16 or 4; i = lane %
// B, q = lane / 16):
//   R(X)  register t: X[i][4 t + q]     the second operand of  c X^T,  the result
//   C(X)  register t: X[4 t + q][i]     the first operand of   X^T r
// so that R(A B) = mfma(C(B), R(A)) with no movement between lanes: m1 =
// alpha g and m2 = beta g leave the matrix cores as the operands of m1 alpha,
// m1 beta, m2 alpha, m2 beta.  R(eps_s) and R(eps_t) stay in registers from an
// instance's set-up to its traces; alpha, beta and g lie in LDS, from where they
// are read as R or as C.
//
// Bound by instruction issue: while an FP64 MFMA runs (64 cycles for
// 16x16x4) its SIMD issues no vector instruction of another wave either
// (measured: MFMA and FP64, FP32 or integer work of two waves add up), so
// an iteration at order 16 takes the 7,168 cycles of its 112 MFMA plus about
// 5,500 of the pivot steps and the rest, 15,000 together.  The kernel it
// replaces (vector ALUs, one wave per instance, every operand in LDS) was
// bound by LDS reads: 80,601 instances of order 16 took 10.5 ms, 6.5 ms now;
// 40,400 of order 8 1.44 ms, 0.80 ms now.  Three waves a SIMD: two with the
// operands of the products kept in registers took 6.95 ms, three with those
// registers spilled 9.2.
#include <algorithm>
#include <utility>

#include "decimate_common.h"

namespace wtsurf {

namespace {

// d of the lane at byte address src / 4.
__device__ __forceinline__ double lane_f64(int src, double d) {
    return __hiloint2double(__builtin_amdgcn_ds_bpermute(src, __double2hiint(d)),
                            __builtin_amdgcn_ds_bpermute(src, __double2loint(d)));
}

// d of the lane that the DPP control names.
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double d) {
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(d), CTRL, 0xf, 0xf, true),
                            __builtin_amdgcn_mov_dpp(__double2loint(d), CTRL, 0xf, 0xf, true));
}

// The sum over lanes l, l ^ 32, then ^ 16, ^ 2, ^ 1, in every lane of them.  (A swap
// of a value with itself leaves the one half, or the even rows, in the first
// result and the other in the second.)
__device__ __forceinline__ double quad_rows_sum(double d) {
    auto a = __builtin_amdgcn_permlane32_swap(__double2hiint(d), __double2hiint(d), false, false);
    auto b = __builtin_amdgcn_permlane32_swap(__double2loint(d), __double2loint(d), false, false);
    d = __hiloint2double(a[0], b[0]) + __hiloint2double(a[1], b[1]);
    a = __builtin_amdgcn_permlane16_swap(__double2hiint(d), __double2hiint(d), false, false);
    b = __builtin_amdgcn_permlane16_swap(__double2loint(d), __double2loint(d), false, false);
    d = __hiloint2double(a[0], b[0]) + __hiloint2double(a[1], b[1]);
    d += dpp_f64<0x4E>(d);     // quad_perm 2,3,0,1
    return d + dpp_f64<0xB1>(d);  // quad_perm 1,0,3,2
}

// The next k tickets of the queue, the first of them to every lane.  The lane
// number is hidden and the barrier keeps the branch where it is: a compiler
// that knows which lanes come from the lane 0 branch at the loop's end sends
// them through this one by a way of their own, and the others then loop on
// without lane 0, whose ticket they need.
__device__ __forceinline__ int take(unsigned *queue, unsigned k) {
    __builtin_amdgcn_wave_barrier();
    int tk = 0;
    if (opaque_tid() == 0) tk = (int)atomicAdd(queue, k);
    __builtin_amdgcn_wave_barrier();
    return uniform(tk);
}

// a b with the roundings spelled out, the same in every kernel.
__device__ __forceinline__ double2 cmul_fma(double2 a, double2 b) {
    return make_double2(fma(-a.y, b.y, a.x * b.x), fma(a.y, b.x, a.x * b.y));
}

// |re| + |im| of a free row; NaN and used rows count as zero.
__device__ __forceinline__ double pivot_value(double re, double im, int free) {
    const double v = fmax_nocanon(fabs(re) + fabs(im), 0.0);
    return __hiloint2double(__double2hiint(v) & free, __double2loint(v) & free);
}

// ---- one instance a wave, orders 9 to 16 -----------------------------------

struct M16 {
    v4d re, im;
};

// R(A B) from C(B) and R(A), K = 4 KS.  Columns from 4 KS on depend on such
// columns of B alone, and nothing reads them: they may hold anything.
template <int KS>
__device__ __forceinline__ M16 mul16(const M16 &c, const M16 &r) {
    using P = Prec<double>;
    M16 d{{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        d.re = P::mfma(c.re[s], r.re[s], d.re);
        d.im = P::mfma(c.re[s], r.im[s], d.im);
        d.re = mfma_neg(c.im[s], r.im[s], d.re);
        d.im = P::mfma(c.im[s], r.re[s], d.im);
    }
    return d;
}

constexpr int kLd16 = 17;

// Natural order, column-major; 12 workgroups fill a CU's LDS.
struct Lds16 {
    double2 g[16 * kLd16];  // the inverse; before it a panel's pivot rows
    double2 al[16 * kLd16], be[16 * kLd16];
};

template <int KS>
__device__ __forceinline__ void write16(const M16 &r, double2 *m, int i, int q) {
#pragma unroll
    for (int t = 0; t < KS; ++t) m[(4 * t + q) * kLd16 + i] = make_double2(r.re[t], r.im[t]);
}
template <int KS>
__device__ __forceinline__ M16 read_r16(const double2 *m, int i, int q) {
    M16 r;
#pragma unroll
    for (int t = 0; t < KS; ++t) {
        const double2 v = m[(4 * t + q) * kLd16 + i];
        r.re[t] = v.x;
        r.im[t] = v.y;
    }
    return r;
}
template <int KS>
__device__ __forceinline__ M16 read_c16(const double2 *m, int i, int q) {
    M16 c;
#pragma unroll
    for (int t = 0; t < KS; ++t) {
        const double2 v = m[i * kLd16 + 4 * t + q];
        c.re[t] = v.x;
        c.im[t] = v.y;
    }
    return c;
}

// x = R(X), the identity (KS <= 2: zero) from row and column n to 4 KS: X^-1 to
// sh.g in natural order, the identity from there on (the identity of order n if
// a pivot column is zero or NaN; returns true then).  Gauss-Jordan with partial
// pivoting on |re| + |im| over the rows not yet used (the izamax rule of zgesv,
// the lowest row on ties), rows never swapped: step c's pivot row p keeps its
// values unscaled, standing for 1/pivot times itself, takes every later step
// like any other row and is scaled once at the end; element (row r, column c) is
// then X^-1[step of r][pivot row of step c].  Rows and columns from n on hold the
// identity, whose steps change nothing, or (KS <= 2: the time of one instance,
// and what the registers of larger orders do not allow) zero, whose steps are
// left out.  Columns are eliminated in panels of 4, one register of every lane,
// and the panel is applied to the rest as X += M T by four MFMA, M the panel's
// columns (with the distance from 1 where a pivot row meets its own column) and T
// its pivot rows.
template <int KS>
__device__ __forceinline__ bool inverse16(M16 &x, int n, Lds16 &sh, int lane) {
    const int i = lane & 15, q = lane >> 4;
    int free = i < 4 * KS ? -1 : 0;
    constexpr bool kSkip = KS <= 2;
    int srow = i < (kSkip ? n : 4 * KS) ? 1 << 20 : i;  // step at which row i was the pivot (not yet)
    double2 myr = make_double2(1.0, 0.0);
    int prow[4] = {q, 4 + q, 8 + q, 12 + q};  // pivot row of the own columns' steps
    int sing = 0;
    auto panel = [&](auto tc) {
        constexpr int t = tc;
        double yr = x.re[t], yi = x.im[t];
        auto step = [&](auto kc) {
            constexpr int k = kc;
            if (kSkip && 4 * t + k >= n) return;
            const int own = (16 * k + i) << 2;
            double fr = lane_f64(own, yr), fi = lane_f64(own, yi);
            // pivot search: the largest high word, and among several rows that
            // have it (seldom) the largest low word
            const double v = pivot_value(yr, yi, free);
            const int hi = __double2hiint(v);
            int key = hi;
            key = std::max(key, __builtin_amdgcn_mov_dpp(key, 0x111, 0xf, 0xf, true));  // row_shr:1
            key = std::max(key, __builtin_amdgcn_mov_dpp(key, 0x112, 0xf, 0xf, true));
            key = std::max(key, __builtin_amdgcn_mov_dpp(key, 0x114, 0xf, 0xf, true));
            key = std::max(key, __builtin_amdgcn_mov_dpp(key, 0x118, 0xf, 0xf, true));
            const int kh = __builtin_amdgcn_readlane(key, 16 * k + 15);
            // (in a column without a positive entry all 16 have the high word 0)
            constexpr int sh0 = 32 * (k / 2), sh1 = 16 * (k % 2);
            unsigned rows = (unsigned)(__ballot(hi == kh) >> sh0) & (0xffffu << sh1);
            if (rows & (rows - 1)) {
                const unsigned lo = hi == kh ? (unsigned)__double2loint(v) : 0u;
                unsigned m = lo;
                m = std::max(m, (unsigned)__builtin_amdgcn_mov_dpp((int)m, 0x111, 0xf, 0xf, true));
                m = std::max(m, (unsigned)__builtin_amdgcn_mov_dpp((int)m, 0x112, 0xf, 0xf, true));
                m = std::max(m, (unsigned)__builtin_amdgcn_mov_dpp((int)m, 0x114, 0xf, 0xf, true));
                m = std::max(m, (unsigned)__builtin_amdgcn_mov_dpp((int)m, 0x118, 0xf, 0xf, true));
                const unsigned ml = (unsigned)__builtin_amdgcn_readlane((int)m, 16 * k + 15);
                rows = (unsigned)(__ballot(hi == kh && lo == ml) >> sh0) & (0xffffu << sh1);
                sing |= kh == 0 && ml == 0 && 4 * t + k < n;
            }
            const int p = __builtin_ctz(rows) - sh1;
            const int src = (p | (lane & 48)) << 2;
            const double2 y = make_double2(lane_f64(src, yr), lane_f64(src, yi));
            double2 r = crecip_scaled(make_double2(readlane_f64(yr, 16 * k + p),
                                                   readlane_f64(yi, 16 * k + p)),
                                      (kh >> 20) - 1022);
            double2 u = cmul_fma(y, r);
            if (q == k) {
                u = r;
                yr = yi = 0.0;
                prow[t] = p;
            }
            if (i == p) {
                fr = fi = 0.0;
                free = 0;
                srow = 4 * t + k;
                myr = r;
            }
            yr = fma(-fr, u.x, fma(fi, u.y, yr));
            yi = fma(-fr, u.y, fma(-fi, u.x, yi));
        };
        each_of(std::make_integer_sequence<int, 4>(), step);
        const int k = srow - 4 * t;
        if (k >= 0 && k < 4) {
#pragma unroll
            for (int v = 0; v < KS; ++v)
                if (v != t) sh.g[20 * k + 4 * v + q] = make_double2(x.re[v], x.im[v]);
        }
        wave_order();
        double2 a = sh.g[20 * q + i];
        wave_order();
        if ((i >> 2) == t) a = make_double2(0.0, 0.0);
        x.re[t] = yr;
        x.im[t] = yi;
        using P = Prec<double>;
        x.re = P::mfma(a.x, yr, x.re);
        x.im = P::mfma(a.x, yi, x.im);
        x.re = mfma_neg(a.y, yi, x.re);
        x.im = P::mfma(a.y, yr, x.im);
        if (prow[t] == i) x.re[t] += 1.0;
    };
    each_of(std::make_integer_sequence<int, KS>(), panel);
#pragma unroll
    for (int t = 0; t < KS; ++t) {
        const double2 e = cmul_fma(make_double2(x.re[t], x.im[t]), myr);
        const int c = 4 * t + q;
        if (sing)
            sh.g[c * kLd16 + i] = make_double2(i == c && i < n ? 1.0 : 0.0, 0.0);
        else
            sh.g[prow[t] * kLd16 + srow] = e;
    }
    wave_order();
    return sing;
}

// The traces of final inverse f (0: GLL, 1: GRR, 2: GB) of one instance in the
// reference's summation order (src/surfstat.f90:150-192,
// src/fermiarc.f90:238-328).  Lane l0 + i has the terms of orbital i: d = Im
// G(i, i) / divisor and s the three of its spin traces (0 where there is
// none).  o: place in the outputs.
struct Terms {
    double d, s[3];
};
__device__ __forceinline__ Terms terms_of(const DecimateArgs &a, double2 d, double2 g, int partner,
                                          bool up) {
    Terms t;
    t.d = d.y / a.divisor;
    t.s[0] = t.s[1] = t.s[2] = 0.0;
    if (a.spin_mode && partner >= 0) {
        t.s[0] = g.y / a.divisor;
        t.s[1] = (up ? g.x : -g.x) / a.divisor;
        t.s[2] = (up ? d.y : -d.y) / a.divisor;
    }
    return t;
}
__device__ __forceinline__ void tiny_traces(const DecimateArgs &a, int f, int o, const Terms &t,
                                            int l0, int lane) {
    const int n = a.n;
    double s = 0.0;
    if (f == 2) {
        for (int i = 0; i < n; ++i) s = s - readlane_f64(t.d, l0 + i);
    } else {
        const int *list = f == 0 ? a.top : a.bot;
        const int cnt = f == 0 ? a.ntop : a.nbot, off = f == 0 ? 0 : n - a.nw;
        for (int e = 0; e < cnt; ++e) s = s - readlane_f64(t.d, l0 + off + uniform(list[e]) - 1);
    }
    if (lane == 0) (f == 0 ? a.dos_l : f == 1 ? a.dos_r : a.dos_bulk)[o] = s;
    __builtin_amdgcn_wave_barrier();
    if (a.spin_mode && f < 2) {
        // surfstat sums GRR's spin traces over the top orbital indices,
        // SurfaceDOSkk over the bottom orbitals of the last layer
        const bool top = f == 0 || a.spin_mode == 1;
        const int *list = top ? a.top : a.bot;
        const int cnt = top ? a.ntop : a.nbot, off = top ? 0 : n - a.nw;
        double s0 = 0.0, s1 = 0.0, s2 = 0.0;
        for (int e = 0; e < cnt; ++e) {
            const int l = l0 + off + uniform(list[e]) - 1;
            s0 = s0 - readlane_f64(t.s[0], l);
            s1 = s1 - readlane_f64(t.s[1], l);
            s2 = s2 - readlane_f64(t.s[2], l);
        }
        if (lane == 0) {
            double *out = a.spin_out(o, f);
            out[0] = s0;
            out[(size_t)a.ninst] = s1;
            out[2 * (size_t)a.ninst] = s2;
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// Waves per SIMD: the loops hold about 160 registers, one 4 x 4 tile 80.
constexpr int kTinyOcc = 3, kTinyOcc1 = 6;

template <int KS>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kTinyOcc)))
tiny16_kernel(DecimateArgs a) {
    __shared__ Lds16 sh;
    const int lane = threadIdx.x, i = lane & 15, q = lane >> 4;
    const int n = a.n;
    for (;;) {
        const int t = take(a.queue, 1u);
        if (queue_empty((unsigned)t, a.ninst)) break;
        int ik;
        double2 z;
        instance_of(a, t, ik, z);
        const double2 *H00 = a.hk + (size_t)ik * 512, *H01 = H00 + 256;
        // eps_s = eps_t = H00, alpha = H01, beta = H01^dagger (src/surfgreen.f90:74-78)
        M16 es{{0, 0, 0, 0}, {0, 0, 0, 0}}, et;
#pragma unroll
        for (int v = 0; v < KS; ++v) {
            const int c = 4 * v + q;
            const double2 h = H00[i + 16 * c], s = H01[c + 16 * i];
            es.re[v] = h.x;
            es.im[v] = h.y;
            sh.al[c * kLd16 + i] = H01[i + 16 * c];
            sh.be[c * kLd16 + i] = make_double2(s.x, -s.y);
        }
        et = es;
        const M16 h0 = es;  // (KS <= 2: H00 stays in registers)
        const int o = a.inst_k ? t : ik + a.nk * (t - ik * a.nomega);
        int it = 1, status = 0;
        // f < 0: the iterations; then G_LL = (z - eps_s)^-1, G_RR = (z -
        // eps_t)^-1 and G_B = (z - eps_i)^-1 (:127-134)
        for (int f = -1; f < 3;) {
            // (the lane's numbers afresh: what derives from them is not kept
            // in registers through the loop)
            const int lane = opaque_tid(), i = lane & 15, q = lane >> 4;
            // g = (z - eps_i)^-1, eps_i = eps_s + eps_t - H00 (src/surfgreen.f90:88-89)
            M16 x{{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
            for (int v = 0; v < KS; ++v) {
                const double2 h = KS <= 2 ? make_double2(h0.re[v], h0.im[v]) : H00[i + 16 * (4 * v + q)];
                double ex = (es.re[v] + et.re[v]) - h.x, ey = (es.im[v] + et.im[v]) - h.y;
                if (f == 0) {
                    ex = es.re[v];
                    ey = es.im[v];
                } else if (f == 1) {
                    ex = et.re[v];
                    ey = et.im[v];
                }
                const bool in = i < n && 4 * v + q < n, dg = i == 4 * v + q;
                x.re[v] = in ? (dg ? z.x : 0.0) - ex : dg && KS > 2 ? 1.0 : 0.0;
                x.im[v] = in ? (dg ? z.y : 0.0) - ey : 0.0;
            }
            if (inverse16<KS>(x, n, sh, lane)) status |= 1;
            if (f >= 0) {
                bool up = false;
                const int pr = a.spin_mode && i < n ? spin_partner(i, a.nw, up) : -1;
                tiny_traces(a, f, o,
                            terms_of(a, sh.g[i * (kLd16 + 1)], sh.g[i + std::max(pr, 0) * kLd16], pr, up),
                            0, lane);
                if (a.gfull) {
                    double2 *full = a.gfull + ((size_t)t * 3 + f) * n * n;
                    for (int e = lane; e < n * n; e += 64) full[e] = sh.g[e % n + (e / n) * kLd16];
                }
                wave_order();
                ++f;
                continue;
            }
            // m1 = alpha g, m2 = beta g (:92-95)
            M16 c = read_c16<KS>(sh.g, i, q);
            const M16 m1 = mul16<KS>(c, read_r16<KS>(sh.al, i, q));
            __builtin_amdgcn_sched_barrier(0);
            const M16 m2 = mul16<KS>(c, read_r16<KS>(sh.be, i, q));
            __builtin_amdgcn_sched_barrier(0);
            // eps_s += m1 beta, beta' = m2 beta (:98-102, 116-117)
            c = read_c16<KS>(sh.be, i, q);
            M16 d = mul16<KS>(c, m1);
            es.re += d.re;
            es.im += d.im;
            __builtin_amdgcn_sched_barrier(0);
            d = mul16<KS>(c, m2);
            wave_order();
            write16<KS>(d, sh.be, i, q);
            __builtin_amdgcn_sched_barrier(0);
            // eps_t += m2 alpha, alpha' = m1 alpha (:107-114)
            c = read_c16<KS>(sh.al, i, q);
            d = mul16<KS>(c, m2);
            et.re += d.re;
            et.im += d.im;
            __builtin_amdgcn_sched_barrier(0);
            d = mul16<KS>(c, m1);
            wave_order();
            write16<KS>(d, sh.al, i, q);
            __builtin_amdgcn_sched_barrier(0);
            // stop when sum_ij |alpha'_ij| <= accuracy (:120-122)
            // (up to order 8 in the order of tiny4_kernel: columns, halves of
            // the rows, columns, rows)
            double asum = 0.0;
#pragma unroll
            for (int v = 0; v < KS; ++v) asum += cabs_scaled(d.re[v], d.im[v]);
            asum += dpp_f64<0x128>(asum);  // row_ror:8
            asum += dpp_f64<0x124>(asum);  // row_ror:4
            asum = quad_rows_sum(asum);
            const bool conv = uniform(asum <= a.accuracy);
            if (conv || it >= a.itermax) {
                if (!conv) status |= 2;
                f = 0;
            } else {
                ++it;
            }
        }
        if (lane == 0) {
            if (a.iters) a.iters[o] = it;
            if (a.status) a.status[o] = status;
            __threadfence();
            atomicAdd(a.queue + 1, 1u);
        }
    }
}

// ---- four instances a wave, orders up to 8 ---------------------------------
// KB x KB tiles of 4 (KB = 1, 2); lane i + 4 b + 16 q, b the instance.

template <int KB>
struct M4 {
    double re[KB][KB], im[KB][KB];
};

__device__ __forceinline__ double mfma4(double a, double b, double c) {
    return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ double mfma4_neg(double a, double b, double c) {
    return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 1);
}

template <int KB>
__device__ __forceinline__ M4<KB> mul4(const M4<KB> &c, const M4<KB> &r) {
    M4<KB> d;
#pragma unroll
    for (int I = 0; I < KB; ++I)
#pragma unroll
        for (int J = 0; J < KB; ++J) d.re[I][J] = d.im[I][J] = 0.0;
#pragma unroll
    for (int K = 0; K < KB; ++K) {
#pragma unroll
        for (int I = 0; I < KB; ++I)
#pragma unroll
            for (int J = 0; J < KB; ++J) {
                d.re[I][J] = mfma4(c.re[K][J], r.re[I][K], d.re[I][J]);
                d.im[I][J] = mfma4(c.re[K][J], r.im[I][K], d.im[I][J]);
            }
#pragma unroll
        for (int I = 0; I < KB; ++I)
#pragma unroll
            for (int J = 0; J < KB; ++J) {
                d.re[I][J] = mfma4_neg(c.im[K][J], r.im[I][K], d.re[I][J]);
                d.im[I][J] = mfma4(c.im[K][J], r.re[I][K], d.im[I][J]);
            }
    }
    return d;
}

// Place of element (r, c) of instance b: lanes along r, and lanes along c, fall
// on different banks.
template <int KB>
__device__ __forceinline__ int at4(int r, int c, int b) {
    return ((r >> 2) * KB + (c >> 2)) * 64 + 16 * (r & 3) + 4 * b + ((r + c) & 3);
}

template <int KB>
struct Lds4 {
    // the four instances' matrices by at4(); before the inverse g holds a
    // panel's pivot rows
    double2 g[KB * KB * 64], al[KB * KB * 64], be[KB * KB * 64];
};

template <int KB>
__device__ __forceinline__ M4<KB> read_c4(const double2 *m, int i, int b, int q) {
    M4<KB> c;
#pragma unroll
    for (int I = 0; I < KB; ++I)
#pragma unroll
        for (int J = 0; J < KB; ++J) {
            const double2 v = m[at4<KB>(4 * I + q, 4 * J + i, b)];
            c.re[I][J] = v.x;
            c.im[I][J] = v.y;
        }
    return c;
}

template <int KB>
__device__ __forceinline__ M4<KB> read_r4(const double2 *m, int i, int b, int q) {
    M4<KB> r;
#pragma unroll
    for (int I = 0; I < KB; ++I)
#pragma unroll
        for (int J = 0; J < KB; ++J) {
            const double2 v = m[at4<KB>(4 * I + i, 4 * J + q, b)];
            r.re[I][J] = v.x;
            r.im[I][J] = v.y;
        }
    return r;
}

template <int KB>
__device__ __forceinline__ void write4(const M4<KB> &r, double2 *m, int i, int b, int q) {
#pragma unroll
    for (int I = 0; I < KB; ++I)
#pragma unroll
        for (int J = 0; J < KB; ++J)
            m[at4<KB>(4 * I + i, 4 * J + q, b)] = make_double2(r.re[I][J], r.im[I][J]);
}

// As inverse16, for the four instances at once; the lanes of a singular one
// return true.
template <int KB>
__device__ __forceinline__ bool inverse4(M4<KB> &x, int n, Lds4<KB> &sh, int lane) {
    const int i = lane & 3, b = (lane >> 2) & 3, q = lane >> 4;
    int free[KB], srow[KB], prow[KB];
    double2 myr[KB];
#pragma unroll
    for (int I = 0; I < KB; ++I) {
        free[I] = -1;
        srow[I] = 1 << 20;
        prow[I] = 4 * I + q;
        myr[I] = make_double2(1.0, 0.0);
    }
    int sing = 0;
    auto panel = [&](auto tc) {
        constexpr int t = tc;
        auto step = [&](auto kc) {
            constexpr int k = kc;
            const int own = (16 * k + (lane & 15)) << 2;
            double2 f[KB];  // the step's column, to every lane of its rows
            // pivot search: the high word of |re| + |im| over the row's tag;
            // where a second row of one of the instances has the same upper
            // bits (seldom), the largest value and the lowest row that has it
            int key = 0, next = 0;  // the larger of the lane's rows, the other
#pragma unroll
            for (int I = 0; I < KB; ++I) {
                f[I] = make_double2(lane_f64(own, x.re[I][t]), lane_f64(own, x.im[I][t]));
                const int kI = (__double2hiint(pivot_value(f[I].x, f[I].y, free[I])) & ~15) | (15 - 4 * I - i);
                next = I == 0 ? 0 : std::min(key, kI);
                key = std::max(key, kI);
            }
            int top = key;
            top = std::max(top, __builtin_amdgcn_mov_dpp(top, 0xB1, 0xf, 0xf, true));  // quad_perm 1,0,3,2
            top = std::max(top, __builtin_amdgcn_mov_dpp(top, 0x4E, 0xf, 0xf, true));  // quad_perm 2,3,0,1
            if (__ballot((key == top ? next : key) >= (top & ~15))) {
                double v[KB], best = 0.0;
#pragma unroll
                for (int I = 0; I < KB; ++I) {
                    v[I] = pivot_value(f[I].x, f[I].y, free[I]);
                    best = fmax_nocanon(best, v[I]);
                }
                best = fmax_nocanon(best, dpp_f64<0xB1>(best));
                best = fmax_nocanon(best, dpp_f64<0x4E>(best));
                int tag = 0;
#pragma unroll
                for (int I = 0; I < KB; ++I) tag = std::max(tag, v[I] == best ? 15 - 4 * I - i : 0);
                tag = std::max(tag, __builtin_amdgcn_mov_dpp(tag, 0xB1, 0xf, 0xf, true));
                tag = std::max(tag, __builtin_amdgcn_mov_dpp(tag, 0x4E, 0xf, 0xf, true));
                sing |= !(best > 0.0) && 4 * t + k < n;
                top = (__double2hiint(best) & ~15) | tag;
            }
            const int p = 15 - (top & 15);
            double sr = x.re[0][t], si = x.im[0][t];
            if constexpr (KB == 2)
                if (p >= 4) {
                    sr = x.re[1][t];
                    si = x.im[1][t];
                }
            const int src = ((p & 3) | (lane & 60)) << 2;
            const double2 y = make_double2(lane_f64(src, sr), lane_f64(src, si));
            // the pivot, from the lane of its row to the others of the column
            auto pivot = [&](auto part) {
                int v = 0;
#pragma unroll
                for (int I = 0; I < KB; ++I) v |= part(f[I]) & (4 * I + i == p ? -1 : 0);
                v |= __builtin_amdgcn_mov_dpp(v, 0xB1, 0xf, 0xf, true);
                return v | __builtin_amdgcn_mov_dpp(v, 0x4E, 0xf, 0xf, true);
            };
            double2 r = crecip_scaled(
                make_double2(__hiloint2double(pivot([](double2 z) { return __double2hiint(z.x); }),
                                              pivot([](double2 z) { return __double2loint(z.x); })),
                             __hiloint2double(pivot([](double2 z) { return __double2hiint(z.y); }),
                                              pivot([](double2 z) { return __double2loint(z.y); }))),
                (top >> 20) - 1022);
            double2 u = cmul_fma(y, r);
            const bool mine = q == k;
            if (mine) {
                u = r;
                prow[t] = p;
            }
#pragma unroll
            for (int I = 0; I < KB; ++I) {
                double yr = mine ? 0.0 : x.re[I][t], yi = mine ? 0.0 : x.im[I][t];
                if (4 * I + i == p) {
                    f[I] = make_double2(0.0, 0.0);
                    free[I] = 0;
                    srow[I] = 4 * t + k;
                    myr[I] = r;
                }
                x.re[I][t] = fma(-f[I].x, u.x, fma(f[I].y, u.y, yr));
                x.im[I][t] = fma(-f[I].x, u.y, fma(-f[I].y, u.x, yi));
            }
        };
        each_of(std::make_integer_sequence<int, 4>(), step);
        if constexpr (KB == 2) {
            constexpr int v = 1 - t;
#pragma unroll
            for (int I = 0; I < KB; ++I) {
                const int k = srow[I] - 4 * t;
                if (k >= 0 && k < 4)
                    sh.g[16 * k + 4 * b + q] = make_double2(x.re[I][v], x.im[I][v]);
            }
            wave_order();
            double2 a = sh.g[lane];
            wave_order();
#pragma unroll
            for (int I = 0; I < KB; ++I) {
                const double mr = x.re[I][t], mi = x.im[I][t];
                x.re[I][v] = mfma4(a.x, mr, x.re[I][v]);
                x.im[I][v] = mfma4(a.x, mi, x.im[I][v]);
                x.re[I][v] = mfma4_neg(a.y, mi, x.re[I][v]);
                x.im[I][v] = mfma4(a.y, mr, x.im[I][v]);
            }
        }
#pragma unroll
        for (int I = 0; I < KB; ++I)
            if (prow[t] == 4 * I + i) x.re[I][t] += 1.0;
    };
    each_of(std::make_integer_sequence<int, KB>(), panel);
#pragma unroll
    for (int I = 0; I < KB; ++I)
#pragma unroll
        for (int J = 0; J < KB; ++J) {
            const int r = sing ? 4 * I + i : srow[I], c = sing ? 4 * J + q : prow[J];
            double2 e = cmul_fma(make_double2(x.re[I][J], x.im[I][J]), myr[I]);
            if (sing) e = make_double2(r == c && r < n ? 1.0 : 0.0, 0.0);
            sh.g[at4<KB>(r, c, b)] = e;
        }
    wave_order();
    return sing;
}

template <int KB>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(KB == 1 ? kTinyOcc1 : kTinyOcc)))
tiny4_kernel(DecimateArgs a) {
    __shared__ Lds4<KB> sh;
    const int lane = threadIdx.x, i = lane & 3, b = (lane >> 2) & 3, q = lane >> 4;
    const int n = a.n;
    for (;;) {
        const int t0 = take(a.queue, 4u);
        if (queue_empty((unsigned)t0, a.ninst)) break;
        // the last wave's spare lanes repeat the last instance
        const int t = t0 + std::min(b, a.ninst - 1 - t0);
        int ik;
        double2 z;
        instance_of(a, t, ik, z);
        const double2 *H00 = a.hk + (size_t)ik * 512, *H01 = H00 + 256;
        M4<KB> es, et;
#pragma unroll
        for (int I = 0; I < KB; ++I)
#pragma unroll
            for (int J = 0; J < KB; ++J) {
                const int r = 4 * I + i, c = 4 * J + q;
                const double2 h = H00[r + 16 * c], v = H01[c + 16 * r];
                es.re[I][J] = h.x;
                es.im[I][J] = h.y;
                sh.al[at4<KB>(r, c, b)] = H01[r + 16 * c];
                sh.be[at4<KB>(r, c, b)] = make_double2(v.x, -v.y);
            }
        et = es;
        const int o = a.inst_k ? t : ik + a.nk * (t - ik * a.nomega);
        const int mine = std::min(4, a.ninst - t0);
        // The instances of a wave start together and stop by themselves: one
        // that has stopped takes no more of the increments.
        int it = 1, myit = 0, status = 0;
        bool live = true;
        for (int f = -1; f < 3;) {
            const int lane = opaque_tid(), i = lane & 3, b = (lane >> 2) & 3, q = lane >> 4;
            M4<KB> x;
#pragma unroll
            for (int I = 0; I < KB; ++I)
#pragma unroll
                for (int J = 0; J < KB; ++J) {
                    const double2 h = H00[4 * I + i + 16 * (4 * J + q)];
                    double ex = (es.re[I][J] + et.re[I][J]) - h.x;
                    double ey = (es.im[I][J] + et.im[I][J]) - h.y;
                    if (f == 0) {
                        ex = es.re[I][J];
                        ey = es.im[I][J];
                    } else if (f == 1) {
                        ex = et.re[I][J];
                        ey = et.im[I][J];
                    }
                    const int r = 4 * I + i, c = 4 * J + q;
                    const bool in = r < n && c < n;
                    x.re[I][J] = in ? (r == c ? z.x : 0.0) - ex : r == c ? 1.0 : 0.0;
                    x.im[I][J] = in ? (r == c ? z.y : 0.0) - ey : 0.0;
                }
            const bool sing = inverse4<KB>(x, n, sh, lane);
            if ((live || f >= 0) && sing) status |= 1;
            if (f >= 0) {
                // lane 8 b' + r: the terms of orbital r of instance b'
                const int r = std::min(lane & 7, 4 * KB - 1), tb = (lane >> 3) & 3;
                bool up = false;
                const int pr = a.spin_mode && r < n ? spin_partner(r, a.nw, up) : -1;
                const Terms te = terms_of(a, sh.g[at4<KB>(r, r, tb)],
                                          sh.g[at4<KB>(r, std::min(std::max(pr, 0), 4 * KB - 1), tb)], pr, up);
                for (int m = 0; m < mine; ++m)
                    tiny_traces(a, f, __builtin_amdgcn_readlane(o, 4 * m), te, 8 * m, lane);
                if (a.gfull)
                    for (int m = 0; m < mine; ++m) {
                        double2 *full = a.gfull + ((size_t)(t0 + m) * 3 + f) * n * n;
                        for (int e = lane; e < n * n; e += 64) full[e] = sh.g[at4<KB>(e % n, e / n, m)];
                    }
                wave_order();
                ++f;
                continue;
            }
            auto add = [&](M4<KB> &e, const M4<KB> &d) {
#pragma unroll
                for (int I = 0; I < KB; ++I)
#pragma unroll
                    for (int J = 0; J < KB; ++J) {
                        e.re[I][J] += live ? d.re[I][J] : 0.0;
                        e.im[I][J] += live ? d.im[I][J] : 0.0;
                    }
            };
            M4<KB> c = read_c4<KB>(sh.g, i, b, q);
            const M4<KB> m1 = mul4<KB>(c, read_r4<KB>(sh.al, i, b, q));
            __builtin_amdgcn_sched_barrier(0);
            const M4<KB> m2 = mul4<KB>(c, read_r4<KB>(sh.be, i, b, q));
            __builtin_amdgcn_sched_barrier(0);
            c = read_c4<KB>(sh.be, i, b, q);
            add(es, mul4<KB>(c, m1));
            __builtin_amdgcn_sched_barrier(0);
            M4<KB> d = mul4<KB>(c, m2);
            wave_order();
            write4<KB>(d, sh.be, i, b, q);
            __builtin_amdgcn_sched_barrier(0);
            c = read_c4<KB>(sh.al, i, b, q);
            add(et, mul4<KB>(c, m2));
            __builtin_amdgcn_sched_barrier(0);
            d = mul4<KB>(c, m1);
            wave_order();
            write4<KB>(d, sh.al, i, b, q);
            __builtin_amdgcn_sched_barrier(0);
            // (in the order of tiny16_kernel)
            double asum = 0.0;
#pragma unroll
            for (int I = 0; I < KB; ++I) {
                double rsum = 0.0;
#pragma unroll
                for (int J = 0; J < KB; ++J) rsum += cabs_scaled(d.re[I][J], d.im[I][J]);
                asum += rsum;
            }
            asum = quad_rows_sum(asum);
            const bool conv = asum <= a.accuracy;
            if (live && (conv || it >= a.itermax)) {
                if (!conv) status |= 2;
                live = false;
                myit = it;
            }
            if (!__ballot(live))
                f = 0;
            else
                ++it;
        }
        if (i == 0 && q == 0 && b < mine) {
            if (a.iters) a.iters[o] = myit;
            if (a.status) a.status[o] = status;
        }
        __builtin_amdgcn_wave_barrier();
        if (lane == 0) {
            __threadfence();
            atomicAdd(a.queue + 1, (unsigned)mine);
        }
    }
}

template <typename K>
int launch_tiny(K kernel, const DecimateArgs &a, int per_wave, int occ, int num_cu, hipStream_t s) {
    const long waves = ((long)a.ninst + per_wave - 1) / per_wave;
    const long want = std::min<long>((long)num_cu * 4 * occ, waves);
    hipLaunchKernelGGL(kernel, dim3((unsigned)std::max<long>(1, want)), dim3(64), 0, s, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace

int decimate_tiny_max_n() { return 16; }

int decimate_tiny_run(const DecimateArgs &a, int num_cu, hipStream_t s) {
    if (a.n < 1 || a.n > decimate_tiny_max_n() || num_cu < 1) return -1;
    // Up to one instance a SIMD an instance
    // of order 8 is faster alone in its wave, whose pivots are then uniform
    // (a call of one instance 222 us as one of four, 160 us alone when the line
    // was drawn; the same bits, since the steps and the order of every sum are the
    // same).
    const bool alone = a.n > 8 || a.ninst <= 4L * num_cu;
    auto one = [&](auto kernel) { return launch_tiny(kernel, a, 1, kTinyOcc, num_cu, s); };
    auto four = [&](auto kernel, int occ) { return launch_tiny(kernel, a, 4, occ, num_cu, s); };
    switch ((a.n + 3) / 4) {
        case 1:
            return alone ? one(tiny16_kernel<1>) : four(tiny4_kernel<1>, kTinyOcc1);
        case 2:
            return alone ? one(tiny16_kernel<2>) : four(tiny4_kernel<2>, kTinyOcc);
        case 3: return one(tiny16_kernel<3>);
        default: return one(tiny16_kernel<4>);
    }
}

}  // namespace wtsurf
