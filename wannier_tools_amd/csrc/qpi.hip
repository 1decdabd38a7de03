// The two QPI sums on gfx950.
//
// 1. Autocorrelation over a k-plane (SurfaceDOSkk's jdos / jsdos,
// src/fermiarc.f90:496-560):
//
//   out(iq1, iq2) = sum_{ik1, ik2} sum_f a_f(ik1, ik2) a_f(ik1q, ik2q)
//   ik1q - 1 = (ik1 - 1 + iq1 - 1) mod m1,   ik2q - 1 = (ik2 - 1 + iq2 - 1) mod m2
//
// The shifted factor only ever reads the m1 x m2 corner of the plane, and the
// unshifted index enters only through (ik - 1) mod m, so the plane is first
// folded onto that torus, E_f(c1, c2) = sum of a_f over ik1 - 1 = c1 (mod m1),
// ik2 - 1 = c2 (mod m2), and the sum becomes the cyclic correlation
//
//   C(p1, p2) = sum_{c1 < m1, c2 < m2} sum_f E_f(c1, c2) a_f((c1 + p1) mod m1, (c2 + p2) mod m2)
//
// with out(iq1, iq2) = C((iq1 - 1) mod m1, (iq2 - 1) mod m2): O((m1 m2)^2) FP64
// multiply-adds, summed as they stand (a transform would leave an absolute
// error of the largest C everywhere, and the fields' peaks span decades).
// correlate_kernel takes R2 values of p2 and all p1 per workgroup, 8
// consecutive p1 per thread: a thread slides an 8-wide window of each of its
// R2 rows of a_f over the row of E_f, one LDS read of a row and one of E
// (broadcast) for 8 R2 multiply-adds, where a thread per (p1, p2) took two
// reads for each: at 257 x 257, moduli 256 and four fields, 6.97 ms, bound by
// the LDS reads, and 0.73 ms now (rows staged one load at a time a thread 0.79,
// windows of two rows 0.81).  Rows go in groups of G values of c2, one per group
// of threads; the sum over c2 is cut into slices so that there are workgroups
// for the whole chip, and expand_kernel adds the slices in order.  Bound by the
// FP64 vector ALUs.
//
// 2. Linear autocorrelation along a k path, per energy (surfstat_jdos,
// src/surfstat.f90:891-907): with h = (nk - 1)/2 and s = iq - h,
//
//   out(iq, j) = sum_{ik = max(1, 1 - s)}^{min(2h + 1, 2h + 1 - s)} a(ik, j) a(ik + s, j)
//
// the terms added in the reference's order.  kpath_jdos_kernel stages JT
// energies of the path in LDS and gives each thread one energy and eight
// consecutive shifts, sliding an 8-wide window over the path: two LDS reads for
// eight multiply-adds (one thread per sum from global memory: 388 us at 512 x
// 512 and four fields, 50 us staged), and the same kernel reads either order of the arrays
// (k or energy fastest), so that no caller transposes.  Paths too long for LDS,
// and the smallest calls, take kpath_jdos_long_kernel, one thread per (iq, j,
// field) from global memory; long paths with the energy fastest are exchanged
// on the device first, for its loads' sake.
#include <algorithm>

#include "wtsurf_device.h"
#include "wtsurf_internal.h"

namespace wtsurf {

namespace {

constexpr int kCorrBlock = 256;

// E_f(c1, c2) for c1 < m1, c2 < m2; fields [nfield][nky][nkx], E [nfield][m2][m1].
__global__ void __launch_bounds__(kCorrBlock) fold_kernel(const double *__restrict__ a, int nkx,
                                                          int nky, int m1, int m2, int nfield,
                                                          double *__restrict__ e) {
    const long total = (long)nfield * m1 * m2;
    for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < total;
         t += (long)gridDim.x * blockDim.x) {
        const int c1 = (int)(t % m1);
        const int c2 = (int)((t / m1) % m2);
        const int f = (int)(t / ((long)m1 * m2));
        const double *af = a + (size_t)f * nkx * nky;
        double s = 0.0;
        for (int i2 = c2; i2 < nky; i2 += m2)
            for (int i1 = c1; i1 < nkx; i1 += m1) s += af[i1 + (size_t)nkx * i2];
        e[t] = s;
    }
}

// Place of element x of a row of a in LDS: two doubles of padding in eight, so
// that the threads' windows (8 apart) fall on different banks and on 16 B.
__host__ __device__ __forceinline__ constexpr int skew(int x) { return x + 2 * (x >> 3); }
// Length of a row of a of len elements, even.
__host__ __device__ __forceinline__ constexpr int row_length(int len) { return (skew(len) + 2) & ~1; }

// Slice blockIdx.y of C(p1, p2) for p2 = R2 blockIdx.x ..: threads tp = tid % TP
// (p1 = 8 tp .. 8 tp + 7) of group g = tid / TP (c2 = c20 + g of each chunk).
// part [slices][m2][m1].  Dynamic LDS: G rows of E (of an even length), G + R2 - 1
// skewed rows of a.
template <int R2>
__global__ void __launch_bounds__(kCorrBlock) correlate_kernel(
    const double *__restrict__ a, const double *__restrict__ e, int nkx, int nky, int m1, int m2,
    int nfield, int TP, int JN, int len, double *__restrict__ part) {
    extern __shared__ __align__(16) double lds[];
    const int G = kCorrBlock / TP;
    const int ld = row_length(len);
    const int le = (m1 + 1) & ~1;
    double *er = lds;                   // [G][le]
    double *ar = lds + (size_t)G * le;  // [G + R2 - 1][ld]
    const int tid = threadIdx.x;
    const int tp = tid % TP, g = tid / TP;
    const int sj = tid % JN, srow = 4 * (tid / JN), sstep = 4 * (kCorrBlock / JN);
    const int p20 = R2 * blockIdx.x;
    const int chunks = (m2 + G - 1) / G;  // per field
    const long total = (long)nfield * chunks;
    const long k0 = total * blockIdx.y / gridDim.y, k1 = total * (blockIdx.y + 1) / gridDim.y;
    double acc[R2][8];
#pragma unroll
    for (int j = 0; j < R2; ++j)
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[j][i] = 0.0;
    for (long k = k0; k < k1; ++k) {
        const int f = (int)(k / chunks), c20 = (int)(k - (long)f * chunks) * G;
        const int ng = min(G, m2 - c20);  // rows of this chunk
        const double *ef = e + ((size_t)f * m2 + c20) * m1;
        const double *af = a + (size_t)f * nkx * nky;
        __syncthreads();  // the previous rows are no longer read
        // (JN threads along a row, the others on other rows; four loads in
        // flight a thread)
        const int p2 = (c20 + p20) % m2, rows = ng + R2 - 1;
        for (int j = sj; j < m1; j += JN) {
            for (int row = srow; row < rows; row += sstep) {
                double v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    int r2 = p2 + std::min(row + u, rows - 1);
                    r2 = r2 < m2 ? r2 : r2 % m2;
                    v[u] = af[(size_t)nkx * r2 + j];
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    for (int x = j; x < len; x += m1)  // around the torus
                        ar[std::min(row + u, rows - 1) * ld + skew(x)] = v[u];
            }
            for (int row = srow; row < ng; row += sstep) {
                double v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = ef[(size_t)std::min(row + u, ng - 1) * m1 + j];
#pragma unroll
                for (int u = 0; u < 4; ++u) er[std::min(row + u, ng - 1) * le + j] = v[u];
            }
        }
        __syncthreads();
        if (g < ng) {
            const double *eg = er + g * le;
            const double *w0 = ar + g * ld + 10 * tp;  // window of p2 = p20 + j: row g + j
            double w[R2][8];
#pragma unroll
            for (int j = 0; j < R2; ++j)
#pragma unroll
                for (int i = 0; i < 8; ++i) w[j][i] = w0[j * ld + i];
            int c1 = 0;
            for (; c1 + 8 <= m1; c1 += 8) {
                w0 += 10;
                double2 e2[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) e2[t] = *reinterpret_cast<const double2 *>(eg + c1 + 2 * t);
#pragma unroll
                for (int t = 0; t < 8; t += 2) {
                    double2 nw[R2];
#pragma unroll
                    for (int j = 0; j < R2; ++j) nw[j] = *reinterpret_cast<const double2 *>(w0 + j * ld + t);
#pragma unroll
                    for (int j = 0; j < R2; ++j) {
#pragma unroll
                        for (int i = 0; i < 8; ++i)
                            acc[j][i] = fma(e2[t / 2].x, w[j][(t + i) & 7], acc[j][i]);
                        w[j][t] = nw[j].x;
                    }
#pragma unroll
                    for (int j = 0; j < R2; ++j) {
#pragma unroll
                        for (int i = 0; i < 8; ++i)
                            acc[j][i] = fma(e2[t / 2].y, w[j][(t + 1 + i) & 7], acc[j][i]);
                        w[j][t + 1] = nw[j].y;
                    }
                }
            }
            w0 += 10;
#pragma unroll
            for (int t = 0; t < 7; ++t)
                if (c1 + t < m1) {
                    const double ev = eg[c1 + t];
#pragma unroll
                    for (int j = 0; j < R2; ++j) {
#pragma unroll
                        for (int i = 0; i < 8; ++i) acc[j][i] = fma(ev, w[j][(t + i) & 7], acc[j][i]);
                        w[j][t] = w0[j * ld + t];
                    }
                }
        }
    }
    // the groups' sums, added in order
    __syncthreads();
    for (int j = 0; j < R2; ++j) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            double v = acc[0][i];
#pragma unroll
            for (int q = 1; q < R2; ++q)
                if (j == q) v = acc[q][i];
            lds[(g * 8 + i) * TP + tp] = v;
        }
        __syncthreads();
        if (p20 + j < m2)
            for (int p1 = tid; p1 < m1; p1 += kCorrBlock) {
                double v = 0.0;
                for (int q = 0; q < G; ++q) v += lds[(q * 8 + (p1 & 7)) * TP + (p1 >> 3)];
                part[((size_t)blockIdx.y * m2 + p20 + j) * m1 + p1] = v;
            }
        __syncthreads();
    }
}

// out(iq1, iq2) = C((iq1 - 1) mod m1, (iq2 - 1) mod m2), C the sum of its slices;
// out [nky][nkx].
__global__ void __launch_bounds__(kCorrBlock) expand_kernel(const double *__restrict__ c, int nkx,
                                                            int nky, int m1, int m2, int slices,
                                                            double *__restrict__ out) {
    const long total = (long)nkx * nky;
    for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < total;
         t += (long)gridDim.x * blockDim.x) {
        const int i1 = (int)(t % nkx), i2 = (int)(t / nkx);
        const double *p = c + (size_t)(i2 % m2) * m1 + (i1 % m1);
        double s = 0.0;
        for (int q = 0; q < slices; ++q) s += p[(size_t)q * m1 * m2];
        out[t] = s;
    }
}

// out_f(iq, j) for JT energies j of one field and 8 kCorrBlock / JT shifts iq;
// element (f, j, ik) at f fs + j js + ik ks.  Dynamic LDS nk (JT + 1) doubles.
template <int JT>
__global__ void __launch_bounds__(kCorrBlock) kpath_jdos_kernel(const double *__restrict__ a,
                                                                int nk, int nomega, size_t fs,
                                                                size_t js, size_t ks,
                                                                double *__restrict__ out) {
    extern __shared__ __align__(16) double lds[];  // [nk][JT + 1]
    constexpr int LD = JT + 1;
    const int tid = threadIdx.x;
    const int nj = (nomega + JT - 1) / JT;
    const int f = blockIdx.x / nj, j0 = (blockIdx.x % nj) * JT;
    const double *src = a + f * fs + j0 * js;
    // the faster of the two indices along the threads
    if (ks == 1) {
        for (int j = 0; j < JT && j0 + j < nomega; ++j)
            for (int ik = tid; ik < nk; ik += kCorrBlock) lds[ik * LD + j] = src[j * js + ik];
    } else {
        for (int e = tid; e < nk * JT; e += kCorrBlock) {
            const int j = e % JT, ik = e / JT;
            if (j0 + j < nomega) lds[ik * LD + j] = src[j * js + ik * ks];
        }
    }
    __syncthreads();
    const int j = tid % JT, h = (nk - 1) / 2;
    const int iq0 = 8 * (blockIdx.y * (kCorrBlock / JT) + tid / JT);
    if (j0 + j >= nomega || iq0 >= nk) return;
    const double *r = lds + j;
    double acc[8], w[8];
    int lo[8], hi[8], first = nk, last = -1, from = 0, to = nk;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        // (past the last shift: that one again, not stored)
        const int sft = min(iq0 + i, nk - 1) + 1 - h;
        lo[i] = sft < 0 ? -sft : 0;                 // 0-based first ik
        hi[i] = sft > 0 ? 2 * h - sft : 2 * h;      // 0-based last ik
        acc[i] = 0.0;
        if (hi[i] >= lo[i]) {
            first = min(first, lo[i]);
            last = max(last, hi[i]);
        }
        from = max(from, lo[i]);
        to = min(to, hi[i]);
    }
    const int s0 = iq0 + 1 - h;
    // the ends of the path, where not every shift has a term
    auto edge = [&](int ik) {
        const double x = r[ik * LD];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (ik >= lo[i] && ik <= hi[i]) acc[i] = fma(x, r[min(ik + s0 + i, nk - 1) * LD], acc[i]);
    };
    int ik = first;
    for (; ik < from && ik <= last; ++ik) edge(ik);
    if (ik + 7 <= to) {
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i] = r[min(ik + s0 + i, nk - 1) * LD];
        for (; ik + 7 <= to; ik += 8) {
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const double x = r[(ik + t) * LD];
#pragma unroll
                for (int i = 0; i < 8; ++i) acc[i] = fma(x, w[(t + i) & 7], acc[i]);
                // the window's next value, past the path after its last use
                const int n = ik + t + s0 + 8;
                w[t] = r[(n < nk ? n : nk - 1) * LD];
            }
        }
    }
    for (; ik <= last; ++ik) edge(ik);
    double *dst = out + f * fs + (j0 + j) * js;
#pragma unroll
    for (int i = 0; i < 8; ++i)
        if (iq0 + i < nk) dst[(iq0 + i) * ks] = acc[i];
}

// out_f(iq, j) from global memory, element (f, j, ik) as above; thread iq of row
// (j, f) = row0 + blockIdx.y.
__global__ void __launch_bounds__(kCorrBlock) kpath_jdos_long_kernel(const double *__restrict__ a,
                                                                     int nk, int nomega, size_t fs,
                                                                     size_t js, size_t ks, int row0,
                                                                     double *__restrict__ out) {
    const int iq = blockIdx.x * kCorrBlock + threadIdx.x;  // 0-based
    if (iq >= nk) return;
    const int rw = row0 + blockIdx.y;
    const size_t row = (rw / nomega) * fs + (rw % nomega) * js;
    const double *r = a + row;
    const int h = (nk - 1) / 2;
    const int sft = iq + 1 - h;
    const int lo = sft < 0 ? -sft : 0;                       // 0-based first ik
    const int hi = sft > 0 ? 2 * h - sft : 2 * h;            // 0-based last ik
    double s = 0.0;
    for (int ik = lo; ik <= hi; ++ik) s += r[ik * ks] * r[(ik + sft) * ks];
    out[row + iq * ks] = s;
}

// dst [nfield][cols][rows] = src [nfield][rows][cols]
__global__ void __launch_bounds__(kCorrBlock) transpose_kernel(const double *__restrict__ src, int rows,
                                                               int cols, long total,
                                                               double *__restrict__ dst) {
    const long plane = (long)rows * cols;
    for (long e = blockIdx.x * (long)kCorrBlock + threadIdx.x; e < total; e += (long)gridDim.x * kCorrBlock) {
        const long f = e / plane, r = e - f * plane;
        dst[e] = src[f * plane + (r % rows) * cols + r / rows];
    }
}

}  // namespace

int kplane_corr_max_m() { return kKplaneMaxM; }

int transpose_launch(const double *src, int rows, int cols, int nfield, double *dst, hipStream_t s) {
    const long total = (long)rows * cols * nfield;
    const unsigned blocks = (unsigned)std::min<long>((total + kCorrBlock - 1) / kCorrBlock, 1 << 16);
    hipLaunchKernelGGL(transpose_kernel, dim3(blocks), dim3(kCorrBlock), 0, s, src, rows, cols, total, dst);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int kpath_jdos_launch(const double *fields, int nk, int nomega, int nfield, bool k_fastest,
                      double *out, hipStream_t s) {
    if (nk < 1 || nomega < 1 || nfield < 1 || (long)nomega * nfield > 65535L * 1024) return -1;
    const size_t fs = (size_t)nk * nomega, js = k_fastest ? nk : 1, ks = k_fastest ? 1 : nomega;
    auto go = [&](auto kernel, int JT) {
        const size_t lds = (size_t)nk * (JT + 1) * sizeof(double);
        if (lds > (size_t)64 * 1024 &&
            hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
            (void)hipGetLastError();  // the launch reports whether the size is accepted
        // (a launch has less than 2^32 threads along x: fields in pieces)
        const int per = 8 * kCorrBlock / JT, nj = (nomega + JT - 1) / JT;
        const int step = std::max(1, (1 << 22) / nj);
        for (int f0 = 0; f0 < nfield; f0 += step)
            hipLaunchKernelGGL(kernel, dim3((unsigned)std::min(step, nfield - f0) * nj, (nk + per - 1) / per),
                               dim3(kCorrBlock), lds, s, fields + f0 * fs, nk, nomega, fs, js, ks,
                               out + f0 * fs);
    };
    // as many energies as keep two workgroups of LDS on a CU, or at last one;
    // the smallest calls are a launch's latency, and staging only adds to it
    // (21 points and energies: 36 us from global memory, 40 staged)
    constexpr int kMaxLds = 80 * 1024 / sizeof(double);
    if (nk > kJdosStagedMaxNk || (nk <= 40 && nfield * nomega <= 256)) {
        for (int r0 = 0; r0 < nfield * nomega; r0 += 65535)
            hipLaunchKernelGGL(kpath_jdos_long_kernel,
                               dim3((nk + kCorrBlock - 1) / kCorrBlock,
                                    (unsigned)std::min(65535, nfield * nomega - r0)),
                               dim3(kCorrBlock), 0, s, fields, nk, nomega, fs, js, ks, r0, out);
    } else if (nk <= kMaxLds / 17)
        go(kpath_jdos_kernel<16>, 16);
    else if (nk <= kMaxLds / 5)
        go(kpath_jdos_kernel<4>, 4);
    else
        go(kpath_jdos_kernel<1>, 1);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

// Launch shape of correlate_kernel: threads along p1 (a power of two, so that
// the groups of threads tile the workgroup), threads along a row when rows are
// staged (a power of two: all of them stage narrow rows too, at m1 = 1, m2 =
// 2000 0.2 ms for 7.1 with one thread to a row's element), the LDS length of a row of
// a, R2 as large as two workgroups of LDS a CU allow, and slices for about
// four workgroups a CU.
struct CorrPlan {
    int tp, jn, len, r2, slices;
    size_t lds;
};
static CorrPlan corr_plan(int m1, int m2, int nfield) {
    CorrPlan p{};
    p.tp = 8;
    while (8 * p.tp < m1) p.tp *= 2;
    p.jn = 1;
    while (p.jn < m1 && p.jn < kCorrBlock) p.jn *= 2;
    p.len = m1 + 8 * p.tp + 8;
    const int G = kCorrBlock / p.tp;
    for (p.r2 = 4;; p.r2 /= 2) {
        const size_t rows = (size_t)G * ((m1 + 1) & ~1) + (size_t)(G + p.r2 - 1) * row_length(p.len);
        p.lds = std::max(rows, (size_t)8 * kCorrBlock) * sizeof(double);
        if (p.r2 == 1 || p.lds <= (size_t)80 * 1024) break;
    }
    const long blocks = (m2 + p.r2 - 1) / p.r2;
    const long chunks = (long)nfield * ((m2 + G - 1) / G);
    p.slices = (int)std::max<long>(1, std::min(chunks, (1024 + blocks - 1) / blocks));
    return p;
}

size_t kplane_corr_doubles(int m1, int m2, int nfield) {
    return (size_t)corr_plan(m1, m2, nfield).slices * m1 * m2;
}

int kplane_corr_launch(const KplaneCorrArgs &k, hipStream_t s) {
    if (k.nkx < 1 || k.nky < 1 || k.m1 < 1 || k.m2 < 1 || k.m1 > k.nkx || k.m2 > k.nky ||
        k.m1 > kKplaneMaxM || k.nfield < 1)
        return -1;
    const long nfold = (long)k.nfield * k.m1 * k.m2;
    const int gfold = (int)std::min<long>((nfold + kCorrBlock - 1) / kCorrBlock, 4096);
    hipLaunchKernelGGL(fold_kernel, dim3(gfold), dim3(kCorrBlock), 0, s, k.fields, k.nkx, k.nky,
                       k.m1, k.m2, k.nfield, k.folded);
    const CorrPlan p = corr_plan(k.m1, k.m2, k.nfield);
    auto go = [&](auto kernel) {
        if (p.lds > (size_t)64 * 1024 &&
            hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.lds) != hipSuccess)
            (void)hipGetLastError();  // the launch reports whether the size is accepted
        hipLaunchKernelGGL(kernel, dim3((k.m2 + p.r2 - 1) / p.r2, p.slices), dim3(kCorrBlock), p.lds,
                           s, k.fields, k.folded, k.nkx, k.nky, k.m1, k.m2, k.nfield, p.tp, p.jn,
                           p.len, k.corr);
    };
    if (p.r2 == 4)
        go(correlate_kernel<4>);
    else if (p.r2 == 2)
        go(correlate_kernel<2>);
    else
        go(correlate_kernel<1>);
    const long nout = (long)k.nkx * k.nky;
    const int gout = (int)std::min<long>((nout + kCorrBlock - 1) / kCorrBlock, 4096);
    hipLaunchKernelGGL(expand_kernel, dim3(gout), dim3(kCorrBlock), 0, s, k.corr, k.nkx, k.nky,
                       k.m1, k.m2, p.slices, k.out);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace wtsurf
