// Device-side building blocks shared by the wtsurf kernels (gfx950 / CDNA4).
//
// Matrix storage convention on the device: every per-instance complex matrix
// is an NP x NP column-major array of (re, im) pairs, NP = 16*Q the order
// rounded up to the MFMA tile edge.  The pad rows/columns hold exact zeros;
// every product of zero-padded operands keeps them zero, so the kernels work
// on the padded shape without masks.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

namespace wtsurf {

constexpr int kWave = 64;
constexpr int kBlock = 512;  // 8 waves, two per SIMD
constexpr int kWaves = kBlock / kWave;
constexpr int kChunk = 8;    // K-chunk (complex) staged through LDS per step
constexpr int kPanel = 8;    // Gauss-Jordan panel width (rank of each MFMA update)

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

// threadIdx.x hidden from loop-invariant code motion: address arithmetic that
// derives from it is then recomputed inside each device-function call instead
// of being hoisted out of the instance loop and held in registers throughout.
__device__ __forceinline__ int opaque_tid() {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

// Values every thread of the workgroup holds identically (read from LDS
// after a barrier) made provably uniform for the compiler.  Loops and
// branches that contain barriers must test only such values: a condition the
// compiler believes divergent lets its structurizer send different lanes of
// one wave around different cycles of the loop, and the barriers then pair
// up wrongly.
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ __forceinline__ double readlane_f64(double v, int lane) {
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ float readlane_f32(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// max(a, b) (a quiet NaN operand yields the other one, as fmax) for operands
// that are never signalling NaNs, which no arithmetic produces: one
// v_max_f64, without the quieting step fmax adds on values the compiler
// cannot prove canonical (every DPP-moved value).
__device__ __forceinline__ double fmax_nocanon(double a, double b) {
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// Median of three, one instruction.
__device__ __forceinline__ int imed3(int a, int b, int c) {
    int r;
    asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// Maximum over the 64 lanes of a wave of values whose maximum is >= 0
// (operands as fmax_nocanon), returned to every lane: DPP row shifts inside
// each row of 16 lanes, then row broadcasts 15 and 31 carry the partial
// maxima up to lane 63.  A shift's lanes without a source read 0 (bound_ctrl),
// which leaves a non-negative maximum as it is; the rows a broadcast does not
// write hold unspecified values, but none of them reaches lane 63.  No old
// value is kept, so no register copy precedes a DPP move.
__device__ __forceinline__ double wave_max_f64(double v) {
#define WT_DPP_MAX_STEP(ctrl, rmask)                                                  \
    {                                                                                  \
        const int hi = __double2hiint(v), lo = __double2loint(v);                      \
        const int h2 = __builtin_amdgcn_mov_dpp(hi, ctrl, rmask, 0xf, true);           \
        const int l2 = __builtin_amdgcn_mov_dpp(lo, ctrl, rmask, 0xf, true);           \
        v = fmax_nocanon(v, __hiloint2double(h2, l2));                                 \
    }
    WT_DPP_MAX_STEP(0x111, 0xf)  // row_shr:1
    WT_DPP_MAX_STEP(0x112, 0xf)  // row_shr:2
    WT_DPP_MAX_STEP(0x114, 0xf)  // row_shr:4
    WT_DPP_MAX_STEP(0x118, 0xf)  // row_shr:8
    WT_DPP_MAX_STEP(0x142, 0xa)  // row_bcast:15
    WT_DPP_MAX_STEP(0x143, 0xc)  // row_bcast:31
#undef WT_DPP_MAX_STEP
    return readlane_f64(v, 63);
}

// Complex arithmetic on (re, im) pairs of either precision.
template <typename C>
__device__ __forceinline__ C cmul(C a, C b) {
    C r;
    r.x = a.x * b.x - a.y * b.y;
    r.y = a.x * b.y + a.y * b.x;
    return r;
}
template <typename C>
__device__ __forceinline__ C cadd(C a, C b) {
    C r;
    r.x = a.x + b.x;
    r.y = a.y + b.y;
    return r;
}
// 1/z = conj(z) / |z|^2 without a division: both parts are scaled by 2^-e,
// e the binary exponent of max(|re|, |im|), so that |z|^2 lies in [1/4, 2)
// (no overflow or underflow whatever the magnitude of z); the hardware
// reciprocal of |z|^2 is refined by Newton steps (two in FP64, one in FP32:
// each step doubles the correct bits of the ~2^-23 estimate) and the result
// is scaled back by 2^-e.  A few ulp from the correctly rounded quotient.
__device__ __forceinline__ double2 crecip_fast(double2 z) {
    const int e = __builtin_amdgcn_frexp_exp(fmax(fabs(z.x), fabs(z.y)));
    const double x = __builtin_amdgcn_ldexp(z.x, -e), y = __builtin_amdgcn_ldexp(z.y, -e);
    const double d = fma(x, x, y * y);
    double r = __builtin_amdgcn_rcp(d);
    r = fma(r, fma(-d, r, 1.0), r);
    r = fma(r, fma(-d, r, 1.0), r);
    return make_double2(__builtin_amdgcn_ldexp(x * r, -e), __builtin_amdgcn_ldexp(-y * r, -e));
}
__device__ __forceinline__ float2 crecip_fast(float2 z) {
    const int e = __builtin_amdgcn_frexp_expf(fmaxf(fabsf(z.x), fabsf(z.y)));
    const float x = __builtin_amdgcn_ldexpf(z.x, -e), y = __builtin_amdgcn_ldexpf(z.y, -e);
    const float d = fmaf(x, x, y * y);
    float r = __builtin_amdgcn_rcpf(d);
    r = fmaf(r, fmaf(-d, r, 1.0f), r);
    return make_float2(__builtin_amdgcn_ldexpf(x * r, -e), __builtin_amdgcn_ldexpf(-y * r, -e));
}

// Per-precision MFMA: one 16x16x4 step, D += A B, with the operand layout
//   A[i][k]: lane i + 16k;  B[k][j]: lane j + 16k;  D[i][j]: lane j + 16*q,
// element v, where (checked on the device with known-answer products)
//   FP64: i = 4v + q       FP32: i = 4q + v.
template <typename R>
struct Prec;
template <>
struct Prec<double> {
    using C = double2;
    using V4 = v4d;
    __device__ static __forceinline__ V4 mfma(double a, double b, V4 c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    __device__ static __forceinline__ int out_row(int q, int v) { return 4 * v + q; }
    __device__ static __forceinline__ double readlane(double x, int l) { return readlane_f64(x, l); }
};
template <>
struct Prec<float> {
    using C = float2;
    using V4 = v4f;
    __device__ static __forceinline__ V4 mfma(float a, float b, V4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    __device__ static __forceinline__ int out_row(int q, int v) { return 4 * q + v; }
    __device__ static __forceinline__ float readlane(float x, int l) { return readlane_f32(x, l); }
};

// sqrt(x^2 + y^2) scaled by the exponent of the larger part, so that the
// squares neither overflow nor underflow.
__device__ __forceinline__ double cabs_scaled(double x, double y) {
    const int e = __builtin_amdgcn_frexp_exp(fmax(fabs(x), fabs(y)));
    const double xs = __builtin_amdgcn_ldexp(x, -e), ys = __builtin_amdgcn_ldexp(y, -e);
    return __builtin_amdgcn_ldexp(sqrt(fma(xs, xs, ys * ys)), e);
}

// D += -A B: the FP64 MFMA's negate bit of the first operand.
__device__ __forceinline__ v4d mfma_neg(double a, double b, v4d c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 1);
}

// Spin partner of orbital i (0-based) in layers of nw orbitals (-1: none), and
// whether i is spin up.
__device__ __forceinline__ int spin_partner(int i, int nw, bool &up) {
    const int nh = nw / 2, l = i % nw;
    up = l < nh;
    return l >= 2 * nh ? -1 : up ? i + nh : i - nh;
}

// 1/z as crecip_fast, the binary exponent e of |re| + |im| given: the scaled
// |z|^2 lies in [1/8, 1).
__device__ __forceinline__ double2 crecip_scaled(double2 z, int e) {
    const double x = __builtin_amdgcn_ldexp(z.x, -e), y = __builtin_amdgcn_ldexp(z.y, -e);
    const double d = fma(x, x, y * y);
    double r = __builtin_amdgcn_rcp(d);
    r = fma(r, fma(-d, r, 1.0), r);
    r = fma(r, fma(-d, r, 1.0), r);
    return make_double2(__builtin_amdgcn_ldexp(x * r, -e), __builtin_amdgcn_ldexp(-y * r, -e));
}

// LDS written by some lanes of a wave is read by others of the same wave
// after this: the LDS keeps a wave's accesses in order, the compiler must too.
__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

template <int... J, typename F>
__device__ __forceinline__ void each_of(std::integer_sequence<int, J...>, F &&step) {
    (step(std::integral_constant<int, J>()), ...);
}

}  // namespace wtsurf
