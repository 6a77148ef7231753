// Device helpers shared by the batched kernels: complex pairs with the fused
// operations written out, the FP64 phasor and the reference's shift factor.
#pragma once

#include "leap_internal.h"
#include "phasor.h"

// Global-memory pointers: pointers read from a descriptor table are otherwise
// generic, and flat memory instructions share the LDS wait counter.
#define LEAP_GLOBAL __attribute__((address_space(1)))

namespace leap {
namespace dev {

// The device clock at the launch's first workgroup.
__device__ inline void stamp(uint64_t* at) {
    if (at && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *at = uint64_t(wall_clock64());
}

// Orders a wave's LDS writes before its later reads (no workgroup barrier).
__device__ inline void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename T>
struct C2 {
    T x, y;
};

// Complex product with the fused operations written out (no contraction), so
// every kernel evaluates it the same way.
template <typename T>
__device__ inline C2<T> cmul(C2<T> a, C2<T> b) {
#pragma clang fp contract(off)
    return {fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x)};
}

// a * z + v with fused multiply-adds.
template <typename T>
__device__ inline C2<T> horner_step(C2<T> a, C2<T> z, C2<T> v) {
    C2<T> r;
    r.x = fma(a.x, z.x, fma(-a.y, z.y, v.x));
    r.y = fma(a.x, z.y, fma(a.y, z.x, v.y));
    return r;
}

constexpr double kTwoPiHi = 6.283185307179586232;           // double(2 pi)
constexpr double kTwoPiLo = 2.4492935982947064e-16;         // 2 pi - double(2 pi)
constexpr double kInvTwoPi = 0.15915494309189533577;

// exp(i theta) with the argument reduced modulo 2 pi in FP64 and the sincos in FP32.
__device__ inline C2<float> phasor_mixed(double theta) {
    const double n = rint(theta * kInvTwoPi);
    double r = fma(-n, kTwoPiHi, theta);
    r = fma(-n, kTwoPiLo, r);
    float s, c;
    sincosf(float(r), &s, &c);
    return {c, s};
}

__device__ inline C2<double> phasor_f64(double theta) {
    const Phasor64 p = phasor64(theta);
    return {p.c, p.s};
}

// exp(i th) by reduction modulo pi / 32 with a two-part constant through FMAs, a 64-entry
// table in LDS and the series to r^8 (cos) and r^7 (sin) on |r| <= pi / 64, whose next terms
// are below 2.5e-20 and 4.6e-18: 17 FP64 instructions, two for the table's address and an LDS
// read.  The multiple k of pi / 32 is rounded by adding 1.5 2^52, which leaves k mod 2^32 in the
// low word.  Accurate for |th| < 2^40, NaN for a th that is not finite.
constexpr int kPhasorTable = 64;

// By every thread of the workgroup; a barrier orders it before the first use.
__device__ inline void phasor_table_init(double2* table) {
    for (uint32_t k = threadIdx.x; k < kPhasorTable; k += blockDim.x) {
        double sn, cs;
        sincospi(double(k) / 32.0, &sn, &cs);
        table[k] = make_double2(cs, sn);
    }
}

__device__ inline double2 phasor_table(const double2* __restrict__ table, double th) {
#pragma clang fp contract(off)
    constexpr double kStep = 10.185916357881301489;         // 32 / pi
    constexpr double kPiO32Hi = 0.098174770424681034875;    // double(pi / 32)
    constexpr double kPiO32Lo = 3.8270212473354786e-18;     // pi / 32 - double(pi / 32)
    constexpr double kRound = 6755399441055744.0;           // 1.5 2^52
    const double m = fma(th, kStep, kRound);
    const double k = m - kRound;
    const double2 t = table[__double2loint(m) & (kPhasorTable - 1)];
    double r = fma(-k, kPiO32Hi, th);
    r = fma(-k, kPiO32Lo, r);
    const double r2 = r * r;
    double s = fma(-1.0 / 5040.0, r2, 1.0 / 120.0);
    s = fma(s, r2, -1.0 / 6.0);
    s = fma(r * r2, s, r);  // sin r
    double c = fma(1.0 / 40320.0, r2, -1.0 / 720.0);
    c = fma(c, r2, 1.0 / 24.0);
    c = fma(c, r2, -0.5) * r2;  // cos r - 1
    return make_double2(fma(-t.y, s, fma(t.x, c, t.x)), fma(t.x, s, fma(t.y, c, t.y)));
}

// -2 pi ((dd . uvw).z - w) (CpuLeapCalibrator.cc:190) with the fused operations written out.
__device__ inline double shift_factor(const double dz[3], double u, double v, double w) {
#pragma clang fp contract(off)
    double t = dz[0] * u;
    t = fma(dz[1], v, t);
    t = fma(dz[2], w, t);
    return -kTwoPi * (t - w);
}

}  // namespace dev
}  // namespace leap
