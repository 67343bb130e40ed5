// site_stream.hpp -- a site's random stream dealt to the lanes of one wave, for
// the kernels that gate a site over many steps in one launch.
#pragma once
#include "mrg32k3a.hpp"

namespace casim {

// Streams in doubles, exact integers throughout (mrg32k3a.hpp has the
// recurrences): a product of 16 x 33 bits is one operation there, where the
// 32-bit integer form takes several quarter-rate multiplies and reductions.
// A channel's state is kept one generator step past the point where its draw
// starts, so that its last words are the draw's first values, and only reduced
// to (-m, 2 m).
constexpr double RM1 = 4294967087.0, RM2 = 4294944443.0;
// x minus a multiple of m, in (-m, 2 m) for |x| < 2^53
__device__ __forceinline__ double near53(double x, double m) {
    return __builtin_fma(-floor(x * (1.0 / m)), m, x);
}
__device__ __forceinline__ double mod53(double v, double m) {  // v in (-m, 2 m)
    v = v < 0.0 ? v + m : v;
    return v >= m ? v - m : v;
}
// sum of three products mod m, a as high and low 16 bits
__device__ __forceinline__ double row53(const double *a, const double *x, double m) {
    const double h = near53(__builtin_fma(a[0], x[0], __builtin_fma(a[2], x[1], a[4] * x[2])), m);
    return near53(__builtin_fma(h, 65536.0, __builtin_fma(a[1], x[0], __builtin_fma(a[3], x[1], a[5] * x[2]))), m);
}
__device__ __forceinline__ void jump53(const double *a, double x[6]) {
    double y[6];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        y[i] = row53(a + 6 * i, x, RM1);
        y[3 + i] = row53(a + 18 + 6 * i, x + 3, RM2);
    }
#pragma unroll
    for (int i = 0; i < 6; ++i) x[i] = y[i];
}
// The first U01 value of the draw that the state x belongs to; the draw itself
// is this plus up to 2^-24 (less 1 when that reaches 1).
__device__ __forceinline__ double first53(const double x[6]) {
    const double d = mod53(x[2], RM1) - mod53(x[5], RM2);
    return (d > 0.0 ? d : d + RM1) * mrg::NORM;
}
// Modular inverse of the recurrences' last coefficients: x_{n-3} = (a12 x_{n-2}
// - x_n) / a13 takes a state one step back.
constexpr uint64_t powmod(uint64_t b, uint64_t e, uint64_t m) {
    uint64_t v = 1;
    for (b %= m; e; e >>= 1, b = b * b % m)
        if (e & 1) v = v * b % m;
    return v;
}
constexpr uint32_t INV13 = (uint32_t)powmod(mrg::A13N, mrg::M1 - 2, mrg::M1);
constexpr uint32_t INV23 = (uint32_t)powmod(mrg::A23N, mrg::M2 - 2, mrg::M2);
static_assert((uint64_t)INV13 * mrg::A13N % mrg::M1 == 1 && (uint64_t)INV23 * mrg::A23N % mrg::M2 == 1, "inverses");
__device__ __forceinline__ void step_back(const uint32_t x[6], uint32_t y[6]) {
    const uint32_t u = mrg::mulmod(mrg::A12, x[0], mrg::C1, mrg::M1), v = mrg::mulmod(mrg::A21, x[4], mrg::C2, mrg::M2);
    const uint32_t du = u >= x[2] ? u - x[2] : u - x[2] + mrg::M1, dv = v >= x[5] ? v - x[5] : v - x[5] + mrg::M2;
    const uint32_t a = mrg::mulmod(du, INV13, mrg::C1, mrg::M1), b = mrg::mulmod(dv, INV23, mrg::C2, mrg::M2);
    y[2] = x[1], y[1] = x[0], y[0] = a;
    y[5] = x[4], y[4] = x[3], y[3] = b;
}

}  // namespace casim
