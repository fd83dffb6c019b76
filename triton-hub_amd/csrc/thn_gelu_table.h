// GeLU from tables in LDS, for the kernels over 16-bit rows in which vector instructions would bound it: the norms with a GeLU
// epilogue.  The normal distribution function Phi and GeLU' = Phi(x) + x*phi(x) are cut into intervals of 1/32 between -14
// and 6, each with a cubic of its own around its middle (10 KiB per table, which a workgroup fills while its first rows arrive).  A value costs 8
// or 9 vector instructions and one 16-byte read of LDS, which another pipe carries out, where the polynomial of thn_act_math.h takes 19 and 20
// slots: 2^25 normally distributed values in registers 15.2 -> 9.1 us, about 16 cycles of LDS per 64 lanes, more than half of them bank
// conflicts of lanes at different nodes.  LayerNorm + GeLU bfloat16 16384 x 4096: 28.1 and 37.6 vector instructions per element -> 21.1 and 28.7,
// forward + backward 145.4 -> 124.8 us, the forward then at the rate of its memory.  Intervals of 1/32 keep the tables small (finer
// ones would be more to fill) at the accuracy below.  Which kernels use it, with both sides over other widths: gelu_tabled() in thn_kernels.h.
//
// The cubics are the Taylor polynomials of degree 5 economised over the interval (the Chebyshev polynomials of degree 4 and 5 taken
// off), off by at most x^4 * 3.1e-10 of the value: below a rounded coefficient for |x| < 4.  Against float64, 2-norm, polynomial -> table: GeLU of
// normal values 3.88e-8 -> 3.23e-8 (at 1.5 times their spread and an offset of 0.25 3.30e-8 -> 3.14e-8), GeLU' 4.83e-8 -> 3.80e-8 (4.26e-8 -> 4.13e-8);
// Phi in bands of x [-2, -1] 1.2e-7 -> 3.6e-8, [-6, -5] 1.1e-6 -> 1.4e-7, [-9, -8] 2.0e-6 -> 9.0e-7, [-13, -12] 5.2e-6 -> 4.6e-6; GeLU' from 1 up, where it is 1 but for a rounded coefficient, 3.4e-8 -> 4.9e-8.
#pragma once

#include "thn_act_math.h"

namespace thn {

constexpr int kGeluPerUnit = 32, kGeluLow = -14, kGeluHigh = 6;
constexpr int kGeluNodes = (kGeluHigh - kGeluLow) * kGeluPerUnit + 1;

struct GeluTables {
    float cdf[kGeluNodes][4], slope[kGeluNodes][4];
};

// The tables, made by the compiler in float64: phi and Phi go from node to node by the series of exp and of the integral of
// phi, from the left, where both are positive sums without cancellation.
constexpr GeluTables make_gelu_tables() {
    GeluTables tables{};
    constexpr double h = 1.0 / kGeluPerUnit, r2 = h * h / 4.0, r4 = r2 * r2;
    double pdf = 1.0966065593889713e-43;      // phi(-14)
    double cdf = 7.793536819192799e-45;         // Phi(-14)
    for (int i = 0; i < kGeluNodes; ++i) {
        const double x = kGeluLow + i * h;
        // phi^(n)(x) = p[n]*phi(x): p[n + 1] = -(x*p[n] + n*p[n - 1])
        double p[18] = {1.0, -x};
        for (int n = 1; n < 17; ++n) p[n + 1] = -(x * p[n] + n * p[n - 1]);
        // coefficients 0 to 5 of Phi(x + d), and of (x + d)*phi(x + d), by powers of d
        double of_cdf[6] = {cdf}, of_slope[6] = {};
        double factorial = 1.0;
        for (int n = 0; n < 6; ++n) {
            if (n > 0) factorial *= n;
            if (n > 0) of_cdf[n] = pdf * p[n - 1] / factorial;
            const double derivative = x * p[n] + (n > 0 ? n * p[n - 1] : 0.0);       // of x*phi, over phi
            of_slope[n] = of_cdf[n] + pdf * derivative / factorial;
        }
        // at both ends the functions are constant from the last node on: 0 and 1
        for (int which = 0; which < 2; ++which) {
            const double* c = which == 0 ? of_cdf : of_slope;
            float* out = which == 0 ? tables.cdf[i] : tables.slope[i];
            if (i == 0 || i == kGeluNodes - 1) {
                out[0] = i == 0 ? 0.0f : 1.0f;
                out[1] = out[2] = out[3] = 0.0f;
            } else {
                out[0] = static_cast<float>(c[0] - c[4] * r4 / 8.0);
                out[1] = static_cast<float>(c[1] - c[5] * r4 * 5.0 / 16.0);
                out[2] = static_cast<float>(c[2] + c[4] * r2);
                out[3] = static_cast<float>(c[3] + c[5] * r2 * 5.0 / 4.0);
            }
        }
        // on to the next node
        double integral = 0.0, ratio = 0.0, power = 1.0;
        for (int n = 0; n < 18; ++n) {
            ratio += p[n] * power;                   // phi(x + h)/phi(x)
            power *= h / (n + 1);
            integral += p[n] * power;                // (Phi(x + h) - Phi(x))/phi(x)
        }
        cdf += pdf * integral;
        pdf *= ratio;
    }
    return tables;
}

static __device__ const GeluTables kGeluTables = make_gelu_tables();

template <bool SLOPE, int BLOCK>
__device__ __forceinline__ void fill_gelu_table(f32x4* table, int tid) {
    const f32x4* from = reinterpret_cast<const f32x4*>(SLOPE ? kGeluTables.slope : kGeluTables.cdf);
#pragma unroll
    for (int i = 0; i < (kGeluNodes + BLOCK - 1) / BLOCK; ++i) {
        const int at = tid + i * BLOCK;
        if (at < kGeluNodes) table[at] = from[at];
    }
    __syncthreads();
}

// A value's place in the table: the cubic of the nearest node, the value within the ends, and the distance to the node.  A value beyond
// the ends is moved to them and a NaN to the lower one, so that the index is in range for any value.
struct GeluPlace {
    f32x4 c;
    float s, d;
};
template <bool SLOPE>
__device__ __forceinline__ GeluPlace gelu_place(float x, const f32x4* table) {
    constexpr float kRound = 12582912.0f;                    // 1.5 * 2^23: the sum's low bits are the nearest whole number
    const float s = __builtin_fminf(__builtin_fmaxf(x, static_cast<float>(kGeluLow)), static_cast<float>(kGeluHigh));
    const float u = __builtin_fmaf(s, static_cast<float>(kGeluPerUnit), kRound);
    const uint32_t node = as_u32(u) - (0x4B400000u + static_cast<uint32_t>(kGeluLow * kGeluPerUnit));
    return GeluPlace{table[node], s, __builtin_fmaf(u - kRound, -1.0f / kGeluPerUnit, SLOPE ? x : s)};
}
// GeLU is x*c0 + s*(Phi - c0): two roundings of the size of the result, those of c0 and of the sum; NaN at NaN and at -inf, inf at inf.
// The slope takes the distance to the node from x itself, times 0 beyond the ends: NaN at NaN and, as x*phi(x) is in the
// reference (gelu.py:77-80), at both infinities.
template <bool SLOPE>
__device__ __forceinline__ float gelu_at(float x, const GeluPlace& p) {
    const float rest = __builtin_fmaf(p.d, __builtin_fmaf(p.d, p.c[3], p.c[2]), p.c[1]);
    return SLOPE ? __builtin_fmaf(p.d, rest, p.c[0]) : __builtin_fmaf(x, p.c[0], p.s * (p.d * rest));
}

// GeLU(x), or GeLU'(x) with SLOPE.
template <bool SLOPE>
__device__ __forceinline__ float gelu_by_table(float x, const f32x4* table) {
    return gelu_at<SLOPE>(x, gelu_place<SLOPE>(x, table));
}

// The same for the N values of a vector, in place.  With BATCH all N reads of the table are under way before the first is used (4
// registers each); the compiler by itself, saving registers, waits for each.
template <bool SLOPE, bool BATCH, int N>
__device__ __forceinline__ void gelu_by_table(float (&z)[N], const f32x4* table) {
    GeluPlace p[N];
#pragma unroll
    for (int e = 0; e < N; ++e) p[e] = gelu_place<SLOPE>(z[e], table);
    if constexpr (BATCH) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < N; ++e) z[e] = gelu_at<SLOPE>(z[e], p[e]);
}

}  // namespace thn
