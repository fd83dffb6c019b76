// Element-wise activation formulas, forward and derivative, shared by the streaming activation kernels (thn_act.h)
// and by the activation epilogue of the norm kernels (thn_kernels.h).  Each formula cites the line of the
// reference it restates (TritonHub/Activations/*.py).
#pragma once

#include <type_traits>

#include "thn_device.h"

namespace thn {

enum : int {
    kGelu = 0, kGeluTanh = 1, kSilu = 2, kRelu = 3, kLeakyRelu = 4, kRelu6 = 5, kSigmoid = 6, kTanh = 7, kMish = 8,
    kSoftplus = 9, kThreshold = 10, kNumActs = 11
};

__device__ __forceinline__ float log_c(float z) { return __logf(z); }
__device__ __forceinline__ double log_c(double z) { return log(z); }

// The float32 formulas below are written for the instruction budget of a streaming kernel: at 16-bit storage a
// compute unit must finish an element in about 25 instruction slots to keep up with HBM, and the quarter-rate
// v_exp_f32 / v_log_f32 / v_rcp_f32 cost four slots each.  Quotients use the hardware reciprocal (1 ulp) and a
// multiplication instead of an IEEE division (10 slots); every result stays within a few float32 ulp of the exact
// function, far inside the test tolerances.
__device__ __forceinline__ float rcp_fast(float x) { return __builtin_amdgcn_rcpf(x); }

// tanh(u) = sign(u) * (1 - t)/(1 + t) with t = exp(-2|u|): no overflow for any u.
__device__ __forceinline__ float tanh_safe(float u) {
    const float t = __expf(-2.0f * __builtin_fabsf(u));
    const float r = (1.0f - t) * rcp_fast(1.0f + t);
    return u < 0.0f ? -r : r;
}

__device__ __forceinline__ float sigmoid_f(float x) { return rcp_fast(1.0f + __expf(-x)); }

// The gate of the tanh form of GeLU: 0.5*(1 + tanh(u)) with u = sqrt(2/pi)*(x + 0.044715 x^3) (gelu.py:23-26) is the
// logistic function of 2u, 1/(1 + exp(-2u)).  One exponential and one reciprocal, no cancellation for negative x
// (where 1 + tanh(u) loses every digit), no overflow: exp(-2u) = inf gives 0, exp(-2u) = 0 gives 1.
struct GateParts { float gate, e; };            // e = exp(-2u), gate = 1/(1 + e)
__device__ __forceinline__ GateParts gelu_tanh_gate_parts(float x) {
    const float inner = __builtin_fmaf(0.044715f * x * x, x, x);
    GateParts p;
    p.e = __builtin_amdgcn_exp2f(-2.302208198144325f * inner);                     // -2*sqrt(2/pi)*log2(e)
    p.gate = rcp_fast(1.0f + p.e);
    return p;
}
__device__ __forceinline__ float gelu_tanh_gate(float x) { return gelu_tanh_gate_parts(x).gate; }

// GeLU from the normal distribution function Phi(x) = 0.5*(1 + erf(x/sqrt 2)).  With t = 1/(1 + c|x|) in (0, 1] both directions
// take Phi(-|x|) = t*Q(t)*exp(-x^2/2), Q a polynomial of degree 7: branch free, accurate in the negative tail (where
// 1 + erf(..) cancels), a third of the instructions of the library erff.  c is free and sets how fast such a fit converges: at
// the c below degree 7 reaches what took degree 9 and 8 at c = 0.35.  The sign of x rides on t, t_s = 1/(sgn + c*x), and
// step = max(sgn, 0), so that one multiply-add takes the place of a comparison, a subtraction and a selection:
//   Phi(x) = step - t_s*Q*exp(-x^2/2),   GeLU'(x) = Phi(x) + x*phi(x) = step + exp(-x^2/2)*(x/sqrt(2 pi) - t_s*Q).
// The exponential is base 2 (the hardware's v_exp_f32), of a^2 with a = x*sqrt(log2(e)/2).  19 instruction slots per element
// forward and 20 backward (a transcendental counts as 2) instead of 21 and 22.  Float32 against float64, 2-norm: x = 1.5 g + 0.25 with g
// normal 3.29e-8 and 4.26e-8 instead of 3.32e-8 and 4.46e-8, g alone 3.88e-8 and 4.83e-8 instead of 3.98e-8 and 5.14e-8; in bands of
// x the roundings fall differently, up to 0.7 and up to 1.23 times as large ([-4, -3] 4.4e-7 -> 3.1e-7 forward, [-2, -1.5] 1.43e-7 -> 1.62e-7).
//
// |t| is a modifier of the polynomial's multiply-adds, which then have no room for a coefficient and read it from a scalar register.
// LITERALS: |t| in a register of its own, an instruction more, and the coefficients in the instructions.  That is the faster
// one where little else is in flight, without -> with, us: the element-wise forward of 2^23 and 2^24 bfloat16 elements 6.8-7.1 -> 6.3-6.7
// and 12.0 -> 11.3 (2^26 42.6 -> 42.3; before degree 7 6.6, 11.5 and 43.7; float16 9.5 -> 9.5 and 12.4 -> 12.3, before 9.2 and 12.0), 2^22 float64
// elements 10.1 -> 9.8, and the norm forwards off the 128-bit path.  Those on it lose 2-4 % by it, and the backwards spill.  (The norms over 16-bit
// rows go by the tables of thn_gelu_table.h instead; the element-wise kernels gained with 2^26 elements, forward + backward 109 -> 106 us, but lost
// up to 4 % at 2^22 and 2^24, where filling the table counts.)
struct NormalParts {
    float tq, e, step;      // t_s*Q(t), exp(-x^2/2), x < 0 ? 0 : 1
};
template <int DEGREE, bool LITERALS>
__device__ __forceinline__ NormalParts normal_parts(float x, float c, const float (&coefficients)[DEGREE + 1]) {
    const float sgn = __builtin_copysignf(1.0f, x);
    const float t = rcp_fast(__builtin_fmaf(c, x, sgn));
    const float a = x * 0.84932180028801907f;
    float size = __builtin_fabsf(t);
    if constexpr (LITERALS) asm("" : "+v"(size));
    float q = coefficients[DEGREE];
#pragma unroll
    for (int i = DEGREE - 1; i >= 0; --i) q = __builtin_fmaf(q, size, coefficients[i]);
    return NormalParts{t * q, __builtin_amdgcn_exp2f(-a * a), sgn > 0.0f ? sgn : 0.0f};
}

// Minimax fit of the relative error of Phi(-|x|) (x in [0, 13.3], behind which the exponential underflows): 1.24e-7 with c and the
// coefficients as stored.
template <bool LITERALS>
__device__ __forceinline__ float normal_cdf(float x) {
    const NormalParts p = normal_parts<7, LITERALS>(x, 0.3036f, {0.12107304f, 0.12204604f, 0.1020654f, 0.12441437f, -0.044881325f,
                                                                 0.19440602f, -0.15598506f, 0.036861554f});
    return __builtin_fmaf(-p.tq, p.e, p.step);
}

// Minimax fit of the error relative to |x|/sqrt(2 pi) + t*Q, which is what GeLU' is made of: 4.5e-8 as stored.  (c = 0.385 to 0.41
// measure alike; beyond 0.415 the fit is worse than degree 8 at 0.354 was.)
__device__ __forceinline__ float gelu_slope(float x) {
    const NormalParts p = normal_parts<7, false>(x, 0.401f, {0.16005206f, 0.15829173f, 0.14927879f, 0.011608556f, 0.21302079f,
                                                             -0.34127876f, 0.18568613f, -0.036659308f});
    return __builtin_fmaf(p.e, __builtin_fmaf(0.39894228040143267794f, x, -p.tq), p.step);
}

// Mish needs t = tanh(softplus(x)) with softplus(x) = x > 20 ? x : log(1 + e^x) (mish.py:19-22).  With w = e^x and
// n = w*(w + 2):  tanh(log(1 + w)) = n/(n + 2)  and  1 - t^2 = 4*(n + 1)/(n + 2)^2 : one exponential, one
// reciprocal, no cancellation for very negative x (where log(1 + e^x) rounds to 0 in float32).  Above 20 the
// reference's branch gives tanh(x), which is 1 in float32.
struct MishParts { float t, one_minus_t2, sig; };
__device__ __forceinline__ MishParts mish_parts(float x) {
    const float w = __expf(x < 20.0f ? x : 20.0f);
    const float n = w * (w + 2.0f);
    const float r = rcp_fast(n + 2.0f);
    MishParts m;
    const bool big = x > 20.0f;
    m.t = big ? 1.0f : n * r;
    m.one_minus_t2 = big ? 0.0f : 4.0f * (n + 1.0f) * r * r;
    m.sig = big ? 1.0f : w * rcp_fast(1.0f + w);          // sigmoid(x) = w/(1 + w); 1 in float32 above 20
    return m;
}

template <int ACT, typename C, bool LITERALS = false>
__device__ __forceinline__ C act_fwd(C x, C p0, C p1) {
    if constexpr (ACT == kGelu) {
        return x * normal_cdf<LITERALS>(x);                                                  // gelu.py:28
    } else if constexpr (ACT == kGeluTanh) {
        return x * gelu_tanh_gate(x);                                                      // gelu.py:23-26
    } else if constexpr (ACT == kSilu) {
        return x * sigmoid_f(x);                                                           // silu.py:19
    } else if constexpr (ACT == kRelu) {
        return x > C(0) ? x : C(0);                                                        // relu.py:19
    } else if constexpr (ACT == kLeakyRelu) {
        return x > C(0) ? x : p0 * x;                                                      // leaky_relu.py:20
    } else if constexpr (ACT == kRelu6) {
        const C r = x > C(0) ? x : C(0);                                                   // relu6.py:19-20
        return r < C(6) ? r : C(6);
    } else if constexpr (ACT == kSigmoid) {
        return sigmoid_f(x);                                                               // sigmoid.py:19
    } else if constexpr (ACT == kTanh) {
        return tanh_safe(x);                                                               // tanh.py:19-21
    } else if constexpr (ACT == kMish) {
        return x * mish_parts(x).t;                                                        // mish.py:19-23
    } else if constexpr (ACT == kSoftplus) {
        if constexpr (std::is_same<C, float>::value) {                                     // softplus.py:21
            // base-2 hardware exponential and logarithm; the factors log2(e)*beta and ln(2)/beta are the same for every
            // element (two multiplications fewer per element than exp and log of base e)
            const float k = p0 * 1.44269504088896341f, inv = 0.69314718055994531f * rcp_fast(p0);
            return x * p0 > p1 ? x : __builtin_amdgcn_logf(1.0f + __builtin_amdgcn_exp2f(k * x)) * inv;
        } else {
            return x * p0 > p1 ? x : log_c(C(1) + exp_c(p0 * x)) / p0;
        }
    } else {
        return x > p0 ? x : p1;                                                            // threshold.py:20
    }
}

// `s` is the saved tensor: the forward's input, or its output for Sigmoid and Tanh.
template <int ACT, typename C>
__device__ __forceinline__ C act_bwd(C s, C g, C p0, C p1) {
    if constexpr (ACT == kGelu) {
        return g * gelu_slope(s);                                                          // gelu.py:77-80
    } else if constexpr (ACT == kGeluTanh) {
        // gelu.py:71-75 with t = tanh(u) = 2*gate - 1: 0.5*(1 + t) = gate, 0.5*(1 - t^2) = 2*gate*(1 - gate)
        const GateParts p = gelu_tanh_gate_parts(s);
        const float gate = p.gate;
        // 1 - gate = e*gate: taken from whichever side does not cancel (e = inf goes with gate = 0 < 0.5)
        const float slope = gate * (gate < 0.5f ? 1.0f - gate : p.e * gate);   // gate*(1 - gate) = sech^2(u)/4
        const float du2 = __builtin_fmaf(3.0f * 0.044715f * 1.59576912160573071f, s * s, 1.59576912160573071f);   // 2*u'
        const float tail = slope == 0.0f ? 0.0f : s * slope * du2;             // exactly 0 once |s| > ~6: no 0 * inf
        return g * (gate + tail);
    } else if constexpr (ACT == kSilu) {
        const float sg = sigmoid_f(s);                                                     // silu.py:56-57
        return g * (sg * (1.0f + s * (1.0f - sg)));
    } else if constexpr (ACT == kRelu) {
        return s > C(0) ? g : C(0);                                                        // relu.py:56
    } else if constexpr (ACT == kLeakyRelu) {
        return s > C(0) ? g : p0 * g;                                                      // leaky_relu.py:59
    } else if constexpr (ACT == kRelu6) {
        const C r = s > C(0) ? g : C(0);                                                   // relu6.py:57-58
        return s < C(6) ? r : C(0);
    } else if constexpr (ACT == kSigmoid) {
        return g * (s * (1.0f - s));                                                       // sigmoid.py:56
    } else if constexpr (ACT == kTanh) {
        return g * (1.0f - s * s);                                                         // tanh.py:58
    } else if constexpr (ACT == kMish) {
        const MishParts m = mish_parts(s);                                                 // mish.py:60-66
        return g * (m.t + s * m.one_minus_t2 * m.sig);
    } else if constexpr (ACT == kSoftplus) {
        if constexpr (std::is_same<C, float>::value) {                                     // softplus.py:62
            const float k = p0 * -1.44269504088896341f;
            return s * p0 > p1 ? g : g * rcp_fast(1.0f + __builtin_amdgcn_exp2f(k * s));
        } else {
            return s * p0 > p1 ? g : g / (C(1) + exp_c(-p0 * s));
        }
    } else {
        return s > p0 ? g : C(0);                                                          // threshold.py:59
    }
}

}  // namespace thn
