// Dropout over a contiguous tensor: y[i] = rand(seed, i) < p ? 0 : x[i] / (1 - p), with rand the uniform float32 that
// Triton's tl.rand(seed, i) returns, so that a seed gives the mask it gives in the reference
// (TritonHub/Layers/dropout.py:12-23; the backward, :56-67, is the same function of the upstream gradient).
//
// tl.rand: the first output word of Philox-4x32 with 10 rounds on counter (i mod 2^32, i div 2^32, 0, 0) and key
// (seed mod 2^32, seed div 2^32), read as int32 v, folded to v < 0 ? -v - 1 : v, converted to float32 and multiplied
// by 4.6566127342e-10.  Every element needs a Philox block of its own: the kernel is bound by integer arithmetic, not
// by memory (two plain streams of a bfloat16 16384 x 4096 tensor take 44 us), so it is written for the number of vector
// instructions per element:
//  * a round's `hi ^ counter ^ key` is one v_bitop3_b32 (truth table 0x96), not two v_xor_b32;
//  * the zero counter words and the words that the first output word does not depend on drop out of the first two and
//    the last two rounds: 17 multiplications and 17 exclusive-ors for offsets below 2^32 (kWide = false), where the
//    second counter word is zero too and half of the second round is the same for every element;
//  * float32(fold(v)) * 4.6566127342e-10 < p is monotone in fold(v), so the host turns p into the number T of folded
//    words that are dropped (dropout_threshold) and the test is one addition and one unsigned comparison: v lies in
//    [-T, T - 1] exactly if uint32(v + T) < 2 T;
//  * a dropped element is selected before it is scaled (0 scales to +0), which leaves no branch.
// Issue costs measured for one wave (cycles): v_mad_u64_u32 / v_mul_hi_u32 4.2, v_bitop3_b32 and v_xor_b32 2.5, v_cmp_u32 4.2,
// v_mul_f64 and the float64 conversions 4.2-4.5.  bfloat16 16384 x 4096, one launch (134 MB in, 134 MB out): 113 -> 86.5 us.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

#include "thn_device.h"

namespace thn {

struct DropoutArgs {
    const char* x;
    char* out;
    int64_t total_vecs;    // whole 16-byte vectors
    int64_t total_elems;
    int64_t first_offset;  // offset of element 0 (0 for a whole tensor)
    float p;
    uint32_t key_lo, key_hi;
    uint32_t threshold;    // dropout_threshold(p)
};

constexpr float kDropoutScale = 4.6566127342e-10f;

// How many of the folded words 0 .. 2^31 - 1 give a uniform value below p: they are the first ones.
inline uint32_t dropout_threshold(float p) {
    uint32_t low = 0u, high = 0x80000000u;
    while (low < high) {
        const uint32_t mid = low + (high - low) / 2u;
        if (static_cast<float>(static_cast<int32_t>(mid)) * kDropoutScale < p) low = mid + 1u;
        else high = mid;
    }
    return low;
}

// The first Philox word of counter (c0, c1, 0, 0); c1 = 0 is taken as given unless kWide.
template <bool kWide>
__device__ __forceinline__ uint32_t philox_first_word(uint32_t i, uint32_t c1_in, uint32_t k0, uint32_t k1) {
    constexpr uint32_t kM0 = 0xD2511F53u, kM1 = 0xCD9E8D57u, kW0 = 0x9E3779B9u, kW1 = 0xBB67AE85u;
    const auto product = [](uint32_t m, uint32_t c) { return static_cast<uint64_t>(m) * c; };
    const auto high = [](uint64_t p) { return static_cast<uint32_t>(p >> 32); };
    const auto low = [](uint64_t p) { return static_cast<uint32_t>(p); };
    const auto xor3 = [](uint32_t a, uint32_t b, uint32_t c) { return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96); };
    // round 1: the third and fourth counter words are 0
    uint64_t pa = product(kM0, i), pb;
    uint32_t c0 = kWide ? c1_in ^ k0 : k0, c1 = 0u, c2 = high(pa) ^ k1, c3 = low(pa);
    k0 += kW0;
    k1 += kW1;
    // round 2: c1 is 0 (and c0 the same for every element unless kWide)
    pa = product(kM0, c0);
    pb = product(kM1, c2);
    c0 = high(pb) ^ k0;
    c1 = low(pb);
    c2 = kWide ? xor3(high(pa), c3, k1) : c3 ^ (high(pa) ^ k1);
    c3 = low(pa);
    k0 += kW0;
    k1 += kW1;
    // round 3: c3 is the same for every element unless kWide
    pa = product(kM0, c0);
    pb = product(kM1, c2);
    c0 = xor3(high(pb), c1, k0);
    c1 = low(pb);
    c2 = kWide ? xor3(high(pa), c3, k1) : high(pa) ^ (c3 ^ k1);
    c3 = low(pa);
#pragma unroll
    for (int round = 4; round <= 8; ++round) {
        k0 += kW0;
        k1 += kW1;
        pa = product(kM0, c0);
        pb = product(kM1, c2);
        c0 = xor3(high(pb), c1, k0);
        c2 = xor3(high(pa), c3, k1);
        c1 = low(pb);
        c3 = low(pa);
    }
    // rounds 9 and 10: only what the first word of the last one needs
    k0 += kW0;
    k1 += kW1;
    pa = product(kM0, c0);
    pb = product(kM1, c2);
    c2 = xor3(high(pa), c3, k1);
    c1 = low(pb);
    k0 += kW0;
    return xor3(high(product(kM1, c2)), c1, k0);
}

template <bool kWide>
__device__ __forceinline__ bool is_dropped(int64_t offset, const DropoutArgs& a) {
    const uint64_t o = static_cast<uint64_t>(offset);
    const uint32_t w = philox_first_word<kWide>(static_cast<uint32_t>(o), static_cast<uint32_t>(o >> 32), a.key_lo, a.key_hi);
    return w + a.threshold < 2u * a.threshold;
}

// x / keep for a float32 divisor shared by all elements, correctly rounded like the division it replaces: the
// float64 product of x and the float64 reciprocal of keep is within 2^-52 of the exact quotient, and a quotient of two
// float32 values is never closer than 2^-49 (relative) to a point where float32 rounding changes direction, so
// rounding the product to float32 gives the same value as rounding the quotient itself (infinities, NaN, signed
// zeros, overflow and subnormal results included).  3 instructions per element instead of the 11 of a division.
struct KeepDivisor {
    double rk64;     // float32 storage types
    double keep64;   // float64 storage
};
__device__ __forceinline__ KeepDivisor make_keep_divisor(float keep) {
    return KeepDivisor{1.0 / static_cast<double>(keep), static_cast<double>(keep)};
}
__device__ __forceinline__ float keep_div(float x, const KeepDivisor& d) {
    float q = static_cast<float>(static_cast<double>(x) * d.rk64);
    asm("" : "+v"(q));      // rounded to float32 here: the compiler would otherwise round the product to a 16-bit type at once
    return q;
}
__device__ __forceinline__ double keep_div(double x, const KeepDivisor& d) { return x / d.keep64; }

constexpr int kDropoutBlock = 256;
constexpr uint32_t kDropAll = 0x80000000u;      // the threshold at which no element is kept (2 T does not fit a word there)

template <typename T, bool kWide>
__global__ void __launch_bounds__(kDropoutBlock) dropout_flat_kernel(const DropoutArgs a) {
    using C = typename std::conditional<T::kBytes == 8, double, float>::type;
    constexpr int VEC = T::VEC;
    const KeepDivisor keep = make_keep_divisor(1.0f - a.p);        // float32 difference, as the reference's `1 - p`
    const int64_t step = static_cast<int64_t>(gridDim.x) * kDropoutBlock;
    const bool all = a.threshold == kDropAll;
    for (int64_t v = static_cast<int64_t>(blockIdx.x) * kDropoutBlock + threadIdx.x; v < a.total_vecs; v += step) {
        if (all) {
            st128u(a.out + v * 16, u32x4{0u, 0u, 0u, 0u});
            continue;
        }
        const u32x4 raw = ld128u(a.x + v * 16);
        C xf[VEC], of[VEC];
        unpack_as<T>(raw, xf);
        const int64_t e0 = a.first_offset + v * VEC;
#pragma unroll
        for (int e = 0; e < VEC; ++e) of[e] = keep_div(is_dropped<kWide>(e0 + e, a) ? C(0) : xf[e], keep);
        st128u(a.out + v * 16, pack_as<T, C>(of));
    }
    // the tail that does not fill a vector
    const int64_t i = a.total_vecs * VEC + threadIdx.x;
    if (blockIdx.x == 0 && i < a.total_elems) {
        const C x = load_elem<T, C>(a.x, i);
        store_elem<T, C>(a.out, i, all || is_dropped<kWide>(a.first_offset + i, a) ? C(0) : keep_div(x, keep));
    }
}

int launch_dropout(int dtype, const DropoutArgs& a, int grid, hipStream_t st);

}  // namespace thn
