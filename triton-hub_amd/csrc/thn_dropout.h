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
//  * a dropped element is selected before it is scaled (0 scales to +0), which leaves no branch;
//  * 16-bit values are scaled by one multiplication where dropout_scale() finds a factor, instead of 3 instructions;
//  * a forward that keeps its decisions shifts each into its word with the comparison's own mask as the carry of one
//    addition, and takes the element's part of the first product as the addend of that multiplication.
// bfloat16 16384 x 4096 (134 MB in, 134 MB out): a forward that keeps its decisions takes 88.6 us under the profiler (41.8 vector
// instructions per element, issuing in 96 % of the cycles in which a compute unit is busy; with 45.4 instructions, registers for
// 7 of the 8 workgroups per compute unit that are launched and no decision before the first vectors had arrived 97.7); with
// its backward 134.0 -> 127.3 among others.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <string.h>
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
    uint32_t* mask;        // dropout_masked_kernel: see there
    float scale;           // dropout_scale(1 - p, type): 0 where the product would not round like the quotient
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

// A float32 r whose product x * r, rounded to float32 and then to a 16-bit type, is for every x of that type what the
// quotient x / keep rounded the same way is; 0 if none of the three next to 1 / keep is one.  The roundings depend on
// x's significand alone, so every one of them is tried: the normal numbers at one exponent (results only grow, keep being
// at most 1: they stay normal, and infinity starts at the rounding boundary of the largest), the subnormal ones in units of
// the smallest, where bfloat16 results below 128 units have been rounded to float32's subnormal grid of 2^-16 units first.
// Found for 92 of the p = 0.01, 0.02 ... 0.99 with bfloat16, for 86 with float16.
// (Loops without an exit, which the compiler makes vector loops of: 1.6 us for float16 and 0.4 for bfloat16 on the host, in the mean
// over those p; one value at a time took 6.1 and 1.4.)
template <int kBits, bool kCoarse>      // significand bits with the hidden one; float32's own subnormal grid matters
inline bool products_round_alike(float keep, float r) {
    constexpr int kHidden = 1 << (kBits - 1), kDrop = 24 - kBits;
    const auto narrow = [](float v) {
        uint32_t u;
        memcpy(&u, &v, 4);
        return static_cast<int32_t>((u + (1u << (kDrop - 1)) - 1u + (u >> kDrop & 1u)) >> kDrop);
    };
    int32_t differ = 0;
    for (int m = kHidden; m < 2 * kHidden; ++m) {
        const float x = static_cast<float>(m);
        differ |= narrow(x / keep) ^ narrow(x * r);
    }
    if (differ != 0) return false;
    // (a float32 result from kHidden units on is a normal number; below it goes to whole units, to even)
    const auto narrow_subnormal = [&](float v) { return narrow(v >= static_cast<float>(kHidden) ? v : (v + 0x1p23f) - 0x1p23f); };
    const auto coarse = [](double exact) { return static_cast<float>(((exact * 65536.0 + 0x1p52) - 0x1p52) / 65536.0); };     // (1 / keep is at most 2^24)
    for (int m = 1; m < kHidden; ++m) {
        const float x = static_cast<float>(m);
        float quotient = x / keep, product = x * r;
        if (kCoarse && quotient < static_cast<float>(kHidden)) quotient = coarse(static_cast<double>(m) / keep);
        if (kCoarse && product < static_cast<float>(kHidden)) product = coarse(static_cast<double>(m) * r);
        differ |= narrow_subnormal(quotient) ^ narrow_subnormal(product);
    }
    return differ == 0;
}
inline float dropout_scale(float keep, int dtype) {
    if (!(keep > 0.0f) || (dtype != kF16 && dtype != kBF16)) return 0.0f;
    const float r = 1.0f / keep;
    const float candidates[3] = {r, nextafterf(r, 0.0f), nextafterf(r, 2.0f * r)};
    for (const float c : candidates) {
        if (dtype == kBF16 ? products_round_alike<8, true>(keep, c) : products_round_alike<11, false>(keep, c)) return c;
    }
    return 0.0f;
}

// The first Philox word of counter (c0, c1, 0, 0), the product of c0 and the first multiplier being given; c1 = 0 is taken
// as given unless kWide.
constexpr uint32_t kPhiloxM0 = 0xD2511F53u;
template <bool kWide>
__device__ __forceinline__ uint32_t philox_first_word(uint64_t first_product, uint32_t c1_in, uint32_t k0, uint32_t k1) {
    constexpr uint32_t kM0 = kPhiloxM0, kM1 = 0xCD9E8D57u, kW0 = 0x9E3779B9u, kW1 = 0xBB67AE85u;
    const auto product = [](uint32_t m, uint32_t c) { return static_cast<uint64_t>(m) * c; };
    const auto high = [](uint64_t p) { return static_cast<uint32_t>(p >> 32); };
    const auto low = [](uint64_t p) { return static_cast<uint32_t>(p); };
    const auto xor3 = [](uint32_t a, uint32_t b, uint32_t c) { return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96); };
    // round 1: the third and fourth counter words are 0
    uint64_t pa = first_product, pb;
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
    const uint32_t w = philox_first_word<kWide>(static_cast<uint64_t>(kPhiloxM0) * static_cast<uint32_t>(o), static_cast<uint32_t>(o >> 32), a.key_lo, a.key_hi);
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
constexpr int kMaskedVecs = 4;                   // vectors per thread and step of dropout_masked_kernel
constexpr int64_t kMaskedMost = int64_t{1} << 32;  // elements at most
constexpr uint32_t kDropAll = 0x80000000u;      // the threshold at which no element is kept (2 T does not fit a word there)

// What a step of the kernels does with one element: the value it stores, `dropped` being the decision.  The float32 value is
// selected before it is widened (the asm keeps the compiler from selecting both halves of the float64 instead).
__device__ __forceinline__ float dropout_value(float x, bool dropped, const KeepDivisor& keep) {
    float kept = dropped ? 0.0f : x;
    asm("" : "+v"(kept));
    return keep_div(kept, keep);
}
__device__ __forceinline__ double dropout_value(double x, bool dropped, const KeepDivisor& keep) { return keep_div(dropped ? 0.0 : x, keep); }
template <bool kProduct, typename C> __device__ __forceinline__ C dropout_value(C x, bool dropped, const KeepDivisor& keep, float scale) {
    if constexpr (kProduct) return (dropped ? 0.0f : x) * scale;
    else return dropout_value(x, dropped, keep);
}

// word = 2^VEC * word + the decisions of a vector, whose lanes' bits the scalar masks hold: an addition with carry each.  A vector
// instruction needs two wait states behind the comparison that writes the scalar mask it reads; the compiler, which
// sees to that for its own instructions, does not look into an asm block, so the block begins with them.  The masks go
// through it: what reads them afterwards reads them behind those wait states too.
template <int VEC> __device__ __forceinline__ void shift_in_decisions(uint32_t& word, uint64_t (&drop)[VEC]) {
    static_assert(VEC == 2 || VEC == 4 || VEC == 8);
#define THN_SHIFT_IN(MASK) "\n\tv_addc_co_u32_e64 %0, vcc, %0, %0, %" #MASK
    if constexpr (VEC == 2) {
        asm("s_nop 1" THN_SHIFT_IN(1) THN_SHIFT_IN(2) : "+v"(word), "+s"(drop[0]), "+s"(drop[1]) : : "vcc");
    } else if constexpr (VEC == 4) {
        asm("s_nop 1" THN_SHIFT_IN(1) THN_SHIFT_IN(2) THN_SHIFT_IN(3) THN_SHIFT_IN(4)
            : "+v"(word), "+s"(drop[0]), "+s"(drop[1]), "+s"(drop[2]), "+s"(drop[3]) : : "vcc");
    } else {
        asm("s_nop 1" THN_SHIFT_IN(1) THN_SHIFT_IN(2) THN_SHIFT_IN(3) THN_SHIFT_IN(4) THN_SHIFT_IN(5) THN_SHIFT_IN(6) THN_SHIFT_IN(7) THN_SHIFT_IN(8)
            : "+v"(word), "+s"(drop[0]), "+s"(drop[1]), "+s"(drop[2]), "+s"(drop[3]), "+s"(drop[4]), "+s"(drop[5]), "+s"(drop[6]), "+s"(drop[7]) : : "vcc");
    }
#undef THN_SHIFT_IN
}

// the tail that does not fill a vector
template <typename T, bool kWide>
__device__ __forceinline__ void dropout_tail(const DropoutArgs& a, const KeepDivisor& keep, bool all) {
    using C = typename std::conditional<T::kBytes == 8, double, float>::type;
    const int64_t i = a.total_vecs * T::VEC + threadIdx.x;
    if (blockIdx.x == 0 && i < a.total_elems) {
        const C x = load_elem<T, C>(a.x, i);
        store_elem<T, C>(a.out, i, all || is_dropped<kWide>(a.first_offset + i, a) ? C(0) : keep_div(x, keep));
    }
}

template <typename T, bool kWide, bool kProduct>
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
        for (int e = 0; e < VEC; ++e) of[e] = dropout_value<kProduct>(xf[e], is_dropped<kWide>(e0 + e, a), keep, a.scale);
        st128u(a.out + v * 16, pack_as<T, C>(of));
    }
    dropout_tail<T, kWide>(a, keep, all);
}

// A forward that keeps its decisions (kRead = false) and the backward that reads them instead of drawing them again.  A
// workgroup takes pieces of 256 x 4 vectors, thread t of it vectors t, t + 256, t + 512 and t + 768 of a piece; word t of the
// piece's 256 words of mask holds their decisions, a byte per vector with the first in the highest byte, the first element of a
// vector in the highest of the byte's VEC low bits.  (One byte per thread and vector cost the forward 14 us.)  The next piece is
// requested before the present one is used, as act_flat_kernel does (kAhead), except by the forward over 16-bit values, whose 8 Philox
// blocks per vector are arithmetic enough to wait on: it requests each vector of the next piece when that of the present one is
// stored (16 registers fewer: 8 workgroups per compute unit).  float32 and float64, with 4 and 2 blocks per vector, lose by that
// (forward of 2^24 float64 49.5 us against 48.4, 2^23 float32 15.3 against 14.7).  Slots past the end repeat the last vector, so
// that no branch stands around a load or a store.  The threshold is below kDropAll (p < 1 in float32), the offsets of the
// elements start at 0 and fit 32 bits.
// bfloat16 16384 x 4096 under the profiler: forward 88.6 us, backward 45.2, which is what two plain streams take (80 drawn again).
template <typename T, bool kRead, bool kProduct>
__global__ void __launch_bounds__(kDropoutBlock, kRead || T::kBytes > 2 ? 1 : 8) dropout_masked_kernel(const DropoutArgs a) {
    using C = typename std::conditional<T::kBytes == 8, double, float>::type;
    constexpr int VEC = T::VEC, U = kMaskedVecs;
    constexpr bool kAhead = kRead || T::kBytes > 2;
    const KeepDivisor keep = make_keep_divisor(1.0f - a.p);
    const uint32_t pieces = static_cast<uint32_t>((a.total_vecs + kDropoutBlock * U - 1) / (kDropoutBlock * U));
    const uint32_t last = static_cast<uint32_t>(a.total_vecs - 1);
    const auto place = [&](uint32_t piece, int u) -> uint32_t {
        const uint32_t v = piece * (kDropoutBlock * U) + u * kDropoutBlock + threadIdx.x;
        return v < last ? v : last;
    };
    const auto load = [&](uint32_t v) { return ld128u(a.x + static_cast<uint64_t>(v) * 16); };
    // The first product of element e of a vector: the part of e is the addend of the multiplication.  (Kept from the compiler,
    // which would add e to the offset first, one instruction more per element; an instruction reads one scalar operand.)
    uint32_t m0 = kPhiloxM0;
    uint64_t of_element[VEC];
    asm("" : "+v"(m0));
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
        of_element[e] = static_cast<uint64_t>(kPhiloxM0) * e;
        asm("" : "+s"(of_element[e]));
    }
    if (blockIdx.x < pieces) {
        u32x4 cur[U], nxt[kAhead ? U : 1];
        uint32_t word = 0u, next_word = 0u;
#pragma unroll
        for (int u = 0; u < U; ++u) cur[u] = load(place(blockIdx.x, u));
        if constexpr (kRead) word = a.mask[static_cast<uint64_t>(blockIdx.x * kDropoutBlock + threadIdx.x)];
        if constexpr (kAhead) drain_vector_memory(cur);
        for (uint32_t piece = blockIdx.x; piece < pieces; piece += gridDim.x) {
            const uint32_t next = piece + gridDim.x < pieces ? piece + gridDim.x : piece;
            if constexpr (kAhead) {
#pragma unroll
                for (int u = 0; u < U; ++u) nxt[u] = load(place(next, u));
            }
            if constexpr (kRead) next_word = a.mask[static_cast<uint64_t>(next * kDropoutBlock + threadIdx.x)];
            else word = 0u;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t v = place(piece, u);
                C xf[VEC], of[VEC];
                if constexpr (kRead) {
                    unpack_as<T>(cur[u], xf);
#pragma unroll
                    for (int e = 0; e < VEC; ++e) {
                        const bool dropped = (word >> (8 * (U - 1 - u) + VEC - 1 - e) & 1u) != 0u;
                        of[e] = dropout_value<kProduct>(xf[e], dropped, keep, a.scale);
                    }
                } else {
                    // the decisions first: nothing waits for the vector before they are made
                    uint64_t drop[VEC];
                    if constexpr (VEC < 8) word <<= 8 - VEC;
#pragma unroll
                    for (int e = 0; e < VEC; ++e) {
                        const uint64_t first = static_cast<uint64_t>(m0) * (v * VEC) + of_element[e];
                        const uint32_t w = philox_first_word<false>(first, 0u, a.key_lo, a.key_hi);
                        drop[e] = __builtin_amdgcn_uicmp(w + a.threshold, 2u * a.threshold, 36);
                    }
                    shift_in_decisions(word, drop);
                    pin_loaded(cur[u]);
                    unpack_as<T>(cur[u], xf);
                    // (the mask as the condition: from the comparison itself the compiler would make a second one, inverted)
#pragma unroll
                    for (int e = 0; e < VEC; ++e) of[e] = dropout_value<kProduct>(xf[e], __builtin_amdgcn_inverse_ballot_w64(drop[e]), keep, a.scale);
                }
                st128u(a.out + static_cast<uint64_t>(v) * 16, pack_as<T, C>(of));
                if constexpr (!kAhead) cur[u] = load(place(next, u));
            }
            if constexpr (!kRead) a.mask[static_cast<uint64_t>(piece * kDropoutBlock + threadIdx.x)] = word;
            if constexpr (kAhead) {
#pragma unroll
                for (int u = 0; u < U; ++u) cur[u] = nxt[u];
            }
            if constexpr (kRead) word = next_word;
        }
    }
    dropout_tail<T, false>(a, keep, false);
}

enum class DropoutMask { kNone, kWrite, kRead };

int launch_dropout(int dtype, DropoutMask mode, const DropoutArgs& a, int grid, hipStream_t st);

}  // namespace thn
