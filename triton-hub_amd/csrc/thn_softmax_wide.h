// Softmax / Softmin / LogSoftmax over rows wider than 64 KiB that one compute unit can still hold in its registers
// (up to 384 KiB: K vectors of 16 bytes in each of 1024 threads), in 16- and 32-bit storage: every tensor is read once.
//
// The looping kernels (thn_softmax.h) walk such a row twice, the second time from the caches: their forward moves 3 and their
// backward 5 tensors through the compute units where a register-resident row moves 2 and 3.  One workgroup fills a compute unit; while it writes vector k of a row it
// requests vector k of its next row into the same registers, so that only the reductions between the passes leave
// the unit without requests, and the units are in different phases.
//
// Measured (looping -> registers, us): log-softmax bfloat16 4096 x 128256 forward 439 -> 394, backward 587 -> 580, both
// 1024 -> 975; softmax backward 721 -> 587, both 1160 -> 983; log-softmax both directions 512 x 151936 171 -> 149, 2000 x 50257
// 216 -> 198, float32 512 x 96000 203 -> 183.  Tensors of 1 GiB stream at 5.3 (forward) and 5.4 TB/s (backward), each byte fetched
// and written once (FETCH_SIZE, WRITE_SIZE), where a bare copy loop reaches 6.15 and a loop with two reads 6.2: between the
// last request of a row and the first of the next lie two reductions over the whole workgroup (backward: one), in which the
// only workgroup of the compute unit asks for nothing.  2, 4 or 8 vectors of lag and 1, 2 or 4 of y ahead stay within 2 % of each
// other.  Which rows and row counts run here: softmax_wide_vecs() in thn_api.hip.
//
// Rows may start at any element: the vectors are those on 16-byte boundaries, and the up to VEC - 1 elements in front of
// and behind them go to one lane each ("edge" elements).  The launcher takes these kernels when all streams sit at the same
// offset from such a boundary in every row.  All accesses are buffer instructions, whose bounds are the row's: a slot past
// the row's end loads 0 and stores nothing, and the row behind the last one is a descriptor of 0 bytes, without a branch.
#pragma once

#include "thn_dispatch.h"
#include "thn_softmax.h"

namespace thn {

constexpr int kWideBlock = 1024;

using rsrc_t = __amdgpu_buffer_rsrc_t;
constexpr int kBufferFlags = 0x00020000;       // raw buffer, 32-bit data format
constexpr int kNonTemporal = 2;                // the nt bit of the instruction's cache policy
constexpr int kOutOfBounds = 0x7ffffff0;

// One row of a stream: its whole vectors, and the row as elements (for the edge elements).
template <typename T> struct WideRow {
    rsrc_t vecs, elems;
    int n_vecs;
    __device__ __forceinline__ WideRow(const char* base, int64_t stride_bytes, int64_t row, int n_cols, bool valid) {
        char* p = const_cast<char*>(base) + row * stride_bytes;
        const int head = static_cast<int>((16u - static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p) & 15u)) & 15u) / T::kBytes;
        n_vecs = (n_cols - head) / T::VEC;
        vecs = __builtin_amdgcn_make_buffer_rsrc(p + head * T::kBytes, 0, valid ? n_vecs * 16 : 0, kBufferFlags);
        elems = __builtin_amdgcn_make_buffer_rsrc(p, 0, valid ? n_cols * T::kBytes : 0, kBufferFlags);
    }
    // Byte offset of the edge element of thread t, or an offset past the row: the elements in front of the vectors
    // belong to the first wave, those behind them to the second.
    __device__ __forceinline__ static int edge_offset(const char* base, int64_t stride_bytes, int64_t row, int n_cols, int t) {
        const uintptr_t p = reinterpret_cast<uintptr_t>(base) + static_cast<uintptr_t>(row * stride_bytes);
        const int head = static_cast<int>((16u - static_cast<uint32_t>(p & 15u)) & 15u) / T::kBytes;
        const int behind = head + (n_cols - head) / T::VEC * T::VEC;
        int c = t < 64 ? (t < head ? t : n_cols) : behind + t - 64;
        return c < n_cols ? c * T::kBytes : kOutOfBounds;
    }
    template <int AUX>
    __device__ __forceinline__ u32x4 load(int offset) const {
        return __builtin_amdgcn_raw_buffer_load_b128(vecs, offset, 0, AUX);
    }
    __device__ __forceinline__ void store(int offset, u32x4 v) const {
        __builtin_amdgcn_raw_buffer_store_b128(v, vecs, offset, 0, kNonTemporal);
    }
    __device__ __forceinline__ uint32_t load_edge(int offset) const {       // the raw bits
        if constexpr (T::kBytes == 2) return __builtin_amdgcn_raw_buffer_load_b16(elems, offset, 0, 0);
        else return __builtin_amdgcn_raw_buffer_load_b32(elems, offset, 0, 0);
    }
    __device__ __forceinline__ void store_edge(int offset, float f) const {
        if constexpr (T::kBytes == 2) {
            typename T::bits_t b;
            T::store1(&b, 0, f);
            __builtin_amdgcn_raw_buffer_store_b16(b, elems, offset, 0, 0);
        } else {
            __builtin_amdgcn_raw_buffer_store_b32(as_u32(f), elems, offset, 0, 0);
        }
    }
    __device__ __forceinline__ static float widen(uint32_t bits) { return T::widen(static_cast<typename T::bits_t>(bits)); }
};

// fn(integral_constant<int, I>) for I = FROM, FROM + STEP, ... below TO.
template <int FROM, int TO, int STEP, typename Fn> __device__ __forceinline__ void static_for(Fn&& fn) {
    if constexpr (FROM < TO) {
        fn(std::integral_constant<int, FROM>{});
        static_for<FROM + STEP, TO, STEP>(fn);
    }
}

// Slots between the request of a vector of the next row and its use in that row's sums, half a row: with fewer the
// kernel waits for memory, with more the sums of the slots that are left over hold up the next row.
template <int K> constexpr int kWideLag = K / 2;

// Forward.  The sums of a row (a running maximum per thread and sum(exp(x - maximum)) in float64, rescaled once per kGroup
// vectors) are taken as its vectors arrive, while the row before it is written; y comes from the same registers.
// KFULL: slots below it lie inside every row.
template <typename T, bool LOG, int K, int KFULL>
__global__ void __launch_bounds__(kWideBlock) softmax_fwd_wide_kernel(const SoftmaxFwdArgs a) {
    constexpr int VEC = T::VEC;
    constexpr int kGroup = 2;
    constexpr int kLag = kWideLag<K>;
    static_assert(K % kGroup == 0 && kLag % kGroup == 0, "whole groups");
    __shared__ float red[RedSmem<kWideBlock, 1, 1>::kFloats];
    __shared__ double red_sum[RedSmem<kWideBlock, 1, 1>::kFloats];
    int phase = 0, phase_sum = 0;
    const int t = threadIdx.x;
    // a wave whose slot lies behind the row computes nothing for it (24 vectors per thread leave no registers for that)
    constexpr bool kSkip = K < 24;
    const int wave = __builtin_amdgcn_readfirstlane(t & ~63);
    const float neg_inf = OpMax::identity<float>();
    // softmin: the sign bits are flipped on the packed vectors
    const uint32_t flip1 = a.sign < 0.0f ? (T::kBytes == 2 ? 0x8000u : 0x80000000u) : 0u;
    const uint32_t flip = T::kBytes == 2 ? flip1 | flip1 << 16 : flip1;

    u32x4 cur[K];
    uint32_t edge;
    float m = neg_inf;
    double acc = 0.0;
    // one group of slots into the sums of its row, which has n_vecs vectors
    const auto absorb = [&](auto first, int n_vecs) {
        constexpr int k0 = decltype(first)::value;
        if (kSkip && k0 >= KFULL && wave + k0 * kWideBlock >= n_vecs) return;
        float f[kGroup][VEC];
        float top = m;
#pragma unroll
        for (int u = 0; u < kGroup; ++u) {
            const int k = k0 + u;
            cur[k] ^= flip;
            pin_loaded(cur[k]);
            T::unpack(cur[k], f[u]);
            const bool in = k < KFULL || t + k * kWideBlock < n_vecs;
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                f[u][e] = in ? f[u][e] : neg_inf;
                top = OpMax::apply(top, f[u][e]);
            }
        }
        const float base = top > neg_inf ? top : 0.0f;      // nothing but -inf so far: exp(-inf - 0) = 0
        acc *= static_cast<double>(exp_c(m - base));
        m = top;
#pragma unroll
        for (int u = 0; u < kGroup; ++u) {
            float part = 0.0f;
#pragma unroll
            for (int e = 0; e < VEC; ++e) part += exp_c(f[u][e] - base);
            acc += static_cast<double>(part);
        }
        asm volatile("" : "+v"(acc));       // group by group: the maxima of all of them first would need every value unpacked
    };
    {
        const WideRow<T> x(a.x, a.x_stride_bytes, blockIdx.x, a.n_cols, true);
        edge = x.load_edge(WideRow<T>::edge_offset(a.x, a.x_stride_bytes, blockIdx.x, a.n_cols, t));
#pragma unroll
        for (int k = 0; k < K; ++k) cur[k] = x.template load<kNonTemporal>((t + k * kWideBlock) * 16);
        static_for<0, K, kGroup>([&](auto k0) { absorb(k0, x.n_vecs); });
    }
    drain_vector_memory();
    for (int64_t row = blockIdx.x; row < a.M; row += gridDim.x) {
        const WideRow<T> y(a.y, a.y_stride_bytes, row, a.n_cols, true);
        const int edge_off = WideRow<T>::edge_offset(a.y, a.y_stride_bytes, row, a.n_cols, t);
        const float fe = edge_off == kOutOfBounds ? neg_inf : WideRow<T>::widen(edge ^ flip1);
        {
            const float top = OpMax::apply(m, fe);
            const float base = top > neg_inf ? top : 0.0f;
            acc = acc * static_cast<double>(exp_c(m - base)) + static_cast<double>(exp_c(fe - base));
            m = top;
        }
        float mx[1] = {m};
        row_allreduce<kWideBlock, 1, 1, OpMax, float>(mx, red, phase, 0, t);
        double s[1] = {acc * static_cast<double>(exp_c(m - (mx[0] > neg_inf ? mx[0] : 0.0f)))};
        row_allreduce<kWideBlock, 1, 1, OpSum, double>(s, red_sum, phase_sum, 0, t);
        const float row_max = mx[0];        // a row of -inf alone: -inf - -inf = NaN
        const float scale = static_cast<float>(LOG ? log(s[0]) : 1.0 / s[0]);

        const int64_t next = row + gridDim.x;
        const WideRow<T> x(a.x, a.x_stride_bytes, next, a.n_cols, next < a.M);
        auto value = [&](float v) {
            const float z = v - row_max;
            if constexpr (LOG) return z - scale;
            else return exp_c(z) * scale;
        };
        y.store_edge(edge_off, value(fe));
        edge = x.load_edge(WideRow<T>::edge_offset(a.x, a.x_stride_bytes, next, a.n_cols, t));
        m = neg_inf;
        acc = 0.0;
        static_for<0, K, 1>([&](auto slot) {
            constexpr int k = decltype(slot)::value;
            const int off = (t + k * kWideBlock) * 16;
            if (!kSkip || k < KFULL || wave + k * kWideBlock < y.n_vecs) {
                float f[VEC];
                pin_loaded(cur[k]);    // packed until here: the values that the sums unpacked are not kept
                T::unpack(cur[k], f);
#pragma unroll
                for (int e = 0; e < VEC; ++e) f[e] = value(f[e]);
                cur[k] = T::pack(f);
            }
            y.store(off, cur[k]);
            cur[k] = x.template load<kNonTemporal>(off);
            if constexpr (k >= kLag && (k - kLag) % kGroup == kGroup - 1) absorb(std::integral_constant<int, k - kLag - (kGroup - 1)>{}, x.n_vecs);
        });
        static_for<K - kLag, K, kGroup>([&](auto k0) { absorb(k0, x.n_vecs); });
    }
}

// Backward.  The row of dy stays in the registers, y is streamed, AHEAD vectors ahead, while dx is written.  The sum of a
// row: log-softmax, of dy, is taken as the vectors arrive, while the row before it is written; softmax, of y * dy, in a pass
// of its own over y, which is then read a second time, from the caches.
template <typename T, bool LOG, int K, int AHEAD>
__global__ void __launch_bounds__(kWideBlock) softmax_bwd_wide_kernel(const SoftmaxBwdArgs a) {
    constexpr int VEC = T::VEC;
    constexpr int kLag = kWideLag<K>;
    static_assert(K % AHEAD == 0, "vector k waits in slot k % AHEAD, also from one pass to the next");
    __shared__ double red_sum[RedSmem<kWideBlock, 1, 1>::kFloats];
    int phase_sum = 0;
    const int t = threadIdx.x;

    u32x4 g[K];
    uint32_t g_edge;
    double acc = 0.0;
    const auto absorb = [&](int k) {
        float gf[VEC];
        pin_loaded(g[k]);
        T::unpack(g[k], gf);
        float part = 0.0f;
#pragma unroll
        for (int e = 0; e < VEC; ++e) part += gf[e];
        acc += static_cast<double>(part);
        asm volatile("" : "+v"(acc));
    };
    {
        const WideRow<T> dy(a.dy, a.dy_stride_bytes, blockIdx.x, a.n_cols, true);
        g_edge = dy.load_edge(WideRow<T>::edge_offset(a.dy, a.dy_stride_bytes, blockIdx.x, a.n_cols, t));
#pragma unroll
        for (int k = 0; k < K; ++k) g[k] = dy.template load<kNonTemporal>((t + k * kWideBlock) * 16);
        if constexpr (LOG) {
#pragma unroll
            for (int k = 0; k < K - kLag; ++k) absorb(k);
        }
    }
    drain_vector_memory(g);
    for (int64_t row = blockIdx.x; row < a.M; row += gridDim.x) {
        const WideRow<T> y(a.y, a.y_stride_bytes, row, a.n_cols, true);
        const int edge_off = WideRow<T>::edge_offset(a.y, a.y_stride_bytes, row, a.n_cols, t);
        u32x4 ahead[AHEAD];
        const uint32_t y_edge = y.load_edge(edge_off);
        const auto request = [&](int k, bool again) {
            const int off = (t + k * kWideBlock) * 16;
            ahead[k % AHEAD] = again ? y.template load<kNonTemporal>(off) : y.template load<0>(off);
        };
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) request(k, LOG);
        if constexpr (LOG) {
#pragma unroll
            for (int k = K - kLag; k < K; ++k) absorb(k);
        } else {
            acc = 0.0;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                float gf[VEC], yf[VEC];
                T::unpack(g[k], gf);
                T::unpack(ahead[k % AHEAD], yf);
                float part = 0.0f;
#pragma unroll
                for (int e = 0; e < VEC; ++e) part = fmaf(yf[e], gf[e], part);
                acc += static_cast<double>(part);
                if (k + AHEAD < K) request(k + AHEAD, false);
                else request(k + AHEAD - K, true);
            }
        }
        const float ye = WideRow<T>::widen(y_edge), ge = WideRow<T>::widen(g_edge);      // past the row: 0
        double s[1] = {acc + static_cast<double>(LOG ? ge : ye * ge)};
        row_allreduce<kWideBlock, 1, 1, OpSum, double>(s, red_sum, phase_sum, 0, t);
        const float total = static_cast<float>(s[0]);

        const int64_t next = row + gridDim.x;
        const WideRow<T> dy(a.dy, a.dy_stride_bytes, next, a.n_cols, next < a.M);
        const WideRow<T> dx(a.dx, a.dx_stride_bytes, row, a.n_cols, true);
        auto value = [&](float yv, float gv) {
            if constexpr (LOG) return fmaf(-exp_c(yv), total, gv) * a.sign;
            else return yv * (gv - total) * a.sign;
        };
        dx.store_edge(edge_off, value(ye, ge));
        g_edge = dy.load_edge(WideRow<T>::edge_offset(a.dy, a.dy_stride_bytes, next, a.n_cols, t));
        acc = 0.0;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int off = (t + k * kWideBlock) * 16;
            float yf[VEC], gf[VEC];
            pin_loaded(g[k]);
            T::unpack(ahead[k % AHEAD], yf);
            T::unpack(g[k], gf);
#pragma unroll
            for (int e = 0; e < VEC; ++e) gf[e] = value(yf[e], gf[e]);
            dx.store(off, T::pack(gf));
            g[k] = dy.template load<kNonTemporal>(off);
            if (k + AHEAD < K) request(k + AHEAD, true);
            if constexpr (LOG) {
                if (k >= kLag) absorb(k - kLag);
            }
        }
    }
}

// (K, slots that lie inside every row, vectors of y ahead): rows of up to K * 1024 vectors and of more than the second
// number * 1024 (the narrowest, of 64 KiB and a few elements, may have one vector less).  With 24 vectors per thread there are registers left for two vectors of y.
#define THN_SM_WIDE_SHAPES(X) X(8, 3, 4) X(12, 8, 4) X(16, 12, 4) X(20, 16, 4) X(24, 20, 2)
constexpr int kWideMaxVecs = 24 * kWideBlock;

#define THN_DECLARE_SOFTMAX_WIDE_LAUNCHERS(NAME)                                                              \
    int launch_softmax_fwd_wide_##NAME(bool is_log, int k, const SoftmaxFwdArgs& a, int grid, hipStream_t st); \
    int launch_softmax_bwd_wide_##NAME(bool is_log, int k, const SoftmaxBwdArgs& a, int grid, hipStream_t st);

THN_DECLARE_SOFTMAX_WIDE_LAUNCHERS(f32)
THN_DECLARE_SOFTMAX_WIDE_LAUNCHERS(f16)
THN_DECLARE_SOFTMAX_WIDE_LAUNCHERS(bf16)

#define THN_SM_WIDE_FWD_CASE(K_, FULL_, AHEAD_)                                                                                  \
    if (k == K_) {                                                                                                       \
        return is_log ? run_kernel<SoftmaxFwdArgs>(softmax_fwd_wide_kernel<T, true, K_, FULL_>, a, grid, kWideBlock, st, nullptr) \
                      : run_kernel<SoftmaxFwdArgs>(softmax_fwd_wide_kernel<T, false, K_, FULL_>, a, grid, kWideBlock, st, nullptr); \
    }
#define THN_SM_WIDE_BWD_CASE(K_, FULL_, AHEAD_)                                                                                  \
    if (k == K_) {                                                                                                       \
        return is_log ? run_kernel<SoftmaxBwdArgs>(softmax_bwd_wide_kernel<T, true, K_, AHEAD_>, a, grid, kWideBlock, st, nullptr) \
                      : run_kernel<SoftmaxBwdArgs>(softmax_bwd_wide_kernel<T, false, K_, AHEAD_>, a, grid, kWideBlock, st, nullptr); \
    }

#define THN_DEFINE_SOFTMAX_WIDE_LAUNCHERS(NAME, TYPE)                                                          \
    int launch_softmax_fwd_wide_##NAME(bool is_log, int k, const SoftmaxFwdArgs& a, int grid, hipStream_t st) { \
        using T = TYPE;                                                                                        \
        THN_SM_WIDE_SHAPES(THN_SM_WIDE_FWD_CASE)                                                               \
        return 1;                                                                                              \
    }                                                                                                          \
    int launch_softmax_bwd_wide_##NAME(bool is_log, int k, const SoftmaxBwdArgs& a, int grid, hipStream_t st) { \
        using T = TYPE;                                                                                        \
        THN_SM_WIDE_SHAPES(THN_SM_WIDE_BWD_CASE)                                                               \
        return 1;                                                                                              \
    }

}  // namespace thn
