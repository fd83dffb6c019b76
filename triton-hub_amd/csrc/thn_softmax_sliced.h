// Softmax / Softmin / LogSoftmax over few wide rows (more than 64 KiB, 16- and 32-bit storage): a row is cut into slices of 32 KiB,
// one workgroup each, so that the whole chip works on them.  Two launches per direction: the first leaves the sums of every
// slice, the second combines those of its row and writes the slice.
//
// The kernels with a workgroup per row (thn_softmax_wide.h, thn_softmax.h) are bound by what one compute unit moves, about 30 GB/s
// in and out, where there are fewer rows than units, and by a second round for a few rows where there are a few more.  Here the
// input is read twice, the second time mostly from the caches: 3 units of traffic forward and 4 (log-softmax) or 5 backward
// instead of 2 and 3 where a row stays in registers, the walking kernels' own where it does not.
// Forward / backward, us: log-softmax bfloat16 16 x 128256 18.4 / 16.5 -> 7.5 / 7.1, 16 x 240000 31.3 / 33.8 -> 7.8 / 8.2, 60 x 179018 25.5 / 31.7 ->
// 13.1 / 15.4, 300 x 240000 90.4 / 110.6 -> 70.3 / 88.9; float32 64 x 128256 28.1 / 42.3 -> 18.0 / 21.6, 153 x 206289 76.9 / 101.4 -> 63.4 / 81.4,
// 325 x 206289 152 / 214 -> 133 / 171; softmax float32 16 x 227155 40.0 / 39.0 -> 9.2 / 11.7, 290 x 227155 152.8 / 263.4 -> 129.8 / 223.8.
// Slices of 16 KiB are as fast up to 16 rows and 5 % slower from 128 on; slices of 64 KiB 3 % faster for float32 and up to 15 % slower for
// 16-bit rows; writing the slices in the reverse of the order in which they were summed changed nothing.
// Which rows and row counts run here: softmax_slicing() in thn_api.hip.
//
// The sums travel through the output, which is written over afterwards: slice i leaves its record in each slice j of its
// row, as the vector number i of that slice.  So a workgroup finds the records of its whole row inside the one slice that nobody but
// itself writes over, and does so behind a barrier.  No workspace, nothing to clear, nothing shared between calls.
//
// As in thn_softmax_wide.h rows may start at any element, all streams of a row at the same offset from a 16-byte boundary; the elements
// in front of the first and behind the last whole vector belong to the first and the last slice; buffer instructions bound
// every access by its slice, the edge elements by the row.
#pragma once

#include "thn_dispatch.h"
#include "thn_softmax.h"
#include "thn_softmax_wide.h"

namespace thn {

constexpr int kSlicedBlock = 512;
constexpr int kSlicedVecs = 4;           // 16-byte vectors per thread
constexpr int kSlicedMost = 64;          // slices of a row at most: each is combined by one lane of a wave

struct Slicing {
    int slices;        // per row
    int vecs;          // 16-byte vectors per slice (the last may have fewer, but more than kSlicedMost)
};

// Slices of even size for rows of `vecs` vectors, give or take the one that a row which starts off a 16-byte boundary has less.
inline Slicing even_slices(int vecs) {
    const int most = kSlicedBlock * kSlicedVecs, n = (vecs + most - 1) / most;
    return Slicing{n, (vecs + n - 1) / n};
}

// What the slices of a row leave for each other: the maximum and sum(exp(x - maximum)), or the sum of the backward.
struct SliceRecord {
    u32x4 bits;
    __device__ static __forceinline__ u32x4 of(float m, double s) {
        const uint64_t u = __builtin_bit_cast(uint64_t, s);
        return u32x4{static_cast<uint32_t>(u), static_cast<uint32_t>(u >> 32), as_u32(m), 0u};
    }
    __device__ __forceinline__ double sum() const {
        const uint32_t lo = bits[0], hi = bits[1];
        return __builtin_bit_cast(double, static_cast<uint64_t>(hi) << 32 | lo);
    }
    __device__ __forceinline__ float max() const { const uint32_t m = bits[2]; return as_f32(m); }
};

// One slice of a row of one stream.
template <typename T> struct RowSlice {
    rsrc_t vecs, elems;
    int n_vecs;        // of this slice
    int edge;          // byte offset of this thread's edge element in the row
    char* first;       // the row's first whole vector
    __device__ __forceinline__ RowSlice(const char* base, int64_t stride_bytes, int64_t row, int n_cols, const Slicing& s, int slice, int t) {
        char* p = const_cast<char*>(base) + row * stride_bytes;
        const int head = static_cast<int>((16u - static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p) & 15u)) & 15u) / T::kBytes;
        const int whole = (n_cols - head) / T::VEC;
        const int from = slice * s.vecs;
        n_vecs = whole - from < s.vecs ? whole - from : s.vecs;
        first = p + head * T::kBytes;
        vecs = __builtin_amdgcn_make_buffer_rsrc(first + static_cast<int64_t>(from) * 16, 0, n_vecs * 16, kBufferFlags);
        elems = __builtin_amdgcn_make_buffer_rsrc(p, 0, n_cols * T::kBytes, kBufferFlags);
        int c = n_cols;
        if (slice == 0 && t < head) c = t;
        if (slice == s.slices - 1 && t >= 64) c = head + whole * T::VEC + t - 64;
        edge = c < n_cols ? c * T::kBytes : kOutOfBounds;
    }
    template <int AUX> __device__ __forceinline__ u32x4 load(int offset) const {
        return __builtin_amdgcn_raw_buffer_load_b128(vecs, offset, 0, AUX);
    }
    __device__ __forceinline__ void store(int offset, u32x4 v) const {
        __builtin_amdgcn_raw_buffer_store_b128(v, vecs, offset, 0, kNonTemporal);
    }
    __device__ __forceinline__ float load_edge() const {
        if constexpr (T::kBytes == 2) return T::widen(__builtin_amdgcn_raw_buffer_load_b16(elems, edge, 0, 0));
        else return T::widen(__builtin_amdgcn_raw_buffer_load_b32(elems, edge, 0, 0));
    }
    __device__ __forceinline__ void store_edge(float f) const {
        if constexpr (T::kBytes == 2) {
            typename T::bits_t b;
            T::store1(&b, 0, f);
            __builtin_amdgcn_raw_buffer_store_b16(b, elems, edge, 0, 0);
        } else {
            __builtin_amdgcn_raw_buffer_store_b32(as_u32(f), elems, edge, 0, 0);
        }
    }
    // Record `slice` into the first vectors of every slice of this (output) row, thread j that of slice j ...
    __device__ __forceinline__ void leave(const Slicing& s, int slice, int t, u32x4 record) const {
        if (t < s.slices) st128_keep(first + (static_cast<int64_t>(t) * s.vecs + slice) * 16, record);
    }
    // ... and lane j's record of slice j from the copy that lies in slice `slice`.
    __device__ __forceinline__ SliceRecord take(const Slicing& s, int slice, int lane) const {
        const int j = lane < s.slices ? lane : s.slices - 1;
        return SliceRecord{ld128_keep(first + (static_cast<int64_t>(slice) * s.vecs + j) * 16)};
    }
};

template <typename T>
__global__ void __launch_bounds__(kSlicedBlock) softmax_fwd_slice_sums_kernel(const SoftmaxFwdArgs a, const Slicing s) {
    constexpr int VEC = T::VEC, K = kSlicedVecs;
    __shared__ float red[RedSmem<kSlicedBlock, 1, 1>::kFloats];
    __shared__ double red_sum[RedSmem<kSlicedBlock, 1, 1>::kFloats];
    int phase = 0, phase_sum = 0;
    const int t = threadIdx.x;
    const int row = blockIdx.x / s.slices, slice = blockIdx.x % s.slices;
    const float neg_inf = OpMax::identity<float>();
    const RowSlice<T> x(a.x, a.x_stride_bytes, row, a.n_cols, s, slice, t);
    u32x4 cur[K];
#pragma unroll
    for (int k = 0; k < K; ++k) cur[k] = x.template load<0>((t + k * kSlicedBlock) * 16);
    const float edge = x.load_edge();
    float m = x.edge == kOutOfBounds ? neg_inf : edge * a.sign;
    const float fe = m;
    float f[K][VEC];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        T::unpack(cur[k], f[k]);
        const bool in = t + k * kSlicedBlock < x.n_vecs;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            f[k][e] = in ? f[k][e] * a.sign : neg_inf;
            m = OpMax::apply(m, f[k][e]);
        }
    }
    float mx[1] = {m};
    row_allreduce<kSlicedBlock, 1, 1, OpMax, float>(mx, red, phase, 0, t);
    const float base = mx[0] > neg_inf ? mx[0] : 0.0f;      // nothing but -inf: exp(-inf - 0) = 0
    double acc[1] = {static_cast<double>(exp_c(fe - base))};
#pragma unroll
    for (int k = 0; k < K; ++k) {
        float part = 0.0f;
#pragma unroll
        for (int e = 0; e < VEC; ++e) part += exp_c(f[k][e] - base);
        acc[0] += static_cast<double>(part);
    }
    row_allreduce<kSlicedBlock, 1, 1, OpSum, double>(acc, red_sum, phase_sum, 0, t);
    const RowSlice<T> y(a.y, a.y_stride_bytes, row, a.n_cols, s, slice, t);
    y.leave(s, slice, t, SliceRecord::of(mx[0], acc[0]));
}

template <typename T, bool LOG>
__global__ void __launch_bounds__(kSlicedBlock) softmax_fwd_slice_write_kernel(const SoftmaxFwdArgs a, const Slicing s) {
    constexpr int VEC = T::VEC, K = kSlicedVecs;
    const int t = threadIdx.x, lane = t & 63;
    const int row = blockIdx.x / s.slices, slice = blockIdx.x % s.slices;
    const float neg_inf = OpMax::identity<float>();
    const RowSlice<T> x(a.x, a.x_stride_bytes, row, a.n_cols, s, slice, t), y(a.y, a.y_stride_bytes, row, a.n_cols, s, slice, t);
    const SliceRecord r = y.take(s, slice, lane);
    u32x4 cur[K];
#pragma unroll
    for (int k = 0; k < K; ++k) cur[k] = x.template load<kNonTemporal>((t + k * kSlicedBlock) * 16);
    const float edge = x.load_edge();
    const float m = lane < s.slices ? r.max() : neg_inf;
    const float row_max = group_allreduce<64, OpMax, float>(m);        // a row of -inf alone: -inf - -inf = NaN
    const double part = lane < s.slices ? r.sum() * static_cast<double>(exp_c(m - (row_max > neg_inf ? row_max : 0.0f))) : 0.0;
    const double total = group_allreduce<64, OpSum, double>(part);
    const float scale = static_cast<float>(LOG ? log(total) : 1.0 / total);
    __syncthreads();        // every wave has its records: they are written over now
    auto value = [&](float v) {
        const float z = v * a.sign - row_max;
        if constexpr (LOG) return z - scale;
        else return exp_c(z) * scale;
    };
    y.store_edge(value(edge));
#pragma unroll
    for (int k = 0; k < K; ++k) {
        float f[VEC];
        T::unpack(cur[k], f);
#pragma unroll
        for (int e = 0; e < VEC; ++e) f[e] = value(f[e]);
        y.store((t + k * kSlicedBlock) * 16, T::pack(f));
    }
}

template <typename T, bool LOG>
__global__ void __launch_bounds__(kSlicedBlock) softmax_bwd_slice_sums_kernel(const SoftmaxBwdArgs a, const Slicing s) {
    constexpr int VEC = T::VEC, K = kSlicedVecs;
    __shared__ double red_sum[RedSmem<kSlicedBlock, 1, 1>::kFloats];
    int phase_sum = 0;
    const int t = threadIdx.x;
    const int row = blockIdx.x / s.slices, slice = blockIdx.x % s.slices;
    const RowSlice<T> y(a.y, a.y_stride_bytes, row, a.n_cols, s, slice, t), dy(a.dy, a.dy_stride_bytes, row, a.n_cols, s, slice, t);
    u32x4 cy[LOG ? 1 : K], cg[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int off = (t + k * kSlicedBlock) * 16;
        cg[k] = dy.template load<0>(off);            // past the slice: 0
        if constexpr (!LOG) cy[k] = y.template load<0>(off);
    }
    const float ge = dy.load_edge();
    double acc[1] = {LOG ? static_cast<double>(ge) : static_cast<double>(y.load_edge() * ge)};
#pragma unroll
    for (int k = 0; k < K; ++k) {
        float gf[VEC], yf[VEC];
        T::unpack(cg[k], gf);
        if constexpr (!LOG) T::unpack(cy[k], yf);
        float part = 0.0f;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            if constexpr (LOG) part += gf[e];
            else part = fmaf(yf[e], gf[e], part);
        }
        acc[0] += static_cast<double>(part);
    }
    row_allreduce<kSlicedBlock, 1, 1, OpSum, double>(acc, red_sum, phase_sum, 0, t);
    const RowSlice<T> dx(a.dx, a.dx_stride_bytes, row, a.n_cols, s, slice, t);
    dx.leave(s, slice, t, SliceRecord::of(0.0f, acc[0]));
}

template <typename T, bool LOG>
__global__ void __launch_bounds__(kSlicedBlock) softmax_bwd_slice_write_kernel(const SoftmaxBwdArgs a, const Slicing s) {
    constexpr int VEC = T::VEC, K = kSlicedVecs;
    const int t = threadIdx.x, lane = t & 63;
    const int row = blockIdx.x / s.slices, slice = blockIdx.x % s.slices;
    const RowSlice<T> y(a.y, a.y_stride_bytes, row, a.n_cols, s, slice, t), dy(a.dy, a.dy_stride_bytes, row, a.n_cols, s, slice, t),
        dx(a.dx, a.dx_stride_bytes, row, a.n_cols, s, slice, t);
    const SliceRecord r = dx.take(s, slice, lane);
    u32x4 cy[K], cg[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int off = (t + k * kSlicedBlock) * 16;
        cy[k] = y.template load<kNonTemporal>(off);
        cg[k] = dy.template load<kNonTemporal>(off);
    }
    const float ye = y.load_edge(), ge = dy.load_edge();
    const float total = static_cast<float>(group_allreduce<64, OpSum, double>(lane < s.slices ? r.sum() : 0.0));
    __syncthreads();        // every wave has its records: they are written over now
    auto value = [&](float yv, float gv) {
        if constexpr (LOG) return fmaf(-exp_c(yv), total, gv) * a.sign;
        else return yv * (gv - total) * a.sign;
    };
    dx.store_edge(value(ye, ge));
#pragma unroll
    for (int k = 0; k < K; ++k) {
        float yf[VEC], gf[VEC];
        T::unpack(cy[k], yf);
        T::unpack(cg[k], gf);
#pragma unroll
        for (int e = 0; e < VEC; ++e) gf[e] = value(yf[e], gf[e]);
        dx.store((t + k * kSlicedBlock) * 16, T::pack(gf));
    }
}

#define THN_DECLARE_SOFTMAX_SLICED_LAUNCHERS(NAME)                                                     \
    int launch_softmax_fwd_sliced_##NAME(bool is_log, const SoftmaxFwdArgs& a, Slicing s, hipStream_t st); \
    int launch_softmax_bwd_sliced_##NAME(bool is_log, const SoftmaxBwdArgs& a, Slicing s, hipStream_t st);

THN_DECLARE_SOFTMAX_SLICED_LAUNCHERS(f32)
THN_DECLARE_SOFTMAX_SLICED_LAUNCHERS(f16)
THN_DECLARE_SOFTMAX_SLICED_LAUNCHERS(bf16)

template <typename Args>
int run_sliced(void (*sums)(const Args, const Slicing), void (*write)(const Args, const Slicing), const Args& a, Slicing s, hipStream_t st) {
    const int grid = static_cast<int>(a.M) * s.slices;
    hipLaunchKernelGGL(sums, dim3(grid), dim3(kSlicedBlock), 0, st, a, s);
    if (hipGetLastError() != hipSuccess) return -1;
    hipLaunchKernelGGL(write, dim3(grid), dim3(kSlicedBlock), 0, st, a, s);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

#define THN_DEFINE_SOFTMAX_SLICED_LAUNCHERS(NAME, T)                                                       \
    int launch_softmax_fwd_sliced_##NAME(bool is_log, const SoftmaxFwdArgs& a, Slicing s, hipStream_t st) { \
        return run_sliced<SoftmaxFwdArgs>(softmax_fwd_slice_sums_kernel<T>,                                \
                                          is_log ? softmax_fwd_slice_write_kernel<T, true> : softmax_fwd_slice_write_kernel<T, false>, a, s, st); \
    }                                                                                                      \
    int launch_softmax_bwd_sliced_##NAME(bool is_log, const SoftmaxBwdArgs& a, Slicing s, hipStream_t st) { \
        return is_log ? run_sliced<SoftmaxBwdArgs>(softmax_bwd_slice_sums_kernel<T, true>, softmax_bwd_slice_write_kernel<T, true>, a, s, st) \
                      : run_sliced<SoftmaxBwdArgs>(softmax_bwd_slice_sums_kernel<T, false>, softmax_bwd_slice_write_kernel<T, false>, a, s, st); \
    }

}  // namespace thn
