// The dropout kernel in the four storage types.
#include "thn_dropout.h"

namespace thn {

// A masked call's offsets start at 0 and end below 2^32 (dropout_launch in thn_api.hip).  kProduct: a.scale is set.
template <typename T, bool kProduct>
static void launch_as(DropoutMask mode, const DropoutArgs& a, int grid, hipStream_t st) {
    const dim3 blocks(grid), threads(kDropoutBlock);
    switch (mode) {
        case DropoutMask::kNone:
            // offsets that all fit 32 bits: the second counter word is zero throughout
            if (a.first_offset + a.total_elems <= (int64_t{1} << 32)) hipLaunchKernelGGL((dropout_flat_kernel<T, false, kProduct>), blocks, threads, 0, st, a);
            else hipLaunchKernelGGL((dropout_flat_kernel<T, true, kProduct>), blocks, threads, 0, st, a);
            break;
        case DropoutMask::kWrite: hipLaunchKernelGGL((dropout_masked_kernel<T, false, kProduct>), blocks, threads, 0, st, a); break;
        case DropoutMask::kRead: hipLaunchKernelGGL((dropout_masked_kernel<T, true, kProduct>), blocks, threads, 0, st, a); break;
    }
}
template <typename T>
static void launch_16bit(DropoutMask mode, const DropoutArgs& a, int grid, hipStream_t st) {
    if (a.scale != 0.0f) launch_as<T, true>(mode, a, grid, st);
    else launch_as<T, false>(mode, a, grid, st);
}

int launch_dropout(int dtype, DropoutMask mode, const DropoutArgs& a, int grid, hipStream_t st) {
    switch (dtype) {
        case kF32: launch_as<F32, false>(mode, a, grid, st); break;
        case kF16: launch_16bit<F16>(mode, a, grid, st); break;
        case kBF16: launch_16bit<BF16>(mode, a, grid, st); break;
        case kF64: launch_as<F64, false>(mode, a, grid, st); break;
        default: return 1;
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace thn
