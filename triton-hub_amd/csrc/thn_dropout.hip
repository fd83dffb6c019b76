// The dropout kernel in the four storage types.
#include "thn_dropout.h"

namespace thn {

template <typename T, bool kWide>
static void launch_mode(DropoutMask mode, const DropoutArgs& a, int grid, hipStream_t st) {
    switch (mode) {
        case DropoutMask::kNone: hipLaunchKernelGGL((dropout_flat_kernel<T, kWide>), dim3(grid), dim3(kDropoutBlock), 0, st, a); break;
        case DropoutMask::kWrite: hipLaunchKernelGGL((dropout_masked_kernel<T, kWide, false>), dim3(grid), dim3(kDropoutBlock), 0, st, a); break;
        case DropoutMask::kRead: hipLaunchKernelGGL((dropout_masked_kernel<T, kWide, true>), dim3(grid), dim3(kDropoutBlock), 0, st, a); break;
    }
}

template <typename T>
static void launch_as(DropoutMask mode, const DropoutArgs& a, int grid, hipStream_t st) {
    // offsets that all fit 32 bits: the second counter word is zero throughout
    if (a.first_offset + a.total_elems <= (int64_t{1} << 32)) launch_mode<T, false>(mode, a, grid, st);
    else launch_mode<T, true>(mode, a, grid, st);
}

int launch_dropout(int dtype, DropoutMask mode, const DropoutArgs& a, int grid, hipStream_t st) {
    switch (dtype) {
        case kF32: launch_as<F32>(mode, a, grid, st); break;
        case kF16: launch_as<F16>(mode, a, grid, st); break;
        case kBF16: launch_as<BF16>(mode, a, grid, st); break;
        case kF64: launch_as<F64>(mode, a, grid, st); break;
        default: return 1;
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace thn
