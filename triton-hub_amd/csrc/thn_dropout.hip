// The dropout kernel in the four storage types.
#include "thn_dropout.h"

namespace thn {

template <typename T>
static void launch_as(const DropoutArgs& a, int grid, hipStream_t st) {
    // offsets that all fit 32 bits: the second counter word is zero throughout
    if (a.first_offset + a.total_elems <= (int64_t{1} << 32)) hipLaunchKernelGGL((dropout_flat_kernel<T, false>), dim3(grid), dim3(kDropoutBlock), 0, st, a);
    else hipLaunchKernelGGL((dropout_flat_kernel<T, true>), dim3(grid), dim3(kDropoutBlock), 0, st, a);
}

int launch_dropout(int dtype, const DropoutArgs& a, int grid, hipStream_t st) {
    switch (dtype) {
        case kF32: launch_as<F32>(a, grid, st); break;
        case kF16: launch_as<F16>(a, grid, st); break;
        case kBF16: launch_as<BF16>(a, grid, st); break;
        case kF64: launch_as<F64>(a, grid, st); break;
        default: return 1;
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace thn
