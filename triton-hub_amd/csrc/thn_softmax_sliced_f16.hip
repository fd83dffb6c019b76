// Softmax / Softmin / LogSoftmax kernels for few rows of more than 64 KiB, cut into slices, F16 storage.
#include "thn_softmax_sliced.h"

namespace thn {
THN_DEFINE_SOFTMAX_SLICED_LAUNCHERS(f16, F16)
}  // namespace thn
