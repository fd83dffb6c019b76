// Softmax / Softmin / LogSoftmax kernels for few rows of more than 64 KiB, cut into slices, BF16 storage.
#include "thn_softmax_sliced.h"

namespace thn {
THN_DEFINE_SOFTMAX_SLICED_LAUNCHERS(bf16, BF16)
}  // namespace thn
