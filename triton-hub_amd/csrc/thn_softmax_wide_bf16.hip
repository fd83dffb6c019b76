// Softmax / Softmin / LogSoftmax kernels for rows of 64 to 384 KiB that stay in registers, BF16 storage.
#include "thn_softmax_wide.h"

namespace thn {
THN_DEFINE_SOFTMAX_WIDE_LAUNCHERS(bf16, BF16)
}  // namespace thn
