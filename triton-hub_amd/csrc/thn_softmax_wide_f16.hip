// Softmax / Softmin / LogSoftmax kernels for rows of 64 to 384 KiB that stay in registers, F16 storage.
#include "thn_softmax_wide.h"

namespace thn {
THN_DEFINE_SOFTMAX_WIDE_LAUNCHERS(f16, F16)
}  // namespace thn
