// Softmax / Softmin / LogSoftmax kernels for rows of 64 to 384 KiB that stay in registers, F32 storage.
#include "thn_softmax_wide.h"

namespace thn {
THN_DEFINE_SOFTMAX_WIDE_LAUNCHERS(f32, F32)
}  // namespace thn
