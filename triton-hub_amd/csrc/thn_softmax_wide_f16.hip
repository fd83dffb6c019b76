// Flat-mapped Softmax / Softmin / LogSoftmax kernels for narrow rows, F16 storage.
#include "thn_softmax_wide.h"

namespace thn {
THN_DEFINE_SOFTMAX_WIDE_LAUNCHERS(f16, F16)
}  // namespace thn
