// The two halves of a dropout that keeps its decisions for the backward, for the host module (thn_host.cpp).  Same function
// and same bits as thn_dropout with first_offset 0 (include/thnorm.h), status codes too.
#pragma once

#include <stdint.h>

namespace thn {

// 32-bit words of the mask of n elements (dropout_masked_kernel in thn_dropout.h): 256 per started piece of 1024 16-byte vectors.
inline int64_t dropout_mask_words(int64_t n, int elem_bytes) { return (n / (16 / elem_bytes) + 1023) / 1024 * 256; }

int dropout_keep_mask(const void* x, void* out, uint32_t* mask, int64_t n, float p, uint64_t seed, int dtype, void* stream);
int dropout_from_mask(const void* x, void* out, const uint32_t* mask, int64_t n, float p, uint64_t seed, int dtype, void* stream);

}  // namespace thn
