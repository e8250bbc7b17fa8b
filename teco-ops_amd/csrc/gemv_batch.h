// gemv_batch.h — weight products of a batch of rows of x (gemv_batch.hip),
// for gemv.hip's dispatch.
#pragma once

#include "common.h"

namespace tecoops {

// y[b, n] = T(sum_k W[n, k] x[b, k] (* scales[n])) for any batch, in slices of
// up to 64 rows of x; W is 16-bit (scales null, type T) or int8 (T = fp16).
// W and x 16-byte aligned, K a multiple of the values in 16 bytes of W.
// INTERNAL_ERROR when a launch fails.
tecoopsStatus_t gemv_batch(hipStream_t s, const void *W, const void *scales, const void *x,
                           void *y, int batch, int n, int k, tecoopsDataType_t dataType, bool i8);

}  // namespace tecoops
