// gemv_batch.h — weight products of a batch of rows of x (gemv_batch.hip),
// for gemv.hip's dispatch.
#pragma once

#include "tecoops.h"

#include <hip/hip_runtime_api.h>

namespace tecoops {

// Rows of x that a launch stages for `batch` (at most 64) rows.
inline int gemv_batch_staged(int batch) {
    return batch <= 4 ? 4 : batch <= 8 ? 8 : (batch + 15) / 16 * 16;
}

// Bytes per element of K that the busiest CU copies into LDS for n rows of W in
// workgroups of r, each with `staged` rows of x.
inline long long gemv_batch_bytes(long long n, int r, int staged, bool i8, int cus) {
    const long long wgs = (n + r - 1) / r;
    return (wgs + cus - 1) / cus * (r * (i8 ? 1 : 2) + 2 * staged);
}

// Rows of W per workgroup: of the sizes built, the one whose busiest CU copies
// the fewest bytes of W and x together, the largest on ties.  Counted in rows
// of W alone, widths between two sizes fell to 8 rows, which copies x most
// often and throws half of every MFMA away (on 256 CUs, µs, then / now: int8
// [22528, 4096] batch 8 41.3 / 18.5, [30720, 4096] batch 32 90.8 / 25.1; bf16
// [14336, 4096] batch 64 73.1 / 23.2).  Over 1656 products (N 64..65536, K
// 1024..16384, batch 2..64) the time of the size it picks is 1 % above that of
// the best size in the mean.  48 rows for up to 8 rows of x, where staging x
// costs least; above 32 rows of x two int8 stages fit in LDS from 32 rows on.
// 16-bit rows of a multiple of 32 KiB keep off 48, and off 16 in several rounds
// (waves of 16 rows then queue on the same memory channels: [12288, 16384]
// batch 8 81.2 at 48, 59.7 at 64, [10240, 16384] batch 3 67.1 at 16, 55.3 at 8).
inline int gemv_batch_rows(int n, int k, int batch, bool i8, int cus) {
    const int staged = gemv_batch_staged(batch);
    int best = 0;
    long long least = 0;
    for (int r : {128, 112, 96, 64, 48, 32, 16, 8}) {
        if (r == 48 && staged > 8) continue;
        if (!i8 && k % 16384 == 0 && (r == 48 || (r == 16 && n > 16 * cus))) continue;
        if (r < 32 && i8 && staged > 32) continue;
        const long long bytes = gemv_batch_bytes(n, r, staged, i8, cus);
        if (best == 0 || bytes < least) {
            least = bytes;
            best = r;
        }
    }
    return best;
}

// y[b, n] = T(sum_k W[n, k] x[b, k] (* scales[n])) for any batch, in slices of
// up to 64 rows of x; W is 16-bit (scales null, type T) or int8 (T = fp16).
// W and x 16-byte aligned, K a multiple of the values in 16 bytes of W.
// INTERNAL_ERROR when a launch fails.
tecoopsStatus_t gemv_batch(hipStream_t s, const void *W, const void *scales, const void *x,
                           void *y, int batch, int n, int k, tecoopsDataType_t dataType, bool i8);

}  // namespace tecoops
