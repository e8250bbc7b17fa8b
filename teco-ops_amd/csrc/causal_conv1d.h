// causal_conv1d.h — the choice between the kernels of token-contiguous rows
// (causal_conv1d.hip).
#pragma once

namespace tecoops {

// Whether a varlen batch of token-contiguous rows runs along the token axis
// (conv1d_axis_kernel) or a wave per sequence and channel (or its grouped form).
// Along the axis a workgroup per channel takes at most 4 groups of 2048 tokens at a
// time, so that it wants channels to fill the chip, and pays where the sequences
// are short against a group, and where they start off the 16-byte boundary, which
// costs a wave per row more.  The host knows their total only: lengths that are
// alike and whole vectors leave one that 8 times their number divides, which other
// lengths hardly ever do.
// Not divided: µs by rows / along the axis on 256 CUs: 44 sequences of 12..23
// tokens, dim 6336 32 / 18; 100 of 9 in the mean, 6360 53 / 23; 26 of 32, 4840 26 /
// 14; 7 of 163, 2704 16 / 9; 6 of 637, 6544 44 / 28; 20 of 1186, 1192 41 / 28; but 7 of
// 62, 4520 11 / 12, and few channels of long ones: 54 of 1106, 272 26 / 36.
// Divided: µs by rows / along the axis, sequences on the boundary, then off it or
// of random length:
//   mean length to 256: dim 512, 64 x 256 18.5 / 15.4, 25.9 / 20.1; dim 384,
//     64 x 256 14.8 / 15.4, 21.7 / 19.1, 512 x 40 29 / 27, 39 / 27; dim 256
//     19.3 / 20.1, 24.8 / 21.1; dim 64, 64 x 256 6.5 / 9.8
//   to 512: dim 4096, 16 x 512 55 / 37, 68 / 50; dim 768, 4 x 512 6.1 / 6.4, 7.9
//     / 8.3; dim 512 8 x 512 6.6 / 7.0, 16 x 512 10.2 / 8.6
//   below 1024: dim 4096, 16 x 1000 69 / 61, 86 / 62, 32 random of 924 in the
//     mean 169 / 109; dim 768 17.4 / 18.0, 20.2 / 18.0; dim 512 13.4 / 14.2, 16.1
//     / 14.7, 24 x 768 15.5 / 18.5; few or longer ones lose: dim 4096, 4 x
//     1024 20.3 / 22.1, 24.6 / 24.7, dim 2048, 8 x 1024 19.1 / 21.4
//   longer: dim 4096, 4 x 4096 50 / 66, 58 / 70; dim 64, 64 x 4096 17 / 109
//   fewer than 2048 tokens: dim 2048, 8 x 128 7.3 / 8.5, 8 x 64 6.0 / 8.3; dim
//     4096, 4 x 256 11.7 / 12.2, 16.0 / 12.3
// and where one or two sequences have too few channels to fill the chip with a
// wave each: dim 1024, 1 x 16384 23.5 / 17.1, 25.8 / 21.5; dim 64 20.8 / 8.0;
// dim 2048 30.4 / 34.9; dim 768, 2 x 4096 10.8 / 8.9, 12.7 / 13.7, 3001 + 900
// tokens 9.9 / 8.2.
// Over 1000 random batches (1..128 sequences, 64..8192 channels, a third alike) the
// choice takes 1.6 % more than the better kernel in the mean.
inline bool conv1d_along_axis(long long batch, long long dim, long long tokens, long long cus) {
    if (batch <= 2 && tokens >= 3072 && batch * dim <= 6 * cus) return true;
    if (tokens % (8 * batch) != 0) {
        if (tokens * dim < (1LL << 20) || dim < cus || tokens > batch * (dim >= 3 * cus ? 2048 : 512)) return false;
        return (tokens >= 448 && batch * dim >= 96 * cus) || (tokens >= 1024 && batch * dim >= 16 * cus);
    }
    if (tokens < 1024 || (tokens < 2048 && tokens * dim < (1LL << 22))) return false;
    const long long mean = (tokens + batch - 1) / batch;
    if (mean <= 256) return 2 * dim >= 3 * cus;
    if (mean <= 512) return dim >= 3 * cus || (dim >= 2 * cus && tokens >= 8192);
    return mean < 1024 && batch >= 8 && dim >= 3 * cus;
}

}  // namespace tecoops
