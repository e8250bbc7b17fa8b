// fa_grid.h — the sequence that a workgroup of the attention kernels serves
// (flash_attention.hip).
#pragma once

namespace tecoops {
namespace fa {

// Sequence (of batch) at place `place` of grid row `row`: the sequences move on by
// one place every 2^turn rows.
constexpr int turned_place(int place, int row, int turn, int batch) {
    return (place + (row >> turn)) % batch;
}

constexpr int kNoTurn = 31;

// The turn of a grid whose rows hold `units` consecutive workgroups of each
// sequence.  Workgroup n runs on XCD n % 8, and an XCD deals its workgroups to its
// 4 shader engines in turn, each workgroup waiting for its own engine: 32 slots,
// n % 32.  With fixed places a long sequence, whose workgroups are the only ones
// with work in the upper rows, has the same slots again after 32 / gcd(32, batch *
// units) rows: all of them with an odd batch, but one engine or a part of the XCDs
// with an even one.  Moving on after as many rows takes it round all slots.  With
// units a multiple of 8 it stays on its XCDs, whose L2 hold its keys and values;
// fewer units would keep it to some of the XCDs, and go round them.
// bf16 causal, D 128, us, fixed / one place each row (or each second one) / this
// rule: 32 heads over 8: 3869 + 3 x 1000 tokens 357 / 164 / 164, + 4 x 1000 173 /
// 191 / 174, 9 of 64..2048 90 / 115 / 90, 24 of 16..1024 84 / 74 / 75; 16 over 2
// (4 units): 3869 + 7 x 1000 356 / 140 / 140, and 162 kept to its XCDs.
constexpr int turn_shift(int units, int batch) {
    if (batch % 2 != 0 || units % 32 == 0) return kNoTurn;
    return 5 - __builtin_ctz((units * batch) | 32);
}

// The same for a prefill of `rows` query rows in all and at most `longest` per
// sequence: sequences alike (within an eighth of the longest in the mean) have
// their work in every row, and nothing to spread (16 heads over 2, 16 x 512 rows,
// on two machines: fixed 36.2 and 37.6, turned 39.7 and 38.2).
constexpr int turn_shift(int units, int batch, int longest, long long rows) {
    return 8 * rows >= 7ll * longest * batch ? kNoTurn : turn_shift(units, batch);
}

}  // namespace fa
}  // namespace tecoops
