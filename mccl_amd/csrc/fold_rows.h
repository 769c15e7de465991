// How a list of binary folds is spread over launches: plain arithmetic, the same for the library and
// for the test that checks it on the CPU.
#pragma once

#include <algorithm>
#include <stdint.h>

#include "ring_cut.h"

namespace mcclhip {

// Layout of one fold: [head scalars][16-byte vectors][tail scalars]; head makes the destination 16-byte
// aligned.  `lead` vectors of the first tile group lie in front of the body, and `dst`, `src` and `nvec`
// count from the group's start.  The launch computes all of it (fold_span), so that a wavefront starts
// with its addresses at hand.
struct __attribute__((aligned(32))) FoldSpan {
    char* dst;
    const char* src;
    uint64_t nvec;
    uint16_t head, tail;  // elements, fewer than 16 bytes each
    uint32_t lead;        // vectors of the first tile group that lie in front of the body
};
constexpr uint64_t fold_blocks(const FoldSpan& f) { return (f.nvec + kFoldBlock - 1) / kFoldBlock; }

// Folds of fewer blocks in all take less time than another launch, and a block of theirs that strides
// finds its operands in the caches; it does so for at most kFoldRounds tiles.
constexpr uint64_t kFoldLarge = 16384, kFoldRounds = 16;

// Calls launch(first, m, blocks) so that every fold of f[0 .. n) is in one launch, as one of m folds with
// `blocks` blocks each.  The folds of a ring step are alike: all go in one launch, with the blocks that the
// longest needs.  In a ragged list most of those would have no work, so no fold gets more than
// twice the average; where the longer ones' blocks would then do several tiles one after the other, and
// the folds are large or the tiles many, the folds above the average get launches of their own.  us, fp32,
// striding / parted: one fold of 26 M elements beside nine of 1000 74.6 / 46.6, twelve of 6.5 M beside 108
// of 1000 265 / 145, 40 of 1000 to 2 M 30.9 / 24.1, one of 1 M beside 119 of 1000 18.2 / 9.1; but one of 2 M
// beside nine of 1000 4.7 / 6.5, eight of 300,000 beside 60 of 1000 6.0 / 7.9.  f comes back in another order.
template <class Launch>
void fold_rows(FoldSpan* f, uint32_t n, Launch&& launch) {
    uint64_t longest = 0, sum = 0;
    for (uint32_t i = 0; i < n; i++) {
        const uint64_t b = fold_blocks(f[i]);
        longest = b > longest ? b : longest;
        sum += b;
    }
    const uint64_t most = 2 * ((sum + n - 1) / n) + 1;
    if (longest > most && (sum > kFoldLarge || longest > kFoldRounds * most)) {
        const uint32_t above = (uint32_t)(std::partition(f, f + n, [&](const FoldSpan& s) { return fold_blocks(s) * n > sum; }) - f);
        fold_rows(f, above, launch);
        fold_rows(f + above, n - above, launch);
        return;
    }
    launch(f, n, longest < most ? longest : most);
}

}  // namespace mcclhip
