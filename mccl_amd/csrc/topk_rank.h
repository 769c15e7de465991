// The last step of a selection in a list: the `want`-th largest of the few entries that share a prefix, the same for the
// kernels and for the test that checks it on the CPU.
#pragma once

#include <stdint.h>

namespace mcclhip {

// Entries of list[from, to) that are as large or larger: the cut is the entry that as many reach as are wanted.  Entries
// differ in their index, so that one is the cut, and no entry where a list in scratch memory that another call
// overwrites holds one twice across it.  (Counting the larger ones instead, two equal entries would both be the cut, and one
// more entry than wanted reach it.)
constexpr uint32_t reaching_entries(const uint64_t* list, uint32_t from, uint32_t to, uint64_t entry) {
    uint32_t n = 0;
#pragma unroll 4
    for (uint32_t j = from; j < to; j++) n += list[j] >= entry ? 1u : 0u;
    return n;
}

// Where no entry is the cut.  An entry's key, in the upper half, has 31 bits: none reaches this one, nor the one above it.
constexpr uint64_t kNoCut = 0xFFFFFFFEFFFFFFFFull;

}  // namespace mcclhip
