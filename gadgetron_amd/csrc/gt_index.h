// gt_index.h -- index rules of the gridding kernels, plain C++ so that a host
// program can check them (tests/cpp/index_check.cpp).
#pragma once

#include <stdint.h>

namespace gt {

// Word that a lane reads of the heads (j, rows) of n table entries, n >= 1, lanes
// 2 e and 2 e + 1 entry e's two words: past the last entry the last one's, so that
// an even lane always gets a sample index and an odd one a row mask.
constexpr uint32_t head_word(uint32_t lane, uint32_t n) {
    const uint32_t e = lane >> 1;
    return 2 * (e < n ? e : n - 1) + (lane & 1);
}

}  // namespace gt
