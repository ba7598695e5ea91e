// index_check.cpp -- the kernels' index rules (gadgetron_amd/csrc/gt_index.h) on
// the host: every lane and entry count they can meet.  Exit status 0 if all hold.
#include <cstdio>

#include "gt_index.h"

int main() {
    int bad = 0;
    // a chunk of 32 entries, n of them before the end of the item, 2 words an entry
    for (uint32_t n = 1; n <= 32; n++)
        for (uint32_t lane = 0; lane < 64; lane++) {
            const uint32_t w = gt::head_word(lane, n);
            const bool in_range = w < 2 * n;
            const bool same_kind = (w & 1) == (lane & 1);  // even lanes: sample indices, odd lanes: row masks
            const bool own = lane / 2 >= n || w == lane;
            if (!in_range || !same_kind || !own) {
                std::printf("head_word: lane %u of %u entries reads word %u\n", lane, n, w);
                bad++;
            }
        }
    std::printf(bad ? "index_check: %d failures\n" : "index_check: ok\n", bad);
    return bad ? 1 : 0;
}
