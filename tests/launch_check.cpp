// Host check of the run counts of h264g_dev.h: every launch of a batch keeps within a grid's room.
#include <cstdio>

#include "h264g_dev.h"

int main() {
    for (int what = 1; what < 4; what++)
        for (int mbaff = 0; mbaff < 2; mbaff++) {
            const bool mbs = what & INTER_MBS, bs = what & INTER_BS;
            const uint64_t most = runs_per_launch(mbs, bs, mbaff), blocks = blocks_of_run(mbs, bs, mbaff);
            const uint64_t want = (mbs ? 64 : 0) + (bs ? (mbaff ? 64 : 32) : 0);
            // the largest batch: 4095 pictures of 2^20 MBs; a launch's threads stay below 2^32, and
            // one run more would not fit
            const uint64_t n = 4095ull * ((1 << 20) / MB_CHUNK);
            const bool ok = blocks == want && most * blocks * 64 < 1ull << 32 && (most + 1) * blocks * 64 >= 1ull << 32 && n < 1ull << 32 &&
                            most >= (1 << 20) / MB_CHUNK;
            if (!ok) {
                std::printf("what %d mbaff %d: %llu runs of %llu blocks\n", what, mbaff, (unsigned long long)most, (unsigned long long)blocks);
                return 1;
            }
        }
    std::puts("ok");
    return 0;
}
