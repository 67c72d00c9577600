// Host check of csrc/readback.h: transfers that take effect only when awaited, one of which
// fails.  Usage: readback_check; prints "ok" or what is wrong.
#include <cstdio>
#include <vector>

#include "readback.h"

struct Io {
    const std::vector<uint8_t> &src;
    unsigned direct_mask;        // planes written by a transfer
    const Plane *first;
    int fail_at;                 // the call that fails (counted from 0), -1 none
    int calls = 0;
    struct Job { uint8_t *to; size_t at, n; };
    std::vector<Job> flying;
    size_t marks[2] = {0, 0}, started = 0, landed = 0;
    bool fails() { return calls++ == fail_at; }
    void land(size_t upto) {
        for (; landed < upto; landed++, flying.erase(flying.begin())) std::memcpy(flying[0].to, &src[flying[0].at], flying[0].n);
    }
    bool direct(const Plane &p, size_t) { return (direct_mask >> (&p - first)) & 1u; }
    int fetch(uint8_t *to, size_t at, size_t n) {
        if (fails()) return -3;
        flying.push_back({to, at, n});
        started++;
        return 0;
    }
    int mark(int h) {
        if (fails()) return -3;
        marks[h] = started;
        return 0;
    }
    int wait(int h) {
        if (fails()) return -3;
        land(marks[h]);
        return 0;
    }
    int wait_all() {
        if (fails()) return -3;  // (a failed wait: the next one succeeds)
        land(started);
        return 0;
    }
};

int main() {
    const size_t half = 16;
    std::vector<uint8_t> src(400);
    for (size_t i = 0; i < src.size(); i++) src[i] = (uint8_t)(i * 37 + 11);
    for (size_t y : {1, 15, 16, 17, 32, 40, 200})
        for (size_t c : {1, 4, 16, 50})
            for (unsigned mask = 0; mask < 8; mask++)
                for (int fail = -1;; fail++) {
                    std::vector<uint8_t> buffer(2 * half), out(y + 2 * c + 3, 0xEE);
                    const Plane p[3] = {{&out[0], y}, {&out[y + 1], c}, {&out[y + c + 2], c}};
                    Io io{src, mask, p, fail};
                    const int rc = read_planes(io, buffer.data(), half, p, p + 3);
                    if (!io.flying.empty()) {
                        std::printf("y %zu c %zu direct %u, call %d fails: %zu transfers in flight\n", y, c, mask, fail, io.flying.size());
                        return 1;
                    }
                    const bool failed = fail >= 0 && fail < io.calls;
                    if ((rc != 0) != (fail >= 0 && io.calls > fail)) {
                        std::printf("y %zu c %zu direct %u, call %d fails: code %d\n", y, c, mask, fail, rc);
                        return 1;
                    }
                    if (!failed) {
                        bool same = out[y] == 0xEE && out[y + c + 1] == 0xEE && out[y + 2 * c + 2] == 0xEE;
                        for (size_t i = 0; i < y; i++) same &= p[0].to[i] == src[i];
                        for (size_t i = 0; i < c; i++) same &= p[1].to[i] == src[y + i] && p[2].to[i] == src[y + c + i];
                        if (!same) {
                            std::printf("y %zu c %zu direct %u: wrong bytes\n", y, c, mask);
                            return 1;
                        }
                        if (fail >= 0) break;  // no call left to fail
                    }
                }
    std::puts("ok");
    return 0;
}
