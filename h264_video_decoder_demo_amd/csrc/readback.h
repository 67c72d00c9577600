// readback.h -- how planes that lie one after the other in a source reach memory of the caller's:
// each by a transfer of its own, or through the two halves of a buffer and a copy.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <cstring>

struct Plane {
    uint8_t *to;
    size_t n;
};

// Io: what starts and awaits transfers, in order (each call 0 or an error code):
//   bool direct(plane, mean)   the plane is written by a transfer (mean: bytes per plane of the call)
//   int fetch(to, at, n)       starts the transfer of n bytes from `at` of the source
//   int mark(half)             wait(half) waits for what has been started so far
//   int wait(half)
//   int wait_all()             waits for everything started
// Planes p .. end - 1, which start at `at`, through the buffer.
template <class Io>
int bounce_planes(Io &io, uint8_t *buffer, size_t half, size_t at, const Plane *p, const Plane *end) {
    size_t total = 0;
    for (const Plane *q = p; q != end; q++) total += q->n;
    size_t done = 0;  // bytes of *p that are there
    const size_t parts = (total + half - 1) / half;
    auto part = [&](size_t k) { return std::min(half, total - k * half); };
    auto fetch = [&](size_t k) -> int {
        if (int rc = io.fetch(buffer + (k & 1) * half, at + k * half, part(k))) return rc;
        return parts > 1 ? io.mark((int)(k & 1)) : 0;
    };
    for (size_t k = 0; k < parts && k < 2; k++)
        if (int rc = fetch(k)) return rc;
    for (size_t k = 0; k < parts; k++) {
        if (int rc = parts > 1 ? io.wait((int)(k & 1)) : io.wait_all()) return rc;
        const uint8_t *src = buffer + (k & 1) * half;
        for (size_t left = part(k); left;) {
            const size_t n = std::min(left, p->n - done);
            std::memcpy(p->to + done, src, n);
            src += n;
            left -= n;
            done += n;
            if (done == p->n) {
                p++;
                done = 0;
            }
        }
        if (k + 2 < parts)
            if (int rc = fetch(k + 2)) return rc;
    }
    return 0;
}

// Planes p .. end - 1.  When it returns, also with an error, no transfer that it started is still
// writing the caller's memory or the buffer.
template <class Io>
int read_planes(Io &io, uint8_t *buffer, size_t half, const Plane *p, const Plane *end) {
    size_t mean = 0;
    for (const Plane *q = p; q != end; q++) mean += q->n / (size_t)(end - p);
    const Plane *first = p;  // planes first .. p - 1, n bytes from `at`, are to go through the buffer
    size_t at = 0, n = 0;
    auto run = [&]() -> int {
        for (; p != end; p++) {
            if (!io.direct(*p, mean)) {
                n += p->n;
                continue;
            }
            if (n)
                if (int rc = bounce_planes(io, buffer, half, at, first, p)) return rc;
            at += n;
            if (int rc = io.fetch(p->to, at, p->n)) return rc;
            at += p->n;
            first = p + 1;
            n = 0;
        }
        if (n)
            if (int rc = bounce_planes(io, buffer, half, at, first, end)) return rc;
        return io.wait_all();
    };
    const int rc = run();
    if (rc) (void)io.wait_all();
    return rc;
}
