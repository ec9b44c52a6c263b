// psim_stage.hip -- copies between device memory and a caller's pageable
// arrays through a pinned staging buffer (host code).
//
// A pageable hipMemcpy costs, on MI355X hosts, 20 us at 24 KB, 0.35 ms at 0.8 MB
// (2.2 GB/s) and 5 ms for 48 MB into fresh pages; the same copies from or to
// pinned memory take 8 us, 0.02 ms and 0.9 ms, and the host's part (a copy
// between the staging buffer and the caller's array, page faults included) is
// spread over a few threads and overlaps the next chunk's transfer.
// Measured, arrays to n x 3 on the device included: a state of 2,097,152
// particles (240 MB) 72 -> 7 ms, of 262,144 7 -> 1 ms, a force_table call at
// 100,003 particles (7.2 MB both ways) 0.83 -> 0.37 ms, a step and a read of
// 1,000 particles 134 -> 105 us.  Halves of 2 MiB instead of 4: 240 MB in
// 12 ms, the force_table call 0.39 ms.
#include "psim_stage.hpp"

#include <algorithm>
#include <cstdio>
#include <cstring>

namespace psim {

namespace {

constexpr size_t kChunk = 4u << 20;   // one half of the staging buffer at most
constexpr size_t kAlign = 64;

inline size_t padded(size_t b) { return (b + kAlign - 1) & ~(kAlign - 1); }

bool ok(hipError_t e, const char *what)
{
    if (e == hipSuccess) return true;
    std::fprintf(stderr, "psim: %s failed: %s\n", what, hipGetErrorString(e));
    return false;
}

// The same copies straight from and to pageable memory (no pinned memory to be
// had).
int unstaged(hipStream_t st, const Xfer *x, int nx, hipMemcpyKind kind)
{
    const bool up = kind == hipMemcpyHostToDevice;
    for (int k = 0; k < nx; ++k)
        if (!ok(hipMemcpyAsync(up ? const_cast<void *>(x[k].dev) : x[k].host,
                               up ? x[k].host : x[k].dev, x[k].bytes, kind, st), "copy"))
            return -1;
    return ok(hipStreamSynchronize(st), "copy") ? 0 : -1;
}

// What stays in flight after a failure still uses the buffer.
int fail(hipStream_t st)
{
    (void)hipStreamSynchronize(st);
    return -1;
}

}  // namespace

bool stage_reserve(HostStage &h, size_t bytes)
{
    const size_t want = std::min(std::max(bytes, (size_t)4096), 2 * kChunk);
    if (h.cap >= want || h.refused) return h.cap != 0;
    // (powers of two: a caller whose calls grow does not reallocate each time)
    size_t cap = 4096;
    while (cap < want) cap *= 2;
    HostStage grown;
    bool made = ok(hipHostMalloc((void **)&grown.buf, cap, hipHostMallocDefault), "hipHostMalloc");
    if (!made) grown.buf = nullptr;
    for (hipEvent_t &e : grown.done)
        made = made && ok(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreate");
    if (!made) {   // the smaller buffer, if there is one, takes more rounds
        (void)hipGetLastError();
        stage_free(grown);
        h.refused = true;   // asked for once
        return h.cap != 0;
    }
    grown.cap = cap;
    stage_free(h);
    h = grown;
    return true;
}

void stage_free(HostStage &h)
{
    if (h.buf) (void)hipHostFree(h.buf);
    for (hipEvent_t &e : h.done) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    h.buf = nullptr;
    h.cap = 0;
}

int stage_read(HostStage &h, hipStream_t st, const Xfer *x, int nx)
{
    size_t total = 0;
    for (int k = 0; k < nx; ++k) total += padded(x[k].bytes);
    if (!stage_reserve(h, total)) return unstaged(st, x, nx, hipMemcpyDeviceToHost);
    if (total <= h.cap) {   // one round
        size_t at = 0;
        for (int k = 0; k < nx; ++k) {
            if (!ok(hipMemcpyAsync(h.buf + at, x[k].dev, x[k].bytes, hipMemcpyDeviceToHost, st),
                    "copy to the host"))
                return fail(st);
            at += padded(x[k].bytes);
        }
        if (!ok(hipStreamSynchronize(st), "copy to the host")) return -1;
        at = 0;
        for (int k = 0; k < nx; ++k) {
            host_copy(x[k].host, h.buf + at, x[k].bytes);
            at += padded(x[k].bytes);
        }
        return 0;
    }
    // chunks through the two halves: the host empties one while the other
    // fills
    const size_t half = h.cap / 2;
    void *to[2] = {nullptr, nullptr};
    size_t len[2] = {0, 0};
    int b = 0;
    auto empty = [&](int k) {
        if (!to[k]) return true;
        if (!ok(hipEventSynchronize(h.done[k]), "copy to the host")) return false;
        host_copy(to[k], h.buf + k * half, len[k]);
        to[k] = nullptr;
        return true;
    };
    for (int k = 0; k < nx; ++k)
        for (size_t off = 0; off < x[k].bytes; off += half, b ^= 1) {
            if (!empty(b)) return fail(st);
            len[b] = std::min(half, x[k].bytes - off);
            if (!ok(hipMemcpyAsync(h.buf + b * half, (const char *)x[k].dev + off, len[b],
                                   hipMemcpyDeviceToHost, st), "copy to the host") ||
                !ok(hipEventRecord(h.done[b], st), "hipEventRecord"))
                return fail(st);
            to[b] = (char *)x[k].host + off;
        }
    return empty(b) && empty(b ^ 1) ? 0 : fail(st);
}

int stage_write(HostStage &h, hipStream_t st, const Xfer *x, int nx)
{
    size_t total = 0;
    for (int k = 0; k < nx; ++k) total += padded(x[k].bytes);
    if (!stage_reserve(h, total)) return unstaged(st, x, nx, hipMemcpyHostToDevice);
    const bool once = total <= h.cap;
    const size_t half = once ? 0 : h.cap / 2;
    size_t at = 0;
    bool used[2] = {false, false};
    int b = 0;
    for (int k = 0; k < nx; ++k) {
        const size_t step = once ? x[k].bytes : half;
        for (size_t off = 0; off < x[k].bytes; off += step) {
            const size_t n = std::min(step, x[k].bytes - off);
            if (!once) {
                if (used[b] && !ok(hipEventSynchronize(h.done[b]), "copy to the device"))
                    return fail(st);
                at = b * half;
            }
            host_copy(h.buf + at, (const char *)x[k].host + off, n);
            if (!ok(hipMemcpyAsync((char *)const_cast<void *>(x[k].dev) + off, h.buf + at, n,
                                   hipMemcpyHostToDevice, st), "copy to the device"))
                return fail(st);
            if (once) {
                at += padded(n);
            } else {
                if (!ok(hipEventRecord(h.done[b], st), "hipEventRecord")) return fail(st);
                used[b] = true;
                b ^= 1;
            }
        }
    }
    // the staging buffer is free again for the next call
    return ok(hipStreamSynchronize(st), "copy to the device") ? 0 : -1;
}

}  // namespace psim
