// psim_stage.hpp -- copies between device memory and a caller's pageable
// arrays through a pinned staging buffer (psim_stage.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace psim {

// A context's pinned buffer, at most 8 MiB: made with the context in the size
// of its state (pinning 8 MiB takes 0.5 ms, which a first call would pay
// otherwise), grown where a call needs more, freed with the context.  Without
// pinned memory the copies go through a smaller buffer made before, or straight
// to pageable memory.  Used by one call on the context at a time, as the context
// is.
struct HostStage {
    char *buf = nullptr;
    size_t cap = 0;
    bool refused = false;   // no more pinned memory to be had
    hipEvent_t done[2] = {nullptr, nullptr};
};

// One array of a copy: its host and device addresses and its size.
struct Xfer {
    void *host;
    const void *dev;
    size_t bytes;
};

// Room for `bytes`, up to the 8 MiB that longer copies pass through in two
// halves; false where there is no buffer at all.
bool stage_reserve(HostStage &h, size_t bytes);
void stage_free(HostStage &h);
// device -> host, in stream order after what is enqueued; the arrays are
// filled on return.  0, or -1 after a message on stderr.
int stage_read(HostStage &h, hipStream_t st, const Xfer *x, int nx);
// host -> device; the device arrays are written when the stream gets past the
// call, the host arrays are free on return.
int stage_write(HostStage &h, hipStream_t st, const Xfer *x, int nx);

// memcpy, spread over a few threads from 1 MiB on (psim_host.cpp)
void host_copy(void *dst, const void *src, size_t bytes);

// One particle's vector in an n x 3 array.
template <class T>
__device__ __forceinline__ void store_aos(T *out, int o, T x, T y, T z)
{
    T *q = out + 3 * (size_t)o;
    q[0] = x;
    q[1] = y;
    q[2] = z;
}

}  // namespace psim
