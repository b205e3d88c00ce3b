// Transfers between host and device through pinned memory (internal).
// Measured: a terminal frame 102 -> 59 us, a 640x480 picture 260 -> 189 us, an
// export of 141 MB 60 -> 4.1 ms (with the wrapper's single allocation).
//
// A copy between pageable memory and the device is staged by the runtime in
// pieces that wait for one another (16 GB/s here, 57 GB/s from pinned
// memory), and each such copy costs a wait of its own.  Here the pinned
// memory comes from a process-wide pool: calls take what they need and give
// it back before they return, so handles share it and a new handle's first
// call finds it warm.
#pragma once
#include <hip/hip_runtime.h>

#include "sloth_host.h"

namespace sloth {

// The pool keeps freed blocks while a handle lives (at most PIN_POOL_BYTES,
// the latest ones; sizes are powers of two, and a lease takes a block of its
// own size only) and frees them with the last one.  Safe from any thread.
constexpr size_t PIN_POOL_BYTES = 64u << 20;
struct PinPoolUser {
    PinPoolUser();
    ~PinPoolUser();
    PinPoolUser(const PinPoolUser&) = delete;
    PinPoolUser& operator=(const PinPoolUser&) = delete;
};

// Pinned memory out of the pool, for the length of a call or of a handle.
// Work enqueued on `s` may use it until the lease ends, which waits for `s`
// unless done() said that this is not needed.  take() again ends the lease
// and begins another.
struct PinLease {
    void* p = nullptr;
    PinLease() = default;
    PinLease(const PinLease&) = delete;
    PinLease& operator=(const PinLease&) = delete;
    ~PinLease() { end(); }
    int take(size_t n, hipStream_t s);
    void done() { busy = false; }
    template <class T> T* as() const { return (T*)p; }

  private:
    void end();
    size_t bytes = 0;
    hipStream_t stream = nullptr;
    bool busy = false;
};

struct Span {
    void* host;
    void* dev;
    size_t bytes;
};

// Copies the spans to the host after everything enqueued on `s`; returns when
// they are there.
int copy_out(const Span* spans, int n, hipStream_t s);
// Enqueues copies of the spans to the device on `s`; the host memory is free
// on return, the lease holds the bytes.
int copy_in(const Span* spans, int n, PinLease& lease, hipStream_t s);

}  // namespace sloth
