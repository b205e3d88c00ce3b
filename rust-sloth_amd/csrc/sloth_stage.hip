// Transfers between host and device through pinned memory: see sloth_stage.h.
#include "sloth_stage.h"

#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>

namespace sloth {

namespace {
struct Block {
    void* p;
    size_t bytes;
};
struct Pool {
    std::mutex mu;
    std::array<Block, 32> idle;   // longest idle first
    size_t n = 0, bytes = 0;
    int users = 0;
    Block remove(size_t i)
    {
        const Block b = idle[i];
        bytes -= b.bytes;
        std::copy(idle.begin() + i + 1, idle.begin() + n--, idle.begin() + i);
        return b;
    }
};
// never destroyed: handles may outlive static destructors
Pool& pool()
{
    static Pool* p = new Pool;
    return *p;
}
}  // namespace

PinPoolUser::PinPoolUser()
{
    std::lock_guard<std::mutex> lk(pool().mu);
    ++pool().users;
}

PinPoolUser::~PinPoolUser()
{
    Pool& q = pool();
    std::lock_guard<std::mutex> lk(q.mu);
    if (--q.users > 0) return;
    for (size_t i = 0; i < q.n; ++i) (void)hipHostFree(q.idle[i].p);
    q.n = q.bytes = 0;
}

int PinLease::take(size_t need, hipStream_t s)
{
    end();
    size_t want = 65536;
    while (want < need) want *= 2;
    stream = s;
    busy = true;
    Pool& q = pool();
    {
        std::lock_guard<std::mutex> lk(q.mu);
        // only a block of this size: a handle that kept a larger one for its
        // life would hold more than it needs, and the next large copy would
        // allocate anew
        for (size_t i = q.n; i-- > 0;)
            if (q.idle[i].bytes == want) {
                p = q.remove(i).p;
                bytes = want;
                return SLOTH_OK;
            }
    }
    const hipError_t e = hipHostMalloc(&p, want, hipHostMallocPortable);
    if (e != hipSuccess) {
        p = nullptr;
        (void)hipGetLastError();
        return fail(SLOTH_ENOMEM, "hipHostMalloc(%zu bytes): %s", want, hipGetErrorString(e));
    }
    bytes = want;
    return SLOTH_OK;
}

void PinLease::end()
{
    if (!p) return;
    if (busy) (void)hipStreamSynchronize(stream);
    const Block own{p, bytes};
    p = nullptr;
    Pool& q = pool();
    std::array<Block, std::tuple_size<decltype(q.idle)>::value> out;   // freed, those longest idle
    size_t n_out = 0;
    {
        std::lock_guard<std::mutex> lk(q.mu);
        if (q.users > 0 && own.bytes <= PIN_POOL_BYTES) {
            while (q.n == q.idle.size() || q.bytes + own.bytes > PIN_POOL_BYTES) out[n_out++] = q.remove(0);
            q.idle[q.n++] = own;
            q.bytes += own.bytes;
        } else {
            out[n_out++] = own;
        }
    }
    for (size_t i = 0; i < n_out; ++i) (void)hipHostFree(out[i].p);
}

int copy_in(const Span* spans, int n, PinLease& lease, hipStream_t s)
{
    size_t total = 0;
    for (int i = 0; i < n; ++i) total += (spans[i].bytes + 255) & ~(size_t)255;
    int rc = lease.take(total, s);
    if (rc) return rc;
    uint8_t* at = lease.as<uint8_t>();
    for (int i = 0; i < n; ++i) {
        if (!spans[i].bytes) continue;
        memcpy(at, spans[i].host, spans[i].bytes);
        HIP_TRY(hipMemcpyAsync(spans[i].dev, at, spans[i].bytes, hipMemcpyHostToDevice, s));
        at += (spans[i].bytes + 255) & ~(size_t)255;
    }
    return SLOTH_OK;
}

// One thread empties pinned memory that the device has just written at about
// 30 GB/s, and at 14 GB/s into memory that was never touched; the link
// carries 57 GB/s.  So from COPY_SHARED bytes on, COPY_THREADS threads share
// that, and start (25 us) while the work before the copy and the copy itself
// run.  Up to COPY_LONG bytes everything lands in one pinned block; longer
// copies go in pieces of COPY_SLOT through two slots a thread, one filled
// while the other is emptied.  (2.4 MB of a 640x480 frame: runtime's pageable
// copies 140 us, one block and one thread 127, this 85.)
static constexpr size_t COPY_SHARED = 1u << 20;
static constexpr size_t COPY_LONG = 8u << 20;
static constexpr size_t COPY_SLOT = 2u << 20;
static constexpr int COPY_THREADS = 4;

// Calls work(w) for w < n on as many threads, the caller's among them.
template <class F, class G>
static void on_threads(int n, F&& work, G&& before_own)
{
    std::array<std::thread, COPY_THREADS> th;
    bool own[COPY_THREADS] = {};
    for (int w = 1; w < n; ++w) {
        try {
            th[w] = std::thread(work, w);
        } catch (...) {
            own[w] = true;   // no thread to be had: this one does its share
        }
    }
    before_own();
    work(0);
    for (int w = 1; w < n; ++w) {
        if (own[w]) work(w);
        else th[w].join();
    }
}

// A value that one thread sets and others wait for: awake for as long as a
// short render and its copy take (a thread that sleeps is back tens of
// microseconds late), asleep from then on (the stream may hold any amount of
// work).
class Gate {
  public:
    int wait()
    {
        const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(200);
        while (!value.load(std::memory_order_acquire)) {
            if (std::chrono::steady_clock::now() >= until) {
                std::unique_lock<std::mutex> lk(mu);
                set.wait(lk, [&] { return value.load(std::memory_order_relaxed) != 0; });
                break;
            }
            std::this_thread::yield();
        }
        return value.load(std::memory_order_acquire);
    }
    void open(int v)
    {
        {
            std::lock_guard<std::mutex> lk(mu);
            value.store(v, std::memory_order_release);
        }
        set.notify_all();
    }

  private:
    std::atomic<int> value{0};
    std::mutex mu;
    std::condition_variable set;
};

static size_t room(size_t n) { return (n + 255) & ~(size_t)255; }

// All spans through one pinned block of `total` bytes.
static int copy_out_block(const Span* spans, int n, size_t total, hipStream_t s)
{
    PinLease lease;
    int rc = lease.take(total, s);
    if (rc) return rc;
    uint8_t* block = lease.as<uint8_t>();
    size_t at = 0;
    for (int i = 0; i < n; at += room(spans[i++].bytes))
        if (spans[i].bytes)
            HIP_TRY(hipMemcpyAsync(block + at, spans[i].dev, spans[i].bytes, hipMemcpyDeviceToHost, s));
    // bytes [lo, hi) of the block
    auto empty = [&](size_t lo, size_t hi) {
        size_t b = 0;
        for (int i = 0; i < n; b += room(spans[i++].bytes)) {
            const size_t x = std::max(lo, b), y = std::min(hi, b + spans[i].bytes);
            if (x < y) memcpy((uint8_t*)spans[i].host + (x - b), block + x, y - x);
        }
    };
    hipError_t e = hipSuccess;
    if (total < COPY_SHARED) {
        e = hipStreamSynchronize(s);
        if (e == hipSuccess) empty(0, total);
    } else {
        Gate there;   // 1: the block is filled, 2: it never will be
        on_threads(
            COPY_THREADS,
            [&](int w) {
                if (there.wait() == 1)
                    empty(total * (size_t)w / COPY_THREADS, total * (size_t)(w + 1) / COPY_THREADS);
            },
            [&] {
                e = hipStreamSynchronize(s);
                there.open(e == hipSuccess ? 1 : 2);
            });
    }
    HIP_TRY(e);
    lease.done();
    return SLOTH_OK;
}

int copy_out(const Span* spans, int n, hipStream_t s)
{
    size_t total = 0;
    for (int i = 0; i < n; ++i) total += room(spans[i].bytes);
    if (total <= COPY_LONG) return copy_out_block(spans, n, total, s);

    PinLease lease;
    int rc = lease.take((size_t)COPY_THREADS * 2 * COPY_SLOT, s);
    if (rc) return rc;
    int dev = 0;
    HIP_TRY(hipGetDevice(&dev));
    std::array<hipEvent_t, 2 * COPY_THREADS> ev{};
    std::atomic<int> bad{(int)hipSuccess};
    auto note = [&](hipError_t e) {
        if (e != hipSuccess) bad.store((int)e);
        return e == hipSuccess;
    };
    for (hipEvent_t& v : ev)
        if (!note(hipEventCreateWithFlags(&v, hipEventDisableTiming))) v = nullptr;
    // piece k of the spans in order, each span cut on its own
    size_t pieces = 0;
    for (int i = 0; i < n; ++i) pieces += (spans[i].bytes + COPY_SLOT - 1) / COPY_SLOT;
    auto piece = [&](size_t k) {
        int i = 0;
        for (;; ++i) {
            const size_t c = (spans[i].bytes + COPY_SLOT - 1) / COPY_SLOT;
            if (k < c) break;
            k -= c;
        }
        const size_t at = k * COPY_SLOT;
        return Span{(uint8_t*)spans[i].host + at, (uint8_t*)spans[i].dev + at, std::min(COPY_SLOT, spans[i].bytes - at)};
    };
    // thread w takes pieces w, w + COPY_THREADS, ... through its own two slots
    auto slot = [&](int w, int q) { return lease.as<uint8_t>() + (size_t)(2 * w + q) * COPY_SLOT; };
    auto issue = [&](int w, size_t k, int q) {
        const Span c = piece(k);
        return note(hipMemcpyAsync(slot(w, q), c.dev, c.bytes, hipMemcpyDeviceToHost, s)) &&
               note(hipEventRecord(ev[2 * w + q], s));
    };
    Gate begun;   // 1: the first piece is there, 2: it never will be
    auto work = [&](int w) {
        if (begun.wait() != 1 || (w && !note(hipSetDevice(dev)))) return;
        int q = 0;
        for (size_t k = (size_t)w; k < pieces; k += COPY_THREADS, q ^= 1) {
            if (k + COPY_THREADS < pieces && !issue(w, k + COPY_THREADS, q ^ 1)) return;
            if (!note(hipEventSynchronize(ev[2 * w + q]))) return;
            const Span c = piece(k);
            memcpy(c.host, slot(w, q), c.bytes);
        }
    };
    // this thread alone waits for the work before the copy, with every
    // thread's first piece enqueued behind it
    auto begin = [&] {
        for (int w = 0; w < COPY_THREADS && (size_t)w < pieces; ++w)
            if (!issue(w, (size_t)w, 0)) break;
        if (bad.load() == (int)hipSuccess) note(hipEventSynchronize(ev[0]));
        begun.open(bad.load() == (int)hipSuccess ? 1 : 2);
    };
    if (bad.load() == (int)hipSuccess) on_threads(COPY_THREADS, work, begin);
    const hipError_t e = (hipError_t)bad.load();
    if (e == hipSuccess) lease.done();   // every piece has been waited for
    for (hipEvent_t v : ev)
        if (v) (void)hipEventDestroy(v);
    HIP_TRY(e);
    return SLOTH_OK;
}

}  // namespace sloth
