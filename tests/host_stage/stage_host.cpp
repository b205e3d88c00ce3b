// The host side of the transfers (csrc/sloth_stage.hip) with a HIP runtime of
// the few functions it calls: "device" memory is host memory, copies happen at
// once, and allocations are counted.  argv[1] names the check.
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime.h>

#include <chrono>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <ctime>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "sloth_stage.hip"

using namespace sloth;

static std::mutex mu;
static std::map<void*, size_t> pinned;
static int allocations = 0;
// the stream's work lasts until then; a waiting thread is awake, as it is in
// the runtime
static std::chrono::steady_clock::time_point busy_until;
static void wait_for_stream()
{
    while (std::chrono::steady_clock::now() < busy_until) std::this_thread::yield();
}

int sloth::fail(int code, const char* fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vfprintf(stderr, fmt, ap);
    va_end(ap);
    return code;
}

extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    std::lock_guard<std::mutex> lk(mu);
    *p = malloc(n);
    pinned[*p] = n;
    ++allocations;
    return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
    std::lock_guard<std::mutex> lk(mu);
    pinned.erase(p);
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t)
{
    wait_for_stream();
    return hipSuccess;
}
hipError_t hipGetDevice(int* d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    *e = (hipEvent_t)1;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t)
{
    wait_for_stream();
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
}

#define CHECK(c)                                                \
    do {                                                        \
        if (!(c)) {                                             \
            printf("line %d: %s\n", __LINE__, #c);              \
            return 1;                                           \
        }                                                       \
    } while (0)

static size_t all_pinned()
{
    size_t n = 0;
    for (auto& b : pinned) n += b.second;
    return n;
}

// A read-back's large block stays with the pool when a handle then takes a
// small one for its life, and the next read-back finds it there.
static int small_lease()
{
    PinPoolUser user;
    std::vector<uint8_t> src(12u << 20, 7), dst(src.size());
    const Span s{dst.data(), src.data(), src.size()};
    CHECK(copy_out(&s, 1, nullptr) == SLOTH_OK && dst == src);
    PinLease handle;
    CHECK(handle.take(40000, nullptr) == SLOTH_OK);
    handle.done();
    CHECK(pinned.at(handle.p) <= 2 * 65536);
    const int before = allocations;
    std::fill(dst.begin(), dst.end(), 0);
    CHECK(copy_out(&s, 1, nullptr) == SLOTH_OK && dst == src);
    CHECK(allocations == before);
    return 0;
}

// Idle blocks stay within the pool's bytes, and a size in use is kept in
// place of sizes that no longer are.
static int pool_bound()
{
    {
        PinPoolUser user;
        for (size_t n = 65536; n <= (64u << 20); n *= 2) {
            PinLease a, b;
            CHECK(a.take(n, nullptr) == SLOTH_OK && b.take(n, nullptr) == SLOTH_OK);
        }
        CHECK(all_pinned() <= PIN_POOL_BYTES);
        for (int k = 0; k < 2; ++k) {
            const int before = allocations;
            PinLease a;
            CHECK(a.take(3u << 20, nullptr) == SLOTH_OK);
            if (k) CHECK(allocations == before);
        }
        CHECK(all_pinned() <= PIN_POOL_BYTES);
        PinLease over;   // more than the pool keeps
        CHECK(over.take(PIN_POOL_BYTES + 1, nullptr) == SLOTH_OK);
    }
    CHECK(pinned.empty());
    return 0;
}

// A read-back behind a long render leaves the processors to others: the
// copying threads sleep until there is something to copy.
static int waits_asleep(size_t bytes)
{
    PinPoolUser user;
    std::vector<uint8_t> src(bytes), dst(src.size());
    for (size_t i = 0; i < src.size(); ++i) src[i] = (uint8_t)(i * 7 + (i >> 12));
    const Span s{dst.data(), src.data(), src.size()};
    CHECK(copy_out(&s, 1, nullptr) == SLOTH_OK && dst == src);
    std::fill(dst.begin(), dst.end(), 0);
    busy_until = std::chrono::steady_clock::now() + std::chrono::milliseconds(400);
    const clock_t t0 = clock();   // of all threads
    CHECK(copy_out(&s, 1, nullptr) == SLOTH_OK);
    const double used = (double)(clock() - t0) / CLOCKS_PER_SEC;
    CHECK(dst == src);
    printf("%.3f s of processor time in a wait of 0.4 s\n", used);
    CHECK(used < 0.6);   // one thread's wait
    return 0;
}

int main(int argc, char** argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "small_lease") return small_lease();
    if (what == "pool_bound") return pool_bound();
    if (what == "waits_asleep") return waits_asleep(4u << 20);
    if (what == "waits_asleep_long") return waits_asleep((33u << 20) + 5);
    return 2;
}
