// The host side of the tiled plan (csrc/sloth_tiled.hip) with a HIP runtime
// whose memory is host memory and whose launches are recorded.  The binning
// kernels are played by launched(): a render meets `careful` careful triangles
// and boxes that ask for `wraps` odd tile columns.  argv[1] names the check.
#include <cxxabi.h>

#include <cstdarg>
#include <cstdio>
#include <map>
#include <string>

#include "sloth_tiled.hip"

using namespace sloth;

static uint32_t careful = 0, wraps = 0;   // of the scene
struct Launch {
    std::string name;
    dim3 grid;
};
static std::vector<Launch> launches;
static std::map<const void*, std::string> names;

int sloth::fail(int code, const char* fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vfprintf(stderr, fmt, ap);
    va_end(ap);
    return code;
}

static void launched(const std::string& name, dim3 grid, void** a)
{
    launches.push_back({name, grid});
    auto u32 = [&](int i) { return *(uint32_t*)a[i]; };
    if (name.find("k_tile_clear(") != std::string::npos) {
        memset(*(uint32_t**)a[4], 0, u32(5) * sizeof(uint32_t));
        memset(*(uint32_t**)a[6], 0, (WRAP_CNT + 1) * sizeof(uint32_t));
    } else if (name.find("k_bin<true") != std::string::npos) {
        uint32_t* cnt = *(uint32_t**)a[10];
        cnt[0] = careful;
        cnt[WRAP_CNT] = wraps;
    } else if (name.find("k_bin<false") != std::string::npos) {
        if (careful > u32(12) || wraps > u32(14)) (*(uint32_t**)a[9])[0] = 1u;
    }
}

struct _hipCall {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
};
static _hipCall call;

extern "C" {
void** __hipRegisterFatBinary(const void*)
{
    static void* h;
    return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* device_name, unsigned, void*, void*, dim3*, dim3*,
                           int*)
{
    int status = 0;
    char* d = abi::__cxa_demangle(device_name, nullptr, nullptr, &status);
    names[f] = d ? d : device_name;
    free(d);
}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s)
{
    call = {grid, block, lds, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s)
{
    *grid = call.grid;
    *block = call.block;
    *lds = call.lds;
    *s = call.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void** args, size_t, hipStream_t)
{
    launched(names[f], grid, args);
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n)
{
    *p = calloc(n, 1);
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
}

#define CHECK(c)                                   \
    do {                                           \
        if (!(c)) {                                \
            printf("line %d: %s\n", __LINE__, #c); \
            return 1;                              \
        }                                          \
    } while (0)

// One frame of one draw, planned, sized and rendered as a job does it.
struct Scene {
    TiledPlan plan;
    std::vector<Frame> frames;
    std::vector<Draw> draws;
    uint32_t flag = 0;
    int sizings = 0;
    Scene(uint32_t W, uint32_t H)
    {
        frames.assign(1, Frame{});
        draws.assign(1, Draw{});
        frames[0].W = W;
        frames[0].H = H;
        frames[0].draw_end = 1;
        frames[0].n_tris = draws[0].n = 1000000;
        plan.overflow = &flag;
    }
    int size()
    {
        ++sizings;
        return plan.size(frames, draws, frames.data(), draws.data(), nullptr);
    }
    int render()
    {
        int rc = plan.plan(frames, draws, frames[0].H);
        if (!rc && !plan.sized) rc = size();
        for (int attempt = 0; !rc && attempt < 4; ++attempt) {
            launches.clear();
            rc = plan.launch(frames, draws, frames.data(), draws.data(), nullptr, 0, 1, nullptr, nullptr, nullptr, false,
                             1, nullptr, nullptr);
            bool ovf = false;
            if (!rc) rc = plan.overflowed(1, nullptr, ovf);
            if (rc || !ovf) return rc;
            plan.outgrow();
            rc = size();
        }
        return rc ? rc : -1;
    }
};
static const Launch* find(const char* what)
{
    for (const Launch& l : launches)
        if (l.name.find(what) != std::string::npos) return &l;
    return nullptr;
}

// The careful list's launch follows the sizing of the present tiles, not the
// largest list that any tile size ever had.
static int careful_room()
{
    Scene sc(1920, 1080);
    CHECK(sc.plan.set_tile(16, 8) == SLOTH_OK);
    careful = 200000;
    CHECK(sc.render() == SLOTH_OK && find("k_careful<false") && find("k_careful<false")->grid.x == 4096);
    CHECK(sc.plan.set_tile(128, 32) == SLOTH_OK);
    careful = 100;
    CHECK(sc.render() == SLOTH_OK && find("k_careful<false"));
    CHECK(find("k_careful<false")->grid.x == (100 + 50 + 1024 + 3) / 4);
    CHECK(sc.plan.set_tile(64, 32) == SLOTH_OK);
    careful = 0;
    CHECK(sc.render() == SLOTH_OK && !find("k_careful<false"));
    // careful triangles come later: sized again, and there is room from then on
    for (uint32_t n : {1, 300, 0, 1000, 5}) {
        careful = n;
        CHECK(sc.render() == SLOTH_OK && find("k_careful<false"));
    }
    CHECK(sc.sizings == 4);
    careful = 5000;
    CHECK(sc.render() == SLOTH_OK && sc.sizings == 5);
    return 0;
}

// Odd widths: a view whose wrapped boxes reach further and further is sized
// again a few times, not for each tile column; any other sizing has the columns
// that the scene needs and no more.
static int odd_reach()
{
    Scene sc(1919, 1079);
    CHECK(sc.plan.set_tile(64, 32) == SLOTH_OK);
    careful = 0;
    wraps = 2;
    CHECK(sc.render() == SLOTH_OK && sc.sizings == 1 && sc.plan.odd_cols() == 2);
    for (wraps = 2; wraps <= 30; ++wraps) {
        CHECK(sc.render() == SLOTH_OK && sc.plan.odd_cols() >= wraps);
        CHECK(find("k_tile_edges")->grid.y <= 30);   // the frame has 30 columns
    }
    printf("%d sizings\n", sc.sizings);
    CHECK(sc.sizings <= 8);
    careful = 7;   // outgrown for another reason
    for (uint32_t w : {1, 0, 17}) {
        wraps = w;
        sc.plan.outgrow();
        CHECK(sc.size() == SLOTH_OK && sc.plan.odd_cols() == (w == 17 ? 22 : w));
    }
    CHECK(sc.plan.set_tile(128, 16) == SLOTH_OK);   // other tiles: sized for what is there
    wraps = 9;
    CHECK(sc.render() == SLOTH_OK && sc.plan.odd_cols() == 9);
    return 0;
}

int main(int argc, char** argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "careful_room") return careful_room();
    if (what == "odd_reach") return odd_reach();
    return 2;
}
