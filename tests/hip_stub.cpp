// A stand-in for the HIP runtime calls of scene creation, in host memory, for test_scene_fallback.py: loaded
// with global visibility before libzombie_amd.so, its symbols are the ones that the library binds to.
// Device memory is limited, launches do nothing or are refused, and one operator new can be made to fail.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <new>

namespace {
constexpr int kSuccess = 0, kOutOfMemory = 2, kInvalidConfiguration = 9;
int64_t limitBytes = INT64_MAX, liveBytes = 0, peakBytes = 0;
uint64_t largestLaunch = 0;   // threads
int refuseLaunches = 0, lastError = kSuccess;
int64_t mallocsUntilNewFails = -1;
bool newFails = false;
struct Dim3 { uint32_t x, y, z; };
Dim3 pushedGrid, pushedBlock;
std::map<void*, int64_t>& sizes() { static auto* m = new std::map<void*, int64_t>(); return *m; }
int fail(int e) { lastError = e; return e; }
}  // namespace

extern "C" {
void stub_reset(int64_t limit, int refuse, int64_t mallocs) {
    limitBytes = limit; refuseLaunches = refuse; mallocsUntilNewFails = mallocs; newFails = false;
    largestLaunch = 0; lastError = kSuccess; peakBytes = liveBytes;
}
int64_t stub_live_bytes() { return liveBytes; }
int64_t stub_peak_bytes() { return peakBytes; }
uint64_t stub_largest_launch() { return largestLaunch; }
int stub_last_error() { return lastError; }

int hipGetDevice(int* d) { *d = 0; return kSuccess; }
int hipMalloc(void** p, size_t n) {
    if (liveBytes + (int64_t)n > limitBytes) return fail(kOutOfMemory);
    *p = std::malloc(n);
    sizes()[*p] = (int64_t)n;
    liveBytes += (int64_t)n;
    if (liveBytes > peakBytes) peakBytes = liveBytes;
    if (mallocsUntilNewFails > 0 && --mallocsUntilNewFails == 0) newFails = true;
    return kSuccess;
}
int hipFree(void* p) {
    auto it = sizes().find(p);
    if (it == sizes().end()) return fail(1);
    liveBytes -= it->second;
    sizes().erase(it);
    std::free(p);
    return kSuccess;
}
int hipMemcpy(void* d, const void* s, size_t n, int) { std::memcpy(d, s, n); return kSuccess; }
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t, void*) { pushedGrid = g; pushedBlock = b; return kSuccess; }
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* shared, void** stream) {
    *g = pushedGrid; *b = pushedBlock; *shared = 0; *stream = nullptr;
    return kSuccess;
}
int hipLaunchKernel(const void*, Dim3 g, Dim3 b, void**, size_t, void*) {
    const uint64_t threads = (uint64_t)g.x * g.y * g.z * b.x * b.y * b.z;
    if (threads > largestLaunch) largestLaunch = threads;
    return refuseLaunches ? fail(kInvalidConfiguration) : kSuccess;
}
int hipStreamSynchronize(void*) { return kSuccess; }
int hipGetLastError() { int e = lastError; lastError = kSuccess; return e; }
const char* hipGetErrorString(int) { return "stub"; }
}

void* operator new(size_t n) {
    if (newFails) { newFails = false; throw std::bad_alloc(); }
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }
