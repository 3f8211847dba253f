// Host check of vh::HostCopy with the HIP calls replaced by host ones: a status
// read by another thread while a download waits does not change what the
// download reports, and neither mixes with the other's data.
#include <hip/hip_runtime.h>

#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <thread>
#include <vector>

#include "../cpu-vh_amd/csrc/vh_hostcopy.hpp"

static std::function<void()> g_on_wait;  // called once, by the wait after the download copied the words
static std::atomic<int> g_small{0};      // copies of the error words so far

extern "C" {
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    return (*p = std::malloc(n)) ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = nullptr; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) {
    if (g_on_wait && g_small.load() > 0) {
        auto f = g_on_wait;
        g_on_wait = nullptr;
        f();
    }
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    if (n == 3 * sizeof(int)) ++g_small;
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *) {
    a->type = hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
}

int main() {
    const int good[3] = {0, 0, 0}, bad[3] = {1, 0, 0};
    std::vector<double> src(1000), out(1000, -1.0);
    for (size_t i = 0; i < src.size(); ++i) src[i] = 0.5 * (double)i;
    vh::HostCopy hc;
    if (hc.init(300) != hipSuccess) return 2;  // a download of four chunks
    bool mine = true, theirs = false;
    std::thread other;
    g_on_wait = [&] {
        other = std::thread([&] { (void)hc.status(bad, nullptr, &theirs); });
        for (int k = 0; k < 100 && g_small.load() < 2; ++k) std::this_thread::sleep_for(std::chrono::milliseconds(1));
    };
    const hipError_t r = hc.fetch(out.data(), src.data(), src.size(), good, nullptr, &mine);
    other.join();
    std::vector<float> hi(1000, 0.25f), lo(1000, 0.125f);
    bool err = true;
    const hipError_t w = hc.fetch_widened(out.data() + 500, hi.data(), lo.data(), 500, good, nullptr, &err);
    bool data = true;
    for (size_t i = 0; i < 1000; ++i) data = data && out[i] == (i < 500 ? src[i] : 0.375);
    std::printf("download %d mine %d theirs %d widened %d err %d data %d\n", (int)r, (int)mine, (int)theirs, (int)w,
                (int)err, (int)data);
    hc.release();
    return r == hipSuccess && !mine && theirs && w == hipSuccess && !err && data ? 0 : 1;
}
