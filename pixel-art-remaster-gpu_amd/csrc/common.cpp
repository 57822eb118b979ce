// common.cpp -- last-error storage and device probing.
#include "common.hpp"

#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <thread>

namespace {
thread_local char g_last_error[512] = "";
}

namespace dpx {

int fail(int code, const char* fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_last_error, sizeof(g_last_error), fmt, ap);
    va_end(ap);
    return code;
}

int require_device()
{
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n <= 0) return fail(DPX_ENODEV, "no GPU visible to this process (%s)", hipGetErrorString(e));
    return DPX_OK;
}

// The runtime copies to memory that is not pinned at 18 GB/s: its own pinned
// blocks, emptied by the calling thread.  Here blocks of kChunk go through
// kSlots pinned slots (the link gives 55 GB/s) and kWorkers threads empty
// them meanwhile: a 256x224 frame's diagram, 20.6 MB, in 530 us instead of
// 1155.  The slots are kept (a pinned allocation takes longer than the copy)
// and freed when the library is unloaded; a call that finds them in use, or
// cannot have them or a thread, copies as before.  So does one whose
// destination the runtime knows: memory that is pinned already takes the
// link's rate directly (a 640x480 frame at 8x, 78.6 MB: 2.2 ms a call, through
// the slots 2.6 to 7.8, by the cores the threads get).
namespace {

constexpr size_t kChunk = 4 << 20, kSlots = 2, kDownloadMin = 4 << 20;
constexpr int kWorkers = 3;

struct Staging {
    std::mutex mu;
    char* pin = nullptr;
    ~Staging()
    {
        if (pin) (void)hipHostFree(pin);
    }
};

Staging& staging()
{
    static Staging s;
    return s;
}

// Is p the runtime's own memory (pinned, managed, a device's)?
bool known(const void* p)
{
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return false;
}

}  // namespace

hipError_t download(void* dst, const void* src, size_t n)
{
    if (n < kDownloadMin || known(dst)) return hipMemcpy(dst, src, n, hipMemcpyDeviceToHost);
    Staging& st = staging();
    std::unique_lock<std::mutex> lock(st.mu, std::try_to_lock);
    if (!lock.owns_lock()) return hipMemcpy(dst, src, n, hipMemcpyDeviceToHost);
    if (!st.pin && hipHostMalloc((void**)&st.pin, kChunk * kSlots, hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        st.pin = nullptr;
        return hipMemcpy(dst, src, n, hipMemcpyDeviceToHost);
    }
    const size_t chunks = (n + kChunk - 1) / kChunk;
    auto bytes = [&](size_t k) { return std::min(kChunk, n - k * kChunk); };
    std::atomic<size_t> ready{ 0 };          // chunks in their slots
    std::atomic<size_t> copied[kSlots] = {};  // parts copied out of a slot
    std::atomic<size_t> parts{ 0 };          // of a chunk, one a worker; 0 until their number is known
    auto work = [&](size_t w) {
        size_t p;
        while ((p = parts.load(std::memory_order_acquire)) == 0) std::this_thread::yield();
        for (size_t k = 0; k < chunks; k++) {
            while (ready.load(std::memory_order_acquire) <= k) std::this_thread::yield();
            const size_t at = bytes(k) * w / p, end = bytes(k) * (w + 1) / p;
            memcpy((char*)dst + k * kChunk + at, st.pin + k % kSlots * kChunk + at, end - at);
            copied[k % kSlots].fetch_add(1, std::memory_order_release);
        }
    };
    std::thread workers[kWorkers];
    size_t started = 0;
    try {
        for (; started < kWorkers; started++) workers[started] = std::thread(work, started);
    } catch (...) {
    }
    if (!started) return hipMemcpy(dst, src, n, hipMemcpyDeviceToHost);
    parts.store(started, std::memory_order_release);
    hipError_t rc = hipSuccess;
    for (size_t k = 0; k < chunks; k++) {
        while (copied[k % kSlots].load(std::memory_order_acquire) < k / kSlots * started) std::this_thread::yield();
        if (rc == hipSuccess)
            rc = hipMemcpy(st.pin + k % kSlots * kChunk, (const char*)src + k * kChunk, bytes(k), hipMemcpyDeviceToHost);
        ready.store(k + 1, std::memory_order_release);  // (after an error too: the workers end)
    }
    for (size_t w = 0; w < started; w++) workers[w].join();
    return rc;
}

}  // namespace dpx

extern "C" const char* dpx_last_error(void) { return g_last_error; }

extern "C" const char* dpx_version(void) { return "depixel-mi355x 0.1 (gfx950)"; }
