// Host double of the HIP runtime calls libbh_hip.so makes, for tests of its host
// code without a GPU (test_host_paths.py): loaded with RTLD_GLOBAL before the
// library, whose references then bind to these. Device memory is host memory,
// kernels do nothing, copies happen at once; what the runtime would still be
// working on until the next wait is kept as counts.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <dirent.h>
#include <new>
#include <thread>

namespace {
constexpr int kOk = 0, kError = 1;
std::atomic<long> ticks{0};        // one per kernel: the clock of the events
std::atomic<int> kernels{0};       // launched since the last wait
std::atomic<int> uploads{0};       // host arrays copied from since the last wait
std::atomic<int> copies{0};        // host-to-device copies so far
std::atomic<int> fail_copy{-1};    // the one of them that fails
std::atomic<int> news{0}, fail_new{-1};
std::atomic<size_t> live{0}, most{0}, base{0};  // device bytes
std::atomic<int> waiting{0};       // most threads seen at a wait for kernels

int threads()
{
    int n = 0;
    if (DIR* d = opendir("/proc/self/task")) {
        while (const dirent* e = readdir(d))
            n += e->d_name[0] != '.';
        closedir(d);
    }
    return n;
}

int wait()
{
    if (kernels > 0)
        waiting = std::max(waiting.load(), threads());
    kernels = 0;
    uploads = 0;
    return kOk;
}

struct Dim {
    uint32_t x, y, z;
};
struct Launch {
    Dim grid, block;
    size_t lds;
    void* stream;
};
thread_local Launch pending_launch;
thread_local int last_error = kOk;
}  // namespace

void* operator new(size_t n)
{
    if (fail_new >= 0 && news++ == fail_new)
        throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1))
        return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

extern "C" {

// -- what the tests set and read
void fake_fail_copy(int k) { copies = 0, fail_copy = k; }
void fake_fail_new(int k) { news = 0, fail_new = k; }
int fake_uploads() { return uploads; }
int fake_kernels() { return kernels; }
int fake_threads() { return threads(); }
int fake_waiting_threads() { return waiting; }
void fake_mark_memory() { base = live.load(), most = live.load(); }
size_t fake_extra_memory() { return most - base; }

// -- the runtime
int __hipPushCallConfiguration(Dim grid, Dim block, size_t lds, void* stream)
{
    pending_launch = {grid, block, lds, stream};
    return kOk;
}
int __hipPopCallConfiguration(Dim* grid, Dim* block, size_t* lds, void** stream)
{
    *grid = pending_launch.grid, *block = pending_launch.block;
    *lds = pending_launch.lds, *stream = pending_launch.stream;
    return kOk;
}
int hipLaunchKernel(const void*, Dim, Dim, void**, size_t, void*)
{
    ++ticks, ++kernels;
    return kOk;
}
int hipGetDeviceCount(int* n) { return *n = 1, kOk; }
int hipGetDevice(int* d) { return *d = 0, kOk; }
int hipGetDevicePropertiesR0600(void*, int) { return kError; }
const char* hipGetErrorString(int) { return "injected"; }
int hipGetLastError()
{
    const int e = last_error;
    last_error = kOk;
    return e;
}
int hipMalloc(void** p, size_t n)
{
    size_t* q = static_cast<size_t*>(std::calloc(n + 64, 1));
    if (!q)
        return kError;
    *q = n;
    live += n;
    most = std::max(most.load(), live.load());
    *p = q + 8;
    return kOk;
}
int hipFree(void* p)
{
    if (p) {
        size_t* q = static_cast<size_t*>(p) - 8;
        live -= *q;
        std::free(q);
    }
    return kOk;
}
int hipHostMalloc(void** p, size_t n, unsigned) { return (*p = std::calloc(n, 1)) ? kOk : kError; }
int hipHostFree(void* p) { return std::free(p), kOk; }
int hipMemsetAsync(void* p, int v, size_t n, void*) { return std::memset(p, v, n), kOk; }
int hipMemset(void* p, int v, size_t n) { return std::memset(p, v, n), kOk; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void*)
{
    if (kind == 1) {  // host to device
        if (copies++ == fail_copy)
            return kError;
        ++uploads;
    }
    std::memcpy(d, s, n);
    return kOk;
}
int hipMemcpy(void* d, const void* s, size_t n, int) { return std::memcpy(d, s, n), wait(); }
int hipStreamCreateWithFlags(void** s, unsigned) { return *s = std::malloc(1), kOk; }
int hipStreamDestroy(void* s) { return std::free(s), kOk; }
int hipStreamSynchronize(void*) { return wait(); }
int hipStreamWaitEvent(void*, void*, unsigned) { return kOk; }
int hipEventCreate(void** e) { return *e = new long(-1), kOk; }  // not recorded
int hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void* e) { return delete static_cast<long*>(e), kOk; }
int hipEventRecord(void* e, void*) { return *static_cast<long*>(e) = ticks, kOk; }
int hipEventSynchronize(void*)
{
    if (kernels > 0)  // a worker that waits for them is there by now
        std::this_thread::sleep_for(std::chrono::milliseconds(20));
    return wait();
}
int hipEventElapsedTime(float* ms, void* a, void* b)
{
    const long x = *static_cast<long*>(a), y = *static_cast<long*>(b);
    if (x < 0 || y < 0)
        return last_error = kError;  // and the thread's last error, as the runtime keeps it
    *ms = static_cast<float>(y - x);
    return kOk;
}
}
