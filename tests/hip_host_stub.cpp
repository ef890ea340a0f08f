// The HIP runtime calls of libflipgpu.so over host memory, for tests of its
// host code without a device: allocations are counted (and refused beyond a
// limit), copies and fills done at once, kernels not run (what they would have
// written stays as it was, zero at first).  A stream counts what was queued on
// it and what has been waited for.  A chosen launch can be made to fail.
// Launches are counted by kernel.  Loaded ahead of the library with its symbols global (test_host_runtime.py).
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <string>

namespace {
struct Stream {
    long queued = 0, done = 0;
};
struct Event {
    Stream* stream = nullptr;
    long mark = 0;
};
struct Dim3 {
    uint32_t x, y, z;
};
struct Config {
    Dim3 grid, block;
    size_t lds;
    Stream* stream;
};
constexpr int kOutOfMemory = 2, kInvalidConfiguration = 9, kLaunchFailure = 719;
std::mutex mu;
std::map<void*, uint64_t> device, pinned;
std::set<Stream*> streams;
std::map<const void*, std::string> kernels;
std::map<const void*, long> launches;
uint64_t device_bytes = 0, limit = ~0ull;
long fail_launch = -1;   // launches until one fails
thread_local int last_error = 0;
thread_local Config config;

int error(int e) { return last_error = e; }
int queue(Stream* s)
{
    std::lock_guard<std::mutex> lock(mu);
    s->queued++;
    return 0;
}
int launch(const void* f, Dim3 g, Dim3 b, Stream* s)
{
    {
        std::lock_guard<std::mutex> lock(mu);
        launches[f]++;
        if (fail_launch >= 0 && fail_launch-- == 0) return error(kLaunchFailure);
    }
    if (!g.x || !g.y || !g.z || !b.x || !b.y || !b.z || b.x * b.y * b.z > 1024) return error(kInvalidConfiguration);
    return queue(s);
}
}  // namespace

extern "C" {
// the tests' side
uint64_t stub_device_bytes() { return device_bytes; }
uint64_t stub_allocations() { return device.size() + pinned.size(); }
void stub_limit(uint64_t bytes) { limit = bytes; }
void stub_fail_launch(long n) { fail_launch = n; }
int stub_launch_failed() { return fail_launch == -1; }
// launches of the kernels whose (mangled) name holds `part` since the last reset
long stub_launches(const char* part)
{
    std::lock_guard<std::mutex> lock(mu);
    long n = 0;
    for (const auto& l : launches)
        if (kernels[l.first].find(part) != std::string::npos) n += l.second;
    return n;
}
void stub_reset_launches() { launches.clear(); }
int stub_busy_streams()
{
    std::lock_guard<std::mutex> lock(mu);
    int n = 0;
    for (Stream* s : streams) n += s->queued > s->done;
    return n;
}

// the runtime's
int hipGetDeviceCount(int* n) { return *n = 1, 0; }
int hipSetDevice(int) { return 0; }
int hipGetLastError()
{
    const int e = last_error;
    last_error = 0;
    return e;
}
const char* hipGetErrorString(int e) { return e == kOutOfMemory ? "out of memory" : e ? "error" : "no error"; }
int hipMalloc(void** p, size_t bytes)
{
    std::lock_guard<std::mutex> lock(mu);
    *p = nullptr;
    if (device_bytes + bytes > limit) return error(kOutOfMemory);
    *p = std::calloc(1, bytes ? bytes : 1);
    device[*p] = bytes;
    device_bytes += bytes;
    return 0;
}
int hipFree(void* p)
{
    std::lock_guard<std::mutex> lock(mu);
    for (Stream* s : streams) s->done = s->queued;
    if (!p) return 0;
    const auto it = device.find(p);
    if (it == device.end()) std::abort();
    device_bytes -= it->second;
    device.erase(it);
    std::free(p);
    return 0;
}
int hipHostMalloc(void** p, size_t bytes, unsigned)
{
    std::lock_guard<std::mutex> lock(mu);
    *p = std::calloc(1, bytes ? bytes : 1);
    pinned[*p] = bytes;
    return 0;
}
int hipHostFree(void* p)
{
    std::lock_guard<std::mutex> lock(mu);
    for (Stream* s : streams) s->done = s->queued;
    if (p && !pinned.erase(p)) std::abort();
    std::free(p);
    return 0;
}
int hipStreamCreateWithFlags(Stream** s, unsigned)
{
    std::lock_guard<std::mutex> lock(mu);
    streams.insert(*s = new Stream);
    return 0;
}
int hipStreamDestroy(Stream* s)
{
    std::lock_guard<std::mutex> lock(mu);
    streams.erase(s);
    delete s;
    return 0;
}
int hipStreamSynchronize(Stream* s)
{
    std::lock_guard<std::mutex> lock(mu);
    s->done = s->queued;
    return 0;
}
int hipEventCreateWithFlags(Event** e, unsigned) { return *e = new Event, 0; }
int hipEventCreate(Event** e) { return *e = new Event, 0; }
int hipEventDestroy(Event* e) { return delete e, 0; }
int hipEventRecord(Event* e, Stream* s)
{
    std::lock_guard<std::mutex> lock(mu);
    e->stream = s;
    e->mark = s->queued;
    return 0;
}
int hipEventSynchronize(Event* e)
{
    std::lock_guard<std::mutex> lock(mu);
    if (e->stream && e->stream->done < e->mark) e->stream->done = e->mark;
    return 0;
}
int hipEventElapsedTime(float* ms, Event*, Event*) { return *ms = 1.0f, 0; }
int hipMemcpyAsync(void* d, const void* s, size_t bytes, int, Stream* q) { return std::memmove(d, s, bytes), queue(q); }
int hipMemsetAsync(void* d, int v, size_t bytes, Stream* q) { return std::memset(d, v, bytes), queue(q); }
int hipMemsetD32Async(void* d, int v, size_t n, Stream* q)
{
    for (size_t k = 0; k < n; k++) static_cast<int*>(d)[k] = v;
    return queue(q);
}
int hipGetSymbolAddress(void** p, const void*)
{
    static void* const scratch = std::calloc(1, 64 << 20);
    return *p = scratch, 0;
}
int hipLaunchKernel(const void* f, Dim3 g, Dim3 b, void**, size_t, Stream* s) { return launch(f, g, b, s); }
int hipExtLaunchKernel(const void* f, Dim3 g, Dim3 b, void**, size_t, Stream* s, Event* a, Event* z, int)
{
    const int e = launch(f, g, b, s);
    if (a) hipEventRecord(a, s);
    if (z) hipEventRecord(z, s);
    return e;
}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t lds, Stream* s) { return config = Config{g, b, lds, s}, 0; }
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* lds, Stream** s)
{
    *g = config.grid;
    *b = config.block;
    *lds = config.lds;
    *s = config.stream;
    return 0;
}
void** __hipRegisterFatBinary(const void*)
{
    static void* handle = nullptr;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
    kernels[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
}
