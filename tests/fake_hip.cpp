// A stand-in for the HIP runtime on the host, for tests of the library's memory
// and copy code without a device: "device" memory is host memory of a settable
// total, kernels do nothing, copies happen at once, and a stream can be blocked
// so that waits for it last until it is released.  The library's own calls
// resolve to these when this is loaded (globally) before it.
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace {
struct Stream {
    bool blocked = false;
};
struct Event {
    Stream* on = nullptr;
};
std::mutex mu;
std::condition_variable cv;
std::map<void*, size_t> blocks, pinned;
std::vector<Stream*> streams;
size_t capacity = (size_t)1 << 40, used = 0;
int64_t n_malloc = 0, n_memcpy = 0;
thread_local int fail_new_after = -1;   // allocations of this thread until one fails (< 0: none does)

// the stand-in's own allocations do not count
struct Own {
    const int keep = fail_new_after;
    Own() { fail_new_after = -1; }
    ~Own() { fail_new_after = keep; }
};

constexpr int kOk = 0, kInvalid = 1, kNoMemory = 2, kNotReady = 600, kCaptureUnsupported = 900;
bool capturing = false, captures_ended = false;   // a stream capture under way elsewhere, and whether a call ended it

bool lives(Stream* s)
{
    for (Stream* x : streams)
        if (x == s) return true;
    return false;
}
int wait_for(Stream* s)
{
    std::unique_lock<std::mutex> lk(mu);
    cv.wait(lk, [s] { return !s || !lives(s) || !s->blocked; });
    return kOk;
}
int wait_for_all()
{
    std::unique_lock<std::mutex> lk(mu);
    cv.wait(lk, [] {
        for (Stream* s : streams)
            if (s->blocked) return false;
        return true;
    });
    return kOk;
}
}  // namespace

void* operator new(size_t n)
{
    if (fail_new_after >= 0 && fail_new_after-- == 0) throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

extern "C" {

// ---- what a test sets and asks
void fake_capacity(size_t bytes) { capacity = bytes; }
size_t fake_used() { return used; }
int64_t fake_mallocs() { return n_malloc; }
int64_t fake_memcpys() { return n_memcpy; }
void fake_fail_new(int after) { fail_new_after = after; }
int fake_n_streams() { return (int)streams.size(); }
void* fake_stream(int i) { return streams[i]; }
void fake_block(void* s, int on)
{
    {
        std::lock_guard<std::mutex> lk(mu);
        ((Stream*)s)->blocked = on != 0;
    }
    cv.notify_all();
}
void fake_capture(int on) { capturing = on != 0; }
int fake_captures_ended() { return captures_ended; }
// whether a device block starts with these bytes
int fake_holds(const void* p, size_t n)
{
    std::lock_guard<std::mutex> lk(mu);
    for (const auto& b : blocks)
        if (b.second >= n && std::memcmp(b.first, p, n) == 0) return 1;
    return 0;
}
void* fake_pinned(size_t n)
{
    Own own;
    std::lock_guard<std::mutex> lk(mu);
    void* p = std::calloc(n, 1);
    pinned[p] = n;
    return p;
}

// ---- the runtime
int hipGetDeviceCount(int* n) { return *n = 2, kOk; }
int hipGetDevice(int* d) { return *d = 0, kOk; }
int hipSetDevice(int) { return kOk; }
int hipGetLastError() { return kOk; }
const char* hipGetErrorString(int e) { return e == kNoMemory ? "out of memory" : "error"; }
int hipDeviceSynchronize()
{
    if (capturing) return captures_ended = true, kCaptureUnsupported;
    return wait_for_all();
}
int hipMalloc(void** p, size_t n)
{
    Own own;
    std::lock_guard<std::mutex> lk(mu);
    *p = nullptr;
    if (used + n > capacity) return kNoMemory;
    *p = std::calloc(n ? n : 1, 1);
    if (!*p) return kNoMemory;
    blocks[*p] = n;
    used += n;
    ++n_malloc;
    return kOk;
}
int hipFree(void* p)
{
    wait_for_all();
    std::lock_guard<std::mutex> lk(mu);
    auto it = blocks.find(p);
    if (it == blocks.end()) return kInvalid;
    used -= it->second;
    blocks.erase(it);
    std::free(p);
    return kOk;
}
int hipHostMalloc(void** p, size_t n, unsigned) { return *p = fake_pinned(n), *p ? kOk : kNoMemory; }
int hipHostFree(void* p)
{
    std::lock_guard<std::mutex> lk(mu);
    pinned.erase(p);
    std::free(p);
    return kOk;
}
int hipStreamCreateWithFlags(void** s, unsigned)
{
    Own own;
    std::lock_guard<std::mutex> lk(mu);
    streams.push_back(new Stream);
    *s = streams.back();
    return kOk;
}
int hipStreamDestroy(void* s)
{
    std::lock_guard<std::mutex> lk(mu);
    for (size_t i = 0; i < streams.size(); ++i)
        if (streams[i] == s) streams.erase(streams.begin() + (long)i);
    return kOk;   // (the object stays: events may point to it)
}
int hipStreamSynchronize(void* s) { return wait_for((Stream*)s); }
int hipStreamWaitEvent(void*, void*, unsigned) { return kOk; }
int hipStreamIsCapturing(void*, int* st) { return *st = 0, kOk; }
int hipEventCreate(void** e)
{
    Own own;
    return *e = new Event, kOk;
}
int hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void* e) { return delete (Event*)e, kOk; }
int hipEventRecord(void* e, void* s) { return ((Event*)e)->on = (Stream*)s, kOk; }
int hipEventSynchronize(void* e) { return wait_for(((Event*)e)->on); }
int hipEventQuery(void* e)
{
    std::lock_guard<std::mutex> lk(mu);
    Stream* s = ((Event*)e)->on;
    return s && lives(s) && s->blocked ? kNotReady : kOk;
}
int hipEventElapsedTime(float* ms, void*, void*) { return *ms = 1.f, kOk; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*)
{
    {
        std::lock_guard<std::mutex> lk(mu);
        ++n_memcpy;
    }
    std::memmove(d, s, n);
    return kOk;
}
int hipMemcpy(void* d, const void* s, size_t n, int) { return std::memmove(d, s, n), kOk; }
struct Attributes {
    int type, device;
    void *on_device, *on_host;
    int managed;
    unsigned flags;
};
int hipPointerGetAttributes(Attributes* a, const void* p)
{
    std::lock_guard<std::mutex> lk(mu);
    *a = Attributes{};
    for (const auto* m : {&blocks, &pinned})
        for (const auto& b : *m)
            if (p >= b.first && p < (const char*)b.first + b.second) a->type = m == &pinned ? 1 : 2;
    return kOk;
}
int hipFuncSetAttribute(const void*, int, int) { return kOk; }
struct dim3v {
    unsigned x, y, z;
};
int hipLaunchKernel(const void*, dim3v, dim3v, void**, size_t, void*) { return kOk; }

}  // extern "C"
