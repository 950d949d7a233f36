// capi_memory.hip -- a context's device blocks and its copies between device
// memory and a caller's pageable arrays.
#include <sched.h>

#include <algorithm>
#include <cstring>

#include "capi_internal.h"

namespace bs2e {

// ---------------------------------------------------------------------------
// device blocks
// ---------------------------------------------------------------------------
namespace {
thread_local int t_quiet_depth = 0;
thread_local bool t_quiet = false;   // nothing uses what this scope releases any more
}  // namespace

QuietScope::QuietScope(bool waited) : waited_(waited), outer_(t_quiet)
{
    ++t_quiet_depth;
    if (waited) t_quiet = true;
}
QuietScope::~QuietScope()
{
    if (--t_quiet_depth == 0) t_quiet = false;
    else if (waited_) t_quiet = outer_;   // (said of this scope's blocks only)
}

namespace {
std::mutex g_pools_mu;               // held before a pool's own
DevicePool* g_pools = nullptr;
}  // namespace

DevicePool::DevicePool()
{
    std::lock_guard<std::mutex> lk(g_pools_mu);
    next_ = g_pools;
    if (next_) next_->prev_ = this;
    g_pools = this;
}

DevicePool::~DevicePool()
{
    if (token_) (void)hipFree(token_);
    std::lock_guard<std::mutex> lk(g_pools_mu);
    (prev_ ? prev_->next_ : g_pools) = next_;
    if (next_) next_->prev_ = prev_;
}

void DevicePool::trim_device(int device)
{
    std::lock_guard<std::mutex> lk(g_pools_mu);
    for (DevicePool* p = g_pools; p; p = p->next_)
        if (p->device == device) p->trim(0);
}

hipError_t device_malloc(int device, void** out, size_t bytes)
{
    hipError_t e = hipMalloc(out, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        DevicePool::trim_device(device);
        e = hipMalloc(out, bytes);
    }
    return e;
}

hipError_t DevicePool::alloc(void** out, size_t bytes)
{
    *out = nullptr;
    const size_t need = (std::max<size_t>(bytes, 1) + 255) / 256 * 256;
    {
        std::lock_guard<std::mutex> lk(mu_);
        // the smallest kept block that holds it without wasting more than a quarter
        auto it = kept_.lower_bound(need);
        if (it != kept_.end() && it->first <= need + need / 4 + ((size_t)64 << 10)) {
            try {
                live_.emplace(it->second.ptr, it->first);
            } catch (...) {
                return hipErrorOutOfMemory;
            }
            *out = it->second.ptr;
            kept_bytes_ -= it->first;
            kept_.erase(it);
            return hipSuccess;
        }
    }
    const hipError_t e = device_malloc(device, out, need);
    if (e != hipSuccess) {
        *out = nullptr;
        return e;
    }
    try {
        std::lock_guard<std::mutex> lk(mu_);
        if (!token_ && hipMalloc(&token_, kToken) != hipSuccess) {
            (void)hipGetLastError();
            token_ = nullptr;
        }
        live_.emplace(*out, need);
    } catch (...) {
        (void)hipFree(*out);
        *out = nullptr;
        return hipErrorOutOfMemory;
    }
    return hipSuccess;
}

// Waits for the device by hipFree of a block held for that.  (Waiting for the
// device as such ends every stream capture under way in the process, other
// threads' and relaxed ones among them; hipFree does not.)
bool DevicePool::wait_idle()
{
    void* t;
    {
        std::lock_guard<std::mutex> lk(mu_);
        t = token_;
        token_ = nullptr;
    }
    if (!t) return false;
    const bool idle = hipFree(t) == hipSuccess;
    if (idle && hipMalloc(&t, kToken) != hipSuccess) {   // (the next allocation tries again)
        (void)hipGetLastError();
        t = nullptr;
    }
    if (t) {
        std::lock_guard<std::mutex> lk(mu_);
        if (!token_) std::swap(t, token_);
    }
    if (t) (void)hipFree(t);   // (an allocation of another thread has made one meanwhile)
    return idle;
}

void DevicePool::release(void* p)
{
    if (!p) return;
    // As hipFree would, wait for the device: kernels of any stream, the
    // caller's own among them, may still read the block.
    (void)hipSetDevice(device);
    bool idle = t_quiet;
    if (!idle) idle = wait_idle();
    size_t size = 0;
    {
        std::lock_guard<std::mutex> lk(mu_);
        auto it = live_.find(p);
        if (it != live_.end()) {
            size = it->second;
            live_.erase(it);
        }
        if (idle && size > 0 && size <= kMaxKept) {
            try {
                kept_.emplace(size, Kept{p, ++stamp_});
                kept_bytes_ += size;
                p = nullptr;
            } catch (...) {   // no memory for the entry: the block goes back
            }
        }
    }
    if (p && hipFree(p) == hipSuccess) idle = true;
    if (t_quiet_depth > 0) t_quiet = idle;
    trim(kMaxKept);
}

void DevicePool::trim(size_t keep)
{
    for (;;) {
        void* victim = nullptr;
        {
            std::lock_guard<std::mutex> lk(mu_);
            if (kept_bytes_ <= keep && kept_.size() <= kMaxBlocks) return;
            if (kept_.empty()) return;
            auto oldest = kept_.begin();
            for (auto it = kept_.begin(); it != kept_.end(); ++it)
                if (it->second.stamp < oldest->second.stamp) oldest = it;
            victim = oldest->second.ptr;
            kept_bytes_ -= oldest->first;
            kept_.erase(oldest);
        }
        (void)hipFree(victim);
    }
}

// ---------------------------------------------------------------------------
// copies to and from pageable memory
// ---------------------------------------------------------------------------
HostCopier::~HostCopier()
{
    {
        std::lock_guard<std::mutex> lk(mu_);
        stop_ = true;
    }
    work_.notify_all();
    for (std::thread& t : threads_) t.join();
    for (auto& r : rings_) r->drop();
}

void HostCopier::Ring::drop()
{
    for (int b = 0; b < kBufs; ++b) {
        if (ev[b]) {
            if (in_flight[b]) (void)hipEventSynchronize(ev[b]);
            (void)hipEventDestroy(ev[b]);
        }
        ev[b] = nullptr;
        in_flight[b] = false;
    }
    if (pin) (void)hipHostFree(pin);
    pin = nullptr;
    buf = 0;
}

// Whether all its copies have run.
bool HostCopier::Ring::idle()
{
    for (int b = 0; b < kBufs; ++b) {
        if (in_flight[b] && hipEventQuery(ev[b]) != hipSuccess) return false;
        in_flight[b] = false;
    }
    return true;
}

// kBufs pinned buffers, an eighth of the copy each (64 KiB to 8 MiB).
bool HostCopier::Ring::prepare(size_t total)
{
    size_t want = kMinBuf;
    while (want < kMaxBuf && want * kBufs < total) want *= 2;
    if (want <= buf) return true;
    drop();
    if (hipHostMalloc((void**)&pin, want * kBufs, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        pin = nullptr;
        return false;
    }
    buf = want;
    for (int b = 0; b < kBufs; ++b)
        if (hipEventCreateWithFlags(&ev[b], hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            ev[b] = nullptr;
            drop();
            return false;
        }
    return true;
}

// A ring for one transfer: one whose copies have all run, else a new one, else
// one that still uploads behind its stream's work, else the next given back;
// nullptr where there is no memory for the first.
HostCopier::Ring* HostCopier::take()
{
    std::unique_lock<std::mutex> lk(rings_mu_);
    for (;;) {
        Ring* busy = nullptr;
        for (auto& r : rings_) {
            if (r->taken) continue;
            if (r->idle()) {
                r->taken = true;
                return r.get();
            }
            busy = r.get();
        }
        if ((int)rings_.size() < max_rings_) {
            try {
                rings_.push_back(std::make_unique<Ring>());
                rings_.back()->taken = true;
                return rings_.back().get();
            } catch (...) {
                if (rings_.empty()) return nullptr;
            }
        }
        if (busy) {
            busy->taken = true;
            return busy;
        }
        rings_cv_.wait(lk);
    }
}

void HostCopier::give(Ring* r)
{
    {
        std::lock_guard<std::mutex> lk(rings_mu_);
        r->taken = false;
    }
    rings_cv_.notify_one();
}

// For copies of some size, once.
void HostCopier::start_threads(size_t total)
{
    if (total <= kSlice || has_threads_) return;
    std::call_once(threads_once_, [this] {
        cpu_set_t set;
        int n = sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) / 2 : 1;
        n = std::min(8, n);
        try {
            for (int i = 0; i < n; ++i) threads_.emplace_back([this] { run(); });
        } catch (...) {   // fewer threads, or none: the caller copies
        }
        has_threads_ = !threads_.empty();
    });
}

void HostCopier::run()
{
    std::unique_lock<std::mutex> lk(mu_);
    for (;;) {
        work_.wait(lk, [this] { return stop_ || !queue_.empty(); });
        if (queue_.empty()) return;
        const Slice s = queue_.front();
        queue_.pop_front();
        lk.unlock();
        std::memcpy(s.dst, s.src, s.bytes);
        lk.lock();
        if (--*s.pending == 0) done_.notify_all();
    }
}

// Copies src to dst in slices on the threads (counted in *pending), or here
// when it is short or there are none.
void HostCopier::spread(void* dst, const void* src, size_t bytes, int* pending)
{
    if (!has_threads_ || bytes <= kSlice / 2) {
        std::memcpy(dst, src, bytes);
        return;
    }
    {
        std::unique_lock<std::mutex> lk(mu_);
        for (size_t o = 0; o < bytes; o += kSlice) {
            try {
                queue_.push_back(Slice{(char*)dst + o, (const char*)src + o, std::min(kSlice, bytes - o), pending});
            } catch (...) {   // no memory for the entry: the rest here
                lk.unlock();
                std::memcpy((char*)dst + o, (const char*)src + o, bytes - o);
                break;
            }
            ++*pending;
        }
    }
    work_.notify_all();
}

void HostCopier::wait_slices(const int* pending)
{
    std::unique_lock<std::mutex> lk(mu_);
    done_.wait(lk, [pending] { return *pending == 0; });
}

void HostCopier::copy(void* dst, const void* src, size_t bytes)
{
    start_threads(bytes);
    int pending = 0;
    spread(dst, src, bytes, &pending);
    wait_slices(&pending);
}

// Whether the runtime knows the array (pinned, or memory of a device): it
// copies straight to and from it.
static bool known_memory(const void* p, size_t bytes)
{
    for (const char* at : {(const char*)p, (const char*)p + (bytes - 1)}) {
        hipPointerAttribute_t a;
        if (hipPointerGetAttributes(&a, at) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        if (a.type == hipMemoryTypeUnregistered) return false;
    }
    return true;
}

hipError_t HostCopier::transfer(const Piece* pieces, size_t n, bool to_host, hipStream_t s)
{
    const size_t line = to_host ? kDirectToHost : kDirectToDevice;
    size_t total = 0;
    for (size_t i = 0; i < n; ++i) total += pieces[i].bytes;
    auto direct = [&](const Piece& p) {
        return hipMemcpyAsync(p.dst, p.src, p.bytes, to_host ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice, s);
    };
    // what takes the ring: of a long transfer, the pageable pieces
    std::array<Piece, kMaxPieces> ringed;
    size_t nr = 0;
    for (size_t i = 0; i < n; ++i) {
        const Piece& p = pieces[i];
        if (p.bytes == 0) continue;
        if (total > line && nr < kMaxPieces && !known_memory(to_host ? p.dst : p.src, p.bytes)) {
            ringed[nr++] = p;
        } else {
            const hipError_t e = direct(p);
            if (e != hipSuccess) return e;
        }
    }
    if (nr > 0) {
        Ring* r = take();
        const bool ready = r && r->prepare(total);
        hipError_t e = hipSuccess;
        if (ready) {
            start_threads(total);
            e = through(*r, ringed.data(), nr, to_host, s);
        } else {
            for (size_t i = 0; i < nr && e == hipSuccess; ++i) e = direct(ringed[i]);
        }
        if (r) give(r);
        if (e != hipSuccess) return e;
        if (ready && nr == n) return hipSuccess;   // (all in place)
    }
    // (the runtime has read a pageable source when it returns)
    return to_host ? hipStreamSynchronize(s) : hipSuccess;
}

hipError_t HostCopier::through(Ring& r, const Piece* pieces, size_t n, bool to_host, hipStream_t s)
{
    const hipMemcpyKind kind = to_host ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice;
    struct Part {
        void* dst;
        const void* src;
        size_t bytes;
    };
    constexpr int kParts = 16;
    Part parts[kBufs][kParts];        // what each buffer holds
    int n_parts[kBufs] = {};
    size_t pi = 0, po = 0;            // next byte to issue
    int64_t head = 0, tail = 0;       // buffers issued, buffers handed on
    hipError_t e = hipSuccess;
    while (e == hipSuccess && (pi < n || tail < head)) {
        if (pi < n && head - tail < kBufs) {
            const int b = (int)(head % kBufs);
            wait_slices(&r.pending[b]);
            if (r.in_flight[b]) {
                e = hipEventSynchronize(r.ev[b]);
                r.in_flight[b] = false;
            }
            char* const base = r.pin + (size_t)b * r.buf;
            size_t used = 0;
            n_parts[b] = 0;
            while (pi < n && used < r.buf && n_parts[b] < kParts) {
                const Piece& p = pieces[pi];
                const size_t m = std::min(p.bytes - po, r.buf - used);
                if (m > 0) {
                    char* const mine = base + used;
                    char* const dst = (char*)p.dst + po;
                    const char* const src = (const char*)p.src + po;
                    if (to_host) {
                        if (e == hipSuccess) e = hipMemcpyAsync(mine, src, m, kind, s);
                    } else {
                        spread(mine, src, m, &r.pending[b]);
                    }
                    parts[b][n_parts[b]++] = Part{dst, mine, m};
                    used += (m + 255) / 256 * 256;
                    po += m;
                }
                if (po == p.bytes) {
                    ++pi;
                    po = 0;
                }
            }
            if (!to_host) {
                wait_slices(&r.pending[b]);
                for (int i = 0; i < n_parts[b] && e == hipSuccess; ++i)
                    e = hipMemcpyAsync(parts[b][i].dst, parts[b][i].src, parts[b][i].bytes, kind, s);
            }
            if (e == hipSuccess) e = hipEventRecord(r.ev[b], s);
            r.in_flight[b] = e == hipSuccess;
            ++head;
            if (!to_host) tail = head;   // (the buffer is free once its event has passed)
            continue;
        }
        const int b = (int)(tail % kBufs);
        e = hipEventSynchronize(r.ev[b]);
        r.in_flight[b] = false;
        if (e == hipSuccess)
            for (int i = 0; i < n_parts[b]; ++i) spread(parts[b][i].dst, parts[b][i].src, parts[b][i].bytes, &r.pending[b]);
        ++tail;
    }
    if (e != hipSuccess) (void)hipStreamSynchronize(s);   // nothing reads or writes the buffers any more
    if (to_host)
        for (int b = 0; b < kBufs; ++b) wait_slices(&r.pending[b]);
    return e;
}

bool ctx_waited(bs2e_ctx* c)
{
    return !c->arena && !c->foreign && hipStreamSynchronize(c->stream) == hipSuccess;
}

HostCopier* ctx_copier(bs2e_ctx* c)
{
    std::lock_guard<std::mutex> lk(c->up_mu);
    if (!c->copier) {
        try {
            c->copier = std::make_shared<HostCopier>(1);
        } catch (...) {
            return nullptr;
        }
    }
    return c->copier.get();
}

static hipError_t transfer(bs2e_ctx* c, std::initializer_list<Piece> pieces, bool to_host)
{
    if (HostCopier* h = ctx_copier(c)) return h->transfer(pieces.begin(), pieces.size(), to_host, c->stream);
    for (const Piece& p : pieces)
        if (p.bytes > 0) {
            const hipError_t e = hipMemcpyAsync(p.dst, p.src, p.bytes, to_host ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice,
                                                c->stream);
            if (e != hipSuccess) return e;
        }
    return hipStreamSynchronize(c->stream);
}

hipError_t copy_to_host(bs2e_ctx* c, std::initializer_list<Piece> pieces) { return transfer(c, pieces, true); }
hipError_t copy_to_device(bs2e_ctx* c, std::initializer_list<Piece> pieces) { return transfer(c, pieces, false); }

}  // namespace bs2e
