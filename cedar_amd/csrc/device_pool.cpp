#include "device_pool.hpp"

#include <algorithm>
#include <cstdlib>
#include <list>
#include <mutex>
#include <unordered_map>
#include <utility>
#include <vector>

namespace cedar {
namespace hip {

namespace {

struct block {
    void *p;
    std::size_t bytes;
    int device;
};

struct pool {
    std::mutex mu;
    std::unordered_map<void *, block> live;  // blocks handed out
    std::list<block> kept;                   // oldest first
    std::size_t kept_bytes = 0, limit = kPoolBytes;
    std::vector<std::pair<int, hipStream_t>> streams;

    pool() {
        const char *v = std::getenv("CEDAR_AMD_POOL_MB");
        char *end = nullptr;
        const unsigned long long mb = v && *v >= '0' && *v <= '9' ? std::strtoull(v, &end, 10) : 0;
        if (end && *end == '\0') limit = (std::size_t)std::min(mb, ~0ull >> 20) << 20;
    }
    // moves the blocks kept longest to out until at most `most` bytes are left (the lock is held)
    void evict(std::size_t most, std::list<block> &out) {
        while (kept_bytes > most) {
            kept_bytes -= kept.front().bytes;
            out.splice(out.end(), kept, kept.begin());
        }
    }
};

// never destroyed: blocks may come back while the process ends
pool &the_pool() {
    static pool *p = new pool;
    return *p;
}

thread_local int idle_device = -1;  // the device whose freed blocks are idle, or -1
thread_local int busy_scopes = 0;   // open pool_busy_scopes

int current_device() {
    int d = 0;
    return hipGetDevice(&d) == hipSuccess ? d : -1;
}

std::size_t release(std::list<block> &out) {
    std::size_t bytes = 0;
    for (const block &b : out) {
        (void)hipFree(b.p);
        bytes += b.bytes;
    }
    out.clear();
    return bytes;
}

}  // namespace

void *pool_malloc(std::size_t bytes, hipError_t *e) {
    pool &P = the_pool();
    bytes = (bytes + 255) / 256 * 256;
    const int dev = current_device();
    {
        std::lock_guard<std::mutex> g(P.mu);
        // the block kept last is the likeliest to be of this size
        for (auto it = P.kept.rbegin(); it != P.kept.rend(); ++it) {
            if (it->bytes != bytes || it->device != dev) continue;
            void *const p = it->p;
            P.live.emplace(p, *it);  // the one that can throw, so first
            P.kept_bytes -= it->bytes;
            P.kept.erase(std::next(it).base());
            *e = hipSuccess;
            return p;
        }
    }
    void *p = nullptr;
    *e = hipMalloc(&p, bytes);
    if (*e == hipErrorOutOfMemory) {
        std::list<block> out;
        {
            std::lock_guard<std::mutex> g(P.mu);
            P.evict(0, out);
        }
        if (!out.empty()) {
            (void)hipGetLastError();
            release(out);
            *e = hipMalloc(&p, bytes);
        }
    }
    if (*e != hipSuccess) return nullptr;
    try {
        std::lock_guard<std::mutex> g(P.mu);
        P.live.emplace(p, block{p, bytes, dev});
    } catch (...) {
        (void)hipFree(p);
        throw;
    }
    return p;
}

void pool_free(void *p) noexcept {
    if (!p) return;
    pool &P = the_pool();
    std::list<block> out;
    try {
        std::list<block> mine(1);  // allocated before anything changes
        std::lock_guard<std::mutex> g(P.mu);
        const auto it = P.live.find(p);
        mine.front() = it == P.live.end() ? block{p, 0, -1} : it->second;
        if (it != P.live.end()) P.live.erase(it);
        const block &b = mine.front();
        if (b.device < 0 || b.device != idle_device || busy_scopes > 0 || b.bytes > P.limit) {
            out.splice(out.end(), mine);
        } else {
            P.kept_bytes += b.bytes;
            P.kept.splice(P.kept.end(), mine);
            P.evict(P.limit, out);
        }
    } catch (...) {  // no host memory for the list: the block goes back all the same
        {
            std::lock_guard<std::mutex> g(P.mu);
            P.live.erase(p);
        }
        (void)hipFree(p);
    }
    release(out);
}

std::size_t pool_set_limit(std::size_t bytes) {
    pool &P = the_pool();
    std::list<block> out;
    std::size_t prev;
    {
        std::lock_guard<std::mutex> g(P.mu);
        prev = P.limit;
        P.limit = bytes;
        P.evict(bytes, out);
    }
    release(out);
    return prev;
}

std::size_t pool_trim() {
    pool &P = the_pool();
    std::list<block> out;
    std::vector<std::pair<int, hipStream_t>> streams;
    {
        std::lock_guard<std::mutex> g(P.mu);
        P.evict(0, out);
        streams.swap(P.streams);
    }
    for (const auto &s : streams) (void)hipStreamDestroy(s.second);
    return release(out);
}

pool_idle_scope::pool_idle_scope(hipStream_t s) : prev_(idle_device) {
    idle_device = -1;
    if (busy_scopes > 0) return;
    if (hipStreamSynchronize(s) == hipSuccess)
        idle_device = current_device();
    else
        (void)hipGetLastError();  // blocks then go back through hipFree, which waits itself
}
pool_idle_scope::~pool_idle_scope() { idle_device = prev_; }

pool_busy_scope::pool_busy_scope() { ++busy_scopes; }
pool_busy_scope::~pool_busy_scope() { --busy_scopes; }

hipStream_t pool_capture_stream(hipError_t *e) {
    pool &P = the_pool();
    const int dev = current_device();
    {
        std::lock_guard<std::mutex> g(P.mu);
        for (auto it = P.streams.begin(); it != P.streams.end(); ++it) {
            if (it->first != dev) continue;
            const hipStream_t s = it->second;
            P.streams.erase(it);
            *e = hipSuccess;
            return s;
        }
    }
    hipStream_t s = nullptr;
    *e = hipStreamCreateWithFlags(&s, hipStreamNonBlocking);
    return *e == hipSuccess ? s : nullptr;
}

void pool_return_capture_stream(hipStream_t s) {
    if (!s) return;
    pool &P = the_pool();
    int dev = -1;
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamGetDevice(s, &dev) == hipSuccess &&
        hipStreamIsCapturing(s, &st) == hipSuccess && st == hipStreamCaptureStatusNone) {
        std::lock_guard<std::mutex> g(P.mu);
        if (P.streams.size() < 16) {
            P.streams.emplace_back(dev, s);
            return;
        }
    }
    (void)hipStreamDestroy(s);
}

}  // namespace hip
}  // namespace cedar
