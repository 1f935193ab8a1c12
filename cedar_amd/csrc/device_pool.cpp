#include "device_pool.hpp"

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
    std::size_t kept_bytes = 0;
    std::vector<std::pair<int, hipStream_t>> streams;
};

// never destroyed: blocks may come back while the process ends
pool &the_pool() {
    static pool *p = new pool;
    return *p;
}

thread_local int idle_device = -1;  // the device whose freed blocks are idle, or -1

int current_device() {
    int d = 0;
    return hipGetDevice(&d) == hipSuccess ? d : -1;
}

void release(std::vector<block> &out) {
    for (const block &b : out) (void)hipFree(b.p);
    out.clear();
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
            const block b = *it;
            P.kept.erase(std::next(it).base());
            P.kept_bytes -= b.bytes;
            P.live.emplace(b.p, b);
            *e = hipSuccess;
            return b.p;
        }
    }
    void *p = nullptr;
    *e = hipMalloc(&p, bytes);
    if (*e == hipErrorOutOfMemory) {
        std::vector<block> out;
        {
            std::lock_guard<std::mutex> g(P.mu);
            out.assign(P.kept.begin(), P.kept.end());
            P.kept.clear();
            P.kept_bytes = 0;
        }
        if (!out.empty()) {
            (void)hipGetLastError();
            release(out);
            *e = hipMalloc(&p, bytes);
        }
    }
    if (*e != hipSuccess) return nullptr;
    std::lock_guard<std::mutex> g(P.mu);
    P.live.emplace(p, block{p, bytes, dev});
    return p;
}

void pool_free(void *p) {
    if (!p) return;
    pool &P = the_pool();
    std::vector<block> out;
    {
        std::lock_guard<std::mutex> g(P.mu);
        const auto it = P.live.find(p);
        const block b = it == P.live.end() ? block{p, 0, -1} : it->second;
        if (it != P.live.end()) P.live.erase(it);
        if (b.device < 0 || b.device != idle_device || b.bytes > kPoolBytes) {
            out.push_back(b);
        } else {
            P.kept.push_back(b);
            P.kept_bytes += b.bytes;
            while (P.kept_bytes > kPoolBytes) {
                P.kept_bytes -= P.kept.front().bytes;
                out.push_back(P.kept.front());
                P.kept.pop_front();
            }
        }
    }
    release(out);
}

void pool_idle_scope::enter(hipError_t waited) {
    prev_ = idle_device;
    if (waited == hipSuccess)
        idle_device = current_device();
    else
        (void)hipGetLastError();  // blocks then go back through hipFree, which waits itself
}

pool_idle_scope::pool_idle_scope() { enter(hipDeviceSynchronize()); }
pool_idle_scope::pool_idle_scope(hipStream_t s) { enter(hipStreamSynchronize(s)); }
pool_idle_scope::~pool_idle_scope() { idle_device = prev_; }

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
