// Device memory and capture streams kept from one solver to the next.
//
// A solver allocates some fifty buffers and frees them together, and every hipFree waits for the
// device and unmaps: 10 of the 31 ms of a differentiated solve of 4 x 1025^2, which builds a solver
// per call, went into it and 2 ms into hipMalloc.  Blocks of a destroyed solver are therefore kept
// for the next one of the same sizes, per device and byte count, up to a limit in all; beyond
// that the ones kept longest are freed, and when an allocation here fails all of them are.  Another
// library's allocation cannot ask for them: pool_trim gives them back at once, and a limit of 0 keeps
// none.
//
// A block may be handed to any thread and stream, so it is only kept while no queued work can still
// use it: inside a pool_idle_scope.  Outside one pool_free is hipFree.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <optional>

namespace cedar {
namespace hip {

// Bytes kept at most, unless CEDAR_AMD_POOL_MB of the environment (MiB, read at the first use) or
// pool_set_limit says otherwise.
constexpr std::size_t kPoolBytes = std::size_t(4) << 30;
// Sets the limit, frees what lies beyond it and returns the previous one.
std::size_t pool_set_limit(std::size_t bytes);
// Frees every kept block and stream; returns the bytes of the blocks.
std::size_t pool_trim();

// nullptr and the error in *e on failure
void *pool_malloc(std::size_t bytes, hipError_t *e);
void pool_free(void *p) noexcept;

// While alive, blocks of the current device that this thread frees are idle: nothing queued uses
// them.  The constructor waits for the stream that alone used them, and not for the device: that
// breaks every capture in the process, whichever thread captures and in whatever mode, where hipFree
// leaves those of other threads alone.
class pool_idle_scope {
public:
    explicit pool_idle_scope(hipStream_t s);
    ~pool_idle_scope();
    pool_idle_scope(const pool_idle_scope &) = delete;
    pool_idle_scope &operator=(const pool_idle_scope &) = delete;

private:
    int prev_;
};

// While alive, no block that this thread frees is idle, whatever scope is opened inside.
class pool_busy_scope {
public:
    pool_busy_scope();
    ~pool_busy_scope();
    pool_busy_scope(const pool_busy_scope &) = delete;
    pool_busy_scope &operator=(const pool_busy_scope &) = delete;
};

// First member of a class that owns buffers used on stream s: its destructor calls enter(s), and as the
// first member is destroyed last, the members after it give their blocks back idle.  Where work of the
// caller's own on other streams may use the buffers (lend: it has pointers to them; lend_if_captured:
// it records what is enqueued on s into a graph), they go back through hipFree, which waits for the
// device.
class pool_guard {
public:
    void lend() { lent_ = true; }
    void lend_if_captured(hipStream_t s) {
        hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
        const hipError_t e = hipStreamIsCapturing(s, &st);
        if (e != hipSuccess) (void)hipGetLastError();
        if (e != hipSuccess || st != hipStreamCaptureStatusNone) lent_ = true;
    }
    void enter(hipStream_t s) {
        if (lent_)
            busy_.emplace();
        else
            idle_.emplace(s);
    }

private:
    std::optional<pool_idle_scope> idle_;
    std::optional<pool_busy_scope> busy_;
    bool lent_ = false;
};

// A non-blocking stream of the current device for captures alone (no work runs on it, so the next
// solver can take it over); nullptr and the error in *e on failure.  At most 16 are kept.
hipStream_t pool_capture_stream(hipError_t *e);
void pool_return_capture_stream(hipStream_t s);

}  // namespace hip
}  // namespace cedar
