// Internal helpers shared by the runtime, the tile-op entry points and the
// codegen target: thread-local error reporting mapped to the HalError
// categories of crates/tile_hal/src/error.rs:5-33.
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>
#include <string>

#include "../../include/tilers_hip.h"

namespace th {

// Record `msg` as this thread's last error and return `code`.
int fail(int code, const std::string& msg);

// hipSuccess -> TH_OK; anything else -> `code` with "<op> failed: <name> (<n>)".
int check_hip(hipError_t err, const char* op, int code);

// Clear the last error (successful calls leave it untouched, like errno).
void clear_error();

// Make `ordinal` the current device of this thread.
int use_device(int ordinal);

// Per-device scratch used by entry points that take an optional workspace.
// Returns a device buffer of at least `bytes` on the current device (grown on
// demand, kept until process exit).
int device_scratch(size_t bytes, void** out);

// Whether work enqueued on `s` is being recorded into a graph (or that cannot be told).
bool stream_capturing(hipStream_t s);

// Per-(device, stream) scratch for entry points without a workspace argument:
// work queued on one stream runs in order, so calls never share the buffer
// concurrently.  (hipStreamPerThread names another stream in every thread: there each
// thread has a buffer of its own, freed some time after the thread has ended unless a graph
// recorded it.)  `hold` locks the buffer until it is destroyed: a caller keeps it until
// everything that uses the buffer is queued, so that another thread's call on the same
// stream queues its work before or after and not in between, and cannot grow the buffer
// meanwhile.  At least `bytes`, grown on demand to at least twice the size and kept until
// process exit.  A buffer that is outgrown stays allocated (all of them together are smaller
// than the current one): queued work and graphs recorded earlier still use it.  Only where
// memory runs out are a stream's buffers given back to make room, after draining the stream,
// but for those that were handed out while a graph was recorded.
using ScratchHold = std::unique_lock<std::recursive_mutex>;
int stream_scratch(hipStream_t stream, size_t bytes, void** out, ScratchHold* hold);

// The same for a caller that can do without: false, and nothing given back, where the memory
// for it cannot be had.
bool try_stream_scratch(hipStream_t stream, size_t bytes, void** out, ScratchHold* hold);

// Whether the stream's buffer holds `bytes` already, so that stream_scratch need not allocate.
bool stream_scratch_ready(hipStream_t stream, size_t bytes);

}  // namespace th

#define TH_TRY(expr)                 \
  do {                               \
    const int th_rc_ = (expr);       \
    if (th_rc_ != TH_OK) return th_rc_; \
  } while (0)
