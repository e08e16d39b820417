// The library's scratch buffers (csrc/runtime.cpp) on a HIP runtime made of counters, so that
// allocation failures, captures and threads can be staged on the CPU.  One scenario per run,
// named by the first argument; exits 0 if it holds.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <thread>
#include <vector>

#include "runtime.hpp"

namespace {
std::map<void*, size_t> g_live;                 // device buffers
size_t g_capacity = size_t(1) << 40;            // bytes that may be live
std::set<hipStream_t> g_capturing;              // streams being recorded, in global mode
thread_local hipStreamCaptureMode t_mode = hipStreamCaptureModeGlobal;
int g_invalidated = 0;                          // captures that a forbidden call broke

bool forbidden() {
  if (g_capturing.empty() || t_mode == hipStreamCaptureModeRelaxed) return false;
  ++g_invalidated;
  return true;
}
size_t live_bytes() {
  size_t n = 0;
  for (const auto& e : g_live) n += e.second;
  return n;
}
}  // namespace

extern "C" {
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorName(hipError_t) { return "fake"; }
hipError_t hipMalloc(void** p, size_t n) {
  if (forbidden()) return hipErrorStreamCaptureUnsupported;
  if (live_bytes() + n > g_capacity) return hipErrorOutOfMemory;
  *p = std::malloc(1);
  g_live[*p] = n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (forbidden()) return hipErrorStreamCaptureUnsupported;
  if (!g_live.erase(p)) return hipErrorInvalidValue;   // (the address is not used again)
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  return g_capturing.count(s) ? hipErrorStreamCaptureUnsupported : hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
  *st = g_capturing.count(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) {
  std::swap(*m, t_mode);
  return hipSuccess;
}
}

namespace {
const hipStream_t kA = reinterpret_cast<hipStream_t>(0x1000);
constexpr size_t MB = 1 << 20;

#define CHECK(x)                                                   \
  do {                                                             \
    if (!(x)) {                                                    \
      std::printf("line %d: not so: %s\n", __LINE__, #x);          \
      std::exit(1);                                                \
    }                                                              \
  } while (0)

void* get(hipStream_t s, size_t bytes) {
  void* p = nullptr;
  th::ScratchHold hold;
  return th::stream_scratch(s, bytes, &p, &hold) == TH_OK ? p : nullptr;
}
void* in_thread(hipStream_t s, size_t bytes) {
  void* p = nullptr;
  std::thread([&] { p = get(s, bytes); }).join();
  return p;
}

// One handle, a stream of its own in every thread: no two threads get the same buffer, each
// keeps its own, and an ordinary stream's buffer is shared.
void per_thread_own() {
  void* mine = get(hipStreamPerThread, MB);
  CHECK(mine && get(hipStreamPerThread, MB) == mine);
  CHECK(th::stream_scratch_ready(hipStreamPerThread, MB));
  void* other = nullptr;
  bool ready = true;
  std::thread([&] {
    ready = th::stream_scratch_ready(hipStreamPerThread, 1);
    other = get(hipStreamPerThread, MB);
  }).join();
  CHECK(!ready && other && other != mine);
  CHECK(get(hipStreamPerThread, MB) == mine);
  CHECK(get(kA, MB) && in_thread(kA, MB) == get(kA, MB));
}

// Many short-lived threads: what they leave is given back, but for what a graph recorded.
void per_thread_bounded() {
  void* graphs = nullptr;
  std::thread([&] {
    get(hipStreamPerThread, MB);
    g_capturing.insert(hipStreamPerThread);
    graphs = get(hipStreamPerThread, MB);
    g_capturing.clear();
  }).join();
  for (int i = 0; i < 200; ++i) {
    void* p = nullptr;
    std::thread([&] { get(hipStreamPerThread, MB), p = get(hipStreamPerThread, 5 * MB); }).join();
    CHECK(p && p != graphs);
  }
  CHECK(g_live.count(graphs));
  CHECK(live_bytes() <= MB + 17 * 6 * MB);
}

// A graph recorded earlier uses its buffer whenever it is replayed: where memory runs out, that
// buffer stays, as the current one or outgrown; others make room.
void short_of_memory() {
  get(kA, 2 * MB);
  g_capturing.insert(kA);
  void* graphs = get(kA, 2 * MB);
  g_capturing.clear();
  g_capacity = 10 * MB;
  CHECK(!get(kA, 12 * MB));
  CHECK(g_live.count(graphs) && get(kA, 2 * MB) == graphs);
  CHECK(get(kA, 3 * MB));   // 4 MB
  CHECK(!get(kA, 9 * MB));
  CHECK(g_live.count(graphs) && live_bytes() == 2 * MB);
  CHECK(get(kA, 8 * MB) && get(kA, 8 * MB) != graphs);
}

// A call that can do without gives nothing back.
void short_of_memory_optional() {
  void* p = get(kA, 2 * MB);
  g_capacity = 10 * MB;
  void* q = nullptr;
  {
    th::ScratchHold hold;
    CHECK(!th::try_stream_scratch(kA, 9 * MB, &q, &hold));
  }
  CHECK(g_live.count(p) && get(kA, 2 * MB) == p);
  CHECK(get(kA, 9 * MB));   // a call that cannot do without makes room
}

// A refused allocation is no lack of memory: the buffer stays.
void refused_while_recording() {
  void* p = get(kA, MB);
  g_capturing.insert(kA);
  CHECK(!get(kA, 5 * MB));
  g_capturing.clear();
  CHECK(get(kA, MB) == p && live_bytes() == MB);
  CHECK(get(kA, 5 * MB) && live_bytes() == 6 * MB);
}

// Another stream is being captured in global mode: allocations and frees here neither fail nor
// break that capture, and the thread's own mode is as it was.
void another_stream_recorded() {
  const hipStream_t other = reinterpret_cast<hipStream_t>(0x2000);
  for (int i = 0; i < 16; ++i) in_thread(hipStreamPerThread, MB);   // left to be freed
  g_capturing.insert(other);
  CHECK(get(kA, MB));
  CHECK(get(kA, 3 * MB));
  CHECK(in_thread(hipStreamPerThread, MB) && live_bytes() == 5 * MB);
  g_capacity = 10 * MB;
  CHECK(get(kA, 7 * MB));   // makes room
  CHECK(g_invalidated == 0 && t_mode == hipStreamCaptureModeGlobal);
}
}  // namespace

int main(int argc, char** argv) {
  const std::map<std::string, void (*)()> all = {
      {"per_thread_own", per_thread_own},
      {"per_thread_bounded", per_thread_bounded},
      {"short_of_memory", short_of_memory},
      {"short_of_memory_optional", short_of_memory_optional},
      {"refused_while_recording", refused_while_recording},
      {"another_stream_recorded", another_stream_recorded},
  };
  const auto it = argc == 2 ? all.find(argv[1]) : all.end();
  CHECK(it != all.end());
  it->second();
  std::puts("ok");
}
