// fake_gpu.cpp -- the HIP runtime and the kernel launchers that the API harness
// links wahgpu_api.hip against.  A launcher computes nothing: it logs one line
// and, where its kernels would hand a result to the host, hands over what the
// test scripted for it (nothing scripted: no fault, result 0).
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

#include <deque>
#include <map>
#include <string>

#include "wah_kernels.h"

namespace {

std::string g_log;
std::map<void*, size_t> g_blocks;  // device memory
size_t g_device_bytes = 0, g_most = ~(size_t)0;
uint64_t g_clock = 0;

struct Script {
  bool ends;  // false: the launch's last block never comes
  uint64_t fault, result, extra[2];
};
std::map<std::string, std::deque<Script>> g_scripts;

void note(const char* fmt, ...) {
  char buf[256];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_log += buf;
  g_log += '\n';
}

Script next(const char* name) {
  auto& q = g_scripts[name];
  if (q.empty()) return Script{true, 0, 0, {0, 0}};
  const Script s = q.front();
  q.pop_front();
  return s;
}

hipError_t busy(hipStream_t s) {
  return s && s->capturing ? hipErrorStreamCaptureUnsupported : hipSuccess;
}

}  // namespace

extern "C" {
const char* fake_log() { return g_log.c_str(); }
void fake_reset() {
  g_log.clear();
  g_scripts.clear();
  g_most = ~(size_t)0;
}
uint64_t fake_device_bytes() { return g_device_bytes; }
void fake_most_bytes(uint64_t bytes) { g_most = bytes; }
void fake_capture(void* stream, int on) { static_cast<hipStream_t>(stream)->capturing = on != 0; }
// What the next launch of `name` leaves behind (queued).
void fake_script(const char* name, int ends, uint64_t fault, uint64_t result, uint64_t extra0,
                 uint64_t extra1) {
  g_scripts[name].push_back(Script{ends != 0, fault, result, {extra0, extra1}});
}
}

const char* hipGetErrorString(hipError_t e) {
  return e == hipErrorOutOfMemory ? "out of memory"
         : e == hipErrorStreamCaptureUnsupported ? "not permitted while a stream is capturing"
                                                 : "error";
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
  memset(p, 0, sizeof(*p));
  strcpy(p->name, "fake");
  strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipMallocBytes(void** p, size_t bytes) {
  *p = nullptr;
  if (bytes > g_most) return hipErrorOutOfMemory;
  // address space only: pages come when they are touched
  void* m = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE,
                 -1, 0);
  if (m == MAP_FAILED) return hipErrorOutOfMemory;
  g_blocks[m] = bytes;
  g_device_bytes += bytes;
  *p = m;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  auto it = g_blocks.find(p);
  if (it == g_blocks.end()) return hipErrorInvalidValue;
  munmap(p, it->second);
  g_device_bytes -= it->second;
  g_blocks.erase(it);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  *p = calloc(1, bytes);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void* dst, const void* src, size_t bytes, hipMemcpyKind) {
  memcpy(dst, src, bytes);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind, hipStream_t) {
  memcpy(dst, src, bytes);
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = new FakeStream; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { delete s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { return busy(s); }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
  *st = s->capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
  s->capturing = true;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
  s->capturing = false;
  *g = new FakeGraph;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, void*, void*, size_t) {
  *e = new FakeGraph;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { note("graph"); return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { delete g; return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { delete e; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = new FakeEvent; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { e->at = ++g_clock; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
  *ms = (float)(b->at - a->at);
  return hipSuccess;
}

// ---- launchers ---------------------------------------------------------------

namespace wah {

// A launch of at least one tile on scan state: its last block's results.
static void scan(const char* name, const ScanRun& a, uint64_t n, bool waits) {
  if (!n) return;
  note("%s n=%llu state=%p captured=%d", name, (unsigned long long)n, (void*)a.state, a.captured);
  const Script s = next(name);
  if (!s.ends) return;
  if (waits) {
    a.host[0] = s.fault;
    a.host[1] = s.result;
  } else if (s.fault) {
    *a.kept = s.fault;
  }
}

void launch_sort(const BuildArgs& a, hipStream_t s, LaunchHook* hook) {
  note("sort cols=%u", a.cols_cap);
  ++g_clock;
  for (int g = 0; hook && g < 5; ++g) hook->mark(s);
}
void launch_tail(const BuildArgs& a, hipStream_t s, LaunchHook* hook) {
  note("tail cols=%u", a.cols_cap);
  ++g_clock;
  if (hook) hook->mark(s);
}
void launch_sort_finalize(const BuildArgs&, hipStream_t) { note("finalize"); }
void launch_small(const BuildArgs& a, hipStream_t) {
  note("small cols=%u", a.inline_desc ? 1u : a.shorts_cap);
  g_clock += 100;
}
void launch_rank_selftest(uint32_t*, hipStream_t) {}
void launch_fill32(uint32_t* p, uint64_t words, uint32_t, hipStream_t) {
  if (words) note("fill %p words=%llu", (void*)p, (unsigned long long)words);
}
void launch_chunks(const uint32_t*, uint64_t, uint32_t*, uint32_t*, hipStream_t) { note("chunks"); }
void launch_fills(const uint32_t*, const uint32_t*, uint64_t, uint32_t*, hipStream_t) { note("fills"); }
void launch_merge(const ScanRun& a, const uint32_t*, const uint32_t*, const uint32_t*, uint64_t n,
                  uint32_t*, uint32_t*, uint32_t*, hipStream_t) {
  scan("merge", a, n, true);
}
void launch_compact(const ScanRun& a, const uint32_t*, const uint32_t*, uint64_t n, int, uint32_t*,
                    hipStream_t) {
  scan("compact", a, n, true);
}
void launch_colen(const ScanRun& a, const uint32_t*, const uint32_t*, uint64_t k, uint32_t*,
                  uint32_t*, uint32_t*, wahgpu_counts_dev*, hipStream_t) {
  scan("colen", a, k, true);
}
void launch_scan(const ScanRun& a, const uint32_t*, const uint32_t*, uint64_t n, uint32_t*, bool,
                 hipStream_t) {
  scan("scan", a, n, false);
}
void launch_decode(const ScanRun& s, const DecodeStream& a, const DecodeStream& b, uint64_t,
                   hipStream_t) {
  scan("decode", s, a.len + b.len, true);
}
void launch_range(const ScanRun& s, const uint32_t*, const uint32_t*, const uint32_t*, uint64_t,
                  const uint32_t*, uint64_t most_words, uint32_t, uint32_t, uint32_t*,
                  uint64_t nrows, uint64_t* table, uint64_t table_cap, bool grow, hipStream_t) {
  note("range nrows=%llu most=%llu table=%llu grow=%d", (unsigned long long)nrows,
       (unsigned long long)most_words, table ? (unsigned long long)table_cap : 0ull, grow);
  const Script x = next("range");
  s.host[3] = x.extra[0];
  s.host[4] = x.extra[1];
  if (!x.ends) return;
  s.host[0] = x.fault;
  s.host[1] = x.result;
}
void launch_encode(const ScanRun& s, const uint32_t*, const uint32_t*, int, uint64_t nrows,
                   uint32_t*, uint64_t, hipStream_t) {
  scan("encode", s, nrows, true);
}

}  // namespace wah
