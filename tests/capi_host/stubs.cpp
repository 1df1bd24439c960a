// stubs.cpp -- definitions for stubs.h
#include "stubs.h"

#include <hip/hip_runtime_api.h>

using namespace bsattn;

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  if (n > stub::memory_limit || !(*p = std::calloc(1, n))) return hipErrorOutOfMemory;
  std::lock_guard<std::mutex> lock(stub::mu);
  stub::memory[*p] = n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> lock(stub::mu);
  CHECK(!p || stub::memory.erase(p) == 1);
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n) {
  std::memset(p, v, n);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stub error"; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 256;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = (hipEvent_t)new stub::Event;
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) {
  delete (stub::Event*)e;
  return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) { return ((stub::Event*)e)->done ? hipSuccess : hipErrorNotReady; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  ((stub::Event*)e)->done = false;
  ++((stub::Event*)e)->records;
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  std::lock_guard<std::mutex> lock(stub::mu);
  if (!((stub::Event*)e)->done) stub::waits.emplace_back(s, (stub::Event*)e);
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 0.f;
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* st) {
  *st = stub::capture;
  return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }
}

namespace bsattn {
using stub::run;
hipError_t noalloc_scratch(int, void** p, uint32_t** a) {
  static std::vector<uint8_t> s(kNoAllocScratchBytes);
  static std::vector<uint32_t> w(kArriveWords);
  *p = s.data();
  *a = w.data();
  return hipSuccess;
}
hipError_t launch_patch(const Geometry& g, const PatchBatch& pb, hipStream_t) { return run(g, &pb); }
hipError_t launch_append(const Geometry& g, const AppendBatch&, const AppendPages& pg, const PatchBatch& pb, int,
                         const void*, const void*, hipStream_t, Timing*) {
  return run(g, pg.given ? &pb : nullptr);
}
hipError_t launch_append_q16(const Geometry& g, const AppendBatch&, const AppendPages& pg, const PatchBatch& pb, int,
                             const void*, const void*, hipStream_t, Timing*) {
  return run(g, pg.given ? &pb : nullptr);
}
hipError_t launch_append_quantized(const Geometry& g, const AppendBatch&, const AppendPages& pg, const PatchBatch& pb,
                                   int, const uint32_t*, const void*, const void*, const uint32_t*, const void*,
                                   const void*, hipStream_t, Timing*) {
  return run(g, pg.given ? &pb : nullptr);
}
hipError_t launch_append_step(const Geometry& g, const AppendBatch&, const void*, const void*, hipStream_t, Timing*) {
  return run(g, nullptr);
}
int candidates(const Geometry& g, int len) { return (len + g.tb - 1) / g.tb - g.nr - g.ns; }
int mfma_err_stride(const Geometry&) { return 64; }
int fused_select_limit(int) { return 2048; }
bool fused_decode_ok(const Geometry&, int, int) { return false; }
int attend_waves(const Geometry&, int) { return kWaves; }
hipError_t launch_select(const Geometry& g, const SeqBatch&, const void*, float*, float*, int32_t*, int, hipStream_t,
                         Timing*, const StepAppend*) {
  return run(g, nullptr);
}
hipError_t launch_attend(const Geometry& g, const SeqBatch&, const void*, const int32_t*, int, float, void*, float*,
                         hipStream_t, Timing*) {
  return run(g, nullptr);
}
hipError_t launch_decode(const Geometry& g, const SeqBatch&, const void*, float*, int32_t*, int, int, float, void*,
                         float*, hipStream_t, Timing*) {
  return run(g, nullptr);
}
hipError_t launch_append_decode(const Geometry& g, const SeqBatch&, const StepAppend& ap, const void*, float*, float*,
                                int32_t*, int32_t*, int, bool, int, float, void*, float*, uint32_t*, hipStream_t,
                                Timing*) {
  return run(g, &ap.pb);
}
hipError_t launch_fused_decode(const Geometry& g, const SeqBatch&, int, const void*, int32_t*, bool, float, void*,
                               float*, uint32_t*, hipStream_t, Timing*) {
  return run(g, nullptr);
}
hipError_t launch_fused_attend(const Geometry& g, const SeqBatch&, int, const void*, const int32_t*, float, void*,
                               float*, uint32_t*, hipStream_t, Timing*) {
  return run(g, nullptr);
}
int prefill_splits(const Geometry&, int, int, int) { return stub::splits; }
hipError_t launch_prefill(const Geometry& g, const SeqBatch&, int, int nsplit, const void*, float, void*, float* ws,
                          hipEvent_t done, hipStream_t s, Timing*) {
  {
    std::lock_guard<std::mutex> lock(stub::mu);
    stub::prefills.push_back({ws, (stub::Event*)done, nsplit});
  }
  const hipError_t e = run(g, nullptr);
  if (e == hipSuccess && done) (void)hipEventRecord(done, s);
  return e;
}
hipError_t launch_export(const Geometry& g, const SeqBatch&, int, void*, void*, hipStream_t) { return run(g, nullptr); }
hipError_t launch_export_quantized(const Geometry& g, const SeqBatch&, int, uint32_t*, void*, void*, uint32_t*, void*,
                                   void*, hipStream_t) {
  return run(g, nullptr);
}
hipError_t launch_export_summaries(const Geometry& g, int, int, void*, hipStream_t) { return run(g, nullptr); }
}  // namespace bsattn
