// The library's host code (gst_decoder.cpp, gst_ans.cpp, gst_serve.cpp) on a stand-in for the
// HIP runtime and for the kernels' launches: what a call leaves behind it, and what it does
// when the runtime refuses it something.  One check an argument; no GPU and no HIP library.
//
// The stand-in keeps device and pinned memory in ordinary memory that is never given back, so
// no two allocations share an address.  Work on created streams is done at once; hipMemset on
// the null stream is done as late as HIP allows: when something waits for that stream or runs
// on it.  The "kernels" write kBlock to every output byte.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <vector>

#include "gst_ans.h"
#include "gst_decoder.h"
#include "gst_internal.h"
#include "gst_serve.h"

#define CHECK(x)                                                        \
  do {                                                                  \
    if (!(x)) {                                                         \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #x);               \
      std::exit(1);                                                     \
    }                                                                   \
  } while (0)

namespace {

constexpr uint8_t kBlock = 0x5A;

struct Fake {
  std::mutex mu;
  std::vector<std::function<void()>> late;  // null-stream clears that were not waited for
  std::set<void *> freed;
  size_t lds = 65536;
  int streams = 0;
  int memsets = 0;       // hipMemsetAsync calls on created streams
  uint32_t raise = 0;    // error bits the next decodes set
  uint32_t images = 0;   // images the last rANS launch found in its plan
  int fail_waits = 0;    // hipStreamSynchronize fails this many times
  size_t most = ~size_t{0};  // the largest device allocation that succeeds
  size_t pinned = 0;     // the largest pinned allocation so far
  bool no_pinned = false;  // hipHostMalloc fails
  void *out = nullptr;   // where the last kernel wrote its output

  void RunLate() {
    std::vector<std::function<void()>> work;
    {
      std::lock_guard<std::mutex> lk(mu);
      work.swap(late);
    }
    for (auto &w : work) w();
  }
  void Before(hipStream_t s) {
    if (!s) RunLate();
  }
};
Fake &F() {
  static Fake f;
  return f;
}

hipError_t NewMemory(void **p, size_t n) {
  *p = std::aligned_alloc(4096, (n + 4095) / 4096 * 4096);
  std::memset(*p, 0xA5, n);
  return hipSuccess;
}

}  // namespace

extern "C" {

hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {
  std::memset(p, 0, sizeof(*p));
  std::strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
  p->maxThreadsPerBlock = 1024;
  p->sharedMemPerBlock = F().lds;
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }

hipError_t hipMalloc(void **p, size_t n) { return n > F().most ? hipErrorOutOfMemory : NewMemory(p, n); }
hipError_t hipFree(void *p) { F().freed.insert(p); return hipSuccess; }
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t) { return hipMalloc(p, n); }
hipError_t hipFreeAsync(void *p, hipStream_t) { F().freed.insert(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  F().pinned = std::max(F().pinned, n);
  return F().no_pinned ? hipErrorOutOfMemory : NewMemory(p, n);
}
hipError_t hipHostFree(void *p) { F().freed.insert(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) { return hipErrorInvalidValue; }
hipError_t hipMemGetAddressRange(hipDeviceptr_t *, size_t *, hipDeviceptr_t) { return hipErrorInvalidValue; }

hipError_t hipMemset(void *p, int v, size_t n) {
  std::lock_guard<std::mutex> lk(F().mu);
  F().late.push_back([=] { std::memset(p, v, n); });
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t s) {
  if (!s) return hipMemset(p, v, n);
  ++F().memsets;
  std::memset(p, v, n);
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  F().RunLate();
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
  F().Before(st);
  std::memcpy(d, s, n);
  return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned flags) {
  CHECK(flags == hipStreamNonBlocking);
  *s = reinterpret_cast<hipStream_t>(static_cast<uintptr_t>(0x1000 + 16 * ++F().streams));
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
  F().Before(s);
  if (F().fail_waits == 0) return hipSuccess;
  --F().fail_waits;
  return hipErrorUnknown;
}
hipError_t hipDeviceSynchronize() { F().RunLate(); return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = reinterpret_cast<hipEvent_t>(0x10); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t s) { F().Before(s); return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0.f; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) { return hipErrorNotSupported; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }

}  // extern "C"

namespace gst {

hipError_t LaunchStage(uint32_t stage, const KernelArgs &a, uint32_t, const StageConfig &, hipStream_t s) {
  F().Before(s);
  if (stage == kStageAns) {
    F().images = a.plan ? a.plan->n_images : 1;
    *a.err |= F().raise;
  }
  if (stage != kStageAssemble) return hipSuccess;
  const uint32_t n = a.plan ? a.plan->n_images : 1;
  for (uint32_t i = 0; i < n; ++i) {
    const ImageDesc &d = a.plan ? reinterpret_cast<const ImageDesc *>(reinterpret_cast<const uint8_t *>(a.plan) +
                                                                      PlanImagesOffset(a.plan_cap))[i]
                                : a.single;
    std::memset(d.out, kBlock, 8 * static_cast<size_t>(d.nv));
    F().out = d.out;
  }
  return hipSuccess;
}
hipError_t LaunchAnsGroups(const uint32_t *, const uint8_t *, uint32_t, uint32_t groups, uint32_t n, uint8_t *out,
                           uint32_t *status, hipStream_t s) {
  F().Before(s);
  std::memset(out, kBlock, static_cast<size_t>(groups) * n * kSymsPerLane);
  std::memset(status, 0, 4 * static_cast<size_t>(groups));
  F().out = out;
  return hipSuccess;
}
hipError_t LaunchExportBits(uint32_t *bits, uint32_t *host, hipStream_t s) {
  F().Before(s);
  *host = *bits;
  *bits = 0;
  return hipSuccess;
}
hipError_t LaunchClearWord(uint32_t *word, hipStream_t s) {
  F().Before(s);
  *word = 0;
  return hipSuccess;
}
hipError_t LaunchGather(const GatherArgs &a, hipStream_t s) {
  F().Before(s);
  for (uint32_t i = 0; i < a.n; ++i) std::memcpy(a.job[i].dst, a.job[i].src, a.job[i].bytes);
  return hipSuccess;
}
hipError_t LaunchCompare(const CompareArgs &, hipStream_t) { return hipSuccess; }
hipError_t ResolveNoAllocScratch(int) { return hipSuccess; }
uint8_t *NoAllocScratch(int) { return nullptr; }

}  // namespace gst

namespace {

// A file of the smallest legal size whose streams hold no words (the stand-in decodes nothing).
std::vector<uint8_t> File(uint32_t width = 128, uint32_t height = 1024) {
  gst_header h{};
  h.width = width;
  h.height = height;
  h.palette_bytes = 8192;
  const uint32_t groups = width * height / 131072;
  h.y_cmp_sz = 2 * groups * 132;
  h.chroma_cmp_sz = 4 * groups * 132;
  h.palette_sz = 132;
  h.indices_sz = groups * 132;
  std::vector<uint8_t> f(sizeof(h) + 2048 + h.y_cmp_sz + h.chroma_cmp_sz + h.palette_sz + h.indices_sz);
  std::memcpy(f.data(), &h, sizeof(h));
  return f;
}

gst_header Header(const std::vector<uint8_t> &f) {
  gst_header h;
  std::memcpy(&h, f.data(), sizeof(h));
  return h;
}

hipStream_t NewStream() {
  hipStream_t s;
  CHECK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking) == hipSuccess);
  return s;
}

gst_batch *NewBatch(const gst_header &h) {
  gst_batch_config c{};
  c.capacity_images = 1;
  c.capacity_blocks = h.width / 4 * (h.height / 4);
  gst_batch *b = nullptr;
  CHECK(gst_batch_create(&c, &b) == GST_OK);
  return b;
}

void Bind(gst_batch *b, const gst_header &h, const std::vector<uint8_t> &f, std::vector<uint8_t> *out, hipStream_t s) {
  const void *in[1] = {f.data()};
  void *o[1] = {out->data()};
  CHECK(gst_batch_bind(b, &h, 1, in, o, s) == GST_OK);
}

// A device without the LDS that the largest kernel asks for is refused when it is set up.
void DeviceWithLittleLds() {
  F().lds = 40959;
  CHECK(gst_initialize_decoder(0) == GST_ERR_NOT_INITIALIZED);
  F().lds = 40960;
  CHECK(gst_initialize_decoder(0) == GST_OK);
}

// A batch made while the null stream is busy, bound on a stream that does not wait for it.
void BatchPlanSurvives() {
  const auto f = File();
  const gst_header h = Header(f);
  std::vector<uint8_t> out(h.width * h.height / 2);
  gst_batch *b = NewBatch(h);
  hipStream_t s = NewStream();
  Bind(b, h, f, &out, s);
  F().RunLate();
  CHECK(gst_batch_decode(b, s) == GST_OK);
  CHECK(F().images == 1);
  for (uint8_t v : out) CHECK(v == kBlock);
  gst_batch_destroy(b);
}

// Bits that a decode sets after they were read and cleared are there for the next read.
void BatchErrorBitsSurvive() {
  const auto f = File();
  const gst_header h = Header(f);
  std::vector<uint8_t> out(h.width * h.height / 2);
  gst_batch *b = NewBatch(h);
  F().RunLate();
  hipStream_t s = NewStream();
  Bind(b, h, f, &out, s);
  for (uint32_t bits : {4u, 2u, 0u, 6u}) {
    F().raise = bits;
    CHECK(gst_batch_decode(b, s) == GST_OK);
    F().RunLate();
    uint32_t got = ~0u;
    CHECK(gst_batch_error_bits(b, s, &got) == GST_OK);
    CHECK(got == bits);
  }
  gst_batch_destroy(b);
}

void StreamErrorBitsSurvive() {
  const auto f = File();
  const gst_header h = Header(f);
  std::vector<uint8_t> out(h.width * h.height / 2), staging(512 + f.size());
  hipStream_t s = NewStream();
  for (uint32_t bits : {4u, 2u, 0u, 6u}) {
    F().raise = bits;
    CHECK(gst_load_compressed_dxt(&h, s, staging.data(), out.data(), 0, nullptr, nullptr) == GST_OK);
    F().RunLate();
    uint32_t got = ~0u;
    CHECK(gst_read_error_bits(s, &got) == GST_OK);
    CHECK(got == bits);
  }
}

// What a caller may record into a graph holds no hipMemsetAsync.
void AsyncErrorBits() {
  const auto f = File();
  const gst_header h = Header(f);
  std::vector<uint8_t> out(h.width * h.height / 2), staging(512 + f.size());
  gst_batch *b = NewBatch(h);
  hipStream_t s = NewStream();
  Bind(b, h, f, &out, s);
  uint32_t got = 0;
  CHECK(gst_read_error_bits(s, &got) == GST_OK);  // the stream's word is there from here on
  const int before = F().memsets;
  for (uint32_t bits : {4u, 0u, 6u}) {
    F().raise = bits;
    CHECK(gst_load_compressed_dxt(&h, s, staging.data(), out.data(), 0, nullptr, nullptr) == GST_OK);
    CHECK(gst_read_error_bits_async(s, &got) == GST_OK);
    CHECK(got == bits);
    CHECK(gst_batch_decode(b, s) == GST_OK);
    CHECK(gst_batch_error_bits_async(b, s, &got) == GST_OK);
    CHECK(got == bits);
  }
  CHECK(F().memsets == before);
  gst_batch_destroy(b);
}

// The server's comparison flags and plans are cleared before its first request.
void ServerLeavesNothingBehind() {
  gst_server_config c{};
  c.hbm_budget_bytes = 1 << 20;
  c.host_staging_bytes = 1 << 20;
  c.max_batch_images = 4;
  c.max_batch_blocks = 1 << 16;
  gst_server *s = nullptr;
  CHECK(gst_server_create(&c, &s) == GST_OK);
  CHECK(F().late.empty());
  gst_server_destroy(s);
}

// One stand-alone stream of one word.
struct AnsCall {
  gst_ans_decoder *d = nullptr;
  uint8_t syms[GST_ANS_SYMBOLS_PER_STREAM] = {};
  AnsCall() {
    const uint32_t counts[2] = {1, 1};
    CHECK(gst_ans_decoder_create(counts, 2, 1, &d) == GST_OK);
  }
  ~AnsCall() { gst_ans_decoder_destroy(d); }
  int Decode() {
    const uint32_t state = 1u << 15;
    const uint8_t word[2] = {};
    const uint8_t *const data[1] = {word};
    const size_t len[1] = {2};
    return gst_ans_decode(d, &state, 1, data, len, 1, syms);
  }
};

// A call whose wait failed may leave a kernel writing to its buffer: no later call gets it.
void PinnedAfterFailedWait() {
  const auto f = File();
  std::vector<uint8_t> out(Header(f).width * Header(f).height / 2);
  CHECK(gst_decompress_dxt(f.data(), f.size(), out.data(), out.size()) == GST_OK);
  void *const first = F().out;
  F().fail_waits = 1;
  CHECK(gst_decompress_dxt(f.data(), f.size(), out.data(), out.size()) == GST_ERR_HIP);
  CHECK(F().out == first);  // kept after the call that succeeded
  CHECK(gst_decompress_dxt(f.data(), f.size(), out.data(), out.size()) == GST_OK);
  CHECK(F().out != first);

  AnsCall a;
  F().fail_waits = 1;
  CHECK(a.Decode() == GST_ERR_HIP);
  void *const failed = F().out;
  CHECK(a.Decode() == GST_OK);
  CHECK(F().out != failed);
}

// Host-to-host calls go on without pinned memory: from the first, and when it runs out.
void NoPinnedMemory() {
  const auto f = File();
  AnsCall a;
  for (bool none : {true, false, true}) {
    F().no_pinned = none;
    if (none) gst_free_decompressor();
    std::vector<uint8_t> out(Header(f).width * Header(f).height / 2);
    CHECK(gst_decompress_dxt(f.data(), f.size(), out.data(), out.size()) == GST_OK);
    for (uint8_t v : out) CHECK(v == kBlock);
    F().raise = 4;
    CHECK(gst_decompress_dxt(f.data(), f.size(), out.data(), out.size()) == GST_ERR_CORRUPT_STREAM);
    F().raise = 0;
    std::memset(a.syms, 0, sizeof(a.syms));
    CHECK(a.Decode() == GST_OK);
    for (uint8_t v : a.syms) CHECK(v == kBlock);
  }
}

// A call that fits the device's memory goes on where the size it would keep does not.
void LittleDeviceMemory() {
  const auto f = File();
  const gst_header h = Header(f);
  std::vector<uint8_t> out(h.width * h.height / 2), staging(512 + f.size());
  CHECK(gst_decompress_dxt(f.data(), f.size(), out.data(), out.size()) == GST_OK);
  gst_free_decompressor();
  F().most = size_t{300} << 10;  // the scratch is 177 KiB, kept scratch at least 1 MiB
  CHECK(gst_decompress_dxt(f.data(), f.size(), out.data(), out.size()) == GST_OK);
  CHECK(gst_load_compressed_dxt(&h, nullptr, staging.data(), out.data(), 0, nullptr, nullptr) == GST_OK);
}

// Calls too large for a buffer that is kept pin nothing for themselves.
void LargeHostCalls() {
  const auto f = File(16384, 8192);
  std::vector<uint8_t> out(size_t{16384} * 8192 / 2);
  CHECK(gst_decompress_dxt(f.data(), f.size(), out.data(), out.size()) == GST_OK);
  for (uint8_t v : out) CHECK(v == kBlock);
  const uint32_t groups = 8192, lanes = 32, counts[2] = {1, 1};
  gst_ans_decoder *d = nullptr;
  CHECK(gst_ans_decoder_create(counts, 2, lanes, &d) == GST_OK);
  const uint8_t word[2] = {};
  const std::vector<uint32_t> states(groups * lanes, 1u << 15);
  const std::vector<const uint8_t *> data(groups, word);
  const std::vector<size_t> lens(groups, 2);
  std::vector<uint8_t> syms(states.size() * GST_ANS_SYMBOLS_PER_STREAM);
  CHECK(gst_ans_decode(d, states.data(), groups * lanes, data.data(), lens.data(), groups, syms.data()) == GST_OK);
  for (uint8_t v : syms) CHECK(v == kBlock);
  gst_ans_decoder_destroy(d);
  CHECK(F().pinned <= size_t{64} << 20);
}

const std::map<std::string, void (*)()> kChecks = {
    {"little_lds", DeviceWithLittleLds},
    {"batch_plan", BatchPlanSurvives},
    {"batch_error_bits", BatchErrorBitsSurvive},
    {"stream_error_bits", StreamErrorBitsSurvive},
    {"async_error_bits", AsyncErrorBits},
    {"server_flags", ServerLeavesNothingBehind},
    {"pinned_after_failed_wait", PinnedAfterFailedWait},
    {"no_pinned_memory", NoPinnedMemory},
    {"little_device_memory", LittleDeviceMemory},
    {"large_host_calls", LargeHostCalls},
};

}  // namespace

int main(int argc, char **argv) {
  if (argc != 2 || !kChecks.count(argv[1])) return 2;
  kChecks.at(argv[1])();
  std::puts("ok");
  return 0;
}
