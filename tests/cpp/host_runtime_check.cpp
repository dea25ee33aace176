// The C ABI's host side without a GPU: this program defines the HIP runtime
// functions that librasterizer_amd.so calls (the program's definitions come
// before the library's own dependencies), with device memory as host memory and
// kernel launches that do nothing but are recorded.  It counts allocations,
// checks that what is freed was allocated, and can make allocations fail.
// Run with the name of a check; exits 0 when it holds (tests/test_host_runtime.py).
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <set>
#include <vector>

#include "rasterizer_amd.h"
#include "rz_kernels.h"
#include "rz_scratch.h"

namespace {

struct Runtime {
  std::set<void*> device, pinned;
  std::vector<size_t> deviceSizes, pinnedSizes;  // of every allocation asked for
  int badFrees = 0;                              // of memory that is not allocated
  int streamSyncs = 0;
  int failDevice = -1, failPinned = -1;  // allocations that succeed before every further one fails (-1: all do)
  dim3 grid;                             // of the last launch
  unsigned largestGrid = 0;
  size_t largestNew = ~size_t(0);        // operator new fails for more
  bool zeroWords = false;                // copies of 16 bytes to the host read as zeros
  hipError_t lastError = hipSuccess;     // what the next hipGetLastError reports
};
Runtime& rt() {
  static Runtime r;
  return r;
}

hipError_t allocate(std::set<void*>& live, std::vector<size_t>& sizes, int& fail, void** p, size_t bytes) {
  sizes.push_back(bytes);
  *p = nullptr;
  if (fail == 0) return rt().lastError = hipErrorOutOfMemory;
  if (fail > 0) --fail;
  *p = std::calloc(bytes ? bytes : 1, 1);  // untouched pages cost nothing
  if (!*p) return hipErrorOutOfMemory;
  live.insert(*p);
  return hipSuccess;
}
hipError_t release(std::set<void*>& live, void* p) {
  if (!p) return hipSuccess;
  if (live.erase(p) == 0) {
    ++rt().badFrees;
    return hipErrorInvalidValue;
  }
  std::free(p);
  return hipSuccess;
}
void copy(void* dst, const void* src, size_t n) { std::memmove(dst, src, n); }

void copy_out(void* dst, const void* src, size_t n, hipMemcpyKind kind) {
  copy(dst, src, n);
  if (kind == hipMemcpyDeviceToHost && n == 16 && rt().zeroWords) std::memset(dst, 0, n);
}

int object;  // what streams, events and graphs point to

}  // namespace

void* operator new(size_t n) {
  void* p = n > rt().largestNew ? nullptr : std::malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  const hipError_t e = allocate(rt().device, rt().deviceSizes, rt().failDevice, p, n);
  if (e == hipSuccess && n <= size_t(1) << 20) std::memset(*p, 0xAB, n);  // device memory is not cleared
  return e;
}
hipError_t hipFree(void* p) { return release(rt().device, p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  return allocate(rt().pinned, rt().pinnedSizes, rt().failPinned, p, n);
}
hipError_t hipHostFree(void* p) { return release(rt().pinned, p); }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { return *d = h, hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return copy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind kind, hipStream_t) {
  return copy_out(d, s, n, kind), hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  return *s = reinterpret_cast<hipStream_t>(&object), hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return ++rt().streamSyncs, hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = reinterpret_cast<hipEvent_t>(&object), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0.0f, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
  std::memset(p, 0, sizeof *p);
  std::strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static void* symbol = std::calloc(size_t(64) << 20, 1);  // the draw's static device array
  return *p = symbol, hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  return *n = 2, hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = rt().lastError;
  rt().lastError = hipSuccess;
  return e;
}
hipError_t hipLaunchKernel(const void*, dim3 grid, dim3, void**, size_t, hipStream_t) {
  rt().grid = grid;
  if (grid.x > rt().largestGrid) rt().largestGrid = grid.x;
  return hipSuccess;
}
hipError_t hipLaunchCooperativeKernel(const void* f, dim3 g, dim3 b, void** a, unsigned s, hipStream_t st) {
  return hipLaunchKernel(f, g, b, a, s, st);
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3, size_t, hipStream_t) { return rt().grid = grid, hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream) {
  *grid = rt().grid;
  *block = dim3(1);
  *shared = 0;
  *stream = nullptr;
  return hipSuccess;
}
}

namespace {

int failures = 0;
#define CHECK(cond)                                                     \
  do {                                                                  \
    if (!(cond)) {                                                      \
      std::printf("line %d: %s does not hold\n", __LINE__, #cond);      \
      ++failures;                                                       \
    }                                                                   \
  } while (0)

rz_context* context(uint32_t w, uint32_t h) {
  rz_context* c = nullptr;
  CHECK(rz_create(w, h, &c) == RZ_OK);
  return c;
}

// rz_sync and rz_readback_raw allocate nothing, on a fresh context too, and
// wait for the stream when no memory can be had.
void blocking_calls() {
  rz_context* c = context(64, 64);
  std::vector<uint16_t> depth(64 * 64), hiz(64 + 8);
  const size_t device = rt().deviceSizes.size(), pinned = rt().pinnedSizes.size();
  rt().failDevice = rt().failPinned = 0;
  for (int i = 0; i < 2; ++i) {
    int before = rt().streamSyncs;
    CHECK(rz_sync(c) == RZ_OK);
    CHECK(rt().streamSyncs > before);
    before = rt().streamSyncs;
    CHECK(rz_readback_raw(c, depth.data(), hiz.data()) == RZ_OK);
    CHECK(rt().streamSyncs > before);
    int visible = 0, clip = 0;
    const float lo[4] = {0, 0, 0, 1}, hi[4] = {1, 1, 1, 1};
    CHECK(rz_query(c, lo, hi, &visible, &clip) == RZ_OK);
    CHECK(rz_query2d(c, 0, 7, 0, 7, 9, &visible) == RZ_OK);
  }
  CHECK(rt().deviceSizes.size() == device && rt().pinnedSizes.size() == pinned);
  rt().failDevice = rt().failPinned = -1;
  CHECK(rz_destroy(c) == RZ_OK);
}

// A context that cannot be made whole is not made, and nothing of it is left.
void failed_creation() {
  for (int n = 0;; ++n) {
    rt().failPinned = n;
    rz_context* c = nullptr;
    const int s = rz_create(64, 64, &c);
    rt().failPinned = -1;
    if (s == RZ_OK) {
      CHECK(n > 0);
      CHECK(rz_destroy(c) == RZ_OK);
      break;
    }
    CHECK(s == RZ_ERR_OUT_OF_MEMORY && !c);
    CHECK(rt().device.empty() && rt().pinned.empty());
  }
}

// An error that another HIP call left behind is not theirs: they wait and give
// their results.
void error_left_behind() {
  rz_context* c = context(64, 64);
  std::vector<uint16_t> depth(64 * 64), hiz(64 + 8);
  int before = rt().streamSyncs;
  rt().lastError = hipErrorInvalidValue;
  CHECK(rz_sync(c) == RZ_OK);
  CHECK(rt().streamSyncs > before);
  before = rt().streamSyncs;
  rt().lastError = hipErrorInvalidValue;
  CHECK(rz_readback_raw(c, depth.data(), hiz.data()) == RZ_OK);
  CHECK(rt().streamSyncs > before);
  CHECK(rz_destroy(c) == RZ_OK);
}

// Scene preparation's working memory: what a call used, and half as much again,
// is one block from the next call on, unless it is more than is kept; a small call
// after such a one allocates no more than it takes.
void scratch() {
  using rzd::Scratch;
  {
    Scratch s;
    auto call = [&](size_t part, int parts) {
      const size_t before = rt().deviceSizes.size();
      Scratch::Frame frame(s);
      for (int i = 0; i < parts; ++i) CHECK(s.take<unsigned char>(part) != nullptr);
      return rt().deviceSizes.size() - before;
    };
    CHECK(call(1 << 20, 46) == 46);
    CHECK(call(1 << 20, 46) == 1 && rt().deviceSizes.back() == size_t(69) << 20);
    CHECK(call(1 << 20, 46) == 0);
    for (int parts = 47; parts < 69; ++parts) CHECK(call(1 << 20, parts) == 0);  // growing calls
    CHECK(call(1000, 3) == 0);
    CHECK(call(Scratch::kKeepDevice / 2, 5) == 5);
    CHECK(rt().device.empty());  // too large to be kept
    CHECK(call(Scratch::kKeepDevice / 2, 5) == 1 && rt().deviceSizes.back() == 5 * Scratch::kKeepDevice / 2);
    CHECK(call(1000, 3) == 3);
    for (size_t k = rt().deviceSizes.size() - 3; k < rt().deviceSizes.size(); ++k) CHECK(rt().deviceSizes[k] == 1024);
    CHECK(call(Scratch::kKeepDevice / 2, 5) > 0);
    CHECK(call(1000, 3) == 3);
    CHECK(call(1000, 3) == 1);
    rt().pinnedSizes.clear();
    for (size_t bytes = 1000; bytes <= Scratch::kMaxHost; bytes += bytes / 16 + 100) CHECK(s.host(bytes) != nullptr);
    CHECK(s.host(Scratch::kMaxHost) != nullptr && s.host(Scratch::kMaxHost + 1) == nullptr);
    CHECK(rt().pinnedSizes.size() <= 18 && rt().pinnedSizes.back() == Scratch::kMaxHost);
    rt().failDevice = 0;
    Scratch::Frame frame(s);
    CHECK(s.take<int>(100) != nullptr && s.take<int>(1 << 20) == nullptr);
    rt().failDevice = -1;
  }
}

// The scene box over as many vertices as a call can have: its launches have
// work-groups, no more than there are partial results.
void scene_box_sizes() {
  for (uint32_t n : {0u, 1u, 256u, 257u, 131072u, 131073u, 0xFFFE0001u, 0xFFFFFF01u, 0xFFFFFFFFu}) {
    rt().largestGrid = 0;
    CHECK(rzd::launch_scene_boxes(nullptr, 8, 8, reinterpret_cast<const float*>(&object), n, nullptr, nullptr, nullptr,
                                  nullptr) == hipSuccess);
    CHECK(rt().largestGrid == (n < 131072u ? n / 256u + (n % 256u != 0u || n == 0u) : rzd::kSceneParts));
  }
}

// Host memory that cannot be had is a status, not an exception through the C ABI.
void no_host_memory() {
  rz_context* c = context(64, 64);
  std::vector<uint64_t> cov(4096);
  rt().largestNew = 4096;
  CHECK(rz_get_tables(c, cov.data(), nullptr) == RZ_OK);
  rt().largestNew = ~size_t(0);
  const uint32_t n = 50000;
  std::vector<float> boxes(size_t(n) * 8);  // from malloc: 16-byte aligned
  std::vector<uint32_t> idx(n), offsets(n + 1);
  uint32_t count = 0;
  rt().zeroWords = true;  // the pass's words: no error, no open range
  CHECK(rz_sah_batches(c, n, boxes.data(), 512, 8, idx.data(), offsets.data(), &count) == RZ_OK);
  rt().largestNew = 4096;
  CHECK(rz_sah_batches(c, n, boxes.data(), 512, 8, idx.data(), offsets.data(), &count) == RZ_ERR_OUT_OF_MEMORY);
  rt().largestNew = ~size_t(0);
  CHECK(rz_destroy(c) == RZ_OK);
}

// Buffers that grow and cannot: the call says so, what it freed is not freed
// again, and the next call with memory works and reports no error of this one.
void failed_growth() {
  std::vector<uint32_t> packets(4 * 8 * 4);
  std::vector<float> boxes(8 * 200000);
  std::vector<uint8_t> visible(200000);
  const float lo[4] = {0, 0, 0, 1}, hi[4] = {1, 1, 1, 1};
  for (int n = 0; n < 12; ++n) {
    rz_context* c = context(64, 64);
    rz_occluder* o = nullptr;
    CHECK(rz_occluder_create(c, packets.data(), 16, lo, hi, lo, hi, &o) == RZ_OK);
    auto draw = [&](uint32_t count) {
      std::vector<const rz_occluder*> items(count, o);
      return rz_draw_frame(c, count, items.data(), nullptr);
    };
    auto query = [&](uint32_t count) { return rz_query_batch(c, count, boxes.data(), visible.data(), nullptr); };
    CHECK(draw(3) == RZ_OK && query(150000) == RZ_OK);
    rt().failDevice = n;
    const int d = draw(1000), q = query(200000);
    CHECK((d == RZ_OK || d == RZ_ERR_OUT_OF_MEMORY) && (q == RZ_OK || q == RZ_ERR_OUT_OF_MEMORY));
    CHECK((d == RZ_OK && q == RZ_OK) == (n >= 12));
    if (n % 2) {
      rt().failDevice = -1;
      CHECK(draw(2000) == RZ_OK && query(200000) == RZ_OK);
    }
    rt().failDevice = -1;
    CHECK(rz_sync(c) == RZ_OK);
    CHECK(rz_occluder_destroy(o) == RZ_OK && rz_destroy(c) == RZ_OK);
    CHECK(rt().badFrees == 0 && rt().device.empty());
  }
}

// The same for a views object's plan and a model's buffers.
void failed_plans() {
  std::vector<uint32_t> packets(4 * 8 * 4);
  std::vector<float> boxes(8 * 1000), x(16 * 1000), grad(5313);
  const float lo[4] = {0, 0, 0, 1}, hi[4] = {1, 1, 1, 1}, eye[3] = {1, 2, 3};
  const uint32_t size[2] = {64, 64}, pairs[2] = {0, 1};
  rz_context* c = context(64, 64);
  rz_occluder* o = nullptr;
  CHECK(rz_occluder_create(c, packets.data(), 16, lo, hi, lo, hi, &o) == RZ_OK);
  bool failed = true;
  for (int n = 0; failed && n < 100; ++n)
    for (int pinned = 0; pinned < 2; ++pinned) {
      int& fail = pinned ? rt().failPinned : rt().failDevice;
      rz_views* v = nullptr;
      rz_mlp* m = nullptr;
      CHECK(rz_views_create(2, size, size, &v) == RZ_OK && rz_mlp_create(1, &m) == RZ_OK);
      for (uint32_t k = 0; k < 2; ++k)
        CHECK(rz_views_set_occluders(v, k, 1, &o) == RZ_OK && rz_views_set_queries(v, k, 1000, boxes.data()) == RZ_OK &&
              rz_views_set_eye(v, k, eye) == RZ_OK);
      fail = n;
      const int r = rz_views_run(v, 0);
      fail = n;
      const int g = rz_mlp_gradients(m, 1000, x.data(), 1, pairs, grad.data(), nullptr);
      fail = -1;
      CHECK((r == RZ_OK || r == RZ_ERR_OUT_OF_MEMORY) && (g == RZ_OK || g == RZ_ERR_OUT_OF_MEMORY));
      CHECK(n > 0 || (r != RZ_OK && g != RZ_OK));
      // No step has run: no box is visible.
      std::vector<uint8_t> visible(1000, 7), clip(1000, 7);
      CHECK(rz_views_read_queries(v, 1, visible.data(), clip.data()) == RZ_OK);
      for (int k = 0; k < 1000; ++k) CHECK(visible[k] == 0 && clip[k] == 0);
      if (!pinned) failed = r != RZ_OK || g != RZ_OK;
      CHECK(rz_views_run(v, 0) == RZ_OK && rz_views_sync(v, nullptr) == RZ_OK);
      CHECK(rz_mlp_gradients(m, 1000, x.data(), 1, pairs, grad.data(), nullptr) == RZ_OK);
      CHECK(rz_views_destroy(v) == RZ_OK && rz_mlp_destroy(m) == RZ_OK && rt().badFrees == 0);
    }
  CHECK(!failed);
  CHECK(rz_occluder_destroy(o) == RZ_OK && rz_destroy(c) == RZ_OK);
}

// Answers of a step come back through a bounded pinned buffer, and without it
// where it cannot be had.
void view_answers() {
  rz_context* c = context(64, 64);
  const uint32_t size[3] = {64, 64, 64}, counts[3] = {1500000, 0, 700000};
  std::vector<float> boxes(size_t(counts[0]) * 8);
  std::vector<uint8_t> visible(counts[0]), clip(counts[0]);
  rz_views* v = nullptr;
  CHECK(rz_views_create(3, size, size, &v) == RZ_OK);
  for (uint32_t k = 0; k < 3; ++k) CHECK(rz_views_set_queries(v, k, counts[k], boxes.data()) == RZ_OK);
  CHECK(rz_views_run(v, 0) == RZ_OK && rz_views_sync(v, nullptr) == RZ_OK);
  for (int pinned : {0, -1}) {
    rt().failPinned = pinned;
    rt().pinnedSizes.clear();
    for (uint32_t k : {2u, 0u, 1u, 2u}) {
      std::memset(visible.data(), 7, visible.size());
      std::memset(clip.data(), 7, clip.size());
      CHECK(rz_views_read_queries(v, k, visible.data(), clip.data()) == RZ_OK);
      for (uint32_t i = 0; i < counts[k]; i += 997) CHECK(visible[i] == 0 && clip[i] == 0);
      CHECK(counts[k] == counts[0] || (visible[counts[k]] == 7 && clip[counts[k]] == 7));
    }
    for (size_t n : rt().pinnedSizes) CHECK(n <= size_t(2) << 20);
  }
  rt().failPinned = -1;
  CHECK(rz_views_destroy(v) == RZ_OK && rz_destroy(c) == RZ_OK);
}

// Batches and views' answers that grow from call to call seldom pin memory anew.
void growing_calls() {
  rz_context* c = context(64, 64);
  std::vector<float> boxes(size_t(131072) * 8);
  std::vector<uint8_t> visible(131072);
  rt().pinnedSizes.clear();
  for (uint32_t n = 500; n <= 131072; n += 500)
    CHECK(rz_query_batch(c, n, boxes.data(), visible.data(), nullptr) == RZ_OK);
  CHECK(rz_query_batch(c, 131072, boxes.data(), visible.data(), nullptr) == RZ_OK);
  CHECK(rt().pinnedSizes.size() <= 9);
  const uint32_t size = 64;
  rz_views* v = nullptr;
  CHECK(rz_views_create(1, &size, &size, &v) == RZ_OK);
  const size_t before = rt().pinnedSizes.size();
  uint32_t steps = 0;
  for (uint32_t n = 1000; n <= 131072; n += 1000, ++steps) {
    CHECK(rz_views_set_queries(v, 0, n, boxes.data()) == RZ_OK);
    CHECK(rz_views_run(v, 0) == RZ_OK && rz_views_sync(v, nullptr) == RZ_OK);
    CHECK(rz_views_read_queries(v, 0, visible.data(), nullptr) == RZ_OK);
  }
  // A changed number of queries makes a new plan, whose view table is pinned.
  CHECK(rt().pinnedSizes.size() - before <= steps + 9);
  CHECK(rz_views_destroy(v) == RZ_OK && rz_destroy(c) == RZ_OK);
}

struct Check {
  const char* name;
  void (*run)();
};
const Check checks[] = {{"blocking_calls", blocking_calls},
                        {"error_left_behind", error_left_behind},
                        {"failed_creation", failed_creation},
                        {"scratch", scratch},
                        {"scene_box_sizes", scene_box_sizes},
                        {"no_host_memory", no_host_memory},
                        {"failed_growth", failed_growth},
                        {"failed_plans", failed_plans},
                        {"view_answers", view_answers},
                        {"growing_calls", growing_calls}};

}  // namespace

int main(int argc, char** argv) {
  for (const Check& c : checks) {
    if (argc > 1 && std::strcmp(argv[1], c.name) != 0) continue;
    c.run();
    CHECK(rt().badFrees == 0);
    CHECK(rt().device.empty() && rt().pinned.empty());
    std::printf("%s: %s\n", c.name, failures ? "failed" : "ok");
    return failures ? 1 : 0;
  }
  std::printf("no such check\n");
  return 2;
}
