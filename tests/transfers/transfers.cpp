// TEST INFRASTRUCTURE ONLY: state uploads and downloads (csrc/host/rsim.cpp) on a runtime of host memory, for what a GPU
// cannot be made to do in a test: a copy that fails between two others, and a device without room. Copies and packs are
// queued and done when the stream is synchronised, so whatever a call leaves queued is still to read or write its caller's
// memory. Prints "ok" or the first check that does not hold.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <functional>
#include <map>
#include <vector>

#include "device/launch.h"
#include "rsim.h"

namespace {
size_t g_room = ~(size_t)0;  // bytes that the device still has
std::map<void*, size_t> g_live;
std::vector<std::function<void()>> g_queue;
int g_mallocs = 0, g_frees = 0, g_copies = 0, g_failing_copy = -1;

#define CHECK(x)                                             \
  do {                                                       \
    if (!(x)) {                                              \
      printf("line %d: %s (%s)\n", __LINE__, #x, rsim_last_error()); \
      exit(0);                                               \
    }                                                        \
  } while (0)
}  // namespace

extern "C" {
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = (hipStream_t)16, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = (hipEvent_t)16, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* st) { return *st = hipStreamCaptureStatusNone, hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorName(hipError_t) { return "error"; }
const char* hipGetErrorString(hipError_t) { return "of the test's runtime"; }
hipError_t hipMalloc(void** p, size_t bytes) {
  ++g_mallocs;
  *p = nullptr;
  if (bytes > g_room) return hipErrorOutOfMemory;
  g_room -= bytes;
  *p = malloc(bytes);
  g_live[*p] = bytes;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  ++g_frees;
  CHECK(g_live.count(p) == 1);
  g_room += g_live[p];
  g_live.erase(p);
  free(p);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  for (auto& f : g_queue) f();
  g_queue.clear();
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) { return g_queue.push_back([=] { memset(p, v, n); }), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  if (g_copies++ == g_failing_copy) return hipErrorUnknown;
  return g_queue.push_back([=] { memcpy(d, s, n); }), hipSuccess;
}
}

namespace rs {
namespace dev {
hipError_t order_scratch_address(uint32_t** out) { return *out = nullptr, hipSuccess; }
hipError_t stepping_static_lds(size_t* bytes) { return *bytes = 0, hipSuccess; }
hipError_t launch_pack_states(hipStream_t, const uint32_t* aos, uint32_t* blocks, uint32_t n) {
  return g_queue.push_back([=] { rsim_aosoa_pack(aos, n, blocks); }), hipSuccess;
}
hipError_t launch_unpack_states(hipStream_t, const uint32_t* blocks, uint32_t* aos, uint32_t n) {
  return g_queue.push_back([=] { rsim_aosoa_unpack(blocks, n, aos); }), hipSuccess;
}
}  // namespace dev
}  // namespace rs

namespace {
std::vector<uint32_t> make_states(uint32_t n, uint32_t seed) {
  std::vector<uint32_t> v((size_t)n * rs::ARENA_WORDS);
  for (size_t i = 0; i < v.size(); ++i) v[i] = (uint32_t)(i * 2654435761u) ^ seed;
  return v;
}
// Up into dst, the buffer's words checked, and down again.
void round_trip(rsim_device* dev, rsim_states* dst, uint32_t n, uint32_t seed) {
  const std::vector<uint32_t> in = make_states(n, seed);
  std::vector<uint32_t> out(in.size()), words(rsim_aosoa_words(n));
  CHECK(rsim_write_states(dev, dst, in.data()) == RSIM_OK && g_queue.empty());
  CHECK(rsim_aosoa_pack(in.data(), n, words.data()) == RSIM_OK);
  CHECK(memcmp(rsim_states_device_ptr(dst), words.data(), words.size() * 4) == 0);
  CHECK(rsim_download_states(dev, dst, out.data()) == RSIM_OK && g_queue.empty());
  CHECK(out == in);
}

// A copy fails with others of the same transfer queued before it: the call returns its error with nothing left queued.
void failing_copy(rsim_device* dev) {
  const uint32_t n = 3 * 6144;
  rsim_states* s = nullptr;
  CHECK(rsim_alloc_states(dev, n, &s) == RSIM_OK);
  std::vector<uint32_t> host = make_states(n, 1);
  for (int k = 0; k < 3; ++k) {
    g_failing_copy = g_copies + k;
    CHECK(rsim_write_states(dev, s, host.data()) == RSIM_ERR_HIP);
    CHECK(g_queue.empty());
    g_failing_copy = g_copies + k;
    CHECK(rsim_download_states(dev, s, host.data()) == RSIM_ERR_HIP);
    CHECK(g_queue.empty());
  }
  round_trip(dev, s, n, 2);
  CHECK(rsim_states_free(s) == RSIM_OK);
}
// A device that has room for the caller's buffers and no more: transfers work all the same.
void full_device(rsim_device* dev) {
  for (uint32_t n : {1u, 200u, 6500u}) {
    rsim_states* s = nullptr;
    g_room = rsim_aosoa_words(n) * 4;
    CHECK(rsim_alloc_states(dev, n, &s) == RSIM_OK);
    round_trip(dev, s, n, 3);
    CHECK(rsim_states_free(s) == RSIM_OK);
    const std::vector<uint32_t> in = make_states(n, 4);
    CHECK(rsim_upload_states(dev, in.data(), n, &s) == RSIM_OK);
    CHECK(rsim_states_free(s) == RSIM_OK);
  }
}
// A device with room for a small staging buffer, or none: the transfers after the first neither free it nor ask for more,
// until a buffer of the device is freed.
void small_stage(rsim_device*& dev) {
  const size_t arena = rs::ARENA_WORDS * 4;
  for (uint32_t room : {0u, 130u, 900u}) {
    rsim_states *s = nullptr, *other = nullptr;
    const uint32_t n = 2000;
    g_room = 2 * rsim_aosoa_words(n) * 4 + room * arena;
    CHECK(rsim_alloc_states(dev, n, &s) == RSIM_OK && rsim_alloc_states(dev, n, &other) == RSIM_OK);
    round_trip(dev, s, n, 5);
    const int mallocs = g_mallocs, frees = g_frees;
    for (uint32_t k = 0; k < 3; ++k) {
      round_trip(dev, s, n, 6 + k);
      CHECK(g_mallocs == mallocs && g_frees == frees);
    }
    CHECK(rsim_states_free(other) == RSIM_OK);
    round_trip(dev, s, n, 9);
    CHECK(g_room == rsim_aosoa_words(n) * 4 + room * arena - n * arena);  // now the whole batch is staged at once
    CHECK(rsim_states_free(s) == RSIM_OK);
    rsim_device* fresh = nullptr;  // the next case starts without a staging buffer
    CHECK(rsim_open(0, &fresh) == RSIM_OK && rsim_close(dev) == RSIM_OK);
    dev = fresh;
  }
}
// The staging buffer stands in no allocation's way: a buffer that fits only without it gets its room.
void given_back(rsim_device* dev) {
  const uint32_t n = 512, worlds = 3;
  const uint64_t words = rsim_aosoa_words(n);
  rsim_states *s = nullptr, *t = nullptr;
  rsim_words* b = nullptr;
  rsim_world* w = nullptr;
  CHECK(rsim_alloc_states(dev, n, &s) == RSIM_OK);
  const std::vector<uint32_t> table((size_t)rs::STATIC_WORDS * worlds);
  for (int kind = 0; kind < 4; ++kind) {
    g_room = (size_t)n * rs::ARENA_WORDS * 4;
    round_trip(dev, s, n, 10 + kind);  // the staging buffer takes all of it
    CHECK(g_room == 0);
    if (kind == 0) CHECK(rsim_alloc_states(dev, n, &t) == RSIM_OK && rsim_states_free(t) == RSIM_OK);
    if (kind == 1) CHECK(rsim_alloc_words(dev, words, &b) == RSIM_OK && rsim_words_free(b) == RSIM_OK);
    if (kind == 2) CHECK(rsim_upload_worlds(dev, table.data(), worlds, &w) == RSIM_OK && rsim_world_free(w) == RSIM_OK);
    if (kind == 3) CHECK(rsim_alloc_words(dev, words + 1, &b) == RSIM_ERR_HIP);
  }
  round_trip(dev, s, n, 14);
  CHECK(rsim_states_free(s) == RSIM_OK);
}
}  // namespace

int main(int argc, char** argv) {
  const char* what = argc > 1 ? argv[1] : "";
  rsim_device* dev = nullptr;
  CHECK(rsim_open(0, &dev) == RSIM_OK);
  if (!strcmp(what, "failing_copy")) failing_copy(dev);
  else if (!strcmp(what, "full_device")) full_device(dev);
  else if (!strcmp(what, "small_stage")) small_stage(dev);
  else if (!strcmp(what, "given_back")) given_back(dev);
  else CHECK(!"a known case");
  CHECK(rsim_close(dev) == RSIM_OK && g_live.empty());
  printf("ok\n");
  return 0;
}
