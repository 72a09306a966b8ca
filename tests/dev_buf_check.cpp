// Host check of csrc/dev_buf.h on a runtime of its own: hipMalloc / hipFree keep
// a list of owned blocks, the capture state is a variable.  Prints "failures=0".
#include <cstdio>
#include <map>

#include "dev_buf.h"

static std::map<void *, size_t> g_owned;
static bool g_capturing = false;
static size_t g_room = (size_t)1 << 40;  // bytes the device still has

hipError_t hipMalloc(void **p, size_t n) {
  if (g_capturing) return hipErrorStreamCaptureUnsupported;
  if (n > g_room) return hipErrorOutOfMemory;
  static size_t next = 0;  // no address twice
  *p = (void *)(next += 4096);
  g_owned[*p] = n;
  g_room -= n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  auto it = g_owned.find(p);
  if (it == g_owned.end()) return hipErrorInvalidValue;
  g_room += it->second;
  g_owned.erase(it);
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *st) {
  *st = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }

static int g_fail = 0;
#define EXPECT(c) \
  do { \
    if (!(c)) std::printf("line %d: %s\n", __LINE__, #c), ++g_fail; \
  } while (0)

using qh::Carve;
using qh::DevBuf;

static Carve carve(size_t bytes) {
  Carve c;
  c.add(bytes);
  return c;
}

// A graph captured on a small block, then a call that needs a larger one.
static void captured_block_outlives_growth() {
  DevBuf b;
  const hipStream_t s = nullptr;
  std::vector<char *> small, big;
  EXPECT(carve(800 << 10).try_bind(b, s, &small));  // eager warm-up
  g_capturing = true;
  std::vector<char *> in_graph;
  EXPECT(carve(800 << 10).try_bind(b, s, &in_graph));
  EXPECT(in_graph[0] == small[0]);
  EXPECT(!carve(2 << 20).try_bind(b, s, &big));  // no growth inside a capture
  EXPECT(b.p == in_graph[0]);
  g_capturing = false;
  EXPECT(carve(2 << 20).try_bind(b, s, &big));
  EXPECT(big[0] != in_graph[0]);
  EXPECT(g_owned.count(in_graph[0]) == 1);  // what a replay writes to
  EXPECT(carve(4 << 20).bind(b, s)[0] != big[0]);
  EXPECT(g_owned.count(in_graph[0]) == 1);
  EXPECT(g_owned.count(big[0]) == 0);  // no graph holds this one
  EXPECT(g_owned.size() == 2);
  b.release();
  EXPECT(g_owned.empty());
}

// The same through bind(), and the kept blocks stay below the one in use.
static void kept_blocks_are_bounded() {
  DevBuf b;
  const hipStream_t s = nullptr;
  for (size_t need = 1 << 20; need <= (size_t)64 << 20; need += 1 << 20) {
    carve(need).bind(b, s);
    g_capturing = true;
    carve(need).bind(b, s);
    g_capturing = false;
  }
  size_t all = 0;
  for (auto &o : g_owned) all += o.second;
  EXPECT(all < 2 * b.cap);
  b.release();
  EXPECT(g_owned.empty());
}

// Without captures a buffer is one block.
static void eager_growth_frees() {
  DevBuf b;
  for (size_t need = 1; need < 10000; need *= 3) carve(need).bind(b, (hipStream_t) nullptr);
  EXPECT(g_owned.size() == 1);
  b.release();
  EXPECT(g_owned.empty() && b.p == nullptr && b.cap == 0);
}

int main() {
  captured_block_outlives_growth();
  kept_blocks_are_bounded();
  eager_growth_frees();
  std::printf("failures=%d\n", g_fail);
  return g_fail != 0;
}
