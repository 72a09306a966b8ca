// Host check of csrc/dev_buf.h on a runtime of its own: hipMalloc / hipFree keep
// a list of owned blocks, the capture state is a variable.  Prints "failures=0".
#include <cstdio>
#include <map>

#include "dev_buf.h"

static std::map<void *, size_t> g_owned;
static bool g_capturing = false;
static size_t g_room = (size_t)1 << 40;  // bytes the device still has
static int g_mallocs = 0, g_frees = 0;

hipError_t hipMalloc(void **p, size_t n) {
  ++g_mallocs;
  if (g_capturing) return hipErrorStreamCaptureUnsupported;
  if (n > g_room) return hipErrorOutOfMemory;
  static size_t next = 0;  // no address twice
  *p = (void *)(next += 4096);
  g_owned[*p] = n;
  g_room -= n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  ++g_frees;
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

// A device without the memory for the larger block: nothing moves, and the
// refused size costs no further calls to the runtime for a while.
static void refused_growth_changes_nothing() {
  DevBuf b;
  const hipStream_t s = nullptr;
  std::vector<char *> out;
  char *const small = carve(1 << 20).bind(b, s)[0];
  const size_t room = g_room;
  g_room = (size_t)64 << 20;
  EXPECT(!carve((size_t)1 << 30).try_bind(b, s, &out));
  EXPECT(b.p == small && b.cap == 1 << 20 && g_owned.count(small) == 1);
  const int m = g_mallocs, f = g_frees;
  for (int i = 0; i < 100; ++i) {
    EXPECT(!carve((size_t)1 << 30).try_bind(b, s, &out));
    EXPECT(carve(1 << 20).bind(b, s)[0] == small);  // the fallback
  }
  EXPECT(g_mallocs == m && g_frees == f);
  EXPECT(carve((size_t)32 << 20).try_bind(b, s, &out));  // a smaller one can be had
  g_room = room;
  int n = 0;
  while (n < 1000 && !carve((size_t)1 << 30).try_bind(b, s, &out)) ++n;
  EXPECT(n < 1000);  // asked for again in the end
  b.release();
  EXPECT(g_owned.empty());
}

// bind() needs its block: where both do not fit, the old one goes first.
static void needed_growth_frees_first_where_both_do_not_fit() {
  DevBuf b;
  const hipStream_t s = nullptr;
  carve((size_t)40 << 20).bind(b, s);
  const size_t room = g_room;
  g_room = (size_t)20 << 20;
  carve((size_t)50 << 20).bind(b, s);
  EXPECT(g_owned.size() == 1 && b.cap == (size_t)50 << 20);
  bool threw = false;
  try {
    carve((size_t)80 << 20).bind(b, s);
  } catch (const qh::GpuError &) {
    threw = true;
  }
  EXPECT(threw);
  b.release();
  EXPECT(g_owned.empty());
  g_room = room;
}

int main() {
  refused_growth_changes_nothing();
  needed_growth_frees_first_where_both_do_not_fit();
  captured_block_outlives_growth();
  kept_blocks_are_bounded();
  eager_growth_frees();
  std::printf("failures=%d\n", g_fail);
  return g_fail != 0;
}
