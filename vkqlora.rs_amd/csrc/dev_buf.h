// dev_buf.h -- the context's growable device buffers and the bump allocator
// that lays a call's scratch out in them.  Host code only.
#pragma once
#include <cstddef>
#include <cstdint>
#include <string>
#include <vector>

#include <hip/hip_runtime_api.h>

namespace qh {

struct GpuError {
  std::string msg;
};

inline void check(hipError_t e, const char *what) {
  if (e != hipSuccess) throw GpuError{std::string(what) + ": " + hipGetErrorString(e)};
}

// True also where the runtime cannot tell (the null stream while another
// stream captures).
inline bool capturing(hipStream_t s) {
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &cs) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return cs != hipStreamCaptureStatusNone;
}

// Growable device buffer.  A captured graph holds the address its calls were
// bound to for as long as it is replayed, and nobody tells the library when
// that ends: growth frees a block only if no captured call was bound to it,
// and keeps it until release() otherwise.  A block that takes a kept one's
// place is twice as large where the device has that, so that the kept ones
// together stay below the one in use.
struct DevBuf {
  void *p = nullptr;
  size_t cap = 0;
  bool captured = false;     // a captured call was bound to p
  std::vector<void *> kept;  // blocks of earlier captures

  // For the calls on stream `s`.
  void *ensure(size_t bytes, hipStream_t s) {
    ensure(bytes);
    if (bytes) mark(s);
    return p;
  }
  // For buffers that only blocking host-slice calls use (never captured).
  void *ensure(size_t bytes) {
    if (bytes <= cap) return p;
    hipError_t e = grow(bytes);
    if (e == hipErrorOutOfMemory && p && !captured) {  // not beside the old block
      check(hipFree(p), "hipFree");
      p = nullptr;
      cap = 0;
      e = grow(bytes);
    }
    check(e, "hipMalloc");
    return p;
  }
  // False, with the buffer as it was, when the device has no such block left.
  // A size that failed is not asked for again on every call (a failing
  // hipMalloc waits for the device): the next attempt comes kRetry calls later.
  bool try_ensure(size_t bytes) {
    if (bytes <= cap) return true;
    if (bytes >= failed && ++refused < kRetry) return false;
    refused = 0;
    if (grow(bytes) != hipSuccess) {
      if (bytes < failed) failed = bytes;
      return false;
    }
    if (bytes >= failed) failed = SIZE_MAX;
    return true;
  }
  // Notes that a call on `s` is bound to the block.
  void mark(hipStream_t s) {
    if (p && !captured) captured = capturing(s);
  }
  void release() {
    for (void *k : kept) (void)hipFree(k);
    kept.clear();
    if (p) (void)hipFree(p);
    p = nullptr;
    cap = 0;
    captured = false;
    failed = SIZE_MAX;
    refused = 0;
  }

 private:
  static constexpr int kRetry = 256;
  size_t failed = SIZE_MAX;  // the smallest size that try_ensure could not have
  int refused = 0;

  // A block for `bytes` in place of the present one, which goes only when the
  // new one is there.
  hipError_t grow(size_t bytes) {
    const auto up = [](size_t n) { return n < 256 ? 256 : (n + 255) / 256 * 256; };
    size_t want = up(bytes);
    if (captured) kept.reserve(kept.size() + 1);
    void *q = nullptr;
    hipError_t e = hipErrorOutOfMemory;
    if (captured && want < 2 * cap && (e = hipMalloc(&q, up(2 * cap))) == hipSuccess)
      want = up(2 * cap);
    if (!q) e = hipMalloc(&q, want);
    if (e != hipSuccess) {
      (void)hipGetLastError();
      return e;
    }
    if (captured) {
      kept.push_back(p);
    } else if (p && (e = hipFree(p)) != hipSuccess) {
      (void)hipFree(q);
      return e;
    }
    p = q;
    cap = want;
    captured = false;
    return hipSuccess;
  }
};

// Bump allocator over one DevBuf: sizes are laid out first, then carved.
struct Carve {
  std::vector<size_t> sizes;
  size_t add(size_t bytes) {
    sizes.push_back((bytes + 255) / 256 * 256);
    return sizes.size() - 1;
  }
  size_t total() const {
    size_t t = 0;
    for (size_t s : sizes) t += s;
    return t;
  }
  // For the calls on stream `s`; without one, for blocking host-slice calls.
  std::vector<char *> bind(DevBuf &b, hipStream_t s) { return bind_at((char *)b.ensure(total(), s)); }
  std::vector<char *> bind(DevBuf &b) { return bind_at((char *)b.ensure(total())); }
  // Binds to `b` unless that needs memory that cannot be had now: a larger
  // buffer during a stream capture (an allocation would end the capture), or
  // more than the device has left.  For paths with a fallback that needs
  // less.
  bool try_bind(DevBuf &b, hipStream_t s, std::vector<char *> *out) {
    const size_t need = total();
    if (need > b.cap && (capturing(s) || !b.try_ensure(need))) return false;
    b.mark(s);
    *out = bind_at((char *)b.p);
    return true;
  }
  std::vector<char *> bind_at(char *base) {
    std::vector<char *> out;
    for (size_t s : sizes) {
      out.push_back(base);
      base += s;
    }
    return out;
  }
};

}  // namespace qh
