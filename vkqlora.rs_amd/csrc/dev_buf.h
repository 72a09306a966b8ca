// dev_buf.h -- the context's growable device buffers and the bump allocator
// that lays a call's scratch out in them.  Host code only.
#pragma once
#include <cstddef>
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
// place is at least twice as large, so that the kept ones together stay below
// the one in use.
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
    const size_t want = rounded(bytes);
    retire();
    check(hipMalloc(&p, want), "hipMalloc");
    cap = want;
    return p;
  }
  // False, with the buffer empty, when the device has no such block left.
  bool try_ensure(size_t bytes) {
    if (bytes <= cap) return true;
    const size_t want = rounded(bytes);
    retire();
    if (hipMalloc(&p, want) != hipSuccess) {
      (void)hipGetLastError();
      p = nullptr;
      return false;
    }
    cap = want;
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
  }

 private:
  size_t rounded(size_t bytes) const {
    if (captured && bytes < 2 * cap) bytes = 2 * cap;
    return bytes < 256 ? 256 : (bytes + 255) / 256 * 256;
  }
  void retire() {
    if (p && captured) {
      kept.push_back(p);
    } else if (p) {
      check(hipFree(p), "hipFree");
    }
    p = nullptr;
    cap = 0;
    captured = false;
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
