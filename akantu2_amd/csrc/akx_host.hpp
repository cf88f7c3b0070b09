// akx_host.hpp -- host-side utilities shared by the translation units of the
// library: status-code errors, HIP error checks, device buffers.
#pragma once

#include "../../include/akantu_mi355x.h"
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <new>
#include <stdexcept>
#include <string>
#include <vector>

namespace akx {

// ---------------------------------------------------------------------------
// Errors: C++ exceptions inside, status codes across the ABI.
// ---------------------------------------------------------------------------
struct Error : std::runtime_error {
  int code;
  Error(int c, const std::string &m) : std::runtime_error(m), code(c) {}
};

extern thread_local std::string g_last_error;

#define HIPCHECK(x)                                                            \
  do {                                                                         \
    hipError_t err_ = (x);                                                     \
    if (err_ != hipSuccess)                                                    \
      throw Error(err_ == hipErrorOutOfMemory ? AKX_ERR_MEMORY : AKX_ERR_HIP,  \
                  std::string(#x) + ": " + hipGetErrorString(err_));           \
  } while (0)

// (a literal's string is built only when it is thrown: checks of every entry of
// an array spent 10 ns each on it)
inline void require(bool c, const char *msg) {
  if (!c)
    throw Error(AKX_ERR_INVALID, msg);
}
inline void require(bool c, const std::string &msg) {
  if (!c)
    throw Error(AKX_ERR_INVALID, msg);
}

// ---------------------------------------------------------------------------
// Device buffer
// ---------------------------------------------------------------------------
template <class T> struct DevBuf {
  T *p = nullptr;
  size_t n = 0;
  DevBuf() = default;
  DevBuf(const DevBuf &) = delete;
  DevBuf &operator=(const DevBuf &) = delete;
  ~DevBuf() { release(); }
  void release() {
    if (p)
      (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
  void alloc(size_t count) {
    if (count == n && p)
      return;
    release();
    if (count == 0)
      return;
    HIPCHECK(hipMalloc(&p, count * sizeof(T)));
    n = count;
  }
  // grow only (keeps the buffer, and its address, when it is big enough)
  void reserve(size_t count) {
    if (count > n || !p)
      alloc(count > 0 ? count : 1);
  }
  size_t bytes() const { return n * sizeof(T); }
};


// The distinct values of a block's node ids in ascending order: a bit per
// node, read back over the words the block spans; ids scattered over far more
// words than there are ids are sorted instead.
class DistinctNodes {
  std::vector<uint64_t> bits;

public:
  explicit DistinctNodes(int64_t nb_nodes) : bits((nb_nodes + 63) / 64, 0) {}
  // appends the distinct values of ids[0 .. n), n > 0, to out
  void append(const int32_t *ids, int64_t n, std::vector<int32_t> &out) {
    const auto mm = std::minmax_element(ids, ids + n);
    const int64_t w0 = *mm.first >> 6, w1 = *mm.second >> 6;
    if (w1 - w0 > 4 * n) {
      const size_t start = out.size();
      out.insert(out.end(), ids, ids + n);
      std::sort(out.begin() + start, out.end());
      out.erase(std::unique(out.begin() + start, out.end()), out.end());
      return;
    }
    for (int64_t i = 0; i < n; ++i)
      bits[ids[i] >> 6] |= uint64_t(1) << (ids[i] & 63);
    for (int64_t w = w0; w <= w1; ++w) {
      for (uint64_t b = bits[w]; b; b &= b - 1)
        out.push_back((int32_t)(w * 64 + __builtin_ctzll(b)));
      bits[w] = 0;
    }
  }
};

// Run f and turn any exception into a status code (nothing throws across
// the C ABI).
template <class F> inline int guard(F &&f) {
  try {
    f();
    return AKX_OK;
  } catch (const Error &e) {
    g_last_error = e.what();
    return e.code;
  } catch (const std::bad_alloc &) {
    g_last_error = "host allocation failed";
    return AKX_ERR_MEMORY;
  } catch (const std::exception &e) {
    g_last_error = e.what();
    return AKX_ERR_INVALID;
  } catch (...) {
    g_last_error = "unknown error";
    return AKX_ERR_INVALID;
  }
}


} // namespace akx
