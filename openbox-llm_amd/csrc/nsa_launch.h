// Host-side helpers shared by the C-ABI entry points: status codes, argument
// checks and launch-error capture.  No allocation and no host synchronisation
// happen here; every launch goes to the caller's stream.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>

#include "nsa_hip.h"

#define NSA_CHECK(cond, code) \
  do {                        \
    if (!(cond)) return (code); \
  } while (0)

static inline int nsa_launch_status() {
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? NSA_OK : NSA_ERR_LAUNCH;
}

// Device of a stream (the null stream: the current device), or -1.
static inline int stream_device(hipStream_t s) {
  hipDevice_t dev = -1;
  if (hipStreamGetDevice(s, &dev) != hipSuccess) return -1;
  return (int)dev;
}

// Compute units of the stream's device, cached per device.  The cache is
// written with relaxed atomics: two threads that race on a first lookup store
// the same value.
static inline int device_cu_count(hipStream_t s) {
  static std::atomic<int> cache[64];
  const int dev = stream_device(s);
  if (dev < 0 || dev >= 64) return 256;
  int n = cache[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cache[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Several tensors in one launch (nsa_prep.hip; the C entry points nsa_transpose_kv,
// nsa_pool_fwd and nsa_pool_bwd are their sets of one): up to three transposed
// copies [BH][L][D] -> [BH][D][Lp], up to two poolings of one shape.
int nsa_transpose_kv_set(const void* const* x, void* const* xt, const int* L, const int* Lp, int n, int BH, int D,
                         int dtype, void* stream);
int nsa_pool_fwd_set(const void* const* x, void* const* out, int m, int B, int H, int T, int D, int l, int d,
                     int dtype, void* stream);
int nsa_pool_bwd_set(const void* const* dpool, int dpool_dtype, void* const* dx, int m, int B, int H, int T, int D,
                     int l, int d, int dtype, void* stream);
