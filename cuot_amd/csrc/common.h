// common.h -- shared device/host definitions for the gfx950 silent-OT engine.
//
// A block is 128 bits in memory byte order (bytes 0..7 = lo).  On the device it
// is handled as four little-endian u32 words (uint4 x,y,z,w = bytes 0-3, 4-7,
// 8-11, 12-15), which is also the column order of the AES state.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <mutex>

#include "../../include/cuot_amd.h"

#define CUOT_DEV __device__ __forceinline__

typedef uint4 blk;

CUOT_DEV blk bxor(blk a, blk b) { return make_uint4(a.x ^ b.x, a.y ^ b.y, a.z ^ b.z, a.w ^ b.w); }
CUOT_DEV blk bzero() { return make_uint4(0u, 0u, 0u, 0u); }
CUOT_DEV blk bsel(bool c, blk a) { return c ? a : bzero(); }

// Plain 16-byte global accessors.  The address space is spelled out: through a
// pointer read from an argument table the compiler would use flat accesses,
// which also count as LDS operations.
typedef uint32_t blk_vec __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) blk_vec* blk_gptr;
typedef const __attribute__((address_space(1))) blk_vec* blk_cgptr;
CUOT_DEV blk ldb(const blk* p) {
  const blk_vec v = *(blk_cgptr)p;
  return make_uint4(v.x, v.y, v.z, v.w);
}
CUOT_DEV void stb(blk* p, blk v) { *(blk_gptr)p = blk_vec{v.x, v.y, v.z, v.w}; }

// ---------------------------------------------------------------------------
// Host-side error plumbing: every extern "C" entry point returns an int status.
// ---------------------------------------------------------------------------
#define CUOT_HIP_TRY(expr)                                  \
  do {                                                      \
    hipError_t _e = (expr);                                 \
    if (_e != hipSuccess) {                                 \
      cuot_set_last_error(hipGetErrorString(_e), __FILE__, __LINE__); \
      return CUOT_ERR_HIP;                                  \
    }                                                       \
  } while (0)

#define CUOT_CHECK_ARG(cond, msg)                           \
  do {                                                      \
    if (!(cond)) {                                          \
      cuot_set_last_error(msg, __FILE__, __LINE__);         \
      return CUOT_ERR_ARG;                                  \
    }                                                       \
  } while (0)

#define CUOT_LAUNCH_CHECK()                                 \
  do {                                                      \
    hipError_t _e = hipGetLastError();                      \
    if (_e != hipSuccess) {                                 \
      cuot_set_last_error(hipGetErrorString(_e), __FILE__, __LINE__); \
      return CUOT_ERR_HIP;                                  \
    }                                                       \
  } while (0)

// One-time set-up of each device (function attributes hold for the device that is
// current when they are set); safe with several threads.
struct CuotDeviceOnce {
  std::mutex mu;
  std::atomic<bool> done[64] = {};

  template <typename F>
  hipError_t run(const F& setup) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
    if (done[dev].load(std::memory_order_acquire)) return hipSuccess;
    std::lock_guard<std::mutex> lk(mu);
    if (done[dev].load(std::memory_order_relaxed)) return hipSuccess;
    e = setup();
    if (e == hipSuccess) done[dev].store(true, std::memory_order_release);
    return e;
  }
};

void cuot_set_last_error(const char* msg, const char* file, int line);
