// pxr_runtime.h -- host-side runtime shared by the C-ABI entry points:
// current stream, error reporting, the device error counter and a small
// cache of library-owned scratch buffers.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "pxrhip.h"

namespace pxr {

constexpr int REPORT_SLOTS = 256;
constexpr int LEAF_BIN_CHUNK = 4096;

struct Runtime {
  int device = -1;
  hipStream_t stream = nullptr;
  bool own_stream = false;  // created by pxrhip_init
  bool capturing = false;   // a graph capture of the stream is open
  bool checks = true;
  // device counter of skipped particles; from [2] on a word per report slot
  unsigned long long *d_bad = nullptr;
  unsigned long long *d_sort_bad = nullptr;  // the leaf sort's own counter of bad keys (d_bad + 1)
  unsigned long long *h_report = nullptr;  // pinned host memory, see report_slot
  int num_cus = 256;
  // leaf deposition summed in LDS blocks (pxr_leafbin.hip) from this many
  // particles on (0: never), in work items of at most leaf_bin_chunk particles;
  // up to LEAF_BIN_CHUNK the routines take smaller ones by themselves, a larger
  // value is taken as it is
  int64_t leaf_bin_min = 1 << 16;
  int leaf_bin_chunk = LEAF_BIN_CHUNK;
  // form of the last large leaf call (pxrhip_get_tuning "last.leaf_*"): 1 block
  // by block; whether its deposition could read records (the GPU decides, and
  // writes its answer behind the report slots)
  int last_leaf_current = 0, last_leaf_rho = 0, last_leaf_gather = 0;
  bool last_leaf_records_asked = false;
  // incremented whenever library-owned device memory that recorded work may
  // point at is freed (a scratch slot that grows, the cached tile table):
  // a HIP graph captured before that refers to freed memory
  unsigned long long mem_gen = 0;
};

Runtime &rt();
int set_error(int code, const char *fmt, ...);
int ensure_init();
// library-owned scratch buffer number `slot`, grown to at least `bytes`; null
// if there is no memory for it (with the runtime's error state cleared, so
// that a caller that has a form without scratch can launch that)
void *scratch(int slot, size_t bytes);
// gives a slot's memory back, once the work that uses it is done (hipFree waits
// for the device)
void scratch_free(int slot);
// bytes held in slot (slot < 0: in all of them)
size_t scratch_bytes(int slot);
// Gives all scratch back and, with bytes > 0, keeps the total at or below so
// much from here on: scratch() then returns null as if there was no more memory.
void scratch_limit(size_t bytes);
// A word of pinned host memory for a kernel to report through: the caller's
// own until as many later calls have asked for one (calls of other threads
// that wait at the same time have theirs).
unsigned long long *report_slot();
// read the bad-particle counter (synchronises the stream), reset it to 0
int take_bad(unsigned long long *n);
// the same for any device counter
int take_counter(unsigned long long *ctr, unsigned long long *n, hipStream_t st);

// the word after the report slots: whether the last current was deposited from
// records
inline unsigned long long *records_word() { return rt().h_report + REPORT_SLOTS; }

inline unsigned grid1d(int64_t n, int block) {
  int64_t b = (n + block - 1) / block;
  return (unsigned)(b < 1 ? 1 : b);
}

}  // namespace pxr

#define PXR_HIP(call)                                                          \
  do {                                                                         \
    hipError_t e_ = (call);                                                    \
    if (e_ != hipSuccess)                                                      \
      return pxr::set_error(PXRHIP_ERR_HIP, "%s failed: %s", #call,           \
                            hipGetErrorString(e_));                            \
  } while (0)

#define PXR_LAUNCHED()                                                         \
  do {                                                                         \
    hipError_t e_ = hipGetLastError();                                         \
    if (e_ != hipSuccess)                                                      \
      return pxr::set_error(PXRHIP_ERR_HIP, "kernel launch failed: %s",        \
                            hipGetErrorString(e_));                            \
  } while (0)

#define PXR_INIT()                                                             \
  do {                                                                         \
    int r_ = pxr::ensure_init();                                               \
    if (r_ != PXRHIP_OK) return r_;                                            \
  } while (0)
