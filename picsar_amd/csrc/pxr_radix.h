// pxr_radix.h -- stable sort of particle indices by a small integer key
// (sorting cell, node block), the common part of the leaf sort and of the
// binned leaf routines.
#pragma once
#include "pxr_device.h"
#include "pxr_runtime.h"

namespace pxr {

constexpr int RX_BITS = 11;  // widest digit

// How n keys below nkeys are sorted: npass least-significant-digit passes
// of `bits` bits, each over nblk blocks of 4 * seg items (a wave owns seg
// consecutive ones).
struct RadixPlan {
  i64 n = 0, seg = 0;
  int npass = 0, bits = 0, nblk = 0;
  i64 hist_ints = 0;  // ints of the histogram buffer
};

// hist_cap: largest histogram buffer the caller can give, in ints (at least
// 2^20)
RadixPlan radix_plan(i64 n, i64 nkeys, i64 hist_cap);

// the largest hist_ints of a plan for n keys or fewer
i64 radix_hist_most(i64 n, i64 nkeys, i64 hist_cap);

// Sorts on stream st.  key[0] holds the keys (all in [0, nkeys)); key[1],
// idx[0] and idx[1] are n ints each, hist plan.hist_ints.  Returns which of
// the two buffers holds the sorted keys and, in key order and in increasing
// order within a key, the indices 0..n-1.  After a single pass hist[d * p.nblk]
// is the number of keys below d.  counted: the caller has left the first
// pass's digit counts of every block in hist (as k_rx_count does).
int radix_sort(const RadixPlan &p, int *const *key, int *const *idx, int *hist, hipStream_t st,
               bool counted = false);

}  // namespace pxr
