// pxr_radix.hip -- stable least-significant-digit radix sort of (key, index)
// pairs.
//
// A pass reads the keys twice and writes the pairs once: per-block digit
// counts, an exclusive scan of them in digit-major order, and the scatter.
// What bounds it: the scattered 8 B writes and, for a million pairs, launch
// latency (four short kernels per pass), so digits are taken as wide as a
// wave's counters in LDS allow (11 bits, 8 KB per wave) and the passes are as
// few as possible: one up to 2048 keys, two up to 4 M.
#include <algorithm>

#include "pxr_radix.h"

namespace pxr {

// Items of a block (a cap on the histogram makes it more).  Few items want
// more blocks than 4096 a block give: 100,000 particles in 24^3 cells 127 ->
// 103 us (the whole leaf sort); from half a million on, the histogram costs
// as much (a million in 48^3 cells 207 and 203 us; ordering two million by
// 729 blocks for the leaf step 1110 and 1170).
constexpr i64 RX_FEW = (i64)1 << 19;
PXR_HD i64 rx_items(i64 n) { return n < RX_FEW ? 1024 : 4096; }
constexpr int RX_SCAN = 2048;    // counts per block of the scan

static void rx_digits(i64 nkeys, RadixPlan &p) {
  int kb = 1;
  while (kb < 31 && ((i64)1 << kb) < nkeys) kb++;
  p.npass = (kb + RX_BITS - 1) / RX_BITS;
  p.bits = (kb + p.npass - 1) / p.npass;
}

// A plan's blocks are at most one per rx_items keys, so the most are those of n
// keys or of the largest number cut into small ones.
i64 radix_hist_most(i64 n, i64 nkeys, i64 hist_cap) {
  RadixPlan p;
  rx_digits(nkeys, p);
  const i64 few = std::min(n, RX_FEW - 1), nblk = std::max((n + 4095) / 4096, (few + 1023) / 1024);
  const i64 m = std::max<i64>(1, std::min(nblk, hist_cap >> p.bits)) << p.bits;
  return m + (m + RX_SCAN - 1) / RX_SCAN;
}

RadixPlan radix_plan(i64 n, i64 nkeys, i64 hist_cap) {
  RadixPlan p;
  p.n = n;
  rx_digits(nkeys, p);
  // a block's sums follow the counts in the histogram buffer
  const i64 cap = hist_cap - hist_cap / 1024;
  const i64 nblk = std::min<i64>((n + rx_items(n) - 1) / rx_items(n), cap >> p.bits);
  p.nblk = (int)std::max<i64>(1, nblk);
  p.seg = ((n + 4 * (i64)p.nblk - 1) / (4 * (i64)p.nblk) + 63) / 64 * 64;
  p.nblk = (int)std::max<i64>(1, (n + 4 * p.seg - 1) / (4 * p.seg));
  const i64 m = (i64)p.nblk << p.bits;
  p.hist_ints = m + (m + RX_SCAN - 1) / RX_SCAN;
  return p;
}

// digit counts of every block, digit-major: hist[d * nblk + block]
__global__ __launch_bounds__(256) void k_rx_count(const int *key, i64 n, i64 seg, int shift,
                                                  int bits, int *hist) {
  __shared__ int cnt[1 << RX_BITS];
  const int nd = 1 << bits;
  for (int d = threadIdx.x; d < nd; d += 256) cnt[d] = 0;
  __syncthreads();
  const i64 b0 = (i64)blockIdx.x * 4 * seg, b1 = min(n, b0 + 4 * seg);
  for (i64 i = b0 + threadIdx.x; i < b1; i += 256)
    atomicAdd(&cnt[(key[i] >> shift) & (nd - 1)], 1);
  __syncthreads();
  for (int d = threadIdx.x; d < nd; d += 256) hist[(i64)d * gridDim.x + blockIdx.x] = cnt[d];
}

__global__ __launch_bounds__(256) void k_rx_sums(const int *hist, i64 m, int *bsum) {
  __shared__ int s[4];
  const i64 b0 = (i64)blockIdx.x * RX_SCAN;
  int acc = 0;
  for (int k = threadIdx.x; k < RX_SCAN; k += 256)
    if (b0 + k < m) acc += hist[b0 + k];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o);
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) bsum[blockIdx.x] = s[0] + s[1] + s[2] + s[3];
}

// exclusive scan in place: every block sums the blocks before it itself
// (at most 1023), which saves a launch
__global__ __launch_bounds__(256) void k_rx_scan(int *hist, i64 m, const int *bsum) {
  constexpr int PER = RX_SCAN / 256;
  __shared__ int s[4], before[4];
  const int t = (int)threadIdx.x, lane = t & 63, w = t >> 6;
  int acc = 0;
  for (int k = t; k < (int)blockIdx.x; k += 256) acc += bsum[k];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o);
  if (lane == 0) before[w] = acc;
  const i64 b0 = (i64)blockIdx.x * RX_SCAN + (i64)t * PER;
  int v[PER], sum = 0;
#pragma unroll
  for (int k = 0; k < PER; k++) {
    v[k] = b0 + k < m ? hist[b0 + k] : 0;
    sum += v[k];
  }
  int inc = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(inc, off);
    if (lane >= off) inc += y;
  }
  if (lane == 63) s[w] = inc;
  __syncthreads();
  int run = before[0] + before[1] + before[2] + before[3] + inc - sum;
  for (int k = 0; k < w; k++) run += s[k];
#pragma unroll
  for (int k = 0; k < PER; k++) {
    if (b0 + k < m) hist[b0 + k] = run;
    run += v[k];
  }
}

// the same for few counts, by one workgroup in one launch
constexpr int RX_SCAN_ONE = 16384;

__global__ __launch_bounds__(1024) void k_rx_scan_one(int *hist, int m) {
  constexpr int PER = RX_SCAN_ONE / 1024;
  __shared__ int s[16];
  const int t = (int)threadIdx.x, lane = t & 63, w = t >> 6;
  const int per = min(PER, (m + 1023) / 1024);
  int v[PER], sum = 0;
#pragma unroll
  for (int k = 0; k < PER; k++) {
    v[k] = k < per && t * per + k < m ? hist[t * per + k] : 0;
    sum += v[k];
  }
  int run = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(run, off);
    if (lane >= off) run += y;
  }
  if (lane == 63) s[w] = run;
  run -= sum;
  __syncthreads();
  for (int k = 0; k < w; k++) run += s[k];
#pragma unroll
  for (int k = 0; k < PER; k++) {
    if (k < per && t * per + k < m) hist[t * per + k] = run;
    run += v[k];
  }
}

// Scatter.  A wave takes its items 64 at a time in order; the lanes that
// hold the same digit are found with one ballot per digit bit, their slots
// claimed with one add on the wave's counter of that digit, so the order of
// equal digits is kept.  idx_in null: the items are 0..n-1.
__global__ __launch_bounds__(256) void k_rx_scatter(const int *key, const int *idx_in, i64 n,
                                                    i64 seg, int shift, int bits,
                                                    const int *hist, int *key_out,
                                                    int *idx_out) {
  extern __shared__ int next[];  // [4][1 << bits]
  const int nd = 1 << bits;
  const int t = (int)threadIdx.x, lane = t & 63, w = t >> 6;
  for (int d = t; d < 4 * nd; d += 256) next[d] = 0;
  __syncthreads();
  int *mine = next + w * nd;
  const i64 i0 = ((i64)blockIdx.x * 4 + w) * seg, i1 = min(n, i0 + seg);
  for (i64 i = i0 + lane; i < i1; i += 64) atomicAdd(mine + ((key[i] >> shift) & (nd - 1)), 1);
  __syncthreads();
  for (int d = t; d < nd; d += 256) {
    int run = hist[(i64)d * gridDim.x + blockIdx.x];
    for (int q = 0; q < 4; q++) {
      const int c = next[q * nd + d];
      next[q * nd + d] = run;
      run += c;
    }
  }
  __syncthreads();
  const unsigned long long below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  for (i64 b = i0; b < i1; b += 64) {
    const i64 i = b + lane;
    const bool act = i < i1;
    const int k = act ? key[i] : 0;
    const int d = (k >> shift) & (nd - 1);
    unsigned long long peers = __ballot(act);
    for (int q = 0; q < bits; q++) {
      const bool bit = (d >> q) & 1;
      const unsigned long long set = __ballot(bit);
      peers &= bit ? set : ~set;
    }
    const int lead = act ? __ffsll((long long)peers) - 1 : lane;
    int slot = 0;
    if (act && lead == lane) slot = atomicAdd(mine + d, __popcll(peers));
    slot = __shfl(slot, lead) + __popcll(peers & below);
    if (act) {
      key_out[slot] = k;
      idx_out[slot] = idx_in ? idx_in[i] : (int)i;
    }
  }
}

int radix_sort(const RadixPlan &p, int *const *key, int *const *idx, int *hist, hipStream_t st,
               bool counted) {
  const i64 m = (i64)p.nblk << p.bits;
  const unsigned nsum = (unsigned)((m + RX_SCAN - 1) / RX_SCAN);
  int *bsum = hist + m;
  const dim3 grd((unsigned)p.nblk), blk(256);
  const size_t lds = 4 * sizeof(int) << p.bits;
  int at = 0;
  for (int pass = 0; pass < p.npass; pass++, at ^= 1) {
    const int shift = pass * p.bits;
    if (pass || !counted)
      hipLaunchKernelGGL(k_rx_count, grd, blk, 0, st, key[at], p.n, p.seg, shift, p.bits, hist);
    if (m <= RX_SCAN_ONE) {
      hipLaunchKernelGGL(k_rx_scan_one, dim3(1), dim3(1024), 0, st, hist, (int)m);
    } else {
      hipLaunchKernelGGL(k_rx_sums, dim3(nsum), blk, 0, st, hist, m, bsum);
      hipLaunchKernelGGL(k_rx_scan, dim3(nsum), blk, 0, st, hist, m, bsum);
    }
    hipLaunchKernelGGL(k_rx_scatter, grd, blk, lds, st, key[at], pass ? idx[at] : nullptr, p.n,
                       p.seg, shift, p.bits, hist, key[at ^ 1], idx[at ^ 1]);
  }
  return at;
}

}  // namespace pxr
