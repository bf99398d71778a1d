// pxr_leafbin.hip -- the leaf routines on large particle sets, block by block in
// LDS: the current and charge deposition (depose_jxjyjz, pxr_depose_rho_n) and
// the field gather.
//
// A caller of the leaf routines hands over particles in any order, anywhere
// in the grid arrays.  Adding every contribution to global memory costs one
// FP64 L2 atomic per node and particle (144 for an order-3 Esirkepov
// particle that keeps its nodes), and those atomics bound the kernel.  Here
// the particles are first keyed by cubic blocks of B^3 nodes (by the node
// floor(x) of their new position, or of the mid position for the direct
// current), ordered by block with a radix sort of their indices, and cut
// into work items of at most `chunk` particles of one block.  A workgroup
// sums its work item's contributions into an LDS copy of the block with its
// halo (the nodes that the shapes and one cell of motion reach) and adds the
// block to the grid array once per non-zero node.
//
// The contributions are the same arithmetic as the global-atomic kernels
// (esirkepov_deposit, direct_deposit, the nodal shapes of pxr_depose_rho_n);
// only the order of the FP64 sums differs.  A call that has no memory for the
// ordering, or that is captured in a HIP graph, takes the unbinned kernel.
//
// The gather of the fields (geteb3d_energy_conserving) uses the same order
// for a large set whose particles are in none.
#include <algorithm>
#include <mutex>

#include "pxr_leafbin.h"
#include "pxr_radix.h"
#include "pxr_runtime.h"

namespace pxr {

// Blocks of B^3 nodes over the padded array; block (bx, by, bz) holds the
// particles whose node floor(x) + guard lies in [bx B, bx B + B).
struct BinGeom {
  int nb[3];   // blocks per axis
  int gd[3];   // guard widths
  int na[3];   // padded node counts
  i64 nblocks;
};

constexpr int LB_EDGE = 8;  // nodes per block edge

static BinGeom make_bin_geom(const GridGeom &g, int B) {
  BinGeom b;
  b.gd[0] = g.gx; b.gd[1] = g.gy; b.gd[2] = g.gz;
  b.na[0] = g.nx + 1 + 2 * g.gx;
  b.na[1] = g.ny + 1 + 2 * g.gy;
  b.na[2] = g.nz + 1 + 2 * g.gz;
  for (int d = 0; d < 3; d++) b.nb[d] = (b.na[d] + B - 1) / B;
  b.nblocks = (i64)b.nb[0] * b.nb[1] * b.nb[2];
  return b;
}

// block index along one axis of normalised position x: floor(x) clamped to
// the array (a particle outside it is rejected by the deposit kernel)
template <int B> PXR_DEV int block_axis(double x, int g, int na) {
  double f = floor(x);
  f = fmin(fmax(f, -(double)g), (double)(na - 1 - g));
  return ((int)f + g) / B;
}

// The eight values of every particle in one record of 64 bytes, written by
// k_lb_keys and read by the deposition if *use is set (null: never).  In block
// order a set in no order reads one value of a cache line from each of the
// eight arrays per particle, which bounds orders 1 and 2: two million particles
// on 64^3 cells 411 and 423 us (Esirkepov), 281 and 317 with the record (the
// LDS adds bound order 3: 448 and 475).  A set in cell order shares those
// lines (177 us at order 1) and would pay for the copy.
struct DepoRec {
  double *rec = nullptr;
  const int *use = nullptr;
  PXR_DEV bool on() const { return use && *use; }
};

struct Particle8 {
  double x, y, z, ux, uy, uz, gi, w;
};

PXR_DEV Particle8 load8(const DepoArgs &a, const DepoRec &r, bool rec, i64 ip) {
  Particle8 p;
  if (rec) {
    const double2 *q = (const double2 *)(r.rec + 8 * ip);
    const double2 q0 = q[0], q1 = q[1], q2 = q[2], q3 = q[3];
    p = Particle8{q0.x, q0.y, q1.x, q1.y, q2.x, q2.y, q3.x, q3.y};
  } else {
    p = Particle8{a.xp[ip], a.yp[ip], a.zp[ip], a.ux[ip], a.uy[ip], a.uz[ip], a.gi[ip], a.w[ip]};
  }
  return p;
}

// positions (and, for the mid positions, velocities and h = dt / (2 dx)) of
// one call
struct LbPos {
  i64 np;
  const double *x, *y, *z, *ux, *uy, *uz, *gi, *w;
  double xmin, ymin, zmin, dxi, dyi, dzi, h[3];
  int l4symtry;
  double *rec;  // not null: the normalised positions go to 6-double records too
  DepoRec packed;
};

// arguments of the binned deposition: the call's, and the particles' records
struct LbDepo {
  DepoArgs c;
  DepoRec packed;
};

// arguments of the binned gather: the call's, and the particles' records
struct LbGather {
  LeafGatherArgs c;
  double *rec;
};

// Block of particle ip, by the node of its position (MID: of its position
// half a step back, where the direct current is deposited).
template <int B, bool MID>
PXR_DEV int lb_key(const LbPos &a, const BinGeom &bg, i64 ip) {
  double x = a.x[ip], y = a.y[ip], z = a.z[ip];
  const bool pack = a.packed.on();
  double ux = 0.0, uy = 0.0, uz = 0.0, gi = 0.0;
  if (MID || pack) ux = a.ux[ip], uy = a.uy[ip], uz = a.uz[ip], gi = a.gi[ip];
  if (pack) {
    double2 *q = (double2 *)(a.packed.rec + 8 * ip);
    q[0] = double2{x, y};
    q[1] = double2{z, ux};
    q[2] = double2{uy, uz};
    q[3] = double2{gi, a.w[ip]};
  }
  x = (x - a.xmin) * a.dxi;
  y = (y - a.ymin) * a.dyi;
  z = (z - a.zmin) * a.dzi;
  if (MID) {
    x -= a.h[0] * (ux * gi);
    y -= a.h[1] * (uy * gi);
    z -= a.h[2] * (uz * gi);
  } else if (a.l4symtry) {
    x = fabs(x);
    y = fabs(y);
  }
  if (a.rec) {
    a.rec[6 * ip] = x;
    a.rec[6 * ip + 1] = y;
    a.rec[6 * ip + 2] = z;
  }
  return block_axis<B>(x, bg.gd[0], bg.na[0]) +
         bg.nb[0] * (block_axis<B>(y, bg.gd[1], bg.na[1]) +
                     bg.nb[1] * block_axis<B>(z, bg.gd[2], bg.na[2]));
}

// keys; clears the blocks' ranges and the number of work items
template <int B, bool MID>
__global__ __launch_bounds__(256) void k_lb_keys(LbPos a, BinGeom bg, int *key, int2 *range,
                                                 int *nitems) {
  const i64 ip = (i64)blockIdx.x * blockDim.x + threadIdx.x;
  if (ip == 0) *nitems = 0;
  if (range && ip < bg.nblocks) range[ip] = make_int2(0, 0);
  if (ip < a.np) key[ip] = lb_key<B, MID>(a, bg, ip);
}

// The same for a set that one pass of the radix sort orders, with the digit
// counts of that pass (k_rx_count).  A small call is a chain of short launches:
// this one less, none for the blocks' ranges and one for the scan of few
// counts take the charge density of 66,000 particles in cell order on 32^3
// cells from 61 to 39 us at order 1, the Esirkepov current from 62 to 41 (100,000:
// 61 and 60 -> 43 and 45; 400,000 on 64^3 67 and 82 -> 58 and 74).
template <int B, bool MID>
__global__ __launch_bounds__(256) void k_lb_keys_count(LbPos a, BinGeom bg, int *key, i64 seg,
                                                       int bits, int *hist, int *nitems) {
  __shared__ int cnt[1 << RX_BITS];
  const int nd = 1 << bits;
  for (int d = threadIdx.x; d < nd; d += 256) cnt[d] = 0;
  if (blockIdx.x == 0 && threadIdx.x == 0) *nitems = 0;
  __syncthreads();
  const i64 b0 = (i64)blockIdx.x * 4 * seg, b1 = min(a.np, b0 + 4 * seg);
#pragma unroll 4
  for (i64 ip = b0 + threadIdx.x; ip < b1; ip += 256) {
    const int k = lb_key<B, MID>(a, bg, ip);
    key[ip] = k;
    atomicAdd(&cnt[k], 1);
  }
  __syncthreads();
  for (int d = threadIdx.x; d < nd; d += 256) hist[(i64)d * gridDim.x + blockIdx.x] = cnt[d];
}

// The sorted particles of each block that has any: the first of a run of
// equal keys writes its start, the last its end.  (One thread per gap used to
// write the starts of the empty blocks in it too: 4.4 ms for a bunch in 512^3
// cells, 275 thousand blocks.)
__global__ __launch_bounds__(256) void k_lb_ranges(i64 np, const int *key, int2 *range) {
  const i64 j = (i64)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= np) return;
  const int k = key[j];
  if (j == 0 || key[j - 1] != k) range[k].x = (int)j;
  if (j == np - 1 || key[j + 1] != k) range[k].y = (int)j + 1;
}

// Where the sorted particles of a block lie: the ranges, or, after a sort in
// one pass, its scanned digit counts (those of a digit's first radix block).
struct BlockRanges {
  const int2 *range;  // or null
  const int *hist;
  int stride, nd, np;
  PXR_DEV int2 of(i64 b) const {
    if (range) return range[b];
    return make_int2(hist[b * stride], b + 1 < nd ? hist[(b + 1) * stride] : np);
  }
};

// The work items (block, first slot, count) of at most `chunk` particles of
// one block, a thread per block.  Their order is that of the blocks inside a
// workgroup, and between workgroups that of their adds to *nitems.  A block of
// more than LB_OWN items is cut by its whole wave (eight million particles in
// one block are 16,000 items).
constexpr int LB_OWN = 8;

__global__ __launch_bounds__(1024) void k_lb_plan(BlockRanges br, i64 nblocks, int chunk,
                                                  int4 *items, int *nitems) {
  __shared__ int s[16], first;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const i64 b = (i64)blockIdx.x * 1024 + t;
  const int2 r = b < nblocks ? br.of(b) : make_int2(0, 0);
  const int c = r.y - r.x, ni = (c + chunk - 1) / chunk;
  int inc = ni;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(inc, off);
    if (lane >= off) inc += y;
  }
  if (lane == 63) s[w] = inc;
  __syncthreads();
  if (t == 0) {
    int sum = 0;
    for (int k = 0; k < 16; k++) sum += s[k];
    first = sum ? atomicAdd(nitems, sum) : 0;
  }
  __syncthreads();
  int at = first + inc - ni;
  for (int k = 0; k < w; k++) at += s[k];
  auto put = [&](int bb, int f, int n, int o, int k) {
    items[o + k] = make_int4(bb, f + k * chunk, min(chunk, n - k * chunk), 0);
  };
  if (ni <= LB_OWN)
    for (int k = 0; k < ni; k++) put((int)b, r.x, c, at, k);
  unsigned long long many = __ballot(ni > LB_OWN);
  for (; many; many &= many - 1) {
    const int l = __ffsll((long long)many) - 1;
    const int bb = __shfl((int)b, l), f = __shfl(r.x, l), n = __shfl(c, l), o = __shfl(at, l);
    const int m = __shfl(ni, l);
    for (int k = lane; k < m; k += 64) put(bb, f, n, o, k);
  }
}

// LDS block of one work item: nodes [o0, o0 + L) per axis (grid indices)
struct LdsBlock {
  double *p;
  int o[3], L, nodes;
  PXR_DEV bool holds(const int *lo, const int *hi) const {
    return lo[0] >= o[0] && lo[1] >= o[1] && lo[2] >= o[2] && hi[0] < o[0] + L &&
           hi[1] < o[1] + L && hi[2] < o[2] + L;
  }
};

// LDS accumulator of the current (FP64 LDS atomics), component c at p + c*nodes
struct LdsAccB {
  double *p;
  int i0, j0, k0, sy, sz, nodes;
  PXR_DEV double *row(int c, int i, int j, int k) const {
    return p + c * nodes + ((i - i0) + sy * (j - j0) + sz * (k - k0));
  }
  PXR_DEV void add_row(double *r, int o, double v) const { atomicAdd(r + o, v); }
  PXR_DEV void add(int c, int i, int j, int k, double v) const { atomicAdd(row(c, i, j, k), v); }
};

// the LDS block of block b: first node and edge; zeroed (after the
// previous work item's flush has read it)
template <int B, int HLO, int HHI>
PXR_DEV void lb_block(const BinGeom &bg, int b, LdsBlock &blk, double *lds, int ncomp) {
  const int bx = b % bg.nb[0], by = (b / bg.nb[0]) % bg.nb[1], bz = b / (bg.nb[0] * bg.nb[1]);
  blk.p = lds;
  blk.L = B + HHI - HLO;
  blk.nodes = blk.L * blk.L * blk.L;
  blk.o[0] = bx * B - bg.gd[0] + HLO;
  blk.o[1] = by * B - bg.gd[1] + HLO;
  blk.o[2] = bz * B - bg.gd[2] + HLO;
  __syncthreads();
  for (int i = threadIdx.x; i < ncomp * blk.nodes; i += blockDim.x) lds[i] = 0.0;
  __syncthreads();
}

// add the LDS block's non-zero nodes to the grid arrays
PXR_DEV void lb_flush(const LdsBlock &blk, const GridGeom &g, double *const *dst, int ncomp) {
  __syncthreads();
  const int L = blk.L;
  for (int t = threadIdx.x; t < blk.nodes; t += blockDim.x) {
    const int i = blk.o[0] + t % L, j = blk.o[1] + (t / L) % L, k = blk.o[2] + t / (L * L);
    if (!g.inside(i, j, k)) continue;  // nothing deposits outside the array
    const i64 ix = g.idx(i, j, k);
    for (int c = 0; c < ncomp; c++) {
      const double v = blk.p[c * blk.nodes + t];
      if (v != 0.0) unsafeAtomicAdd(dst[c] + ix, v);
    }
  }
}

// A thread of 256 takes S = ceil(n / 256) consecutive particles of a work item
// in turn, lanes S apart, so that in cell-ordered input the lanes of a wave sit
// in different cells.
PXR_DEV int lb_stride(int n) { return (n + (int)blockDim.x - 1) / (int)blockDim.x; }

// The first of them.  At order 3, whose adds at one address cost the most, S
// apart is too near in the small work items of dense sets in cell order: where
// LB_RUN particles on the caller's order has not changed yet (a block's row of
// eight cells with 12 or more particles each), the lanes of a wave spread over
// the whole item, 4 S apart, and the four waves share what lies between.
// Esirkepov current and charge density with items of 4096 as they were once, of
// 2048, and so (us): sixteen million on 64^3 cells 3757 and 1722, 6212 and 2876,
// 2248 and 1152; four million 755 and 408, 701 and 358, 609 and 309; a bunch of
// four million, up to 1200 a cell, 2650 and 1300, 2912 and 1353, 2176 and 1049.
// (At 8 a cell it loses, sixteen million on 128^3 2306 -> 2425 us, and in no
// order, where it scatters the reads of perm: eight million on 64^3 1534 ->
// 1702.)
constexpr int LB_RUN = 48;

template <int N> PXR_DEV int lb_first(const int *perm, int n, int S) {
  const int t = threadIdx.x, lane = t & 63;
  if (N == 3 && n > 256) {
    const int p = lane * 4 * S;  // (every wave finds the same)
    const bool run = p + LB_RUN < n && perm[p + LB_RUN] == perm[p] + LB_RUN;
    if (__popcll(__ballot(run)) >= 32) return p + (t >> 6) * S;
  }
  return t * S;
}

// Esirkepov current: the box of an order-N particle lies within
// [floor(x) - 2, floor(x) + 3] (order 1: [-1, +2]) on each axis.
// (Order 3 at three waves per SIMD, the three workgroups that fit the LDS: two
// registers more and it runs two, 1512 -> 1655 us for eight million particles
// in no order on 64^3 cells.)
template <int N, int B>
__global__ __launch_bounds__(256, N == 3 ? 3 : 1) void k_lb_esirkepov(LbDepo d, BinGeom bg, const int *perm,
                                                      const int4 *items, const int *nitems) {
  const DepoArgs &a = d.c;
  const bool rec = d.packed.on();
  constexpr int HLO = (N == 1) ? -1 : -2, HHI = (N == 1) ? 2 : 3;
  extern __shared__ double lds[];
  const i64 o = a.g.idx(0, 0, 0);
  const GlobalAcc gacc{{a.jx + o, a.jy + o, a.jz + o}, a.g.NX, a.g.NX * a.g.NY};
  double *dst[3] = {a.jx, a.jy, a.jz};
  const int nit = *nitems;
  for (int w = blockIdx.x; w < nit; w += gridDim.x) {
  const int4 it = items[w];
  LdsBlock blk;
  lb_block<B, HLO, HHI>(bg, it.x, blk, lds, 3);
  const LdsAccB acc{lds, blk.o[0], blk.o[1], blk.o[2], blk.L, blk.L * blk.L, blk.nodes};
  const int n = it.z, S = lb_stride(n), first = lb_first<N>(perm + it.y, n, S);
  for (int k = 0; k < S; k++) {
    const int p = first + k;
    if (p >= n) break;
    const Particle8 q = load8(a, d.packed, rec, perm[it.y + p]);
    EsirkepovIn<double> in;
    esirkepov_prepare<N, double>(in, q.x, q.y, q.z, q.ux, q.uy, q.uz, q.gi, q.w, a.ec);
    int lo[3], hi[3];
    if (!esirkepov_box<N, double>(in, lo, hi) || !a.g.inside(lo[0], lo[1], lo[2]) ||
        !a.g.inside(hi[0], hi[1], hi[2])) {
      count_bad(a.bad);
      continue;
    }
    if (blk.holds(lo, hi)) esirkepov_deposit<N, double>(in, acc);
    else esirkepov_deposit<N, double>(in, gacc);  // a position that is not a number
  }
  lb_flush(blk, a.g, dst, 3);
  }
}

// Direct current: the nodes of an order-N particle lie within
// [floor(m) - 2, floor(m) + 3] of its mid position m (order 1: [-1, +2]) on
// each axis.
//
// Global FP64 atomics bound the unbinned form (k_direct: 24, 81 or 192 adds
// per particle into L2; 2.75 ms for a million order-2 particles on 64^3
// cells); here they go to LDS and one add per node and block remains
// (0.12 ms, and 0.06 ms to key and order the particles).
template <int N, int B>
__global__ __launch_bounds__(256) void k_lb_direct(LbDepo d, BinGeom bg, const int *perm,
                                                   const int4 *items, const int *nitems) {
  const DepoArgs &a = d.c;
  const bool rec = d.packed.on();
  constexpr int HLO = (N == 1) ? -1 : -2, HHI = (N == 1) ? 2 : 3;
  extern __shared__ double lds[];
  const i64 o = a.g.idx(0, 0, 0);
  const GlobalAcc gacc{{a.jx + o, a.jy + o, a.jz + o}, a.g.NX, a.g.NX * a.g.NY};
  double *dst[3] = {a.jx, a.jy, a.jz};
  const int nit = *nitems;
  for (int w = blockIdx.x; w < nit; w += gridDim.x) {
    const int4 it = items[w];
    LdsBlock blk;
    lb_block<B, HLO, HHI>(bg, it.x, blk, lds, 3);
    const LdsAccB acc{lds, blk.o[0], blk.o[1], blk.o[2], blk.L, blk.L * blk.L, blk.nodes};
    const int n = it.z, S = lb_stride(n), first = lb_first<N>(perm + it.y, n, S);
    for (int k = 0; k < S; k++) {
      const int p = first + k;
      if (p >= n) break;
      const Particle8 q = load8(a, d.packed, rec, perm[it.y + p]);
      DirectIn<double> in;
      direct_prepare<N, double>(in, q.x, q.y, q.z, q.ux, q.uy, q.uz, q.gi, q.w, a.q, a.xmin, a.ymin, a.zmin, a.dt, a.dx, a.dy,
                                a.dz, a.s);
      int lo[3], hi[3];
      direct_box<N>(in, lo, hi);
      if (!a.g.inside(lo[0], lo[1], lo[2]) || !a.g.inside(hi[0], hi[1], hi[2])) {
        count_bad(a.bad);
        continue;
      }
      if (blk.holds(lo, hi)) direct_deposit<N, double>(in, acc);
      else direct_deposit<N, double>(in, gacc);  // a position that is not a number
    }
    lb_flush(blk, a.g, dst, 3);
  }
}

// charge density: nodes [floor(x) - 1, floor(x) + 2] (order 1: [0, 1])
template <int N, int B>
__global__ __launch_bounds__(256) void k_lb_rho(RhoArgs a, BinGeom bg, const int *perm,
                                                const int4 *items, const int *nitems) {
  constexpr int HLO = (N == 1) ? 0 : -1, HHI = (N == 1) ? 1 : 2;
  extern __shared__ double lds[];
  double *dst[1] = {a.rho};
  const int nit = *nitems;
  for (int w = blockIdx.x; w < nit; w += gridDim.x) {
  const int4 it = items[w];
  LdsBlock blk;
  lb_block<B, HLO, HHI>(bg, it.x, blk, lds, 1);
  const int L = blk.L;
  const int n = it.z, S = lb_stride(n), first = lb_first<N>(perm + it.y, n, S);
  for (int k = 0; k < S; k++) {
    const int p = first + k;
    if (p >= n) break;
    const i64 ip = perm[it.y + p];
    double x = (a.xp[ip] - a.xmin) * a.dxi, y = (a.yp[ip] - a.ymin) * a.dyi;
    const double z = (a.zp[ip] - a.zmin) * a.dzi;
    if (a.l4symtry) {
      x = fabs(x);
      y = fabs(y);
    }
    double sx[N + 1], sy[N + 1], sz[N + 1];
    const int j = shape_nodal<N, double>(x, sx);
    const int kk = shape_nodal<N, double>(y, sy);
    const int l = shape_nodal<N, double>(z, sz);
    if (!a.g.inside(j, kk, l) || !a.g.inside(j + N, kk + N, l + N)) {
      count_bad(a.bad);
      continue;
    }
    const double wq =
        a.per_particle_weight ? a.q * a.w[ip] * a.invvol : a.q * a.invvol * a.w[0];
    const int lo[3] = {j, kk, l}, hi[3] = {j + N, kk + N, l + N};
    const bool in_lds = blk.holds(lo, hi);
    double *r = in_lds ? lds + ((j - blk.o[0]) + L * ((kk - blk.o[1]) + L * (l - blk.o[2])))
                       : a.rho + a.g.idx(j, kk, l);
    const i64 sy_ = in_lds ? L : a.g.NX, sz_ = in_lds ? (i64)L * L : a.g.NX * a.g.NY;
#pragma unroll
    for (int c = 0; c <= N; c++)
#pragma unroll
      for (int b = 0; b <= N; b++)
#pragma unroll
        for (int e = 0; e <= N; e++) {
          const double v = sx[e] * sy[b] * sz[c] * wq;
          if (in_lds) atomicAdd(r + e + sy_ * b + sz_ * c, v);
          else unsafeAtomicAdd(r + e + sy_ * b + sz_ * c, v);
        }
  }
  lb_flush(blk, a.g, dst, 1);
  }
}

// Gather: the stencils of a particle at x lie within [floor(x) - 1,
// floor(x) + 2], and with a staggered shape of order 3 from floor(x) - 2 on.
// One workgroup per work item stages the six blocks, as the tiled kernel
// does, and its particles read them there.
//
// In random order k_gather is bound by its cache lines: 96 rows of three or
// four nodes per order-3 particle, each in lines that no other lane of the
// wave wants.  Staged, a line is read once per work item.  What is left are
// the particles' own scattered accesses, so those go through one record of
// 48 bytes per particle (its position, then its six field values) instead of
// three reads and six read-modify-writes in nine arrays.  Two million order-3
// particles on 64^3 cells: 1.35 ms plain, 0.67 ms staged, 0.46 ms with the
// records (ordering 0.09 ms); 16 million on 128^3: 22.9 -> 3.6 ms.
template <int N, int M, int B>
__global__ __launch_bounds__(512) void k_lb_gather(LbGather a, BinGeom bg, const int *perm,
                                                   const int4 *items, const int *nitems) {
  constexpr int HLO = M == 3 ? -2 : -1, HHI = 2, L = B + HHI - HLO, LN = L * L * L;
  extern __shared__ double lds[];
  const int nit = *nitems;
  const i64 org = a.c.g.idx(0, 0, 0);
  FieldView<double> fg[6];
  const double *F[6] = {a.c.exg, a.c.eyg, a.c.ezg, a.c.bxg, a.c.byg, a.c.bzg};
  for (int f = 0; f < 6; f++) fg[f] = FieldView<double>{F[f] + org, a.c.g.NX, a.c.g.NX * a.c.g.NY};
  for (int w = blockIdx.x; w < nit; w += gridDim.x) {
    const int4 it = items[w];
    const int b = it.x;
    const int o[3] = {b % bg.nb[0] * B - bg.gd[0] + HLO, b / bg.nb[0] % bg.nb[1] * B - bg.gd[1] + HLO,
                      b / (bg.nb[0] * bg.nb[1]) * B - bg.gd[2] + HLO};
    __syncthreads();  // the previous item's block is no longer read
    for (int t = threadIdx.x; t < LN; t += 512) {
      const int i = o[0] + t % L, j = o[1] + t / L % L, k = o[2] + t / (L * L);
      const bool in = a.c.g.inside(i, j, k);
      const i64 ix = in ? a.c.g.idx(i, j, k) : 0;
      double v[6];
#pragma unroll
      for (int f = 0; f < 6; f++) v[f] = in ? F[f][ix] : 0.0;
#pragma unroll
      for (int f = 0; f < 6; f++) lds[f * LN + t] = v[f];
    }
    __syncthreads();
    LdsView<double> fl[6];
    for (int f = 0; f < 6; f++) fl[f] = LdsView<double>{lds + f * LN, o[0], o[1], o[2], L, L * L};
    for (int p = threadIdx.x; p < it.z; p += 512) {
      double *rec = a.rec + 6 * (i64)perm[it.y + p];
      const double x = rec[0], y = rec[1], z = rec[2];
      GatherStencil<N, M, double> st;
      gather_stencil<N, M, double>(st, x, y, z, a.c.s);
      int lo[3], hi[3];
      gather_bounds<N, M, double>(st, lo, hi);
      bool held = a.c.g.inside(lo[0], lo[1], lo[2]) && a.c.g.inside(hi[0], hi[1], hi[2]);
      for (int d = 0; d < 3; d++) held = held && lo[d] >= o[d] && hi[d] < o[d] + L;
      double e[6];
      if (held) {
        gather_apply<N, M, double>(st, fl, e);
      } else if (!gather_eb<N, M, double>(x, y, z, a.c.s, a.c.g, fg, e)) {
        count_bad(a.c.bad);  // outside the arrays
        for (int f = 0; f < 6; f++) e[f] = -0.0;  // the outputs stay as they are
      }
#pragma unroll
      for (int f = 0; f < 6; f++) rec[f] = e[f];
    }
  }
}

// the records' field values added to the caller's arrays
__global__ __launch_bounds__(256) void k_lb_gather_add(LeafGatherArgs a, const double *rec) {
  const i64 ip = (i64)blockIdx.x * blockDim.x + threadIdx.x;
  if (ip >= a.np) return;
  const double2 *r = (const double2 *)(rec + 6 * ip);
  const double2 r0 = r[0], r1 = r[1], r2 = r[2];
  a.ex[ip] += r0.x;
  a.ey[ip] += r0.y;
  a.ez[ip] += r1.x;
  a.bx[ip] += r1.y;
  a.by[ip] += r2.x;
  a.bz[ip] += r2.y;
}

// One workgroup looks at 64 runs of 64 consecutive particles spread over the
// set: it is in no order if more than 24 of the 63 in a run have another block
// than their predecessor, on average (a set in cell order crosses blocks a few
// times a run, one in random order nearly always).  `spread` > 0: and if the
// 4096 particles are spread over at least about that many blocks, by the number
// of pairs that share one (counted in 4096 hashed counters; n particles in N
// blocks evenly: n^2 / N).
template <int B>
__global__ __launch_bounds__(1024) void k_lb_probe(LbPos a, BinGeom bg, int spread, int *out,
                                                  unsigned long long *host_out) {
  __shared__ int s[16], pairs[16], cnt[4096];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int b[4], n = 0;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const i64 ip = (a.np - 64) * (4 * wave + r) / 63 + lane;
    b[r] = block_axis<B>((a.x[ip] - a.xmin) * a.dxi, bg.gd[0], bg.na[0]) +
           bg.nb[0] * (block_axis<B>((a.y[ip] - a.ymin) * a.dyi, bg.gd[1], bg.na[1]) +
                       bg.nb[1] * block_axis<B>((a.z[ip] - a.zmin) * a.dzi, bg.gd[2], bg.na[2]));
  }
#pragma unroll
  for (int r = 0; r < 4; r++) n += __popcll(__ballot(lane > 0 && b[r] != __shfl_up(b[r], 1)));
  if (lane == 0) s[wave] = n;
  __syncthreads();
  n = 0;
  for (int w = 0; w < 16; w++) n += s[w];
  int scattered = n > 64 * 24;
  if (scattered && spread > 0) {  // (the same for all threads)
#pragma unroll
    for (int r = 0; r < 4; r++) cnt[threadIdx.x + 1024 * r] = 0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; r++) atomicAdd(&cnt[(unsigned)b[r] * 2654435761u >> 20], 1);
    __syncthreads();
    int q = 0;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int c = cnt[threadIdx.x + 1024 * r];
      q += c * (c - 1);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) q += __shfl_down(q, o);
    if (lane == 0) pairs[wave] = q;
    __syncthreads();
    q = 0;  // at most 2^24
    for (int w = 0; w < 16; w++) q += pairs[w];
    scattered = q <= (1 << 24) / spread;
  }
  if (threadIdx.x == 0) {
    *out = scattered;
    *host_out = scattered;
  }
}

// Particles below which keys and counts take one launch: the radix sort's
// blocks are of 1024 there, four a thread; of 4096 the key pass would have too
// few waves in flight.
constexpr i64 LB_COUNTED = 1 << 19;

// Scratch: the ordering's, and the records'.
enum { LB_KEYS = 24, LB_IDX, LB_HIST, LB_RANGES, LB_ITEMS, LB_NITEMS, LB_REC };
constexpr i64 LB_HIST_CAP = (i64)1 << 21;  // ints of the sort's counts
// Largest buffer kept from one call to the next.  A call that has waited for
// itself gives larger ones back (allocating and freeing a few GB takes 0.6 ms,
// a call that needs them 5 ms and more).
constexpr size_t LB_KEEP = (size_t)1 << 30;

// Buffers that order up to np particles at a time.
struct LbOrder {
  BinGeom bg;
  i64 maxitems = 0;
  int *keys, *idxs, *hist, *nitems;
  int2 *range;
  int4 *items;
  int *perm;  // set by lb_sort
};

// Returns false for a set there is no memory or index range for.  The records
// are asked for after this; those that an earlier call has left behind are
// given up for it.
static bool lb_alloc(i64 np, const GridGeom &g, int chunk, LbOrder &o) {
  o.bg = make_bin_geom(g, LB_EDGE);
  o.maxitems = o.bg.nblocks + np / chunk + 1;
  if (np >= (i64)1 << 31 || o.bg.nblocks >= (i64)1 << 31 || o.maxitems >= (i64)1 << 31)
    return false;
  const i64 hist = radix_hist_most(np, o.bg.nblocks, LB_HIST_CAP);
  for (int attempt = 0; attempt < 2; attempt++) {
    o.keys = (int *)scratch(LB_KEYS, 2 * sizeof(int) * (size_t)np);
    o.idxs = (int *)scratch(LB_IDX, 2 * sizeof(int) * (size_t)np);
    o.hist = (int *)scratch(LB_HIST, sizeof(int) * (size_t)hist);
    o.range = (int2 *)scratch(LB_RANGES, sizeof(int2) * (size_t)o.bg.nblocks);
    o.items = (int4 *)scratch(LB_ITEMS, sizeof(int4) * (size_t)o.maxitems);
    o.nitems = (int *)scratch(LB_NITEMS, sizeof(int));
    if (o.keys && o.idxs && o.hist && o.range && o.items && o.nitems) return true;
    if (!scratch_bytes(LB_REC)) return false;
    scratch_free(LB_REC);
  }
  return false;
}

// Particle indices in block order (radix sort: the input order is kept
// inside a block) and the work items.  Counting and placing the particles
// with global atomics on the blocks' counters took 0.32 ms for two million
// in random order (every particle its own atomic), this 0.09 ms.
template <int B, bool MID>
static void lb_sort(const LbPos &a, int chunk, hipStream_t st, LbOrder &o) {
  const i64 np = a.np;
  const BinGeom &bg = o.bg;
  const RadixPlan plan = radix_plan(np, bg.nblocks, LB_HIST_CAP);
  int *keys = o.keys, *idxs = o.idxs, *hist = o.hist, *nitems = o.nitems;
  // one pass of the sort: its counts say where the blocks lie
  const bool one = plan.npass == 1;
  int2 *range = one ? nullptr : o.range;
  int *key[2] = {keys, keys + np}, *idx[2] = {idxs, idxs + np};
  const bool counted = one && np < LB_COUNTED;
  if (counted)
    hipLaunchKernelGGL((k_lb_keys_count<B, MID>), dim3((unsigned)plan.nblk), dim3(256), 0, st, a,
                       bg, keys, plan.seg, plan.bits, hist, nitems);
  else
    hipLaunchKernelGGL((k_lb_keys<B, MID>), dim3(grid1d(std::max(np, bg.nblocks), 256)), dim3(256),
                       0, st, a, bg, keys, range, nitems);
  const int at = radix_sort(plan, key, idx, hist, st, counted);
  o.perm = idx[at];
  if (!one)
    hipLaunchKernelGGL(k_lb_ranges, dim3(grid1d(np, 256)), dim3(256), 0, st, np, key[at], range);
  const BlockRanges br{range, hist, plan.nblk, 1 << plan.bits, (int)np};
  hipLaunchKernelGGL(k_lb_plan, dim3(grid1d(bg.nblocks, 1024)), dim3(1024), 0, st, br, bg.nblocks,
                     chunk, o.items, nitems);
}

// The ordering and the kernels behind it share scratch.  A call launches them
// all before another thread's.  With checks off it may still be running when
// the next one comes on another stream, which therefore waits for its event
// first (7 us a call, two million particles on 64^3 cells 1122 -> 1139 us for
// a gather and a deposition; with checks on every call waits for itself and
// records none).  Where the event cannot be had the stream is waited for.
class OrderTurn {
  friend void leaf_trim();
  static std::mutex mutex;
  static hipEvent_t last;  // end of the last call's work
  std::lock_guard<std::mutex> lock{mutex};
  hipStream_t st;
  bool checks = rt().checks;

 public:
  explicit OrderTurn(hipStream_t s) : st(s) {
    if (last) (void)hipStreamWaitEvent(st, last, 0);
  }
  ~OrderTurn() {
    if (checks) return;
    if (!last && hipEventCreateWithFlags(&last, hipEventDisableTiming) != hipSuccess) last = nullptr;
    if (!last || hipEventRecord(last, st) != hipSuccess) {
      (void)hipStreamSynchronize(st);
      (void)hipGetLastError();
    }
  }
};
void leaf_trim() {
  if (!rt().checks) return;
  for (int k = LB_KEYS; k <= LB_REC; k++)
    if (scratch_bytes(k) > LB_KEEP) {
      std::lock_guard<std::mutex> lock(OrderTurn::mutex);
      if (scratch_bytes(k) > LB_KEEP) scratch_free(k);
    }
}
std::mutex OrderTurn::mutex;
hipEvent_t OrderTurn::last = nullptr;

// Particles from which a gather asks for their order.  The question costs a
// call in cell order 4 to 8 us, so it has to be a small part of the call.  A
// million on 64^3 cells: order 3 151 -> 155 us in cell order and 618 -> 293 in
// random order, order 2 106 -> 109 and 428 -> 227 (600000 on 48^3, order 2:
// 180 -> 187).  At order 1, where a particle reads eight nodes of a field, the
// staged form gains little on a small grid: one, two and four million on 64^3
// 170 -> 175, 324 -> 293 and 650 -> 580 us (four million on 128^3 995 -> 692).
constexpr i64 GATHER_BIN_MIN1 = 3 << 20, GATHER_BIN_MIN = 3 << 18;
// And particles per block of the grid: a block's six fields are staged whole,
// 1331 nodes or more each, however few particles read them.  Random order,
// plain -> staged at about this many per block and at half of it:
// order 1: four million on 200^3 (228) 1037 -> 896 us, eight on 256^3 (223)
// 2040 -> 1800; two on 200^3 (114) 530 -> 601, four on 256^3 (111) 1042 -> 1195;
// order 2: one on 200^3 (57) 749 -> 614, two on 256^3 (56) 1473 -> 1162; four
// on 384^3 (34) 3450 -> 3464, one on 256^3 (28) 756 -> 1041;
// order 3: one on 256^3 (28) 1518 -> 1222, eight on 512^3 (29) 14101 -> 9257;
// two on 384^3 (17) 3234 -> 3828, four on 512^3 (15) 7014 -> 8710.
// (A million on 512^3, 3.6 a block: 356 -> 5191, 917 -> 6589, 1747 -> 7976.)
constexpr int GATHER_PER_BLOCK[4] = {0, 192, 48, 24};
// And blocks over which the particles are spread: in few of them (a bunch) the
// plain kernel reads the fields from the caches.  A bunch of sigma cells in 128^3,
// plain and staged (us): order 1, four million, sigma 3 222 and 533, sigma 12
// (about 150 blocks) 393 and 651, a slab 4 thick (about 330) 313 and 636, 16
// thick (700) 644 and 628, sigma 24 883 and 699; order 2, a million, sigma 6
// (about 20) 181 and 209, sigma 12 254 and 239; four million, sigma 3 508 and
// 556, sigma 6 699 and 603; order 3, a million, sigma 3 234 and 244, sigma 6 342
// and 270; two million, sigma 3 445 and 398; four million, sigma 1.5 689 and 623.
static int gather_spread(int order, i64 np) {
  const bool small = np < (i64)3 << 19;
  return order == 1 ? 448 : order == 2 ? (small ? 64 : 10) : (small ? 10 : 0);
}
constexpr i64 DEPO_REC_MIN = 1 << 19;  // a million random: 236 -> 164 us (Esirkepov, order 1)
constexpr int GATHER_CHUNK = 1024;  // particles of a gather's work item

// persistent workgroups: as many as the CUs hold at this LDS size, or one
// per work item if there are fewer
static unsigned lb_grid(i64 maxitems, size_t lds) {
  const i64 per_cu = (i64)(160 * 1024 / (lds + 1024));
  const i64 g = (i64)rt().num_cus * (per_cu < 1 ? 1 : per_cu);
  return (unsigned)(maxitems < g ? maxitems : g);
}

#define LB_LAUNCH(KERNEL, ARGS)                                                               \
  do {                                                                                       \
    PXR_HIP(hipFuncSetAttribute((const void *)&KERNEL,                                      \
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));     \
    hipLaunchKernelGGL(KERNEL, grd, blk, lds, st, ARGS, o.bg, o.perm, o.items, o.nitems);     \
  } while (0)

// Work recorded into a graph, the library's or one of the caller's own, may
// not refer to scratch that a later call frees when it needs more.
static bool recording(hipStream_t st) {
  if (rt().capturing) return true;
  hipStreamCaptureStatus s = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &s) != hipSuccess) (void)hipGetLastError();
  return s != hipStreamCaptureStatusNone;
}

static bool pays(i64 np, const GridGeom &g, int per_block) {
  const Runtime &r = rt();
  return r.leaf_bin_min > 0 && np >= r.leaf_bin_min &&
         np >= per_block * make_bin_geom(g, LB_EDGE).nblocks && !recording(r.stream);
}

// Particles of a work item, of which the routine would take `own`.
static int item_size(int own) {
  const int most = rt().leaf_bin_chunk;
  return most > LEAF_BIN_CHUNK ? most : std::min(most, own);
}

int leaf_last_items(int64_t *n) {
  int *nitems = (int *)scratch(LB_NITEMS, sizeof(int)), v = 0;
  if (!nitems) return set_error(PXRHIP_ERR_HIP, "scratch allocation failed");
  PXR_HIP(hipStreamSynchronize(rt().stream));
  PXR_HIP(hipMemcpy(&v, nitems, sizeof(int), hipMemcpyDeviceToHost));
  *n = v;
  return PXRHIP_OK;
}

static LbPos gather_pos(const LeafGatherArgs &a, double *rec) {
  return LbPos{a.np, a.xp, a.yp, a.zp, nullptr, nullptr, nullptr, nullptr, nullptr, a.xmin, a.ymin,
               a.zmin, a.dxi, a.dyi, a.dzi, {0.0, 0.0, 0.0}, 0, rec, {}};
}

DepoArgs DepoArgs::part(i64 first, i64 n) const {
  DepoArgs p = *this;
  p.np = n;
  for (const double **q : {&p.xp, &p.yp, &p.zp, &p.ux, &p.uy, &p.uz, &p.gi, &p.w}) *q += first;
  return p;
}

LeafGatherArgs LeafGatherArgs::part(i64 first, i64 n) const {
  LeafGatherArgs p = *this;
  p.np = n;
  for (const double **q : {&p.xp, &p.yp, &p.zp}) *q += first;
  for (double **q : {&p.ex, &p.ey, &p.ez, &p.bx, &p.by, &p.bz}) *q += first;
  return p;
}

bool leaf_binned_gather_may_pay(const LeafGatherArgs &a, int order) {
  return rt().checks && a.np >= (order == 1 ? GATHER_BIN_MIN1 : GATHER_BIN_MIN) &&
         pays(a.np, a.g, GATHER_PER_BLOCK[order]);
}

// host: where the answer goes on the host (null: the probe's report slot)
static void launch_probe(const LbPos &pos, const GridGeom &g, int spread, hipStream_t st,
                         LeafProbe &probe, unsigned long long *host = nullptr) {
  unsigned long long *slot = report_slot();
  probe.host = host ? host : slot;
  probe.dev = (int *)(rt().d_bad + 2 + (slot - rt().h_report));
  hipLaunchKernelGGL(k_lb_probe<LB_EDGE>, dim3(1), dim3(1024), 0, st, pos,
                     make_bin_geom(g, LB_EDGE), spread, probe.dev, probe.host);
}

int leaf_probe_start(LeafGatherArgs &a, int order, hipStream_t st, LeafProbe &probe) {
  PXR_HIP(hipEventCreateWithFlags(&probe.done, hipEventDisableTiming));
  launch_probe(gather_pos(a, nullptr), a.g, gather_spread(order, a.np), st, probe);
  PXR_LAUNCHED();
  PXR_HIP(hipEventRecord(probe.done, st));
  a.skip = probe.dev;
  return PXRHIP_OK;
}

// Particles ordered at a time, in equal parts: 8 million, or 512 per block of
// the grid, which bounds the records (48 or 64 bytes a particle).  Fewer per
// block cost more than they save: a hundred million in no order on 512^3 cells,
// order 1, in one part, three, six and twelve 22.8, 26.2, 31.4 and 40.7 ms
// (Esirkepov; without records 33.4) and 24.6, 33.6, 46.0 and 77.1 (gather).
static i64 part_size(i64 np, const GridGeom &g) {
  const i64 most = std::max<i64>((i64)1 << 23, 512 * make_bin_geom(g, LB_EDGE).nblocks);
  const i64 nparts = (np + most - 1) / most;
  return (np + nparts - 1) / nparts;
}

int leaf_probe_read(LeafProbe &probe, bool &scattered) {
  PXR_HIP(hipEventSynchronize(probe.done));
  scattered = *(volatile unsigned long long *)probe.host != 0;
  return PXRHIP_OK;
}

int leaf_binned_gather(const LeafGatherArgs &a, int order, bool lower, hipStream_t st,
                       i64 &done) {
  i64 size = part_size(a.np, a.g);
  const int chunk = item_size(GATHER_CHUNK);
  const int L = LB_EDGE + (order == 3 && !lower ? 4 : 3);
  const size_t lds = sizeof(double) * 6 * (size_t)(L * L * L);
  const OrderTurn turn(st);
  done = 0;
  LbGather ga;
  LbOrder o;
  if (!lb_alloc(size, a.g, chunk, o)) return PXRHIP_OK;
  // smaller parts where there is no memory for the records of larger ones
  while (!(ga.rec = (double *)scratch(LB_REC, 6 * sizeof(double) * (size_t)size))) {
    if (size < GATHER_BIN_MIN) return PXRHIP_OK;
    size = (size + 1) / 2;
  }
  while (done < a.np) {
    ga.c = a.part(done, std::min(size, a.np - done));
    lb_sort<LB_EDGE, false>(gather_pos(ga.c, ga.rec), chunk, st, o);
    const dim3 grd(lb_grid(o.maxitems, lds)), blk(512);
    switch (order * 2 + (lower ? 1 : 0)) {
      case 2: LB_LAUNCH((k_lb_gather<1, 1, LB_EDGE>), ga); break;
    case 3: LB_LAUNCH((k_lb_gather<1, 0, LB_EDGE>), ga); break;
    case 4: LB_LAUNCH((k_lb_gather<2, 2, LB_EDGE>), ga); break;
      case 5: LB_LAUNCH((k_lb_gather<2, 1, LB_EDGE>), ga); break;
      case 6: LB_LAUNCH((k_lb_gather<3, 3, LB_EDGE>), ga); break;
      default: LB_LAUNCH((k_lb_gather<3, 2, LB_EDGE>), ga); break;
    }
    hipLaunchKernelGGL(k_lb_gather_add, dim3(grid1d(ga.c.np, 256)), dim3(256), 0, st, ga.c,
                       ga.rec);
    PXR_LAUNCHED();
    done += ga.c.np;
  }
  return PXRHIP_OK;
}

// Particles per block of the grid from which a direct current is summed block
// by block.  A block's three LDS arrays are cleared and added up whole, so few
// particles do not repay it.  Unbinned and binned at orders 1, 2 and 3: 66,000
// on 200^3 cells (3.8 a block) 98, 268, 604 and 154, 355, 626 us; a million on
// 512^3 (3.6) 1209, 3752, 8629 and 1590, 4834, 9520; on 384^3 (8.5) 1176, 3670,
// 8501 and 869, 2331, 4483; 300,000 on 200^3 (17) 346, 1110, 2561 and 234, 448,
// 727.  (The Esirkepov current and the charge density are faster binned at one
// a block already.)
constexpr int DIRECT_PER_BLOCK = 8;

bool leaf_binned_current_pays(i64 np, const GridGeom &g, bool direct) {
  return pays(np, g, direct ? DIRECT_PER_BLOCK : 1);
}
bool leaf_binned_rho_pays(i64 np, const GridGeom &g) { return pays(np, g, 1); }

// the current of a.np particles, in parts that bound the records' memory
template <bool MID>
static int binned_current(const DepoArgs &a, int order, hipStream_t st, i64 &done) {
  const OrderTurn turn(st);
  const EsirkConst<double> &c = a.ec;
  // (with checks off nobody waits, and larger records would be kept)
  const bool records = order <= 2 && a.np >= DEPO_REC_MIN &&
                       (rt().checks ||
                        8 * sizeof(double) * (size_t)part_size(a.np, a.g) <= LB_KEEP);
  const i64 size = records ? part_size(a.np, a.g) : a.np;
  const int L = LB_EDGE + (order == 1 ? 3 : 5);
  const size_t lds = sizeof(double) * 3 * (size_t)(L * L * L);
  // A full block holds a few thousand particles at the densities of interest,
  // and the blocks of a modest grid are too few to share evenly among the CUs:
  // smaller work items, until clearing and adding up the LDS blocks costs as
  // much.  Two million in cell order on 64^3 cells, 4096 particles an item and
  // so: order 1 374 -> 177 us, order 2 402 -> 255, order 3 446 -> 410.
  const int chunk = item_size(order == 1 ? 512 : order == 2 ? 1024 : 2048);
  done = 0;
  LbDepo d;
  rt().last_leaf_records_asked = false;
  LbOrder o;
  if (!lb_alloc(size, a.g, chunk, o)) return PXRHIP_OK;
  if (records)  // (without memory for them the arrays are read)
    d.packed.rec = (double *)scratch(LB_REC, 8 * sizeof(double) * (size_t)size);
  while (done < a.np) {
    d.c = a.part(done, std::min(size, a.np - done));
    LbPos pos{d.c.np, d.c.xp, d.c.yp, d.c.zp, d.c.ux, d.c.uy, d.c.uz, d.c.gi, d.c.w, c.xmin,
              c.ymin, c.zmin, c.dxi, c.dyi, c.dzi,
              {0.5 * c.dtsdx0, 0.5 * c.dtsdy0, 0.5 * c.dtsdz0}, 0, nullptr, {}};
    if (d.packed.rec) {
      LeafProbe probe;
      launch_probe(pos, a.g, 0, st, probe, records_word());
      rt().last_leaf_records_asked = true;
      d.packed.use = probe.dev;
      pos.packed = d.packed;
    }
    lb_sort<LB_EDGE, MID>(pos, chunk, st, o);
    const dim3 grd(lb_grid(o.maxitems, lds)), blk(256);
    if constexpr (MID) {
      if (order == 1) LB_LAUNCH((k_lb_direct<1, LB_EDGE>), d);
      else if (order == 2) LB_LAUNCH((k_lb_direct<2, LB_EDGE>), d);
      else LB_LAUNCH((k_lb_direct<3, LB_EDGE>), d);
    } else {
      if (order == 1) LB_LAUNCH((k_lb_esirkepov<1, LB_EDGE>), d);
      else if (order == 2) LB_LAUNCH((k_lb_esirkepov<2, LB_EDGE>), d);
      else LB_LAUNCH((k_lb_esirkepov<3, LB_EDGE>), d);
    }
    PXR_LAUNCHED();
    done += d.c.np;
  }
  return PXRHIP_OK;
}

int leaf_binned_direct(const DepoArgs &a, int order, hipStream_t st, i64 &done) {
  return binned_current<true>(a, order, st, done);
}

int leaf_binned_esirkepov(const DepoArgs &a, int order, hipStream_t st, i64 &done) {
  return binned_current<false>(a, order, st, done);
}

int leaf_binned_rho(const RhoArgs &a, int order, hipStream_t st, bool &done) {
  const OrderTurn turn(st);
  done = false;
  constexpr int E = LB_EDGE;
  LbOrder o;
  const LbPos pos{a.np, a.xp, a.yp, a.zp, nullptr, nullptr, nullptr, nullptr, nullptr, a.xmin, a.ymin,
                  a.zmin, a.dxi, a.dyi, a.dzi, {0.0, 0.0, 0.0}, a.l4symtry, nullptr, {}};
  // work items as for the currents: 33.6 million in cell order on 128^3 cells,
  // 4096 particles an item and so, 3.46 -> 1.58, 3.44 -> 1.83 and 3.47 -> 2.85
  // ms at orders 1 to 3
  const int chunk = item_size(order == 3 ? 2048 : 1024);
  if (!lb_alloc(a.np, a.g, chunk, o)) return PXRHIP_OK;
  lb_sort<E, false>(pos, chunk, st, o);
  const int L = E + (order == 1 ? 1 : 3);
  const size_t lds = sizeof(double) * (size_t)(L * L * L);
  const dim3 grd(lb_grid(o.maxitems, lds)), blk(256);
  if (order == 1) LB_LAUNCH((k_lb_rho<1, E>), a);
  else if (order == 2) LB_LAUNCH((k_lb_rho<2, E>), a);
  else LB_LAUNCH((k_lb_rho<3, E>), a);
  PXR_LAUNCHED();
  done = true;
  return PXRHIP_OK;
}

}  // namespace pxr
