// pxr_leafbin.hip -- the leaf current and charge deposition (depose_jxjyjz,
// pxr_depose_rho_n) for large particle sets, summed block by block in LDS.
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
// only the order of the FP64 sums differs.  Nothing synchronises with the
// host, so the sequence can be captured in a HIP graph once its scratch is
// allocated.
#include <algorithm>

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

// positions (and, for the mid positions, velocities and h = dt / (2 dx)) of
// one call
struct LbPos {
  i64 np;
  const double *x, *y, *z, *ux, *uy, *uz, *gi;
  double xmin, ymin, zmin, dxi, dyi, dzi, h[3];
  int l4symtry;
};

// Block of every particle, by the node of its position (MID: of its
// position half a step back, where the direct current is deposited).
template <int B, bool MID>
__global__ __launch_bounds__(256) void k_lb_keys(LbPos a, BinGeom bg, int *key) {
  const i64 ip = (i64)blockIdx.x * blockDim.x + threadIdx.x;
  if (ip >= a.np) return;
  double x = (a.x[ip] - a.xmin) * a.dxi, y = (a.y[ip] - a.ymin) * a.dyi;
  double z = (a.z[ip] - a.zmin) * a.dzi;
  if (MID) {
    const double gi = a.gi[ip];
    x -= a.h[0] * (a.ux[ip] * gi);
    y -= a.h[1] * (a.uy[ip] * gi);
    z -= a.h[2] * (a.uz[ip] * gi);
  } else if (a.l4symtry) {
    x = fabs(x);
    y = fabs(y);
  }
  key[ip] = block_axis<B>(x, bg.gd[0], bg.na[0]) +
            bg.nb[0] * (block_axis<B>(y, bg.gd[1], bg.na[1]) +
                        bg.nb[1] * block_axis<B>(z, bg.gd[2], bg.na[2]));
}

// first[b]: the first sorted particle of block b (first[nblocks] = np)
__global__ __launch_bounds__(256) void k_lb_first(i64 np, const int *key, i64 nblocks,
                                                  int *first) {
  const i64 j = (i64)blockIdx.x * blockDim.x + threadIdx.x;
  if (j > np) return;
  const i64 prev = j ? key[j - 1] : -1, here = j < np ? key[j] : nblocks;
  for (i64 b = prev + 1; b <= here; b++) first[b] = (int)j;
}

// One workgroup: the work items (block, first slot, count) of at most
// `chunk` particles of one block.  Each thread owns a contiguous range of
// blocks.
__global__ __launch_bounds__(1024) void k_lb_plan(const int *first, i64 nblocks, int chunk,
                                                  int4 *items, int *nitems) {
  __shared__ int s[16];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const i64 per = (nblocks + 1023) / 1024;
  const i64 b0 = min(nblocks, (i64)t * per), b1 = min(nblocks, b0 + per);
  int ni = 0;
  for (i64 b = b0; b < b1; b++) ni += (first[b + 1] - first[b] + chunk - 1) / chunk;
  int inc = ni;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(inc, off);
    if (lane >= off) inc += y;
  }
  if (lane == 63) s[w] = inc;
  __syncthreads();
  int it = inc - ni;
  for (int k = 0; k < w; k++) it += s[k];
  for (i64 b = b0; b < b1; b++) {
    const int f = first[b], c = first[b + 1] - f;
    for (int k = 0; k < c; k += chunk) items[it++] = make_int4((int)b, f + k, min(chunk, c - k), 0);
  }
  if (t == 1023) *nitems = it;
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

// Lanes take particles S = ceil(n / 256) apart, so that in cell-ordered
// input the lanes of a wave sit in different cells.
PXR_DEV int lb_stride(int n) { return (n + (int)blockDim.x - 1) / (int)blockDim.x; }

// Esirkepov current: the box of an order-N particle lies within
// [floor(x) - 2, floor(x) + 3] (order 1: [-1, +2]) on each axis.
template <int N, int B>
__global__ __launch_bounds__(256) void k_lb_esirkepov(DepoArgs a, BinGeom bg, const int *perm,
                                                      const int4 *items, const int *nitems) {
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
  const int n = it.z, S = lb_stride(n);
  for (int k = 0; k < S; k++) {
    const int p = (int)threadIdx.x * S + k;
    if (p >= n) break;
    const i64 ip = perm[it.y + p];
    EsirkepovIn<double> in;
    esirkepov_prepare<N, double>(in, a.xp[ip], a.yp[ip], a.zp[ip], a.ux[ip], a.uy[ip],
                                 a.uz[ip], a.gi[ip], a.w[ip], a.ec);
    int lo[3], hi[3];
    if (!esirkepov_box<N, double>(in, lo, hi) || !a.g.inside(lo[0], lo[1], lo[2]) ||
        !a.g.inside(hi[0], hi[1], hi[2])) {
      count_bad(a.bad);
      continue;
    }
    if (blk.holds(lo, hi)) esirkepov_deposit<N, double>(in, acc);
    else esirkepov_deposit<N, double>(in, gacc);  // not reached: the halo holds every box
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
__global__ __launch_bounds__(256) void k_lb_direct(DepoArgs a, BinGeom bg, const int *perm,
                                                   const int4 *items, const int *nitems) {
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
    const int n = it.z, S = lb_stride(n);
    for (int k = 0; k < S; k++) {
      const int p = (int)threadIdx.x * S + k;
      if (p >= n) break;
      const i64 ip = perm[it.y + p];
      DirectIn<double> in;
      direct_prepare<N, double>(in, a.xp[ip], a.yp[ip], a.zp[ip], a.ux[ip], a.uy[ip], a.uz[ip],
                                a.gi[ip], a.w[ip], a.q, a.xmin, a.ymin, a.zmin, a.dt, a.dx, a.dy,
                                a.dz, a.s);
      int lo[3], hi[3];
      direct_box<N>(in, lo, hi);
      if (!a.g.inside(lo[0], lo[1], lo[2]) || !a.g.inside(hi[0], hi[1], hi[2])) {
        count_bad(a.bad);
        continue;
      }
      if (blk.holds(lo, hi)) direct_deposit<N, double>(in, acc);
      else direct_deposit<N, double>(in, gacc);  // not reached: the halo holds every box
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
  const int n = it.z, S = lb_stride(n);
  for (int k = 0; k < S; k++) {
    const int p = (int)threadIdx.x * S + k;
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

// Particle indices in block order (radix sort: the input order is kept
// inside a block) and the work items.  Counting and placing the particles
// with global atomics on the blocks' counters took 0.32 ms for two million
// in random order (every particle its own atomic), this 0.09 ms.
template <int B, bool MID>
static int lb_sort(const LbPos &a, const GridGeom &g, int chunk, hipStream_t st, BinGeom &bg,
                   int *&perm, int4 *&items, int *&nitems, i64 &maxitems) {
  bg = make_bin_geom(g, B);
  const i64 np = a.np;
  maxitems = bg.nblocks + np / chunk + 1;
  if (np >= (i64)1 << 31 || bg.nblocks >= (i64)1 << 31 || maxitems >= (i64)1 << 31)
    return set_error(PXRHIP_ERR_ARG, "binned deposition: more than 2^31 particles or blocks");
  const RadixPlan plan = radix_plan(np, bg.nblocks, (i64)1 << 21);
  int *keys = (int *)scratch(24, 2 * sizeof(int) * (size_t)np);
  int *idxs = (int *)scratch(25, 2 * sizeof(int) * (size_t)np);
  int *hist = (int *)scratch(26, sizeof(int) * (size_t)plan.hist_ints);
  int *first = (int *)scratch(27, sizeof(int) * (size_t)(bg.nblocks + 1));
  items = (int4 *)scratch(28, sizeof(int4) * (size_t)maxitems);
  nitems = (int *)scratch(29, sizeof(int));
  if (!keys || !idxs || !hist || !first || !items || !nitems)
    return set_error(PXRHIP_ERR_HIP, "binned deposition: out of device memory");
  int *key[2] = {keys, keys + np}, *idx[2] = {idxs, idxs + np};
  hipLaunchKernelGGL((k_lb_keys<B, MID>), dim3(grid1d(np, 256)), dim3(256), 0, st, a, bg, keys);
  const int at = radix_sort(plan, key, idx, hist, st);
  perm = idx[at];
  hipLaunchKernelGGL(k_lb_first, dim3(grid1d(np + 1, 256)), dim3(256), 0, st, np, key[at],
                     bg.nblocks, first);
  hipLaunchKernelGGL(k_lb_plan, dim3(1), dim3(1024), 0, st, first, bg.nblocks, chunk, items,
                     nitems);
  PXR_LAUNCHED();
  return PXRHIP_OK;
}

constexpr int LB_EDGE = 8;  // nodes per block edge

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
    hipLaunchKernelGGL(KERNEL, grd, blk, lds, st, ARGS, bg, perm, items, nitems);             \
  } while (0)

static bool pays(i64 np, const GridGeom &g, int edge) {
  const Runtime &r = rt();
  return r.leaf_bin_min > 0 && np >= r.leaf_bin_min && !r.capturing &&
         np >= make_bin_geom(g, edge).nblocks;
}

bool leaf_binned_current_pays(i64 np, const GridGeom &g) { return pays(np, g, LB_EDGE); }
bool leaf_binned_rho_pays(i64 np, const GridGeom &g) { return pays(np, g, LB_EDGE); }

int leaf_binned_direct(const DepoArgs &a, int order, hipStream_t st) {
  BinGeom bg;
  int *perm, *nitems;
  int4 *items;
  i64 maxitems;
  const EsirkConst<double> &c = a.ec;
  const LbPos pos{a.np, a.xp, a.yp, a.zp, a.ux, a.uy, a.uz, a.gi, c.xmin, c.ymin, c.zmin, c.dxi,
                  c.dyi, c.dzi, {0.5 * c.dtsdx0, 0.5 * c.dtsdy0, 0.5 * c.dtsdz0}, 0};
  int r = lb_sort<LB_EDGE, true>(pos, a.g, rt().leaf_bin_chunk, st, bg, perm, items, nitems,
                                 maxitems);
  if (r) return r;
  const int L = LB_EDGE + (order == 1 ? 3 : 5);
  const size_t lds = sizeof(double) * 3 * (size_t)(L * L * L);
  const dim3 grd(lb_grid(maxitems, lds)), blk(256);
  if (order == 1) LB_LAUNCH((k_lb_direct<1, LB_EDGE>), a);
  else if (order == 2) LB_LAUNCH((k_lb_direct<2, LB_EDGE>), a);
  else LB_LAUNCH((k_lb_direct<3, LB_EDGE>), a);
  PXR_LAUNCHED();
  return PXRHIP_OK;
}

int leaf_binned_esirkepov(const DepoArgs &a, int order, hipStream_t st) {
  BinGeom bg;
  int *perm, *nitems;
  int4 *items;
  i64 maxitems;
  const EsirkConst<double> &c = a.ec;
  const LbPos pos{a.np, a.xp, a.yp, a.zp, nullptr, nullptr, nullptr, nullptr, c.xmin, c.ymin,
                  c.zmin, c.dxi, c.dyi, c.dzi, {0.0, 0.0, 0.0}, 0};
  int r = lb_sort<LB_EDGE, false>(pos, a.g, rt().leaf_bin_chunk, st, bg, perm, items, nitems,
                                  maxitems);
  if (r) return r;
  const int L = LB_EDGE + (order == 1 ? 3 : 5);
  const size_t lds = sizeof(double) * 3 * (size_t)(L * L * L);
  const dim3 grd(lb_grid(maxitems, lds)), blk(256);
  if (order == 1) LB_LAUNCH((k_lb_esirkepov<1, LB_EDGE>), a);
  else if (order == 2) LB_LAUNCH((k_lb_esirkepov<2, LB_EDGE>), a);
  else LB_LAUNCH((k_lb_esirkepov<3, LB_EDGE>), a);
  PXR_LAUNCHED();
  return PXRHIP_OK;
}

int leaf_binned_rho(const RhoArgs &a, int order, hipStream_t st) {
  constexpr int E = LB_EDGE;
  BinGeom bg;
  int *perm, *nitems;
  int4 *items;
  i64 maxitems;
  const LbPos pos{a.np, a.xp, a.yp, a.zp, nullptr, nullptr, nullptr, nullptr, a.xmin, a.ymin,
                  a.zmin, a.dxi, a.dyi, a.dzi, {0.0, 0.0, 0.0}, a.l4symtry};
  int r = lb_sort<E, false>(pos, a.g, rt().leaf_bin_chunk, st, bg, perm, items, nitems, maxitems);
  if (r) return r;
  const int L = E + (order == 1 ? 1 : 3);
  const size_t lds = sizeof(double) * (size_t)(L * L * L);
  const dim3 grd(lb_grid(maxitems, lds)), blk(256);
  if (order == 1) LB_LAUNCH((k_lb_rho<1, E>), a);
  else if (order == 2) LB_LAUNCH((k_lb_rho<2, E>), a);
  else LB_LAUNCH((k_lb_rho<3, E>), a);
  PXR_LAUNCHED();
  return PXRHIP_OK;
}

}  // namespace pxr
