// pxr_leafbin.h -- arguments of the leaf deposition kernels (global
// atomics, pxr_leaf.hip) and of their binned form (pxr_leafbin.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "pxr_device.h"
#include "pxr_kernels.h"

namespace pxr {

// current deposition of one call of depose_jxjyjz
struct DepoArgs {
  i64 np;
  const double *xp, *yp, *zp, *ux, *uy, *uz, *gi, *w;
  double q, xmin, ymin, zmin, dt, dx, dy, dz, s;
  EsirkConst<double> ec;
  GridGeom g;
  double *jx, *jy, *jz;
  unsigned long long *bad;
  DepoArgs part(i64 first, i64 n) const;  // the same call for n particles from `first`
};

// one call of geteb3d_energy_conserving with one order on all axes
struct LeafGatherArgs {
  i64 np;
  const double *xp, *yp, *zp;
  double *ex, *ey, *ez, *bx, *by, *bz;
  double xmin, ymin, zmin, dxi, dyi, dzi, s;
  GridGeom g;
  const double *exg, *eyg, *ezg, *bxg, *byg, *bzg;
  unsigned long long *bad;
  const int *skip;  // not null: k_gather leaves the set alone if *skip is set
  LeafGatherArgs part(i64 first, i64 n) const;  // the same call for n particles from `first`
};

// charge density of one call of pxr_depose_rho_n
struct RhoArgs {
  i64 np;
  const double *xp, *yp, *zp, *w;
  double q, xmin, ymin, zmin, dxi, dyi, dzi, invvol;
  int per_particle_weight, l4symtry;
  GridGeom g;
  double *rho;
  unsigned long long *bad;
};

// global-memory accumulator of the current (FP64 atomics), node (0,0,0)
// at p[c]
struct GlobalAcc {
  double *p[3];
  i64 sy, sz;
  PXR_DEV void add(int c, int i, int j, int k, double v) const {
    unsafeAtomicAdd(p[c] + (i + sy * j + sz * k), v);
  }
  PXR_DEV double *row(int c, int i, int j, int k) const { return p[c] + (i + sy * j + sz * k); }
  PXR_DEV void add_row(double *r, int o, double v) const { unsafeAtomicAdd(r + o, v); }
};

// Binned forms: the particles are ordered by cubic blocks of nodes
// and each block's current (or charge) is summed in LDS
// before one global add per node.  They launch and do not wait.  Without memory
// for the order they return PXRHIP_OK with nothing done (done = 0 or false),
// and the unbinned kernels take the particles from `done` on.
int leaf_binned_esirkepov(const DepoArgs &a, int order, hipStream_t st, i64 &done);
int leaf_binned_direct(const DepoArgs &a, int order, hipStream_t st, i64 &done);
int leaf_binned_rho(const RhoArgs &a, int order, hipStream_t st, bool &done);
// whether a call of np particles on grid g takes the binned form: at least
// the runtime's leaf_bin_min particles and one per block (eight for the direct
// current), and no graph capture open (the scratch may have to grow)
bool leaf_binned_current_pays(i64 np, const GridGeom &g, bool direct);
bool leaf_binned_rho_pays(i64 np, const GridGeom &g);

// The gather of a set in no order: particles ordered by blocks, the block's
// fields staged in LDS.  A set in cell order reads the grid arrays through the
// caches faster without, so for a call that may gain a probe looks at the
// order first.  leaf_probe_start sets a.skip, so that the plain kernel can be
// launched behind it at once and steps aside for a set in no order;
// leaf_probe_read waits for the answer.  leaf_binned_gather returns how many
// particles are done: all of them, or fewer where it ran out of memory.
bool leaf_binned_gather_may_pay(const LeafGatherArgs &a, int order);
struct LeafProbe {
  hipEvent_t done = nullptr;
  unsigned long long *host = nullptr;
  int *dev = nullptr;
  ~LeafProbe() {
    if (done) (void)hipEventDestroy(done);
  }
};
int leaf_probe_start(LeafGatherArgs &a, int order, hipStream_t st, LeafProbe &probe);
int leaf_probe_read(LeafProbe &probe, bool &scattered);
// gives scratch beyond 1 GiB a buffer back, after a call that has waited
void leaf_trim();
// work items of the last call, or part of one, that went block by block
int leaf_last_items(int64_t *n);
int leaf_binned_gather(const LeafGatherArgs &a, int order, bool lower, hipStream_t st, i64 &done);

}  // namespace pxr
