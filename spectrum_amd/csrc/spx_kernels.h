// spx_kernels.h -- launch-side types shared by the kernels and the host runtime.
#pragma once

#include <stdint.h>
#include <hip/hip_runtime.h>

#include "spx_plan.h"
#include "spx_acc.h"
#include "../../include/spectrum_amd.h"

namespace spx {

// Device-side control block of one run or served query.
struct RunCtl {
   unsigned long long next;             // next trajectory id handed out
   unsigned long long done;             // trajectories finished (accepted or failed)
   unsigned long long failed;           // trajectories that exhausted their attempts
   unsigned long long steps_done;       // accepted steps of finished trajectories
   unsigned long long steps_executed;   // every executed step (throughput counter)
   unsigned long long discards[8];      // discarded attempts by reason
   unsigned long long tmin_bits, tmax_bits;
};

// One run, or one served query: what its trajectories share.  Lives in device memory and is read
// with scalar loads; each slot pool holds a table of them.
struct QueryDesc {
   const spx_plan_desc* plan;
   RunCtl* ctl;
   spx_rng_desc rng;                    // replay pointers are device pointers here
   uint64_t first, end;                 // trajectory id range
   int32_t n_dist, pad_;
   int64_t hist_off[SPX_MAX_DIST];      // offsets of each distribution in this query's counts (bins)
   int64_t acc_off[SPX_MAX_DIST];       // and in its exact sums (bin components)
   unsigned long long* hist_counts;
   unsigned long long* hist_acc;        // SPX_ACC_LIMBS limbs per bin component (spx_acc.h)
   unsigned long long* hist_events;     // per distribution
   spx_traj_record* records;            // optional per-trajectory records
   uint64_t rec_first, rec_n;
};

// A pool of trajectory slots (kernel argument block, in device memory).  The slots of one wave always
// work for the same query; a wave moves on to the oldest admitted query with trajectories left when
// all of its slots are idle and its own query has none.
struct Launch {
   const QueryDesc* queries;            // query table
   const int32_t* queue;                // admitted query indices, oldest first
   int32_t n_queue;
   int32_t n_queries;                   // size of the query table
   uint64_t n_lanes;                    // a multiple of the block size: waves are always full
   int32_t* slot_q;                     // query index of each slot (-1: none)
   // lane state (structure of arrays, n_lanes each; boundary arrays SPX_MAX_BND * n_lanes)
   int32_t* active;
   double *t, *x, *y, *z, *m0, *m1, *m2, *amp, *wgt, *dt_prev, *src_old, *ds_prev, *dmax, *dt_adapt;
   double* pf;                          // momentum magnitude of the slot's last field evaluation (guiding centre)
   float* kc;                           // SPX_KC * n_lanes: compensation terms of the FP32-step kernels' FP64 sums
   double *bdelta, *bdelta_old;
   int32_t *bcross, *bstat;
   uint64_t* traj;
   uint32_t *nn, *nu;
   int32_t* attempt;
   int64_t* steps;
   int32_t* n_events;
   // start state (read when an event is binned)
   double *t0, *x0, *y0, *z0, *m00, *m01, *m02;
   // last event per distribution (SPX_MAX_DIST * n_lanes)
   int32_t* ev_bin;
   double* ev_w;
   // events queued by the step kernel for the service kernel: 3 classes x 9 fields x n_lanes
   double* evs;
   int32_t* ev_bnd;                     // 3 * n_lanes
   int32_t* ev_pending;                 // bit per class
   int32_t* ex_code;                    // discard reason of the last step kernel
   // compaction (LaunchShape::list): the place of each running slot among its query's, the running slots of each
   // query counted by the service kernel (two sets of n_queries, used in turn), and the list of running slots
   int32_t* rank;
   uint32_t* n_running;
   int32_t* list;
};

// Slot states
enum { SLOT_IDLE = 0, SLOT_RUN = 1, SLOT_START = 2, SLOT_EVENT = 3, SLOT_DONE = 4, SLOT_DISCARD = 5 };

// Thread i of n_threads of the packing pass of a launch, one per slot of the span and per list place at least: a running
// slot goes to its query's part of the list, a place that no slot takes gets -1, and the other set of counts is cleared
// for the next packed launch, all of it however large the query table is.  The parts follow the admission order, each
// from a wave boundary.
template <typename LP>
__host__ __device__ __forceinline__ void pack_place(LP L, int32_t packed, uint64_t span, uint64_t list_span, uint64_t i, uint64_t n_threads)
{
   const uint32_t* n_running = L->n_running + (int64_t)packed * L->n_queries;
   uint32_t* other = L->n_running + (int64_t)(1 - packed) * L->n_queries;
   const int32_t q = i < span && L->active[i] == SLOT_RUN ? L->slot_q[i] : -1;
   uint64_t start = 0;
   bool taken = false;
   for (int k = 0; k < L->n_queue; k++) {
      const int32_t c = L->queue[k];
      const uint32_t n = n_running[c];
      if (c == q) L->list[start + (uint64_t)L->rank[i]] = (int32_t)i;
      taken = taken || (i >= start && i < start + n);
      start += (n + 63u) & ~63u;
   }
   if (i < list_span && !taken) L->list[i] = -1;
   for (uint64_t c = i; c < (uint64_t)L->n_queries; c += n_threads) other[c] = 0u;
}

// What one engine launch covers.
struct LaunchShape {
   uint64_t span = 0;                   // slots the service kernel covers: the first `span`, whole blocks
   int32_t n_steps = 0;                 // steps per running slot
   bool few = false;                    // the few-wave step kernel
   // The step kernel takes the running slots from a list that packs them into full waves, a query's in consecutive
   // places from a wave boundary; -1: the slots in place.  0 or 1 picks the set of n_running the launch uses.
   int32_t packed = -1;
   int64_t turn = -1;                   // launches of the run so far, where a launch may leave slots for the next (step_window)
   uint64_t list_span = 0;              // list places the step kernel covers (whole waves): at least those in use
};

// Compensated FP64 accumulation of the FP32-step kernels: the sums t, x, y, z and p (Parker) or
// t, x, y, z (guiding centre) each carry a Kahan compensation term, kept per slot across launches.
#define SPX_KC 5

// Host-side dispatch.  One engine launch is the service kernel followed by the step kernel on
// `stream`; when `mid` is not null it is recorded between the two, so the caller can time each
// kernel with events.  launch_f64 / launch_f32 pick the instantiation for (transport, background,
// flow, diffusion) of each precision; they live in separately compiled units.  The step kernels of has_few exist in
// two forms with the same results: one for a device full of waves, and one for few resident waves (`few`, in units of
// their own), where a launch lasts as long as the longest step chain of one wave and most of the chip idles.
// A wave then issues one instruction every 4 cycles whatever its independence, so the way to a shorter step is
// fewer instructions per lane: four lanes share a trajectory (quad_get in spx_engine.h).
enum { LAUNCH_BOTH = 0, LAUNCH_FEW = 1, LAUNCH_SERVICE = 2 };   // dispatch templates: service + step, the few-wave step, service alone
hipError_t launch_f64(const spx_plan_desc& host_plan, const LaunchShape& shape, const Launch* dev_launch, hipStream_t stream, hipEvent_t mid);
hipError_t launch_f32(const spx_plan_desc& host_plan, const LaunchShape& shape, const Launch* dev_launch, hipStream_t stream, hipEvent_t mid);
hipError_t launch_few_f64(const spx_plan_desc& host_plan, const LaunchShape& shape, const Launch* dev_launch, hipStream_t stream);
hipError_t launch_few_f32(const spx_plan_desc& host_plan, const LaunchShape& shape, const Launch* dev_launch, hipStream_t stream);
// The list of the running slots after a service kernel that counted them (spx_kernels_f64.hip).
hipError_t pack_running(const LaunchShape& shape, const Launch* dev_launch, hipStream_t stream);

// Which step kernels have the few-wave form.  Measured on one wave per SIMD, one pass: FP64 modulation 15.6 -> 9.4 ms
// (64 trajectories), guiding centre 265 -> 189 ms (5000), gridded wind with anisotropic kappa 565 -> 306 ms (10^4);
// FP32 with kappa ~ T r^2 41 -> 26 ms (2000), gridded anisotropic 289 -> 134 ms (500).
inline bool has_few(const spx_plan_desc& p, int precision)
{
   if (precision == SPX_PREC_FP64) return p.traj_type <= SPX_TRAJ_FIELDLINE;
   const bool parker = p.traj_type == SPX_TRAJ_PARKER || p.traj_type == SPX_TRAJ_PARKER_SOURCE || p.traj_type == SPX_TRAJ_FIELDLINE;
   return parker && (p.bg.kind == SPX_BG_SOLARWIND || p.bg.kind == SPX_BG_GRID);
}

// FP32 cell records of a Cartesian grid (spx_grid_desc::c32) from its device zone records (nz[0] x nz[1] x
// nz[2], x fastest, SPX_GRID_REC doubles each): for every zone, the 8 zones of the stencil whose lowest
// corner it is, in corner order i + 2j + 4k (corners beyond the last zone repeat it; no stencil reads them).
hipError_t grid_expand_cells(const double* zones, const int32_t nz[3], float* c32, hipStream_t st);

inline hipError_t launch_transport(const spx_plan_desc& host_plan, const LaunchShape& shape, const Launch* dev_launch,
                                   int precision, hipStream_t stream, hipEvent_t mid)
{
   return precision == SPX_PREC_MIXED ? launch_f32(host_plan, shape, dev_launch, stream, mid)
                                      : launch_f64(host_plan, shape, dev_launch, stream, mid);
}

}  // namespace spx
