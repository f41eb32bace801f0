// gxt_kernels.h -- kernel argument blocks and host-side launchers.
#pragma once

#include <hip/hip_runtime.h>

#include "gxt_types.h"

namespace gxt {

// Histogram rows: workgroup b adds into row b % nrows, bins[row * stride + (z | nz
// + r | nz + nr + vol)] and spec[row * 3 * kSpecBins + species * kSpecBins + bin].
struct TallyRows {
  double *bins;
  unsigned long long *spec;
  int64_t stride;
  int nrows;
  int pad;
};

// Arguments of a step-loop launch (k_loop) and of the injection.
struct LoopArgs {
  const DevParams *P;
  Counters *cnt;
  DevEvent *ev;
  int *ev_live;      // live tracks of event slot e from ev_live[e * kLiveStride] on (kLive*)
  char *pages;       // npages pages of page_bytes<R>()
  uint32_t *list;    // ring of the pages with tracks, mask + 1 entries (Rings)
  uint32_t *freel;   // ring of the free pages, mask + 1 entries
  PageSeg *seg;      // two arrays of `groups` (Rings::parity)
  uint32_t mask;
  int npages;
  TallyRows rows;
  double *trace;
  int64_t trace_cap;
  int mode;          // transport: 0 plain, 1 with e-/e+ multiple scattering, 2 e-/e+ in a field map with
                     // the local helix, 3 with the RK45 stepper, 4 the volume tree
  int lds_tables;    // staged in LDS (kLds*)
  int lds_tab_bytes; // dynamic LDS they take
  int lds_bytes;     // dynamic LDS with the event sums
  int ev_slots;      // events with sums in LDS
  int groups;        // workgroups launched (at most)
  int keep;          // workgroups keep their pages from launch to launch
  int max_tracks;    // tracks the pool holds (one workgroup); 0: as many as find pages
  int once;          // transport each track once at most
  long long iter_end;  // Rings::iters from which no task runs; LLONG_MAX: no limit
  int ticks;         // 100 MHz ticks after which a workgroup starts no further task
  int prof;          // accumulate the time of the loop's parts (kStatTime*)
};

struct SampleArgs {
  int n;
  const double *ekin;
  const double *dir;
  uint32_t *rng;
  double *out_ekin;
  double *out_dir;
  double *out_edep;
  int32_t *nsec;
  int32_t *sec_species;
  double *sec_ekin;
  double *sec_dir;
};

// LDS of a launch beside its tables and event sums, and all of a workgroup's.
constexpr int kLoopLdsFixed = 31 * 1024;
constexpr int kEventSumBytes = 72;
constexpr int kMinEvSlots = 128, kMaxEvSlots = 512;
constexpr int kLoopLds = 160 * 1024;
// Raises the LDS limit of the loop of a mode (LoopArgs::mode, lds_tables) on the
// current device, where its launches need it: once for every context, on the
// device of its stream, as launches may come from threads with another current
// device.
template <class R>
hipError_t prepare_loop(int mode, int lds_tables);
template <class R, int kMode>
hipError_t prepare_loop_mode(int lds_tables);
// One launch of the step loop (gxt_loop.h) on a.groups workgroups.  e0, e1 (may
// be null) take the kernel's start and end.
template <class R>
hipError_t launch_loop(const LoopArgs &a, hipStream_t st, hipEvent_t e0, hipEvent_t e1);
// The launch of one transport mode (each mode is compiled in a unit of its own).
template <class R, int kMode>
hipError_t launch_loop_mode(const LoopArgs &a, hipStream_t st, hipEvent_t e0, hipEvent_t e1);
// Primaries or tracks in flight (gxt_primary, gxt_track) of up to kInjectRanges
// jobs, injected together: entry i, first[r] <= i < first[r + 1], is src[r][i -
// first[r]] and its event slot .event + base[r].
constexpr int kInjectRanges = 64;
struct InjectArgs {
  const void *src[kInjectRanges];
  int first[kInjectRanges + 1];
  int base[kInjectRanges];
  int nr;
  int n[2];  // of the entries, photons and e-/e+
  int fill;  // tracks per page, if there are free pages enough
};
template <class R, class In>
hipError_t launch_inject(const LoopArgs &a, const InjectArgs &in, hipStream_t st);
// Clears the rings and makes all pages free.
hipError_t launch_pages_init(const LoopArgs &a, hipStream_t st);

// What the host reads of the device's state after a launch.
struct Snapshot {
  long long live;    // tracks in pages
  long long peak;    // Rings::peak
  long long iters;   // Rings::iters
  unsigned int ran;  // workgroups that ran a task in the last launch
  int overflow;
};
// The host's snapshot, into pinned host memory (device addresses out,
// out_live, out_peak): each event's live tracks and the most that were live at
// once (kLivePeak, which it brings up to date), e < n.
hipError_t launch_snapshot(const Counters *cnt, int *ev_live, int n, Snapshot *out, int *out_live, int *out_peak,
                           hipStream_t st);
hipError_t launch_rng_init(const DevParams *P, const uint32_t *seed, const uint64_t *idx, int n, uint32_t *out,
                           hipStream_t st);
hipError_t launch_rng_draw(uint32_t *states, int n, int k, double *out, hipStream_t st);
hipError_t launch_table_value(const DevParams *P, int precision, int slot, int table, const double *x, double *out,
                              int n, hipStream_t st);
hipError_t launch_macro_xs(const DevParams *P, int precision, int slot, int species, int proc, const double *e,
                           double *out, int n, hipStream_t st);
hipError_t launch_sample(const DevParams *P, int precision, int slot, int model, const SampleArgs &s, hipStream_t st);
hipError_t launch_helix(const double B[3], int precision, const double *charge, const double *mom, const double *step,
                        double *pos, double *dir, int n, hipStream_t st);
// Straight-line navigation of the analytic geometry (gxt_slab_distance);
// pstep and boundary may be null.
hipError_t launch_slab_distance(const DevParams *P, const double *pos, const double *dir, const double *pstep,
                                int32_t *vol, double *snext, int32_t *next, double *safety, int32_t *boundary, int n,
                                hipStream_t st);
hipError_t launch_field_value(const DevField &F, const double *pos, double *b, int n, hipStream_t st);
hipError_t launch_field_step(const DevField &F, int precision, const double *charge, const double *mom,
                             const double *step, double *pos, double *dir, double *err, int n, hipStream_t st);

// Volume-tree queries over n points (pos, dir: [3n] SoA) in the tree g (the
// step kernels check touchable[i] against g.ntouch).  lds_bytes > 0: the
// tree is one allocation of lds_bytes (a multiple of 16, at most 48 KiB)
// starting at g.node, which each workgroup copies into LDS; 0: it is read in
// place.
hipError_t launch_nav_locate(const DevNav &g, int lds_bytes, const double *pos, const double *dir, int32_t *out,
                             int n, hipStream_t st);
hipError_t launch_nav_step(const DevNav &g, int lds_bytes, const int32_t *touchable, const double *pos,
                           const double *dir, double *snext, int32_t *next, double *safety, int n, hipStream_t st);
hipError_t launch_nav_find_next_boundary(const DevNav &g, int lds_bytes, const int32_t *touchable, const double *pos,
                                        const double *dir, const double *pstep, double *snext, int32_t *next,
                                        double *safety, int32_t *boundary, int n, hipStream_t st);

}  // namespace gxt
