// gxt_types.h -- host/device layout of the physics data, geometry, track
// pool and counters of the MI355X step loop.
#pragma once

#include <stdint.h>

#include "../../include/gxt.h"

namespace gxt {

constexpr int kMaxVol = 128;      // volumes (calorimeter: 2 per layer)
constexpr int kMaxElem = 3;       // elements per material
constexpr int kMaxSlots = 2;      // materials per setup
constexpr int kMaxZBins = 64;
constexpr int kMaxRBins = 64;
constexpr int kNumQueues = 9;     // (species, process) interaction queues + positrons at rest
constexpr int kQueueAtRest = 8;
constexpr int kSpecBins = 64;     // secondary spectrum bins per species
constexpr int kInvRangeHints = 256;  // search-hint bins per inverse-range vector
constexpr int kMaxShells = 128;   // shell binding energies over the elements of the slots
// Statistics counters are spread over kStripes rows (workgroup b adds to row
// b % kStripes).
constexpr int kStripes = 16;
// Words per row of the substream jump table: the first rows of both components'
// matrices; 8 bytes of the index x 256 values x 24 bytes = 48 KB.
constexpr int kJumpRow = 6;
constexpr int kJumpWords = 8 * 256 * kJumpRow;

// One node of a physics vector: abscissa (energy or range), value, second
// derivative, 1 / (distance to the next node); a spline lookup reads two
// adjacent nodes, 64 B (32 B in FP32).
struct alignas(32) Node64 {
  double x, y, d2, idx;
};
struct alignas(16) Node32 {
  float x, y, d2, idx;
};

// What a step-loop launch stages in LDS: nothing; the photon tables, the jump
// table, the Sandia rows and the search hints; those and the e-/e+ tables.
enum { kLdsNone = 0, kLdsPhotons, kLdsAll };

// One physics vector inside the node array (nodes [off, off+n)).
struct DevTable {
  int off;
  int n;
  int loff;  // first node in the LDS copy of its kernel's tables (DevParams::lds_*), -1: none
  int lpad;
  double dl, base;  // log-binning: bin = log(E)/dl - base
  double x0, xn, y0, yn;  // first and last node (the clamps of a lookup)
  double idl;             // 1 / dl
  float dlf, basef, idlf;
  float fpad;
  float x0f, xnf, y0f, ynf;
  // search hints of a non-log vector (inverse range): hints[hint + k] is the
  // last node below x[0] 2^(k / hscale), k < nhint (hint < 0: none)
  int hint, nhint;
  float hlog0, hscale;  // log2 x[0]; hint bins per octave
};

struct DevElement {
  int Z;
  int sb;          // offset of the element's Seltzer-Berger grid (x[32], y[57], v[57][32])
  int sandia;      // offset of its Sandia rows (5 doubles each)
  int nint;        // number of Sandia intervals
  int shell;       // offset of its shell binding energies (MeV)
  int nshell;
  double natoms;   // atoms per mm3
  double zoa;      // Sandia Z/A ratio
  double wbrem;    // n Z (Z+1): element weight for pair and brems
};

struct DevMaterial {
  double ne;          // electrons per mm3
  double migdal;      // k_p^2 = migdal * E_tot^2
  double cut_gamma;   // gamma production threshold (MeV)
  double cut_e;       // electron production threshold (MeV)
  double cut_length;  // production cut (mm)
  double compt_split; // Lambda.compt upper edge: above it LambdaPrim.compt / E
  double phot_emin;   // LambdaPrim.phot lower edge: below it Sandia
  int nel;
  int pad;
  DevElement el[kMaxElem];
  DevTable tab[GXT_NTAB];
  // Sandia photo-absorption by merged interval: the sx_n breakpoints
  // sx[sx_b .. sx_b + sx_n) (keV, ascending) are every element's interval
  // edges but its first; interval j (sx[sx_b + j - 1] <= E < sx[sx_b + j])
  // holds each element's coefficients a1..a4 at sx[sx_c + (j * nel + i) * 4].
  // A search starts at hints[sx_hint + k], the interval of the lower end of
  // log2 bin k (sx_hscale bins per octave from sx_hlog0).
  int sx_b, sx_c, sx_n, sx_hint, sx_nhint;
  float sx_hlog0, sx_hscale;
};

struct NavNode;
struct NavGrid;

// A volume tree on the device.
struct DevNav {
  const NavNode *node;
  const NavGrid *grid;   // per volume
  const int32_t *idx;
  int ntouch;
  int pad;
};

// The transport geometry.  Slab form (tree = 0): nvol volumes between the
// planes z[v] and z[v + 1], |x| <= hx, |y| <= hy; a track's volume is v.
// Tree form (tree = 1): a track's volume is a touchable of nav, and
// cell[touchable] its tally cell; cells [0, nvol - 1) are the touchables
// with a material, in touchable order, and cell nvol - 1 is vacuum (slot -1).
// slot[] and visible[] are per cell (in the slab form cells are volumes).
struct DevGeometry {
  int nvol;
  int tree;
  double hx, hy;
  double z[kMaxVol + 1];
  int slot[kMaxVol];
  int visible[kMaxVol];
  const int32_t *cell;
  DevNav nav;
};

// Magnetic field seen by the general (non-uniform or Runge-Kutta)
// propagation: a cylindrical (r, z) map, or the uniform field b.
struct DevField {
  const double *v;         // (Br, Bphi, Bz) in tesla at (ir * nz + iz) * 3; null: uniform b
  int nr, nz;
  double r0, z0, dr, dz;   // first node and spacing (mm)
  double idr, idz;         // 1 / spacing
  double origin[3];        // setup origin in the map frame (mm)
  double b[3];             // uniform field (tesla) when v is null
  int stepper;             // GXT_STEPPER_*
  int general;             // e-/e+ take the general propagation (a map, or RK45)
};

// One placed box of a volume tree (a touchable), in global coordinates: boxes
// are placed by translations only.  Touchables are numbered breadth-first, so
// the daughters of a touchable are [first, first + count).
struct alignas(16) NavBox {
  double c[3];     // centre (mm)
  double h[3];     // half-lengths (mm)
  int32_t parent;  // -1 for the world
  int32_t first;
  int32_t count;
  int32_t volume;  // index into the caller's volume array
};
struct alignas(64) NavNode : NavBox {};

// Daughter index of a volume with many daughters: nb bins of its extent
// along axis ax (mother frame, bin = (x + h) inv); the daughters that may hold
// a point of bin b are ordinals idx[idx[off + b] .. idx[off + b + 1]), in
// ascending order.  nb = 0: no index (the daughters are scanned).
struct NavGrid {
  double inv;
  int32_t ax, nb, off, pad;
};

// Bin of mother-frame coordinate x in a daughter index (clamped; NaN -> 0).
// The same function places the daughters' extents when the index is built:
// it is monotone in x, so a point inside a daughter's extent falls in one of
// the daughter's bins.
__host__ __device__ inline int nav_bin(double x, double h, double inv, int nb) {
  const double u = (x + h) * inv;
  if (!(u >= 0.0)) return 0;
  if (u >= (double)nb) return nb - 1;
  return (int)u;
}

// Most points per call of the entry points that take [3n] structure-of-arrays
// (their kernels index them with 32-bit k n + i).
constexpr int kMaxSoaPoints = 1 << 29;

// Largest tree (nodes, grids and index) the navigation kernels copy into LDS.
constexpr int kNavLdsMax = 48 * 1024;

// Everything a kernel needs besides the pool: lives in one device buffer.
struct DevParams {
  DevMaterial mat[kMaxSlots];
  DevGeometry geo;
  double B[3], ub[3];  // uniform field and its unit vector
  double bmag;
  DevField field;
  double tracking_cut;
  double zbin, rbin;
  int nz, nr;
  int max_steps;
  int trace_events;   // events [0, trace_events) are traced
  int trace_steps;
  int msc;            // e-/e+ multiple scattering
  uint32_t seed[6];
  int nsandia, nshells;     // doubles in the Sandia and shell arrays
  int nsx, nhints;          // entries of sx and hints, both to whole 16-byte words
  const uint32_t *jump8;    // first row of A_c^(d 2^(76+8k)) mod m_c at (k * 256 + d) * kJumpRow + 3 c
  const Node64 *nd;             // physics-vector nodes, FP64
  const Node32 *nf;             // FP32 mirror
  const double *sbd;            // Seltzer-Berger grids, FP64
  const float *sbf;             // FP32 mirror
  const double *sandia;         // Sandia rows (edge keV, a1..a4)
  const double *sx;             // merged Sandia breakpoints and coefficients (DevMaterial::sx_*)
  const int *hints;             // search hints of the inverse-range vectors
  // the Seltzer-Berger grid every element shares: reduced photon energy k / T
  // (32 nodes) and ln(T / MeV) (57 nodes), FP64 and FP32; the step loop
  // reads them from its LDS copy of DevParams
  double sbx[32], sby[57];
  float sbxf[32], sbyf[57];
  // shell binding energies (MeV) of every element of the slots, falling, the
  // innermost first (DevElement::shell, nshell), read where DevParams is
  double shell_e[kMaxShells];
  // LDS copies of the physics vectors a transport kernel reads: layout 0 the
  // photon tables (GXT_TAB_LAMBDA_COMPT .. GXT_TAB_LAMBDAPRIM_PHOT), layout 1
  // the e-/e+ tables (GXT_TAB_LAMBDA_BREM_EM .. GXT_TAB_INVRANGE_EP), one
  // contiguous node span per material slot: nodes [lds_src[l][s], +
  // lds_cnt[l][s]) of the node array, in slot order
  int lds_src[2][kMaxSlots];
  int lds_cnt[2][kMaxSlots];
  int lds_nodes[2];
};

// ------------------------------------------------------------------ track pages
// Live tracks sit in pages of 64, one structure-of-arrays block per page, so a
// wave loads or fills a page with contiguous accesses.  Every page holds
// tracks that wait for the same task: type 0 photon transport, 1 e-/e+
// transport, 2 + q the interaction queue q.  R is the precision of the
// physics state (double, or float in the precision form); positions and
// tallies stay FP64.
constexpr int kPageTracks = 64;
constexpr int kTypes = 2 + kNumQueues;
enum PageF64 { kPx = 0, kPy, kPz,
               kPtedep, kPuid,  // tracing only: step deposit, substream index
               kPageF64 };
enum PageR { kPdx = 0, kPdy, kPdz, kPe, kPnil0, kPnil1, kPnil2, kPageR };
enum PageU32 { kPrng = 0, kPevent = 6, kPmeta, kPnsteps, kPageU32 };  // meta: volume | species << 16
template <class R>
__host__ __device__ constexpr int page_bytes() {
  return kPageTracks * (kPageF64 * 8 + kPageR * (int)sizeof(R) + kPageU32 * 4);
}

// A page with tracks, as the step loop's list holds it between launches.
__host__ __device__ constexpr uint32_t page_entry(uint32_t page, int type, int count) {
  return page << 10 | (uint32_t)type << 6 | (uint32_t)(count - 1);
}
constexpr uint32_t kMaxPages = 1u << 22;

// The step loop's page lists in device memory, two rings of `mask + 1` entries
// (at least twice the pages, so that what a launch writes never reaches what it
// has still to read): list (page_entry of the pages with tracks, [lhead,
// ltail)) and free pages ([fhead, ftail)).  A launch of the loop takes entries
// from the heads and writes behind the tails (counted by lpush, fpush); its
// last workgroup to end moves the heads and tails, so that a launch reads only
// what was written before it began.  Each workgroup's entries are contiguous
// within [seg_lo, seg_hi), what the last launch wrote: PageSeg of the
// workgroup in the array of `parity`; the entries before (left over) and
// behind (injected) belong to none.
struct alignas(128) Rings {
  unsigned long long lhead, ltail, fhead, ftail;
  unsigned long long lpush, fpush;
  unsigned int done;        // workgroups of the launch that have ended
  unsigned int ran, ran_last;  // workgroups that ran a task in this launch, in the last one
  int parity;
  unsigned long long seg_lo, seg_hi;
  long long live;           // tracks in pages when the last launch ended
  long long net, grow;      // tracks made less those ended in this launch; sum of the workgroups' largest growths
  long long peak;           // most tracks that may have been live at once
  long long iters;          // transports of any track so far, at most
  int launch_iters;         // the same of this launch
  unsigned int inj[2];      // photons, e-/e+ placed by an injection in progress
  unsigned int inj_done;    // its workgroups that have ended
};
struct PageSeg {
  uint32_t first, count;    // entries [seg_lo + first, + count)
};
constexpr int kMaxGroups = 512;
// Free pages per workgroup at its start, at least (one workgroup: what there is):
// an open page for each type and what 12 running tasks may need.
constexpr int kMinFree = 96;

enum StatKind { kStatSteps = 0, kStatStepsCharged, kStatKilled, kStatInteractions, kStatCreated, kStatLoaded0,
                kStatLoaded1, kStatInteractions0, kStatCreated0,
                // wave time (100 MHz ticks) in the loop's parts, with profiling on
                kStatTimeN, kStatTimeC, kStatTimeIN, kStatTimeIC, kStatTimeD, kNumStats };
struct alignas(256) Counters {
  Rings rings;
  unsigned long long stat[kStripes][16];  // 128 B per stripe
  int32_t overflow;        // the pages ran out: the tracks that found none are lost
  int32_t pad[31];
  unsigned long long trace_n; // trace records written
  __host__ __device__ unsigned long long total(int k) const {
    unsigned long long t = 0;
    for (int s = 0; s < kStripes; ++s) t += stat[s][k];
    return t;
  }
};

// Live tracks of event e: kLive.. at ev_live[e * kLiveStride + ..], one 128-byte
// line per event, so the atomics of one event's tracks never queue behind another
// event's.  Its live count exists only when a launch ends, and an event may grow,
// shrink and end in between; so each workgroup gives, beside the change, the
// largest growth that it saw, and the sum of those on top of the count before
// bounds what was live at once (exact for an event in one workgroup).  The growths
// cost 10,000 e- of 10 GeV 2 % in FP32 (33.8 -> 34.5 ms), 0.3 % in FP64.
constexpr int kLiveStride = 32;
enum { kLiveNow = 0,
       kLiveGrow,    // sum of the growths since the last snapshot
       kLiveBefore,  // count at the last snapshot
       kLivePeak };  // largest bound until the last snapshot

// Per-event tallies on the device (FP64, atomics), one or more whole 128-byte
// lines per event for the same reason.
struct alignas(128) DevEvent {
  double edep, visible, leak, clen;
  unsigned long long nsec[3];
  unsigned long long nsteps, npairs, nannihil;
  int pad0, pad1;
};

}  // namespace gxt
