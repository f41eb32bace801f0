// gxt_step.h -- what the kernels of the step loop share: wave helpers, the
// loop's histograms, track page I/O, deposits, GPIL.
#pragma once

#include <hip/hip_runtime.h>

#include "gxt_device.h"
#include "gxt_kernels.h"

namespace gxt {

// ------------------------------------------------------------------ wave helpers
__device__ __forceinline__ int lane() { return (int)__lane_id(); }

// Scans by DPP moves: VALU instructions, where a shuffle is an LDS access of
// over 100 cycles in a chain of six.  All 64 lanes must be active.
template <int kCtrl, int kRows>
__device__ __forceinline__ int dpp_or(int other, int v) {
  return __builtin_amdgcn_update_dpp(other, v, kCtrl, kRows, 0xf, false);
}

// Inclusive sum within each row of 16 lanes.
__device__ __forceinline__ int row_incl_scan(int v) {
  v += dpp_or<0x111, 0xf>(0, v);  // row_shr 1, 2, 4, 8
  v += dpp_or<0x112, 0xf>(0, v);
  v += dpp_or<0x114, 0xf>(0, v);
  v += dpp_or<0x118, 0xf>(0, v);
  return v;
}

// Largest of lanes 0 .. 15, in every lane.
__device__ __forceinline__ int row0_max(int v) {
  v = max(v, dpp_or<0x111, 0xf>(v, v));
  v = max(v, dpp_or<0x112, 0xf>(v, v));
  v = max(v, dpp_or<0x114, 0xf>(v, v));
  v = max(v, dpp_or<0x118, 0xf>(v, v));
  return __builtin_amdgcn_readlane(v, 15);
}

__device__ __forceinline__ int wave_incl_scan(int v) {
  v = row_incl_scan(v);
  v += dpp_or<0x142, 0xa>(0, v);  // row_bcast 15: the sum of rows 0, 2 to rows 1, 3
  v += dpp_or<0x143, 0xc>(0, v);  // row_bcast 31: the sum of rows 0, 1 to rows 2, 3
  return v;
}

// ------------------------------------------------------------------ tallies
// Row of the calling workgroup: z bins, r bins, volumes; then its spectrum row.
__device__ __forceinline__ double *tally_row(const TallyRows &r) {
  return r.bins + (int64_t)(blockIdx.x % r.nrows) * r.stride;
}

// Histograms of the workgroup in LDS.  Deposits of a wave's lanes often share a
// bin (a homogeneous block has one volume; the shower core fills the first
// radial bins), which serialises global atomics in L2; LDS atomics resolve
// those conflicts, and at the end of the launch the workgroup adds its
// non-zero bins to its row with no-return atomics.
struct Hist {
  double z[kMaxZBins];
  double r[kMaxRBins];
  double v[kMaxVol];
  unsigned int spec[3 * kSpecBins];
};

// By all threads of the workgroup, with a barrier after clearing and before
// flushing.
__device__ __forceinline__ void hist_clear(Hist &h) {
  for (int i = (int)threadIdx.x; i < kMaxZBins; i += (int)blockDim.x) h.z[i] = 0.0;
  for (int i = (int)threadIdx.x; i < kMaxRBins; i += (int)blockDim.x) h.r[i] = 0.0;
  for (int i = (int)threadIdx.x; i < kMaxVol; i += (int)blockDim.x) h.v[i] = 0.0;
  for (int i = (int)threadIdx.x; i < 3 * kSpecBins; i += (int)blockDim.x) h.spec[i] = 0u;
}

__device__ __forceinline__ void hist_flush(const TallyRows &rows, const DevParams *P, const Hist &h) {
  const int nz = P->nz, nr = P->nr, nv = P->geo.nvol;
  double *row = tally_row(rows);
  if (nv == 1 && threadIdx.x < 64) {
    // the one volume's deposit: that of all z bins (Dep::flush)
    static_assert(kMaxZBins == 64, "a z bin per lane");
    double s = (int)threadIdx.x < nz ? h.z[threadIdx.x] : 0.0;
    for (int d = 32; d > 0; d >>= 1) s += __shfl_xor(s, d, 64);
    if (threadIdx.x == 0 && s != 0.0) unsafeAtomicAdd(&row[nz + nr], s);
  }
  for (int i = (int)threadIdx.x; i < nz + nr + (nv == 1 ? 0 : nv); i += (int)blockDim.x) {
    const double v = i < nz ? h.z[i] : (i < nz + nr ? h.r[i - nz] : h.v[i - nz - nr]);
    if (v != 0.0) unsafeAtomicAdd(&row[i], v);
  }
  unsigned long long *srow = rows.spec + (int64_t)(blockIdx.x % rows.nrows) * 3 * kSpecBins;
  for (int i = (int)threadIdx.x; i < 3 * kSpecBins; i += (int)blockDim.x)
    if (h.spec[i]) atomicAdd(&srow[i], (unsigned long long)h.spec[i]);
}

__device__ __forceinline__ void spectrum(Hist &h, int species, double e) {
  const int b = (int)floor((m_log10(e) + 3.0) * 8.0);
  if (b >= 0 && b < kSpecBins) atomicAdd(&h.spec[species * kSpecBins + b], 1u);
}

// ------------------------------------------------------------------ pool I/O
// The three interaction lengths are named members so that, with the process
// loops unrolled, every access is static and stays in registers.
template <class R>
struct TrackRegs {
  double pos[3];
  R dir[3];
  R e;
  R nil0, nil1, nil2;
  Rng rng;
  int event, vol, species, nsteps;
  uint64_t uid;
  // value selects (a store through a selected member address would force the
  // whole struct out of registers)
  __device__ __forceinline__ void set_nil(int p, R v) {
    nil0 = p == 0 ? v : nil0;
    nil1 = p == 1 ? v : nil1;
    nil2 = p == 2 ? v : nil2;
  }
};

// Fields of the track in slot `slot` of a page, slot folded into the pointers.
template <class R>
struct PageSlot {
  char *d, *r, *u;
  __device__ __forceinline__ PageSlot(char *page, int slot)
      : d(page + slot * 8),
        r(page + kPageTracks * kPageF64 * 8 + slot * (int)sizeof(R)),
        u(page + kPageTracks * (kPageF64 * 8 + kPageR * (int)sizeof(R)) + slot * 4) {}
  __device__ __forceinline__ double &f64(int k) const {
    return *reinterpret_cast<double *>(d + k * kPageTracks * 8);
  }
  __device__ __forceinline__ uint64_t &u64(int k) const {
    return *reinterpret_cast<uint64_t *>(d + k * kPageTracks * 8);
  }
  __device__ __forceinline__ R &f(int k) const {
    return *reinterpret_cast<R *>(r + k * kPageTracks * (int)sizeof(R));
  }
  __device__ __forceinline__ uint32_t &u32(int k) const {
    return *reinterpret_cast<uint32_t *>(u + k * kPageTracks * 4);
  }
};

template <class R>
__device__ __forceinline__ void load_track(const PageSlot<R> &p, TrackRegs<R> &t, bool trace) {
  t.pos[0] = p.f64(kPx);
  t.pos[1] = p.f64(kPy);
  t.pos[2] = p.f64(kPz);
  t.dir[0] = p.f(kPdx);
  t.dir[1] = p.f(kPdy);
  t.dir[2] = p.f(kPdz);
  t.e = p.f(kPe);
  t.nil0 = p.f(kPnil0);
  t.nil1 = p.f(kPnil1);
  t.nil2 = p.f(kPnil2);
#pragma unroll
  for (int k = 0; k < 6; ++k) t.rng.s[k] = p.u32(kPrng + k);
  t.event = (int)p.u32(kPevent);
  const int meta = (int)p.u32(kPmeta);
  t.vol = meta & 0xffff;
  t.species = meta >> 16;
  t.nsteps = (int)p.u32(kPnsteps);
  t.uid = trace ? p.u64(kPuid) : 0;
}

template <class R>
__device__ __forceinline__ void store_track(const PageSlot<R> &p, const TrackRegs<R> &t, bool trace) {
  p.f64(kPx) = t.pos[0];
  p.f64(kPy) = t.pos[1];
  p.f64(kPz) = t.pos[2];
  p.f(kPdx) = t.dir[0];
  p.f(kPdy) = t.dir[1];
  p.f(kPdz) = t.dir[2];
  p.f(kPe) = t.e;
  p.f(kPnil0) = t.nil0;
  p.f(kPnil1) = t.nil1;
  p.f(kPnil2) = t.nil2;
#pragma unroll
  for (int k = 0; k < 6; ++k) p.u32(kPrng + k) = t.rng.s[k];
  p.u32(kPevent) = (uint32_t)t.event;
  p.u32(kPmeta) = (uint32_t)(t.vol | (t.species << 16));
  p.u32(kPnsteps) = (uint32_t)t.nsteps;
  if (trace) p.u64(kPuid) = t.uid;
}

// A track created by an interaction or an annihilation at rest, at the
// position, volume and event of its parent, with the RNG state rng of its
// substream uid.
template <class R>
__device__ __forceinline__ void store_new(const PageSlot<R> &p, const TrackRegs<R> &par, int species, R e, R d0,
                                          R d1, R d2, uint64_t uid, const uint32_t rng[6], bool trace) {
  p.f64(kPx) = par.pos[0];
  p.f64(kPy) = par.pos[1];
  p.f64(kPz) = par.pos[2];
  p.f(kPdx) = d0;
  p.f(kPdy) = d1;
  p.f(kPdz) = d2;
  p.f(kPe) = e;
  p.f(kPnil0) = R(-1);
  p.f(kPnil1) = R(-1);
  p.f(kPnil2) = R(-1);
#pragma unroll
  for (int k = 0; k < 6; ++k) p.u32(kPrng + k) = rng[k];
  p.u32(kPevent) = (uint32_t)par.event;
  p.u32(kPmeta) = (uint32_t)(par.vol | (species << 16));
  p.u32(kPnsteps) = 0u;
  if (trace) p.u64(kPuid) = uid;
}

// A deposit held back until the kernel's stores, when flush() adds it to the
// workgroup's histograms and EventAdd::deposit to its event.  Every add() of
// one Dep is at the same point.  (Sums kept with the track until its death were
// 24 of the 140 bytes read and written per task: 10,000 e- of 10 GeV took 40.9
// ms in FP64 and 36.6 in FP32, now 40.0 and 35.5; 1,000 in a volume tree 10.0,
// now 9.7.)
struct Dep {
  double e = 0.0, visible = 0.0;
  int iz = 0, ir = 0, vol = 0;
  // v: the track's volume (kGeo as geo_cell)
  template <int kGeo = 2>
  __device__ __forceinline__ void add(const DevParams *P, double de, const double p[3], int v) {
    if (de <= 0.0) return;
    v = geo_cell<kGeo>(P->geo, v);
    if (P->geo.visible[v]) visible += de;
    if (e == 0.0) {
      int z = (int)floor(p[2] / P->zbin);
      iz = z < 0 ? 0 : (z >= P->nz ? P->nz - 1 : z);
      const double r = sqrt(p[0] * p[0] + p[1] * p[1]);
      int rr = (int)(r / P->rbin);
      ir = rr < 0 ? 0 : (rr >= P->nr ? P->nr - 1 : rr);
      vol = v;
    }
    e += de;
  }
  // volumes: more than one.  A single volume takes its sum from the z bins: 64
  // lanes adding to one word were 2 % of the time (10,000 e- of 10 GeV in
  // PbWO4: 39.7 -> 39.0 ms in FP64, 34.7 -> 34.0 in FP32).
  __device__ __forceinline__ void flush(Hist &h, bool volumes) const {
    if (e <= 0.0) return;
    if (volumes) unsafeAtomicAdd(&h.v[vol], e);
    unsafeAtomicAdd(&h.z[iz], e);
    unsafeAtomicAdd(&h.r[ir], e);
  }
};

template <class R>
__device__ __forceinline__ void trace_rec(const LoopArgs &a, const TrackRegs<R> &t, int proc, double edep) {
  if (t.event >= a.P->trace_events || t.nsteps > a.P->trace_steps) return;
  const unsigned long long k = atomicAdd(&a.cnt->trace_n, 1ULL);
  if ((int64_t)k >= a.trace_cap) return;
  double *r = a.trace + 12 * k;
  uint64_t u = t.uid;
  double ub;
  __builtin_memcpy(&ub, &u, 8);
  r[0] = ub;
  r[1] = t.nsteps;
  r[2] = t.species;
  r[3] = proc;
  r[4] = (double)t.e;
  r[5] = t.pos[0];
  r[6] = t.pos[1];
  r[7] = t.pos[2];
  r[8] = (double)t.dir[0];
  r[9] = (double)t.dir[1];
  r[10] = (double)t.dir[2];
  r[11] = edep;
}

// PostStep GPIL of process p (ProxyEmProcess.hpp:122-151): resample the
// number of interaction lengths when exhausted, propose nil / lambda.
template <int p, class R, class NS>
__device__ __forceinline__ void gpil(const DevParams *P, const NS &N, const DevMaterial &m, int species, R e,
                                     R le, R &nil, R &xs, Rng &rng, double &bestd, int &sel) {
  xs = macro_xs(P, N, m, species, p, e, le);
  if (nil <= R(0)) nil = -m_log(rng.template u<R>());
  const double sp = xs > R(0) ? (double)(nil / xs) : kHuge;
  if (sp < bestd) {
    bestd = sp;
    sel = p;
  }
}

}  // namespace gxt
