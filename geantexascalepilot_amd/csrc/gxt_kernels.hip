// gxt_kernels.hip -- gfx950 kernels around the step loop (injection, the host's
// snapshot) and of the component entry points.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "gxt_step.h"

namespace gxt {

constexpr int kBlock = 256;

// ------------------------------------------------------------------ injection
// The state a primary starts from: no interaction lengths yet, the
// substream's initial RNG state, located from its position and direction.
template <class R>
__device__ __forceinline__ void inject_state(const DevParams *P, const LoopArgs &a, const gxt_primary &p,
                                             TrackRegs<R> &t) {
  t.nil0 = t.nil1 = t.nil2 = R(-1);
  t.nsteps = 0;
  t.vol = geo_locate(P->geo, t.pos, p.dir);
  if (t.vol >= 0) substream_state(P->jump8, P->seed, t.uid, t.rng.s);
}

// A track in flight continues from its own interaction lengths, RNG state,
// volume (located when not given) and step count; the event's step tally
// is credited with -nsteps now, so that the track's full count added when it
// dies leaves only the steps taken here (modulo 2^64 arithmetic).
template <class R>
__device__ __forceinline__ void inject_state(const DevParams *P, const LoopArgs &a, const gxt_track &p,
                                             TrackRegs<R> &t) {
  t.nil0 = (R)p.nil[0];
  t.nil1 = (R)p.nil[1];
  t.nil2 = (R)p.nil[2];
  t.nsteps = p.nsteps;
  t.vol = p.volume >= 0 ? p.volume : geo_locate(P->geo, t.pos, p.dir);
  if (t.vol >= 0) {
#pragma unroll
    for (int k = 0; k < 6; ++k) t.rng.s[k] = p.rng[k];
    if (p.nsteps > 0) atomicAdd(&a.ev[t.event].nsteps, (unsigned long long)(-(long long)p.nsteps));
  }
}

// Entries In (gxt_primary or gxt_track) become tracks that wait for their
// transport.  Photons and e-/e+ fill free pages one after the other, `fill`
// tracks each, so that an injection takes no more pages than its tracks need,
// however many jobs they come from (a page or more for each job, and for each
// wave of it and species class, were 98,000 pages for 400 jobs of 256 photons
// where 1,600 do).  Fewer than 64 per page, to spread few tracks over the
// workgroups, only where the free pages leave every workgroup its share.  The
// last workgroup to end puts the pages on the list.
template <class R, class In>
__global__ __launch_bounds__(kBlock) void k_inject(LoopArgs a, InjectArgs in) {
  const DevParams *P = a.P;
  Rings &rg = a.cnt->rings;
  const unsigned long long fhead = rg.fhead, ftail = rg.ftail, ltail = rg.ltail;
  const long long spare = (long long)(ftail - fhead);
  int fill = in.fill;
  if ((in.n[0] + fill - 1) / fill + (in.n[1] + fill - 1) / fill + (long long)a.groups * kMinFree > spare)
    fill = kPageTracks;
  const int np[2] = {(in.n[0] + fill - 1) / fill, (in.n[1] + fill - 1) / fill};  // pages set aside for each class
  const bool trace = P->trace_events > 0;
  const int n = in.n[0] + in.n[1];
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  TrackRegs<R> t;
  int region = -1;
  if (i < n) {
    // the job whose entries hold i
    int lo = 0, hi = in.nr;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (in.first[mid] <= i)
        lo = mid;
      else
        hi = mid;
    }
    const In &p = static_cast<const In *>(in.src[lo])[i - in.first[lo]];
    t.species = p.species;
    t.event = p.event + in.base[lo];
    t.e = (R)p.ekin;
    for (int k = 0; k < 3; ++k) {
      t.pos[k] = p.pos[k];
      t.dir[k] = (R)p.dir[k];
    }
    t.uid = p.substream;
    inject_state(P, a, p, t);
    if (t.vol < 0) {
      unsafeAtomicAdd(&a.ev[t.event].leak, p.ekin);
    } else {
      region = t.species == 0 ? 0 : 1;
      int *live = a.ev_live + (int64_t)t.event * kLiveStride;
      atomicAdd(&live[kLiveNow], 1);
      atomicAdd(&live[kLiveGrow], 1);
    }
  }
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const unsigned long long m = __ballot(region == r);
    if (!m) continue;
    unsigned int at = 0;
    if (lane() == 0) at = atomicAdd(&rg.inj[r], (unsigned int)__popcll(m));
    at = __builtin_amdgcn_readfirstlane(at);
    if (region == r) {
      const unsigned int slot = at + (unsigned int)__popcll(m & ((1ULL << lane()) - 1));
      const long long k = (long long)(slot / (unsigned int)fill) + (r == 0 ? 0 : np[0]);
      if (k < spare) {
        const unsigned int page = a.freel[(uint32_t)(fhead + (unsigned long long)k) & a.mask];
        store_track(PageSlot<R>(a.pages + (int64_t)page * page_bytes<R>(), (int)(slot % (unsigned int)fill)), t, trace);
      } else {
        atomicOr(&a.cnt->overflow, 1);
      }
    }
  }
  __shared__ unsigned int placed[2];
  __shared__ int last;
  __threadfence();
  __syncthreads();
  if (threadIdx.x == 0) {
    last = atomicAdd(&rg.inj_done, 1u) == gridDim.x - 1;
    if (last) {
      placed[0] = atomicExch(&rg.inj[0], 0u);
      placed[1] = atomicExch(&rg.inj[1], 0u);
      rg.inj_done = 0;
    }
  }
  __syncthreads();
  if (!last) return;
  // pages taken: set aside and there; filled: those with tracks (entries
  // outside the world took none)
  const long long take = min((long long)np[0] + np[1], spare);
  const long long u0 = min((long long)((placed[0] + fill - 1) / fill), take);
  const long long u1 = max(min((long long)((placed[1] + fill - 1) / fill), take - np[0]), 0LL);
  for (long long k = threadIdx.x; k < take; k += blockDim.x) {
    const int r = k < np[0] ? 0 : 1;
    const long long v = k - (r == 0 ? 0 : np[0]);
    const uint32_t page = a.freel[(uint32_t)(fhead + (unsigned long long)k) & a.mask];
    if (v < (r == 0 ? u0 : u1))
      a.list[(uint32_t)(ltail + (unsigned long long)(v + (r == 0 ? 0 : u0))) & a.mask] =
          page_entry(page, r, (int)min((long long)placed[r] - v * fill, (long long)fill));
    else
      a.freel[(uint32_t)(ftail + (unsigned long long)(v - (r == 0 ? u0 : u1) + (r == 0 ? 0 : min((long long)np[0], take) - u0))) &
              a.mask] = page;
  }
  if (threadIdx.x == 0) {
    rg.ltail = ltail + (unsigned long long)(u0 + u1);
    rg.fhead = fhead + (unsigned long long)take;
    rg.ftail = ftail + (unsigned long long)(take - u0 - u1);
    rg.live += (long long)placed[0] + placed[1];
    rg.peak = max(rg.peak, rg.live);
  }
}

__global__ __launch_bounds__(kBlock) void k_pages_init(Counters *cnt, uint32_t *freel, PageSeg *seg, int npages,
                                                       int groups) {
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i < npages) freel[i] = (uint32_t)i;
  if (i < 2 * groups) seg[i] = PageSeg{0u, 0u};
  if (i == 0) {
    Rings &r = cnt->rings;
    r.lhead = r.ltail = r.fhead = r.lpush = r.fpush = 0;
    r.ftail = (unsigned long long)npages;
    r.done = r.ran = r.ran_last = 0;
    r.parity = 0;
    r.seg_lo = r.seg_hi = 0;
    r.live = r.net = r.grow = r.peak = 0;
    r.iters = r.launch_iters = 0;
    r.inj[0] = r.inj[1] = r.inj_done = 0;
  }
}

// ------------------------------------------------------------------ component kernels
__global__ void k_rng_init(const DevParams *P, const uint32_t *seed, const uint64_t *idx, int n, uint32_t *out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint32_t v1[3], v2[3];
  jump_substream(P->jump8, seed, idx[i], v1, v2);
  out[6 * i + 0] = v1[0];
  out[6 * i + 1] = v1[1];
  out[6 * i + 2] = v1[2];
  out[6 * i + 3] = v2[0];
  out[6 * i + 4] = v2[1];
  out[6 * i + 5] = v2[2];
}

// Takes any 32-bit words: the recurrence (Rng) holds residues, so a word of 2^32 -
// c or more enters as its residue; given back are the last three values of each
// component, of which those before the draws are the caller's words as they were.
__global__ void k_rng_draw(uint32_t *states, int n, int k, double *out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint32_t in[6];
  Rng r;
  for (int j = 0; j < 6; ++j) r.s[j] = in[j] = states[6 * i + j];
  reduce3<kC1>(r.s);
  reduce3<kC2>(r.s + 3);
  for (int j = 0; j < k; ++j) out[(int64_t)i * k + j] = r.uniform();
  for (int c = 0; c < 6; c += 3) {
    states[6 * i + c] = k == 0 ? in[c] : (k == 1 ? in[c + 1] : (k == 2 ? in[c + 2] : r.s[c]));
    states[6 * i + c + 1] = k == 0 ? in[c + 1] : (k == 1 ? in[c + 2] : r.s[c + 1]);
    states[6 * i + c + 2] = k == 0 ? in[c + 2] : r.s[c + 2];
  }
}

// Straight-line navigation of the analytic geometry for n points (the
// locate, dist_out and safety of the step loop).
__global__ void k_slab_distance(const DevParams *P, const double *pos, const double *dir, const double *pstep,
                                int32_t *vol, double *snext, int32_t *next, double *saf, int32_t *boundary, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const DevGeometry &g = P->geo;
  const double p[3] = {pos[i], pos[n + i], pos[2 * n + i]};
  const double d0 = dir[i], d1 = dir[n + i], d2 = dir[2 * n + i];
  int v = vol[i];
  if (v < 0) v = locate(g, p, d0, d1, d2);
  vol[i] = v;
  if (v < 0) {
    snext[i] = 0.0;
    saf[i] = 0.0;
    next[i] = -1;
    if (boundary) boundary[i] = 1;
    return;
  }
  int face;
  const double s = dist_out(g, v, p, d0, d1, d2, face);
  int nv = -1;
  if (face == 0 || face == 1) {
    nv = face == 1 ? v + 1 : v - 1;
    if (nv >= g.nvol) nv = -1;
  }
  snext[i] = s;
  next[i] = nv;
  saf[i] = safety(g, v, p);
  if (boundary) boundary[i] = pstep ? !(pstep[i] < s) : 1;
}

template <class R>
__global__ void k_table_value(const DevParams *P, int slot, int table, const double *x, double *out, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const Nodes<R> N(P);
  const DevTable &t = P->mat[slot].tab[table];
  const bool inv = table == GXT_TAB_INVRANGE_EM || table == GXT_TAB_INVRANGE_EP;
  out[i] = (double)(inv ? pvec_inv_value(N, t, (R)x[i]) : pvec_value(N, t, (R)x[i]));
}

template <class R>
__global__ void k_macro_xs(const DevParams *P, int slot, int species, int proc, const double *e, double *out, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const Nodes<R> N(P);
  out[i] = (double)macro_xs(P, N, P->mat[slot], species, proc, (R)e[i]);
}

template <class R>
__global__ void k_sample(const DevParams *P, int slot, int model, SampleArgs s) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = s.n;
  if (i >= n) return;
  Rng r;
  for (int j = 0; j < 6; ++j) r.s[j] = s.rng[6 * i + j];
  const R d[3] = {(R)s.dir[i], (R)s.dir[n + i], (R)s.dir[2 * n + i]};
  Interaction<R> o;
  sample_model<R>(P, Nodes<R>(P), P->mat[slot], model, (R)s.ekin[i], d, r, o);
  for (int j = 0; j < 6; ++j) s.rng[6 * i + j] = r.s[j];
  s.out_ekin[i] = (double)o.ekin;
  s.out_dir[i] = (double)o.d[0];
  s.out_dir[n + i] = (double)o.d[1];
  s.out_dir[2 * n + i] = (double)o.d[2];
  s.out_edep[i] = (double)o.edep;
  s.nsec[i] = o.nsec;
  for (int k = 0; k < 2; ++k) {
    const bool has = k < o.nsec;
    s.sec_species[2 * i + k] = has ? o.sec[k].species : -1;
    s.sec_ekin[2 * i + k] = has ? (double)o.sec[k].e : 0.0;
    for (int j = 0; j < 3; ++j) s.sec_dir[6 * i + 3 * k + j] = has ? (double)o.sec[k].d[j] : 0.0;
  }
}

template <class R>
__global__ void k_helix(double b0, double b1, double b2, const double *charge, const double *mom, const double *step,
                        double *pos, double *dir, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double B[3] = {b0, b1, b2};
  const double bmag = sqrt(b0 * b0 + b1 * b1 + b2 * b2);
  double p[3] = {pos[i], pos[n + i], pos[2 * n + i]};
  R d[3] = {(R)dir[i], (R)dir[n + i], (R)dir[2 * n + i]};
  const R ub[3] = {(R)(B[0] / bmag), (R)(B[1] / bmag), (R)(B[2] / bmag)};
  helix_step<R>(ub, bmag, (R)charge[i], (R)mom[i], (R)step[i], p, d);
  for (int k = 0; k < 3; ++k) {
    pos[k * n + i] = p[k];
    dir[k * n + i] = (double)d[k];
  }
}

__global__ void k_field_value(DevField F, const double *pos, double *b, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double B[3];
  map_field(F, pos[i], pos[n + i], pos[2 * n + i], B);
  for (int k = 0; k < 3; ++k) b[k * n + i] = B[k];
}

// Volume-tree queries.  With kLds the workgroup first copies the whole tree
// (nodes, grids and daughter index: lds_bytes, a multiple of 16, read from
// one padded allocation) into LDS, where the node lookups of all its lanes are
// served; the grid then strides over the queries.  Without it the lookups go
// to the tree in device memory.
extern __shared__ uint4 nav_lds[];

template <bool kLds>
__device__ __forceinline__ auto nav_view(const DevNav &g, int lds_bytes) {
  if constexpr (!kLds) {
    return g;
  } else {
    constexpr int w = kNavLdsNode / 16;
    const uint4 *src = reinterpret_cast<const uint4 *>(g.node);
    const int nodes = 4 * g.ntouch;
    for (int k = threadIdx.x; k < lds_bytes / 16; k += blockDim.x)
      nav_lds[k < nodes ? (k >> 2) * w + (k & 3) : k + (w - 4) * g.ntouch] = src[k];
    __syncthreads();
    const char *lds = reinterpret_cast<const char *>(nav_lds);
    const char *rest = lds + (kNavLdsNode - 64) * g.ntouch;
    const char *base = reinterpret_cast<const char *>(g.node);
    return NavLds{lds, reinterpret_cast<const NavGrid *>(rest + (reinterpret_cast<const char *>(g.grid) - base)),
                  reinterpret_cast<const int32_t *>(rest + (reinterpret_cast<const char *>(g.idx) - base)), g.ntouch};
  }
}

template <bool kLds>
__global__ __launch_bounds__(kBlock) void k_nav_locate(DevNav g0, int lds_bytes, const double *pos, const double *dir,
                                                       int32_t *out, int n) {
  const auto g = nav_view<kLds>(g0, lds_bytes);
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const double p[3] = {pos[i], pos[n + i], pos[2 * n + i]};
    const double v[3] = {dir[i], dir[n + i], dir[2 * n + i]};
    out[i] = nav_locate(g, p, v);
  }
}

// A touchable outside [0, g.ntouch) gives next = -2 and NaN distances.
template <bool kLds>
__global__ __launch_bounds__(kBlock) void k_nav_step(DevNav g0, int lds_bytes, const int32_t *touchable,
                                                     const double *pos, const double *dir, double *snext,
                                                     int32_t *next, double *safety, int n) {
  const auto g = nav_view<kLds>(g0, lds_bytes);
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const int t = touchable[i];
    if (t < 0 || t >= g.ntouch) {
      next[i] = -2;
      snext[i] = __builtin_nan("");
      safety[i] = __builtin_nan("");
      continue;
    }
    const double p[3] = {pos[i], pos[n + i], pos[2 * n + i]};
    const double v[3] = {dir[i], dir[n + i], dir[2 * n + i]};
    double s, saf;
    next[i] = nav_step(g, t, p, v, s, saf);
    snext[i] = s;
    safety[i] = saf;
  }
}

// A touchable outside [0, g.ntouch) or a pstep that is negative or not
// finite gives next = -2 and NaN distances.
template <bool kLds>
__global__ __launch_bounds__(kBlock) void k_nav_find_next_boundary(DevNav g0, int lds_bytes, const int32_t *touchable,
                                                                   const double *pos, const double *dir,
                                                                   const double *pstep, double *snext, int32_t *next,
                                                                   double *safety, int32_t *boundary, int n) {
  const auto g = nav_view<kLds>(g0, lds_bytes);
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const int t = touchable[i];
    const double ps = pstep[i];
    if (t < 0 || t >= g.ntouch || !(ps >= 0.0) || !(ps <= 1e300)) {
      next[i] = -2;
      snext[i] = __builtin_nan("");
      safety[i] = __builtin_nan("");
      boundary[i] = 0;
      continue;
    }
    const double p[3] = {pos[i], pos[n + i], pos[2 * n + i]};
    const double v[3] = {dir[i], dir[n + i], dir[2 * n + i]};
    double s, saf;
    int b;
    next[i] = nav_find_next_boundary(g, t, p, v, ps, s, saf, b);
    snext[i] = s;
    safety[i] = saf;
    boundary[i] = b;
  }
}

template <class R>
__global__ void k_field_step(DevField F, const double *charge, const double *mom, const double *step, double *pos,
                             double *dir, double *err, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double p[3] = {pos[i], pos[n + i], pos[2 * n + i]};
  R d[3] = {(R)dir[i], (R)dir[n + i], (R)dir[2 * n + i]};
  double B[3];
  field_at(F, p, B);
  const double bm = sqrt(B[0] * B[0] + B[1] * B[1] + B[2] * B[2]);
  double ex = 0.0, eu = 0.0;
  field_advance<R>(F, B, bm, (R)charge[i], (R)mom[i], step[i], p, d, ex, eu);
  for (int k = 0; k < 3; ++k) {
    pos[k * n + i] = p[k];
    dir[k * n + i] = (double)d[k];
  }
  if (err) {
    err[i] = ex;
    err[n + i] = eu;
  }
}

// ------------------------------------------------------------------ launchers
static inline int grid_for(int n) { return (n + kBlock - 1) / kBlock; }

template <class R>
hipError_t launch_loop(const LoopArgs &a, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
  switch (a.mode) {
    case 0: return launch_loop_mode<R, 0>(a, st, e0, e1);
    case 1: return launch_loop_mode<R, 1>(a, st, e0, e1);
    case 2: return launch_loop_mode<R, 2>(a, st, e0, e1);
    case 3: return launch_loop_mode<R, 3>(a, st, e0, e1);
    default: return launch_loop_mode<R, 4>(a, st, e0, e1);
  }
}
template <class R>
hipError_t prepare_loop(int mode, int lds_tables) {
  switch (mode) {
    case 0: return prepare_loop_mode<R, 0>(lds_tables);
    case 1: return prepare_loop_mode<R, 1>(lds_tables);
    case 2: return prepare_loop_mode<R, 2>(lds_tables);
    case 3: return prepare_loop_mode<R, 3>(lds_tables);
    default: return prepare_loop_mode<R, 4>(lds_tables);
  }
}
template hipError_t prepare_loop<double>(int, int);
template hipError_t prepare_loop<float>(int, int);
template hipError_t launch_loop<double>(const LoopArgs &, hipStream_t, hipEvent_t, hipEvent_t);
template hipError_t launch_loop<float>(const LoopArgs &, hipStream_t, hipEvent_t, hipEvent_t);

template <class R, class In>
hipError_t launch_inject(const LoopArgs &a, const InjectArgs &in, hipStream_t st) {
  const int n = in.n[0] + in.n[1];
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL((k_inject<R, In>), dim3(grid_for(n)), dim3(kBlock), 0, st, a, in);
  return hipGetLastError();
}
template hipError_t launch_inject<double, gxt_primary>(const LoopArgs &, const InjectArgs &, hipStream_t);
template hipError_t launch_inject<float, gxt_primary>(const LoopArgs &, const InjectArgs &, hipStream_t);
template hipError_t launch_inject<double, gxt_track>(const LoopArgs &, const InjectArgs &, hipStream_t);
template hipError_t launch_inject<float, gxt_track>(const LoopArgs &, const InjectArgs &, hipStream_t);

hipError_t launch_pages_init(const LoopArgs &a, hipStream_t st) {
  hipLaunchKernelGGL(k_pages_init, dim3(grid_for(std::max(a.npages, 2 * a.groups))), dim3(kBlock), 0, st, a.cnt,
                     a.freel, a.seg, a.npages, a.groups);
  return hipGetLastError();
}

// The host's snapshot of the step loop, written straight into its pinned
// buffers: the per-event live counts and bounds of their peaks packed, the tracks
// in pages, the overflow flag.
__global__ void k_snapshot(const Counters *cnt, int *ev_live, int n, Snapshot *out, int *out_live, int *out_peak) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e < n) {
    int *L = ev_live + (int64_t)e * kLiveStride;
    const int live = L[kLiveNow], grow = L[kLiveGrow], before = L[kLiveBefore];
    int peak = L[kLivePeak];
    if (grow) {
      peak = max(peak, before + grow);
      L[kLivePeak] = peak;
      L[kLiveGrow] = 0;
    }
    if (live != before) L[kLiveBefore] = live;
    out_live[e] = live;
    out_peak[e] = peak;
  }
  if (e == 0) {
    out->peak = cnt->rings.peak;
    out->iters = cnt->rings.iters;
    out->live = cnt->rings.live;
    out->ran = cnt->rings.ran_last;
    out->overflow = cnt->overflow;
  }
}

hipError_t launch_snapshot(const Counters *cnt, int *ev_live, int n, Snapshot *out, int *out_live, int *out_peak,
                           hipStream_t st) {
  const int grid = n > kBlock ? (n + kBlock - 1) / kBlock : 1;
  hipLaunchKernelGGL(k_snapshot, dim3(grid), dim3(kBlock), 0, st, cnt, ev_live, n, out, out_live, out_peak);
  return hipGetLastError();
}

hipError_t launch_rng_init(const DevParams *P, const uint32_t *seed, const uint64_t *idx, int n, uint32_t *out,
                           hipStream_t st) {
  hipLaunchKernelGGL(k_rng_init, dim3(grid_for(n)), dim3(kBlock), 0, st, P, seed, idx, n, out);
  return hipGetLastError();
}

hipError_t launch_rng_draw(uint32_t *states, int n, int k, double *out, hipStream_t st) {
  hipLaunchKernelGGL(k_rng_draw, dim3(grid_for(n)), dim3(kBlock), 0, st, states, n, k, out);
  return hipGetLastError();
}

hipError_t launch_table_value(const DevParams *P, int precision, int slot, int table, const double *x, double *out,
                              int n, hipStream_t st) {
  if (precision == GXT_FP32)
    hipLaunchKernelGGL(k_table_value<float>, dim3(grid_for(n)), dim3(kBlock), 0, st, P, slot, table, x, out, n);
  else
    hipLaunchKernelGGL(k_table_value<double>, dim3(grid_for(n)), dim3(kBlock), 0, st, P, slot, table, x, out, n);
  return hipGetLastError();
}

hipError_t launch_macro_xs(const DevParams *P, int precision, int slot, int species, int proc, const double *e,
                           double *out, int n, hipStream_t st) {
  if (precision == GXT_FP32)
    hipLaunchKernelGGL(k_macro_xs<float>, dim3(grid_for(n)), dim3(kBlock), 0, st, P, slot, species, proc, e, out, n);
  else
    hipLaunchKernelGGL(k_macro_xs<double>, dim3(grid_for(n)), dim3(kBlock), 0, st, P, slot, species, proc, e, out, n);
  return hipGetLastError();
}

hipError_t launch_sample(const DevParams *P, int precision, int slot, int model, const SampleArgs &s, hipStream_t st) {
  if (precision == GXT_FP32)
    hipLaunchKernelGGL(k_sample<float>, dim3(grid_for(s.n)), dim3(kBlock), 0, st, P, slot, model, s);
  else
    hipLaunchKernelGGL(k_sample<double>, dim3(grid_for(s.n)), dim3(kBlock), 0, st, P, slot, model, s);
  return hipGetLastError();
}

hipError_t launch_helix(const double B[3], int precision, const double *charge, const double *mom, const double *step,
                        double *pos, double *dir, int n, hipStream_t st) {
  if (precision == GXT_FP32)
    hipLaunchKernelGGL(k_helix<float>, dim3(grid_for(n)), dim3(kBlock), 0, st, B[0], B[1], B[2], charge, mom, step,
                       pos, dir, n);
  else
    hipLaunchKernelGGL(k_helix<double>, dim3(grid_for(n)), dim3(kBlock), 0, st, B[0], B[1], B[2], charge, mom, step,
                       pos, dir, n);
  return hipGetLastError();
}

hipError_t launch_slab_distance(const DevParams *P, const double *pos, const double *dir, const double *pstep,
                                int32_t *vol, double *snext, int32_t *next, double *safety, int32_t *boundary, int n,
                                hipStream_t st) {
  hipLaunchKernelGGL(k_slab_distance, dim3(grid_for(n)), dim3(kBlock), 0, st, P, pos, dir, pstep, vol, snext, next,
                     safety, boundary, n);
  return hipGetLastError();
}

hipError_t launch_field_value(const DevField &F, const double *pos, double *b, int n, hipStream_t st) {
  hipLaunchKernelGGL(k_field_value, dim3(grid_for(n)), dim3(kBlock), 0, st, F, pos, b, n);
  return hipGetLastError();
}

// LDS form (trees of at most kNavLdsMax bytes): as many workgroups as the
// CUs hold at once, striding over the queries (one copy of the tree each and
// no partial second round: the step's registers leave 6 per CU, held to 8 they
// spill, 192 us for 81; loading the next query ahead changes nothing);
// otherwise one thread per query.
template <class K>
static dim3 nav_grid(K kernel, int n, int lds_bytes) {
  const int g = grid_for(n);
  if (lds_bytes == 0) return dim3(g);
  int dev = 0, ncu = 0, per = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) !=
                                              hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, kBlock, lds_bytes) != hipSuccess || per < 1 ||
      ncu < 1) {
    (void)hipGetLastError();
    per = 4;
    ncu = 256;
  }
  const int r = per * ncu;
  return dim3(g < r ? g : r);
}

// LDS of a workgroup's copy of a tree of lds_bytes.
static int nav_lds_size(const DevNav &g, int lds_bytes) { return lds_bytes + (kNavLdsNode - 64) * g.ntouch; }

hipError_t launch_nav_locate(const DevNav &g, int lds_bytes, const double *pos, const double *dir, int32_t *out,
                             int n, hipStream_t st) {
  if (lds_bytes > 0)
    hipLaunchKernelGGL(k_nav_locate<true>, nav_grid(k_nav_locate<true>, n, nav_lds_size(g, lds_bytes)), dim3(kBlock),
                       nav_lds_size(g, lds_bytes), st, g, lds_bytes, pos, dir, out, n);
  else
    hipLaunchKernelGGL(k_nav_locate<false>, dim3(grid_for(n)), dim3(kBlock), 0, st, g, 0, pos, dir, out, n);
  return hipGetLastError();
}

hipError_t launch_nav_step(const DevNav &g, int lds_bytes, const int32_t *touchable, const double *pos,
                           const double *dir, double *snext, int32_t *next, double *safety, int n, hipStream_t st) {
  if (lds_bytes > 0)
    hipLaunchKernelGGL(k_nav_step<true>, nav_grid(k_nav_step<true>, n, nav_lds_size(g, lds_bytes)), dim3(kBlock),
                       nav_lds_size(g, lds_bytes), st, g, lds_bytes, touchable, pos, dir, snext, next, safety, n);
  else
    hipLaunchKernelGGL(k_nav_step<false>, dim3(grid_for(n)), dim3(kBlock), 0, st, g, 0, touchable, pos, dir, snext, next,
                       safety, n);
  return hipGetLastError();
}

hipError_t launch_nav_find_next_boundary(const DevNav &g, int lds_bytes, const int32_t *touchable, const double *pos,
                                        const double *dir, const double *pstep, double *snext, int32_t *next,
                                        double *safety, int32_t *boundary, int n, hipStream_t st) {
  if (lds_bytes > 0)
    hipLaunchKernelGGL(k_nav_find_next_boundary<true>,
                       nav_grid(k_nav_find_next_boundary<true>, n, nav_lds_size(g, lds_bytes)), dim3(kBlock),
                       nav_lds_size(g, lds_bytes), st, g, lds_bytes, touchable, pos, dir, pstep, snext, next, safety,
                       boundary, n);
  else
    hipLaunchKernelGGL(k_nav_find_next_boundary<false>, dim3(grid_for(n)), dim3(kBlock), 0, st, g, 0, touchable, pos,
                       dir, pstep, snext, next, safety, boundary, n);
  return hipGetLastError();
}

hipError_t launch_field_step(const DevField &F, int precision, const double *charge, const double *mom,
                             const double *step, double *pos, double *dir, double *err, int n, hipStream_t st) {
  if (precision == GXT_FP32)
    hipLaunchKernelGGL(k_field_step<float>, dim3(grid_for(n)), dim3(kBlock), 0, st, F, charge, mom, step, pos, dir,
                       err, n);
  else
    hipLaunchKernelGGL(k_field_step<double>, dim3(grid_for(n)), dim3(kBlock), 0, st, F, charge, mom, step, pos, dir,
                       err, n);
  return hipGetLastError();
}

}  // namespace gxt
