// gxt_loop.h -- the step loop as one persistent kernel.
//
// A launch runs on one workgroup of 8 or 12 waves per CU.  Each workgroup takes a
// share of the pages with tracks (64 tracks that wait for the same task:
// photon transport, e-/e+ transport, or one of the interactions) and of the
// free pages, and its waves work on their own: a wave takes a page, runs its
// task on the 64 tracks, and writes the tracks that come out, by value, into
// the workgroup's open page of their next task; a page that is full joins the
// ready pages of its task.  What the waves share (ready, open and free pages)
// is in LDS, so a step costs no launch, no wait for the slowest
// wave of a grid, no returning atomic in device memory and no gather: pages
// are read and filled with contiguous accesses.  After its time a workgroup
// hands its pages back; the next launch shares them out again.
//
// Every event's result is independent of the order of the tasks: a track's
// randomness is its own substream, and tallies are sums.
#pragma once

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <climits>

#include "gxt_step.h"

namespace gxt {

constexpr int kLoopWaves = GXT_LOOP_WAVES;  // per workgroup: kLoopWaves / 4 per SIMD
constexpr int kLoopBlock = 64 * kLoopWaves;
constexpr int kLP = 512;    // pages a workgroup holds at once, at most
constexpr int kTake = 256;  // of which with tracks at its start, at most

// Shared state of a workgroup.  A page is known by its local number lp < kLP.
// The waves work on it with LDS atomics and no lock: a lock around each of
// the three accesses of a task cost 12,000 cycles per task, 28 % of the waves'
// time (10 GeV e- in PbWO4, FP64).
//  - Ready pages of a type are a ring: a writer draws a ticket from tail and
//    fills its entry, a reader draws one from head (by compare-and-swap, below
//    tail) and waits for the entry to be filled, which its writer does at once.
//  - Free pages are a stack: a writer draws a ticket upwards from ftop, a reader
//    downwards, and each entry is a mailbox whose writers and readers come in
//    equal number.  `avail` counts the pages that no running task may still
//    need, and a task starts only when its needs are covered, so a ticket
//    always has, or is about to have, its entry.  A page is written again soon
//    after it was read, while it is in the L2 (as a ring, 10,000 e- of 10 GeV
//    took 42.3 ms in FP64, now 40.9; 1,000 in a volume tree 10.7, now 10.0).
//    Ready pages that way, of one type or all, cost 3 to 5 % with many events
//    in flight, and one ring for all types 9 % for 20,011 photons in lead.
//  - A type's open page and its entries given out are one word, changed by
//    compare-and-swap; cnt counts the tracks written into a page.
constexpr uint16_t kNone16 = 0xffffu;
constexpr uint32_t kNoEntry = 0xffffffffu;
// Sched::stop: no free pages for the next task; more tracks than the pool holds;
// no iterations left.
constexpr int kNoPages = 1, kFull = 2, kNoIters = 3;
struct Sched {
  int head[16], tail[16];  // tickets of the ready rings, by type
  int open[16];            // lp << 7 | entries given out (1 .. 63); -1: none
  int until[16];           // tickets below are tasks of this launch; INT_MAX: all, and open pages
  int busy;                // running tasks, + 256 x tasks ended
  int avail;
  int ftop;                // tickets of the free stack
  int stop;                // no further tasks, and why
  int live, top, max_live;  // tracks made less those ended since the launch's start, their largest number, the
                            // number from which the pool is full
  int ran;                 // a task has run
  unsigned int base[2];
  int cnt[kLP];
  uint32_t gpage[kLP];     // local page -> page
  uint16_t rq[kTypes][kLP];  // lp | (tracks - 1) << 9; kNone16: not filled
  uint32_t fs[kLP];        // the free stack: lp; kNoEntry: empty
  int16_t dest[kLoopWaves][kTypes][4];  // pages of a wave's outputs by type, in order of entry / 64
  unsigned long long stat[16];
};
static_assert(kLP == 512, "ready entries hold 9 bits of page");

template <class T>
__device__ __forceinline__ T lds_ld(const T &x) {
  return __hip_atomic_load(&x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
template <class T>
__device__ __forceinline__ void lds_st(T &x, T v) {
  __hip_atomic_store(&x, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ int lds_add(int &x, int v) {
  return __hip_atomic_fetch_add(&x, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ bool lds_cas(int &x, int from, int to) {
  return __hip_atomic_compare_exchange_strong(&x, &from, to, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_WORKGROUP);
}
// The entry of a drawn ticket, once filled; emptied for the ring's next round.
__device__ __forceinline__ int ring_take(uint16_t &e) {
  uint16_t v;
  while ((v = lds_ld(e)) == kNone16) __builtin_amdgcn_s_sleep(1);
  lds_st(e, kNone16);
  return v;
}

// Fills the entry of a drawn ticket, once the reader of the ring's last round
// has emptied it.
__device__ __forceinline__ void ring_put(uint16_t &e, int v) {
  while (lds_ld(e) != kNone16) __builtin_amdgcn_s_sleep(1);
  lds_st(e, (uint16_t)v);
}

// The entry of a drawn ticket, once filled; emptied for the next writer.
__device__ __forceinline__ uint32_t slot_take(uint32_t &e) {
  uint32_t v;
  while ((v = __hip_atomic_exchange(&e, kNoEntry, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) == kNoEntry)
    __builtin_amdgcn_s_sleep(1);
  return v;
}

// Fills the entry of a drawn ticket, once the reader before has emptied it.
__device__ __forceinline__ void slot_put(uint32_t &e, uint32_t v) {
  uint32_t none = kNoEntry;
  while (!__hip_atomic_compare_exchange_strong(&e, &none, v, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_WORKGROUP)) {
    none = kNoEntry;
    __builtin_amdgcn_s_sleep(1);
  }
}

// Pages a task of n tracks may take beside its own, which it frees first:
// photons go on to 4 types, e-/e+ to 7 (at most one new page each); an
// interaction gives up to 3 photons and 3 e-/e+ per track.
__device__ __forceinline__ int task_need(int type, int n) {
  return type == 0 ? 3 : (type == 1 ? 6 : 2 * ((62 + 3 * n) >> 6) - 1);
}

struct Task {
  int type, lp, n;  // type < 0: the wave ends
  int need;
  int live;  // Sched::live with the task's tracks (lane 0, from reserve on)
};

// The next task of a wave: a ready page of the type that has most of them;
// with none ready, the fullest open page that no wave is writing to; with
// neither and no task running, or after the launch's time, none.  While other
// waves run tasks the wave waits for one to end or begin.  (A launch of one
// iteration transports only the pages that it began with, Sched::until.)
__device__ __forceinline__ Task next_task(Sched &S, long long t_end) {
  const int l = lane();
  Task t;
  t.type = -1;
  t.lp = t.n = t.need = t.live = 0;
  for (;;) {
    const bool over = wall_clock64() - t_end >= 0;
    const int busy = __builtin_amdgcn_readfirstlane(lds_ld(S.busy));
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    int key = -1, h = 0, o = -1;
    if (l < kTypes) {
      h = lds_ld(S.head[l]);
      const int until = lds_ld(S.until[l]);
      const int r = min(lds_ld(S.tail[l]), until) - h;
      o = lds_ld(S.open[l]);
      if (r > 0)
        key = (1 << 16) | (r << 4) | l;
      else if (o >= 0 && until == INT_MAX && lds_ld(S.cnt[o >> 7]) == (o & 127))
        key = ((o & 127) << 4) | l;
    }
    key = row0_max(key);
    // (a launch runs a task wherever it can, so that one that ran none is short of pages)
    if (__builtin_amdgcn_readfirstlane(lds_ld(S.stop)) != 0 ||
        (over && __builtin_amdgcn_readfirstlane(lds_ld(S.ran)) != 0))
      return t;
    bool wait = false;
    if (key < 0) {
      if ((busy & 255) == 0 && __builtin_amdgcn_readfirstlane(lds_ld(S.busy)) == busy) return t;
      wait = true;
    } else {
      const int type = key & 15;
      const bool ready = (key >> 16) != 0;
      const int need = task_need(type, ready ? kPageTracks : key >> 4);
      // counted as running before it holds pages, so that a wave that finds none
      // left sees who may give some back
      int had = 0;
      if (l == 0) {
        lds_add(S.busy, 1);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        int v = lds_ld(S.avail);
        while (v >= need && !lds_cas(S.avail, v, v - need)) v = lds_ld(S.avail);
        had = v >= need;
      }
      had = __builtin_amdgcn_readfirstlane(had);
      int ok = 0;
      if (had && l == type) ok = ready ? lds_cas(S.head[type], h, h + 1) : lds_cas(S.open[type], o, -1);
      ok = __builtin_amdgcn_readlane(ok, type);
      if (ok) {
        int v = 0;
        if (l == type) {
          if (ready) {
            v = ring_take(S.rq[type][h & (kLP - 1)]);
          } else {
            // closed: only the tracks given out before are still to come
            while (lds_ld(S.cnt[o >> 7]) != (o & 127)) __builtin_amdgcn_s_sleep(1);
            v = (o >> 7) | ((o & 127) - 1) << 9;
          }
          lds_st(S.ran, 1);
        }
        v = __builtin_amdgcn_readlane(v, type);
        t.type = type;
        t.lp = v & (kLP - 1);
        t.n = (v >> 9) + 1;
        t.need = need;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        return t;
      }
      if (l == 0) {
        if (had) lds_add(S.avail, need);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        lds_add(S.busy, -1);
      }
      if (!had) {
        // short of pages: a running task may free some, otherwise the
        // workgroup hands its pages back
        wait = (busy & 255) != 0;
        if (!wait && __builtin_amdgcn_readfirstlane(lds_ld(S.busy)) == busy) {
          if (l == 0) lds_st(S.stop, kNoPages);
          return t;
        }
      }
    }
    if (wait)
      while (__builtin_amdgcn_readfirstlane(lds_ld(S.busy)) == busy) __builtin_amdgcn_s_sleep(2);
  }
}

// Frees the task's page and gives out entries: lane t < kTypes asks for n
// entries of type t and gets its first entry f; entry e of the type is slot
// e % 64 of page S.dest[wave][t][e / 64].
__device__ __forceinline__ int reserve(Sched &S, Task &task, int n) {
  const int l = lane();
  const int w = (int)(threadIdx.x >> 6);
  // the task's tracks have been read before the page may be written again
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  if (l == 0) slot_put(S.fs[lds_add(S.ftop, 1)], (uint32_t)task.lp);
  int f = 0, o = -1, np = 0, hv = 0;
  int p0 = 0, p1 = 0, p2 = 0;  // new pages in hand (at most 3: n <= 192)
  bool todo = l < kTypes && n > 0;
  do {
    int ex = 0;
    if (todo) {
      o = lds_ld(S.open[l]);
      f = o >= 0 ? o & 127 : 0;
      np = ((f + n + 63) >> 6) - (o >= 0 ? 1 : 0);
      ex = max(np - hv, 0);
    }
    const int incl = row_incl_scan(ex);
    const int total = __builtin_amdgcn_readlane(incl, kTypes - 1);
    if (total > 0) {
      int tk = 0;
      if (l == 0) tk = lds_add(S.ftop, -total) - total;
      tk = __builtin_amdgcn_readfirstlane(tk) + incl - ex;
      for (int j = 0; j < ex; ++j) {
        const int pg = (int)slot_take(S.fs[tk + j]);
        lds_st(S.cnt[pg], 0);
        p0 = hv == 0 ? pg : p0;
        p1 = hv == 1 ? pg : p1;
        p2 = hv == 2 ? pg : p2;
        ++hv;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    }
    if (todo) {
      const int rem = (f + n) & 63;
      const int last = np == 0 ? o >> 7 : (np == 1 ? p0 : (np == 2 ? p1 : p2));
      todo = !lds_cas(S.open[l], o, rem ? last << 7 | rem : -1);
    }
  } while (__any(todo));
  if (l < kTypes && n > 0) {
    int16_t *d = S.dest[w][l];
    const bool have = o >= 0;
    d[0] = (int16_t)(have ? o >> 7 : p0);
    d[1] = (int16_t)(have ? p0 : p1);
    d[2] = (int16_t)(have ? p1 : p2);
    d[3] = (int16_t)p2;
    // a page too many, when the open page changed in between
    if (hv > np) {
      const int pg = np == 0 ? p0 : (np == 1 ? p1 : p2);
      slot_put(S.fs[lds_add(S.ftop, 1)], (uint32_t)pg);
    }
  }
  // what the task did not take of its needs, and its own page; the tracks it
  // gives beyond its own
  const int sum = __builtin_amdgcn_readlane(row_incl_scan(np | n << 8), kTypes - 1);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  if (l == 0) {
    lds_add(S.avail, task.need + 1 - (sum & 255));
    const int net = (sum >> 8) - task.n;
    task.live = lds_add(S.live, net) + net;
  }
  return f;
}

// The wave's outputs are written: lane t's n entries of type t from entry f
// on.  Pages that are now whole become ready; the task has ended.
__device__ __forceinline__ void commit(Sched &S, const Task &task, int f, int n) {
  const int l = lane();
  const int w = (int)(threadIdx.x >> 6);
  // the tracks' stores before the other waves can see the pages
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  if (l < kTypes && n > 0) {
    const int last = (f + n - 1) >> 6;
    for (int j = 0; j <= last; ++j) {
      const int c = min(f + n, 64 * (j + 1)) - max(f, 64 * j);
      const int pg = S.dest[w][l][j];
      if (lds_add(S.cnt[pg], c) + c == kPageTracks)
        ring_put(S.rq[l][lds_add(S.tail[l], 1) & (kLP - 1)], pg | (kPageTracks - 1) << 9);
    }
  }
  if (l == 0) {
    atomicMax(&S.top, task.live);
    if (task.live > S.max_live) lds_st(S.stop, kFull);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  if (l == 0) lds_add(S.busy, 256 - 1);
}

// ------------------------------------------------------------------ event tallies
// The workgroup's sums per event, in LDS, added to the events' records when the
// launch ends.  A workgroup keeps its pages from launch to launch, so its
// tracks belong to few events; one that finds no place goes to its record
// directly.  (With every death, secondary and live count an atomic in device
// memory, 0.99e9 of them bounded the loop: 10,000 e- of 10 GeV in FP32 took
// 55.5 ms with and 39.7 ms without them.)
// The slots (LoopArgs::ev_slots, a power of two) are what the tables leave of
// the LDS, 128 at least: a burst of requests has more events in flight than a
// batch (with 128 of them 13.7 ms per 100 events, with 512 11.9).
constexpr int kEvProbe = 4;
struct EventSum {
  double edep, visible, leak, clen;
  unsigned long long nsteps;
  int tag;  // event slot, -1: none
  int live;
  unsigned int nsec[3], npairs, nannihil;
  int grow;  // largest `live` in this launch
};
static_assert(sizeof(EventSum) == kEventSumBytes, "LDS of the event sums");
struct EventSums {
  EventSum *slot;
  int n;
};

// Where the event's sums are kept, -1: in its record.
__device__ __forceinline__ int event_slot(const EventSums &E, int event) {
  for (int k = 0; k < kEvProbe; ++k) {
    const int s = (event + k) & (E.n - 1);
    int &tag_s = E.slot[s].tag;
    const int tag = lds_ld(tag_s);
    if (tag == event) return s;
    if (tag < 0 && (lds_cas(tag_s, -1, event) || lds_ld(tag_s) == event)) return s;
  }
  return -1;
}

// A task's contribution to a track's event.
struct EventAdd {
  double edep = 0.0, visible = 0.0, leak = 0.0, clen = 0.0;
  int nsteps = 0, live = 0;
  unsigned int nsec0 = 0, nsec1 = 0, nsec2 = 0, npairs = 0, nannihil = 0;
  __device__ __forceinline__ void deposit(const Dep &d) {
    edep += d.e;
    visible += d.visible;
  }
};

__device__ __forceinline__ void event_add(const LoopArgs &a, const EventSums &S, int event, const EventAdd &c) {
  const int s = event_slot(S, event);
  if (s >= 0) {
    EventSum &E = S.slot[s];
    if (c.edep != 0.0) unsafeAtomicAdd(&E.edep, c.edep);
    if (c.visible != 0.0) unsafeAtomicAdd(&E.visible, c.visible);
    if (c.leak != 0.0) unsafeAtomicAdd(&E.leak, c.leak);
    if (c.clen != 0.0) unsafeAtomicAdd(&E.clen, c.clen);
    if (c.nsteps) atomicAdd(&E.nsteps, (unsigned long long)c.nsteps);
    if (c.live > 0)
      atomicMax(&E.grow, atomicAdd(&E.live, c.live) + c.live);
    else if (c.live)
      atomicAdd(&E.live, c.live);
    if (c.nsec0) atomicAdd(&E.nsec[0], c.nsec0);
    if (c.nsec1) atomicAdd(&E.nsec[1], c.nsec1);
    if (c.nsec2) atomicAdd(&E.nsec[2], c.nsec2);
    if (c.npairs) atomicAdd(&E.npairs, c.npairs);
    if (c.nannihil) atomicAdd(&E.nannihil, c.nannihil);
  } else {
    DevEvent &E = a.ev[event];
    if (c.edep != 0.0) unsafeAtomicAdd(&E.edep, c.edep);
    if (c.visible != 0.0) unsafeAtomicAdd(&E.visible, c.visible);
    if (c.leak != 0.0) unsafeAtomicAdd(&E.leak, c.leak);
    if (c.clen != 0.0) unsafeAtomicAdd(&E.clen, c.clen);
    if (c.nsteps) atomicAdd(&E.nsteps, (unsigned long long)c.nsteps);
    int *live = a.ev_live + (int64_t)event * kLiveStride;
    if (c.live) atomicAdd(&live[kLiveNow], c.live);
    if (c.live > 0) atomicAdd(&live[kLiveGrow], c.live);
    if (c.nsec0) atomicAdd(&E.nsec[0], (unsigned long long)c.nsec0);
    if (c.nsec1) atomicAdd(&E.nsec[1], (unsigned long long)c.nsec1);
    if (c.nsec2) atomicAdd(&E.nsec[2], (unsigned long long)c.nsec2);
    if (c.npairs) atomicAdd(&E.npairs, (unsigned long long)c.npairs);
    if (c.nannihil) atomicAdd(&E.nannihil, (unsigned long long)c.nannihil);
  }
}

__device__ __forceinline__ void events_clear(const EventSums &S) {
  for (int s = (int)threadIdx.x; s < S.n; s += (int)blockDim.x) {
    EventSum &E = S.slot[s];
    E.edep = E.visible = E.leak = E.clen = 0.0;
    E.nsteps = 0;
    E.tag = -1;
    E.live = 0;
    E.nsec[0] = E.nsec[1] = E.nsec[2] = E.npairs = E.nannihil = 0;
    E.grow = 0;
  }
}

// By all threads of the workgroup, with a barrier before.
__device__ __forceinline__ void events_flush(const LoopArgs &a, const EventSums &S) {
  for (int s = (int)threadIdx.x; s < S.n; s += (int)blockDim.x) {
    const EventSum &L = S.slot[s];
    const int event = L.tag;
    if (event < 0) continue;
    DevEvent &E = a.ev[event];
    if (L.edep != 0.0) unsafeAtomicAdd(&E.edep, L.edep);
    if (L.visible != 0.0) unsafeAtomicAdd(&E.visible, L.visible);
    if (L.leak != 0.0) unsafeAtomicAdd(&E.leak, L.leak);
    if (L.clen != 0.0) unsafeAtomicAdd(&E.clen, L.clen);
    if (L.nsteps) atomicAdd(&E.nsteps, L.nsteps);
    int *live = a.ev_live + (int64_t)event * kLiveStride;
    if (L.live) atomicAdd(&live[kLiveNow], L.live);
    if (L.grow) atomicAdd(&live[kLiveGrow], L.grow);
    for (int k = 0; k < 3; ++k)
      if (L.nsec[k]) atomicAdd(&E.nsec[k], (unsigned long long)L.nsec[k]);
    if (L.npairs) atomicAdd(&E.npairs, (unsigned long long)L.npairs);
    if (L.nannihil) atomicAdd(&E.nannihil, (unsigned long long)L.nannihil);
  }
}

template <class R>
__device__ __forceinline__ char *page_at(const LoopArgs &a, const Sched &S, int lp) {
  return a.pages + (int64_t)S.gpage[lp] * page_bytes<R>();
}

// ------------------------------------------------------------------ staging
extern __shared__ uint4 tab_lds[];

// DevParams into LDS in 8-byte words: every thread issues its loads before its
// stores, so the copy costs one memory latency.
constexpr int kParamWords = (int)(sizeof(DevParams) / 8);
constexpr int kParamPer = (kParamWords + kLoopBlock - 1) / kLoopBlock;

__device__ __forceinline__ void stage_params(const DevParams *P, DevParams &sP) {
  static_assert(sizeof(DevParams) % 8 == 0, "DevParams is copied in 8-byte words");
  const unsigned long long *src = reinterpret_cast<const unsigned long long *>(P);
  unsigned long long *dst = reinterpret_cast<unsigned long long *>(&sP);
  unsigned long long v[kParamPer];
#pragma unroll
  for (int j = 0; j < kParamPer; ++j) {
    const int k = j * kLoopBlock + (int)threadIdx.x;
    if (k < kParamWords) v[j] = src[k];
  }
#pragma unroll
  for (int j = 0; j < kParamPer; ++j) {
    const int k = j * kLoopBlock + (int)threadIdx.x;
    if (k < kParamWords) dst[k] = v[j];
  }
}

// n 16-byte words from src to LDS dst by the workgroup's threads, four loads
// in flight per thread before their stores.
__device__ __forceinline__ void copy_words16(uint4 *dst, const uint4 *src, int n) {
  for (int k = (int)threadIdx.x; k < n; k += 4 * kLoopBlock) {
    const int k1 = k + kLoopBlock, k2 = k + 2 * kLoopBlock, k3 = k + 3 * kLoopBlock;
    const uint4 v0 = src[k];
    const uint4 v1 = k1 < n ? src[k1] : v0;
    const uint4 v2 = k2 < n ? src[k2] : v0;
    const uint4 v3 = k3 < n ? src[k3] : v0;
    dst[k] = v0;
    if (k1 < n) dst[k1] = v1;
    if (k2 < n) dst[k2] = v2;
    if (k3 < n) dst[k3] = v3;
  }
}

// The physics vectors of layout `layout` (one node span per material slot)
// into dynamic LDS from 16-byte word dst on; returns the word after them.
template <class R>
__device__ __forceinline__ int stage_tables(const DevParams *P, int layout, int dst) {
  using T = typename NodeType<R>::T;
  constexpr int w = sizeof(T) / sizeof(uint4);
  const uint4 *src = reinterpret_cast<const uint4 *>(NodeType<R>::global(P));
  for (int s = 0; s < kMaxSlots; ++s) {
    const int n16 = P->lds_cnt[layout][s] * w;
    copy_words16(tab_lds + dst, src + (int64_t)P->lds_src[layout][s] * w, n16);
    dst += n16;
  }
  return dst;
}

// ------------------------------------------------------------------ transport task
constexpr int kPhotonSteps = 8;  // most steps of a photon in one task

// The steps of one page of photons (kCharged false) or e-/e+; the species
// class is a compile-time constant so each variant carries only its own code.
// kMode as LoopArgs::mode.
template <class R, bool kCharged, int kMode, class NS>
__device__ __forceinline__ void transport_task(const LoopArgs &a, const DevParams *P, const NS &N, Sched &S,
                                               Hist &wh, const EventSums &ES, Task &task) {
  const bool trace = P->trace_events > 0;
  const R mine = (R)P->tracking_cut;
  constexpr int kG = kMode == 4 ? 1 : 0;  // geo_cell form
  const bool volumes = P->geo.nvol > 1;
  const bool active = lane() < task.n;
  TrackRegs<R> t;
  int q = -1;
  bool survive = false, annihilate = false, dies = false, killed = false, escaped = false;
  int nsub = 0;  // steps taken in this task
  EventAdd add;
  double edep = 0.0;
  if (active) {
    load_track(PageSlot<R>(page_at<R>(a, S, task.lp), lane()), t, trace);
    if (!kCharged) t.species = 0;
    // species as a value the compiler can bound: 0 here, or 1 / 2 there
    const int sp = kCharged ? (t.species == 2 ? 2 : 1) : 0;
    const bool charged = kCharged;
    // A photon that neither interacts nor ends steps on in the task while at
    // least half of the page's do (kPhotonSteps at most); what is left then,
    // and every e-/e+ after its step, goes into a page with others.  Stepping
    // the stragglers of a wave (up to 2 steps in the block, 4 in a
    // calorimeter) ran most passes with few lanes: 10 GeV e-, Runge-Kutta in
    // a solenoid map 19.7 -> 12.5 ms per 100, calorimeter with multiple
    // scattering 20.2 -> 14.2 per 257, 4 T calorimeter 16.9 -> 13.6 per 613,
    // volume tree 13.0 -> 10.6 per 1000; PbWO4 block 43.8 -> 42.6 per 10000.
    // Photons at a quarter or 3/8: the same, e-/e+ at 3/4: msc 14.7, at 1/2:
    // 16.8.
    for (;;) {
      survive = false;
      edep = 0.0;
      Dep dA, dB;  // along-step loss (mid-step, pre-step volume); local deposit at the end point
      // material slot of the track's volume; -1 (tree form only): vacuum, no
      // physics, the track flies to the next boundary
      const int mslot = P->geo.slot[geo_cell<kG>(P->geo, t.vol)];
      const bool vac = kMode == 4 && mslot < 0;
      const DevMaterial &m = P->mat[vac ? 0 : mslot];
      R xs0 = R(0), xs1 = R(0), xs2 = R(0);
      double bestd = kHuge;
      int sel = -1;
      double lam1 = kMscNone;
      // the step's table lookups share log(E) and the e-/e+ range at E
      const R le = m_log(t.e);
      R range = R(0);
      if (!vac) {
        gpil<0>(P, N, m, sp, t.e, le, t.nil0, xs0, t.rng, bestd, sel);
        gpil<1>(P, N, m, sp, t.e, le, t.nil1, xs1, t.rng, bestd, sel);
        if (sp != 1) gpil<2>(P, N, m, sp, t.e, le, t.nil2, xs2, t.rng, bestd, sel);
        if (charged) {
          const double al = (double)along_limit(N, m, sp == 2, t.e, le, mine, range);
          if (al < bestd) {
            bestd = al;
            sel = -1;
          }
        }
        // multiple scattering: its step limit; then the geometric length of the
        // true path is propagated (the step is the true path for interaction
        // lengths and loss); its tables are not among those in LDS
        if constexpr (kMode != 0) {
          if (charged && P->msc) {
            lam1 = msc_lambda1<R>(Nodes<R>(P), m, sp == 2, t.e, le);
            if (lam1 < kMscNone) {
              const double saf = kMode == 4 ? nav_safety(P->geo.nav, nav_box(P->geo.nav, t.vol), t.pos) : safety(P->geo, t.vol, t.pos);
              const double tlim = fmax(fmax(kMscFacRange * fmax((double)range, lam1), kMscFacSafety * saf), kMscTmin);
              if (tlim < bestd) {
                bestd = tlim;
                sel = -1;
              }
            }
          }
        }
      }
      const double pre[3] = {t.pos[0], t.pos[1], t.pos[2]};
      const int prevol = t.vol;
      double step = 0.0;
      int status;
      if constexpr (kMode != 0) {
        const bool msc_on = lam1 < kMscNone;
        const double request = msc_on ? msc_geom(bestd, lam1) : bestd;
        double gstep = 0.0;
        if constexpr (kMode == 4)
          status = propagate_tree<R>(P, sp, t.e, t.pos, t.dir, t.vol, request, gstep);
        else if constexpr (kMode == 2)
          status = propagate_general<R, GXT_STEPPER_HELIX>(P, sp, t.e, t.pos, t.dir, t.vol, request, gstep);
        else if constexpr (kMode == 3)
          status = propagate_general<R, GXT_STEPPER_RK45>(P, sp, t.e, t.pos, t.dir, t.vol, request, gstep);
        else
          status = propagate<R>(P, sp, t.e, t.pos, t.dir, t.vol, request, gstep);
        step = msc_on ? (status == kPhysics ? bestd : msc_true(gstep, lam1, bestd)) : gstep;
      } else {
        status = propagate<R>(P, sp, t.e, t.pos, t.dir, t.vol, bestd, step);
      }
      if (xs0 > R(0)) t.nil0 -= (R)step * xs0;
      if (xs1 > R(0)) t.nil1 -= (R)step * xs1;
      if (xs2 > R(0)) t.nil2 -= (R)step * xs2;
      t.nsteps++;
      if (charged && !vac) {
        add.clen = step;
        R loss = R(0);
        t.e = along_doit(N, m, t.species == 2, t.e, le, range, (R)step, mine, loss);
        const double mid[3] = {0.5 * (pre[0] + t.pos[0]), 0.5 * (pre[1] + t.pos[1]), 0.5 * (pre[2] + t.pos[2])};
        dA.add<kG>(P, (double)loss, mid, prevol);
        edep += (double)loss;
        if constexpr (kMode != 0) {
          if (lam1 < kMscNone && status != kEscaped && t.e > R(0) && step > 0.0)
            msc_deflect<R>(step / lam1, t.dir, t.rng);
        }
      }
      int tproc = status == kPhysics ? sel : (status == kBoundary ? -2 : (status == kEscaped ? -3 : -1));
      if (status == kPhysics && sel < 0) tproc = -1;
      if (status == kEscaped) {
        if (trace) trace_rec(a, t, tproc, edep);
        escaped = true;
        dies = true;
      } else if (t.e <= R(0)) {
        if (trace) trace_rec(a, t, tproc, edep);
        annihilate = t.species == 2;
        dies = !annihilate;
      } else if (status == kPhysics && sel >= 0) {
        t.set_nil(sel, R(-1));
        q = queue_of(t.species, sel);
      } else {
        if (trace) trace_rec(a, t, tproc, edep);
        if (t.e < mine) {
          dB.add<kG>(P, (double)t.e, t.pos, t.vol);
          annihilate = t.species == 2;
          dies = !annihilate;
        } else if (t.nsteps >= P->max_steps) {
          dB.add<kG>(P, (double)t.e, t.pos, t.vol);
          killed = true;
          dies = true;
        } else {
          survive = true;
        }
      }
      // positron at rest: its two photons are made by the interaction task
      if (annihilate) q = kQueueAtRest;
      dA.flush(wh, volumes);
      dB.flush(wh, volumes);
      add.deposit(dA);
      add.deposit(dB);
      ++nsub;
      if (kCharged || !survive || nsub >= kPhotonSteps || 2 * (int)__popcll(__ballot(survive)) < task.n) break;
    }
  }
  // the track's next task, and its entry among the wave's tracks of that type
  const int type = q >= 0 ? 2 + q : (survive ? (kCharged ? 1 : 0) : -1);
  const unsigned long long lt = (1ULL << lane()) - 1;
  int rank = 0, n = 0;
  constexpr int kOut = kCharged ? kNumQueues - 3 + 1 : 3 + 1;
#pragma unroll
  for (int k = 0; k < kOut; ++k) {
    const int ty = k == 0 ? (kCharged ? 1 : 0) : (kCharged ? 4 + k : 1 + k);
    const unsigned long long m = __ballot(type == ty);
    if (type == ty) rank = (int)__popcll(m & lt);
    if (lane() == ty) n = (int)__popcll(m);
  }
  const int f = reserve(S, task, n);
  const int e = __shfl(f, type >= 0 ? type : 0, 64) + rank;
  if (type >= 0) {
    const PageSlot<R> p(page_at<R>(a, S, S.dest[threadIdx.x >> 6][type][e >> 6]), e & 63);
    store_track(p, t, trace);
    if (trace && q >= 0 && q != kQueueAtRest) p.f64(kPtedep) = edep;
  }
  commit(S, task, f, n);
  if (killed) atomicAdd(&S.stat[kStatKilled], 1ULL);
  if (dies) {
    add.nsteps = t.nsteps;
    add.live = -1;
    if (escaped) add.leak = (double)t.e;
  }
  if (active && (dies || add.clen != 0.0 || add.edep != 0.0)) event_add(a, ES, t.event, add);
  const int steps = __builtin_amdgcn_readlane(wave_incl_scan(nsub), 63);
  if (lane() == 0) {
    atomicAdd(&S.stat[kStatSteps], (unsigned long long)steps);
    if (kCharged) atomicAdd(&S.stat[kStatStepsCharged], (unsigned long long)steps);
    atomicAdd(&S.stat[kCharged ? kStatLoaded1 : kStatLoaded0], (unsigned long long)task.n);
  }
}

// ------------------------------------------------------------------ interaction task
// Fate of a secondary: 1 pushed (>= tracking cut), 0 deposited, 2 deposited
// and, a positron, annihilated at rest.
template <class R>
__device__ __forceinline__ int sec_fate(const DevParams *P, const TrackRegs<R> &t, Dep &dp, const Sec<R> &s, R mine,
                                        int &outN, int &outC, int &nannih) {
  if (s.e < mine) {
    dp.add(P, (double)s.e, t.pos, t.vol);
    if (s.species == 2) {
      ++nannih;
      outN += 2;
      return 2;
    }
    return 0;
  }
  if (s.species == 0)
    outN++;
  else
    outC++;
  return 1;
}

// One page of queue q: sample the final states, write the survivors and the
// tracks created, each with its RNG state.
template <class R, class NS>
__device__ __forceinline__ void interact_task(const LoopArgs &a, const DevParams *P, const NS &N,
                                              const uint32_t *jump, Sched &S, Hist &wh, const EventSums &ES,
                                              Task &task, long long &t_derive) {
  const bool trace = P->trace_events > 0;
  const R mine = (R)P->tracking_cut;
  const int q = task.type - 2;
  const bool active = lane() < task.n;
  TrackRegs<R> t;
  Interaction<R> o;
  o.nsec = 0;
  int fate0 = 0, fate1 = 0;
  bool survive = false, prim_rest = false, killed = false, pair = false;
  int outN = 0, outC = 0, nannih = 0;
  Dep dp;  // every deposit of an interaction is at the track's position
  if (active) {
    const PageSlot<R> p(page_at<R>(a, S, task.lp), lane());
    load_track(p, t, trace);
    if (q == kQueueAtRest) {
      // positron stopped by the continuous loss or the tracking cut
      ++nannih;
      prim_rest = true;
      outN = 2;
      t.e = R(0);
    } else {
      // an interacting track is in a material (the tree form's vacuum has no physics)
      const DevMaterial &m = P->mat[max(P->geo.slot[geo_cell<2>(P->geo, t.vol)], 0)];
      if (q < 3)
        sample_neutral<R>(P, N, m, q, t.e, t.dir, t.rng, o);
      else
        sample_charged<R>(P, N, m, q, t.e, t.dir, t.rng, o);
      pair = q == 1 && o.nsec == 2;
      if (q == 7) ++nannih;
      dp.add(P, (double)o.edep, t.pos, t.vol);
      t.e = o.ekin;
      t.dir[0] = o.d[0];
      t.dir[1] = o.d[1];
      t.dir[2] = o.d[2];
      if (trace) trace_rec(a, t, queue_proc(q), p.f64(kPtedep) + (double)o.edep);
      if (o.nsec > 0) fate0 = sec_fate(P, t, dp, o.sec[0], mine, outN, outC, nannih);
      if (o.nsec > 1) fate1 = sec_fate(P, t, dp, o.sec[1], mine, outN, outC, nannih);
    }
    if (t.e > R(0)) {
      if (t.e < mine) {
        dp.add(P, (double)t.e, t.pos, t.vol);
        if (t.species == 2) {
          ++nannih;
          prim_rest = true;
          outN += 2;
        }
      } else if (t.nsteps >= P->max_steps) {
        dp.add(P, (double)t.e, t.pos, t.vol);
        killed = true;
      } else {
        survive = true;
        if (t.species == 0)
          outN++;
        else
          outC++;
      }
    }
  }
  const int inclN = wave_incl_scan(outN), inclC = wave_incl_scan(outC);
  const int totN = __builtin_amdgcn_readlane(inclN, 63), totC = __builtin_amdgcn_readlane(inclC, 63);
  const int n = lane() == 0 ? totN : (lane() == 1 ? totC : 0);
  const int f = reserve(S, task, n);
  int kN = __builtin_amdgcn_readlane(f, 0) + inclN - outN;
  int kC = __builtin_amdgcn_readlane(f, 1) + inclC - outC;
  const int w = (int)(threadIdx.x >> 6);
  const long long t0 = a.prof ? wall_clock64() : 0;
  EventAdd c;
  // new tracks in the oracle's draw order: secondary 0, secondary 1, then the
  // primary's annihilation at rest (two back-to-back 511 keV photons,
  // isotropic); the survivor last
#pragma unroll 1
  for (int k = 0; k < 3; ++k) {
    const int fate = k == 0 ? fate0 : (k == 1 ? fate1 : (prim_rest ? 2 : 0));
    if (!__any(fate != 0)) continue;
    const Sec<R> &s1 = o.sec[1];
    int species = k == 1 ? s1.species : o.sec[0].species;
    R e = k == 1 ? s1.e : o.sec[0].e;
    R d0 = k == 1 ? s1.d[0] : o.sec[0].d[0], d1 = k == 1 ? s1.d[1] : o.sec[0].d[1],
      d2 = k == 1 ? s1.d[2] : o.sec[0].d[2];
    if (fate == 2) {
      const double cost = 2.0 * t.rng.uniform() - 1.0;
      const double sint = sqrt((1.0 - cost) * (1.0 + cost));
      const double phi = kTwoPi * t.rng.uniform();
      d0 = (R)(sint * m_cos(phi));
      d1 = (R)(sint * m_sin(phi));
      d2 = (R)cost;
      e = (R)kMe;
      species = 0;
    }
#pragma unroll 1
    for (int j = 0; j < 2; ++j) {
      const bool go = fate == 2 || (fate == 1 && j == 0);
      if (!__any(go)) break;
      if (go) {
        const uint64_t uid = child_substream(t.rng);
        uint32_t rng[6];
        substream_state(jump, P->seed, uid, rng);
        const int idx = species == 0 ? kN++ : kC++;
        const int pg = S.dest[w][species == 0 ? 0 : 1][idx >> 6];
        store_new(PageSlot<R>(page_at<R>(a, S, pg), idx & 63), t, species, e, d0, d1, d2, uid, rng, trace);
        c.nsec0 += species == 0;
        c.nsec1 += species == 1;
        c.nsec2 += species == 2;
        spectrum(wh, species, (double)e);
        d0 = -d0;
        d1 = -d1;
        d2 = -d2;
      }
    }
  }
  if (survive) {
    const int idx = t.species == 0 ? kN : kC;
    const int pg = S.dest[w][t.species == 0 ? 0 : 1][idx >> 6];
    store_track(PageSlot<R>(page_at<R>(a, S, pg), idx & 63), t, trace);
  }
  commit(S, task, f, n);
  if (a.prof) t_derive += wall_clock64() - t0;
  if (active) {
    dp.flush(wh, P->geo.nvol > 1);
    if (killed) atomicAdd(&S.stat[kStatKilled], 1ULL);
    c.deposit(dp);
    c.npairs = pair ? 1u : 0u;
    c.nannihil = (unsigned int)nannih;
    if (!survive) c.nsteps = t.nsteps;
    c.live = outN + outC - 1;
    event_add(a, ES, t.event, c);
  }
  const int made = totN + totC - (int)__popcll(__ballot(survive));
  if (lane() == 0) {
    atomicAdd(&S.stat[kStatInteractions], (unsigned long long)task.n);
    if (q < 3) atomicAdd(&S.stat[kStatInteractions0], (unsigned long long)task.n);
    atomicAdd(&S.stat[kStatCreated], (unsigned long long)made);
    if (q < 3) atomicAdd(&S.stat[kStatCreated0], (unsigned long long)made);
  }
}

// ------------------------------------------------------------------ sharing out
// With many events in flight (LoopArgs::keep) a workgroup keeps its pages from
// launch to launch, so that an event stays with few workgroups; what it has
// beyond the average goes to those with less, after the pages that belong to
// none (injected since).  The workgroups' counts n of the last launch give
// each its own part: with q = ceil(pages / G), s = max(n - q, 0) and d = max(q
// - n, 0), the surplus is the sequence of the pages of none and the s pages of
// each workgroup in order, and a workgroup takes from it d pages behind those
// the workgroups before it take (all find one: the sum of d is at least the sum
// of s and none, as q G is at least the number of pages).
struct Shares {
  uint32_t first[kMaxGroups];  // PageSeg::first
  int sur[kMaxGroups];         // surplus pages of the workgroups before, + none
  int wave[8][3];
  int q, none, own, nt, take0;  // of this workgroup: its own pages, all, its first place in the surplus
  int rank, groups;             // workgroups with pages: before it, all
};

__device__ __forceinline__ void share_out(Shares &sh, const PageSeg *seg, int none, int q, int b, int G) {
  const int tid = (int)threadIdx.x, w = tid >> 6;
  const PageSeg e = tid < G ? seg[tid] : PageSeg{0u, 0u};
  const int n = (int)e.count;
  const int s = max(n - q, 0), d = tid < G ? max(q - n, 0) : 0;
  const int is = wave_incl_scan(s), id = wave_incl_scan(d);
  if (lane() == 63 && w < 8) {
    sh.wave[w][0] = is;
    sh.wave[w][1] = id;
  }
  __syncthreads();
  int bs = none, bd = 0, total = none;
  for (int k = 0; k < 8; ++k) {
    if (k < w) {
      bs += sh.wave[k][0];
      bd += sh.wave[k][1];
    }
    total += sh.wave[k][0];
  }
  const int take0 = bd + id - d;
  const int nt = tid < G ? min(n, q) + min(max(total - take0, 0), d) : 0;
  const int ia = wave_incl_scan(nt > 0 ? 1 : 0);
  if (lane() == 63 && w < 8) sh.wave[w][2] = ia;
  if (tid < G) {
    sh.first[tid] = e.first;
    sh.sur[tid] = bs + is - s;
  }
  __syncthreads();
  if (tid == b) {
    int r = 0, all = 0;
    for (int k = 0; k < 8; ++k) {
      if (k < w) r += sh.wave[k][2];
      all += sh.wave[k][2];
    }
    sh.q = q;
    sh.none = none;
    sh.own = min(n, q);
    sh.nt = nt;
    sh.take0 = take0;
    sh.rank = r + ia - (nt > 0 ? 1 : 0);
    sh.groups = all;
  }
  __syncthreads();
}

// Ring position of page j of the workgroup.
__device__ __forceinline__ unsigned long long share_entry(const Shares &sh, int j, unsigned long long lhead,
                                                          unsigned long long seg_lo, unsigned long long seg_hi) {
  if (j < sh.own) return seg_lo + sh.first[blockIdx.x] + (unsigned)j;
  const int p = sh.take0 + j - sh.own;
  if (p < sh.none) {
    const unsigned long long front = seg_lo - lhead;
    return (unsigned long long)p < front ? lhead + (unsigned)p : seg_hi + ((unsigned long long)p - front);
  }
  // the workgroup whose surplus holds place p: the last with sur <= p
  int lo = 0, hi = (int)gridDim.x;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (sh.sur[mid] <= p)
      lo = mid;
    else
      hi = mid;
  }
  return seg_lo + sh.first[lo] + (unsigned)(sh.q + p - sh.sur[lo]);
}

// ------------------------------------------------------------------ the loop
// kLds: the tables in LDS (LoopArgs::lds_tables).
template <class R, int kMode, int kLds>
__global__ __launch_bounds__(kLoopBlock, kLoopWaves / 4) void k_loop(LoopArgs a) {
  __shared__ Sched S;
  __shared__ DevParams sP;
  __shared__ Hist wh;
  // behind the tables: the event sums, and where they will be, until the
  // pages are taken, the shares
  const EventSums ES = {reinterpret_cast<EventSum *>(tab_lds + a.lds_tab_bytes / 16), a.ev_slots};
  Shares &sh = *reinterpret_cast<Shares *>(ES.slot);
  static_assert(sizeof(Shares) <= kMinEvSlots * sizeof(EventSum), "the shares and the event sums");
  static_assert(sizeof(Sched) + sizeof(DevParams) + sizeof(Hist) <= kLoopLdsFixed,
                "LDS beside the tables");
  const int tid = (int)threadIdx.x;
  Rings &rg = a.cnt->rings;
  // what the launch shares out (the heads and tails move when its last
  // workgroup ends)
  const unsigned long long lhead = rg.lhead, ltail = rg.ltail, fhead = rg.fhead, ftail = rg.ftail;
  const unsigned long long seg_lo = rg.seg_lo, seg_hi = rg.seg_hi;
  const int parity = rg.parity;
  const long long have = (long long)(ltail - lhead);
  const long long spare = (long long)(ftail - fhead);
  const int b = (int)blockIdx.x, G = (int)gridDim.x;
  // by rank: one of `groups` workgroups takes entries lhead + b + groups j
  const bool by_rank = !a.keep || have > (long long)G * kTake || spare < (long long)G * kMinFree;
  int groups = 1, nt = 0, at_free = 0;
  long long taken = have;
  if (by_rank) {
    groups = (int)max(min(min((long long)G, have), spare / kMinFree), 1LL);
    taken = min(have, (long long)groups * kTake);
    nt = b < groups ? (int)((taken - b + groups - 1) / groups) : 0;
    at_free = b;
  } else if (have > 0) {
    share_out(sh, a.seg + (int64_t)parity * G, (int)(have - (long long)(seg_hi - seg_lo)), (int)((have + G - 1) / G),
              b, G);
    groups = max(sh.groups, 1);
    nt = sh.nt;
    at_free = sh.rank;
  }
  // iterations left to a run that counts them
  const bool none_left = rg.iters >= a.iter_end;
  const int nf = have > 0 ? (int)min(spare / groups, (long long)(kLP - kTake)) : 0;
  PageSeg my_seg = {0u, 0u};
  if (nt > 0) {
    const long long t_end = wall_clock64() + a.ticks;
    hist_clear(wh);
    stage_params(a.P, sP);
    // (in 16-byte words) photon tables, e-/e+ tables, jump table, Sandia rows, hints
    int at_jump = 0, at_sx = 0, at_hints = 0;
    if (kLds != kLdsNone) {
      at_jump = stage_tables<R>(a.P, 0, 0);
      if (kLds == kLdsAll) at_jump = stage_tables<R>(a.P, 1, at_jump);
      at_sx = at_jump + kJumpWords / 4;
      at_hints = at_sx + a.P->nsx / 2;
      copy_words16(tab_lds + at_jump, reinterpret_cast<const uint4 *>(a.P->jump8), kJumpWords / 4);
      copy_words16(tab_lds + at_sx, reinterpret_cast<const uint4 *>(a.P->sx), a.P->nsx / 2);
      copy_words16(tab_lds + at_hints, reinterpret_cast<const uint4 *>(a.P->hints), a.P->nhints / 4);
    }
    if (tid < 16) {
      S.head[tid] = S.tail[tid] = 0;
      S.open[tid] = -1;
      S.until[tid] = INT_MAX;
      S.stat[tid] = 0;
    }
    if (tid == 0) {
      S.busy = S.stop = S.ran = S.live = S.top = 0;
      S.ftop = S.avail = nf;
      // (a pool of one workgroup: all tracks are here or in the list)
      S.max_live = a.max_tracks ? a.max_tracks - (int)rg.live : INT_MAX;
    }
    for (int j = tid; j < kTypes * kLP; j += kLoopBlock) S.rq[j / kLP][j % kLP] = kNone16;
    for (int j = tid; j < kLP; j += kLoopBlock) S.fs[j] = kNoEntry;
    __syncthreads();
    // local pages: [0, nt) with tracks, [nt, nt + nf) free
    for (int j = tid; j < nt + nf; j += kLoopBlock) {
      if (j < nt) {
        const unsigned long long at = by_rank ? lhead + (unsigned)b + (unsigned long long)groups * j
                                              : share_entry(sh, j, lhead, seg_lo, seg_hi);
        const uint32_t en = a.list[(uint32_t)at & a.mask];
        const int type = (int)(en >> 6 & 15u), n = (int)(en & 63u) + 1;
        S.gpage[j] = en >> 10;
        S.cnt[j] = n;
        // the first partial page of a type is filled further (not with tracks that
        // the launch is not to transport again), the others are tasks as they are
        if (n == kPageTracks || (a.once && type < 2) || !lds_cas(S.open[type], -1, j << 7 | n))
          S.rq[type][lds_add(S.tail[type], 1)] = (uint16_t)(j | (n - 1) << 9);
      } else {
        S.gpage[j] = a.freel[(uint32_t)(fhead + (unsigned long long)at_free * nf + (j - nt)) & a.mask];
        S.fs[j - nt] = (uint32_t)j;
      }
    }
    __syncthreads();
    events_clear(ES);
    if (a.once && tid < 2) S.until[tid] = S.tail[tid];
    if (none_left && tid == 0) S.stop = kNoIters;
    __syncthreads();
    {
      const DevParams *P = &sP;
      using T = typename NodeType<R>::T;
      constexpr bool kSmall = kLds != kLdsNone;
      const int *hints = reinterpret_cast<const int *>(tab_lds + at_hints);
      const double *sx = reinterpret_cast<const double *>(tab_lds + at_sx);
      const NodesT<R, kSmall, kSmall> N0 = [&] {
        if constexpr (kSmall)
          return NodesT<R, true, true>(reinterpret_cast<const T *>(tab_lds), hints, sx);
        else
          return NodesT<R>(P);
      }();
      const NodesT<R, (kLds == kLdsAll), kSmall> N1 = [&] {
        if constexpr (kLds == kLdsAll)
          return NodesT<R, true, true>(reinterpret_cast<const T *>(tab_lds) + P->lds_nodes[0], hints, sx);
        else if constexpr (kSmall)
          return NodesT<R, false, true>(NodeType<R>::global(P), hints, sx);
        else
          return NodesT<R>(P);
      }();
      const uint32_t *jump = [&] {
        if constexpr (kLds != kLdsNone)
          return reinterpret_cast<const uint32_t *>(tab_lds + at_jump);
        else
          return P->jump8;
      }();
      for (;;) {
        Task task = next_task(S, t_end);
        if (task.type < 0) break;
        const long long t0 = a.prof ? wall_clock64() : 0;
        long long td = 0;
        if (task.type == 0)
          transport_task<R, false, (kMode == 4 ? 4 : 0)>(a, P, N0, S, wh, ES, task);
        else if (task.type == 1)
          transport_task<R, true, kMode>(a, P, N1, S, wh, ES, task);
        else
          interact_task<R>(a, P, N0, jump, S, wh, ES, task, td);
        if (a.prof && lane() == 0) {
          const int part = task.type < 2 ? kStatTimeN + task.type : (task.type < 5 ? kStatTimeIN : kStatTimeIC);
          atomicAdd(&S.stat[part], (unsigned long long)(wall_clock64() - t0 - td));
          if (td) atomicAdd(&S.stat[kStatTimeD], (unsigned long long)td);
        }
      }
    }
    __syncthreads();
    // hand back: pages with tracks (ready, then open ones) and free pages
    const int nfree = S.ftop;
    if (tid == 0) {
      int np = 0;
      for (int t = 0; t < kTypes; ++t) np += S.tail[t] - S.head[t] + (S.open[t] >= 0 ? 1 : 0);
      const unsigned long long lp = atomicAdd(&rg.lpush, (unsigned long long)np);
      const unsigned long long fp = atomicAdd(&rg.fpush, (unsigned long long)nfree);
      S.base[0] = (uint32_t)(ltail + lp);
      my_seg = PageSeg{(uint32_t)lp, (uint32_t)np};
      S.base[1] = (uint32_t)(ftail + fp);
      if (S.ran) {
        atomicAdd(&rg.ran, 1u);
        // (no track's chain of tasks is longer than all the workgroup's)
        atomicMax(&rg.launch_iters, a.once ? 1 : S.busy >> 8);
      }
      if (S.live) atomicAdd((unsigned long long *)&rg.net, (unsigned long long)(long long)S.live);
      if (S.top) atomicAdd((unsigned long long *)&rg.grow, (unsigned long long)S.top);
      if (S.stop == kFull) atomicOr(&a.cnt->overflow, 1);
    }
    __syncthreads();
    uint32_t at = S.base[0];
    for (int t = 0; t < kTypes; ++t) {
      const int h = S.head[t], n = S.tail[t] - h;
      for (int j = tid; j < n; j += kLoopBlock) {
        const int v = S.rq[t][(h + j) & (kLP - 1)];
        const int c = (v >> 9) + 1;
        a.list[(at + (uint32_t)j) & a.mask] = page_entry(S.gpage[v & (kLP - 1)], t, c);
      }
      at += (uint32_t)n;
      const int o = S.open[t];
      if (o >= 0) {
        if (tid == 0) a.list[at & a.mask] = page_entry(S.gpage[o >> 7], t, o & 127);
        ++at;
      }
    }
    for (int j = tid; j < nfree; j += kLoopBlock)
      a.freel[(S.base[1] + (uint32_t)j) & a.mask] = S.gpage[S.fs[j]];
    hist_flush(a.rows, a.P, wh);
    events_flush(a, ES);
    if (tid < kNumStats && S.stat[tid]) atomicAdd(&a.cnt->stat[b % kStripes][tid], S.stat[tid]);
  }
  if (tid == 0) a.seg[(int64_t)(1 - parity) * G + b] = my_seg;
  // the last workgroup to end moves the rings on
  __threadfence();
  __syncthreads();
  if (tid == 0 && atomicAdd(&rg.done, 1u) == gridDim.x - 1) {
    const unsigned long long lp = atomicExch(&rg.lpush, 0ULL), fp = atomicExch(&rg.fpush, 0ULL);
    rg.lhead = lhead + (unsigned long long)taken;
    rg.ltail = ltail + lp;
    rg.seg_lo = ltail;
    rg.seg_hi = ltail + lp;
    rg.parity = 1 - parity;
    rg.fhead = fhead + (unsigned long long)groups * nf;
    rg.ftail = ftail + fp;
    rg.ran_last = atomicExch(&rg.ran, 0u);
    const long long net = (long long)atomicExch((unsigned long long *)&rg.net, 0ULL);
    const long long grow = (long long)atomicExch((unsigned long long *)&rg.grow, 0ULL);
    rg.peak = max(rg.peak, rg.live + grow);
    rg.live += net;
    rg.iters += atomicExch(&rg.launch_iters, 0);
    rg.done = 0;
  }
}

template <class R, int kMode, int kLds>
static hipError_t launch_one(const LoopArgs &a, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
  auto kernel = k_loop<R, kMode, kLds>;
  if (e0 || e1)
    hipExtLaunchKernelGGL(kernel, dim3(a.groups), dim3(kLoopBlock), (uint32_t)a.lds_bytes, st, e0, e1, 0, a);
  else
    hipLaunchKernelGGL(kernel, dim3(a.groups), dim3(kLoopBlock), (size_t)a.lds_bytes, st, a);
  return hipGetLastError();
}

template <class R, int kMode>
hipError_t launch_loop_mode(const LoopArgs &a, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
  switch (a.lds_tables) {
    case kLdsAll: return launch_one<R, kMode, kLdsAll>(a, st, e0, e1);
    case kLdsPhotons: return launch_one<R, kMode, kLdsPhotons>(a, st, e0, e1);
    default: return launch_one<R, kMode, kLdsNone>(a, st, e0, e1);
  }
}

template <class R, int kMode>
hipError_t prepare_loop_mode(int lds_tables) {
  auto kernel = lds_tables == kLdsAll ? k_loop<R, kMode, kLdsAll>
                                      : (lds_tables == kLdsPhotons ? k_loop<R, kMode, kLdsPhotons>
                                                                   : k_loop<R, kMode, kLdsNone>);
  return hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                             kLoopLds - kLoopLdsFixed);
}

}  // namespace gxt
