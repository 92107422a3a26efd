// expert_cache_manage on gfx950: one policy step of one layer's cache in ONE workgroup.
//
// Behaviour follows kernels/expert_cache.hip:191-282 and tests/test_policy.py:83-132
// (the step is restated in oracle/policy.c); the structure is this file's own:
//
//  * The workgroup has W waves, as many as give every expert and every slot a thread of its
//    own (64 W >= E and S; above 1024 experts 16 waves walk the experts). What bounds the
//    step is latency, and the instructions a wave runs through are a large part of it. With
//    one element a thread every phase is one short piece of straight code, whatever E and S.
//  * Every global load the step needs (step counter, ids, slot_expert, slot_stamp, table) is
//    issued up front, so the step costs one memory round trip plus the stores. Cross-lane
//    traffic is DPP and ballots, cross-wave traffic LDS behind barriers that wait for LDS
//    operations only.
//  * The LDS holds the routed flags and the table so that the remap can read the updated
//    table without another trip to memory.
//  * Misses are enumerated in ascending expert id with ballot + popcount prefixes.
//  * Victims are the nact smallest keys (stamp << 20 | slot) among the slots whose expert is
//    not routed this step, assigned in ascending key order to the misses in ascending id
//    order. They are found on 32-bit keys that order the same way (victim_key32): the first
//    wave takes the minimum of all keys once per insert where inserts are few; otherwise
//    every wave sorts its 64 keys in registers and the first wave merges the sorted lists
//    down to the 64 smallest, or, for more victims than that, a key's rank is found by a
//    binary search in each list. A stamp too far above the others for a 32-bit key needs
//    none while enough slots have one; where one lies below the keys they are counted again
//    from the smallest, and only where that leaves too few are 64-bit keys ranked by counting.
//
// Measured on MI355X, us for a graph of 48 launches, against a one-wave kernel that held up to
// 16 slots and 8 experts a lane: 128 experts, 64 slots, 8 ids 111 -> 99; 256, 192, 128 ids,
// 6.6 inserts a launch 246 -> 152; 512, 257, 50 ids, 2.6 inserts 274 -> 146.
#pragma once
#include <type_traits>

#include "wave.h"

namespace ec {

constexpr int kSlotBits = 20;
constexpr int kSlotMask = (1 << kSlotBits) - 1;
constexpr int kMaxSlots = 1024;
constexpr int kMaxInserts = 1024;
constexpr int kLdsExperts = 1024;   // flags + table are in LDS up to this many experts
constexpr long long kKeyMax = 0x7FFFFFFFFFFFFFFFll;
constexpr unsigned kKeyNone = 0xFFFFFFFFu;  // 32-bit key of a slot that cannot be evicted

struct ManageArgs {
  const void* ids;
  int mk, E, S, max_distinct, max_inserts;
  int* table;
  int* map_cold;
  int* slot_expert;
  long long* slot_stamp;
  unsigned char* routed;
  long long* step;
  int* miss;
  int* n_miss;
  int policy, decay;
  void* out;  // remap output (dtype of ids), or null
};

// Experts above kLdsExperts (GLOBAL_E) keep their flags in the caller's `routed` buffer and
// read the table from memory; the LDS arrays for them shrink to one element.
template <int W, bool GLOBAL_E>
struct ManageLds {
  static constexpr int T = W * kWave;
  // expert routed this step: a word each, so that the marks of many ids spread over the banks
  int flag[GLOBAL_E ? 1 : T];
  alignas(16) unsigned char hit[T];  // slot refreshed by a routed expert this step
  int tab[GLOBAL_E ? 1 : T];
  unsigned key[T];      // victim keys (sorted within each wave where every wave sorts)
  int ins[T];           // slot -> insert it takes, or -1
  int mis[T];           // insert r -> missing expert
  int vic[T];           // insert r -> slot, where the caller asks for it
  alignas(16) long long key64[T];  // 64-bit victim keys, where the stamps need them
  long long wmin[W];
  int wsum[2][W], wev[W];
};

typedef int i32x4 __attribute__((ext_vector_type(4)));

template <int IDB>
__device__ __forceinline__ long long load_id(const void* p, int i) {
  if constexpr (IDB == 8)
    return reinterpret_cast<const long long*>(p)[i];
  else
    return (long long)reinterpret_cast<const int*>(p)[i];
}

template <int IDB>
__device__ __forceinline__ void store_id(void* p, int i, int v) {
  if constexpr (IDB == 8)
    reinterpret_cast<long long*>(p)[i] = (long long)v;
  else
    reinterpret_cast<int*>(p)[i] = v;
}

template <bool GLOBAL_E>
__device__ __forceinline__ void step_sync() {
  if constexpr (GLOBAL_E)
    mem_sync();
  else
    lds_sync();
}

__device__ __forceinline__ int wave_index() {
  return __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
}

__device__ __forceinline__ long long victim_key(long long stamp, int slot) {
  return (long long)(((unsigned long long)stamp << kSlotBits) | (unsigned long long)slot);
}

// The 32-bit key of a stamp at or above `base` >= 1 (and below 2^43, where victim_key does
// not overflow), in the order of victim_key: SB low bits of slot, above them 0 for stamp -1
// (a pending prefetch), 1 for stamp 0 (an empty slot), then stamp - base + 2. `fits` is
// false where the stamp has no such key.
template <int SB>
__device__ __forceinline__ unsigned victim_key32(long long stamp, long long base, int slot,
                                                 bool& fits) {
  constexpr unsigned long long kTop = (1ull << (32 - SB)) - 1;  // never a key: see kKeyNone
  const unsigned long long rel =
      stamp > 0 ? (unsigned long long)(stamp - base) + 2 : (unsigned long long)(stamp + 1);
  fits = rel < kTop && stamp >= -1 && stamp < (1ll << 43) && (stamp <= 0 || stamp >= base);
  return (unsigned)rel << SB | (unsigned)slot;
}

// Up to how many inserts the first wave finds the victims one by one. Measured on MI355X in
// a graph of dependent launches that evict at every step (us a launch, one by one / sorted):
// S = 48 of 64 experts 2.25 / 2.32 at 3 inserts, 2.37 / 2.33 at 5; S = 64 of 128 2.45 / 2.53
// at 1, 2.58 / 2.55 at 3; S = 192 of 256 2.75 / 2.84 at 3, 3.07 / 2.87 at 6; S = 257 of 512
// 3.21 / 3.34 at 4, 3.41 / 3.36 at 6; S = 900 of 1024 4.77 / 4.99 at 8, 5.09 / 4.93 at 10.
// One by one costs 0.05-0.2 us more an insert, sorted stays level, so the line rises with
// the number of lists to merge.
template <int W>
__device__ __forceinline__ int few_inserts(int S) {
  return W == 1 ? 3 : 2 + S / 128;
}

// The smallest stamp above zero among the slots `ev` of the workgroup; negative where one of
// those slots has a stamp without a 32-bit key whatever the base. All threads call it.
template <int W, bool GLOBAL_E>
__device__ __forceinline__ long long smallest_stamp(ManageLds<W, GLOBAL_E>& L, bool ev,
                                                    long long stamp) {
  long long low = kKeyMax;
  if (ev) low = stamp < -1 || stamp >= 1ll << 43 ? -1 : stamp > 0 ? stamp : kKeyMax;
  low = wave_min_i64(low);
  if constexpr (W > 1) {
    if (__lane_id() == 0) L.wmin[wave_index()] = low;
    lds_sync();
#pragma unroll 1
    for (int w = 0; w < W; ++w) low = min(low, L.wmin[w]);
  }
  return low;
}

__device__ __forceinline__ long long uniform_i64(long long v) {
  const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned long long)v);
  const unsigned hi =
      (unsigned)__builtin_amdgcn_readfirstlane((int)((unsigned long long)v >> 32));
  return (long long)(((unsigned long long)hi << 32) | lo);
}

// Makes the kernel arguments that the step needs late live in SGPRs at this point, so that
// the compiler loads them together, instead of each where it is used, behind a wait.
__device__ __forceinline__ void args_in_sgprs(const ManageArgs& a) {
  asm volatile("" ::"s"(a.map_cold), "s"(a.routed), "s"(a.miss), "s"(a.n_miss), "s"(a.out),
               "s"(a.max_distinct), "s"(a.max_inserts), "s"(a.policy), "s"(a.decay));
}

// What one thread (expert `tid`, slot `tid`) has to store for a step. A kernel whose
// workgroups all run the step has one of them store it, once all have read the state.
struct StepStores {
  bool inserting;   // there were misses to insert, whether or not slots for them
  int routed;       // the expert's flag
  int miss;         // the expert's index in the miss list, or -1
  int dropped;      // expert of a pending prefetch install that leaves the slot, or -1
  int evicted;      // expert that leaves the slot for `expert`, or -1
  int insert;       // insert the slot takes, or -1
  int expert;       // ... and its expert
  bool moved, aged; // slot_expert, slot_stamp change, to
  int slot_expert;
  long long slot_stamp, step;
  int nact;
};

// What a caller adds to the step:
//  kEarly  early() runs once the loads are issued; its stores have completed, for every
//          wave, before the step's own, and before the step returns;
//  kDefer  the step's global stores go into `stores` (and the inserts' slots to L.vic)
//          instead of to memory, and every wave's loads have returned before the step does.
struct PlainStep {
  static constexpr bool kEarly = false, kDefer = false;
  __device__ __forceinline__ void early() const {}
};

template <class F>
struct EarlyStep : PlainStep {
  static constexpr bool kEarly = true;
  F f;
  __device__ __forceinline__ explicit EarlyStep(const F& fn) : f(fn) {}
  __device__ __forceinline__ void early() const { f(); }
};

struct DeferredStep : PlainStep {
  static constexpr bool kDefer = true;
  StepStores& stores;
  __device__ __forceinline__ explicit DeferredStep(StepStores& s) : stores(s) {}
};

// One policy step. On return, the updated table is in L.tab (or in memory for GLOBAL_E),
// behind a sync that the caller makes, and idv holds ids[threadIdx.x] (or -1 past mk).
//
// PF makes it the prefetch step for predicted ids: the step counter is neither read nor
// written, resident predicted experts keep their stamps, there is no ageing, and installs
// get stamp -1, which marks them pending. Victims are chosen exactly as in a real step (a
// pending slot's key is below every real key, so older unconfirmed predictions go first).
//
// A real step settles the pending slots it finds once it is served (past the read-through
// check): a slot whose expert is routed is confirmed and ends the step with the stamp a
// real install of this step gets (st under LRU, 1 under LFU; after any ageing); a slot
// whose expert is not routed is dropped -- the expert leaves the table and the slot is left
// empty at stamp 0, so a prefetch copy still in flight may stop short. The reference never
// holds a negative stamp, so on its states none of this runs.
template <int W, bool GLOBAL_E, int IDB, bool PF = false, class Caller = PlainStep>
__device__ __forceinline__ void manage_step(const ManageArgs& a, ManageLds<W, GLOBAL_E>& L,
                                            long long& idv, const Caller& caller = Caller()) {
  constexpr bool kDefer = Caller::kDefer;
  static_assert(!GLOBAL_E || !(Caller::kEarly || kDefer));
  static_assert(!PF || !kDefer);
  static_assert(!PF || IDB == 4, "prefetch takes int32 ids");
  static_assert(!GLOBAL_E || W == 16, "insert lists of 1024 experts");
  constexpr int T = W * kWave;
  constexpr int SB = W == 1 ? 6 : W == 2 ? 7 : W == 4 ? 8 : W == 8 ? 9 : 10;
  const int tid = threadIdx.x, lane = __lane_id(), wave = wave_index();
  const int E = a.E, S = a.S, mk = a.mk;
  const bool slot = tid < S;

  // ---- every independent load, issued together ---------------------------------------
  // Addresses are clamped into range instead of predicated, so no load waits behind a
  // branch; threads past the end substitute their sentinel after the loads return. The step
  // counter is a vector load: a scalar load would count in lgkmcnt, and every LDS fence
  // below would stall on it.
  long long st_v = 0;
  if constexpr (!PF)
    st_v = __hip_atomic_load(a.step, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // No branch around the id load either (a branch join would make the compiler wait for
  // it before issuing the rest): with no ids, it reads the 8-byte step counter (the
  // prefetch step: the first table entry) instead.
  using IdT = typename std::conditional<IDB == 8, long long, int>::type;
  const IdT* dummy = PF ? reinterpret_cast<const IdT*>(a.table)
                        : reinterpret_cast<const IdT*>(a.step);
  const IdT* ip = mk > 0 ? reinterpret_cast<const IdT*>(a.ids) : dummy;
  const IdT raw = ip[min(tid, max(mk - 1, 0))];
  int se = a.slot_expert[min(tid, S - 1)];
  long long sp = a.slot_stamp[min(tid, S - 1)];
  int tv = -1;
  if constexpr (!GLOBAL_E) tv = a.table[min(tid, E - 1)];

  caller.early();

  // clears: four bytes a thread
  typename std::conditional<GLOBAL_E, unsigned char, int>::type* flag;
  if constexpr (GLOBAL_E) {
    flag = a.routed;
    for (int e = tid; e < E; e += T) flag[e] = 0;
  } else {
    flag = L.flag;
    flag[tid] = 0;
  }
  if (tid < T / 4) reinterpret_cast<unsigned*>(L.hit)[tid] = 0;
  step_sync<GLOBAL_E>();
  // while the loads above are in flight; where `early` ran, its own arguments came first, and
  // waiting for these here measured slower (8 fused ids 140.5 -> 142.0 us for 48 launches,
  // against 99.8 -> 98.1 for the policy step alone)
  if constexpr (!Caller::kEarly) args_in_sgprs(a);

  // ---- routed flags (ids outside [0,E) are padding; int64 ids truncate like .to(int32))
  // The sentinels for threads past mk / S are applied only now, after the first fence, so
  // that fence does not wait for the loads.
  idv = tid < mk ? (long long)raw : -1;
  if (!slot) se = -1;
  {
    const int e = (int)idv;
    if (e >= 0 && e < E) flag[e] = 1;
  }
  if (__builtin_expect(mk > T, 0)) {
    const auto mark = [&](int e) {
      if (e >= 0 && e < E) flag[e] = 1;
    };
    unsigned done = T;  // ids marked
    if constexpr (IDB == 4) {
      // four ids a load and four loads in flight; the first T ids are marked once more
      if ((reinterpret_cast<uintptr_t>(a.ids) & 15) == 0) {
        const i32x4* v = reinterpret_cast<const i32x4*>(a.ids);
        const unsigned n = (unsigned)mk / 4;
        for (unsigned i = tid; i < n; i += 4 * T) {
          i32x4 e[4];
#pragma unroll
          for (int k = 0; k < 4; ++k) e[k] = v[min(i + k * T, n - 1)];
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            mark(e[k].x);
            mark(e[k].y);
            mark(e[k].z);
            mark(e[k].w);
          }
        }
        done = 4 * n;
      }
    }
    for (unsigned i = done + tid; i < (unsigned)mk; i += 4 * T) {
      int e[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) e[k] = (int)ip[min(i + k * T, (unsigned)(mk - 1))];
#pragma unroll
      for (int k = 0; k < 4; ++k) mark(e[k]);
    }
  }
  if constexpr (!GLOBAL_E) L.tab[tid] = tv;  // entries past E are written too: nothing reads them
  if constexpr (kDefer) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  step_sync<GLOBAL_E>();
  StepStores keep{false, 0, -1, -1, -1, -1, 0, false, false, 0, 0, 0, 0};

  // ---- distinct count (the caller's `routed` is left holding the flags); hits mark their
  // ---- slot; misses enumerate in ascending expert id ----------------------------------
  const bool held = slot & (se >= 0) & (se < E);
  const bool fx = held & (flag[held ? se : 0] != 0);  // the slot's expert is routed
  int total = 0, distinct = 0;
  if constexpr (!GLOBAL_E) {
    const int fb = flag[tid];  // zero past E
    const bool m = (fb != 0) & (tv < 0);
    if (!PF && fb != 0 && tv >= 0 && tv < S) L.hit[tv] = 1;
    const unsigned long long mask = ballot(m);
    // both counts in one word: neither exceeds 1024 over the workgroup
    const int mine = (int)(__popcll(ballot(fb != 0)) << 16 | __popcll(mask));
    int before = 0, all = mine;
    if constexpr (PF) {
      // the prefetch step has no step counter to measure stamps from
      const long long low = wave_min_i64(slot && sp > 0 ? sp : kKeyMax);
      if (lane == 0) L.wmin[wave] = low;
    }
    if constexpr (W > 1) {
      if (lane == 0) L.wsum[0][wave] = mine;
    }
    // no store of the step's own precedes this sync: where `early` made some, they have had
    // the load's round trip to complete, and waiting for them here costs little
    if constexpr (Caller::kEarly) mem_sync();
    if constexpr (kDefer)
      keep.routed = fb;
    else if (tid < E)
      a.routed[tid] = (unsigned char)fb;
    if constexpr (!Caller::kEarly) lds_sync();
    if constexpr (W > 1) wave_sums<W>(L.wsum[0], wave, before, all);
    distinct = all >> 16;
    total = all & 0xFFFF;
    const int j = (before & 0xFFFF) + __popcll(mask & lanes_below());
    if (m && j < a.max_inserts && distinct <= a.max_distinct) {
      L.mis[j] = tid;
      if constexpr (kDefer)
        keep.miss = j;
      else
        a.miss[2 * j] = tid;
    }
  } else {
    int n = 0;
    for (int e = tid; e < E; e += T) n += flag[e] != 0;
    n = wave_incl_scan(n);
    if (lane == kWave - 1) L.wsum[1][wave] = n;
    if constexpr (PF) {
      const long long low = wave_min_i64(slot && sp > 0 ? sp : kKeyMax);
      if (lane == 0) L.wmin[wave] = low;
    }
    lds_sync();
    int before;
    wave_sums<W>(L.wsum[1], wave, before, distinct);
    lds_sync();
    if (distinct <= a.max_distinct) {
      int buf = 0;
      for (int base = 0; base < E; base += T, buf ^= 1) {
        const int e = base + tid;
        const bool f = e < E && flag[e];
        const int t = f ? a.table[e] : -1;
        if (!PF && f && t >= 0 && t < S) L.hit[t] = 1;
        const bool m = f && t < 0;
        const unsigned long long mask = ballot(m);
        if (lane == 0) L.wsum[buf][wave] = __popcll(mask);
        lds_sync();
        int all;
        wave_sums<W>(L.wsum[buf], wave, before, all);
        const int j = total + before + __popcll(mask & lanes_below());
        if (m && j < a.max_inserts) {
          L.mis[j] = e;
          a.miss[2 * j] = e;
        }
        total += all;
      }
    }
  }
  const long long st = uniform_i64(st_v) + 1;
  // Wide step: read through, nothing else changes. The deferring caller's max_distinct admits
  // every step, so its arm is not reached; but without this branch the compiler holds more of
  // that kernel's arguments across the step than fit the SGPRs (42 of their words spilled for
  // 26, and 32 layer-steps of 96 of 128 slots took 374 us for 367).
  if (__builtin_expect(distinct > a.max_distinct, 0)) {
    if constexpr (kDefer) {
      keep.step = st;
      caller.stores = keep;
    } else if (tid == 0) {
      if constexpr (!PF) a.step[0] = st;
      a.n_miss[0] = 0;
    }
    return;
  }
  const int nins = min(total, a.max_inserts);

  // ---- slot side: pending prefetch installs confirmed or dropped, refreshed stamps -------
  const bool lru = a.policy == 0;
  const long long fresh = PF ? -1 : lru ? st : 1;
  const bool ageing = !PF && !lru && nins > 0 && a.decay > 0 && (st % (long long)a.decay) == 0;
  bool hit = !PF && slot && L.hit[tid] != 0;
  bool moved = false;  // slot_expert[tid] changes
  bool aged = false;   // slot_stamp[tid] changes
  if (__builtin_expect(!PF && held && sp < 0, 0)) {
    // A routed one is handed to the hit refresh below at the stamp that makes it end the
    // step at an install's stamp: 0 (+1 = 1 under LFU; st under LRU), or 1 when this step
    // ages (+1, halved = 1). Distinct slots hold distinct experts: no write conflicts.
    if (fx) {
      sp = ageing ? 1 : 0;
      hit = true;
    } else {
      if constexpr (kDefer) {
        keep.dropped = se;
      } else {
        a.table[se] = -1;
        a.map_cold[se] = se;
      }
      if constexpr (!GLOBAL_E) L.tab[se] = -1;
      se = -1;
      sp = 0;
      moved = aged = true;
    }
  }
  if (hit) {
    sp = lru ? st : (long long)((unsigned long long)sp + 1ull);
    aged = true;
  }
  int nact = 0;
  if (nins > 0) {
    if (ageing) {  // LFU ageing on inserting steps where st % decay == 0
      sp >>= 1;
      aged = true;
    }

    // ---- keys of the evictable slots (expert not routed this step) -------------------
    const bool ev = slot & !fx;
    long long base = 1;
    if constexpr (PF) {
      base = kKeyMax;
      for (int w = 0; w < W; ++w) base = min(base, L.wmin[w]);
    } else {
      if (lru) base = max(1ll, st - ((1ll << (32 - SB)) - 8));
    }
    bool fits;
    unsigned key = victim_key32<SB>(sp, base, tid, fits);
    if (!(ev & fits)) key = kKeyNone;
    // Evictable slots, and from bit 16 those among them whose stamp is too far above `base`
    // for a key: it is above all stamps that have one, so such a slot is no victim where
    // `nact` others have keys. (Without ageing a popular expert's count passes 2^22 in a
    // layer of more than 512 slots; with every such step ranked by counting, one insert at
    // 900 slots took 22 us on MI355X, and takes 4.) From bit 27 waves with a stamp below
    // `base`, or without a key at any base: then the upper half alone exceeds the slots.
    int nev_wave = (int)__popcll(ballot(ev));
    const unsigned long long far = ballot(ev & !fits);
    if (__builtin_expect(far != 0, 0)) {
      const unsigned long long above = ballot(ev & !fits & (sp > base) & (sp < 1ll << 43));
      nev_wave |= (int)((unsigned)__popcll(above) << 16 | (above != far ? 1u << 27 : 0u));
    }
    int nev = nev_wave;
    const auto keyed = [&] { return nact <= (nev & 0xFFFF) - (int)((unsigned)nev >> 16); };
    // Keys again, counted from the smallest evictable stamp: under LRU, for a slot that was
    // last used millions of steps ago (one insert at 900 slots 9.5 us, by counting 22).
    const auto rebase = [&]() -> bool {
      base = smallest_stamp(L, ev, sp);
      key = victim_key32<SB>(sp, base, tid, fits);
      if (!ev || !fits) key = kKeyNone;
      return base > 0;
    };
    bool by_count = false;
    const bool few = nins <= few_inserts<W>(S);
    int r = -1;  // insert this thread's slot takes
    if constexpr (W > 1) {
      // a wave without an evictable slot has nothing to sort
      const unsigned sorted = few || (nev_wave & 0xFFFF) == 0 ? key : wave_sort(key);
      L.key[tid] = sorted;
      L.ins[tid] = -1;
      if (lane == 0) L.wev[wave] = nev_wave;
      lds_sync();
      int before;
      wave_sums<W>(L.wev, wave, before, nev);
      nact = min(nins, nev & 0xFFFF);
      if (__builtin_expect(keyed() && nact <= kWave, 1)) {
        if (wave == 0) {
          unsigned v = sorted;  // to become, in lane i, the i-th smallest key
          if (few) {
            unsigned k[W];
#pragma unroll
            for (int c = 0; c < W; ++c)
              k[c] = c * kWave < S ? L.key[c * kWave + lane] : kKeyNone;
#pragma unroll 1
            for (int i = 0; i < nact; ++i) {
              unsigned m = k[0];
#pragma unroll
              for (int c = 1; c < W; ++c) m = min(m, k[c]);
              m = wave_min_u32(m);
              if (lane == i) v = m;
#pragma unroll
              for (int c = 0; c < W; ++c)
                if (k[c] == m) k[c] = kKeyNone;
            }
          } else {
#pragma unroll 1
            for (int c = kWave; c < S; c += kWave)
              v = wave_merge_low(v, L.key[c + kWave - 1 - lane]);
          }
          if (lane < nact) L.ins[v & (T - 1)] = lane;
        }
        lds_sync();
        r = L.ins[tid];
      } else {
        unsigned mine = sorted;
        if (!keyed()) {
          by_count = !rebase();
          mine = wave_sort(key);
          L.key[tid] = mine;
          const int n = (int)__popcll(ballot(key != kKeyNone));
          if (lane == 0) L.wev[wave] = n;
          lds_sync();
          int keys;
          wave_sums<W>(L.wev, wave, before, keys);
          by_count |= keys < nact;
        }
        // more victims than lanes: rank of this thread's sorted key, the keys below it in
        // every wave's sorted list (in its own, its lane), four lists searched at a time
        if (!by_count && mine != kKeyNone) {
          int rank = 0;
          const int lists = (S + kWave - 1) / kWave;
#pragma unroll 1
          for (int w0 = 0; w0 < lists; w0 += 4) {
            int p[4] = {0, 0, 0, 0};
#pragma unroll
            for (int step = 32; step > 0; step >>= 1) {
#pragma unroll
              for (int q = 0; q < 4; ++q)
                if (q < W && L.key[min(w0 + q, W - 1) * kWave + p[q] + step - 1] < mine)
                  p[q] += step;
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              if (q < W && w0 + q < lists)
                rank += p[q] + (L.key[(w0 + q) * kWave + p[q]] < mine ? 1 : 0);
            }
          }
          if (rank < nact) L.ins[mine & (T - 1)] = rank;
        }
        // the slots of a wave's keys are its own threads': ordered within the wave
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
        r = L.ins[tid];
      }
    } else {
      nact = min(nins, nev & 0xFFFF);
      if (__builtin_expect(!keyed(), 0))
        by_count = !rebase() || (int)__popcll(ballot(key != kKeyNone)) < nact;
      if (!by_count) {
        if (nact <= few_inserts<W>(S)) {
#pragma unroll 1
          for (int i = 0; i < nact; ++i) {
            const unsigned m = wave_min_u32(key);
            if (key == m) {
              r = i;
              key = kKeyNone;
            }
          }
        } else {
          const unsigned sorted = wave_sort(key);
          L.ins[tid] = -1;
          if (lane < nact && sorted != kKeyNone) L.ins[sorted & (T - 1)] = lane;
          lds_sync();
          r = L.ins[tid];
        }
      }
    }
    if (__builtin_expect(by_count, 0)) {
      // stamps too far apart for 32-bit keys: rank by counting on the 64-bit ones, two a read
      // (entries past S hold the largest)
      typedef long long i64x2 __attribute__((ext_vector_type(2)));
      const long long k64 = ev ? victim_key(sp, tid) : kKeyMax;
      L.key64[tid] = k64;
      lds_sync();
      if (ev) {
        const i64x2* pair = reinterpret_cast<const i64x2*>(L.key64);
        int rank = 0;
#pragma unroll 4
        for (int i = 0; i < (S + 1) / 2; ++i) {
          const i64x2 k = pair[i];
          rank += (k.x < k64) + (k.y < k64);
        }
        if (rank < nact) r = rank;
      }
    }

    // ---- installs, each by the thread of the victim slot: distinct slots, distinct experts,
    // ---- disjoint table entries, so they need no ordering among themselves ---------------
    if constexpr (W == 1) lds_sync();  // L.mis, in the paths above that made no sync
    if (r >= 0) {
      const int e = L.mis[r];
      const bool evicts = se >= 0 && se < E;
      if constexpr (kDefer) {
        if (evicts) keep.evicted = se;
        keep.insert = r;
        keep.expert = e;
        L.vic[r] = tid;
      } else {
        if (evicts) {
          a.table[se] = -1;
          a.map_cold[se] = se;
        }
        a.table[e] = tid;
        a.map_cold[e] = -1;
        a.miss[2 * r + 1] = tid;
      }
      if constexpr (!GLOBAL_E) {
        if (evicts) L.tab[se] = -1;
        L.tab[e] = tid;
      }
      se = e;
      sp = fresh;
      moved = aged = true;
    }
  }
  if constexpr (kDefer) {
    keep.inserting = nins > 0;
    keep.moved = slot && moved;
    keep.aged = slot && aged;
    keep.slot_expert = se;
    keep.slot_stamp = sp;
    keep.step = st;
    keep.nact = nact;
    caller.stores = keep;
  } else {
    if (slot && aged) a.slot_stamp[tid] = sp;
    if (slot && moved) a.slot_expert[tid] = se;
    if (tid == 0) {
      if constexpr (!PF) a.step[0] = st;
      a.n_miss[0] = nact;
    }
  }
}

// A deferred step's stores.
__device__ __forceinline__ void store_step(const ManageArgs& a, const StepStores& s) {
  const int tid = threadIdx.x;
  if (tid < a.E) a.routed[tid] = (unsigned char)s.routed;
  if (s.miss >= 0) a.miss[2 * s.miss] = tid;
  if (s.dropped >= 0) {
    a.table[s.dropped] = -1;
    a.map_cold[s.dropped] = s.dropped;
  }
  if (s.insert >= 0) {
    if (s.evicted >= 0) {
      a.table[s.evicted] = -1;
      a.map_cold[s.evicted] = s.evicted;
    }
    a.table[s.expert] = tid;
    a.map_cold[s.expert] = -1;
    a.miss[2 * s.insert + 1] = tid;
  }
  if (s.aged) a.slot_stamp[tid] = s.slot_stamp;
  if (s.moved) a.slot_expert[tid] = s.slot_expert;
  if (tid == 0) {
    a.step[0] = s.step;
    a.n_miss[0] = s.nact;
  }
}

// out[i] = table[ids[i]] against the updated table, negative ids wrapping.
template <int W, bool GLOBAL_E, int IDB>
__device__ __forceinline__ void remap_tail(const ManageArgs& a,
                                           const ManageLds<W, GLOBAL_E>& L, long long idv) {
  const int tid = threadIdx.x;
  const int E = a.E, mk = a.mk;
  auto lookup = [&](long long v) -> int {
    if (v < 0) v += E;
    if (v < 0 || v >= E) return -1;
    if constexpr (GLOBAL_E)
      return a.table[v];
    else
      return L.tab[v];
  };
  if (tid < mk) store_id<IDB>(a.out, tid, lookup(idv));
  for (int i = tid + W * kWave; i < mk; i += W * kWave)
    store_id<IDB>(a.out, i, lookup(load_id<IDB>(a.ids, i)));
}

// What the step's first loads need are a kernel's first arguments, outside the struct: the
// build has the command processor preload up to 14 words of leading scalar arguments into
// SGPRs, so those loads wait for no argument load (a struct is not preloaded); the struct's
// own loads are then in flight beside them. Measured on MI355X, us for a graph of 48
// launches: policy step 101.4 -> 100.2 at 8 ids, 152.3 -> 150.4 at 50 ids of 512 experts,
// 158.4 -> 154.4 at 128 of 256; fused call at 8 ids 146.6 -> 141.2.
#define EC_STEP_PARAMS                                                                   \
  const void *ids, long long *step, int *slot_expert, long long *slot_stamp, int *table, \
      int mk, int E, int S
#define EC_STEP_ARGS(a) \
  (a).ids, (a).step, (a).slot_expert, (a).slot_stamp, (a).table, (a).mk, (a).E, (a).S

__device__ __forceinline__ ManageArgs step_args(EC_STEP_PARAMS, const ManageArgs& rest) {
  ManageArgs a = rest;
  a.ids = ids;
  a.step = step;
  a.slot_expert = slot_expert;
  a.slot_stamp = slot_stamp;
  a.table = table;
  a.mk = mk;
  a.E = E;
  a.S = S;
  return a;
}

template <int W, bool GLOBAL_E, int IDB, bool REMAP>
__global__ __launch_bounds__(W* kWave) void manage_k(EC_STEP_PARAMS, ManageArgs rest) {
  __shared__ ManageLds<W, GLOBAL_E> L;
  const ManageArgs a =
      step_args(ids, step, slot_expert, slot_stamp, table, mk, E, S, rest);
  long long idv;
  manage_step<W, GLOBAL_E, IDB>(a, L, idv);
  if constexpr (REMAP) {
    step_sync<GLOBAL_E>();
    remap_tail<W, GLOBAL_E, IDB>(a, L, idv);
  }
}

// The prefetch step (manage_step with PF) for int32 predicted ids.
template <int W, bool GLOBAL_E>
__global__ __launch_bounds__(W* kWave) void prefetch_k(ManageArgs a) {
  __shared__ ManageLds<W, GLOBAL_E> L;
  long long idv;
  manage_step<W, GLOBAL_E, 4, true>(a, L, idv);
}

// Two workgroups, two layers: workgroup 0 runs layer a's policy step and remap (manage_k
// with REMAP), workgroup 1 the prefetch step of another layer p (prefetch_k). The host
// rejects states that share arrays, so the workgroups touch disjoint memory and need no
// ordering between them; the pair occupies one node of the stream instead of two.
template <int W, bool GLOBAL_E, int IDB>
__global__ __launch_bounds__(W* kWave) void manage_prefetch_k(ManageArgs a, ManageArgs p) {
  __shared__ ManageLds<W, GLOBAL_E> L;
  long long idv;
  if (blockIdx.x == 0) {
    manage_step<W, GLOBAL_E, IDB>(a, L, idv);
    step_sync<GLOBAL_E>();
    remap_tail<W, GLOBAL_E, IDB>(a, L, idv);
  } else {
    manage_step<W, GLOBAL_E, 4, true>(p, L, idv);
  }
}

// Standalone remap, any grid; one id per lane per iteration.
template <int IDB>
__global__ __launch_bounds__(256) void remap_k(const void* ids, int n, const int* table, int E,
                                               void* out) {
  const int stride = gridDim.x * blockDim.x;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    long long v = load_id<IDB>(ids, i);
    if (v < 0) v += E;
    store_id<IDB>(out, i, (v >= 0 && v < E) ? table[v] : -1);
  }
}

}  // namespace ec
