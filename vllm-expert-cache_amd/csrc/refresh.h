// expert_cache_refresh on gfx950: a layer's policy step, remap and gather in one launch.
//
// As two launches the gather's workgroups wait for a node of their own and then for the miss
// list to come back from memory. Here every workgroup of the gather's grid runs the whole
// policy step for itself: the state is a few KB, the step is latency and not work, and the
// miss list is then in each workgroup's own LDS, so its first host reads follow at once. No
// workgroup waits for another:
//
//  * A step that inserts nothing is stored by the first workgroup at once. It changes stamps
//    and flags, and takes unrouted experts of dropped prefetches out of the table; whether
//    there is anything to insert depends on the ids and their table entries alone, so a
//    workgroup that reads the state late finds the same. That holds because `out` does not
//    overlap the ids, and because nothing but the routed experts' entries decides: no step
//    reads through (max_distinct is min(E, ids)) and the insert budget is S, so a step without
//    inserts is one without misses.
//  * A step that inserts is stored by the last workgroup to have read the state (they count
//    themselves in `arrived`), after its share of the copy, when its ticket has come back. A
//    workgroup takes its ticket after the step, whose second sync waits for all of its loads
//    of the state (DeferredStep).
//    Counting at every step, before it is known whether it inserts, put the ticket's round
//    trip (over a microsecond) into the steps that insert nothing and gained nothing.
//
// Measured on MI355X, us for a graph of 32 layer-steps, against the two launches of a one-wave
// step and the gather: 128 experts of 4.7 MB, 8 ids, 96 slots, 0.1 inserts a step 422 -> 374;
// 64 slots, 0.45 inserts 1334 -> 1290 (the host link's time is 1172). Four refreshes called
// from Python 65 -> 47.
#pragma once
#include "gather.h"
#include "manage.h"

namespace ec {

// The gather's tiles take 256 threads, so the step has four waves: E and S up to 256.
constexpr int kRefreshWaves = kGatherThreads / kWave;

// Largest grid that refreshes in one launch. The arrivals are atomics on one word, about
// 10 ns each, which the copy of a small expert does not hide. Measured on MI355X, us a launch
// with one 4 KB insert at 128 experts and 64 slots, one launch / two: 32 workgroups 5.0 / 5.8,
// 128 5.6 / 5.8, 160 5.9 / 5.9, 192 6.3 / 5.9, 256 7.0 / 5.8, 1024 15.5 / 5.9; a 1 MB insert,
// whose copy hides them, 23.8 / 26.1 at 128.
constexpr long long kRefreshGroups = 128;

template <int IDB>
__global__ __launch_bounds__(kGatherThreads) void refresh_k(EC_STEP_PARAMS, ManageArgs rest,
                                                            GatherArgs g, unsigned* arrived) {
  constexpr int W = kRefreshWaves;
  __shared__ ManageLds<W, false> L;
  __shared__ int last;
  const ManageArgs a =
      step_args(ids, step, slot_expert, slot_stamp, table, mk, E, S, rest);
  StepStores stores;
  long long idv;
  manage_step<W, false, IDB>(a, L, idv, DeferredStep(stores));
  lds_sync();
  const unsigned wg = blockIdx.y * gridDim.x + blockIdx.x;
  unsigned ticket = 0;
  if (stores.inserting) {
    if (threadIdx.x == 0)
      ticket = __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    gather_pairs<kGatherUnroll, true, false, false>(
        g, stores.nact,
        [&](int j, int& e, int& sl) {
          e = __builtin_amdgcn_readfirstlane(L.mis[j]);
          sl = __builtin_amdgcn_readfirstlane(L.vic[j]);
        },
        nullptr, wg);
    if (threadIdx.x == 0) last = ticket == gridDim.x * gridDim.y - 1;
    lds_sync();
    if (!last) return;
    // for the next launch
    if (threadIdx.x == 0)
      __hip_atomic_store(arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else if (wg != 0) {
    return;
  }
  store_step(a, stores);
  remap_tail<W, false, IDB>(a, L, idv);
}

}  // namespace ec
