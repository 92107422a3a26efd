// libexpertcache.so: C-ABI entry points (declared in include/expert_cache.h).
//
// Argument checks run on the host before any HIP call and return -1, exactly where the
// reference's C-ABI does (kernels/expert_cache.hip:596-598, :616-618, :631-634); otherwise
// each entry point launches one kernel on the caller's stream (two: the fused one for prefill
// chunks, and the refresh above 256 experts or slots, on large grids, or where the slot ids
// overwrite the routing ids) and returns hipGetLastError().
// The library keeps no state and allocates nothing.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "../../include/expert_cache.h"
#include "align.h"
#include "gather.h"
#include "manage.h"
#include "refresh.h"

namespace ec {
namespace {

// [p, p + pn) and [q, q + qn) share a byte
bool ranges_meet(const void* p, long long pn, const void* q, long long qn) {
  const long long a = (long long)reinterpret_cast<uintptr_t>(p);
  const long long b = (long long)reinterpret_cast<uintptr_t>(q);
  return pn > 0 && qn > 0 && a < b + qn && b < a + pn;
}

bool manage_args_bad(int E, int S, int max_inserts, int policy) {
  if (E <= 0 || S <= 0 || S > kMaxSlots || S > kSlotMask) return true;
  if (max_inserts < 0 || max_inserts > kMaxInserts) return true;
  if (policy < 0 || policy > 1) return true;
  return false;
}

// Waves of the policy step's workgroup: one thread for every expert and every slot, and a
// quarter of one for every id (prefill chunks route far more ids than there are experts).
int waves_for(int E, int S, int ids) {
  const int n = E > S ? E : S;
  const int threads = ids / 4 > n ? ids / 4 : n;
  int w = 1;
  while (w < 16 && w * kWave < threads) w *= 2;
  return w;
}

// Calls f with the number of waves as a compile-time constant.
template <class F>
void with_waves(int w, F&& f) {
  switch (w) {
    case 1: f(std::integral_constant<int, 1>()); break;
    case 2: f(std::integral_constant<int, 2>()); break;
    case 4: f(std::integral_constant<int, 4>()); break;
    case 8: f(std::integral_constant<int, 8>()); break;
    default: f(std::integral_constant<int, 16>()); break;
  }
}

template <int IDB, bool REMAP>
int launch_manage(const ManageArgs& a, hipStream_t stream) {
  if (a.E > kLdsExperts) {
    hipLaunchKernelGGL((manage_k<16, true, IDB, REMAP>), dim3(1), dim3(16 * kWave), 0, stream,
                       EC_STEP_ARGS(a), a);
  } else {
    with_waves(waves_for(a.E, a.S, a.mk), [&](auto w) {
      hipLaunchKernelGGL((manage_k<w(), false, IDB, REMAP>), dim3(1), dim3(w() * kWave), 0,
                         stream, EC_STEP_ARGS(a), a);
    });
  }
  return (int)hipGetLastError();
}

int launch_prefetch(const ManageArgs& a, hipStream_t stream) {
  if (a.E > kLdsExperts) {
    hipLaunchKernelGGL((prefetch_k<16, true>), dim3(1), dim3(16 * kWave), 0, stream, a);
  } else {
    with_waves(waves_for(a.E, a.S, a.mk), [&](auto w) {
      hipLaunchKernelGGL((prefetch_k<w(), false>), dim3(1), dim3(w() * kWave), 0, stream, a);
    });
  }
  return (int)hipGetLastError();
}

// Both layers share E and S, so one variant serves the two workgroups.
template <int IDB>
int launch_manage_prefetch(const ManageArgs& a, const ManageArgs& p, hipStream_t stream) {
  if (a.E > kLdsExperts) {
    hipLaunchKernelGGL((manage_prefetch_k<16, true, IDB>), dim3(2), dim3(16 * kWave), 0,
                       stream, a, p);
  } else {
    with_waves(waves_for(a.E, a.S, a.mk > p.mk ? a.mk : p.mk), [&](auto w) {
      hipLaunchKernelGGL((manage_prefetch_k<w(), false, IDB>), dim3(2), dim3(w() * kWave), 0,
                         stream, a, p);
    });
  }
  return (int)hipGetLastError();
}

int launch_fused(const ManageArgs& a, const AlignArgs& g, hipStream_t stream) {
  if (a.mk <= kFusedIds) {
    with_waves(waves_for(a.E, a.S, 4 * a.mk), [&](auto w) {
      hipLaunchKernelGGL((fused_k<w()>), dim3(1), dim3(w() * kWave), 0, stream,
                         EC_STEP_ARGS(a), a, g);
    });
    return (int)hipGetLastError();
  }
  // the fills get a workgroup per 16 K outputs a side
  const int fills = g.L / 16384 < 255 ? g.L / 16384 + 1 : 256;
  with_waves(waves_for(a.E, a.S, a.mk), [&](auto w) {
    hipLaunchKernelGGL((manage_defaults_k<w()>), dim3(1 + fills), dim3(w() * kWave), 0, stream,
                       EC_STEP_ARGS(a), a, g);
  });
  const int rc = (int)hipGetLastError();
  if (rc) return rc;
  hipLaunchKernelGGL(align_k, dim3((a.mk - 1) / 1024 + 1), dim3(1024), 0, stream,
                     static_cast<const int*>(a.ids), a.mk, a.E, a.S, a.table, g);
  return (int)hipGetLastError();
}

ManageArgs make_args(const void* ids, int mk, int E, int S, int max_distinct, int max_inserts,
                     int* table, int* map_cold, int* slot_expert, long long* slot_stamp,
                     unsigned char* routed, long long* step, int* miss, int* n_miss,
                     int policy, int decay, void* out) {
  ManageArgs a;
  a.ids = ids;
  a.mk = mk;
  a.E = E;
  a.S = S;
  a.max_distinct = max_distinct;
  a.max_inserts = max_inserts;
  a.table = table;
  a.map_cold = map_cold;
  a.slot_expert = slot_expert;
  a.slot_stamp = slot_stamp;
  a.routed = routed;
  a.step = step;
  a.miss = miss;
  a.n_miss = n_miss;
  a.policy = policy;
  a.decay = decay;
  a.out = out;
  return a;
}

}  // namespace
}  // namespace ec

using namespace ec;

extern "C" {

int expert_cache_manage(const int* topk_ids, int mk, int E, int S, int max_distinct,
                        int max_inserts, int* table, int* map_cold, int* slot_expert,
                        long long* slot_stamp, unsigned char* routed, long long* step,
                        int* miss, int* n_miss, int policy, int decay, hipStream_t stream) {
  if (manage_args_bad(E, S, max_inserts, policy)) return -1;
  const ManageArgs a = make_args(topk_ids, mk, E, S, max_distinct, max_inserts, table, map_cold,
                                 slot_expert, slot_stamp, routed, step, miss, n_miss, policy,
                                 decay, nullptr);
  return launch_manage<4, false>(a, stream);
}

int expert_cache_manage_remap(const void* ids, int id_bytes, int mk, int E, int S,
                              int max_distinct, int max_inserts, int* table, int* map_cold,
                              int* slot_expert, long long* slot_stamp, unsigned char* routed,
                              long long* step, int* miss, int* n_miss, int policy, int decay,
                              void* out, hipStream_t stream) {
  if (manage_args_bad(E, S, max_inserts, policy)) return -1;
  if (id_bytes != 4 && id_bytes != 8) return -1;
  if (mk > 0 && out == nullptr) return -1;
  const ManageArgs a = make_args(ids, mk, E, S, max_distinct, max_inserts, table, map_cold,
                                 slot_expert, slot_stamp, routed, step, miss, n_miss, policy,
                                 decay, out);
  return id_bytes == 8 ? launch_manage<8, true>(a, stream) : launch_manage<4, true>(a, stream);
}

int expert_cache_prefetch(const int* pred_ids, int mk, int E, int S, int max_inserts,
                          int* table, int* map_cold, int* slot_expert, long long* slot_stamp,
                          unsigned char* routed, int* miss, int* n_miss, hipStream_t stream) {
  if (manage_args_bad(E, S, max_inserts, 0) || mk < 0) return -1;
  // max_distinct = E: a prediction never reads through; no step counter is touched
  const ManageArgs a = make_args(pred_ids, mk, E, S, E, max_inserts, table, map_cold,
                                 slot_expert, slot_stamp, routed, nullptr, miss, n_miss, 0, 0,
                                 nullptr);
  return launch_prefetch(a, stream);
}

int expert_cache_manage_remap_prefetch(
    const void* ids, int id_bytes, int mk, int E, int S, int max_distinct, int max_inserts,
    int* table, int* map_cold, int* slot_expert, long long* slot_stamp, unsigned char* routed,
    long long* step, int* miss, int* n_miss, int policy, int decay, void* out,
    const int* pred_ids, int pk, int pf_max_inserts, int* pf_table, int* pf_map_cold,
    int* pf_slot_expert, long long* pf_slot_stamp, unsigned char* pf_routed, int* pf_miss,
    int* pf_n_miss, hipStream_t stream) {
  if (manage_args_bad(E, S, max_inserts, policy)) return -1;
  if (id_bytes != 4 && id_bytes != 8) return -1;
  if (mk > 0 && out == nullptr) return -1;
  if (manage_args_bad(E, S, pf_max_inserts, 0) || pk < 0) return -1;
  // the two workgroups run unordered: the layers must not share any array
  const long long e4 = 4LL * E, s4 = 4LL * S;
  if (ranges_meet(table, e4, pf_table, e4) || ranges_meet(map_cold, e4, pf_map_cold, e4) ||
      ranges_meet(slot_expert, s4, pf_slot_expert, s4) ||
      ranges_meet(slot_stamp, 2 * s4, pf_slot_stamp, 2 * s4) ||
      ranges_meet(routed, E, pf_routed, E) ||
      ranges_meet(miss, 8LL * max_inserts, pf_miss, 8LL * pf_max_inserts) ||
      ranges_meet(n_miss, 4, pf_n_miss, 4))
    return -1;
  const ManageArgs a = make_args(ids, mk, E, S, max_distinct, max_inserts, table, map_cold,
                                 slot_expert, slot_stamp, routed, step, miss, n_miss, policy,
                                 decay, out);
  const ManageArgs p = make_args(pred_ids, pk, E, S, E, pf_max_inserts, pf_table, pf_map_cold,
                                 pf_slot_expert, pf_slot_stamp, pf_routed, nullptr, pf_miss,
                                 pf_n_miss, 0, 0, nullptr);
  return id_bytes == 8 ? launch_manage_prefetch<8>(a, p, stream)
                       : launch_manage_prefetch<4>(a, p, stream);
}

int expert_cache_remap(const void* ids, int n, int id_bytes, const int* table, int E,
                       void* out, hipStream_t stream) {
  if (E <= 0 || n < 0 || (id_bytes != 4 && id_bytes != 8)) return -1;
  if (n == 0) return 0;
  const int blocks = (n + 255) / 256 < 1024 ? (n + 255) / 256 : 1024;
  if (id_bytes == 8)
    hipLaunchKernelGGL((remap_k<8>), dim3(blocks), dim3(256), 0, stream, ids, n, table, E, out);
  else
    hipLaunchKernelGGL((remap_k<4>), dim3(blocks), dim3(256), 0, stream, ids, n, table, E, out);
  return (int)hipGetLastError();
}

int expert_cache_fused(const int* topk_ids, int mk, int E, int S, int max_distinct,
                       int max_inserts, int* table, int* map_cold, int* slot_expert,
                       long long* slot_stamp, unsigned char* routed, long long* step,
                       int* miss, int* n_miss, int bs, int L, int NB, int* sorted_hot,
                       int* eids_hot, int* npad_hot, int* sorted_cold, int* eids_cold,
                       int* npad_cold, hipStream_t stream) {
  if (E <= 0 || E > kMaxAlignExperts || S <= 0 || S > kMaxSlots || S > kSlotMask) return -1;
  if (bs <= 0 || L <= 0 || NB <= 0 || mk < 0) return -1;
  if (max_inserts < 0 || max_inserts > kMaxAlignExperts) return -1;
  const ManageArgs a = make_args(topk_ids, mk, E, S, max_distinct, max_inserts, table, map_cold,
                                 slot_expert, slot_stamp, routed, step, miss, n_miss, 0, 0,
                                 nullptr);
  AlignArgs g;
  set_block_size(g, bs);
  g.L = L;
  g.NB = NB;
  g.sorted_hot = sorted_hot;
  g.eids_hot = eids_hot;
  g.npad_hot = npad_hot;
  g.sorted_cold = sorted_cold;
  g.eids_cold = eids_cold;
  g.npad_cold = npad_cold;
  return launch_fused(a, g, stream);
}

int expert_cache_refresh(const expert_cache_layer* c, const void* ids, int id_bytes, int mk,
                         void* out, hipStream_t stream) {
  if (c == nullptr || c->arrived == nullptr || mk < 0) return -1;
  if (manage_args_bad(c->E, c->S, c->S, c->policy)) return -1;
  if (id_bytes != 4 && id_bytes != 8) return -1;
  if (mk > 0 && out == nullptr) return -1;
  GatherArgs g;
  if (c->n_miss == nullptr || !gather_plan(c->dst, c->src, c->bytes, c->chunks, c->lanes, g))
    return -1;
  const ManageArgs a = make_args(ids, mk, c->E, c->S, c->E < mk ? c->E : mk, c->S, c->table,
                                 c->map_cold, c->slot_expert, c->slot_stamp, c->routed, c->step,
                                 c->miss, c->n_miss, c->policy, c->decay, out);
  const dim3 grid(c->chunks, c->lanes), block(kGatherThreads);
  // Of one launch's workgroups the first may write `out` while others still read `ids`, so
  // ids that are rewritten in place take two launches.
  const long long id_range = (long long)mk * id_bytes;
  if (c->E <= kGatherThreads && c->S <= kGatherThreads &&
      (long long)c->chunks * c->lanes <= kRefreshGroups &&
      !ranges_meet(ids, id_range, out, id_range)) {
    if (id_bytes == 8)
      hipLaunchKernelGGL((refresh_k<8>), grid, block, 0, stream, EC_STEP_ARGS(a), a, g,
                         c->arrived);
    else
      hipLaunchKernelGGL((refresh_k<4>), grid, block, 0, stream, EC_STEP_ARGS(a), a, g,
                         c->arrived);
    return (int)hipGetLastError();
  }
  const int rc = id_bytes == 8 ? launch_manage<8, true>(a, stream)
                               : launch_manage<4, true>(a, stream);
  if (rc) return rc;
  hipLaunchKernelGGL((gather_k<kGatherUnroll, true, false, false>), grid, block, 0, stream, g,
                     c->miss, c->n_miss, nullptr);
  return (int)hipGetLastError();
}

int expert_cache_gather(void* d0, const void* s0, long b0, void* d1, const void* s1, long b1,
                        void* d2, const void* s2, long b2, void* d3, const void* s3, long b3,
                        void* d4, const void* s4, long b4, void* d5, const void* s5, long b5,
                        const int* miss, const int* n_miss, int chunks, int lanes,
                        hipStream_t stream) {
  void* const dst[kGatherBufs] = {d0, d1, d2, d3, d4, d5};
  const void* const src[kGatherBufs] = {s0, s1, s2, s3, s4, s5};
  const long bytes[kGatherBufs] = {b0, b1, b2, b3, b4, b5};
  GatherArgs g;
  if (n_miss == nullptr || !gather_plan(dst, src, bytes, chunks, lanes, g)) return -1;
  hipLaunchKernelGGL((gather_k<kGatherUnroll, true, false, false>), dim3(chunks, lanes),
                     dim3(kGatherThreads), 0, stream, g, miss, n_miss, nullptr);
  return (int)hipGetLastError();
}

int expert_cache_gather_live(void* d0, const void* s0, long b0, void* d1, const void* s1,
                             long b1, void* d2, const void* s2, long b2, void* d3,
                             const void* s3, long b3, void* d4, const void* s4, long b4,
                             void* d5, const void* s5, long b5, const int* miss,
                             const int* n_miss, const int* slot_expert, int chunks, int lanes,
                             hipStream_t stream) {
  void* const dst[kGatherBufs] = {d0, d1, d2, d3, d4, d5};
  const void* const src[kGatherBufs] = {s0, s1, s2, s3, s4, s5};
  const long bytes[kGatherBufs] = {b0, b1, b2, b3, b4, b5};
  GatherArgs g;
  if (n_miss == nullptr || slot_expert == nullptr) return -1;
  if (!gather_plan(dst, src, bytes, chunks, lanes, g)) return -1;
  hipLaunchKernelGGL((gather_k<kGatherUnroll, true, false, true>), dim3(chunks, lanes),
                     dim3(kGatherThreads), 0, stream, g, miss, n_miss, slot_expert);
  return (int)hipGetLastError();
}

}  // extern "C"
