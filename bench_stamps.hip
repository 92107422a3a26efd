// bench_stamps.so: the decode chain's two kernels with clock stamps, for bench.py's
// in-chain timing (built by __graft_entry__.build(); not part of libexpertcache.so).
//
// Each stamped kernel runs the product kernel's device code unchanged between two reads of
// the GPU's constant-rate clock (s_memrealtime) -- the first as the kernel's first
// instruction, the second after its own stores have completed (s_waitcnt 0, and for the
// gather a workgroup barrier) -- and writes the pair with vector stores into a row of the
// caller's stamp buffer: row[0] = entry, row[1] = exit. So the bench can read, per launch in
// the decode graph, how long the kernel ran and how long the chain took to start it, with
// no event packets between the nodes and no profiler attached.
//
//   stamped_manage_remap  expert_cache_manage_remap (int32 ids, E <= 4096) + one row
//   stamped_gather        expert_cache_gather + one row per workgroup (chunks x lanes rows)
//   stamped_empty         an empty kernel + one row: the chain's floor
//   stamped_clock_khz     the nominal rate of the stamps' clock, as the device reports it
#include <hip/hip_runtime.h>

#include "vllm-expert-cache_amd/csrc/gather.h"
#include "vllm-expert-cache_amd/csrc/manage.h"

namespace {

using namespace ec;

__device__ __forceinline__ unsigned long long clock_now() {
  return __builtin_amdgcn_s_memrealtime();
}

__device__ __forceinline__ void put_row(unsigned long long* row, unsigned long long t0,
                                        unsigned long long t1) {
  typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
  *reinterpret_cast<u64x2*>(row) = u64x2{t0, t1};
}

// manage_k<W, GLOBAL_E, 4, true> with stamps
template <int W, bool GLOBAL_E>
__global__ __launch_bounds__(W* kWave) void stamped_manage_k(EC_STEP_PARAMS, ManageArgs rest,
                                                             unsigned long long* row) {
  const unsigned long long t0 = clock_now();
  __shared__ ManageLds<W, GLOBAL_E> L;
  const ManageArgs a =
      step_args(ids, step, slot_expert, slot_stamp, table, mk, E, S, rest);
  long long idv;
  manage_step<W, GLOBAL_E, 4>(a, L, idv);
  step_sync<GLOBAL_E>();
  remap_tail<W, GLOBAL_E, 4>(a, L, idv);
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  const unsigned long long t1 = clock_now();
  if (threadIdx.x == 0) put_row(row, t0, t1);
}

// gather_k<kGatherUnroll, true, false, false> with stamps, one row per workgroup
__global__ __launch_bounds__(kGatherThreads) void stamped_gather_k(
    GatherArgs g, const int* __restrict__ miss, const int* __restrict__ n_miss,
    unsigned long long* rows) {
  const unsigned long long t0 = clock_now();
  const long long wg = (long long)blockIdx.y * gridDim.x + blockIdx.x;
  gather_walk<kGatherUnroll, true, false, false>(g, miss, n_miss, nullptr, wg);
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  const unsigned long long t1 = clock_now();
  if (threadIdx.x == 0) put_row(rows + 2 * wg, t0, t1);
}

__global__ __launch_bounds__(kWave) void stamped_empty_k(unsigned long long* row) {
  const unsigned long long t0 = clock_now();
  if (__lane_id() == 0) put_row(row, t0, clock_now());
}

template <int W, bool GLOBAL_E = false>
void launch_waves(const ManageArgs& a, unsigned long long* row, hipStream_t s) {
  hipLaunchKernelGGL((stamped_manage_k<W, GLOBAL_E>), dim3(1), dim3(W * kWave), 0, s,
                     EC_STEP_ARGS(a), a, row);
}

}  // namespace

extern "C" {

// expert_cache_manage_remap's arguments (int32 ids only, E <= 4096) plus the stamp row.
int stamped_manage_remap(const void* ids, int id_bytes, int mk, int E, int S, int max_distinct,
                         int max_inserts, int* table, int* map_cold, int* slot_expert,
                         long long* slot_stamp, unsigned char* routed, long long* step,
                         int* miss, int* n_miss, int policy, int decay, void* out,
                         unsigned long long* row, hipStream_t stream) {
  if (E <= 0 || E > 4096 || S <= 0 || S > kMaxSlots || id_bytes != 4) return -1;
  if (max_inserts < 0 || max_inserts > kMaxInserts || policy < 0 || policy > 1) return -1;
  if ((mk > 0 && out == nullptr) || row == nullptr) return -1;
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
  // the product's choice for decode steps: a thread for every expert and every slot
  const int n = E > S ? E : S;
  if (E > kLdsExperts)
    launch_waves<16, true>(a, row, stream);
  else if (n <= 64)
    launch_waves<1>(a, row, stream);
  else if (n <= 128)
    launch_waves<2>(a, row, stream);
  else if (n <= 256)
    launch_waves<4>(a, row, stream);
  else if (n <= 512)
    launch_waves<8>(a, row, stream);
  else
    launch_waves<16>(a, row, stream);
  return (int)hipGetLastError();
}

// expert_cache_gather's arguments plus the stamp rows (one per workgroup: chunks x lanes).
int stamped_gather(void* d0, const void* s0, long b0, void* d1, const void* s1, long b1,
                   void* d2, const void* s2, long b2, void* d3, const void* s3, long b3,
                   void* d4, const void* s4, long b4, void* d5, const void* s5, long b5,
                   const int* miss, const int* n_miss, int chunks, int lanes,
                   unsigned long long* rows, hipStream_t stream) {
  void* const dst[kGatherBufs] = {d0, d1, d2, d3, d4, d5};
  const void* const src[kGatherBufs] = {s0, s1, s2, s3, s4, s5};
  const long bytes[kGatherBufs] = {b0, b1, b2, b3, b4, b5};
  GatherArgs g;
  if (n_miss == nullptr || rows == nullptr || !gather_plan(dst, src, bytes, chunks, lanes, g))
    return -1;
  hipLaunchKernelGGL(stamped_gather_k, dim3(chunks, lanes), dim3(kGatherThreads), 0, stream, g,
                     miss, n_miss, rows);
  return (int)hipGetLastError();
}

int stamped_empty(unsigned long long* row, hipStream_t stream) {
  if (row == nullptr) return -1;
  hipLaunchKernelGGL(stamped_empty_k, dim3(1), dim3(kWave), 0, stream, row);
  return (int)hipGetLastError();
}

// The device's nominal rate of the clock the stamps read, in kHz (-1 if not reported).
int stamped_clock_khz(int device) {
  int v = 0;
  if (hipDeviceGetAttribute(&v, hipDeviceAttributeWallClockRate, device) != hipSuccess) return -1;
  return v;
}

}  // extern "C"
