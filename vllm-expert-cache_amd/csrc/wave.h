// Wave64 primitives for gfx950 (CDNA4): DPP reductions/scans, a 64-lane sort, lane matching,
// and workgroup syncs.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ec {

constexpr int kWave = 64;

// Orders the workgroup's LDS accesses before/after this point. The local-address-space
// fences wait for LDS operations (lgkmcnt) only, so global loads and stores stay in flight
// across it; for a workgroup of one wave the compiler drops the s_barrier.
__device__ __forceinline__ void lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Orders the workgroup's LDS and global accesses before/after this point, and waits until
// its outstanding memory operations have completed.
__device__ __forceinline__ void mem_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  __builtin_amdgcn_s_waitcnt(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
}

// The lanes where `p` holds (HIP's __ballot takes an int: two more instructions).
__device__ __forceinline__ unsigned long long ballot(bool p) {
  return __builtin_amdgcn_ballot_w64(p);
}

__device__ __forceinline__ unsigned long long lanes_below() {
  return (1ull << __lane_id()) - 1ull;
}

// One DPP step of a signed 64-bit min: lanes whose DPP source is outside the row pattern
// (or in a row the mask leaves out) combine with INT64_MAX, i.e. keep their value.
template <int CTRL, int ROWMASK>
__device__ __forceinline__ long long dpp_min_step(long long v) {
  const int lo = (int)(unsigned long long)v;
  const int hi = (int)((unsigned long long)v >> 32);
  const int olo = __builtin_amdgcn_update_dpp((int)0xFFFFFFFF, lo, CTRL, ROWMASK, 0xF, false);
  const int ohi = __builtin_amdgcn_update_dpp(0x7FFFFFFF, hi, CTRL, ROWMASK, 0xF, false);
  const long long o = (long long)(((unsigned long long)(unsigned)ohi << 32) | (unsigned)olo);
  return o < v ? o : v;
}

// Minimum of `v` over all 64 lanes, returned to every lane (all lanes must be active).
// row_shr 1,2,4,8 leaves each row's minimum in its lane 15; row_bcast 15 and 31 fold the
// four rows into lane 63, which is read back as a wave-uniform value.
__device__ __forceinline__ long long wave_min_i64(long long v) {
  v = dpp_min_step<0x111, 0xF>(v);
  v = dpp_min_step<0x112, 0xF>(v);
  v = dpp_min_step<0x114, 0xF>(v);
  v = dpp_min_step<0x118, 0xF>(v);
  v = dpp_min_step<0x142, 0xA>(v);
  v = dpp_min_step<0x143, 0xC>(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned long long)v, 63);
  const unsigned hi =
      (unsigned)__builtin_amdgcn_readlane((int)((unsigned long long)v >> 32), 63);
  return (long long)(((unsigned long long)hi << 32) | lo);
}

template <int CTRL, int ROWMASK>
__device__ __forceinline__ int dpp_add_step(int v) {
  return v + __builtin_amdgcn_update_dpp(0, v, CTRL, ROWMASK, 0xF, false);
}

// Inclusive prefix sum over the 64 lanes in lane order (all lanes must be active).
__device__ __forceinline__ int wave_incl_scan(int v) {
  v = dpp_add_step<0x111, 0xF>(v);
  v = dpp_add_step<0x112, 0xF>(v);
  v = dpp_add_step<0x114, 0xF>(v);
  v = dpp_add_step<0x118, 0xF>(v);
  v = dpp_add_step<0x142, 0xA>(v);
  v = dpp_add_step<0x143, 0xC>(v);
  return v;
}

// Minimum of `v` over all 64 lanes, returned to every lane (all lanes must be active).
template <int CTRL, int ROWMASK>
__device__ __forceinline__ unsigned dpp_umin_step(unsigned v) {
  const unsigned o =
      (unsigned)__builtin_amdgcn_update_dpp((int)0xFFFFFFFF, (int)v, CTRL, ROWMASK, 0xF, false);
  return o < v ? o : v;
}

__device__ __forceinline__ unsigned wave_min_u32(unsigned v) {
  v = dpp_umin_step<0x111, 0xF>(v);
  v = dpp_umin_step<0x112, 0xF>(v);
  v = dpp_umin_step<0x114, 0xF>(v);
  v = dpp_umin_step<0x118, 0xF>(v);
  v = dpp_umin_step<0x142, 0xA>(v);
  v = dpp_umin_step<0x143, 0xC>(v);
  return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

// The value of lane (own lane xor X). Rows of 16 lanes and quads are permuted by DPP, halves
// of the wave by the permlane swaps (both operands `v`: the first result then holds the even
// row / low half of each pair, the second the odd row / high half).
template <int X>
__device__ __forceinline__ unsigned lane_xor(unsigned v) {
  static_assert(X == 1 || X == 2 || X == 3 || X == 4 || X == 7 || X == 8 || X == 15 ||
                X == 16 || X == 31 || X == 32 || X == 63);
  if constexpr (X == 1) return (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true);
  if constexpr (X == 2) return (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, true);
  if constexpr (X == 3) return (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x1B, 0xF, 0xF, true);
  if constexpr (X == 7) return (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xF, 0xF, true);
  if constexpr (X == 8) return (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xF, 0xF, true);
  if constexpr (X == 15) return (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x140, 0xF, 0xF, true);
  if constexpr (X == 4) return lane_xor<3>(lane_xor<7>(v));
  if constexpr (X == 31) return lane_xor<16>(lane_xor<15>(v));
  if constexpr (X == 63) return lane_xor<32>(lane_xor<31>(v));
  if constexpr (X == 16) {
    const auto p = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return (__lane_id() & 16) ? p[0] : p[1];
  }
  if constexpr (X == 32) {
    const auto p = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return (__lane_id() & 32) ? p[0] : p[1];
  }
}

// One compare-exchange of every lane with lane xor X: the lane with bit B set keeps the
// larger value.
template <int X, int B>
__device__ __forceinline__ unsigned sort_step(unsigned v) {
  const unsigned o = lane_xor<X>(v);
  return (__lane_id() & B) ? max(v, o) : min(v, o);
}

// `v` sorted ascending over each row of 16 lanes: 10 compare-exchanges in registers. Each
// merge starts with a mirrored exchange, so all of them run in ascending order.
__device__ __forceinline__ unsigned row_sort(unsigned v) {
  v = sort_step<1, 1>(v);
  v = sort_step<3, 2>(v);
  v = sort_step<1, 1>(v);
  v = sort_step<7, 4>(v);
  v = sort_step<2, 2>(v);
  v = sort_step<1, 1>(v);
  v = sort_step<15, 8>(v);
  v = sort_step<4, 4>(v);
  v = sort_step<2, 2>(v);
  v = sort_step<1, 1>(v);
  return v;
}

// `v` sorted ascending over the 64 lanes: 11 more.
__device__ __forceinline__ unsigned wave_sort(unsigned v) {
  v = row_sort(v);
  v = sort_step<31, 16>(v);
  v = sort_step<8, 8>(v);
  v = sort_step<4, 4>(v);
  v = sort_step<2, 2>(v);
  v = sort_step<1, 1>(v);
  v = sort_step<63, 32>(v);
  v = sort_step<16, 16>(v);
  v = sort_step<8, 8>(v);
  v = sort_step<4, 4>(v);
  v = sort_step<2, 2>(v);
  v = sort_step<1, 1>(v);
  return v;
}

// The 64 smallest of two sorted lists of 64, sorted: `v` ascending over the lanes, `down`
// the other list descending. Their lane-wise minimum is those 64 as a bitonic sequence.
__device__ __forceinline__ unsigned wave_merge_low(unsigned v, unsigned down) {
  v = min(v, down);
  v = sort_step<32, 32>(v);
  v = sort_step<16, 16>(v);
  v = sort_step<8, 8>(v);
  v = sort_step<4, 4>(v);
  v = sort_step<2, 2>(v);
  v = sort_step<1, 1>(v);
  return v;
}

// For a lane with v >= 0, the lanes whose `v` equals its own, compared on the low `bits`
// bits (all lanes must be active). One ballot per bit: needs no LDS, and no order among the
// lanes is assumed.
__device__ __forceinline__ unsigned long long wave_match(int v, int bits) {
  const unsigned long long valid = ballot(v >= 0);
  unsigned lo = (unsigned)valid, hi = (unsigned)(valid >> 32);
#pragma unroll 1
  for (int b = 0; b < bits; b += 3) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int bit = __builtin_amdgcn_sbfe(v, b + k, 1);  // 0 or -1
      const unsigned long long set = ballot(bit != 0);
      lo &= ~((unsigned)set ^ (unsigned)bit);
      hi &= ~((unsigned)(set >> 32) ^ (unsigned)bit);
    }
  }
  return (unsigned long long)hi << 32 | lo;
}

// Sums over the waves of a workgroup, from one word per wave in LDS (W <= 16): the words of
// the waves before this one, and of all waves. Wave-uniform.
template <int W>
__device__ __forceinline__ void wave_sums(const int* word, int wave, int& before, int& all) {
  if constexpr (W == 1) {
    before = 0;
    all = __builtin_amdgcn_readfirstlane(word[0]);
  } else {
    const int lane = __lane_id();
    int v = word[min(lane, W - 1)];
    v = dpp_add_step<0x111, 0xF>(v);
    if constexpr (W > 2) v = dpp_add_step<0x112, 0xF>(v);
    if constexpr (W > 4) v = dpp_add_step<0x114, 0xF>(v);
    if constexpr (W > 8) v = dpp_add_step<0x118, 0xF>(v);
    all = __builtin_amdgcn_readlane(v, W - 1);
    const int prev = __builtin_amdgcn_readlane(v, max(wave - 1, 0));
    before = wave > 0 ? prev : 0;
  }
}

}  // namespace ec
