// expert_cache_fused on gfx950: the LRU policy step followed by both moe_align_block_size
// outputs (kernels/expert_cache.hip:431-588 semantics).
//
// The policy half is manage_step with policy 0 and no decay (a hit and an install both stamp
// the current step). The align half buckets every routing id against the updated table --
// resident ids by slot ("hot"), the rest by expert id ("cold") -- pads each bucket to a
// multiple of the block size, scans, and places each id at its bucket offset plus its rank
// among the earlier ids of the same bucket, so the output is in token order within every
// bucket for every mk (the reference is token-ordered for mk <= 256 and unordered above).
//
// An id's rank is found without a pass over earlier ids: its lane's rank among the lanes of
// its wave with the same bucket (wave_match), plus the counts of the earlier waves, which
// each wave leaves in its own row of a small count matrix in LDS, plus, where several
// workgroups share the ids, the count of the workgroup's earlier ids. No output position is
// written twice (an id, its bucket's padding, or the default past the padded total), so
// nothing is staged and no store is waited for.
//
//  * fused_k, up to kFusedIds ids: the policy step and both alignments in one workgroup,
//    one id, one expert and one slot a thread.
//  * align_k, more ids: a workgroup per 1024 ids, after a launch of the policy step alone.
//    Each workgroup counts the ids before and after its own itself (they come from the L2),
//    which costs less than the node or the cross-XCD handoff that sharing the counts would.
//
// Measured on MI355X, us a launch in a graph, against the same work in one wave that staged
// its output in LDS: 8 ids (128 experts, 64 slots, block 16) 4.7 -> 3.9; 512 ids (256, 128,
// 16) 12.6 -> 7.3; 16384 ids (128, 64, 64) 232 -> 15.6.
#pragma once
#include "manage.h"

namespace ec {

constexpr int kMaxAlignExperts = 1024;
constexpr int kFusedIds = 1024;  // most ids of the one-workgroup kernel: one a thread

struct AlignArgs {
  int bs, L, NB;
  int* sorted_hot;
  int* eids_hot;
  int* npad_hot;
  int* sorted_cold;
  int* eids_cold;
  int* npad_cold;
};

// Buckets are slots 0 .. S-1 (hot), then S + e for expert e (cold): at most 2T.
template <int W>
struct AlignLds {
  static constexpr int T = W * kWave;
  unsigned short cnt[W][2 * T];  // ids per bucket of each wave, then of the waves before it
  int start[2 * T];  // position of the workgroup's first id of the bucket
  int end[2 * T];    // position past the bucket's last id
  int wsum[2][W];
};

// What one workgroup's thread needs after align_place: the padded totals of both sides.
struct AlignTotals {
  int hot, cold;
};

// Bucket of one routing id, -1 for padding and out-of-range ids.
__device__ __forceinline__ int align_key(int e, int E, int S, const int* tab) {
  if (e < 0 || e >= E) return -1;
  const int s = tab[e];
  return ((unsigned)s < (unsigned)S) ? s : S + e;
}

// x / bs for the wave-uniform block size: a shift for powers of two (vLLM's block sizes).
struct BlockDiv {
  int bs, shift;
  __device__ __forceinline__ explicit BlockDiv(int b)
      : bs(b), shift((b & (b - 1)) == 0 ? __builtin_ctz((unsigned)b) : -1) {}
  __device__ __forceinline__ int div(int x) const { return shift >= 0 ? x >> shift : x / bs; }
  __device__ __forceinline__ int pad(int x) const { return div(x + bs - 1) * bs; }
};

typedef int i32x4 __attribute__((ext_vector_type(4)));

// dst[from, to) = v over `n` threads of which this is number `me`; 16-byte stores when dst is
// 16-byte aligned.
__device__ __forceinline__ void fill_i32(int* dst, int from, int to, int v, int me, int n) {
  if (from >= to) return;
  if ((reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
    const int a0 = min((from + 3) & ~3, to);
    const int a1 = a0 + ((to - a0) & ~3);
    if (me < a0 - from) dst[from + me] = v;
    for (long long p = a0 + 4ll * me; p < a1; p += 4ll * n)
      *reinterpret_cast<i32x4*>(dst + p) = i32x4{v, v, v, v};
    if (me < to - a1) dst[a1 + me] = v;
  } else {
    for (long long p = from + me; p < to; p += n) dst[p] = v;
  }
}

// Clears the rows of the count matrix that `waves` waves fill; the caller syncs.
template <int W>
__device__ __forceinline__ void align_clear(AlignLds<W>& A, int waves, int buckets) {
  constexpr int T = W * kWave;
  unsigned* rows = reinterpret_cast<unsigned*>(A.cnt);
  if (2 * (int)threadIdx.x < buckets)
    for (int w = 0; w < waves; ++w) rows[w * T + threadIdx.x] = 0;
}

// Places id `i` of bucket `kk` (-1: none) for every thread of the workgroup, whose ids are
// consecutive and lie in its first `waves` waves. The count matrix is clear. With PART the
// workgroup holds only some of the ids: on entry A.start and A.end hold, per bucket, the
// counts of the ids before and after its own. On return A.end and, per bucket, A.start are
// positions as declared (behind the sync made here).
template <int W, bool PART>
__device__ __forceinline__ AlignTotals align_place(const AlignArgs& g, AlignLds<W>& A, int E,
                                                   int S, BlockDiv d, int kk, int i,
                                                   int waves) {
  const int tid = threadIdx.x, lane = __lane_id(), wave = wave_index();
  int rank = 0;
  if (wave < waves) {
    const unsigned long long m = wave_match(kk, 32 - __clz(S + E - 1));
    rank = __popcll(m & lanes_below());
    // the bucket's last lane in the wave leaves the wave's count
    if (kk >= 0 && (m >> lane) == 1ull) A.cnt[wave][kk] = (unsigned short)(rank + 1);
  }
  lds_sync();
  // thread b: slot bucket b and expert bucket S + b
  int n[2] = {0, 0}, before[2] = {0, 0};
  const int size[2] = {S, E};
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int b = tid + (h ? S : 0);
    if (tid < size[h]) {
      if (waves == 1) {
        n[h] = A.cnt[0][b];
        A.cnt[0][b] = 0;
      } else {
        for (int w0 = 0; w0 < waves; w0 += 4) {
          int c[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) c[q] = w0 + q < waves ? A.cnt[min(w0 + q, W - 1)][b] : 0;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            if (w0 + q < waves) A.cnt[min(w0 + q, W - 1)][b] = (unsigned short)n[h];
            n[h] += c[q];
          }
        }
      }
      if constexpr (PART) {
        before[h] = A.start[b];
        n[h] += before[h] + A.end[b];
      }
    }
  }
  // exclusive scans of the padded counts of both sides over the threads
  const int padded[2] = {d.pad(n[0]), d.pad(n[1])};
  int first[2], total[2];
  int scan[2] = {wave_incl_scan(padded[0]), wave_incl_scan(padded[1])};
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    first[h] = scan[h] - padded[h];
    total[h] = __builtin_amdgcn_readlane(scan[h], kWave - 1);
    if constexpr (W > 1) {
      if (lane == 0) A.wsum[h][wave] = total[h];
    }
  }
  if constexpr (W > 1) {
    lds_sync();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      int b;
      wave_sums<W>(A.wsum[h], wave, b, total[h]);
      first[h] += b;
    }
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (tid < size[h]) {
      const int b = tid + (h ? S : 0);
      A.start[b] = first[h] + before[h];
      A.end[b] = first[h] + n[h];
    }
  }
  lds_sync();
  if (kk >= 0) {
    const int pos = A.start[kk] + A.cnt[wave][kk] + rank;
    int* sorted = kk < S ? g.sorted_hot : g.sorted_cold;
    if (pos < g.L) sorted[pos] = i;
  }
  return {total[0], total[1]};
}

// The padding of each bucket (mk) and its blocks' expert ids, a wave per bucket of the
// launch's `nwaves`, this one being number `me`. `from` is the bucket's first position.
template <int W>
__device__ __forceinline__ void align_pad(const AlignArgs& g, const AlignLds<W>& A, int E,
                                          int S, int mk, BlockDiv d, int me, int nwaves,
                                          const int* from) {
  const int lane = __lane_id();
  for (int b = me; b < S + E; b += nwaves) {
    const int p0 = from[b], p1 = A.end[b];
    if (p0 == p1) continue;
    const int p2 = p0 + d.pad(p1 - p0);
    int* sorted = b < S ? g.sorted_hot : g.sorted_cold;
    int* eids = b < S ? g.eids_hot : g.eids_cold;
    const int id = b < S ? b : b - S;
    for (int p = p1 + lane; p < min(p2, g.L); p += kWave) sorted[p] = mk;
    const int q1 = min(d.div(p2), g.NB);
    for (int q = d.div(p0) + lane; q < q1; q += kWave) eids[q] = id;
  }
}

// Past the padded totals the outputs hold mk and -1.
__device__ __forceinline__ void align_rest(const AlignArgs& g, int mk, BlockDiv d,
                                           AlignTotals t, int me, int n) {
  if (me == 0) {
    g.npad_hot[0] = t.hot;
    g.npad_cold[0] = t.cold;
  }
  fill_i32(g.sorted_hot, min(t.hot, g.L), g.L, mk, me, n);
  fill_i32(g.sorted_cold, min(t.cold, g.L), g.L, mk, me, n);
  fill_i32(g.eids_hot, min(d.div(t.hot), g.NB), g.NB, -1, me, n);
  fill_i32(g.eids_cold, min(d.div(t.cold), g.NB), g.NB, -1, me, n);
}

// One workgroup: T >= E, S and mk.
template <int W>
__global__ __launch_bounds__(W* kWave) void fused_k(ManageArgs a, AlignArgs g) {
  constexpr int T = W * kWave;
  __shared__ ManageLds<W, false> L;
  __shared__ AlignLds<W> A;
  // per side, the bucket of each block below the padded total: no more blocks than ids
  __shared__ unsigned short block[2][T];
  args_in_sgprs(a);
  const int tid = threadIdx.x;
  const int E = a.E, S = a.S, mk = a.mk, waves = (mk + kWave - 1) / kWave;
  const BlockDiv d(g.bs);
  align_clear<W>(A, max(waves, 1), S + E);
  long long idv;
  manage_step<W, false, 4>(a, L, idv);
  lds_sync();
  const int kk = align_key((int)idv, E, S, L.tab);
  const AlignTotals t = align_place<W, false>(g, A, E, S, d, kk, tid, max(waves, 1));
  align_rest(g, mk, d, t, tid, T);
  // thread b names the blocks of its two buckets
  if (tid < S)
    for (int q = d.div(A.start[tid]), q1 = d.div(A.end[tid] + g.bs - 1); q < q1; ++q)
      block[0][q] = (unsigned short)tid;
  if (tid < E)
    for (int q = d.div(A.start[S + tid]), q1 = d.div(A.end[S + tid] + g.bs - 1); q < q1; ++q)
      block[1][q] = (unsigned short)tid;
  lds_sync();
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int total = h ? t.cold : t.hot;
    const int* end = A.end + (h ? S : 0);
    int* sorted = h ? g.sorted_cold : g.sorted_hot;
    int* eids = h ? g.eids_cold : g.eids_hot;
    const int q1 = min(d.div(total), g.NB);
    for (int q = tid; q < q1; q += T) eids[q] = block[h][q];
    const int p1 = min(total, g.L);
    for (int p = tid; p < p1; p += T)
      if (p >= end[block[h][d.div(p)]]) sorted[p] = mk;
  }
}

// A workgroup per 1024 ids, against the table as it is.
__global__ __launch_bounds__(1024) void align_k(const int* ids, int mk, int E, int S,
                                                const int* table, AlignArgs g) {
  constexpr int W = 16, T = W * kWave;
  __shared__ AlignLds<W> A;
  __shared__ int from[2 * T];           // first position of each bucket
  __shared__ unsigned short bucket[T];  // of each expert
  const int tid = threadIdx.x, part = blockIdx.x, parts = gridDim.x;
  const int first = part * T;
  const BlockDiv d(g.bs);
  if (tid < E) {
    const int s = table[tid];
    bucket[tid] = (unsigned short)((unsigned)s < (unsigned)S ? s : S + tid);
  }
  align_clear<W>(A, W, S + E);
  A.start[tid] = A.start[T + tid] = A.end[tid] = A.end[T + tid] = 0;
  lds_sync();
  // ids of the other workgroups, counted per bucket: before this one's, and after
  auto count = [&](int e, int i) {
    if (e >= 0 && e < E) atomicAdd(&(i < first ? A.start : A.end)[bucket[e]], 1);
  };
  const int mine = first + tid < mk ? ids[first + tid] : -1;
  if ((reinterpret_cast<uintptr_t>(ids) & 15) == 0) {
    // four ids a load; `first` is a multiple of four and only the last workgroup's ids end
    // at mk, so no vector straddles a boundary except the one cut off here
    const int n4 = mk & ~3;
    for (int i = 4 * tid; i < n4; i += 4 * T) {
      if (i >= first && i < first + T) continue;
      const i32x4 e = *reinterpret_cast<const i32x4*>(ids + i);
      count(e.x, i);
      count(e.y, i);
      count(e.z, i);
      count(e.w, i);
    }
    const int i = n4 + tid;
    if (i < mk && (i < first || i >= first + T)) count(ids[i], i);
  } else {
    for (int i = tid; i < mk; i += T)
      if (i < first || i >= first + T) count(ids[i], i);
  }
  lds_sync();
  // positions of the buckets' starts: align_place leaves this workgroup's own in A.start
  int before[2] = {tid < S ? A.start[tid] : 0, tid < E ? A.start[S + tid] : 0};
  const int kk = mine >= 0 && mine < E ? bucket[mine] : -1;
  const AlignTotals t = align_place<W, true>(g, A, E, S, d, kk, first + tid, W);
  if (tid < S) from[tid] = A.start[tid] - before[0];
  if (tid < E) from[S + tid] = A.start[S + tid] - before[1];
  lds_sync();
  align_rest(g, mk, d, t, first + tid, parts * T);
  align_pad<W>(g, A, E, S, mk, d, part * W + wave_index(), parts * W, from);
}

}  // namespace ec
