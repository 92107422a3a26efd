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
// workgroups share the ids, the count of the workgroup's earlier ids.
//
//  * fused_k, up to kFusedIds ids: the policy step and both alignments in one workgroup,
//    one id, one expert and one slot a thread. Up to 64 ids are placed by one wave that
//    sorts them in registers.
//  * align_k, more ids: a workgroup per 1024 ids, after a launch whose first workgroup runs
//    the policy step while the others store the outputs' defaults (manage_defaults_k).
//    Each workgroup counts the ids before and after its own itself (they come from the L2),
//    which costs less than the node or the cross-XCD handoff that sharing the counts would.
//
// Measured on MI355X, us a launch in a graph, against the same work in one wave that staged
// its output in LDS: 8 ids (128 experts, 64 slots, block 16) 4.7 -> 2.9; 512 ids (256, 128,
// 16) 12.5 -> 5.3; 16384 ids (128, 64, 64) 232 -> 12.3; 65536 ids 800 -> 18.
#pragma once
#include "manage.h"

namespace ec {

constexpr int kMaxAlignExperts = 1024;
constexpr int kFusedIds = 1024;  // most ids of the one-workgroup kernel: one a thread

struct AlignArgs {
  int bs, L, NB;
  unsigned div_mul;  // x / bs = x * div_mul >> div_shift for 0 <= x < 2^31
  int div_shift;
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
  int end[2 * T];    // ids of the bucket after the workgroup's
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

// The multiplier and shift of the division by bs: with l = ceil(log2 bs), the multiplier is
// 2^(31 + l) / bs rounded up (below 2^32), and the excess, below 1 / bs over x < 2^31, never
// reaches the next quotient.
inline void set_block_size(AlignArgs& g, int bs) {
  int l = 0;
  while ((1ll << l) < bs) ++l;
  g.bs = bs;
  g.div_shift = 31 + l;
  g.div_mul = (unsigned)((((unsigned __int128)1 << g.div_shift) + bs - 1) / bs);
}

struct BlockDiv {
  int bs, shift;
  unsigned mul;
  __device__ __forceinline__ explicit BlockDiv(const AlignArgs& g)
      : bs(g.bs), shift(g.div_shift), mul(g.div_mul) {}
  __device__ __forceinline__ int div(int x) const {
    return (int)((unsigned long long)(unsigned)x * mul >> shift);
  }
  __device__ __forceinline__ int pad(int x) const { return div(x + bs - 1) * bs; }
};

// x[0, n) = y[0, n) = v over `threads` threads of which this is number `me`; 16-byte stores
// where both are 16-byte aligned.
__device__ __forceinline__ void fill_pair(int* x, int* y, int n, int v, int me, int threads) {
  unsigned p = 0;
  if (((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 15) == 0) {
    const unsigned n4 = (unsigned)n / 4;
    for (p = me; p < n4; p += threads) reinterpret_cast<i32x4*>(x)[p] = i32x4{v, v, v, v};
    for (p = me; p < n4; p += threads) reinterpret_cast<i32x4*>(y)[p] = i32x4{v, v, v, v};
    p = 4 * n4;
  }
  for (p += me; p < (unsigned)n; p += threads) x[p] = y[p] = v;
}

// The defaults of all outputs: mk and -1.
__device__ __forceinline__ void align_defaults(const AlignArgs& g, int mk, int me,
                                               int threads) {
  fill_pair(g.sorted_hot, g.sorted_cold, g.L, mk, me, threads);
  fill_pair(g.eids_hot, g.eids_cold, g.NB, -1, me, threads);
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
// consecutive and lie in its first `waves` waves, and names the blocks of the buckets. The
// count matrix is clear and the outputs hold their defaults. With PART the workgroup is
// number `part` of `parts` and holds only some of the ids: on entry A.start and A.end hold,
// per bucket, the counts of the ids before and after its own.
template <int W, bool PART>
__device__ __forceinline__ AlignTotals align_place(const AlignArgs& g, AlignLds<W>& A, int E,
                                                   int S, BlockDiv d, int kk, int i,
                                                   int waves, int part, int parts) {
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
  constexpr int kRows = W < 8 ? W : 8;  // rows read together
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int b = tid + (h ? S : 0);
    if (tid < size[h]) {
      for (int w0 = 0; w0 < waves; w0 += kRows) {
        int c[kRows];
#pragma unroll
        for (int q = 0; q < kRows; ++q) c[q] = A.cnt[w0 + q][b];
#pragma unroll
        for (int q = 0; q < kRows; ++q) {
          A.cnt[w0 + q][b] = (unsigned short)n[h];
          if (w0 + q < waves) n[h] += c[q];  // the rows past the ids' are not clear
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
    }
  }
  lds_sync();
  // Thread b names the blocks of its two buckets; the first workgroups of a launch, as many
  // as a power of two, take each its share of every wave's buckets. A bucket of many blocks
  // is left to its whole wave.
  const int sharing = min(1 << (31 - __clz(parts)), kWave);
  if (part < sharing) {
    const bool own = (lane & (sharing - 1)) == part;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      int* eids = h ? g.eids_cold : g.eids_hot;
      const int q0 = d.div(first[h]), q1 = min(d.div(first[h] + padded[h]), g.NB);
      const bool many = own && q1 - q0 > 8;
      if (own && !many)
        for (int q = q0; q < q1; ++q) eids[q] = tid;
      for (unsigned long long m = ballot(many); m != 0; m &= m - 1) {
        const int l = __ffsll((long long)m) - 1;
        const int end = __builtin_amdgcn_readlane(q1, l);
        for (int q = __builtin_amdgcn_readlane(q0, l) + lane; q < end; q += kWave)
          eids[q] = wave * kWave + l;
      }
    }
  }
  if (kk >= 0) {
    const int pos = A.start[kk] + A.cnt[wave][kk] + rank;
    int* sorted = kk < S ? g.sorted_hot : g.sorted_cold;
    if (pos < g.L) sorted[pos] = i;
  }
  return {total[0], total[1]};
}

// align_place for up to 64 ids, in one wave's registers: lane -> id `lane` of bucket `kk`. The
// ids are sorted by (bucket, token); a bucket is then a run of lanes, and one scan over the
// padded lengths of the runs gives every position.
__device__ __forceinline__ AlignTotals align_place_wave(const AlignArgs& g, int S, int mk,
                                                        BlockDiv d, int kk) {
  const int lane = __lane_id();
  const unsigned none = 0xFFFFFFFFu;
  const unsigned key = kk >= 0 ? (unsigned)kk << 6 | (unsigned)lane : none;
  const unsigned s = mk <= 16 ? row_sort(key) : wave_sort(key);
  const int b = (int)(s >> 6);
  const bool valid = s != none;
  const int prev = __builtin_amdgcn_update_dpp(-1, b, 0x138, 0xF, 0xF, false);  // lane - 1's
  const unsigned long long heads = ballot(valid & (b != prev));
  const unsigned long long upto = lanes_below() << 1 | 1ull;  // this lane and those below
  const int head = 63 - __clzll((long long)(heads & upto));
  const unsigned long long later = heads & ~upto;
  const int nvalid = (int)__popcll(ballot(valid));
  const int next = later ? __ffsll((long long)later) - 1 : nvalid;
  const int padded = d.pad(next - head);
  const bool first = valid & (b != prev);
  const int scan = wave_incl_scan(first ? padded : 0);
  const int nhot = (int)__popcll(ballot(valid & (b < S)));
  const int all = __builtin_amdgcn_readlane(scan, kWave - 1);
  const int at = __builtin_amdgcn_readlane(scan, max(nhot - 1, 0));
  const int hot = nhot > 0 ? at : 0;
  if (valid) {
    const bool is_hot = b < S;
    const int start = scan - padded - (is_hot ? 0 : hot);
    int* sorted = is_hot ? g.sorted_hot : g.sorted_cold;
    const int pos = start + lane - head;
    if (pos < g.L) sorted[pos] = (int)(s & 63);
    if (first) {
      int* eids = is_hot ? g.eids_hot : g.eids_cold;
      const int q1 = min(d.div(start + padded), g.NB);
      for (int q = d.div(start); q < q1; ++q) eids[q] = is_hot ? b : b - S;
    }
  }
  return {hot, all - hot};
}

// One workgroup: T >= E, S and mk. All outputs get their defaults while the policy step's
// loads are in flight (the step's second sync waits for those stores); the ids and the
// blocks' experts are then stored over them, so padding needs no pass of its own.
template <int W>
__global__ __launch_bounds__(W* kWave) void fused_k(EC_STEP_PARAMS, ManageArgs rest, AlignArgs g) {
  constexpr int T = W * kWave;
  __shared__ ManageLds<W, false> L;
  __shared__ AlignLds<W> A;
  const ManageArgs a =
      step_args(ids, step, slot_expert, slot_stamp, table, mk, E, S, rest);
  const int tid = threadIdx.x;
  const int waves = (mk + kWave - 1) / kWave;
  // the alignments' arguments arrive with the step's
  asm volatile("" ::"s"(g.sorted_hot), "s"(g.sorted_cold), "s"(g.eids_hot), "s"(g.eids_cold),
               "s"(g.L), "s"(g.NB), "s"(g.bs), "s"(g.div_mul), "s"(g.div_shift));
  const BlockDiv d(g);
  long long idv;
  const auto early = [&] {
    align_defaults(g, mk, tid, T);
    if (mk > kWave) align_clear<W>(A, waves, S + E);
  };
  manage_step<W, false, 4>(a, L, idv, EarlyStep<decltype(early)>(early));
  lds_sync();
  AlignTotals t;
  if (mk <= kWave) {
    if (wave_index() != 0) return;
    t = align_place_wave(g, S, mk, d, align_key((int)idv, E, S, L.tab));
  } else {
    t = align_place<W, false>(g, A, E, S, d, align_key((int)idv, E, S, L.tab), tid, waves, 0,
                              1);
  }
  if (tid == 0) {
    g.npad_hot[0] = t.hot;
    g.npad_cold[0] = t.cold;
  }
}

// A workgroup per 1024 ids, against the table as it is, over outputs that hold their
// defaults.
__global__ __launch_bounds__(1024) void align_k(const int* ids, int mk, int E, int S,
                                                const int* table, AlignArgs g) {
  constexpr int W = 16, T = W * kWave;
  __shared__ AlignLds<W> A;
  __shared__ unsigned short expert_bucket[T];
  // ids of the other workgroups per expert, before this one's ids and after: four counts of
  // each, by lane, so that a popular expert's ids do not all meet at one address
  __shared__ i32x4 count[2][T];
  const int tid = threadIdx.x, part = blockIdx.x, parts = gridDim.x;
  const unsigned first = part * T;
  const BlockDiv d(g);
  int bucket = -1;  // of expert `tid`
  if (tid < E) {
    const int s = table[tid];
    bucket = (unsigned)s < (unsigned)S ? s : S + tid;
  }
  const int mine = first + tid < (unsigned)mk ? ids[first + tid] : -1;
  align_clear<W>(A, W, S + E);
  A.start[tid] = A.start[T + tid] = A.end[tid] = A.end[T + tid] = 0;
  count[0][tid] = count[1][tid] = i32x4{0, 0, 0, 0};
  lds_sync();
  const int copy = tid & 3;
  auto add = [&](int e, unsigned i) {
    if ((unsigned)e < (unsigned)E)
      atomicAdd(reinterpret_cast<int*>(&count[i < first ? 0 : 1][e]) + copy, 1);
  };
  unsigned done = 0;  // ids counted
  if ((reinterpret_cast<uintptr_t>(ids) & 15) == 0) {
    // four ids a load and four loads in flight; `first` is a multiple of four, and the
    // workgroup's own ids end at a multiple of four or at mk
    const i32x4* v = reinterpret_cast<const i32x4*>(ids);
    const unsigned n = (unsigned)mk / 4;
    for (unsigned i = tid; i < n; i += 4 * T) {
      i32x4 e[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) e[k] = v[min(i + k * T, n - 1)];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const unsigned j = 4 * (i + k * T);
        if (j < 4 * n && (j < first || j >= first + T)) {
          add(e[k].x, j);
          add(e[k].y, j);
          add(e[k].z, j);
          add(e[k].w, j);
        }
      }
    }
    done = 4 * n;
  }
  for (unsigned i = done + tid; i < (unsigned)mk; i += T)
    if (i < first || i >= first + T) add(ids[i], i);
  lds_sync();
  if (bucket >= 0) {
    const i32x4 b = count[0][tid], c = count[1][tid];
    atomicAdd(&A.start[bucket], b.x + b.y + b.z + b.w);
    atomicAdd(&A.end[bucket], c.x + c.y + c.z + c.w);
    expert_bucket[tid] = (unsigned short)bucket;
  }
  lds_sync();
  const int kk = (unsigned)mine < (unsigned)E ? expert_bucket[mine] : -1;
  const AlignTotals t = align_place<W, true>(g, A, E, S, d, kk, first + tid, W, part, parts);
  if (part == 0 && tid == 0) {
    g.npad_hot[0] = t.hot;
    g.npad_cold[0] = t.cold;
  }
}

// The policy step in the launch's first workgroup; the others store the alignments' defaults.
template <int W>
__global__ __launch_bounds__(W* kWave) void manage_defaults_k(EC_STEP_PARAMS, ManageArgs rest,
                                                               AlignArgs g) {
  __shared__ ManageLds<W, false> L;
  const ManageArgs a =
      step_args(ids, step, slot_expert, slot_stamp, table, mk, E, S, rest);
  if (blockIdx.x > 0) {
    align_defaults(g, a.mk, (blockIdx.x - 1) * W * kWave + threadIdx.x,
                   (gridDim.x - 1) * W * kWave);
    return;
  }
  long long idv;
  manage_step<W, false, 4>(a, L, idv);
}

}  // namespace ec
