// Multi-query PFXT: Q independent top-K queries expanded together.
//
// Every query q owns a set of roots and its own bound U_q, histogram
// window and K_q; the node store, the batch and every kernel are shared,
// and a node carries the id of its query.  The queries run on the disjoint
// union of their graphs (batched designs), whose SFXT is each graph's own
// SFXT, so one level loop serves all of them.  Per round, for every query
// at once:
//   1. histograms of its stored paths at or below U_q and of the unexpanded
//      ones (its own kMqBins bins each).  They persist: the count pass adds
//      every child it finds, and the store is only scanned for a query that
//      is new, whose trial fell short or whose window's resolution changed
//      (the scan's two global atomics per stored path, every round, were 5.8
//      of 23 ms for 24 served queries and 3.6 of 14.6 for a batch of 48),
//   2. the batch threshold from its unexpanded paths below U_q,
//   3. a count pass over the batch histogramming its children (< U_q),
//   4. U_q tightened to the top of the bin where the running count of its
//      stored paths and counted children reaches K_q (the bin's upper
//      edge: at least K_q paths cost no more; a per-bin largest key would
//      be tighter by under one of the kMqBins bins, at the price of a
//      second global atomic per counted child, and atomics are performed
//      at memory),
//   5. a fill pass storing its children <= U_q (inclusive: the counted
//      children at U_q are needed).
// A query whose roots' walks are long starts with its roots and a trial bound
// a little above the cheapest (the single query's probe, without its host
// round trips; the others start unbounded, all roots at once): a round
// counts the children of the roots under the trial bound, and if the roots
// and they are fewer than K_q it stores nothing, puts the roots back and
// widens the bound for the next round.  Without a first bound round 0 walks
// every root's whole chain: on a batch of 48 designs the first two rounds
// took 49 ms counting and 11 ms storing of a 67-76 ms run.
// The per-query semantics equal the single-query rounds' (see pfxt.hip);
// the final selection sorts (query, cost, level) so each query's K_q
// results are contiguous.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"
#include "walk.hpp"

namespace cpg {

namespace {

constexpr int kMqBlock = 256;
constexpr int kMqSelBlock = 256;

__device__ inline uint32_t mq_bin(uint32_t k, uint32_t klo, uint32_t shift) {
  if (k < klo) return 0;
  const uint32_t b = (k - klo) >> shift;
  return b < static_cast<uint32_t>(kMqBins) ? b : static_cast<uint32_t>(kMqBins - 1);
}

__device__ inline uint32_t mq_shift(uint32_t klo, uint32_t khi) {
  uint32_t s = 0;
  const uint64_t span = khi >= klo ? static_cast<uint64_t>(khi - klo) : 0;
  while ((span >> s) >= static_cast<uint64_t>(kMqBins)) ++s;
  return s;
}

// Block-wide first bin at which the running sum of h[0..last] reaches
// target; kMqBins if the total is smaller.  *total receives the sum.  (Bins
// past the bound's hold children counted under an older, looser bound.)
__device__ uint32_t mq_crossing(const unsigned* h, uint32_t last, unsigned long long target,
                                unsigned long long* total) {
  constexpr int kPer = kMqBins / kMqSelBlock;
  __shared__ unsigned long long s_part[kMqSelBlock];
  __shared__ unsigned s_bin;
  const int t = threadIdx.x;
  auto at = [&](int i) { return static_cast<uint32_t>(t * kPer + i) <= last ? h[t * kPer + i] : 0u; };
  unsigned long long mine = 0;
  for (int i = 0; i < kPer; ++i) mine += at(i);
  s_part[t] = mine;
  if (t == 0) s_bin = kMqBins;
  __syncthreads();
  for (int off = 1; off < kMqSelBlock; off <<= 1) {
    const unsigned long long v = t >= off ? s_part[t - off] : 0ull;
    __syncthreads();
    s_part[t] += v;
    __syncthreads();
  }
  const unsigned long long incl = s_part[t];
  const unsigned long long excl = incl - mine;
  *total = s_part[kMqSelBlock - 1];
  if (excl < target && incl >= target) {
    unsigned long long run = excl;
    for (int i = 0; i < kPer; ++i) {
      run += at(i);
      if (run >= target) { s_bin = static_cast<uint32_t>(t * kPer + i); break; }
    }
  }
  __syncthreads();
  const uint32_t b = s_bin;
  __syncthreads();
  return b;
}

}  // namespace

__global__ void __launch_bounds__(kMqBlock) mq_roots_kernel(MqArgs a, const int* root_v,
                                                            const int* root_q, int nroots) {
  for (int base = blockIdx.x * blockDim.x; base < nroots; base += gridDim.x * blockDim.x) {
    const int i = base + threadIdx.x;
    const bool take = i < nroots;
    const uint64_t slot = wave_reserve(&a.ctl->node_n, take);
    if (take) {
      const int s = root_v[i];
      const float c = a.distf[s];
      a.nodes.cost[slot] = c;
      a.nodes.to[slot] = s;
      a.nodes.from[slot] = -1;
      a.nodes.parent[slot] = -1;
      a.nodes.level[slot] = 0;
      a.nodes.key[slot] = float_key(c);
      a.nodes.flag[slot] = 0;
      a.nq[slot] = root_q[i];
    }
  }
}

// Opens a round: the counters, and the histograms that are to be counted again.
__global__ void __launch_bounds__(kMqSelBlock) mq_open_kernel(MqArgs a) {
  const int q = blockIdx.x;
  if (q == 0 && threadIdx.x == 0) {
    a.ctl->active = 0;
    a.ctl->batch_n = 0;
  }
  const MqQuery* qs = a.qs + q;
  if (qs->done || !qs->rebuild) return;
  unsigned* h = a.hist + static_cast<size_t>(q) * kMqHistStride;
  for (int j = threadIdx.x; j < kMqHistStride; j += blockDim.x) h[j] = 0u;
  if (threadIdx.x == 0) atomicAdd(&a.ctl->rebuild, 1);
}

// Histograms of the stored paths at or below the bound for the queries that
// count theirs again: nonzero keys, and the unexpanded paths below the bound.
__global__ void __launch_bounds__(kMqBlock) mq_hist_kernel(MqArgs a) {
  if (a.ctl->rebuild == 0) return;
  const uint64_t n = a.ctl->node_n < a.nodes.cap ? a.ctl->node_n : a.nodes.cap;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
    const int q = a.nq[i];
    const MqQuery& qs = a.qs[q];
    if (qs.done || !qs.rebuild) continue;
    const uint32_t k = a.nodes.key[i];
    if (k > qs.ukey) continue;
    const uint32_t b = mq_bin(k, qs.klo, qs.shift);
    unsigned* h = a.hist + static_cast<size_t>(q) * kMqHistStride;
    if (!key_is_zero(k)) atomicAdd(&h[b], 1u);
    if (k < qs.ukey && a.nodes.flag[i] == 0) atomicAdd(&h[kMqBins + b], 1u);
  }
}

// One block per query: the batch threshold (target unexpanded paths below
// the bound); a query with none left is done.  The bins the batch takes are
// cleared.  (The counts may hold a path at the bound itself, which is never
// expanded: that costs a round with nothing to expand, not a missed one.)
__global__ void __launch_bounds__(kMqSelBlock) mq_select_batch_kernel(MqArgs a) {
  const int q = blockIdx.x;
  if (q == 0 && threadIdx.x == 0) a.ctl->rebuild = 0;
  MqQuery* qs = a.qs + q;
  if (qs->done) return;
  unsigned* h = a.hist + static_cast<size_t>(q) * kMqHistStride + kMqBins;
  unsigned long long total = 0;
  const bool take_all = qs->all || qs->trial;
  const uint32_t last = mq_bin(qs->ukey, qs->klo, qs->shift);
  const uint32_t b = mq_crossing(h, last, take_all ? ~0ull : qs->batch_target, &total);
  for (uint32_t j = threadIdx.x; j <= b && j < static_cast<uint32_t>(kMqBins); j += blockDim.x) h[j] = 0u;
  if (threadIdx.x == 0) {
    qs->all = 0;
    qs->rebuild = 0;
    if (total == 0) {
      qs->done = 1;
    } else if (b >= static_cast<uint32_t>(kMqBins)) {
      qs->thkey = qs->ukey;
    } else {
      const uint64_t up = static_cast<uint64_t>(qs->klo) + ((static_cast<uint64_t>(b) + 1) << qs->shift) - 1;
      const uint32_t upk = up > 0xFFFFFFFFull ? 0xFFFFFFFFu : static_cast<uint32_t>(up);
      qs->thkey = upk < qs->ukey ? upk : qs->ukey;
    }
    if (total != 0) atomicAdd(&a.ctl->active, 1);
  }
}

// A block takes tiles of eight slots per thread and reserves a tile's batch
// entries with one atomic (one address for the whole grid).
__global__ void __launch_bounds__(kMqBlock) mq_make_batch_kernel(MqArgs a) {
  const uint64_t n = a.ctl->node_n < a.nodes.cap ? a.ctl->node_n : a.nodes.cap;
  constexpr int kPer = 8;
  constexpr uint64_t kTile = static_cast<uint64_t>(kMqBlock) * kPer;
  for (uint64_t base = static_cast<uint64_t>(blockIdx.x) * kTile; base < n;
       base += static_cast<uint64_t>(gridDim.x) * kTile) {
    const uint64_t i0 = base + threadIdx.x;
    unsigned mask = 0, cnt = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const uint64_t i = i0 + static_cast<uint64_t>(j) * kMqBlock;
      if (i >= n || a.nodes.flag[i] != 0) continue;
      const MqQuery& qs = a.qs[a.nq[i]];
      const uint32_t k = a.nodes.key[i];
      if (!qs.done && k <= qs.thkey && k < qs.ukey) {
        mask |= 1u << j;
        ++cnt;
      }
    }
    uint64_t slot = block_reserve<kMqBlock>(&a.ctl->batch_n, cnt);
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      if (!(mask & (1u << j))) continue;
      const uint64_t i = i0 + static_cast<uint64_t>(j) * kMqBlock;
      a.nodes.flag[i] = 1;
      a.batch[slot++] = static_cast<uint32_t>(i);
    }
  }
}

// Count pass (kFill false): histograms each query's children < U_q, as paths
// and as unexpanded ones.
// Fill pass: stores each query's children <= U_q.
// In the count pass a block counts the children of the query its first
// parent belongs to in an LDS histogram and adds its nonzero bins to the
// query's global histogram at the end of the step: a block's 256
// consecutive batch entries mostly belong to one query (a parent's
// children are stored together), and every global atomic is performed at
// memory.  Parents of other queries count with global atomics.
// In the fill pass a wave stages its children in LDS and stores them with
// one atomic on node_n per kMqStage of them (one address for the whole grid:
// an atomic per wave step bound the pass).
// A block takes one contiguous chunk of the batch, so that one LDS histogram
// serves all of it.
constexpr int kMqStage = 256;
template <bool kFill, int kLanes>
__global__ void __launch_bounds__(kMqBlock) mq_walk_kernel(MqArgs a) {
  __shared__ unsigned s_h[kFill ? 1 : kMqBins];
  __shared__ int s_q;
  constexpr int kW = kMqBlock / 64, kS = kFill ? kMqStage : 1;
  __shared__ float s_cost[kW][kS];
  __shared__ int s_to[kW][kS], s_from[kW][kS], s_parent[kW][kS], s_level[kW][kS], s_nq[kW][kS];
  const int wave = static_cast<int>(threadIdx.x) >> 6, lane = __lane_id();
  int staged = 0;  // wave-uniform
  MqCtl* ctl = a.ctl;
  const uint64_t nb = ctl->batch_n;
  unsigned long long hops = 0, devv = 0, nonmono = 0;
  auto flush = [&]() {
    if (staged == 0) return;
    __builtin_amdgcn_wave_barrier();
    unsigned long long base = 0;
    if (lane == 0) base = atomicAdd(&ctl->node_n, static_cast<unsigned long long>(staged));
    base = __shfl(base, 0);
    for (int j = lane; j < staged; j += 64) {
      const uint64_t slot = base + static_cast<uint64_t>(j);
      if (slot >= a.nodes.cap) {
        atomicExch(&ctl->overflow, 1);
        continue;
      }
      const float cost = s_cost[wave][j];
      a.nodes.cost[slot] = cost;
      a.nodes.to[slot] = s_to[wave][j];
      a.nodes.from[slot] = s_from[wave][j];
      a.nodes.parent[slot] = s_parent[wave][j];
      a.nodes.level[slot] = s_level[wave][j];
      a.nodes.key[slot] = float_key(cost);
      a.nodes.flag[slot] = 0;
      a.nq[slot] = s_nq[wave][j];
    }
    __builtin_amdgcn_wave_barrier();
    staged = 0;
  };
  constexpr uint64_t kParents = kMqBlock / kLanes;  // kLanes lanes per parent
  const uint64_t chunk = ((nb + gridDim.x - 1) / gridDim.x + kParents - 1) / kParents * kParents;
  const uint64_t lo = static_cast<uint64_t>(blockIdx.x) * chunk;
  if (lo >= nb) return;  // block-uniform
  const uint64_t hi = lo + chunk < nb ? lo + chunk : nb;
  if (!kFill) {
    if (threadIdx.x == 0) s_q = a.nq[a.batch[lo]];
    for (int j = threadIdx.x; j < kMqBins; j += blockDim.x) s_h[j] = 0u;
    __syncthreads();
  }
  for (uint64_t base = lo; base < hi; base += kParents) {  // block-uniform
    const uint64_t i = base + threadIdx.x / kLanes;
    int p = 0, lvl = 0, q = 0, to = -1;
    float c = 0.0f;
    MqQuery qs{};
    qs.ukey = kKeyInf;
    if (i < hi) {
      p = static_cast<int>(a.batch[i]);
      c = a.nodes.cost[p];
      to = a.nodes.to[p];
      lvl = a.nodes.level[p];
      q = a.nq[p];
      qs = a.qs[q];
    }
    const bool back = kFill && i < hi && qs.retry;  // a trial that fell short
    if (back) a.nodes.flag[p] = 0;
    const float U = key_float(qs.ukey);
    ChainWalk<kLanes> w;
    w.start(i < hi && !back, c, to, U, qs.ukey != kKeyInf, qs.mag, qs.vrec, qs.devinfo);
    unsigned* h = a.hist + static_cast<size_t>(q) * kMqHistStride;
    const bool local = !kFill && q == s_q;  // count in the block's LDS histogram
    unsigned stored = 0;  // fill: children this lane stored for its parent
    while (__ballot(w.alive)) {
      float cc = 0.0f;
      int cw = 0, from = 0;
      const bool emit = w.step(qs.vrec, qs.devinfo, qs.devs, U, !kFill, qs.step_limit, &ctl->err,
                               &hops, &devv, &nonmono, &cc, &cw, &from);
      if (!kFill) {
        if (emit) {
          const uint32_t k = float_key(cc);
          const uint32_t b = mq_bin(k, qs.klo, qs.shift);
          if (key_is_zero(k)) {  // expanded, never reported
            atomicAdd(&h[kMqBins + b], 1u);
          } else if (local) {
            atomicAdd(&s_h[b], 1u);
          } else {
            atomicAdd(&h[b], 1u);
            atomicAdd(&h[kMqBins + b], 1u);
          }
        }
        continue;
      }
      const uint64_t m = __ballot(emit);
      if (m) {
        const int add = static_cast<int>(__popcll(m));
        if (staged + add > kS) flush();
        if (emit) {
          const int j = staged + static_cast<int>(__popcll(m & lanemask_lt()));
          s_cost[wave][j] = cc;
          s_to[wave][j] = cw;
          s_from[wave][j] = from;
          s_parent[wave][j] = p;
          s_level[wave][j] = lvl + 1;
          s_nq[wave][j] = q;
          ++stored;
        }
        staged += add;
      }
    }
    if (kFill) {
      // per-query stored counts: one atomic per distinct query among the
      // wave's lanes that stored children
      uint64_t pend = __ballot(stored > 0);
      while (pend) {
        const int leader = __ffsll(static_cast<long long>(pend)) - 1;
        const int lq = __shfl(q, leader);
        const bool mine = stored > 0 && q == lq;
        unsigned long long sum = mine ? stored : 0;
        for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
        if (__lane_id() == leader) atomicAdd(&a.qs[lq].stored, sum);
        pend &= ~__ballot(mine);
      }
    }
  }
  if (!kFill) {  // the block's LDS counts into its query's histogram
    __syncthreads();
    unsigned* hq = a.hist + static_cast<size_t>(s_q) * kMqHistStride;
    for (int j = threadIdx.x; j < kMqBins; j += blockDim.x) {
      const unsigned v = s_h[j];
      if (v) {
        atomicAdd(&hq[j], v);
        atomicAdd(&hq[kMqBins + j], v);
      }
    }
  }
  if (kFill) flush();
  (void)hops;
  (void)devv;
  for (int o = 32; o > 0; o >>= 1) nonmono += __shfl_xor(nonmono, o);
  if (kFill && __lane_id() == 0 && nonmono) atomicAdd(&ctl->nonmono, nonmono);  // once per expansion
}

// Next bound of a query whose trial found too few paths (total < K_q).
// Counts grow steeply with the bound: model total ~ gap^alpha, alpha fitted
// to the last two trials (8 at first), aim 5% past K_q and widen by at most
// 1.5x, then 2x: the counts' exponent itself grows with the gap (to ten and
// more on deep graphs), and a trial far too wide walks a hundred times the
// paths of one more narrow trial.  Past every distance without a new path,
// or after kMqTrials, the query goes on unbounded, all its roots at once.
constexpr int kMqTrials = 24;
__device__ inline void mq_widen(MqQuery* qs, unsigned long long total) {
  const double gap = qs->gap;
  qs->retry = 1;
  if (qs->trial >= kMqTrials || (gap > static_cast<double>(qs->mag) && total == qs->prev_total)) {
    qs->trial = 0;
    qs->all = 1;
    qs->ukey = kKeyInf;
    return;
  }
  double alpha = 8.0;
  if (qs->trial > 1 && qs->prev_total > 0 && total > qs->prev_total)
    alpha = fmin(32.0, fmax(1.0, log(static_cast<double>(total) / static_cast<double>(qs->prev_total)) /
                                     log(gap / qs->prev_gap)));
  const double f = pow(static_cast<double>(qs->k) / static_cast<double>(total > 0 ? total : 1ull), 1.0 / alpha) * 1.05;
  const double most = qs->trial == 1 ? 1.5 : 2.0;
  qs->prev_total = total;
  qs->prev_gap = gap;
  qs->gap = gap * fmin(most, fmax(1.05, f));
  qs->trial += 1;
  qs->ukey = float_key(static_cast<float>(static_cast<double>(qs->cmin) + qs->gap));
}

// One block per query: U_q = the upper edge of the bin where the running
// count of stored paths and counted children reaches K_q.
__global__ void __launch_bounds__(kMqSelBlock) mq_select_bound_kernel(MqArgs a) {
  const int q = blockIdx.x;
  MqQuery* qs = a.qs + q;
  if (qs->done) return;
  const unsigned* h = a.hist + static_cast<size_t>(q) * kMqHistStride;
  unsigned long long total = 0;
  const uint32_t b = mq_crossing(h, mq_bin(qs->ukey, qs->klo, qs->shift), qs->k, &total);
  if (threadIdx.x == 0) {
    qs->retry = 0;
    uint32_t uk = qs->ukey;
    if (b < static_cast<uint32_t>(kMqBins)) {
      const uint64_t up = static_cast<uint64_t>(qs->klo) + ((static_cast<uint64_t>(b) + 1) << qs->shift) - 1;
      if (up < uk) uk = static_cast<uint32_t>(up);
      qs->ukey = uk;
      if (!qs->trial && qs->batch_target < qs->target_max)
        qs->batch_target = qs->batch_target * 4 < qs->target_max ? qs->batch_target * 4 : qs->target_max;
      qs->trial = 0;
    } else if (qs->trial) {
      mq_widen(qs, total);
    }
    else if (qs->batch_target < qs->target_max)
      qs->batch_target = qs->batch_target * 4 < qs->target_max ? qs->batch_target * 4 : qs->target_max;
    const uint32_t shift = mq_shift(qs->klo, qs->ukey);
    // children counted but not stored, or another window: count again
    if (qs->retry || shift != qs->shift) qs->rebuild = 1;
    qs->shift = shift;
    qs->rounds += 1;
  }
}

// Sort input: each stored path with a nonzero key <= its query's bound as
// (query << 48 | key << 16 | level) -> node, for the queries sel marks
// (every query when sel is null).
// Blocks take tiles of eight slots per thread, one atomic per tile on the
// path count; the queries' counts gather in LDS while there are at most
// kMqLdsQ of them (a wave's taken nodes of one query add together).
constexpr int kMqLdsQ = 1024;
__global__ void __launch_bounds__(kMqBlock) mq_build_keys_kernel(MqArgs a, const uint8_t* sel,
                                                                 uint64_t* key, uint32_t* val,
                                                                 unsigned long long* count,
                                                                 unsigned long long* per_q) {
  __shared__ unsigned s_cnt[kMqLdsQ];
  const bool lds = a.nq_count <= kMqLdsQ;
  for (int j = threadIdx.x; j < kMqLdsQ; j += blockDim.x) s_cnt[j] = 0;
  __syncthreads();
  const uint64_t n = a.ctl->node_n < a.nodes.cap ? a.ctl->node_n : a.nodes.cap;
  constexpr int kPer = 8;
  constexpr uint64_t kTile = static_cast<uint64_t>(kMqBlock) * kPer;
  for (uint64_t base = static_cast<uint64_t>(blockIdx.x) * kTile; base < n;
       base += static_cast<uint64_t>(gridDim.x) * kTile) {
    const uint64_t i0 = base + threadIdx.x;
    unsigned mask = 0, cnt = 0;
    uint32_t ks[kPer];
    int qv[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const uint64_t i = i0 + static_cast<uint64_t>(j) * kMqBlock;
      ks[j] = 0;
      qv[j] = 0;
      bool take = false;
      if (i < n) {
        qv[j] = a.nq[i];
        ks[j] = a.nodes.key[i];
        take = (!sel || sel[qv[j]]) && ks[j] <= a.qs[qv[j]].ukey && !key_is_zero(ks[j]);
      }
      if (take) {
        mask |= 1u << j;
        ++cnt;
      }
      uint64_t pend = __ballot(take);
      while (pend) {
        const int leader = __ffsll(static_cast<long long>(pend)) - 1;
        const int lq = __shfl(qv[j], leader);
        const uint64_t peers = __ballot(take && qv[j] == lq);
        if (__lane_id() == leader) {
          if (lds) atomicAdd(&s_cnt[lq], static_cast<unsigned>(__popcll(peers)));
          else atomicAdd(&per_q[lq], static_cast<unsigned long long>(__popcll(peers)));
        }
        pend &= ~peers;
      }
    }
    uint64_t slot = block_reserve<kMqBlock>(count, cnt);
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      if (!(mask & (1u << j))) continue;
      const uint64_t i = i0 + static_cast<uint64_t>(j) * kMqBlock;
      key[slot] = (static_cast<uint64_t>(qv[j]) << 48) | (static_cast<uint64_t>(ks[j]) << 16) |
                  static_cast<uint32_t>(a.nodes.level[i] & 0xffff);
      val[slot] = static_cast<uint32_t>(i);
      ++slot;
    }
  }
  __syncthreads();
  if (lds)
    for (int j = threadIdx.x; j < a.nq_count; j += blockDim.x)
      if (s_cnt[j]) atomicAdd(&per_q[j], static_cast<unsigned long long>(s_cnt[j]));
}

// Compaction of the shared node store (served queries): a node is live
// while its query's slot is not done.  Tiles of kCompactTile nodes keep
// their order; parents are remapped through newidx afterwards.
constexpr int kCompactChunks = 16;
constexpr int kCompactTile = kMqBlock * kCompactChunks;

__global__ void __launch_bounds__(kMqBlock) mq_count_live_kernel(MqArgs a, uint64_t n,
                                                                 unsigned* tile_cnt) {
  __shared__ unsigned s_cnt;
  if (threadIdx.x == 0) s_cnt = 0;
  __syncthreads();
  const uint64_t t = blockIdx.x;
  unsigned c = 0;
  for (int j = 0; j < kCompactChunks; ++j) {
    const uint64_t i = t * kCompactTile + static_cast<uint64_t>(j) * kMqBlock + threadIdx.x;
    if (i < n && !a.qs[a.nq[i]].done) ++c;
  }
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
  if (__lane_id() == 0) atomicAdd(&s_cnt, c);
  __syncthreads();
  if (threadIdx.x == 0) tile_cnt[t] = s_cnt;
}

__global__ void __launch_bounds__(kMqBlock) mq_compact_kernel(MqArgs a, uint64_t n, NodeStore dst,
                                                              int* dst_nq, const unsigned* tile_off,
                                                              int* newidx) {
  constexpr int kW = kMqBlock / 64;
  __shared__ unsigned s_wave[kW];
  __shared__ unsigned s_run;
  const int lane = __lane_id(), wave = threadIdx.x >> 6;
  if (threadIdx.x == 0) s_run = 0;
  __syncthreads();
  const uint64_t t = blockIdx.x;
  const uint64_t base = tile_off[t];
  for (int j = 0; j < kCompactChunks; ++j) {
    const uint64_t i = t * kCompactTile + static_cast<uint64_t>(j) * kMqBlock + threadIdx.x;
    int q = 0;
    bool live = false;
    if (i < n) {
      q = a.nq[i];
      live = !a.qs[q].done;
    }
    const uint64_t m = __ballot(live);
    const unsigned rank = static_cast<unsigned>(__popcll(m & lanemask_lt()));
    if (lane == 0) s_wave[wave] = static_cast<unsigned>(__popcll(m));
    __syncthreads();
    unsigned off = s_run;
    for (int w = 0; w < wave; ++w) off += s_wave[w];
    if (live) {
      const uint64_t d = base + off + rank;
      dst.cost[d] = a.nodes.cost[i];
      dst.to[d] = a.nodes.to[i];
      dst.from[d] = a.nodes.from[i];
      dst.parent[d] = a.nodes.parent[i];
      dst.level[d] = a.nodes.level[i];
      dst.key[d] = a.nodes.key[i];
      dst.flag[d] = a.nodes.flag[i];
      dst_nq[d] = q;
      newidx[i] = static_cast<int>(d);
    } else if (i < n) {
      newidx[i] = -1;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      unsigned tot = 0;
      for (int w = 0; w < kW; ++w) tot += s_wave[w];
      s_run += tot;
    }
    __syncthreads();
  }
}

// Appends a single-query node store's first cnt paths (a
// query's roots) at dst[base..) for query slot q, parents shifted.
__global__ void mq_seed_kernel(NodeStore src, uint64_t cnt, NodeStore dst, int* dst_nq,
                               uint64_t base, int q) {
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < cnt;
       i += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
    const uint64_t d = base + i;
    const int p = src.parent[i];
    dst.cost[d] = src.cost[i];
    dst.to[d] = src.to[i];
    dst.from[d] = src.from[i];
    dst.parent[d] = p < 0 ? -1 : static_cast<int>(base + static_cast<uint64_t>(p));
    dst.level[d] = src.level[i];
    dst.key[d] = src.key[i];
    dst.flag[d] = src.flag[i];
    dst_nq[d] = q;
  }
}

__global__ void mq_set_node_n_kernel(MqCtl* ctl, unsigned long long n) { ctl->node_n = n; }

__global__ void mq_remap_parents_kernel(int* parent, const int* newidx, uint64_t n) {
  for (uint64_t j = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; j < n;
       j += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
    const int p = parent[j];
    if (p >= 0) parent[j] = newidx[p];
  }
}

__global__ void mq_gather_costs_kernel(const uint32_t* val, const float* cost, uint64_t n,
                                       float* out) {
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<uint64_t>(gridDim.x) * blockDim.x)
    out[i] = cost[val[i]];
}

__global__ void zero_u32_kernel(unsigned* p, uint64_t n) {
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<uint64_t>(gridDim.x) * blockDim.x)
    p[i] = 0;
}

void launch_zero_u32(unsigned* p, uint64_t n, hipStream_t s) {
  if (n == 0) return;
  const uint64_t g = std::min<uint64_t>(1024, (n + 255) / 256);
  hipLaunchKernelGGL(zero_u32_kernel, dim3(static_cast<unsigned>(g)), dim3(256), 0, s, p, n);
  CPG_HIP(hipGetLastError());
}

void launch_mq_roots(const MqArgs& a, const int* root_v, const int* root_q, int nroots, hipStream_t s) {
  if (nroots <= 0) return;
  hipLaunchKernelGGL(mq_roots_kernel, dim3((nroots + kMqBlock - 1) / kMqBlock), dim3(kMqBlock), 0, s,
                     a, root_v, root_q, nroots);
  CPG_HIP(hipGetLastError());
}

void launch_mq_round(const MqArgs& a, int grid, hipStream_t s) {
  hipLaunchKernelGGL(mq_open_kernel, dim3(a.nq_count), dim3(kMqSelBlock), 0, s, a);
  CPG_HIP(hipGetLastError());
  hipLaunchKernelGGL(mq_hist_kernel, dim3(grid), dim3(kMqBlock), 0, s, a);
  CPG_HIP(hipGetLastError());
  hipLaunchKernelGGL(mq_select_batch_kernel, dim3(a.nq_count), dim3(kMqSelBlock), 0, s, a);
  CPG_HIP(hipGetLastError());
  hipLaunchKernelGGL(mq_make_batch_kernel, dim3(grid), dim3(kMqBlock), 0, s, a);
  CPG_HIP(hipGetLastError());
  // four lanes per parent: a batch of 48 designs took 20.8 / 18.3 / 17.3 / 17.5
  // ms with 1 / 2 / 4 / 8, 24 served queries 35.3 / 33.6 / 33.1 / 34.8
  hipLaunchKernelGGL((mq_walk_kernel<false, 4>), dim3(grid), dim3(kMqBlock), 0, s, a);
  CPG_HIP(hipGetLastError());
  hipLaunchKernelGGL(mq_select_bound_kernel, dim3(a.nq_count), dim3(kMqSelBlock), 0, s, a);
  CPG_HIP(hipGetLastError());
  hipLaunchKernelGGL((mq_walk_kernel<true, 4>), dim3(grid), dim3(kMqBlock), 0, s, a);
  CPG_HIP(hipGetLastError());
}

void launch_mq_build_keys(const MqArgs& a, const uint8_t* sel, uint64_t nmax, uint64_t* key,
                          uint32_t* val, unsigned long long* count, unsigned long long* per_q,
                          int grid, hipStream_t s) {
  if (nmax == 0) return;
  hipLaunchKernelGGL(mq_build_keys_kernel, dim3(grid), dim3(kMqBlock), 0, s, a, sel, key, val,
                     count, per_q);
  CPG_HIP(hipGetLastError());
}

uint64_t mq_compact_tiles(uint64_t n) { return (n + kCompactTile - 1) / kCompactTile; }

void launch_mq_seed(const NodeStore& src, uint64_t cnt, const NodeStore& dst, int* dst_nq,
                    uint64_t base, int q, MqCtl* ctl, int grid, hipStream_t s) {
  if (cnt > 0) {
    hipLaunchKernelGGL(mq_seed_kernel, dim3(grid), dim3(kMqBlock), 0, s, src, cnt, dst, dst_nq, base, q);
    CPG_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL(mq_set_node_n_kernel, dim3(1), dim3(1), 0, s, ctl,
                     static_cast<unsigned long long>(base + cnt));
  CPG_HIP(hipGetLastError());
}

void launch_mq_count_live(const MqArgs& a, uint64_t n, unsigned* tile_cnt, hipStream_t s) {
  const uint64_t nt = mq_compact_tiles(n);
  if (nt == 0) return;
  hipLaunchKernelGGL(mq_count_live_kernel, dim3(static_cast<unsigned>(nt)), dim3(kMqBlock), 0, s, a,
                     n, tile_cnt);
  CPG_HIP(hipGetLastError());
}

void launch_mq_compact(const MqArgs& a, uint64_t n, const NodeStore& dst, int* dst_nq,
                       const unsigned* tile_off, int* newidx, uint64_t n_live, int grid,
                       hipStream_t s) {
  const uint64_t nt = mq_compact_tiles(n);
  if (nt == 0) return;
  hipLaunchKernelGGL(mq_compact_kernel, dim3(static_cast<unsigned>(nt)), dim3(kMqBlock), 0, s, a, n,
                     dst, dst_nq, tile_off, newidx);
  CPG_HIP(hipGetLastError());
  if (n_live == 0) return;
  hipLaunchKernelGGL(mq_remap_parents_kernel, dim3(grid), dim3(kMqBlock), 0, s, dst.parent, newidx,
                     n_live);
  CPG_HIP(hipGetLastError());
}

void launch_mq_gather_costs(const uint32_t* val, const float* cost, uint64_t n, float* out,
                            hipStream_t s) {
  if (n == 0) return;
  const uint64_t g = std::min<uint64_t>(4096, (n + 255) / 256);
  hipLaunchKernelGGL(mq_gather_costs_kernel, dim3(static_cast<unsigned>(g)), dim3(256), 0, s, val,
                     cost, n, out);
  CPG_HIP(hipGetLastError());
}

}  // namespace cpg
