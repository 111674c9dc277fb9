// PFXT: exact top-K prefix-tree expansion in bounded best-first rounds.
//
// A path is a root (a source followed by its suffix chain,
// gpucpg/gpucpg.cu:18502-18513) or a parent plus one deviation edge u->w
// taken at a vertex u of the parent's suffix chain, with cost
//   ((parent + distf[w]) + w_e) - distf[u]
// evaluated left to right in binary32 exactly as
// compute_short_long_path_counts / expand_short_pile do
// (gpucpg/gpucpg.cu:2670-2676, :3271-3276).
//
// Instead of the reference's short/long piles and split schedule
// (gpucpg/gpucpg.cu:19134-21228), every generated path stays in the node
// store with its orderable cost key and an expanded flag, and each round
//   1. histograms the stored paths at or below the bound U (all nonzero
//      ones, and the unexpanded ones),
//   2. picks the cheapest unexpanded paths as the batch (histogram select),
//   3. walks their suffix chains and stores every child with cost <= U,
//   4. tightens U to the K-th smallest nonzero cost among the stored paths
//      (histogram of the old paths plus the new children).
// While U is unbounded a count pass histograms the children before the
// fill pass stores them, so that only paths at or below the tightened U
// are stored.  U is always the upper end of the histogram bin where the
// running count of K distinct stored paths is reached, so no path of the
// final top K lies above it while child cost >= parent cost.
// The walk skips chain segments via the deviation index built by the SFXT:
// a vertex whose smallest deviation delta exceeds X = (U - parent) + slack
// is skipped through its next-smaller pointer and its sorted deviation
// list is cut at the first delta > X.  slack bounds the rounding gap
// between delta and the binary32 cost recurrence, so the skip never hides
// a child whose computed cost is <= U; the exact comparison cost <= U
// decides emission.
#include "common.hpp"
#include "kernels.hpp"
#include "walk.hpp"

namespace cpg {

namespace {

constexpr int kBlock = 256;
constexpr int kSelBlock = 1024;
constexpr int kHistBlock = 1024;

// Block-wide search for the first bin at which the running sum of h (words
// other blocks of the launch wrote) reaches target (1-based count).  Returns
// kHistBins if the total is smaller; *total receives the sum.  Must be called
// by all threads of a kSelBlock block.
__device__ uint32_t find_crossing(const unsigned* h, unsigned long long target,
                                  unsigned long long* total) {
  constexpr int kPer = kHistBins / kSelBlock, kW = kSelBlock / 64;
  __shared__ unsigned s_wave[kW];
  __shared__ unsigned s_bin;
  const int t = threadIdx.x, lane = __lane_id(), wave = t >> 6;
  // 32-bit sums: a node store holds fewer than 2^31 paths (ensure_pfxt_buffers
  // refuses more), and a count pass adds at most as many keys (ckeys_cap)
  unsigned v[kPer], mine = 0;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    v[i] = dev_load(h + t * kPer + i);
    mine += v[i];
  }
  unsigned incl = mine;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned x = __shfl_up(incl, o);
    if (lane >= o) incl += x;
  }
  if (lane == 63) s_wave[wave] = incl;
  if (t == 0) s_bin = kHistBins;
  __syncthreads();
  unsigned before = 0, sum = 0;
#pragma unroll
  for (int w = 0; w < kW; ++w) {
    const unsigned x = s_wave[w];
    if (w < wave) before += x;
    sum += x;
  }
  *total = sum;
  unsigned long long run = before + incl - mine;
  if (run < target && run + mine >= target) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      if (run < target && run + v[i] >= target) s_bin = static_cast<uint32_t>(t * kPer + i);
      run += v[i];
    }
  }
  __syncthreads();
  const uint32_t b = s_bin;
  __syncthreads();
  return b;
}

__global__ void __launch_bounds__(kBlock) roots_kernel(const int* srcs, const uint8_t* keep, int nsrc,
                                                       const int* dist, const float* distf,
                                                       NodeStore nodes, PfxtCtl* ctl) {
  for (int base = blockIdx.x * blockDim.x; base < nsrc; base += gridDim.x * blockDim.x) {
    const int i = base + threadIdx.x;
    bool take = false;
    int s = 0;
    if (i < nsrc) {
      s = srcs[i];
      take = keep[i] != 0 && dist[s] != kIntMax;
    }
    const uint64_t slot = wave_reserve(&ctl->node_n, take);
    if (take) {
      const float c = distf[s];
      nodes.cost[slot] = c;
      nodes.to[slot] = s;
      nodes.from[slot] = -1;
      nodes.parent[slot] = -1;
      nodes.level[slot] = 0;
      nodes.key[slot] = float_key(c);
      nodes.flag[slot] = 0;
    }
  }
}

// Slots one histogram pass covers: every stored path, this round's children,
// or the keys a count pass wrote; [lo, nn) lies within the buffer (after a
// node-store overflow node_n and fill_node_base exceed the capacity, and the
// vector loop reads the group of four holding lo, so lo must not pass nn).
__device__ inline void hist_range(const PfxtCtl* ctl, int mode, uint64_t cap, uint64_t ckeys_cap, uint64_t& lo,
                                  uint64_t& nn) {
  lo = 0;
  if (mode == 2) {
    const uint64_t c = ctl->child_n;
    nn = c < ckeys_cap ? c : ckeys_cap;
  } else {
    const uint64_t c = ctl->node_n;
    nn = c < cap ? c : cap;
    if (mode == 1) {
      const uint64_t b = ctl->fill_node_base;
      lo = b < nn ? b : nn;
    }
  }
}

// Blocks that take part in a pass over that many slots: each leaves one
// partial histogram of 48 KB, which the reduction reads again, so a small
// store uses few (8,192 slots per block; one block up to there).
constexpr uint64_t kHistChunk = 8192;
__device__ inline unsigned hist_parts(uint64_t lo, uint64_t nn) {
  const uint64_t p = (nn - lo + kHistChunk - 1) / kHistChunk;
  return static_cast<unsigned>(p < 1 ? 1 : p > kHistParts ? kHistParts : p);
}

// Per-block histograms over the window (klo, shift), counted in LDS and
// written out as one partial per block: the nonzero keys <= U with the
// largest key of each bin, and (with_pend) the unexpanded paths with key
// < U (those still to be expanded).  mode 0 covers every stored path,
// mode 1 this round's children only, mode 2 the keys a count pass wrote
// (ckeys, no flags).  Each thread reads four consecutive keys and flags
// with one vector load each (the arrays are padded to a multiple of four
// slots).
__global__ void __launch_bounds__(kHistBlock) hist_nodes_kernel(NodeStore nodes, const uint32_t* ckeys,
                                                                uint64_t ckeys_cap, const PfxtCtl* ctl,
                                                                int mode, int with_pend,
                                                                unsigned* part_all, unsigned* part_pend,
                                                                unsigned* part_max) {
  __shared__ unsigned h_all[kHistBins];
  __shared__ unsigned h_pend[kHistBins];
  __shared__ unsigned h_max[kHistBins];
  if (ctl->done) return;
  uint64_t lo, nn;
  hist_range(ctl, mode, nodes.cap, ckeys_cap, lo, nn);
  const unsigned parts = hist_parts(lo, nn);
  if (blockIdx.x >= parts) return;
  for (int j = threadIdx.x; j < kHistBins; j += blockDim.x) {
    h_all[j] = 0;
    h_max[j] = 0;
    if (with_pend) h_pend[j] = 0;
  }
  __syncthreads();
  const uint32_t uk = ctl->ukey;
  const uint32_t klo = ctl->klo, shift = ctl->shift;
  const uint4* key4 = reinterpret_cast<const uint4*>(mode == 2 ? ckeys : nodes.key);
  const uint32_t* flag4 = reinterpret_cast<const uint32_t*>(nodes.flag);
  for (uint64_t g = lo / 4 + static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
       g < (nn + 3) / 4; g += static_cast<uint64_t>(parts) * blockDim.x) {
    const uint4 kv = key4[g];
    const uint32_t fv = with_pend ? flag4[g] : 0u;
    const uint32_t ks[4] = {kv.x, kv.y, kv.z, kv.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint64_t i = 4 * g + q;
      const uint32_t k = ks[q];
      if (i < lo || i >= nn || k > uk) continue;
      const uint32_t b = key_bin(k, klo, shift);
      if (!key_is_zero(k)) {
        atomicAdd(&h_all[b], 1u);
        atomicMax(&h_max[b], k);
      }
      if (with_pend && k < uk && ((fv >> (8 * q)) & 0xffu) == 0) atomicAdd(&h_pend[b], 1u);
    }
  }
  __syncthreads();
  const size_t at = static_cast<size_t>(blockIdx.x) * kHistBins;
  for (int j = threadIdx.x; j < kHistBins; j += blockDim.x) {
    part_all[at + j] = h_all[j];
    part_max[at + j] = h_max[j];
    if (with_pend) part_pend[at + j] = h_pend[j];
  }
}

// Sums the pass's partials into hist_all (and hist_pend), takes the maximum of
// the per-bin largest keys, combined with what is there when accumulate and
// written over it otherwise; then the last block to finish makes the choice
// (HistSelect).  A block of kSelBlock threads covers 64 bins of one plane
// (blockIdx.y: counts, largest keys, unexpanded): its 16 groups of 64 lanes
// add an interleaved share of the partials and meet in LDS.  What was a
// reduction per plane and a one-block selection, four launches of about 3 us
// each, twice a round, is one: on a 5K-vertex query the two kinds of kernels
// took 330 of 850 us.
__global__ void __launch_bounds__(kSelBlock) reduce_select_kernel(const unsigned* part, unsigned* hist_all,
                                                                  unsigned* hist_pend, PfxtCtl* ctl, uint64_t cap,
                                                                  uint64_t ckeys_cap, int mode, int accumulate,
                                                                  int select, unsigned long long target,
                                                                  unsigned long long nroots) {
  constexpr int kGroups = kSelBlock / 64;
  __shared__ unsigned s_sum[kGroups][64];
  __shared__ int s_last;
  if (ctl->done) return;
  const size_t plane = static_cast<size_t>(kHistParts) * kHistBins;
  uint64_t lo, nn;
  hist_range(ctl, mode, cap, ckeys_cap, lo, nn);
  const unsigned parts = hist_parts(lo, nn);
  const int lane = threadIdx.x & 63, grp = threadIdx.x >> 6;
  const int j = blockIdx.x * 64 + lane;
  const bool take_max = blockIdx.y == 1;
  // planes of part: counts, unexpanded, largest keys
  const unsigned* src = part + (blockIdx.y == 0 ? 0 : blockIdx.y == 1 ? 2 * plane : plane);
  unsigned* out = blockIdx.y == 0 ? hist_all : blockIdx.y == 1 ? hist_all + kHistBins : hist_pend;
  unsigned sum = 0;
#pragma unroll 4
  for (unsigned q = static_cast<unsigned>(grp); q < parts; q += kGroups) {
    const unsigned v = src[static_cast<size_t>(q) * kHistBins + j];
    sum = take_max ? max(sum, v) : sum + v;
  }
  s_sum[grp][lane] = sum;
  __syncthreads();
  if (grp == 0) {
    unsigned tot = accumulate ? out[j] : 0u;
#pragma unroll
    for (int g2 = 0; g2 < kGroups; ++g2) tot = take_max ? max(tot, s_sum[g2][lane]) : tot + s_sum[g2][lane];
    dev_store(out + j, tot);
    __builtin_amdgcn_s_waitcnt(0);  // landed before this block is counted
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned n = gridDim.x * gridDim.y;
    s_last = __hip_atomic_fetch_add(&ctl->ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n - 1;
  }
  __syncthreads();
  if (!s_last) return;
  unsigned long long total = 0;
  const uint32_t b = find_crossing(select == kSelectBatch ? hist_pend : hist_all, target, &total);
  if (threadIdx.x != 0) return;
  ctl->ticket = 0;
  const uint32_t uk = ctl->ukey;
  if (select == kSelectBatch) {
    ctl->batch_n = 0;
    ctl->child_n = 0;
    ctl->fill_node_base = ctl->node_n;
    if (total == 0) {
      ctl->done = 1;
    } else if (b >= static_cast<uint32_t>(kHistBins)) {
      ctl->thkey = uk;
    } else {
      const uint32_t up = bin_upper_key(b, ctl->klo, ctl->shift);
      ctl->thkey = up < uk ? up : uk;
    }
    return;
  }
  uint32_t nk = uk;
  if (b < static_cast<uint32_t>(kHistBins)) {
    const uint32_t top = dev_load(hist_all + kHistBins + b);  // largest key in the crossing bin
    if (top < nk) nk = top;
  }
  ctl->ukey = nk;
  ctl->shift = window_shift(ctl->klo, nk);
  if (select == kSelectBound) {
    ctl->expanded += ctl->batch_n;
    ctl->rounds += 1;
  } else {  // a probe's bound: at least target nonzero paths are stored, the roots count as expanded
    ctl->batch_n = 0;
    ctl->child_n = 0;
    ctl->expanded += nroots;
  }
}

// Marks the stored paths with key <= thkey and < U that are not expanded
// yet and appends them to the batch; one counter atomic per block and tile.
// A path at U itself is not expanded: at least K stored paths cost <= U,
// so its children (cost >= U) cannot change the K smallest costs.  A tile is
// 8,192 slots, taken 2,048 at a time, eight consecutive ones per thread (two
// 16-byte key loads, one 8-byte flag load): the counter is one address, about
// 10 ns an atomic, and 2,048-slot tiles made it the bound (16.9 us at 4M
// slots).
__global__ void __launch_bounds__(kBlock) make_batch_kernel(NodeStore nodes, PfxtCtl* ctl,
                                                            uint32_t* batch) {
  if (ctl->done) return;
  const uint64_t n = ctl->node_n < nodes.cap ? ctl->node_n : nodes.cap;
  const uint32_t th = ctl->thkey, uk = ctl->ukey;
  constexpr int kSub = 4;
  constexpr uint64_t kStep = static_cast<uint64_t>(kBlock) * 8, kTile = kStep * kSub;
  const uint4* key4 = reinterpret_cast<const uint4*>(nodes.key);
  const uint2* flag8 = reinterpret_cast<const uint2*>(nodes.flag);
  for (uint64_t base = static_cast<uint64_t>(blockIdx.x) * kTile; base < n;
       base += static_cast<uint64_t>(gridDim.x) * kTile) {
    const uint64_t i0 = base + 8ull * threadIdx.x;
    uint32_t mask = 0;  // byte s: the thread's slots of step s
#pragma unroll
    for (int s = 0; s < kSub; ++s) {
      const uint64_t i = i0 + s * kStep;
      if (i >= n) continue;
      const uint4 ka = key4[i / 4], kb = key4[i / 4 + 1];
      const uint2 fv = flag8[i / 8];
      const uint32_t ks[8] = {ka.x, ka.y, ka.z, ka.w, kb.x, kb.y, kb.z, kb.w};
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const uint32_t f = ((q < 4 ? fv.x : fv.y) >> (8 * (q & 3))) & 0xffu;
        if (i + q < n && f == 0 && ks[q] <= th && ks[q] < uk) mask |= 1u << (8 * s + q);
      }
    }
    uint64_t slot = block_reserve<kBlock>(&ctl->batch_n, static_cast<unsigned>(__popcll(mask)));
    for (; mask; mask &= mask - 1) {
      const int j = __ffsll(static_cast<long long>(mask)) - 1;
      const uint64_t i = i0 + static_cast<uint64_t>(j >> 3) * kStep + static_cast<uint64_t>(j & 7);
      nodes.flag[i] = 1;
      batch[slot++] = static_cast<uint32_t>(i);
    }
  }
}

constexpr int kStage = 256;  // per-wave LDS slots for children awaiting a flush

// Walks the suffix chains of the batch's parents and finds every child
// with cost < U (cost <= U when a.strict == 0).  Count pass (kFill =
// false): write the children's keys to ckeys and count them in child_n
// (hist_nodes_kernel mode 2 histograms them).  Fill pass: append them to
// the node store, unexpanded.  Children are staged per wave in LDS and
// written with one counter atomic per flush.
template <bool kFill, int kLanes>
__global__ void __launch_bounds__(kBlock) walk_kernel(WalkArgs a) {
  constexpr int kParents = kBlock / kLanes;  // kLanes lanes per parent
  constexpr int kWaves = kBlock / 64;
  constexpr int kS = kStage;
  constexpr int kSF = kFill ? kStage : 1;  // node fields are staged by the fill pass only
  __shared__ float s_cost[kWaves][kS];
  __shared__ int s_to[kWaves][kSF];
  __shared__ int s_from[kWaves][kSF];
  __shared__ int s_parent[kWaves][kSF];
  __shared__ int s_level[kWaves][kSF];
  PfxtCtl* ctl = a.ctl;
  if (ctl->done) return;
  const int wave = threadIdx.x >> 6;
  const int lane = __lane_id();
  const uint64_t nb = ctl->batch_n;
  const uint32_t ukey = ctl->ukey;
  const bool bounded = ukey != kKeyInf;
  const float U = key_float(ukey);
  const uint64_t cap = a.nodes.cap;
  const float mag = 2.0f * a.max_abs_distf + a.max_abs_wgt + 1.0f;
  unsigned long long hops = 0, devv = 0, nonmono = 0;
  int staged = 0;  // wave-uniform

  // Writes the wave's staged children: one atomic on node_n (fill) or
  // child_n (count: keys only, into ckeys), then each lane stores every
  // 64th child.  All lanes of the wave call it together.
  auto flush = [&]() {
    if (staged == 0) return;
    __builtin_amdgcn_wave_barrier();
    unsigned long long base = 0;
    if (lane == 0)
      base = atomicAdd(kFill ? &ctl->node_n : &ctl->child_n, static_cast<unsigned long long>(staged));
    base = __shfl(base, 0);
    if (!kFill) {
      for (int q = lane; q < staged; q += 64)
        if (base + q < a.ckeys_cap) a.ckeys[base + q] = float_key(s_cost[wave][q]);
      __builtin_amdgcn_wave_barrier();
      staged = 0;
      return;
    }
    for (int q = lane; q < staged; q += 64) {
      const uint64_t slot = base + q;
      const float cost = s_cost[wave][q];
      if (slot < cap) {
        a.nodes.cost[slot] = cost;
        a.nodes.to[slot] = s_to[wave][q];
        a.nodes.from[slot] = s_from[wave][q];
        a.nodes.parent[slot] = s_parent[wave][q];
        a.nodes.level[slot] = s_level[wave][q];
        a.nodes.key[slot] = float_key(cost);
        a.nodes.flag[slot] = 0;
      } else {
        atomicExch(&ctl->overflow, 1);
      }
    }
    __builtin_amdgcn_wave_barrier();
    staged = 0;
  };

  for (uint64_t base = static_cast<uint64_t>(blockIdx.x) * kParents; base < nb;
       base += static_cast<uint64_t>(gridDim.x) * kParents) {
    const uint64_t i = base + threadIdx.x / kLanes;
    int p = 0, lvl = 0;
    float c = 0.0f;
    int to = -1;
    if (i < nb) {
      p = static_cast<int>(a.batch[i]);
      c = a.nodes.cost[p];
      to = a.nodes.to[p];
      lvl = a.nodes.level[p];
    }
    ChainWalk<kLanes> cw_state;
    cw_state.start(i < nb, c, to, U, bounded, mag, a.vrec, a.devinfo);
    while (__ballot(cw_state.alive)) {
      float cc = 0.0f;
      int cw = 0, from = 0;
      const bool emit = cw_state.step(a.vrec, a.devinfo, a.devs, U, a.strict != 0, a.step_limit,
                                      &ctl->err, &hops, &devv, &nonmono, &cc, &cw, &from);
      const uint64_t m = __ballot(emit);
      if (m) {
        const int add = static_cast<int>(__popcll(m));
        if (staged + add > kS) flush();
        if (emit) {
          const int q = staged + static_cast<int>(__popcll(m & lanemask_lt()));
          s_cost[wave][q] = cc;
          if (kFill) {
            s_to[wave][q] = cw;
            s_from[wave][q] = from;
            s_parent[wave][q] = p;
            s_level[wave][q] = lvl + 1;
          }
        }
        staged += add;
      }
    }
  }
  flush();
  for (int o = 32; o > 0; o >>= 1) nonmono += __shfl_xor(nonmono, o);
  if (kFill && lane == 0 && nonmono) atomicAdd(&ctl->nonmono, nonmono);  // once per expansion
  if (a.collect_stats) {
    for (int o = 32; o > 0; o >>= 1) {
      hops += __shfl_xor(hops, o);
      devv += __shfl_xor(devv, o);
    }
    if (lane == 0) {
      atomicAdd(&ctl->hops, hops);
      atomicAdd(&ctl->devvis, devv);
    }
  }
}

// Bound probe: the walk's inputs for one trial bound ukey over the roots
// (node slots 0..nroots-1, listed in batch by iota_kernel); the node store
// is cut back to the roots, dropping an earlier trial's children.
__global__ void probe_setup_kernel(PfxtCtl* ctl, uint32_t ukey, uint32_t shift,
                                   unsigned long long nb, unsigned long long nroots) {
  ctl->ukey = ukey;
  ctl->shift = shift;
  ctl->batch_n = nb;
  ctl->child_n = 0;
  ctl->done = 0;
  ctl->node_n = nroots;
  ctl->fill_node_base = nroots;
  ctl->overflow = 0;
}

__global__ void iota_kernel(uint32_t* p, uint64_t n) {
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<uint64_t>(gridDim.x) * blockDim.x)
    p[i] = static_cast<uint32_t>(i);
}

}  // namespace

void launch_roots(const int* srcs, const uint8_t* keep, int nsrc, const int* dist,
                  const float* distf, NodeStore nodes, PfxtCtl* ctl, hipStream_t s) {
  if (nsrc <= 0) return;
  const int grid = (nsrc + kBlock - 1) / kBlock;
  hipLaunchKernelGGL(roots_kernel, dim3(grid), dim3(kBlock), 0, s, srcs, keep, nsrc, dist, distf,
                     nodes, ctl);
  CPG_HIP(hipGetLastError());
}

void launch_probe_setup(PfxtCtl* ctl, uint32_t ukey, uint32_t shift, unsigned long long nb,
                        unsigned long long nroots, hipStream_t s) {
  hipLaunchKernelGGL(probe_setup_kernel, dim3(1), dim3(1), 0, s, ctl, ukey, shift, nb, nroots);
  CPG_HIP(hipGetLastError());
}

void launch_iota(uint32_t* p, uint64_t n, int grid, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(iota_kernel, dim3(grid), dim3(kBlock), 0, s, p, n);
  CPG_HIP(hipGetLastError());
}

void launch_hist_select(const NodeStore& nodes, const uint32_t* ckeys, uint64_t ckeys_cap, PfxtCtl* ctl, int mode,
                        bool with_pend, unsigned* part, unsigned* hist_all, unsigned* hist_pend, bool accumulate,
                        HistSelect select, unsigned long long target, unsigned long long nroots, hipStream_t s) {
  const size_t plane = static_cast<size_t>(kHistParts) * kHistBins;
  hipLaunchKernelGGL(hist_nodes_kernel, dim3(kHistParts), dim3(kHistBlock), 0, s, nodes, ckeys, ckeys_cap, ctl, mode,
                     with_pend ? 1 : 0, part, part + plane, part + 2 * plane);
  CPG_HIP(hipGetLastError());
  hipLaunchKernelGGL(reduce_select_kernel, dim3(kHistBins / 64, with_pend ? 3 : 2), dim3(kSelBlock), 0, s, part,
                     hist_all, hist_pend, ctl, nodes.cap, ckeys_cap, mode, accumulate ? 1 : 0,
                     static_cast<int>(select), target, nroots);
  CPG_HIP(hipGetLastError());
}

void launch_make_batch(const NodeStore& nodes, PfxtCtl* ctl, uint32_t* batch, int grid,
                       hipStream_t s) {
  hipLaunchKernelGGL(make_batch_kernel, dim3(grid), dim3(kBlock), 0, s, nodes, ctl, batch);
  CPG_HIP(hipGetLastError());
}

void launch_walk(const WalkArgs& a, bool fill, int grid, hipStream_t s) {
  // Lanes per parent: 4, and 2 where fanouts are short (a mean below 3), where
  // four lanes mostly find one deviation.  Whole queries with 1 / 2 / 4 / 8
  // lanes: 1.5M vertices (mean 2.7), K = 1M 4.26 / 4.09 / 4.28 / 4.38 ms;
  // 1.1M (5.3) 4.60 / 4.32 / 4.19 / 4.19; 400K (20) 3.17 / 2.62 / 2.52 / 2.54;
  // 250K (27), endpoint subset 4.89 / 4.16 / 3.82 / 3.73.
  const dim3 g(grid), b(kBlock);
  if (a.lanes == 2) {
    if (fill) hipLaunchKernelGGL((walk_kernel<true, 2>), g, b, 0, s, a);
    else hipLaunchKernelGGL((walk_kernel<false, 2>), g, b, 0, s, a);
  } else {
    if (fill) hipLaunchKernelGGL((walk_kernel<true, 4>), g, b, 0, s, a);
    else hipLaunchKernelGGL((walk_kernel<false, 4>), g, b, 0, s, a);
  }
  CPG_HIP(hipGetLastError());
}

namespace {
// Stored paths when `rounds` rounds have completed.
__global__ void round_log_kernel(const PfxtCtl* ctl, unsigned long long* rlog, int cap) {
  const int r = ctl->rounds;
  if (r >= 0 && r < cap) rlog[r] = ctl->node_n < ctl->node_cap ? ctl->node_n : ctl->node_cap;
}
}  // namespace

void launch_round_log(const PfxtCtl* ctl, unsigned long long* rlog, int cap, hipStream_t s) {
  hipLaunchKernelGGL(round_log_kernel, dim3(1), dim3(1), 0, s, ctl, rlog, cap);
  CPG_HIP(hipGetLastError());
}

}  // namespace cpg
