// SFXT without device allocation: levelize + relax + successor of a graph
// that is already on the device, for callers that cannot call hipMalloc
// (serving loops that forbid it, harnesses that check for it).
//
// Every intermediate buffer of the level loop (the fanin counters, the
// relax candidates, the level-order queue and offsets, the float suffix
// distances and the loop's control block) lives in one file-scope device
// array, `scratch`, sized for kNoallocMaxVerts vertices.  Its device
// address is taken once per device with hipGetSymbolAddress (the array's
// host-side name is not a device address) and kept per device; kernels get
// pointers into it.  Each device holds its own copy until the process
// ends.  Calls that overlap on one device race on it: callers serialise
// them (one stream, or one call at a time).  The control block is cleared
// by a kernel at the start of every call.
#include <mutex>

#include "common.hpp"
#include "kernels.hpp"
#include "slots.hpp"

namespace cpg {

namespace {

constexpr int kNoallocMaxVerts = 1 << 20;  // 1,048,576 vertices
constexpr size_t kAlign = 256;
constexpr size_t align_up(size_t x) { return (x + kAlign - 1) / kAlign * kAlign; }
// layout: control block, best (8 B), deps, queue, distf (4 B each), lvlp
// (n + 2 ints); best and deps carry the level loop's kSfxtPad no-op slots
constexpr size_t kOffCtl = 0;
constexpr size_t kOffBest = align_up(sizeof(SfxtCtl));
constexpr size_t kOffDeps = kOffBest + align_up(8ull * (kNoallocMaxVerts + kSfxtPad));
constexpr size_t kOffQueue = kOffDeps + align_up(4ull * (kNoallocMaxVerts + kSfxtPad));
constexpr size_t kOffDistf = kOffQueue + align_up(4ull * kNoallocMaxVerts);
constexpr size_t kOffLvlp = kOffDistf + align_up(4ull * kNoallocMaxVerts);
constexpr size_t kScratchBytes = kOffLvlp + align_up(4ull * (kNoallocMaxVerts + 2));  // ~25 MiB

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

// Level-loop grid, by the width of the levels as they come: 32 blocks on one
// XCD (every 8th block) where they are narrow, whose barrier is cheaper, 64
// over all XCDs from two levels of more than 8,000 vertices together on, and
// back below 2,000; a change is another launch and a host synchronisation, so
// there are at most six, and graphs of fewer than 131,072 vertices, which it
// would cost more than it gives, stay on one XCD.  One XCD / all (ms): 346
// vertices a level 1.54 / 1.89, 1,000 3.9 / 5.1, 2,000 2.50 / 2.71, 3,333 2.17 /
// 1.76, 5,000 1.92 / 1.43, 10,000 1.66 / 0.89, 33,000 1.33 / 0.71.
constexpr int kNarrowBlocks = 32;
constexpr int kNarrowStride = 8;
constexpr int kWideBlocks = 64;
constexpr int kWideLevels = 8000;
constexpr int kNarrowLevels = 2000;
constexpr int kNoallocChanges = 6;
constexpr int kNoallocParts = 1 << 17;
constexpr int kMaxDevices = 64;
std::mutex g_mu;
unsigned char* g_scratch[kMaxDevices] = {};

// The current device's address of `scratch`, taken on its first use there.
unsigned char* scratch_ptr() {
  int dev = 0;
  CPG_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) throw std::runtime_error("device index out of range");
  std::lock_guard<std::mutex> lk(g_mu);
  if (!g_scratch[dev]) {
    void* p = nullptr;
    CPG_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) throw std::runtime_error("no device address for the scratch array");
    g_scratch[dev] = static_cast<unsigned char*>(p);
  }
  return g_scratch[dev];
}

__global__ void noalloc_clear_ctl_kernel(SfxtCtl* ctl) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *ctl = SfxtCtl{};
}

// Ahead of a loop's next part: its barrier starts over.
__global__ void noalloc_next_part_kernel(SfxtCtl* ctl) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    ctl->lvl_bar[0] = ctl->lvl_bar[1] = 0ull;
    ctl->cont_d = 0;
  }
}

}  // namespace

int sfxt_noalloc_max_verts() { return kNoallocMaxVerts; }

int sfxt_noalloc(int n, const int* oadjp, const int* iadjp, const int2* iedge, const int* sinks,
                 int nsinks, int* dist, int* succ, int* level, hipStream_t stream) {
  if (n < 0 || nsinks < 0 || nsinks > n) throw std::runtime_error("bad vertex or sink count");
  if (n > kNoallocMaxVerts)
    throw std::runtime_error("graph has " + std::to_string(n) + " vertices; the no-allocation SFXT takes at most " +
                             std::to_string(kNoallocMaxVerts));
  if (n == 0) return 0;
  if (!oadjp || !iadjp || !iedge || (nsinks > 0 && !sinks) || !dist || !succ || !level)
    throw std::runtime_error("null device pointer");
  unsigned char* base = scratch_ptr();
  SfxtArgs a{};
  a.n = n;
  a.nsinks = nsinks;
  a.oadjp = oadjp;
  a.iadjp = iadjp;
  a.iedge = iedge;
  a.sinks = sinks;
  a.ctl = reinterpret_cast<SfxtCtl*>(base + kOffCtl);
  a.best = reinterpret_cast<unsigned long long*>(base + kOffBest);
  a.deps = reinterpret_cast<int*>(base + kOffDeps);
  a.queue = reinterpret_cast<int*>(base + kOffQueue);
  a.distf = reinterpret_cast<float*>(base + kOffDistf);
  a.lvlp = reinterpret_cast<int*>(base + kOffLvlp);
  a.dist = dist;
  a.succ = succ;
  a.level = level;
  hipLaunchKernelGGL(noalloc_clear_ctl_kernel, dim3(1), dim3(64), 0, stream, a.ctl);
  CPG_HIP(hipGetLastError());
  launch_sfxt_dataflow_init(a, stream);  // counters, candidates, queue = sinks then -1
  SfxtCtl c{};
  bool wide = false;
  for (int changes = 0;; ++changes) {
    a.place_stride = wide ? 1 : kNarrowStride;
    a.leave = n < kNoallocParts || changes >= kNoallocChanges ? 0 : wide ? -kNarrowLevels : kWideLevels;
    LoopLease lease;
    launch_sfxt_levels_edges(a, lease.take(wide ? kWideBlocks : kNarrowBlocks, a.place_stride), stream);
    CPG_HIP(hipMemcpyAsync(&c, a.ctl, sizeof(SfxtCtl), hipMemcpyDeviceToHost, stream));
    CPG_HIP(hipStreamSynchronize(stream));
    if (c.err) throw std::runtime_error("SFXT grid barrier did not complete");
    if (c.cont_d == 0) return c.num_levels;
    a.d0 = c.cont_d;
    a.lb0 = c.cont_lb;
    a.le0 = c.cont_le;
    wide = !wide;
    hipLaunchKernelGGL(noalloc_next_part_kernel, dim3(1), dim3(64), 0, stream, a.ctl);
    CPG_HIP(hipGetLastError());
  }
}

}  // namespace cpg
