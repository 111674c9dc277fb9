// A walk over a parent path's suffix chain: the enumeration of
// the parent's children shared by the single-query and multi-query PFXT.
//
// A child of a parent with cost c takes one deviation edge u->w at a vertex
// u of the parent's suffix chain; its cost is ((c + distf[w]) + w_e) -
// distf[u] in binary32, left to right (gpucpg/gpucpg.cu:2670-2676,
// :3271-3276).  The walk reads the deviation index of the SFXT: a chain
// vertex whose smallest delta exceeds X = (U - c) + slack is skipped
// through its next-smaller pointer, and its delta-sorted deviation list is
// cut at the first delta > X.  The slack bounds the rounding gap between
// a delta and the binary32 recurrence, so no child with cost within the
// bound is skipped; the exact comparison decides emission.
#pragma once

#include "common.hpp"

namespace cpg {

// kLanes lanes walk one parent's chain together.  The walk is bound by the
// latency of its dependent loads, so a step makes one round trip do all it
// can: a vertex's record and deviation range were loaded in the step before,
// and a step loads up to kLanes of its deviations, one per lane, beside the
// next chain vertex's record and range (known from this one's).  A lane of
// its own per parent took a trip for the record, one per deviation and one
// for the deviation past the bound, on a quarter of the waves.
template <int kLanes>
struct ChainWalk {
  int4 r;        // record of the chain vertex v: {min delta, nsv, succ, distf}
  int2 di;       // its deviations {first, count}
  int4 nr;       // the next chain vertex's, loaded while v's deviations are scanned
  int2 ndi;
  int v, nv;
  int j, je;     // deviations of v still to scan
  int steps;
  bool alive, scan;
  float c, X;

  // mag = 2 max|distf| + max|w| + 1 (a bound on the terms' magnitudes).
  __device__ inline void start(bool active, float cost, int to, float U, bool bounded, float mag, const int4* vrec,
                               const int2* devinfo) {
    v = to;
    alive = active && to != -1;
    scan = false;
    steps = 0;
    j = je = 0;
    nv = -1;
    c = cost;
    X = bounded ? (U - cost) + ldexpf(fabsf(U) + fabsf(cost) + mag, -17) : __builtin_huge_valf();
    r = nr = make_int4(0, -1, -1, 0);
    di = ndi = make_int2(0, 0);
    if (alive) {
      r = vrec[v];
      di = devinfo[v];
    }
  }

  // One step, by all lanes of the wave together.  Returns true on a lane that
  // found a child with cost < U (cost <= U when !strict); *cc, *cw and *from
  // receive its cost, its deviation head w and the deviation vertex u.  A
  // walk visits each chain vertex and each deviation at most once, so more
  // than step_limit steps means a corrupt index: the walk stops and *err is
  // raised.  *nonmono counts the children whose binary32 cost comes out below
  // the parent's (a deviation whose int-scaled delta is 0, or a negative
  // weight): where one sits at the bound, a path just below U can descend
  // from a parent at or above U, which is never expanded.
  __device__ inline bool step(const int4* vrec, const int2* devinfo, const int4* devs, float U,
                              bool strict, int step_limit, int* err, unsigned long long* hops,
                              unsigned long long* devv, unsigned long long* nonmono, float* cc,
                              int* cw, int* from) {
    const int sub = __lane_id() % kLanes;
    if (alive && ++steps > step_limit) {
      atomicExch(err, 1);
      alive = scan = false;
    }
    *from = v;
    bool fresh = false;  // the next vertex's record is loaded in this step
    if (alive && !scan) {
      if (sub == 0) ++*hops;
      scan = !(__int_as_float(r.x) > X);
      nv = scan ? r.z : r.y;
      j = di.x;
      je = di.x + di.y;
      fresh = nv != -1;
    }
    int4 d = make_int4(0, 0, 0, 0);
    const bool in = alive && scan && j + sub < je;
    if (in) d = devs[j + sub];
    if (fresh) {
      nr = vrec[nv];
      ndi = devinfo[nv];
    }
    bool emit = false;
    const bool ok = in && !(__int_as_float(d.w) > X);
    if (in) ++*devv;
    if (ok) {
      const float x = ((c + __int_as_float(d.z)) + __int_as_float(d.y)) - __int_as_float(r.w);
      if (x < c) ++*nonmono;
      if (strict ? x < U : x <= U) {
        emit = true;
        *cc = x;
        *cw = d.x;
      }
    }
    // the list is cut at its first delta > X: go on only when every lane of
    // the group took one
    const uint64_t took = __ballot(ok) >> (__lane_id() - sub);
    constexpr uint64_t kAll = kLanes == 64 ? ~0ull : (1ull << kLanes) - 1;
    j += kLanes;
    if (alive && !(scan && (took & kAll) == kAll && j < je)) {
      v = nv;
      r = nr;
      di = ndi;
      scan = false;
      alive = nv != -1;
    }
    return emit;
  }
};

}  // namespace cpg
