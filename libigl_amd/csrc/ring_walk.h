// ring_walk.h -- one query's walk of a rope-ordered tree shared by the 64
// lanes of a wavefront (frontier_walk).
//
// A sequential walk is a chain of dependent record fetches as long as the
// query's path.  Here the wavefront keeps a ring of pending records in LDS;
// each round every lane takes one, evaluates it and, if the walk descends
// there, pushes the record's children.  Every record the sequential walk would
// decide on is decided on here too, each by one lane.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace gwn {

constexpr uint32_t kRopeLeaf = 0x80000000u;  // link word of a leaf record

__device__ __forceinline__ uint32_t lanes_below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// LDS writes of the wavefront's lanes become visible to all of them
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A node's children enter the ring together (their positions in the rope are
// kept per record, kids), so a query takes about as many rounds as the tree
// has levels, plus one per 64 records: 7.5 rounds where pushing ranges of
// siblings, one sibling a round, took 21.4 (81,920 triangles, accuracy_scale
// 2), 20.6 against 28.7 at 4.9.  Exact triangles go to a queue
// and are evaluated 64 at a time by the whole wavefront, where evaluating
// each where it is met keeps the lanes that found none idle.
constexpr int kFrontier = 1024;                // records per wavefront (4 KiB of LDS)
constexpr int kExactQueue = 128;               // triangles waiting per wavefront and kind
constexpr uint32_t kNoKid = 0xFFFFFFFFu;       // absent child in kids
enum class Visit { kDone, kDescend, kExact, kExactNear };

// Triangles waiting for the wavefront (LDS, read as a ring): at most 63 between
// rounds, a round adds at most 64.
struct ExactQueue {
  uint32_t* q;
  uint32_t head = 0, n = 0;  // wave-uniform
  __device__ __forceinline__ void push(bool mine, uint32_t t) {
    const uint64_t m = __ballot(mine);
    if (mine) q[(head + n + lanes_below(m)) % kExactQueue] = t;
    n += (uint32_t)__popcll(m);
  }
  // evaluates up to 64 of them, when there are BATCH or no more will come
  template <int BATCH, typename Exact>
  __device__ __forceinline__ void serve(uint32_t lane, bool last, Exact&& exact) {
    if (n >= BATCH || (last && n > 0)) {
      const uint32_t cnt = min(n, 64u);
      if (lane < cnt) exact(q[(head + lane) % kExactQueue]);
      head += cnt;
      n -= cnt;
      wave_lds_sync();
    }
  }
};

// The frontier walk of one query by the calling wavefront.  ring: kFrontier
// entries of LDS; q, qn: kExactQueue each (qn only when kExactNear is
// returned).  kids[i]: the positions of record i's children, kNoKid where
// there are fewer than four or i is a leaf; kids[nslots]: the root's.
// visit(i, k, link, t) evaluates record i for the query, adds its far field (if
// any) to the lane's own sums and says what is to be done; it sets link (the
// record's link word) and k (kids[i]) for kDescend and t (the triangle) for
// kExact and kExactNear, and may set them where they are not read.  exact(t)
// and exact_near(t) add a triangle to the calling lane's own sums;
// subtree(first, end) adds records first .. end - 1, the children of a record
// descended into that a full ring has no room for.
template <int BATCH = 64, typename VisitFn, typename Exact, typename ExactNear, typename Subtree>
__device__ __forceinline__ void frontier_walk(uint32_t* __restrict__ ring, uint32_t* __restrict__ q,
                                              uint32_t* __restrict__ qn, uint32_t lane,
                                              const uint4* __restrict__ kids, uint32_t nslots, VisitFn&& visit,
                                              Exact&& exact, ExactNear&& exact_near, Subtree&& subtree) {
  ExactQueue far{q}, near{qn};
  uint32_t head = 0, tail;  // wave-uniform ring positions
  {
    const uint4 k = kids[nslots];
    const uint32_t mine = lane == 0 ? k.x : lane == 1 ? k.y : lane == 2 ? k.z : lane == 3 ? k.w : kNoKid;
    if (mine != kNoKid) ring[lane] = mine;  // the absent ones are the last
    tail = (uint32_t)__popcll(__ballot(mine != kNoKid));
  }
  wave_lds_sync();
  for (;;) {
    const uint32_t take = min(tail - head, 64u);
    Visit what = Visit::kDone;
    uint32_t link = 0, t = 0;
    uint4 k = make_uint4(kNoKid, kNoKid, kNoKid, kNoKid);
    if (lane < take) what = visit(ring[(head + lane) % kFrontier], k, link, t);
    head += take;
    const bool down = what == Visit::kDescend;
    if (__ballot(down) != 0) {
      const uint32_t np = !down ? 0u : 1u + (k.y != kNoKid) + (k.z != kNoKid) + (k.w != kNoKid);
      const uint64_t b0 = __ballot(np & 1u), b1 = __ballot(np & 2u), b2 = __ballot(np & 4u);
      const uint32_t below = lanes_below(b0) + 2u * lanes_below(b1) + 4u * lanes_below(b2);
      // lanes that fit are a prefix in lane order: their children are contiguous
      const bool fits = below + np <= kFrontier - (tail - head);
      if (down && fits) {
        const uint32_t at = tail + below;
        ring[at % kFrontier] = k.x;
        if (np > 1) ring[(at + 1) % kFrontier] = k.y;
        if (np > 2) ring[(at + 2) % kFrontier] = k.z;
        if (np > 3) ring[(at + 3) % kFrontier] = k.w;
      }
      const uint64_t in = __ballot(fits);
      tail += (uint32_t)__popcll(b0 & in) + 2u * (uint32_t)__popcll(b1 & in) + 4u * (uint32_t)__popcll(b2 & in);
      if (down && !fits) subtree(k.x, link);  // (fits is false for later lanes that do not descend, too)
    }
    far.push(what == Visit::kExact, t);
    near.push(what == Visit::kExactNear, t);
    wave_lds_sync();
    const bool last = head == tail;
    far.serve<BATCH>(lane, last, exact);
    near.serve<BATCH>(lane, last, exact_near);
    if (last && far.n + near.n == 0) break;
  }
}

// sum of the lanes' partial sums in a fixed order; every lane gets the same value
__device__ __forceinline__ double wave_sum(double v) {
  for (int off = 32; off >= 1; off >>= 1) v = __dadd_rn(v, __shfl_xor(v, off, 64));
  return v;
}
__device__ __forceinline__ float wave_sum(float v) {
  for (int off = 32; off >= 1; off >>= 1) v = __fadd_rn(v, __shfl_xor(v, off, 64));
  return v;
}

}  // namespace gwn
