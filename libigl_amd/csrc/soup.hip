// soup.hip -- triangle-soup fast winding number on gfx950.
//
// Pipeline for one mesh (gwn_soup_build):
//   k_tri_setup     per triangle: float box (the reference's K1 loop,
//                   FastWindingNumberForSoups.h:6566-6590) and a packed
//                   a,b,c record for exact evaluation
//   tree            host SAH4 (reference topology) or device LBVH
//   k_parent/k_depth, level buckets
//   k_upward<T>     one launch per tree level, deepest first: per node, the
//                   reference's item()/post() moment formulas -> BoxData,
//                   LocalData for the parent, and the subtree slot count
//   k_positions     one launch per level, root first: first slot of each node
//                   in the rope (skip-pointer) layout
//   k_write_slots   one 96-byte record per non-empty child slot
//
// Query (gwn_soup_query*): k_rs_keys + radix sort orders queries along a
// Hilbert curve so a wavefront's 64 queries walk similar paths; k_traverse walks
// the rope layout with no stack: a far child slot (|q-P|^2 > maxP2*beta^2 and
// a finite Taylor value) adds its order-0/1/2 term and jumps to its skip
// pointer, a near internal slot steps into its first child slot (the next
// record), a near triangle slot adds the exact Van Oosterom-Strackee angle.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <mutex>
#include <string>
#include <vector>

#include "device_math.h"
#include "gwn_internal.h"
#include "radix_keys.h"
#include "ring_walk.h"
#include "soup_moments.h"

namespace gwn {

constexpr uint32_t LINK_LEAF = 0x80000000u;
constexpr double PI_D = 3.1415926535897932384626433832795;

// ---------------------------------------------------------------------------
// setup
__global__ void k_tri_setup(const float* __restrict__ U, const int32_t* __restrict__ F, int64_t nf,
                            float* __restrict__ boxes, float* __restrict__ tri) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nf) return;
  const int32_t* t = F + 3 * i;
  float p[3][3];
  for (int k = 0; k < 3; ++k)
    for (int a = 0; a < 3; ++a) p[k][a] = U[3 * (int64_t)t[k] + a];
  for (int a = 0; a < 3; ++a) {
    float lo = p[0][a], hi = p[0][a];
    lo = fmin_h(lo, p[1][a]);
    hi = fmax_h(hi, p[1][a]);
    lo = fmin_h(lo, p[2][a]);
    hi = fmax_h(hi, p[2][a]);
    boxes[6 * i + 2 * a] = lo;
    boxes[6 * i + 2 * a + 1] = hi;
  }
  for (int k = 0; k < 3; ++k)
    for (int a = 0; a < 3; ++a) tri[9 * i + 3 * k + a] = p[k][a];
}

__global__ void k_parent(const uint32_t* __restrict__ nodes, int64_t nn, int32_t* __restrict__ parent) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nn) return;
  if (i == 0) parent[0] = -1;
  for (int s = 0; s < 4; ++s) {
    const uint32_t c = nodes[4 * i + s];
    if (c != NODE_EMPTY && (c & NODE_INTERNAL)) parent[c & ~NODE_INTERNAL] = (int32_t)i;
  }
}

// Depth of every node and the per-depth counts.  Counts are gathered per
// block in LDS first (depths below 64; deeper ones go straight to memory):
// a global atomic per node on the few per-depth counters serialised.
constexpr int kLdsDepths = 64;

__global__ __launch_bounds__(256) void k_depth(const int32_t* __restrict__ parent, int64_t nn,
                                               int32_t* __restrict__ depth, uint32_t* __restrict__ hist,
                                               int32_t* __restrict__ maxdepth) {
  __shared__ uint32_t h[kLdsDepths];
  __shared__ int32_t dmax;
  if (threadIdx.x < kLdsDepths) h[threadIdx.x] = 0;
  if (threadIdx.x == 0) dmax = 0;
  __syncthreads();
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nn) {
    int d = 0;
    int32_t p = parent[i];
    while (p >= 0 && d < 4096) {
      ++d;
      p = parent[p];
    }
    depth[i] = d;
    if (d < kLdsDepths)
      atomicAdd(&h[d], 1u);
    else
      atomicAdd(&hist[d], 1u);
    atomicMax(&dmax, d);
  }
  __syncthreads();
  if (threadIdx.x < kLdsDepths && h[threadIdx.x]) atomicAdd(&hist[threadIdx.x], h[threadIdx.x]);
  if (threadIdx.x == 0) atomicMax(maxdepth, dmax);
}

// order[] grouped by depth: each block reserves one range per depth with a
// single atomic and places its nodes inside it (the order within a depth is
// immaterial: the nodes of a level are processed independently)
__global__ __launch_bounds__(256) void k_bucket(const int32_t* __restrict__ depth, int64_t nn,
                                                uint32_t* __restrict__ cursor, int32_t* __restrict__ order) {
  __shared__ uint32_t cnt[kLdsDepths], base[kLdsDepths];
  if (threadIdx.x < kLdsDepths) cnt[threadIdx.x] = 0;
  __syncthreads();
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int d = i < nn ? depth[i] : -1;
  uint32_t local = 0;
  if (d >= 0 && d < kLdsDepths) local = atomicAdd(&cnt[d], 1u);
  __syncthreads();
  if (threadIdx.x < kLdsDepths && cnt[threadIdx.x]) base[threadIdx.x] = atomicAdd(&cursor[threadIdx.x], cnt[threadIdx.x]);
  __syncthreads();
  if (d >= kLdsDepths) order[atomicAdd(&cursor[d], 1u)] = (int32_t)i;
  else if (d >= 0) order[base[d] + local] = (int32_t)i;
}

// ---------------------------------------------------------------------------
// upward pass: one level
template <typename T>
__global__ void k_upward(const int32_t* __restrict__ level_nodes, int64_t count, const uint32_t* __restrict__ nodes,
                         const float* __restrict__ U, const int32_t* __restrict__ F,
                         const float* __restrict__ boxes, int order, Local<T>* __restrict__ local,
                         T* __restrict__ boxdata, uint32_t* __restrict__ nslots_sub) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= count) return;
  const int32_t node = level_nodes[t];
  Local<T> ch[4];
  int nch = 0;
  uint32_t cnt = 0;
  for (int s = 0; s < 4; ++s) {
    const uint32_t c = nodes[4 * (int64_t)node + s];
    if (c == NODE_EMPTY) break;
    if (c & NODE_INTERNAL) {
      const uint32_t ci = c & ~NODE_INTERNAL;
      ch[s] = local[ci];
      cnt += 1 + nslots_sub[ci];
    } else {
      tri_local<T>(U, F, boxes, c, order, ch[s]);
      cnt += 1;
    }
    ++nch;
  }
  T bd[92];
  Local<T> out;
  node_post<T>(ch, nch, order, bd, out);
  local[node] = out;
  for (int k = 0; k < 92; ++k) boxdata[92 * (int64_t)node + k] = bd[k];
  nslots_sub[node] = cnt;
}

// top-down: first slot position of each child node
__global__ void k_positions(const int32_t* __restrict__ level_nodes, int64_t count,
                            const uint32_t* __restrict__ nodes, const uint32_t* __restrict__ nslots_sub,
                            uint32_t* __restrict__ first_slot) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= count) return;
  const int32_t node = level_nodes[t];
  uint32_t pos = first_slot[node];
  for (int s = 0; s < 4; ++s) {
    const uint32_t c = nodes[4 * (int64_t)node + s];
    if (c == NODE_EMPTY) break;
    if (c & NODE_INTERNAL) {
      const uint32_t ci = c & ~NODE_INTERNAL;
      first_slot[ci] = pos + 1;
      pos += 1 + nslots_sub[ci];
    } else {
      pos += 1;
    }
  }
}

// Slot record (6 x float4): [P.xyz, maxP2] and the far field of
// far_field_bracket (device_math.h) for b = -N with the link word in b.w.
// The reference's terms (7199-7245), with x = q/|q|:
//   -(x.N)/|q|^2 + (tr Nd - 3 x'Nd x)/|q|^3 + (1.5 (x.s) - 7.5 K(x))/|q|^4,
// s and the cubic K as in the reference (temp0/temp1), are rewritten with
// |x| = 1 as m^2 [ x.(-N) + m ( Qf(x) + m G(x) ) ], m = 1/|q|, with the
// quadratic form Qf(x) = tr |x|^2 - 3 x'Nd x and the cubic
// G(x) = 1.5 (s.x) |x|^2 - 7.5 K(x).  The coefficients are formed in FP64 from
// the BoxData of the record's precision (the reference's in FP32) and rounded
// once.  link = skip index for an internal child, LINK_LEAF|triangle for an item.
template <typename T>
__device__ __forceinline__ void slot_far_field(const T* __restrict__ bd, int s, T* r) {
  const double nd0 = bd[BD_ND + s], nd1 = bd[BD_ND + 4 + s], nd2 = bd[BD_ND + 8 + s];
  const double tr = nd0 + nd1 + nd2;
  const double k0 = bd[BD_NKD + s], k1 = bd[BD_NKD + 4 + s], k2 = bd[BD_NKD + 8 + s];
  const double cxxy = bd[BD_CXXY + s], cxxz = bd[BD_CXXZ + s], cyyz = bd[BD_CYYZ + s];
  const double cyyx = bd[BD_CYYX + s], czzx = bd[BD_CZZX + s], czzy = bd[BD_CZZY + s];
  const double s0 = 3.0 * k0 + (cyyx + czzx), s1 = 3.0 * k1 + (czzy + cxxy), s2 = 3.0 * k2 + (cxxz + cyyz);
  const double b[3] = {-(double)bd[BD_N + s], -(double)bd[BD_N + 4 + s], -(double)bd[BD_N + 8 + s]};
  const double q[6] = {tr - 3.0 * nd0, tr - 3.0 * nd1, tr - 3.0 * nd2, -3.0 * (double)bd[BD_NXY + s],
                       -3.0 * (double)bd[BD_NYZ + s], -3.0 * (double)bd[BD_NZX + s]};
  const double g[10] = {1.5 * s0 - 7.5 * k0,   1.5 * s1 - 7.5 * k1,   1.5 * s2 - 7.5 * k2,   1.5 * s1 - 7.5 * cxxy,
                        1.5 * s2 - 7.5 * cxxz, 1.5 * s0 - 7.5 * cyyx, 1.5 * s2 - 7.5 * cyyz, 1.5 * s0 - 7.5 * czzx,
                        1.5 * s1 - 7.5 * czzy, -7.5 * (double)bd[BD_SP + s]};
  pack_far_field(b, q, g, r);
}
// Rope positions of a node's children, whose first record is `pos`; kNoKid
// where there are fewer than four.
__device__ __forceinline__ uint4 kid_positions(const uint32_t* __restrict__ nodes,
                                               const uint32_t* __restrict__ nslots_sub, uint32_t node, uint32_t pos) {
  uint32_t k[4] = {kNoKid, kNoKid, kNoKid, kNoKid};
  for (int s = 0; s < 4; ++s) {
    const uint32_t c = nodes[4 * (int64_t)node + s];
    if (c == NODE_EMPTY) break;
    k[s] = pos;
    pos += (c & NODE_INTERNAL) ? 1 + nslots_sub[c & ~NODE_INTERNAL] : 1;
  }
  return make_uint4(k[0], k[1], k[2], k[3]);
}

__global__ void k_write_slots(int64_t nn, const uint32_t* __restrict__ nodes, const float* __restrict__ boxdata,
                              const uint32_t* __restrict__ nslots_sub, const uint32_t* __restrict__ first_slot,
                              uint32_t nslots, float4* __restrict__ slots, uint4* __restrict__ kids) {
  int64_t node = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (node >= nn) return;
  const float* bd = boxdata + 92 * node;
  uint32_t pos = first_slot[node];
  if (node == 0) kids[nslots] = kid_positions(nodes, nslots_sub, 0, 0);
  for (int s = 0; s < 4; ++s) {
    const uint32_t c = nodes[4 * node + s];
    if (c == NODE_EMPTY) break;
    uint32_t link, next;
    if (c & NODE_INTERNAL) {
      next = pos + 1 + nslots_sub[c & ~NODE_INTERNAL];
      link = next;
      kids[pos] = kid_positions(nodes, nslots_sub, c & ~NODE_INTERNAL, pos + 1);
    } else {
      next = pos + 1;
      link = LINK_LEAF | c;
      kids[pos] = make_uint4(kNoKid, kNoKid, kNoKid, kNoKid);
    }
    float4* r = slots + 6 * (int64_t)pos;
    float v[20];
    slot_far_field(bd, s, v);
    r[0] = make_float4(bd[BD_P + s], bd[BD_P + 4 + s], bd[BD_P + 8 + s], bd[BD_MAXP2 + s]);
    r[1] = make_float4(v[0], v[1], v[2], __uint_as_float(link));
    for (int k = 1; k < 5; ++k) r[1 + k] = make_float4(v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]);
    pos = next;
  }
}

// FP64 slot record: 24 doubles in the order of the FP32 record's 24 floats,
// the link word in the low half of the eighth.
__global__ void k_write_slots64(int64_t nn, const uint32_t* __restrict__ nodes, const double* __restrict__ bd64,
                                const uint32_t* __restrict__ first_slot, const uint32_t* __restrict__ nslots_sub,
                                double* __restrict__ slots64) {
  int64_t node = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (node >= nn) return;
  const double* bd = bd64 + 92 * node;
  uint32_t pos = first_slot[node];
  for (int s = 0; s < 4; ++s) {
    const uint32_t c = nodes[4 * node + s];
    if (c == NODE_EMPTY) break;
    const uint32_t next = (c & NODE_INTERNAL) ? pos + 1 + nslots_sub[c & ~NODE_INTERNAL] : pos + 1;
    double* r = slots64 + 24 * (int64_t)pos;
    for (int k = 0; k < 3; ++k) r[k] = bd[BD_P + 4 * k + s];
    r[3] = bd[BD_MAXP2 + s];
    double v[20];
    slot_far_field(bd, s, v);
    v[3] = __longlong_as_double((long long)((c & NODE_INTERNAL) ? next : (LINK_LEAF | c)));
    for (int k = 0; k < 20; ++k) r[4 + k] = v[k];
    pos = next;
  }
}

// ---------------------------------------------------------------------------
// closest-point support: a bounding box per slot record, from the FP64
// vertices and rounded outward to float, so a box distance computed from it
// never exceeds the distance to anything inside.
__device__ __forceinline__ float round_down_f(double x) {
  float f = (float)x;
  return ((double)f > x) ? nextafterf(f, -INFINITY) : f;
}
__device__ __forceinline__ float round_up_f(double x) {
  float f = (float)x;
  return ((double)f < x) ? nextafterf(f, INFINITY) : f;
}
__device__ __forceinline__ void tri_box64(const double* __restrict__ V, const int32_t* __restrict__ F, uint32_t t,
                                          float lo[3], float hi[3]) {
  for (int a = 0; a < 3; ++a) {
    double l = V[3 * (int64_t)F[3 * (int64_t)t] + a], h = l;
    for (int k = 1; k < 3; ++k) {
      const double v = V[3 * (int64_t)F[3 * (int64_t)t + k] + a];
      l = v < l ? v : l;
      h = v > h ? v : h;
    }
    lo[a] = round_down_f(l);
    hi[a] = round_up_f(h);
  }
}

__global__ void k_node_boxes(const int32_t* __restrict__ level_nodes, int64_t count, const uint32_t* __restrict__ nodes,
                             const double* __restrict__ V, const int32_t* __restrict__ F, float* __restrict__ nbox) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= count) return;
  const int32_t node = level_nodes[t];
  float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (int s = 0; s < 4; ++s) {
    const uint32_t c = nodes[4 * (int64_t)node + s];
    if (c == NODE_EMPTY) break;
    float cl[3], chh[3];
    if (c & NODE_INTERNAL) {
      const float* b = nbox + 6 * (int64_t)(c & ~NODE_INTERNAL);
      for (int a = 0; a < 3; ++a) {
        cl[a] = b[a];
        chh[a] = b[3 + a];
      }
    } else {
      tri_box64(V, F, c, cl, chh);
    }
    for (int a = 0; a < 3; ++a) {
      lo[a] = fminf(lo[a], cl[a]);
      hi[a] = fmaxf(hi[a], chh[a]);
    }
  }
  for (int a = 0; a < 3; ++a) {
    nbox[6 * (int64_t)node + a] = lo[a];
    nbox[6 * (int64_t)node + 3 + a] = hi[a];
  }
}

// first slot of each child node from the parent's first slot and the links
__global__ void k_positions_rope(const int32_t* __restrict__ level_nodes, int64_t count,
                                 const uint32_t* __restrict__ nodes, const float4* __restrict__ slots,
                                 uint32_t* __restrict__ first_slot) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= count) return;
  const int32_t node = level_nodes[t];
  uint32_t pos = first_slot[node];
  for (int s = 0; s < 4; ++s) {
    const uint32_t c = nodes[4 * (int64_t)node + s];
    if (c == NODE_EMPTY) break;
    if (c & NODE_INTERNAL) {
      first_slot[c & ~NODE_INTERNAL] = pos + 1;
      pos = __float_as_uint(slots[6 * (int64_t)pos + 1].w);
    } else {
      pos += 1;
    }
  }
}

// slot box record (2 x float4): [lo.xyz, link] [hi.xyz, 0], in rope order
__global__ void k_write_dbox(int64_t nn, const uint32_t* __restrict__ nodes, const float* __restrict__ nbox,
                             const double* __restrict__ V, const int32_t* __restrict__ F,
                             const uint32_t* __restrict__ first_slot, const float4* __restrict__ slots,
                             float4* __restrict__ dbox) {
  const int64_t node = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (node >= nn) return;
  uint32_t pos = first_slot[node];
  for (int s = 0; s < 4; ++s) {
    const uint32_t c = nodes[4 * node + s];
    if (c == NODE_EMPTY) break;
    float lo[3], hi[3];
    if (c & NODE_INTERNAL) {
      const float* b = nbox + 6 * (int64_t)(c & ~NODE_INTERNAL);
      for (int a = 0; a < 3; ++a) {
        lo[a] = b[a];
        hi[a] = b[3 + a];
      }
    } else {
      tri_box64(V, F, c, lo, hi);
    }
    const float link = slots[6 * (int64_t)pos + 1].w;
    dbox[2 * (int64_t)pos] = make_float4(lo[0], lo[1], lo[2], link);
    dbox[2 * (int64_t)pos + 1] = make_float4(hi[0], hi[1], hi[2], 0.0f);
    const uint32_t l = __float_as_uint(link);
    pos = (l & LINK_LEAF) ? pos + 1 : l;
  }
}

// Planes of a face for a lower bound of its distance (k_closest): the unit
// normal's plane and, through each edge, the plane across the face with the
// unit normal pointing out of it, as (n, d) with n.(p - centre) + d the signed
// distance.  Zero where an edge or the normal has no direction, which bounds
// nothing.
__global__ void k_face_planes(const double* __restrict__ V, const int32_t* __restrict__ F, int64_t nf, float cx,
                              float cy, float cz, float4* __restrict__ planes) {
  const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= nf) return;
  double v[3][3], n[3];
  const double c[3] = {cx, cy, cz};
  for (int k = 0; k < 3; ++k)
    for (int a = 0; a < 3; ++a) v[k][a] = V[3 * (int64_t)F[3 * f + k] + a] - c[a];
  const auto cross = [](const double* x, const double* y, double* z) {
    for (int a = 0; a < 3; ++a) z[a] = x[(a + 1) % 3] * y[(a + 2) % 3] - x[(a + 2) % 3] * y[(a + 1) % 3];
  };
  const auto plane = [&](const double* dir, const double* at) {
    const double l = sqrt(dir[0] * dir[0] + dir[1] * dir[1] + dir[2] * dir[2]);
    if (!(l > 1e-150 && l < 1e150)) return make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const double u[3] = {dir[0] / l, dir[1] / l, dir[2] / l};
    return make_float4((float)u[0], (float)u[1], (float)u[2], (float)-(u[0] * at[0] + u[1] * at[1] + u[2] * at[2]));
  };
  double e[3][3];
  for (int k = 0; k < 3; ++k)
    for (int a = 0; a < 3; ++a) e[k][a] = v[(k + 1) % 3][a] - v[k][a];
  cross(e[0], e[1], n);
  // a sliver's normal is mostly rounding: bound nothing with it
  const double l0 = e[0][0] * e[0][0] + e[0][1] * e[0][1] + e[0][2] * e[0][2];
  const double l1 = e[1][0] * e[1][0] + e[1][1] * e[1][1] + e[1][2] * e[1][2];
  const double nn = n[0] * n[0] + n[1] * n[1] + n[2] * n[2];
  const bool flat = nn > 1e-14 * l0 * l1;
  planes[4 * f] = flat ? plane(n, v[0]) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  for (int k = 0; k < 3; ++k) {
    double out[3];
    cross(e[k], n, out);
    planes[4 * f + 1 + k] = flat ? plane(out, v[k]) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  }
}

// ---------------------------------------------------------------------------
// exact triangle solid angle: UTsignedSolidAngleTri (6070-6110)
// (not inlined: the sums below call it for few terms)
template <typename T>
__device__ __attribute__((noinline)) T tri_solid_angle(T ax, T ay, T az, T bx, T by, T bz, T cx, T cy, T cz, T qx, T qy,
                                             T qz) {
  T a0 = ax - qx, a1 = ay - qy, a2 = az - qz;
  T b0 = bx - qx, b1 = by - qy, b2 = bz - qz;
  T c0 = cx - qx, c1 = cy - qy, c2 = cz - qz;
  const T al = sqrt(a0 * a0 + a1 * a1 + a2 * a2);
  const T bl = sqrt(b0 * b0 + b1 * b1 + b2 * b2);
  const T cl = sqrt(c0 * c0 + c1 * c1 + c2 * c2);
  if (al == T(0) || bl == T(0) || cl == T(0)) return T(0);
  const T ra = T(1) / al, rb = T(1) / bl, rc = T(1) / cl;
  a0 *= ra; a1 *= ra; a2 *= ra;
  b0 *= rb; b1 *= rb; b2 *= rb;
  c0 *= rc; c1 *= rc; c2 *= rc;
  const T u0 = b0 - a0, u1 = b1 - a1, u2 = b2 - a2;
  const T w0 = c0 - a0, w1 = c1 - a1, w2 = c2 - a2;
  const T num = a0 * (u1 * w2 - u2 * w1) + a1 * (u2 * w0 - u0 * w2) + a2 * (u0 * w1 - u1 * w0);
  if (num == T(0)) return T(0);
  const T den = T(1) + (a0 * b0 + a1 * b1 + a2 * b2) + (a0 * c0 + a1 * c1 + a2 * c2) + (b0 * c0 + b1 * c1 + b2 * c2);
  return T(2) * atan2(num, den);
}

// ---- FP32 fast path of the traversal (atan2_fast: device_math.h) ----
// UTsignedSolidAngleTri (6070-6110) with hardware reciprocal square roots for
// the normalisation; same zero-length and zero-numerator rules.
__device__ __forceinline__ float tri_solid_angle_fast(float ax, float ay, float az, float bx, float by, float bz,
                                                      float cx, float cy, float cz, float qx, float qy, float qz) {
  float a0 = ax - qx, a1 = ay - qy, a2 = az - qz;
  float b0 = bx - qx, b1 = by - qy, b2 = bz - qz;
  float c0 = cx - qx, c1 = cy - qy, c2 = cz - qz;
  const float la = fmaf(a2, a2, fmaf(a1, a1, a0 * a0));
  const float lb = fmaf(b2, b2, fmaf(b1, b1, b0 * b0));
  const float lc = fmaf(c2, c2, fmaf(c1, c1, c0 * c0));
  if (la == 0.0f || lb == 0.0f || lc == 0.0f) return 0.0f;
  if (fminf(la, fminf(lb, lc)) < 1e-30f)  // keep rsq away from denormals
    return tri_solid_angle<float>(ax, ay, az, bx, by, bz, cx, cy, cz, qx, qy, qz);
  const float ra = __builtin_amdgcn_rsqf(la), rb = __builtin_amdgcn_rsqf(lb), rc = __builtin_amdgcn_rsqf(lc);
  a0 *= ra; a1 *= ra; a2 *= ra;
  b0 *= rb; b1 *= rb; b2 *= rb;
  c0 *= rc; c1 *= rc; c2 *= rc;
  const float u0 = b0 - a0, u1 = b1 - a1, u2 = b2 - a2;
  const float w0 = c0 - a0, w1 = c1 - a1, w2 = c2 - a2;
  const float k0 = fmaf(u1, w2, -(u2 * w1)), k1 = fmaf(u2, w0, -(u0 * w2)), k2 = fmaf(u0, w1, -(u1 * w0));
  const float num = fmaf(a2, k2, fmaf(a1, k1, a0 * k0));
  if (num == 0.0f) return 0.0f;
  const float ab = fmaf(a2, b2, fmaf(a1, b1, a0 * b0));
  const float ac = fmaf(a2, c2, fmaf(a1, c1, a0 * c0));
  const float bc = fmaf(b2, c2, fmaf(b1, c1, b0 * c0));
  const float den = ((1.0f + ab) + ac) + bc;
  return 2.0f * atan2_fast(num, den);
}

struct D4 {
  double x, y, z, w;
};

__device__ __forceinline__ float tri_rsqrt(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ double tri_rsqrt(double x) { return rsqrt64(x); }

// Signed solid angles of triangles (UTsignedSolidAngleTri, 6070-6110), summed.
// The half angles atan2(num, den) go into an AngleSum; a term it does not
// take, and a triangle with a corner (nearly) at the query, is summed on its
// own as the per-triangle functions above give it.
template <typename T>
struct SolidAngleSum {
  AngleSum<T> half;
  T extra = T(0);

  __device__ __forceinline__ void add(const float* __restrict__ p, T qx, T qy, T qz) {
    constexpr T tiny = sizeof(T) == 4 ? T(1e-30) : T(1e-290);  // keeps the reciprocal square roots away from denormals
    T a0 = p[0] - qx, a1 = p[1] - qy, a2 = p[2] - qz;
    T b0 = p[3] - qx, b1 = p[4] - qy, b2 = p[5] - qz;
    T c0 = p[6] - qx, c1 = p[7] - qy, c2 = p[8] - qz;
    const T la = fma(a2, a2, fma(a1, a1, a0 * a0));
    const T lb = fma(b2, b2, fma(b1, b1, b0 * b0));
    const T lc = fma(c2, c2, fma(c1, c1, c0 * c0));
    if (fmin(la, fmin(lb, lc)) < tiny) {
      extra += tri_solid_angle<T>(p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8], qx, qy, qz);
      return;
    }
    const T ra = tri_rsqrt(la), rb = tri_rsqrt(lb), rc = tri_rsqrt(lc);
    a0 *= ra; a1 *= ra; a2 *= ra;
    b0 *= rb; b1 *= rb; b2 *= rb;
    c0 *= rc; c1 *= rc; c2 *= rc;
    const T u0 = b0 - a0, u1 = b1 - a1, u2 = b2 - a2;
    const T w0 = c0 - a0, w1 = c1 - a1, w2 = c2 - a2;
    T num;
    if constexpr (sizeof(T) == 4) {
      const T k0 = fma(u1, w2, -(u2 * w1)), k1 = fma(u2, w0, -(u0 * w2)), k2 = fma(u0, w1, -(u1 * w0));
      num = fma(a2, k2, fma(a1, k1, a0 * k0));
    } else {
      num = a0 * (u1 * w2 - u2 * w1) + a1 * (u2 * w0 - u0 * w2) + a2 * (u0 * w1 - u1 * w0);
    }
    if (sizeof(T) == 4 && num == T(0)) return;
    const T ab = fma(a2, b2, fma(a1, b1, a0 * b0));
    const T ac = fma(a2, c2, fma(a1, c1, a0 * c0));
    const T bc = fma(b2, c2, fma(b1, c1, b0 * c0));
    const T den = ((T(1) + ab) + ac) + bc;
    // FP64: the vector (den, num) turns by the roundings of den over its
    // length; where it is short (the query near an edge) the term is
    // tri_solid_angle's.  Sums over the triangles near 6,000 queries, half of
    // them 1e-6 from the surface, differ from that form's by 4.6e-16 (rms) and
    // 4e-15 (at most); with a line at 1e-9 by 6.7e-15 and 4.6e-13, and lay
    // further from the true sums.  One term in 20,000 there is so short.  The
    // same for a query (nearly) in the triangle's plane and inside it, where
    // whether num is zero, and its sign, hang on the last bits, and with them
    // a whole turn of the angle.
    const bool fine = sizeof(T) == 4 || (fmax(fabs(num), fabs(den)) > T(1e-2) && fabs(num) >= T(-1e-9) * den);
    if (!fine || !half.add(num, den))
      extra += tri_solid_angle<T>(p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8], qx, qy, qz);
  }
  __device__ __forceinline__ double total() const { return (double)extra + 2.0 * half.total(); }
};

// ---------------------------------------------------------------------------
// traversal: FP32 (reference arithmetic) and mixed (FP32 far field and
// running sum; FP64 solid angles and sum of the triangles near the query)
//
// Wave-coherent rope walk.  The slot records are in depth-first ("rope")
// order: a far child adds its Taylor value and skips to `link` (the record
// after its subtree), a near internal child is entered (next record), an item
// is evaluated exactly when near.  Each lane keeps `skip`, the next record it
// needs; the wavefront walks one shared index i and a lane takes part in a
// record exactly when i == skip.  (k_traverse tests skip <= i: a lane that
// enters a child or evaluates an item leaves skip where it was, and only a
// lane that takes a far field moves it past the subtree.)  The wave steps to
// i+1 when some lane needs it (a near child, or an item) and otherwise to
// link(i): every lane that is not taking part needs a record at or beyond
// link(i), because the subtrees of the rope are nested intervals.  So each lane
// visits exactly the records of its own walk, in the same order, and sums the same terms in the same
// order as an independent per-lane walk; but every record (and triangle) a
// wave reads is the same for all its lanes, so it is fetched once per wave
// through the scalar cache instead of 64 times through the vector memory path.
__device__ __forceinline__ uint32_t wave_uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// Mixed form: a triangle slot that may lie within near_d of the query
// (|q - P| < sqrt(maxP2) + near_d, P the slot's centre and maxP2 its squared
// radius) has its solid angle computed in FP64 (UTsignedSolidAngleTri,
// 6070-6110, in double) and summed in an FP64 accumulator of its own; the far
// field and every other exact term go to the FP32 sums.  The square root is the
// hardware's, within an ulp: where the line lies is a choice, not a bound.
__device__ __forceinline__ bool near_triangle(float maxp2, float l2, float near_d) {
  const float rr = __builtin_amdgcn_sqrtf(maxp2) + near_d;
  return l2 < rr * rr;
}

// Near-triangle FP64 terms of the mixed form are deferred: a lane notes each
// such triangle in its own column of an LDS list and evaluates the list, in
// the order noted, after the walk.  In the wave-coherent walk this turns FP64
// work that one lane of a wavefront needs at a record (which every lane would
// sit through) into work all lanes do together at the end, and keeps the FP64
// code and its registers out of the walk.  The terms and the order of their
// FP64 additions are those of evaluating each where it is met.  A query that
// meets more than kDefer near triangles gets W = NaN, which sends it to the
// FP64 re-evaluation pass with the ambiguous queries.
constexpr int kDefer = 16;
constexpr int kTravThreads = 256;

struct NearList {
  uint32_t* lds;  // column threadIdx.x of a kDefer x kTravThreads array
  uint32_t n;     // kDefer + 1 after an overflow
};

__device__ __forceinline__ void note_near(NearList& L, uint32_t t) {
  if (L.n < (uint32_t)kDefer) L.lds[L.n * kTravThreads] = t;
  L.n = L.n < (uint32_t)kDefer ? L.n + 1 : (uint32_t)kDefer + 1;
}

// Exact triangles of the wave-coherent walks wait in a per-lane LDS list until
// some lane's is full; then every lane evaluates its own.  At a record only
// the lanes near that triangle need it (61 of a lane's 1,180 records on the
// 81,920-triangle workload at accuracy_scale 4.9, but some lane at 133 of the
// wavefront's 1,502), so evaluating it there keeps the other lanes idle for
// some 90 instructions; together the lanes take about 72 turns.  A lane's
// triangles enter its sum in the order met, whatever its neighbours do, so a
// query's result does not depend on its wavefront.
template <int N>
struct Pending {
  uint32_t* lds;  // column threadIdx.x of an N x kTravThreads array
  uint32_t n = 0;
  __device__ __forceinline__ void push(uint32_t t) { lds[n++ * kTravThreads] = t; }
  template <typename T>
  __device__ __forceinline__ void flush(const float* __restrict__ tri, T qx, T qy, T qz, SolidAngleSum<T>& ex) {
    for (uint32_t k = 0; k < n; ++k) ex.add(tri + 9 * (size_t)lds[k * kTravThreads], qx, qy, qz);
    n = 0;
  }
};

// W of a walk: the far fields' FP32 sum and the exact triangles' angles, plus
// (mixed form) the noted near triangles' FP64 solid angles summed in order;
// NaN after an overflow.
template <bool MIXED>
__device__ __forceinline__ double finish_walk(float sum, const SolidAngleSum<float>& ex, const NearList& L,
                                              const float* __restrict__ tri, float qx, float qy, float qz) {
  const double w = (double)sum + ex.total();
  if (!MIXED) return w / (4.0 * PI_D);
  if (L.n > (uint32_t)kDefer) return __longlong_as_double(0x7FF8000000000000ll);
  SolidAngleSum<double> near;
  for (uint32_t k = 0; k < L.n; ++k) near.add(tri + 9 * (size_t)L.lds[k * kTravThreads], qx, qy, qz);
  return (w + near.total()) / (4.0 * PI_D);
}

// Both walks are held to 8 wavefronts per SIMD (64 VGPRs): the walk loop fits
// in that, and only the mixed form's end-of-walk FP64 code would take more
// (94 VGPRs, 5 wavefronts); it keeps some of its constants in scratch instead.
// Per-lane rope walk from record j to the end: each lane follows its own skip
// pointers and gathers its own records.  The wave-coherent walk hands over to
// it where its wavefront's lanes have stopped sharing records; records, terms
// and their order are the same in both walks.
template <int ORDER, bool MIXED>
__device__ __forceinline__ void lane_walk(const float4* __restrict__ slots, uint32_t nslots,
                                          const float* __restrict__ tri, uint32_t j, float qx, float qy, float qz,
                                          float acc2, float near_d, float& sum, SolidAngleSum<float>& ex,
                                          NearList& L) {
  while (j < nslots) {
    const float4* r = slots + 6 * (size_t)j;
    const float4 a = r[0], b = r[1];
    const uint32_t link = __float_as_uint(b.w);
    const float x = qx - a.x, y = qy - a.y, z = qz - a.z;
    const float l2 = __fadd_rn(__fadd_rn(__fmul_rn(x, x), __fmul_rn(y, y)), __fmul_rn(z, z));
    const bool leaf = (link & LINK_LEAF) != 0;
    if (!(l2 <= __fmul_rn(a.w, acc2))) {
      float4 c, d, e, f;
      if (ORDER >= 1) {
        c = r[2];
        d = r[3];
      }
      if (ORDER >= 2) {
        e = r[4];
        f = r[5];
      }
      const float m = __builtin_amdgcn_rsqf(l2);
      const float o = far_field_bracket<ORDER>(x, y, z, m, b, c, d, e, f), m2 = __fmul_rn(m, m);
      if (isfinite(__fmul_rn(m2, o))) {  // otherwise the reference descends / evaluates the item
        sum = fmaf(m2, o, sum);
        j = leaf ? j + 1 : link;
        continue;
      }
    }
    if (leaf) {
      const uint32_t t = link & ~LINK_LEAF;
      if (MIXED && near_triangle(a.w, l2, near_d)) note_near(L, t);
      else ex.add(tri + 9 * (size_t)t, qx, qy, qz);
    }
    ++j;
  }
}

// A kernel argument copied into a VGPR: a VALU instruction reads at most one
// SGPR, so the product of the slot radius (an SGPR in the wave-coherent walk)
// and accuracy_scale^2 would otherwise need a move at every step.
__device__ __forceinline__ float in_vgpr(float x) {
  float v;
  asm("v_mov_b32 %0, %1" : "=v"(v) : "s"(x));
  return v;
}

// HANDOVER: a wavefront whose lanes have stopped sharing records (fewer than
// 16 lanes per step on average over a window of 256 steps: the union of their
// paths exceeds the longest by far, as on fans of thin triangles) hands over
// to the per-lane walk, each lane from the record it needs next.  Results are
// unchanged (same records, terms and order); the check costs about a tenth of
// the walk's time on coherent batches, so only latency-bound callers (the
// serving engine, on large trees) take it.
//
// The walk is bound by VALU issue, so its step holds only what a lane cannot
// do without: which lanes take part, are far and stay near is kept in scalar
// lane masks, and a far field is added without asking whether it is finite.
// The reference descends where it is not; a sum that ends up not finite is
// walked again by lane_walk, which asks.  A step takes 12 VALU instructions, a
// far field 32 more and a waiting triangle's turn about 75: 66,000 per
// wavefront on 81,920 triangles, 1M queries, accuracy_scale 4.9 (82,700 with
// the conditions in VGPRs, the homogeneous polynomial and each triangle
// evaluated, with an atan2 of its own, where it is met), and 1.70 ms a call
// against 2.06; 1.31M triangles, 10M queries, mixed form: 19.4 against 22.4.
template <int ORDER, bool MIXED, bool HANDOVER>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void k_traverse(
    const float4* __restrict__ slots, uint32_t nslots, const float* __restrict__ tri, const float* __restrict__ Q,
    const uint32_t* __restrict__ perm, const uint32_t* __restrict__ order, int64_t nq, float acc2_arg, float near_d,
    double* __restrict__ W) {
  const int64_t t = (int64_t)(order ? order[xcd_block()] : xcd_block()) * blockDim.x + threadIdx.x;
  if (t >= nq) return;
  const float acc2 = in_vgpr(acc2_arg);
  const int64_t qi = perm ? (int64_t)perm[t] : t;
  const float qx = Q[3 * qi], qy = Q[3 * qi + 1], qz = Q[3 * qi + 2];
  float sum = 0.0f;
  SolidAngleSum<float> ex;
  // mixed form: the noted near triangles take LDS too, and eight blocks of it
  // fit a CU only with a shorter list of waiting ones
  constexpr int kPend = MIXED ? 4 : 16;
  __shared__ uint32_t pend_lds[kPend * kTravThreads];
  __shared__ uint32_t near_lds[MIXED ? kDefer * kTravThreads : 1];
  Pending<kPend> pend{pend_lds + threadIdx.x};
  NearList L{near_lds + threadIdx.x, 0};
  uint32_t skip = 0;
  uint32_t i = 0;
  uint32_t steps = 0, taken = 0;  // wave-uniform: steps in this window, lanes taking part summed over them
  while (i < nslots) {
    const float4* r = slots + 6 * (size_t)i;
    const float4 a = r[0], b = r[1];
    float4 c, d, e, f;
    if (ORDER >= 1) {
      c = r[2];
      d = r[3];
    }
    if (ORDER >= 2) {
      e = r[4];
      f = r[5];
    }
    // the whole record is requested together (one scalar-cache round trip)
    // rather than where each part is first used
    if (ORDER >= 2) asm volatile("" ::"s"(a.x), "s"(b.w), "s"(c.x), "s"(e.x), "s"(f.w));
    else if (ORDER >= 1) asm volatile("" ::"s"(a.x), "s"(b.w), "s"(c.x), "s"(d.w));
    else asm volatile("" ::"s"(a.x), "s"(b.w));
    const uint32_t link = __float_as_uint(b.w);
    const bool leaf = (link & LINK_LEAF) != 0;
    // the record after this one's subtree, picked in scalar code so that a
    // lane taking the far field only copies it
    const uint32_t past = leaf ? i + 1 : link;
    // skip >= i holds for every lane (nested intervals), so skip <= i means
    // skip == i; a lane that descends or evaluates an item leaves skip at i,
    // which is <= i + 1, the record it needs next
    const uint64_t part = lanes_at_most(skip, i);
    const float x = qx - a.x, y = qy - a.y, z = qz - a.z;
    // |q-P|^2 rounded as the reference rounds it (no fused multiply-add),
    // so every near/far decision is the reference's
    const float l2 = __fadd_rn(__fadd_rn(__fmul_rn(x, x), __fmul_rn(y, y)), __fmul_rn(z, z));
    const uint64_t beyond = lanes_beyond(l2, __fmul_rn(a.w, acc2));
    if (lane_in(part & beyond)) {
      const float m = __builtin_amdgcn_rsqf(l2);
      sum = fmaf(__fmul_rn(m, m), far_field_bracket<ORDER>(x, y, z, m, b, c, d, e, f), sum);
      skip = past;
    }
    const uint64_t stay = part & ~beyond;
    if (leaf && stay != 0) {
      if (lane_in(stay)) {
        const uint32_t tr = link & ~LINK_LEAF;
        if (MIXED && near_triangle(a.w, l2, near_d)) note_near(L, tr);
        else pend.push(tr);
      }
      if (__ballot(pend.n == (uint32_t)kPend) != 0) pend.flush(tri, qx, qy, qz, ex);
    }
    i = wave_uniform((leaf || stay != 0) ? i + 1 : link);
    if (HANDOVER) taken += (uint32_t)__popcll(part);
    if (HANDOVER && ++steps == 256) {
      if (taken < 256u * 16u) break;
      steps = taken = 0;
    }
  }
  pend.flush(tri, qx, qy, qz, ex);
  // after a hand-over each lane continues from the record it needs next
  if (HANDOVER && i < nslots)
    lane_walk<ORDER, MIXED>(slots, nslots, tri, skip > i ? skip : i, qx, qy, qz, acc2, near_d, sum, ex, L);
  // a query that is not finite meets no finite term: its sum stays NaN
  if (!isfinite(sum) && isfinite(qx) && isfinite(qy) && isfinite(qz)) {
    sum = 0.0f;
    ex = SolidAngleSum<float>();
    L.n = 0;
    lane_walk<ORDER, MIXED>(slots, nslots, tri, 0, qx, qy, qz, acc2, near_d, sum, ex, L);
  }
  W[qi] = finish_walk<MIXED>(sum, ex, L, tri, qx, qy, qz);
}

// FP64 far field of record i for query q: added to part when the query is
// beyond the record's radius and the value is finite, else false.  link: the
// record's link word.
// descend() is called before the far field's part of the record is read
// (or, where the value is not finite, after) when it returns false.
template <int ORDER, typename Descend>
__device__ __forceinline__ bool record_far64(const double* __restrict__ s64, uint32_t i, uint32_t& link, double qx,
                                             double qy, double qz, double acc2, double& part, Descend&& descend) {
  const double* r = s64 + 24 * (size_t)i;
  const D4 b{r[4], r[5], r[6], r[7]};
  link = (uint32_t)__double_as_longlong(b.w);
  const double x = qx - r[0], y = qy - r[1], z = qz - r[2];
  const double l2 = x * x + y * y + z * z;
  const bool beyond = !(l2 <= r[3] * acc2);
  if (!beyond) descend();
  if (beyond) {
    const D4 c{r[8], r[9], r[10], r[11]}, d{r[12], r[13], r[14], r[15]}, e{r[16], r[17], r[18], r[19]},
        f{r[20], r[21], r[22], r[23]};
    const double m = rsqrt64(l2), m2 = __dmul_rn(m, m);
    const double o = far_field_bracket<ORDER>(x, y, z, m, b, c, d, e, f);
    if (isfinite(__dmul_rn(m2, o))) {
      part = fma(m2, o, part);
      return true;
    }
    descend();
  }
  return false;
}

// all-FP64 form: FP64 moments, far field, atan2 and sum
// The step of k_traverse in FP64, bound by FP64 VALU issue on large batches
// and by the length of its few wavefronts on small ones.  The far field as
// one polynomial with a refined reciprocal square root (it was a division, a
// square root and the moments' own form, about twice the operations) and the
// triangles as one AngleSum took 200,003 queries on 81,920 triangles at
// accuracy_scale 2 from 0.92 to 0.55 ms.  Eight wavefronts per SIMD (64 VGPRs,
// some spilled outside the step): 1.5M queries at 4.9 took 3.97 ms at eight,
// 4.43 at seven, 4.63 at six, 4.50 at five and 4.96 at four.
constexpr int kPend64 = 16;
template <int ORDER>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void k_traverse64(
    const double* __restrict__ s64, uint32_t nslots, const float* __restrict__ tri, const float* __restrict__ Q,
    const uint32_t* __restrict__ perm, const uint32_t* __restrict__ order, int64_t nq, double acc2,
    double* __restrict__ W) {
  // the same wave-coherent rope walk as k_traverse, over the FP64 records;
  // order (when given) is the block order
  const int64_t t = (int64_t)(order ? order[xcd_block()] : xcd_block()) * blockDim.x + threadIdx.x;
  if (t >= nq) return;
  const int64_t qi = perm ? (int64_t)perm[t] : t;
  const double qx = Q[3 * qi], qy = Q[3 * qi + 1], qz = Q[3 * qi + 2];
  double sum = 0.0;
  SolidAngleSum<double> ex;
  __shared__ uint32_t pend_lds[kPend64 * kTravThreads];
  Pending<kPend64> pend{pend_lds + threadIdx.x};
  uint32_t skip = 0;
  uint32_t i = 0;
  while (i < nslots) {
    const double* r = s64 + 24 * (size_t)i;
    const D4 a{r[0], r[1], r[2], r[3]}, b{r[4], r[5], r[6], r[7]};
    asm volatile("" ::"s"(a.x), "s"(b.w));
    const uint32_t link = (uint32_t)__double_as_longlong(b.w);
    const bool leaf = (link & LINK_LEAF) != 0;
    const uint32_t past = leaf ? i + 1 : link;
    const uint64_t part = lanes_at_most(skip, i);
    const double x = qx - a.x, y = qy - a.y, z = qz - a.z;
    const double l2 = x * x + y * y + z * z;
    const uint64_t beyond = lanes_beyond(l2, a.w * acc2);
    if (lane_in(part & beyond)) {
      const D4 c{r[8], r[9], r[10], r[11]}, d{r[12], r[13], r[14], r[15]}, e{r[16], r[17], r[18], r[19]},
          f{r[20], r[21], r[22], r[23]};
      const double m = rsqrt64(l2);
      sum = fma(__dmul_rn(m, m), far_field_bracket<ORDER>(x, y, z, m, b, c, d, e, f), sum);
      skip = past;
    }
    const uint64_t stay = part & ~beyond;
    if (leaf && stay != 0) {
      if (lane_in(stay)) pend.push(link & ~LINK_LEAF);
      if (__ballot(pend.n == (uint32_t)kPend64) != 0) pend.flush(tri, qx, qy, qz, ex);
    }
    i = wave_uniform((leaf || stay != 0) ? i + 1 : link);
  }
  pend.flush(tri, qx, qy, qz, ex);
  if (!isfinite(sum) && isfinite(qx) && isfinite(qy) && isfinite(qz)) {
    // a far field was not finite: the walk again, descending where it is not
    sum = 0.0;
    ex = SolidAngleSum<double>();
    for (uint32_t j = 0; j < nslots;) {
      uint32_t link;
      const bool far = record_far64<ORDER>(s64, j, link, qx, qy, qz, acc2, sum, [] {});
      const bool leaf = (link & LINK_LEAF) != 0;
      if (leaf && !far) ex.add(tri + 9 * (size_t)(link & ~LINK_LEAF), qx, qy, qz);
      j = (far && !leaf) ? link : j + 1;
    }
  }
  W[qi] = (sum + ex.total()) / (4.0 * PI_D);
}

// ---- FP64 re-evaluation of a few scattered queries: one wavefront per query ----
// A sequential walk is a chain of dependent record fetches as long as the
// query's path (thousands on a large mesh): a pass over a few hundred queries
// runs a handful of wavefronts for milliseconds.  Here the 64 lanes of a
// wavefront share one query's walk (frontier_walk, ring_walk.h).  The records
// visited and the terms are those of the sequential walk (each record's
// decision depends on the record and the query only); their FP64 sum is taken
// per lane and then across lanes in a fixed order, so the result is
// deterministic and differs from the sequential sum only by rounding.

// Records first .. end - 1 in rope order, every angle a term of its own: what
// a frontier walk whose ring is full leaves to one lane.
template <int ORDER>
__device__ __attribute__((noinline)) double subtree64(const double* __restrict__ s64, const float* __restrict__ tri,
                                                      uint32_t first, uint32_t end, double qx, double qy, double qz,
                                                      double acc2) {
  double sum = 0.0;
  for (uint32_t j = first; j < end;) {
    uint32_t link;
    const bool far = record_far64<ORDER>(s64, j, link, qx, qy, qz, acc2, sum, [] {});
    const bool leaf = (link & LINK_LEAF) != 0;
    if (leaf && !far) {
      const float* p = tri + 9 * (size_t)(link & ~LINK_LEAF);
      sum = __dadd_rn(sum, tri_solid_angle<double>(p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8], qx, qy, qz));
    }
    j = (far && !leaf) ? link : j + 1;
  }
  return sum;
}

// LDS of one query's frontier walk
struct FrontierLds {
  uint32_t ring[kFrontier];
  uint32_t far[kExactQueue];
};

// FP64 frontier walk of a query: W = sum / 4 pi, the same on every lane
template <int ORDER>
__device__ __forceinline__ double frontier_walk64(FrontierLds& lds, uint32_t lane, const double* __restrict__ s64,
                                                  const uint4* __restrict__ kids, uint32_t nslots,
                                                  const float* __restrict__ tri, double qx, double qy, double qz,
                                                  double acc2) {
  double part = 0.0;
  SolidAngleSum<double> ex;
  const auto exact = [&](uint32_t t) { ex.add(tri + 9 * (size_t)t, qx, qy, qz); };
  frontier_walk(
      lds.ring, lds.far, nullptr, lane, kids, nslots,
      [&](uint32_t i, uint4& k, uint32_t& link, uint32_t& t) {
        const auto descend = [&] {
          if (!(link & LINK_LEAF)) k = kids[i];
        };
        if (record_far64<ORDER>(s64, i, link, qx, qy, qz, acc2, part, descend)) return Visit::kDone;
        t = link & ~LINK_LEAF;
        return (link & LINK_LEAF) ? Visit::kExact : Visit::kDescend;
      },
      exact, exact,
      [&](uint32_t first, uint32_t end) {
        part = __dadd_rn(part, subtree64<ORDER>(s64, tri, first, end, qx, qy, qz, acc2));
      });
  return wave_sum(part + ex.total()) / (4.0 * PI_D);
}

// list[k] (k itself when list is null) for k < count (count = *dcount when
// given, else n): 4 queries per 256-thread block, one per wavefront,
// grid-strided.
template <int ORDER>
__global__ __launch_bounds__(256) void k_reeval64(const double* __restrict__ s64, const uint4* __restrict__ kids,
                                                  uint32_t nslots,
                                                  const float* __restrict__ tri,
                                                  const float* __restrict__ Q, const uint32_t* __restrict__ list,
                                                  int64_t n, const uint32_t* __restrict__ dcount, double acc2,
                                                  double* __restrict__ W) {
  __shared__ FrontierLds lds[4];
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t count = dcount ? (int64_t)*dcount : n;
  for (int64_t k = (int64_t)blockIdx.x * 4 + wv; k < count; k += (int64_t)gridDim.x * 4) {
    const int64_t qi = list ? (int64_t)list[k] : k;
    const double w = frontier_walk64<ORDER>(lds[wv], lane, s64, kids, nslots, tri, Q[3 * qi], Q[3 * qi + 1],
                                        Q[3 * qi + 2], acc2);
    if (lane == 0) W[qi] = w;
  }
}

// ---- small batches: one wavefront per query for the whole query ----
// A batch of a few thousand queries fills few wavefronts with the lane walk,
// and each lane's sequential walk is a chain of dependent record fetches as
// long as its path: at accuracy_scale 4.9 on a 434k-triangle mesh a batch of
// 1,000 queries takes 1.4 ms however few queries it has.  Here each query gets
// a wavefront and the frontier walk (ring_walk.h), so a query takes about one
// round per tree level and per 64 records.  The records visited and each term
// are those of the sequential walk (FP32 decisions and terms with the
// reference's rounding, FP64 near triangles in the mixed form); the sum is
// taken per lane and then across lanes in a fixed order, so results are
// deterministic and differ from the sequential walks' running sums only by
// rounding.  In the mixed form k_reeval64_band then walks the queries whose W
// falls in the ambiguous band again in FP64, so the batch needs no collection
// pass and no count.
//
// Few queries wait for memory, many queries for the vector cache, which
// serves one lane's 16 bytes a cycle where every lane reads another record.
// EARLY (below kEarlyFetchBelow queries) requests the whole record and the
// children's positions at once; otherwise the first 32 bytes decide what else
// a lane reads (5 pieces of 16 bytes a record instead of 7).  81,920
// triangles, early / as needed: 10.3 / 10.8 us (1,000 queries at
// accuracy_scale 2), 34 / 39 us (1,000 at 4.9), 41.5 / 41.9 us (2,000 at 4.9),
// 90 / 67 us (4,000 at 4.9).  Fetching records through LDS, eight lanes a
// record, measured between the two: its 8 KiB a wavefront halve the
// wavefronts in flight.  Against the walk by ranges of siblings with each
// triangle evaluated where it was met: 1,000 queries at 2 25 -> 10 us, 20,000
// at 2 108 -> 60 us, 60,000 at 3 399 -> 321 us; mixed form, 5,003 queries on
// 119,000 triangles at 4.9 182 -> 138 us, 60,000 on 5,000 triangles at 3
// 458 -> 171 us.
constexpr int64_t kEarlyFetchBelow = 2048;

// Records first .. end - 1 in rope order, the mixed form's near triangles in
// FP64: what a frontier walk whose ring is full leaves to one lane.
template <int ORDER, bool MIXED>
__device__ __attribute__((noinline)) double subtree32(const float4* __restrict__ slots,
                                                      const float* __restrict__ tri, uint32_t first, uint32_t end,
                                                      float qx, float qy, float qz, float acc2, float near_d) {
  float sum = 0.0f;
  double sum64 = 0.0;
  for (uint32_t j = first; j < end;) {
    const float4* r = slots + 6 * (size_t)j;
    const float4 a = r[0], b = r[1];
    const uint32_t link = __float_as_uint(b.w);
    const bool leaf = (link & LINK_LEAF) != 0;
    const float x = qx - a.x, y = qy - a.y, z = qz - a.z;
    const float l2 = __fadd_rn(__fadd_rn(__fmul_rn(x, x), __fmul_rn(y, y)), __fmul_rn(z, z));
    if (!(l2 <= __fmul_rn(a.w, acc2))) {
      const float o = far_field_poly<ORDER>(x, y, z, l2, b, r[2], r[3], r[4], r[5]);
      if (isfinite(o)) {
        sum = __fadd_rn(sum, o);
        j = leaf ? j + 1 : link;
        continue;
      }
    }
    if (leaf) {
      const float* p = tri + 9 * (size_t)(link & ~LINK_LEAF);
      if (MIXED && near_triangle(a.w, l2, near_d))
        sum64 = __dadd_rn(sum64,
                          tri_solid_angle<double>(p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8], qx, qy, qz));
      else
        sum = __fadd_rn(sum, tri_solid_angle_fast(p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8], qx, qy, qz));
    }
    ++j;
  }
  return (double)sum + sum64;
}

// FP32 and mixed forms (the FP64 form is k_reeval64 over every query).  FP32
// fits 8 wavefronts per SIMD; the mixed form's FP64 terms spill outside the
// walk at 8 and took 2 to 4% less time at 6 on batches of 60,000.
template <int ORDER, bool MIXED, bool EARLY>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(MIXED ? 6 : 8))) void k_walk_ring(
    const float4* __restrict__ slots, const uint4* __restrict__ kids, uint32_t nslots, const float* __restrict__ tri,
    const float* __restrict__ Q, int64_t nq, float acc2f, float near_d, double* __restrict__ W) {
  __shared__ FrontierLds lds[4];
  __shared__ uint32_t near_all[MIXED ? 4 * kExactQueue : 1];
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int64_t qi = (int64_t)blockIdx.x * 4 + wv; qi < nq; qi += (int64_t)gridDim.x * 4) {
    const float qx = Q[3 * qi], qy = Q[3 * qi + 1], qz = Q[3 * qi + 2];
    float p32 = 0.0f;
    double rest = 0.0;
    const auto exact = [&](uint32_t t) {
      const float* p = tri + 9 * (size_t)t;
      p32 = __fadd_rn(p32, tri_solid_angle_fast(p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8], qx, qy, qz));
    };
    const auto exact_near = [&](uint32_t t) {
      const float* p = tri + 9 * (size_t)t;
      if (MIXED)
        rest = __dadd_rn(rest, tri_solid_angle<double>(p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8], qx, qy, qz));
    };
    frontier_walk(
        lds[wv].ring, lds[wv].far, near_all + (MIXED ? wv * kExactQueue : 0), lane, kids, nslots,
        [&](uint32_t i, uint4& k, uint32_t& link, uint32_t& t) {
          const float4* r = slots + 6 * (size_t)i;
          const float4 a = r[0], b = r[1];
          float4 c, d, e, f;
          if (EARLY) c = r[2], d = r[3], e = r[4], f = r[5], k = kids[i];
          link = __float_as_uint(b.w);
          const bool leaf = (link & LINK_LEAF) != 0;
          const float x = qx - a.x, y = qy - a.y, z = qz - a.z;
          // rounded as the reference rounds it (no fused multiply-add)
          const float l2 = __fadd_rn(__fadd_rn(__fmul_rn(x, x), __fmul_rn(y, y)), __fmul_rn(z, z));
          const bool beyond = !(l2 <= __fmul_rn(a.w, acc2f));
          if (!EARLY && !beyond && !leaf) k = kids[i];  // on its way while the far fields are read
          if (beyond) {
            if (!EARLY) c = r[2], d = r[3], e = r[4], f = r[5];
            const float o = far_field_poly<ORDER>(x, y, z, l2, b, c, d, e, f);
            if (isfinite(o)) {
              p32 = __fadd_rn(p32, o);
              return Visit::kDone;
            }
            if (!EARLY && !leaf) k = kids[i];
          }
          if (!leaf) return Visit::kDescend;
          t = link & ~LINK_LEAF;
          return MIXED && near_triangle(a.w, l2, near_d) ? Visit::kExactNear : Visit::kExact;
        },
        exact, exact_near,
        [&](uint32_t first, uint32_t end) {
          rest = __dadd_rn(rest, subtree32<ORDER, MIXED>(slots, tri, first, end, qx, qy, qz, acc2f, near_d));
        });
    const float s32 = wave_sum(p32);
    double w = (double)s32;
    if (__ballot(rest != 0.0) != 0) w += wave_sum(rest);
    if (lane == 0) W[qi] = w / (4.0 * PI_D);
  }
}

// Mixed form after k_walk_ring: queries whose W falls in the ambiguous band
// are walked again in FP64, one wavefront per query (the others exit at once).
// A kernel of its own so that the FP64 walk's registers do not limit the
// occupancy of the FP32 walk.
template <int ORDER>
__global__ __launch_bounds__(256) void k_reeval64_band(const double* __restrict__ s64, const uint4* __restrict__ kids,
                                                  uint32_t nslots,
                                                       const float* __restrict__ tri, const float* __restrict__ Q,
                                                       int64_t nq, double acc2, double band, double* __restrict__ W) {
  __shared__ FrontierLds lds[4];
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int64_t qi = (int64_t)blockIdx.x * 4 + wv; qi < nq; qi += (int64_t)gridDim.x * 4) {
    if (fabs(W[qi] - 0.5) >= band) continue;  // wave-uniform; NaN is walked again
    const double w = frontier_walk64<ORDER>(lds[wv], lane, s64, kids, nslots, tri, Q[3 * qi], Q[3 * qi + 1],
                                        Q[3 * qi + 2], acc2);
    if (lane == 0) W[qi] = w;
  }
}

// queries with |w - 0.5| < band, and queries whose walk gave NaN (more near
// triangles than the walk notes), are collected for the FP64 re-evaluation
__global__ void k_collect_ambiguous(const double* __restrict__ W, int64_t nq, double band, uint32_t* __restrict__ list,
                                    uint32_t* __restrict__ count) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nq) return;
  const double w = W[i];
  if (isnan(w) || fabs(w - 0.5) < band) {
    const uint32_t p = atomicAdd(count, 1u);
    list[p] = (uint32_t)i;
  }
}

// Morton key of a query (30 bits) over the mesh bbox, for query ordering
__device__ __forceinline__ uint32_t expand_bits10(uint32_t v) {
  v = (v * 0x00010001u) & 0xFF0000FFu;
  v = (v * 0x00000101u) & 0x0F00F00Fu;
  v = (v * 0x00000011u) & 0xC30C30C3u;
  v = (v * 0x00000005u) & 0x49249249u;
  return v;
}
__global__ void k_morton_q(const float* __restrict__ Q, int64_t nq, float lx, float ly, float lz, float sx, float sy,
                           float sz, uint32_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nq) return;
  float fx = (Q[3 * i] - lx) * sx, fy = (Q[3 * i + 1] - ly) * sy, fz = (Q[3 * i + 2] - lz) * sz;
  fx = fminf(fmaxf(fx, 0.0f), 1023.0f);
  fy = fminf(fmaxf(fy, 0.0f), 1023.0f);
  fz = fminf(fmaxf(fz, 0.0f), 1023.0f);
  keys[i] = (expand_bits10((uint32_t)fx) << 2) | (expand_bits10((uint32_t)fy) << 1) | expand_bits10((uint32_t)fz);
  vals[i] = (uint32_t)i;
}

// 30-bit Hilbert key of a query (10 bits per axis, same quantisation as the
// Morton key), by Skilling's transpose algorithm ("Programming the Hilbert
// curve", AIP Conf. Proc. 707, 2004): undo the excess work, Gray-encode,
// interleave.  Consecutive keys are always neighbouring cells (the Morton
// curve jumps), so a wavefront of consecutive queries spans a more compact
// region: a CPU simulation of the wave walk on the 81,920-triangle workload
// at accuracy_scale 4.9 gave 1,471 record steps per wavefront against 1,544.
__device__ __forceinline__ uint32_t hilbert3_10(uint32_t x0, uint32_t x1, uint32_t x2) {
  uint32_t X[3] = {x0, x1, x2};
  // branch-free: m is all ones where bit q of X[i] is set
#pragma unroll
  for (int b = 9; b >= 1; --b) {
    const uint32_t p = (1u << b) - 1u;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const uint32_t m = 0u - ((X[i] >> b) & 1u);
      X[0] ^= p & m;
      const uint32_t t = (X[0] ^ X[i]) & p & ~m;
      X[0] ^= t;
      X[i] ^= t;
    }
  }
  X[1] ^= X[0];
  X[2] ^= X[1];
  uint32_t t = 0;
#pragma unroll
  for (int b = 9; b >= 1; --b) t ^= ((1u << b) - 1u) & (0u - ((X[2] >> b) & 1u));
  X[0] ^= t;
  X[1] ^= t;
  X[2] ^= t;
  uint32_t h = 0;
#pragma unroll
  for (int b = 9; b >= 0; --b) h = (h << 3) | (((X[0] >> b) & 1u) << 2) | (((X[1] >> b) & 1u) << 1) | ((X[2] >> b) & 1u);
  return h;
}
struct HilbertKey {
  const float* Q;
  float lx, ly, lz, sx, sy, sz;
  __device__ __forceinline__ uint32_t operator()(int64_t i) const {
    float fx = (Q[3 * i] - lx) * sx, fy = (Q[3 * i + 1] - ly) * sy, fz = (Q[3 * i + 2] - lz) * sz;
    fx = fminf(fmaxf(fx, 0.0f), 1023.0f);
    fy = fminf(fmaxf(fy, 0.0f), 1023.0f);
    fz = fminf(fmaxf(fz, 0.0f), 1023.0f);
    return hilbert3_10((uint32_t)fx, (uint32_t)fy, (uint32_t)fz);
  }
};

// ---------------------------------------------------------------------------
// host orchestration
void compute_levels(const uint32_t* nodes, int64_t nn, Levels& L, hipStream_t st) {
  DevBuf<int32_t> parent(nn), depth(nn);
  DevBuf<uint32_t> hist(4097);
  DevBuf<int32_t> maxd(1);
  GWN_HIP(hipMemsetAsync(hist.p, 0, hist.bytes(), st));
  GWN_HIP(hipMemsetAsync(maxd.p, 0, sizeof(int32_t), st));
  const unsigned g = div_up(nn, 256);
  hipLaunchKernelGGL(k_parent, dim3(g), dim3(256), 0, st, nodes, nn, parent.p);
  check_launch("k_parent");
  hipLaunchKernelGGL(k_depth, dim3(g), dim3(256), 0, st, parent.p, nn, depth.p, hist.p, maxd.p);
  check_launch("k_depth");
  int32_t md = 0;
  GWN_HIP(hipMemcpyAsync(&md, maxd.p, sizeof(int32_t), hipMemcpyDeviceToHost, st));
  GWN_HIP(hipStreamSynchronize(st));
  GWN_CHECK(md < 4000, GWN_ERR_INVALID, "tree too deep");
  std::vector<uint32_t> h(md + 1);
  GWN_HIP(hipMemcpyAsync(h.data(), hist.p, sizeof(uint32_t) * (md + 1), hipMemcpyDeviceToHost, st));
  GWN_HIP(hipStreamSynchronize(st));
  L.maxdepth = md;
  L.offset.assign(md + 2, 0);
  for (int d = 0; d <= md; ++d) L.offset[d + 1] = L.offset[d] + h[d];
  GWN_HIP(hipMemcpyAsync(hist.p, L.offset.data(), sizeof(uint32_t) * (md + 1), hipMemcpyHostToDevice, st));
  L.order.alloc(nn);
  hipLaunchKernelGGL(k_bucket, dim3(g), dim3(256), 0, st, depth.p, nn, hist.p, L.order.p);
  check_launch("k_bucket");
  GWN_HIP(hipStreamSynchronize(st));
}

// First slot of every node in the rope layout, top-down from the root's 0.
void rope_first_slots(const Levels& L, const uint32_t* nodes, const uint32_t* nsub, uint32_t* first,
                      hipStream_t st) {
  GWN_HIP(hipMemsetAsync(first, 0, sizeof(uint32_t), st));
  for (int d = 0; d <= L.maxdepth; ++d) {
    const int64_t cnt = L.offset[d + 1] - L.offset[d];
    if (!cnt) continue;
    hipLaunchKernelGGL(k_positions, dim3(div_up(cnt, 256)), dim3(256), 0, st, L.order.p + L.offset[d], cnt, nodes,
                       nsub, first);
    check_launch("k_positions");
  }
}

template <typename T>
static void upward(gwn_soup* s, const Levels& L, T* boxdata, DevBuf<uint32_t>& nsub, hipStream_t st) {
  const int64_t nn = s->nnodes;
  DevBuf<Local<T>> local(nn);
  for (int d = L.maxdepth; d >= 0; --d) {
    const int64_t cnt = L.offset[d + 1] - L.offset[d];
    if (!cnt) continue;
    hipLaunchKernelGGL(k_upward<T>, dim3(div_up(cnt, 128)), dim3(128), 0, st, L.order.p + L.offset[d], cnt,
                       s->nodes.p, s->U.p, s->F.p, s->boxes.p, s->order, local.p, boxdata, nsub.p);
    check_launch("k_upward");
  }
  GWN_HIP(hipStreamSynchronize(st));
}

// FP64 moments of every slot (the reference's item()/post() in double), in
// the field order of k_write_slots64: the all-FP64 form and the FP64
// re-evaluation of the mixed form read them.
static void build_fp64_moments(gwn_soup* s, const Levels& L, hipStream_t st) {
  const int64_t nn = s->nnodes;
  DevBuf<double> bd64(92 * nn);
  DevBuf<uint32_t> nsub(nn), first(nn);
  upward<double>(s, L, bd64.p, nsub, st);
  rope_first_slots(L, s->nodes.p, nsub.p, first.p, st);
  s->slots64.alloc(24 * (size_t)s->nslots);
  hipLaunchKernelGGL(k_write_slots64, dim3(div_up(nn, 256)), dim3(256), 0, st, nn, s->nodes.p, bd64.p, first.p,
                     nsub.p, s->slots64.p);
  check_launch("k_write_slots64");
  GWN_HIP(hipStreamSynchronize(st));
}

static void build_cost_grid(gwn_soup* s, hipStream_t st);

// Tree levels, FP32 BoxData (the reference's), the rope-ordered slot records,
// their FP64 moments and the cost grid.  After this the handle is read-only
// to queries.
void soup_finish_build(gwn_soup* s, hipStream_t st) {
  const int64_t nn = s->nnodes;
  if (nn == 0) {
    s->nslots = 0;
    return;
  }
  Levels L;
  compute_levels(s->nodes.p, nn, L, st);
  s->depth = L.maxdepth;
  s->boxdata.alloc(92 * nn);
  DevBuf<uint32_t> nsub(nn), first(nn);
  upward<float>(s, L, s->boxdata.p, nsub, st);
  uint32_t total = 0;
  GWN_HIP(hipMemcpyAsync(&total, nsub.p, sizeof(uint32_t), hipMemcpyDeviceToHost, st));
  rope_first_slots(L, s->nodes.p, nsub.p, first.p, st);
  GWN_HIP(hipStreamSynchronize(st));
  s->nslots = total;
  s->slots.alloc(6 * (size_t)total);
  s->kids.alloc((size_t)total + 1);
  hipLaunchKernelGGL(k_write_slots, dim3(div_up(nn, 256)), dim3(256), 0, st, nn, s->nodes.p, s->boxdata.p, nsub.p,
                     first.p, total, s->slots.p, s->kids.p);
  check_launch("k_write_slots");
  if (!s->boxes_only) {
    build_fp64_moments(s, L, st);
    build_cost_grid(s, st);
  }
  GWN_HIP(hipStreamSynchronize(st));
}

// Slot boxes for closest-point queries (and the antipodal rays), built by the
// first call that needs them.  Concurrent first calls on one handle build
// them once: the others wait on dist_mu, and the boxes are complete on the
// device (the build ends with a stream synchronisation) before dist_ready is
// set.
void soup_ensure_dist(gwn_soup* s, hipStream_t st) {
  if (s->dist_ready.load(std::memory_order_acquire) || s->nnodes == 0) return;
  std::lock_guard<std::mutex> lock(s->dist_mu);
  if (s->dist_ready.load(std::memory_order_relaxed)) return;
  const int64_t nn = s->nnodes;
  Levels L;
  compute_levels(s->nodes.p, nn, L, st);
  DevBuf<float> nbox(6 * (size_t)nn);
  for (int d = L.maxdepth; d >= 0; --d) {
    const int64_t cnt = L.offset[d + 1] - L.offset[d];
    if (!cnt) continue;
    hipLaunchKernelGGL(k_node_boxes, dim3(div_up(cnt, 128)), dim3(128), 0, st, L.order.p + L.offset[d], cnt,
                       s->nodes.p, s->V64.p, s->F.p, nbox.p);
    check_launch("k_node_boxes");
  }
  // first slot of every node, top-down, following the links of the rope
  DevBuf<uint32_t> first(nn);
  GWN_HIP(hipMemsetAsync(first.p, 0, sizeof(uint32_t), st));
  for (int d = 0; d <= L.maxdepth; ++d) {
    const int64_t cnt = L.offset[d + 1] - L.offset[d];
    if (!cnt) continue;
    hipLaunchKernelGGL(k_positions_rope, dim3(div_up(cnt, 256)), dim3(256), 0, st, L.order.p + L.offset[d], cnt,
                       s->nodes.p, s->slots.p, first.p);
    check_launch("k_positions_rope");
  }
  DevBuf<float4> db(2 * (size_t)s->nslots);
  hipLaunchKernelGGL(k_write_dbox, dim3(div_up(nn, 256)), dim3(256), 0, st, nn, s->nodes.p, nbox.p, s->V64.p,
                     s->F.p, first.p, s->slots.p, db.p);
  check_launch("k_write_dbox");
  DevBuf<float4> planes;
  for (int k = 0; k < 3; ++k) {
    const float c = 0.5f * s->bbox[k] + 0.5f * s->bbox[3 + k];
    s->centre[k] = std::isfinite(c) ? c : 0.0f;
  }
  if (!s->boxes_only) {
    planes.alloc(4 * (size_t)s->nf);
    hipLaunchKernelGGL(k_face_planes, dim3(div_up(s->nf, 256)), dim3(256), 0, st, s->V64.p, s->F.p, s->nf,
                       s->centre[0], s->centre[1], s->centre[2], planes.p);
    check_launch("k_face_planes");
  }
  GWN_HIP(hipStreamSynchronize(st));
  s->dbox = std::move(db);
  s->planes = std::move(planes);
  s->dist_ready.store(true, std::memory_order_release);
}

void soup_setup(gwn_soup* s, hipStream_t st) {
  const int64_t nf = s->nf;
  s->boxes.alloc(6 * (size_t)nf);
  s->tri.alloc(9 * (size_t)nf);
  if (nf > 0) {
    hipLaunchKernelGGL(k_tri_setup, dim3(div_up(nf, 256)), dim3(256), 0, st, s->U.p, s->F.p, nf, s->boxes.p,
                       s->tri.p);
    check_launch("k_tri_setup");
  }
}

// Workspace of one sorted query call: Hilbert keys, the query permutation,
// sort temp, and the list and count of ambiguous queries (mixed form).
size_t soup_query_work_bytes(int64_t nq) {
  const size_t a = 256;
  auto up = [&](size_t b) { return (b + a - 1) / a * a; };
  return up(4 * (size_t)nq) * 2 + up(radix_sort_temp_bytes(nq, false)) + up(4 * (size_t)nq) + up(4);
}

// 30-bit Morton keys of the queries over a box (queries outside are clamped
// to it), and the identity permutation to be sorted along with them
void morton_keys(const float* Q, int64_t nq, const float* bb, uint32_t* keys, uint32_t* vals, hipStream_t st) {
  const float ex = std::max(bb[3] - bb[0], 1e-30f), ey = std::max(bb[4] - bb[1], 1e-30f),
              ez = std::max(bb[5] - bb[2], 1e-30f);
  hipLaunchKernelGGL(k_morton_q, dim3(div_up(nq, 256)), dim3(256), 0, st, Q, nq, bb[0], bb[1], bb[2], 1024.0f / ex,
                     1024.0f / ey, 1024.0f / ez, keys, vals);
  check_launch("k_morton_q");
}


// ---------------------------------------------------------------------------
// Block order of the wave walks.  A wavefront's walk time is the union of its
// 64 queries' paths, and it varies several-fold over a batch (queries near the
// surface open many more records); dispatched in Hilbert order, the costly
// blocks of a region can start last and run on alone at the end of the
// launch.  The walks instead take each XCD's blocks costliest first (longest
// processing time first), with a block's cost estimated from the cost grid
// built with the tree.  The order changes which blocks run when, never which
// queries a wavefront holds, so every result is the same bit for bit.

// Records a query at each cell centre of the cost grid visits at accuracy
// scale 2 (the near/far decisions of k_traverse, without the sums), as a
// log-scale byte: min(255, 15 log2(1 + n)).
__global__ __launch_bounds__(256) void k_cost_grid(const float4* __restrict__ slots, uint32_t nslots, float lx,
                                                   float ly, float lz, float hx, float hy, float hz,
                                                   uint8_t* __restrict__ grid) {
  constexpr int G = kCostGrid;
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= G * G * G) return;
  const float qx = lx + (c % G + 0.5f) * hx, qy = ly + ((c / G) % G + 0.5f) * hy, qz = lz + (c / (G * G) + 0.5f) * hz;
  uint32_t i = 0, n = 0;
  while (i < nslots) {
    const float4 a = slots[6 * (size_t)i];
    const uint32_t link = __float_as_uint(slots[6 * (size_t)i + 1].w);
    const bool leaf = (link & LINK_LEAF) != 0;
    const float x = qx - a.x, y = qy - a.y, z = qz - a.z;
    const float l2 = x * x + y * y + z * z;
    ++n;
    if (!(l2 <= a.w * 4.0f)) {
      i = leaf ? i + 1 : link;
    } else {
      n += leaf;
      ++i;
    }
  }
  grid[c] = (uint8_t)fminf(255.0f, 15.0f * log2f(1.0f + (float)n));
}

static void build_cost_grid(gwn_soup* s, hipStream_t st) {
  constexpr int G = kCostGrid;
  s->cost_grid.alloc((size_t)G * G * G);
  const float* bb = s->bbox;
  hipLaunchKernelGGL(k_cost_grid, dim3(div_up(G * G * G, 256)), dim3(256), 0, st, s->slots.p, (uint32_t)s->nslots,
                     bb[0], bb[1], bb[2], (bb[3] - bb[0]) / G, (bb[4] - bb[1]) / G, (bb[5] - bb[2]) / G,
                     s->cost_grid.p);
  check_launch("k_cost_grid");
}

// Estimated cost of each block of 256 sorted queries: the grid's largest
// value over the block's queries.
__global__ __launch_bounds__(256) void k_block_cost(const float* __restrict__ Q, const uint32_t* __restrict__ perm,
                                                    int64_t nq, float lx, float ly, float lz, float sx, float sy,
                                                    float sz, const uint8_t* __restrict__ grid,
                                                    uint8_t* __restrict__ cost) {
  constexpr int G = kCostGrid;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int v = 0;
  if (t < nq) {
    const int64_t qi = perm[t];
    const int ix = min(G - 1, max(0, (int)((Q[3 * qi] - lx) * sx)));
    const int iy = min(G - 1, max(0, (int)((Q[3 * qi + 1] - ly) * sy)));
    const int iz = min(G - 1, max(0, (int)((Q[3 * qi + 2] - lz) * sz)));
    v = grid[(iz * G + iy) * G + ix];
  }
  for (int o = 32; o >= 1; o >>= 1) v = max(v, __shfl_xor(v, o));
  __shared__ int wmax[4];
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) cost[blockIdx.x] = (uint8_t)max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
}

// Block order: one workgroup per XCD's range of logical blocks (the ranges of
// xcd_block()), a counting sort of its blocks by decreasing cost.  Blocks of
// equal cost land in any order.
__global__ __launch_bounds__(256) void k_block_order(const uint8_t* __restrict__ cost, uint32_t nb,
                                                     uint32_t* __restrict__ order) {
  __shared__ uint32_t count[256];
  const uint32_t x = blockIdx.x, q = nb / 8, r = nb % 8;
  const uint32_t lo = x * q + (x < r ? x : r), hi = lo + q + (x < r ? 1 : 0);
  count[threadIdx.x] = 0;
  __syncthreads();
  for (uint32_t b = lo + threadIdx.x; b < hi; b += blockDim.x) atomicAdd(&count[255 - cost[b]], 1u);
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t run = lo;
    for (int k = 0; k < 256; ++k) {
      const uint32_t n = count[k];
      count[k] = run;
      run += n;
    }
  }
  __syncthreads();
  for (uint32_t b = lo + threadIdx.x; b < hi; b += blockDim.x) order[atomicAdd(&count[255 - cost[b]], 1u)] = b;
}

// order (nb = ceil(nq / 256) entries) and cost (nb bytes) are workspace
void block_order(const uint8_t* grid, const float* bb, const float* Q, const uint32_t* perm, int64_t nq,
                 uint32_t* order, uint8_t* cost, hipStream_t st) {
  constexpr int G = kCostGrid;
  const uint32_t nb = (uint32_t)div_up(nq, 256);
  const float ex = std::max(bb[3] - bb[0], 1e-30f), ey = std::max(bb[4] - bb[1], 1e-30f),
              ez = std::max(bb[5] - bb[2], 1e-30f);
  hipLaunchKernelGGL(k_block_cost, dim3(nb), dim3(256), 0, st, Q, perm, nq, bb[0], bb[1], bb[2], G / ex, G / ey,
                     G / ez, grid, cost);
  check_launch("k_block_cost");
  hipLaunchKernelGGL(k_block_order, dim3(8), dim3(256), 0, st, cost, nb, order);
  check_launch("k_block_order");
}

// 30-bit Hilbert keys of the queries over a box (clamped to it): the order in
// which the tree walks take their queries
void hilbert_keys(const float* Q, int64_t nq, const float* bb, uint32_t* keys, uint32_t* vals, void* tmp,
                  hipStream_t st) {
  const float ex = std::max(bb[3] - bb[0], 1e-30f), ey = std::max(bb[4] - bb[1], 1e-30f),
              ez = std::max(bb[5] - bb[2], 1e-30f);
  const HilbertKey key{Q, bb[0], bb[1], bb[2], 1024.0f / ex, 1024.0f / ey, 1024.0f / ez};
  const int64_t nt = radix_tiles(nq);
  hipLaunchKernelGGL(k_rs_keys<HilbertKey>, dim3((unsigned)nt), dim3(RS_KEY_THREADS), 0, st, key, nq, keys, vals,
                     radix_counts_u32(tmp, nq), nt);
  check_launch("k_rs_keys");
}

// ---------------------------------------------------------------------------
// Scratch-free query (gwn_soup_query_device_noalloc).  Its workspace is this
// file-scope device array, not pooled memory: each device that runs the
// library holds one copy for the life of the process.  Host code never uses
// the array's name as an address; it uses the device address that
// hipGetSymbolAddress returns, looked up once per device (with that device
// current) on the first call there.  Every call on a device shares that
// device's copy, so calls that overlap on one device race; the contents a
// call needs zeroed (the ambiguous-query count) are zeroed by a kernel on the
// call's stream.
constexpr int64_t kNoAllocMaxQueries = (int64_t)1 << 20;
constexpr size_t kNoAllocScratchBytes = (size_t)22 << 20;  // >= soup_query_work_bytes(kNoAllocMaxQueries)
constexpr int kNoAllocMaxDevices = 64;
static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

static uint8_t* noalloc_scratch() {
  static std::mutex mu;
  static uint8_t* ptr[kNoAllocMaxDevices] = {};
  int dev = 0;
  GWN_HIP(hipGetDevice(&dev));
  GWN_CHECK(dev >= 0 && dev < kNoAllocMaxDevices, GWN_ERR_NODEVICE, "device ordinal out of range");
  std::lock_guard<std::mutex> lock(mu);
  if (ptr[dev] == nullptr) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) {
      (void)hipGetLastError();
      throw Error{GWN_ERR_HIP, std::string("hipGetSymbolAddress of the query scratch failed: ") + hipGetErrorString(e)};
    }
    GWN_CHECK(soup_query_work_bytes(kNoAllocMaxQueries) <= kNoAllocScratchBytes, GWN_ERR_INVALID,
              "scratch-free query: workspace layout exceeds the static scratch");
    ptr[dev] = static_cast<uint8_t*>(p);
  }
  return ptr[dev];
}

int64_t soup_noalloc_max_queries() { return kNoAllocMaxQueries; }

int soup_walk_for(const gwn_soup* s, int64_t nq, bool latency_bound) {
  if (nq < kRingMaxQueries) return WALK_RING;
  return latency_bound && s->nslots >= (1 << 17) ? WALK_WAVE_HANDOVER : WALK_WAVE;
}

void soup_query_device(const gwn_soup* s, const float* Q, int64_t nq, float accuracy_scale, int precision,
                       double* W, hipStream_t st) {
  if (nq <= 0) return;
  const int walk = soup_walk_for(s, nq, false);
  if (walk == WALK_RING) {
    soup_query_device_ws(s, Q, nq, accuracy_scale, precision, W, st, nullptr, 0, WALK_RING);
    return;
  }
  Scratch ws(soup_query_work_bytes(nq), st);
  soup_query_device_ws(s, Q, nq, accuracy_scale, precision, W, st, ws.p, ws.capacity, walk);
}

// The scratch-free form of soup_query_device: same kernels, same results;
// the workspace is the static scratch, the mixed form's FP64 re-evaluation is
// sized on the device (no host round trip) and no timing events are made.
void soup_query_device_noalloc(const gwn_soup* s, const float* Q, int64_t nq, float accuracy_scale, int precision,
                               double* W, hipStream_t st) {
  GWN_CHECK(nq <= kNoAllocMaxQueries, GWN_ERR_INVALID,
            "scratch-free query: at most 1,048,576 queries per call (got " + std::to_string(nq) + ")");
  if (nq <= 0) return;
  const int walk = soup_walk_for(s, nq, false);
  if (walk == WALK_RING) {
    soup_query_device_ws(s, Q, nq, accuracy_scale, precision, W, st, nullptr, 0, WALK_RING, WS_NO_PROFILE);
    return;
  }
  uint8_t* ws = noalloc_scratch();
  soup_query_device_ws(s, Q, nq, accuracy_scale, precision, W, st, ws, kNoAllocScratchBytes, walk,
                       WS_DEVICE_COUNT | WS_NO_PROFILE);
}

// FP64 walk over nq queries in the order perm
static void launch_traverse64(const gwn_soup* s, unsigned g, hipStream_t st, const float* Q, const uint32_t* perm,
                              const uint32_t* order, int64_t nq, double a2, double* W) {
  const uint32_t ns = (uint32_t)s->nslots;
  switch (s->order) {
    case 0: hipLaunchKernelGGL(k_traverse64<0>, dim3(g), dim3(256), 0, st, s->slots64.p, ns, s->tri.p, Q, perm, order, nq, a2, W); break;
    case 1: hipLaunchKernelGGL(k_traverse64<1>, dim3(g), dim3(256), 0, st, s->slots64.p, ns, s->tri.p, Q, perm, order, nq, a2, W); break;
    default: hipLaunchKernelGGL(k_traverse64<2>, dim3(g), dim3(256), 0, st, s->slots64.p, ns, s->tri.p, Q, perm, order, nq, a2, W); break;
  }
  check_launch("k_traverse64");
}

// one wavefront per query (k_walk_ring), 4 per block
static void launch_walk_ring(const gwn_soup* s, const float* Q, int64_t nq, float accuracy_scale, int precision,
                             double* W, hipStream_t st, bool prof_on) {
  const uint32_t ns = (uint32_t)s->nslots;
  const float acc2 = accuracy_scale * accuracy_scale;
  const double a2 = (double)accuracy_scale * (double)accuracy_scale;
  const float nd = s->mixed.near_dist;
  const double band = (double)s->mixed.ambiguous_band;
  const unsigned g = (unsigned)div_up(nq, 4);
  ProfileScope prof("soup_walk_ring", st, prof_on);
  if (precision == GWN_PREC_FP64) {
    switch (s->order) {
      case 0: hipLaunchKernelGGL(k_reeval64<0>, dim3(g), dim3(256), 0, st, s->slots64.p, s->kids.p, ns, s->tri.p, Q, nullptr, nq, nullptr, a2, W); break;
      case 1: hipLaunchKernelGGL(k_reeval64<1>, dim3(g), dim3(256), 0, st, s->slots64.p, s->kids.p, ns, s->tri.p, Q, nullptr, nq, nullptr, a2, W); break;
      default: hipLaunchKernelGGL(k_reeval64<2>, dim3(g), dim3(256), 0, st, s->slots64.p, s->kids.p, ns, s->tri.p, Q, nullptr, nq, nullptr, a2, W); break;
    }
    check_launch("k_reeval64");
    return;
  }
  const bool early = nq < kEarlyFetchBelow;
#define GWN_LAUNCH_R(O, M)                                                                                          \
  do {                                                                                                              \
    if (early)                                                                                                      \
      hipLaunchKernelGGL((k_walk_ring<O, M, true>), dim3(g), dim3(256), 0, st, s->slots.p, s->kids.p, ns, s->tri.p, \
                         Q, nq, acc2, nd, W);                                                                       \
    else                                                                                                            \
      hipLaunchKernelGGL((k_walk_ring<O, M, false>), dim3(g), dim3(256), 0, st, s->slots.p, s->kids.p, ns,          \
                         s->tri.p, Q, nq, acc2, nd, W);                                                             \
  } while (0)
  const bool mixed = precision == GWN_PREC_MIXED;
  switch (s->order) {
    case 0: if (mixed) GWN_LAUNCH_R(0, true); else GWN_LAUNCH_R(0, false); break;
    case 1: if (mixed) GWN_LAUNCH_R(1, true); else GWN_LAUNCH_R(1, false); break;
    default: if (mixed) GWN_LAUNCH_R(2, true); else GWN_LAUNCH_R(2, false); break;
  }
#undef GWN_LAUNCH_R
  check_launch("k_walk_ring");
  if (mixed) {
    switch (s->order) {
      case 0: hipLaunchKernelGGL(k_reeval64_band<0>, dim3(g), dim3(256), 0, st, s->slots64.p, s->kids.p, ns, s->tri.p, Q, nq, a2, band, W); break;
      case 1: hipLaunchKernelGGL(k_reeval64_band<1>, dim3(g), dim3(256), 0, st, s->slots64.p, s->kids.p, ns, s->tri.p, Q, nq, a2, band, W); break;
      default: hipLaunchKernelGGL(k_reeval64_band<2>, dim3(g), dim3(256), 0, st, s->slots64.p, s->kids.p, ns, s->tri.p, Q, nq, a2, band, W); break;
    }
    check_launch("k_reeval64_band");
  }
}

// Query with caller-provided device workspace of soup_query_work_bytes(nq)
// bytes (none for WALK_RING); calls with distinct workspaces may run
// concurrently on distinct streams against the same tree.  flags:
// WS_DEVICE_COUNT launches the mixed form's FP64 re-evaluation over every
// query with the count read on the device (no host round trip); WS_NO_PROFILE
// creates no kernel-timing events.
void soup_query_device_ws(const gwn_soup* s, const float* Q, int64_t nq, float accuracy_scale, int precision,
                          double* W, hipStream_t st, uint8_t* workspace, size_t ws_bytes, int walk, int flags) {
  if (nq <= 0) return;
  const bool prof_on = (flags & WS_NO_PROFILE) == 0;
  if (s->nslots == 0) {
    fill_device<double>(W, nq, 0.0, st);
    return;
  }
  if (walk == WALK_RING) {
    launch_walk_ring(s, Q, nq, accuracy_scale, precision, W, st, prof_on);
    return;
  }
  GWN_CHECK(walk == WALK_WAVE || walk == WALK_WAVE_HANDOVER, GWN_ERR_INVALID, "unknown walk");
  GWN_CHECK(ws_bytes >= soup_query_work_bytes(nq), GWN_ERR_INVALID, "query workspace too small");
  uint8_t* w = workspace;
  auto take = [&](size_t b) {
    uint8_t* p = w;
    w += (b + 255) / 256 * 256;
    return p;
  };
  uint32_t* keys = (uint32_t*)take(4 * (size_t)nq);
  uint32_t* perm = (uint32_t*)take(4 * (size_t)nq);
  {
    const size_t tmpb = radix_sort_temp_bytes(nq, false);
    void* tmp = take(tmpb);
    hilbert_keys(Q, nq, s->bbox, keys, perm, tmp, st);
    ProfileScope prof("radix_sort", st, prof_on);
    radix_sort_counted_u32(keys, perm, nq, 30, tmp, tmpb, st);
  }
  uint32_t* amb = (uint32_t*)take(4 * (size_t)nq);
  uint32_t* ambn = (uint32_t*)take(4);
  const unsigned g = div_up(nq, 256);
  // the sort keys are spent: their space holds the block order (g entries)
  // and the block costs (g bytes), 5g <= 4 nq bytes rounded up to 256
  uint32_t* border = keys;
  {
    ProfileScope prof("block_order", st, prof_on);
    block_order(s->cost_grid.p, s->bbox, Q, perm, nq, border, (uint8_t*)(border + g), st);
  }

  const float acc2 = accuracy_scale * accuracy_scale;
  const uint32_t ns = (uint32_t)s->nslots;
  if (precision == GWN_PREC_FP64) {
    const double a2 = (double)accuracy_scale * (double)accuracy_scale;
    ProfileScope prof("soup_traverse64", st, prof_on);
    launch_traverse64(s, g, st, Q, perm, border, nq, a2, W);
    return;
  }
  const bool mixed = precision == GWN_PREC_MIXED;
  const float nd = s->mixed.near_dist;
#define GWN_LAUNCH_T(O, M)                                                                                      \
  do {                                                                                                          \
    if (walk == WALK_WAVE)                                                                                      \
      hipLaunchKernelGGL((k_traverse<O, M, false>), dim3(g), dim3(256), 0, st, s->slots.p, ns, s->tri.p, Q, perm, \
                         border, nq, acc2, nd, W);                                                              \
    else                                                                                                        \
      hipLaunchKernelGGL((k_traverse<O, M, true>), dim3(g), dim3(256), 0, st, s->slots.p, ns, s->tri.p, Q, perm, \
                         border, nq, acc2, nd, W);                                                              \
  } while (0)
  {
    ProfileScope prof("soup_traverse", st, prof_on);
    if (mixed) {
      switch (s->order) {
        case 0: GWN_LAUNCH_T(0, true); break;
        case 1: GWN_LAUNCH_T(1, true); break;
        default: GWN_LAUNCH_T(2, true); break;
      }
    } else {
      switch (s->order) {
        case 0: GWN_LAUNCH_T(0, false); break;
        case 1: GWN_LAUNCH_T(1, false); break;
        default: GWN_LAUNCH_T(2, false); break;
      }
    }
  }
#undef GWN_LAUNCH_T
  check_launch("k_traverse");
  if (mixed) {
    fill_device<uint32_t>(ambn, 1, 0u, st);
    hipLaunchKernelGGL(k_collect_ambiguous, dim3(g), dim3(256), 0, st, W, nq, (double)s->mixed.ambiguous_band, amb,
                       ambn);
    check_launch("k_collect_ambiguous");
    const double a2 = (double)accuracy_scale * (double)accuracy_scale;
    int64_t na64 = 0;
    const uint32_t* dcount = nullptr;
    if (flags & WS_DEVICE_COUNT) {
      // bounded by every query; the kernel reads the count on the device
      na64 = nq;
      dcount = ambn;
    } else {
      // the count comes back to the host so that the FP64 pass is launched at
      // its size, or not at all
      uint32_t na = 0;
      GWN_HIP(hipMemcpyAsync(&na, ambn, 4, hipMemcpyDeviceToHost, st));
      GWN_HIP(hipStreamSynchronize(st));
      na64 = na;
    }
    if (na64 > 0) {
      // one wavefront per query, four per block; with the count on the
      // device the grid is capped and strides over the list
      const unsigned gr = dcount ? (unsigned)std::min<int64_t>(div_up(na64, 4), 2048) : (unsigned)div_up(na64, 4);
      ProfileScope prof("soup_reeval64", st, prof_on);
      switch (s->order) {
        case 0: hipLaunchKernelGGL(k_reeval64<0>, dim3(gr), dim3(256), 0, st, s->slots64.p, s->kids.p, ns, s->tri.p, Q, amb, na64, dcount, a2, W); break;
        case 1: hipLaunchKernelGGL(k_reeval64<1>, dim3(gr), dim3(256), 0, st, s->slots64.p, s->kids.p, ns, s->tri.p, Q, amb, na64, dcount, a2, W); break;
        default: hipLaunchKernelGGL(k_reeval64<2>, dim3(gr), dim3(256), 0, st, s->slots64.p, s->kids.p, ns, s->tri.p, Q, amb, na64, dcount, a2, W); break;
      }
      check_launch("k_reeval64");
    }
  }
}

}  // namespace gwn
