// NMH traversal on gfx950: the reference's intersect()/intersectAny()
// (src/kernels/lib/intersect.cuh:36-152) with identical results.
//
// The reference pops a state, tests the node's slab on the node's axis
// (Ray::intersect(slab), src/kernels/lib/ray.cuh:49-61), tests both triangles
// (one-sided Moller-Trumbore, ray.cuh:22-47, strict t < ray.t so the first
// hit wins ties), then pushes R and L (L popped first; L/R swapped when the
// ray direction on the children's axis is negative).  The same tests run here
// in the same order, with changes that do not alter any result:
//   * a node's children slabs are stored in the node record, so both
//     children are tested when their parent is visited; the t-dependent part
//     of the test (range.x <= ray.t) is still applied when a child is taken,
//     exactly when the reference would pop it;
//   * the near child is taken directly; only the far child is deferred;
//   * a deferred child is the sibling of the current path's node at its
//     depth, so the per-lane stack holds only its range (8 bytes, a
//     compact LIFO stack in depth order) plus one trail bit per depth; the
//     child's heap index is recomputed from the last visited node when it is
//     resumed;
//   * the slab quotient (s - p) / d uses the ray's correctly rounded
//     reciprocal y = RN(1/d) and one residual correction,
//         q0 = RN(n y),  e = n - d q0 (exact, FMA),  q = RN(q0 + e y),
//     which equals RN(n / d) (Markstein's theorem) while no step under- or
//     overflows: used only for 2^-60 <= |d| <= 16 and n = 0 or
//     2^-96 <= |n| <= 2^60, true division otherwise.  Inside the loop the
//     numerator range follows from a per-node flag (all four child slab
//     values pass normal_coord) and a per-ray check of the origin;
//   * a node's two triangles first take a reject test on the record's
//     reduced copy (trav_test), whose threshold bounds every rounding and
//     quantisation error: a triangle it rejects fails the reference's test.
//     The others (about one visit in 80 for meshes) take the reference's test on
//     their exact vertices (trav_exact), in order, before the traversal of
//     their ray goes on;
//   * 1/det is HIP's correctly rounded reciprocal sequence without its
//     scaling and fix-up steps, which are identities for 2^-24 <= det <= 2^64
//     (det < kEpsilon is rejected before the value is used; det > 2^64 takes
//     true division); the ray's reciprocals use the same sequence (needed
//     only for 2^-60 <= |d| <= 16).
//
// The traversal is a small state machine (trav_init, then trav_test,
// trav_exact while candidates remain and trav_next per node visit) so that persistent kernels can refill finished lanes.
#pragma once

#include "common.h"

namespace aur {

// Bitwise (not short-circuit) conditions keep these tests free of branches.
__device__ __forceinline__ bool fast_num(float n) {
  const float a = fabsf(n);
  return (n == 0.0f) | ((a >= 0x1p-96f) & (a <= 0x1p60f));
}

// RN(n / d) by the reciprocal quotient (valid when fast_num(n) and fast_d).
__device__ __forceinline__ float quot_fast(float n, float d, float y) {
  const float q = n * y;
  return __builtin_fmaf(__builtin_fmaf(-d, q, n), y, q);
}

// v_min_f32 / v_max_f32 on operands that are never signaling NaNs (every
// operand here is the result of arithmetic, or a copy of one): with IEEE mode
// on, these instructions return the other operand for a quiet NaN, exactly
// fminf / fmaxf.  The compiler cannot prove that through the join of the fast
// and exact quotient paths or the loop-carried range, and would quiet each
// operand first (one more instruction per operand).
__device__ __forceinline__ float min_q(float a, float b) {
  float r;
  __asm__("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float max_q(float a, float b) {
  float r;
  __asm__("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

__device__ __forceinline__ float2 clip(float2 r, float d0, float d1) {
  return make_float2(max_q(min_q(d0, d1), r.x), min_q(max_q(d0, d1), r.y));
}

__device__ __forceinline__ float2 narrow(float2 r, float slo, float shi, float p, float d, float y,
                                         bool fast_d) {
  const float n0 = slo - p, n1 = shi - p;
  float d0 = quot_fast(n0, d, y), d1 = quot_fast(n1, d, y);
  const bool f0 = fast_num(n0), f1 = fast_num(n1);
  if (!(fast_d & f0 & f1)) {
    d0 = n0 / d;
    d1 = n1 / d;
  }
  return clip(r, d0, d1);
}

// RN(1/x) for 2^-60 <= |x| <= 2^64: the steps of HIP's IEEE division 1/x
// (reciprocal estimate, one Newton step, quotient and two residual
// corrections) without the operand scaling and result fix-up, which do
// nothing on this range.
constexpr float kRecipMax = 0x1p64f;
__device__ __forceinline__ float recip_rn(float x) {
  const float r0 = __builtin_amdgcn_rcpf(x);
  const float r1 = __builtin_fmaf(__builtin_fmaf(-x, r0, 1.0f), r0, r0);
  const float q1 = __builtin_fmaf(__builtin_fmaf(-x, r1, 1.0f), r1, r1);
  return __builtin_fmaf(__builtin_fmaf(-x, q1, 1.0f), r1, q1);
}

// The reference's one-sided Moller-Trumbore test after its determinant:
// accept iff !(det < eps), u in [0,1], v >= 0 and u + v <= 1 (NaN passes
// these as in the reference and is rejected by the caller's t test).
__device__ __forceinline__ bool tri_finish(V3 o, V3 d, V3 v1, V3 e1, V3 e2, V3 P, float det,
                                           float invdet, float& u, float& v, float& t) {
  const V3 T = o - v1;
  u = dot(T, P) * invdet;
  const V3 Q = cross(T, e1);
  v = dot(d, Q) * invdet;
  t = dot(e2, Q) * invdet;
  return !(det < kEpsilon) & !(u < 0.0f) & !(u > 1.0f) & !(v < 0.0f) & !(u + v > 1.0f);
}

// Traversal counters of the reference's loop: popped = states popped with an
// in-range index (P), passed = states whose slab test passed (S).  Exact for
// closest-hit traversal, where every pushed state is eventually popped.
struct TraceCount {
  uint32_t popped = 0, passed = 0;
};

// Counters of the reject test: node visits, triangles it left to the exact
// test, and rejected triangles that the exact test accepts.
struct RejectCount {
  uint32_t visits = 0, exact = 0, missed = 0;
};

// Node indices are kept 1-based (K = k + 1: children 2K and 2K + 1, sibling
// K ^ 1, ancestor by shift) and depths one-hot (depth d: 1 << d), so that the
// axis and a pending entry's depth are bit tests.
struct Trav {
  V3 o, d, y;      // origin, direction, RN(1/direction)
  float rj_size, rj_far, rj;  // the reject test's threshold terms (trav_test)
  uint32_t fast;   // bit m: the children of a node at depth m take the reciprocal quotient
  float t, u, v;   // current closest hit (t = ray.t)
  int32_t id;
  uint32_t K, depth;  // node, one-hot depth
  uint32_t trail;  // depths with a pending entry
  uint32_t top;    // stack position (units of the stack)
  float2 r;        // range of the node after its slab test
  float4 slab;     // the node's children's slabs
  uint32_t flags;  // the node's scale_b
};
// Depths whose children's axis (depth + 1) % 3 is x, y, z.
constexpr uint32_t kChildX = 0x24924924u, kChildY = 0x49249249u, kChildZ = 0x92492492u;
constexpr uint32_t kExactShare = 12u;  // exact tests run once candidates wait in a twelfth of the active lanes

// Per-lane stack of deferred ranges.  A deferred child is always deeper
// than every entry already pending (entries sit on the current path's
// siblings and are popped deepest first), so the entries form a LIFO stack
// sorted by depth and entry i is at index i = popcount(trail) at push time:
// at most levels - 1 entries, indices <= levels - 2.
//
// LdsStack: every row in LDS (lane-strided, conflict-free); the state's top
// is the number of entries in 8-byte units of the row stride.
struct LdsStack {
  float2* lds;  // row r of this lane at lds[r * stride]
  uint32_t stride;
  __device__ __forceinline__ void push(uint32_t& top, float2 v) const {
    lds[top] = v;
    top += stride;
  }
  __device__ __forceinline__ float2 pop(uint32_t& top) const {
    top -= stride;
    return lds[top];
  }
};

// SplitStack: rows [0, klds) in LDS, deeper rows in a per-lane column of
// global memory, so that a small LDS window leaves room for more resident
// waves.  The LDS side uses an LDS-qualified pointer and the global side
// stores through a global pointer and loads through a buffer resource, so
// the two stay separate instructions (merged, they would become generic
// "flat" accesses, slower for the common LDS case).
typedef float vf2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) vf2 lds_vf2;
typedef __attribute__((address_space(1))) vf2 glb_vf2;
struct SplitStack {
  lds_vf2* lds;            // row r < klds at lds[r * lstride]
  uint32_t lstride;
  glb_vf2* glb;            // row r >= klds at glb[(r - klds) * gstride]
  __amdgpu_buffer_rsrc_t rsrc;  // the whole global stack buffer
  uint32_t lane_bytes;     // byte offset of glb from the buffer start
  uint32_t gstride;
  uint32_t klds;
  __device__ __forceinline__ void push(uint32_t& top, float2 v) const {
    const vf2 w = {v.x, v.y};
    const uint32_t r = top++;
    if (r < klds)
      lds[r * lstride] = w;
    else
      glb[(size_t)(r - klds) * gstride] = w;
  }
  __device__ __forceinline__ float2 pop(uint32_t& top) const {
    const uint32_t r = --top;
    if (r < klds) {
      const vf2 w = lds[r * lstride];
      return make_float2(w.x, w.y);
    }
    const auto w = __builtin_amdgcn_raw_buffer_load_b64(rsrc, lane_bytes + (r - klds) * gstride * 8u,
                                                        0, 0);
    return make_float2(__uint_as_float(w[0]), __uint_as_float(w[1]));
  }
};

__device__ __forceinline__ LdsStack lds_stack(float2* lane_column, uint32_t stride) {
  return LdsStack{lane_column, stride};
}

// The reciprocal quotient's range.  (An origin below 2^57 keeps the slabs of
// missing children, kNoSlab, beyond any range.)
__device__ __forceinline__ bool fast_axis(float o, float d) {
  const float a = fabsf(d);
  const bool normal = normal_coord(o);
  return (a >= 0x1p-60f) & (a <= 16.0f) & normal & (fabsf(o) <= 0x1p57f);
}

// The root's own slab (record 0 of a tree).
struct RootInfo {
  float lo, hi;
};

// The tree a lane traverses: node records, the triangles' vertices in tree
// order and the node count.
struct TreeRef {
  const NodeRec* nodes;
  const float* tris;
  uint32_t n_nodes;
  RootInfo root;
};

__device__ __forceinline__ RootInfo root_info(const NodeRec* __restrict__ nodes) {
  return RootInfo{nodes[0].cslab[0], nodes[0].cslab[1]};
}

// The reject test's threshold (trav_test).
constexpr float kRejA = 1.6e-3f;                            // times 2 |C|max
constexpr float kRejSize = 2.0f * 3.4f * kRejA;             // 2 thr's terms times D: z,
constexpr float kRejB = 2.0f * 8.125f * 0x1p-12f;           // constant,
constexpr float kRejFar = 48.0f * 0x1p-24f;                 // and D times 2 sigma t

// Sets up a ray; returns false when the root's slab culls it (finished, miss).
// The reciprocals y serve only axes with 2^-60 <= |d| <= 16, where recip_rn
// equals 1.0f / d.
template <bool kCount>
__device__ __forceinline__ bool trav_init_root(Trav& s, RootInfo root, V3 o, V3 d, float tmax,
                                               TraceCount* cnt) {
  s.o = o;
  s.d = d;
  s.y = mk(recip_rn(d.x), recip_rn(d.y), recip_rn(d.z));
  // keep the reciprocals in registers: without this barrier the compiler
  // re-derives them at every use inside the loop
  __asm__ volatile("" : "+v"(s.y.x), "+v"(s.y.y), "+v"(s.y.z));
  const bool fx = fast_axis(o.x, d.x), fy = fast_axis(o.y, d.y), fz = fast_axis(o.z, d.z);
  s.fast = (fx ? kChildX : 0u) | (fy ? kChildY : 0u) | (fz ? kChildZ : 0u);
  {
    // terms of the reject test's threshold, or NaN (no triangle is rejected)
    // for rays outside its bound's range
    const float dm = fmaxf(fmaxf(fabsf(d.x), fabsf(d.y)), fabsf(d.z));
    const float om = fmaxf(fmaxf(fabsf(o.x), fabsf(o.y)), fabsf(o.z));
    const float all = ((d.x + d.y) + d.z) + ((o.x + o.y) + o.z);  // NaN if any is
    const bool in = (dm >= kRejectDirMin) & (dm <= kRejectDirMax) & (om <= kRejectCoord) & (all == all);
    s.rj = in ? dm * kRejB : __builtin_nanf("");
    s.rj_size = dm * kRejSize;
    s.rj_far = dm * dm * kRejFar;
  }
  s.t = tmax;
  s.u = s.v = 0.0f;
  s.id = -1;
  s.K = s.depth = 1;
  s.trail = s.top = 0;
  if (kCount) cnt->popped += 1;  // the root
  s.r = narrow(make_float2(kEpsilon, kInfinity), root.lo, root.hi, o.x, d.x, s.y.x, fx);
  return (s.r.x <= s.r.y) && (s.r.x <= s.t);
}

template <bool kCount>
__device__ __forceinline__ bool trav_init(Trav& s, const TreeRef& tree, V3 o, V3 d, float tmax,
                                          TraceCount* cnt) {
  return trav_init_root<kCount>(s, root_info(tree.nodes), o, d, tmax, cnt);
}

// ---- the reject test ----
//
// Loads the node's record and says which of its triangles may
// pass the reference's test.  VALU issue bounds a visit, and the vector L1
// comes next: a load of 64 lanes that read 64 nodes is 64 lookups.  Both
// triangles' exact test took 125 VALU instructions and a 96-byte record 6
// loads; this test takes 67 and the 64-byte record 4, and what it leaves over
// (1.2% of the visits at 1M triangles) costs 6 more per visit.  2^24 incoherent
// rays into 1M triangles take 4.6 ms (7.3 with the exact tests in every visit):
// 2.38e9 VALU instructions at 0.88 of the issue rate, 2.98e9 L1 lookups at 1.10
// per cycle and CU (lanes that read random 64-byte records of a buffer that the
// L1 holds reach 1.48).  More resident waves than 16 per CU are slower: the
// lines of their visits no longer fit the 32 KB L1 between a record's four
// loads.
//
// With T = p - v1 for any point p of the ray's line and C = T x d, the
// Moller-Trumbore numerators are u det = e2 . C, v det = -(e1 . C) and
// det = -d . (e1 x e2); the reference's test accepts only if none of the
// three edge functions u det, v det and (1 - u - v) det is negative (but for
// rounding).  p = o + t d is the ray's entry into the node's range, so that T
// is no larger than the node's group, and lengths are in units of the group's
// size.  T is computed as (o - v1) + t d, whose rounding does not grow with the
// coordinates: with p computed first and a threshold for the largest coordinate
// of the tree, 2^22 incoherent rays into 1M triangles in a box of 100 over a
// ground plane 2e6 wide took 2.95 ms, 1.56 now (1.40 without the plane; 2.10 with
// the exact tests in every visit), 2e5 wide 2.20 ms, 1.55 now.
//
// Bound.  D = the largest |direction component|, z = the triangle's size (each
// |e| component <= z), q = 2^-11 + 2^-15, t = the range's entry; sigma = 2^-k,
// half of the record's scale (T, and so C and the numerators, come out doubled).
//   edges: rounding to half moves a component by at most q z (2^-11 relative,
//     2^-25 absolute, z >= 2^-10);
//   T: off by at most 2^-12 (dv, |dv| <= 1) + 2^-15 (roundings of dv and T,
//     |T| <= 4) + 2^-24 sigma |o - v1|max (one fma for o - v1; the scale is a
//     power of two); C by 2 D times that and 2^-22 D;
//   u det, v det: z (3 q |C|max + D (6.82 2^-12 + 6 2^-24 sigma |o - v1|max));
//   det: e1 x e2 in half, 3 D ((4.01 q + 3 2^-11) z^2 + 2^-24);
//   the reference's floats: 36 2^-24 z D sigma |o - v1|max per numerator
//     (T, P or Q and the dot product).
// With |T| <= 4 (5 for the second triangle), sigma |o - v1|max <= sigma t D + 5,
// so the terms in sigma are at most 42 2^-24 z D (sigma t D + 5): only a ray
// that comes from some 10^5 sizes of the group away loses the test's use.  A
// triangle that the reference accepts has, with
//   thr = A |C|max + 3.4 A z D + D (B + 48 2^-24 sigma t D),
// u det >= -z thr, v det >= -z thr and (1 - u - v) det >= -2 z thr:
// A = 1.6e-3 >= 3 q = 1.557e-3; half the third function's error is that of
// one numerator plus z D 5.32e-3 z, below 3.4 A z = 5.44e-3 z, plus 0.38 2^-12
// z D, and B = 8.125 2^-12 >= (6.82 + 0.38 + 0.06) 2^-12 + 2^-15 with a margin for
// the float roundings of this test itself (below 2^-18 z D).  Nothing here over-
// or underflows for D in 2^-40 .. 2^40 and coordinates up to 2^40, nor does
// the reference's test of a triangle that it accepts.
// Comparisons are written so that NaN and infinity keep a triangle.
__device__ __forceinline__ float lo16(half2v h) { return (float)h.x; }
__device__ __forceinline__ float hi16(half2v h) { return (float)h.y; }
__device__ __forceinline__ float max3abs(float a, float b, float c) {
  return fmaxf(fmaxf(fabsf(a), fabsf(b)), fabsf(c));
}

// a - b with b the low or high half of h (one instruction; the compiler would
// convert first).
__device__ __forceinline__ float sub_lo16(float a, half2v h) {
  float r;
  __asm__("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(a));
  return r;
}
__device__ __forceinline__ float sub_hi16(float a, half2v h) {
  float r;
  __asm__("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(a));
  return r;
}

// Whether the triangle may be accepted: T doubled, edges e1 and e2, size and
// det in the record's units; base = 2 D (B + 48 2^-24 sigma t D).
__device__ __forceinline__ bool may_hit(V3 T, V3 d, V3 e1, V3 e2, float det, float size, float rj_size, float base) {
  const float cx = __builtin_fmaf(T.y, d.z, -(T.z * d.y));
  const float cy = __builtin_fmaf(T.z, d.x, -(T.x * d.z));
  const float cz = __builtin_fmaf(T.x, d.y, -(T.y * d.x));
  const float un = __builtin_fmaf(e2.z, cz, __builtin_fmaf(e2.y, cy, __builtin_fmaf(e2.x, cx, 0.0f)));
  const float vn = __builtin_fmaf(-e1.z, cz, __builtin_fmaf(-e1.y, cy, __builtin_fmaf(-e1.x, cx, 0.0f)));
  const float wn = __builtin_fmaf(-0.5f, un + vn, det);
  const float m = fminf(fminf(un, vn), wn);
  const float thr = __builtin_fmaf(max3abs(cx, cy, cz), kRejA, __builtin_fmaf(size, rj_size, base));
  return !(__builtin_fmaf(size, thr, m) < 0.0f);
}

// kWide: the record's address takes 64-bit arithmetic per lane (trees of 2^26
// nodes and more, and lanes with trees of their own); else it is a 32-bit
// offset from a wave-uniform base.
template <bool kCount, bool kWide>
__device__ __forceinline__ void trav_test(Trav& s, const TreeRef& tree, TraceCount* cnt, bool& may_a, bool& may_b) {
  if (kCount) {
    cnt->passed += 1;
    cnt->popped += (2 * s.K <= tree.n_nodes) + (2 * s.K + 1 <= tree.n_nodes);
  }
  const size_t offset = kWide ? (size_t)s.K * sizeof(NodeRec) : (size_t)(s.K * (uint32_t)sizeof(NodeRec));
  const uint4* rec = reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(tree.nodes) + offset);
  const uint4 a1 = rec[1], a2 = rec[2], a3 = rec[3], a0 = rec[0];
  s.slab = make_float4(__uint_as_float(a0.x), __uint_as_float(a0.y), __uint_as_float(a0.z), __uint_as_float(a0.w));
  s.flags = a1.w;
  const auto h2 = [](uint32_t x) { return __builtin_bit_cast(half2v, x); };
  const half2v e1x = h2(a2.x), e1y = h2(a2.y), e1z = h2(a2.z), e2x = h2(a2.w), e2y = h2(a3.x), e2z = h2(a3.y);
  const half2v dxy = h2(a3.z), dza = h2(a3.w), szb = h2(a1.w);
  const float scale = __uint_as_float(a1.w & 0x7F800000u);
  const V3 d = s.d;
  const float ts = s.r.x * scale;
  const V3 Ta = mk(__builtin_fmaf(ts, d.x, __builtin_fmaf(s.o.x, scale, -__uint_as_float(a1.x))),
                   __builtin_fmaf(ts, d.y, __builtin_fmaf(s.o.y, scale, -__uint_as_float(a1.y))),
                   __builtin_fmaf(ts, d.z, __builtin_fmaf(s.o.z, scale, -__uint_as_float(a1.z))));
  const V3 Tb = mk(sub_lo16(Ta.x, dxy), sub_hi16(Ta.y, dxy), sub_lo16(Ta.z, dza));
  const float base = __builtin_fmaf(ts, s.rj_far, s.rj);
  // e1 x e2 of both triangles at once
  const half2v nx = __builtin_elementwise_fma(e1y, e2z, -(e1z * e2y));
  const half2v ny = __builtin_elementwise_fma(e1z, e2x, -(e1x * e2z));
  const half2v nz = __builtin_elementwise_fma(e1x, e2y, -(e1y * e2x));
  const float deta = __builtin_fmaf(-lo16(nz), d.z, __builtin_fmaf(-lo16(ny), d.y, __builtin_fmaf(-lo16(nx), d.x, 0.0f)));
  const float detb = __builtin_fmaf(-hi16(nz), d.z, __builtin_fmaf(-hi16(ny), d.y, __builtin_fmaf(-hi16(nx), d.x, 0.0f)));
  const bool far = !(max3abs(Ta.x, Ta.y, Ta.z) <= 8.0f);
  may_a = far | may_hit(Ta, d, mk(lo16(e1x), lo16(e1y), lo16(e1z)), mk(lo16(e2x), lo16(e2y), lo16(e2z)), deta,
                        hi16(dza), s.rj_size, base);
  may_b = far | may_hit(Tb, d, mk(hi16(e1x), hi16(e1y), hi16(e1z)), mk(hi16(e2x), hi16(e2y), hi16(e2z)), detb,
                        lo16(szb), s.rj_size, base);
  // every load has returned here: with the slabs' still in flight on some
  // path, the next visit's address, in one of their registers, waited for all
  // outstanding memory operations, stores included
  __asm__ volatile("" : "+v"(s.slab.x), "+v"(s.slab.y), "+v"(s.slab.z), "+v"(s.slab.w));
}

// The slabs and flags alone, for visits that test both triangles exactly.
__device__ __forceinline__ void trav_slabs(Trav& s, const TreeRef& tree) {
  const uint4* rec = reinterpret_cast<const uint4*>(tree.nodes + s.K);
  const uint4 a0 = rec[0];
  s.flags = rec[1].w;
  s.slab = make_float4(__uint_as_float(a0.x), __uint_as_float(a0.y), __uint_as_float(a0.z), __uint_as_float(a0.w));
}

// The reference's test (Ray::intersect, src/kernels/lib/ray.cuh:22-47) of a
// triangle on the vertices it was uploaded with, for any t above kEpsilon.
__device__ __forceinline__ bool tri_accept(const Trav& s, const float* __restrict__ tris, uint32_t tri, float& u,
                                           float& v, float& t) {
  const float* p = tris + (size_t)tri * 9;  // points layout: x1 x2 x3 y1 y2 y3 z1 z2 z3
  const V3 v1 = mk(p[0], p[3], p[6]);
  const V3 e1 = mk(p[1], p[4], p[7]) - v1, e2 = mk(p[2], p[5], p[8]) - v1;
  const V3 P = cross(s.d, e2);
  const float det = dot(e1, P);
  float inv = recip_rn(det);
  if (det > kRecipMax) inv = 1.0f / det;
  return tri_finish(s.o, s.d, v1, e1, e2, P, det, inv, u, v, t) & (t > kEpsilon);
}

// The same of the node's first or second triangle; returns whether it became
// the closest hit.
__device__ __forceinline__ bool trav_exact(Trav& s, const float* __restrict__ tris, bool first) {
  const uint32_t tri = 2 * s.K - (first ? 2u : 1u);
  float u, v, t;
  const bool hit = tri_accept(s, tris, tri, u, v, t) & (t < s.t);
  if (hit) {
    s.t = t;
    s.u = u;
    s.v = v;
    s.id = (int32_t)tri;
  }
  return hit;
}

// Leaves the node (both triangles done) for the next one; returns true when
// the traversal has finished.  The near child is taken directly, the far one
// deferred; without a child to take, one pending entry is popped, and if its
// range now starts beyond the closest hit (again = true) the lane pops again,
// with popping set, in the next step (1.8% of the steps at 1M triangles; an inner loop until an
// entry passes made every lane of the wave wait through its iterations).
template <class Stk>
__device__ __forceinline__ bool trav_next(Trav& s, uint32_t n_nodes, const Stk& stk, bool popping, bool& again) {
  const bool ax = (s.depth & kChildX) != 0u, ay = (s.depth & kChildY) != 0u;
  // by value: a select of members would keep the state in memory
  const auto pick = [](bool c, float a, float b) { return c ? a : b; };
  const float oc = pick(ax, s.o.x, pick(ay, s.o.y, s.o.z));
  const float dc = pick(ax, s.d.x, pick(ay, s.d.y, s.d.z));
  const float yc = pick(ax, s.y.x, pick(ay, s.y.y, s.y.z));
  // the near child and each child's entry plane by the direction's sign: the
  // quotients of a slab's planes are ordered as the planes are (rounded
  // division is monotonic), so fminf / fmaxf of them are selections
  const bool sw = dc < 0.0f;
  const float n0 = pick(sw, s.slab.w, s.slab.x) - oc, n1 = pick(sw, s.slab.z, s.slab.y) - oc;
  const float n2 = pick(sw, s.slab.y, s.slab.z) - oc, n3 = pick(sw, s.slab.x, s.slab.w) - oc;
  float nx = quot_fast(n0, dc, yc), ny = quot_fast(n1, dc, yc);
  float fx = quot_fast(n2, dc, yc), fy = quot_fast(n3, dc, yc);
  if (((s.fast & s.depth) == 0u) | ((int32_t)s.flags < 0)) {
    // true division, with the reference's fminf / fmaxf (NaN, division by 0)
    const float a = n0 / dc, b = n1 / dc, c = n2 / dc, e = n3 / dc;
    nx = min_q(a, b);
    ny = max_q(a, b);
    fx = min_q(c, e);
    fy = max_q(c, e);
    const bool left = 2 * s.K <= n_nodes, right = 2 * s.K < n_nodes;  // which children exist
    if (!(sw ? right : left)) nx = __builtin_inff();
    if (!(sw ? left : right)) fx = __builtin_inff();
  }
  nx = max_q(nx, s.r.x);
  ny = min_q(ny, s.r.y);
  fx = max_q(fx, s.r.x);
  fy = min_q(fy, s.r.y);
  const bool far = !popping & (fx <= fy);
  const bool take_near = !popping & (nx <= ny) & (nx <= s.t);
  const bool take_far = !take_near & far & (fx <= s.t);
  if (take_near & far) {
    stk.push(s.top, make_float2(fx, fy));
    s.trail |= s.depth << 1;
  }
  if (take_near | take_far) {
    s.K = 2 * s.K + (uint32_t)(sw ^ take_far);
    s.depth <<= 1;
    s.r = make_float2(take_near ? nx : fx, take_near ? ny : fy);
    return false;
  }
  if (s.trail == 0u) return true;
  const float2 e = stk.pop(s.top);
  const uint32_t z = (uint32_t)__builtin_clz(s.trail);
  const uint32_t bit = 0x80000000u >> z;
  s.trail ^= bit;
  // the entry is the sibling of the path's node at its depth
  s.K = (s.K >> (z - (uint32_t)__builtin_clz(s.depth))) ^ 1u;
  s.depth = bit;
  s.r = e;
  again = !(e.x <= s.t);
  return false;
}

// Lane mask of a condition, without materialising it as an integer.
__device__ __forceinline__ uint64_t ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }

// A persistent wave's lanes as masks, so that their states live in scalar
// registers and branch conditions cost no vector instructions.
struct WaveState {
  uint64_t active = 0;        // lanes with a ray
  uint64_t may_a = 0, may_b = 0;  // ... whose node's first, second triangle is still to be tested exactly
  uint64_t popping = 0;       // ... that take the next pending entry
  uint64_t any = 0;           // lanes with an any-hit query (mixed launches)
};
__device__ __forceinline__ bool in(uint64_t mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); }

// One step of a persistent wave; returns the lanes whose traversal has
// finished.  Lanes whose node left candidates wait until they are a twelfth of
// the active lanes (or all of them): the exact test costs about a visit's
// instructions for however few lanes run it (a fifth was 3% slower on the
// 1080p frame, an eighth 1%).
template <bool kAny, bool kMixed, bool kWide, class Stk>
__device__ __forceinline__ uint64_t trav_visit(Trav& s, WaveState& w, const TreeRef& tree, const Stk& stk) {
  bool a = false, b = false;
  if (in(w.active & ~(w.may_a | w.may_b | w.popping))) trav_test<false, kWide>(s, tree, nullptr, a, b);
  w.may_a |= ballot(a);
  w.may_b |= ballot(b);
  const uint64_t pending = w.may_a | w.may_b;
  uint64_t finished = 0;
  if (pending != 0 && (uint32_t)__popcll(pending) * kExactShare >= (uint32_t)__popcll(w.active)) {
    bool hit = false;
    if (in(pending)) hit = trav_exact(s, tree.tris, in(w.may_a));
    w.may_b &= w.may_a;  // lanes that tested their first triangle
    w.may_a = 0;
    if (kAny || kMixed) {
      finished = ballot(hit) & (kAny ? ~0ull : w.any);
      w.may_b &= ~finished;
      w.active &= ~finished;
    }
  }
  const uint64_t go = w.active & ~(w.may_a | w.may_b);
  bool end = false, again = false;
  if (in(go)) end = trav_next(s, tree.n_nodes, stk, in(w.popping), again);
  w.popping = (w.popping & ~go) | ballot(again);
  const uint64_t ended = ballot(end);
  w.active &= ~ended;
  return finished | ended;
}

// The items a wave of a persistent launch takes from [0, n): first a range of
// its own, then chunks from a counter, so that waves whose rays end early take
// over the work of others.  With one fixed range per wave, a launch lasted as
// long as its dearest range: 2^21 camera rays, whose ranges see sky or
// geometry, took 1.00 ms alone, now 0.62 ms; a 256^2 Cornell frame 2.35 ->
// 2.17 ms; the differentiable step at 512^2 25.1 -> 20.1 ms.  The first range
// is one ray per lane below 512 rays a wave and half of an even share above; a
// chunk is a sixteenth of a share, at least one ray per lane (first ranges of
// 128 and 192 rays, chunks of 128 and first ranges of 3/4 of a share were up
// to 25% slower on the camera rays).  Launches of at most one first range per
// wave use no counter.  The blocks form kWorkGroups groups, each with a
// counter of its own in its own cache line (group g's t-th chunk is chunk
// t * groups + g): one address takes an atomic about every 12 ns, which
// bounded launches of short rays (the Cornell frame took 2.68 ms with a
// single counter).  (Asking for the next ticket ahead and letting a request
// reach over the end of a chunk was 10% slower on the camera rays.)
constexpr uint32_t kWorkGroups = 8;
constexpr uint32_t kWorkStride = 32;  // words between groups' counters
struct WaveWork {
  uint64_t next, end;  // the current range
  uint64_t n, first_total;
  uint32_t chunk, group, groups;
  uint32_t* ticket;  // the group's, zero before the launch
  bool more;         // the counter may have chunks left

  __device__ __forceinline__ WaveWork(uint64_t items, uint32_t* tickets) : n(items) {
    const uint32_t waves = (gridDim.x * blockDim.x) >> 6;
    const uint32_t wave = __builtin_amdgcn_readfirstlane((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    const uint64_t share = n >> 32 ? n / waves : (uint64_t)((uint32_t)n / waves);
    const uint64_t first = share < 512 ? 64 : (share / 2) & ~63ull;
    const uint64_t sixteenth = (share / 16 + 63) & ~63ull;
    chunk = sixteenth < 64 ? 64u : (sixteenth > (1u << 20) ? 1u << 20 : (uint32_t)sixteenth);
    groups = gridDim.x < kWorkGroups ? gridDim.x : kWorkGroups;
    group = blockIdx.x % kWorkGroups;
    ticket = tickets + group * kWorkStride;
    first_total = first * waves;
    more = first_total < n;
    next = first * wave;
    end = next + first < n ? next + first : n;
  }
  // The next chunk, when the range is used up; wave-uniform.
  __device__ __forceinline__ void refill() {
    if (next < end || !more) return;
    uint32_t t = 0;
    if ((threadIdx.x & 63u) == 0) t = atomicAdd(ticket, 1u);
    t = __builtin_amdgcn_readfirstlane(t);
    next = first_total + ((uint64_t)t * groups + group) * chunk;
    end = next + chunk < n ? next + chunk : n;
    more = next < n;
  }
};

// Persistent-wave traversal of a work range [0, n) of closest-hit and any-hit
// queries: between node visits, once at least `refill` lanes are idle (or all
// are), idle lanes take the next items of the wave's work, ranked by ballot.
// fetch(i, o, d, tmax, tree, any) loads item i, may replace the lane's tree
// (initially tree0; batches of scenes) and, with kMixed, sets any for an
// any-hit query; store(i, s) receives the finished
// state.  A fetch that never
// writes `tree` keeps the tree wave-uniform.  (Splitting a refill over two
// iterations, so that the item loads overlap the active lanes' node step,
// measured slower: the new lanes lose a step.)
template <bool kAny, bool kMixed, bool kWide, class Stk, class Fetch, class Store>
__device__ __forceinline__ void persistent_trace(TreeRef tree0, uint64_t n, uint32_t* ticket, uint32_t refill,
                                                 const Stk& stk, Fetch fetch, Store store) {
  TreeRef tree = tree0;
  WaveWork work(n, ticket);
  const uint32_t lane = threadIdx.x & 63u;
  const uint64_t lt = lane ? (~0ull >> (64 - lane)) : 0ull;
  Trav s;
  WaveState w;
  uint64_t done = 0;  // lanes whose result of `item` is not stored yet
  uint64_t item = 0;
  for (;;) {
    const uint64_t idle = ~w.active;
    const uint32_t nidle = __popcll(idle);
    if (nidle >= refill || nidle == 64) {
      // finished lanes' results together: loads and stores complete in order,
      // so a store per finished ray would hold up the next visit's loads
      if (in(done)) store(item, s);
      done = 0;
      work.refill();
      if (work.next < work.end) {
        bool enter = false, miss = false, any = false;
        if (in(idle)) {
          const uint64_t i = work.next + __popcll(idle & lt);
          if (i < work.end) {
            V3 o, d;
            float tmax;
            fetch(i, o, d, tmax, tree, any);
            item = i;
            enter = trav_init_root<false>(s, tree.root, o, d, tmax, nullptr);
            miss = !enter;
          }
        }
        w.active |= ballot(enter);
        if (kMixed) w.any = (w.any & ~idle) | ballot(any);
        done = ballot(miss);
        work.next += nidle;
      } else if (nidle == 64) {
        break;
      }
    }
    done |= trav_visit<kAny, kMixed, kWide>(s, w, tree, stk);
  }
}

// Whole traversal of one ray by one lane.
// stk: this lane's stack column, stk[depth * stride].
template <bool kAny, bool kCount = false, bool kCheck = false, bool kReject = true>
__device__ __forceinline__ void trace_ray(Trav& s, const TreeRef& tree, V3 o, V3 d, float tmax, float2* stk,
                                          uint32_t stride, TraceCount* cnt = nullptr, RejectCount* rej = nullptr) {
  const LdsStack st = lds_stack(stk, stride);
  if (!trav_init<kCount>(s, tree, o, d, tmax, cnt)) return;
  bool popping = false;
  for (;;) {
    if (!popping) {
      bool a = true, b = true;
      if (kReject)
        trav_test<kCount, true>(s, tree, cnt, a, b);
      else
        trav_slabs(s, tree);
      if (kCheck) {
        float u, v, t;
        const bool hit_a = tri_accept(s, tree.tris, 2 * s.K - 2, u, v, t);
        const bool hit_b = tri_accept(s, tree.tris, 2 * s.K - 1, u, v, t);
        rej->visits += 1;
        rej->exact += (uint32_t)a + (uint32_t)b;
        rej->missed += (uint32_t)(!a & hit_a) + (uint32_t)(!b & hit_b);
      }
      if (a && trav_exact(s, tree.tris, true) && kAny) return;
      if (b && trav_exact(s, tree.tris, false) && kAny) return;
    }
    bool again = false;
    if (trav_next(s, tree.n_nodes, st, popping, again)) return;
    popping = again;
  }
}

}  // namespace aur
