// Device layout of a built LBVH and the device-side geometry helpers shared by
// the builder and the traversal kernels.
//
// HBM layout (per BVH of n triangles):
//   nodes  [n-1] x 64 B  Karras internal node i: both child boxes + child refs
//                        (a ref with bit 31 set is a leaf = sorted position)
//   wide   [n-1] x 64 B  the traversal's own node of each even-level internal
//                        node (WNode; absent for the largest builds and for
//                        vertices that are not finite or beyond 2^40)
//   tris   [n]   x 48 B  triangle soup in Morton order: v0.xyz + original id,
//                        v1.xyz, v2.xyz (three 16-byte loads per test)
//   parity arrays (codes, order, split, ranges, parents, flags) kept for export
#pragma once
#include "common.hpp"

namespace flg {

struct alignas(16) BNode {
  float4 a;  // L.lo.x L.lo.y L.lo.z L.hi.x
  float4 b;  // L.hi.y L.hi.z R.lo.x R.lo.y
  float4 c;  // R.lo.z R.hi.x R.hi.y R.hi.z
  int4 d;    // refL refR - -
};
static_assert(sizeof(BNode) == 64, "node is 64 bytes");

struct alignas(16) BTri {
  float4 v0;  // w = original triangle id (bit pattern)
  float4 v1;
  float4 v2;
};
static_assert(sizeof(BTri) == 48, "triangle is 48 bytes");

constexpr uint32_t kLeafBit = 0x80000000u;

// The traversal's own node: up to four subtrees below a binary node, in the
// order in which the reference's depth-first traversal meets them.  An entry
// is either a binary node's subtree, with that node's box, or a leaf group,
// the one or two leaf children of one binary node, with that node's box (a
// leaf's test depends on its parent's box).  The boxes are kept as bytes on a
// grid of the node's own, rounded outwards: 64 bytes for four boxes, two
// levels of the tree, in four 16-byte loads.  A traversal of these boxes
// visits a superset of what the reference visits, in its order; traverse.hpp
// says why its hits are the reference's all the same.
struct alignas(16) WNode {
  float px, py, pz;     // the grid's origin
  uint32_t exps;        // its steps: byte k the exponent field of axis k's step, a power of two
  uint32_t lo[3];       // per axis: lower bounds of entries 0..3, a byte each, in steps
  uint32_t hi[3];       // upper bounds
  uint32_t unused[2];
  int4 ref;  // binary node index, or kLeafBit | kPairBit (two leaves) | sorted position; 0: no entry
};
static_assert(sizeof(WNode) == 64, "wide node is 64 bytes");
constexpr uint32_t kPairBit = 0x40000000u;  // positions are below 2^30

struct SharedBlock {
  void* ptr = nullptr;
  size_t bytes = 0;
  int refs = 0;
};

// The context's pool of LBVH output blocks (lbvh.hip): a destroyed BVH's
// block is kept for a later build; released with the context.
void bvh_pool_give(flg_ctx* ctx, void* p, size_t bytes);
void bvh_pool_release(flg_ctx* ctx);

}  // namespace flg

struct flg_bvh {
  flg_ctx* ctx = nullptr;
  int32_t n = 0;
  uint32_t flags = 0;
  float bound[6] = {0, 0, 0, 0, 0, 0};  // host copy of the global bound
  flg::BNode* nodes = nullptr;
  flg::WNode* wide = nullptr;         // wide node of each binary node, or null (binary traversal)
  flg::BTri* tris = nullptr;
  uint32_t* morton = nullptr;         // original order
  uint32_t* morton_sorted = nullptr;
  uint32_t* order = nullptr;          // sorted position -> original triangle
  int32_t* split = nullptr;
  int32_t* rlo = nullptr;
  int32_t* rhi = nullptr;
  int32_t* parent = nullptr;
  uint8_t* leafflags = nullptr;       // bit 0: left child is a leaf, bit 1: right
  int32_t* leaf_parent = nullptr;
  float* gbound = nullptr;            // device copy of the global bound (6 floats)
  uint64_t bytes = 0;
  flg::SharedBlock* block = nullptr;
};

namespace flg {

// Pluecker watertight ray/triangle test (src/experimental/intersector.hpp:
// msub :41-43, StableTriangleNormal :45-60, PlueckerTriangleIntersect :63-101,
// StableNormalize src/common/vector.h:495-504 in double).
FLG_HD float msub(float a, float b, float c) { return __builtin_fmaf(a, b, -c); }

FLG_HD V3 stable_triangle_normal(V3 a, V3 b, V3 c) {
  const float ab_x = a.z * b.y, ab_y = a.x * b.z, ab_z = a.y * b.x;
  const float bc_x = b.z * c.y, bc_y = b.x * c.z, bc_z = b.y * c.x;
  V3 cab = v3(msub(a.y, b.z, ab_x), msub(a.z, b.x, ab_y), msub(a.x, b.y, ab_z));
  V3 cbc = v3(msub(b.y, c.z, bc_x), msub(b.z, c.x, bc_y), msub(b.x, c.y, bc_z));
  const bool sx = fabsf(ab_x) < fabsf(bc_x);
  const bool sy = fabsf(ab_y) < fabsf(bc_y);
  const bool sz = fabsf(ab_z) < fabsf(bc_z);
  return v3(sx ? cab.x : cbc.x, sy ? cab.y : cbc.y, sz ? cab.z : cbc.z);
}

// On the device the three quotients float(x / sqrt(sq)) come from one
// reciprocal square root, refined to y = (1 + e) / sqrt(sq) with |e| below
// 2^-51 by one third-order step on the hardware's approximation.  The step
// leaves 2.5 d^3 of a relative error d, and its own rounding: that asks for d
// below 2^-17.5, and the instruction's is below 2^-24.1 (2^27 inputs over 256
// binades).  x y then differs from the correctly rounded x / sqrt(sq) by fewer
// than 8 units in the last place of a double, so it rounds to the same float
// unless its low 29 bits lie within 8 of the halfway point between two
// floats; those, results below the normal floats (where the halfway points lie
// elsewhere) and lengths outside [2^-300, 2^300] take the division itself.
// About 45 instructions instead of 110.
FLG_HD V3 stable_normalize(V3 v, bool compat) {
  double x = v.x, y = v.y, z = v.z;
  double sq = compat ? (x * x + y * y + z + z) : (x * x + y * y + z * z);
#if defined(__HIP_DEVICE_COMPILE__)
  if (sq >= 0x1p-300 && sq <= 0x1p300) {
    const double y0 = __builtin_amdgcn_rsq(sq);
    const double e = __builtin_fma(-(sq * y0), y0, 1.0);
    const double inv = __builtin_fma(y0 * e, __builtin_fma(e, 0.375, 0.5), y0);
    const double qx = x * inv, qy = y * inv, qz = z * inv;
    const V3 f = v3((float)qx, (float)qy, (float)qz);
    auto off = [](double q) {  // distance test of the low 29 bits from the halfway point
      return ((uint32_t)__builtin_bit_cast(uint64_t, q) & 0x1fffffffu) - (0x10000000u - 16u);
    };
    const uint32_t near = off(qx) < off(qy) ? off(qx) : off(qy);
    if (fminf(fminf(fabsf(f.x), fabsf(f.y)), fabsf(f.z)) >= 0x1p-125f && (near < off(qz) ? near : off(qz)) > 32u)
      return f;
  }
#endif
  double r = __builtin_sqrt(sq);
  return v3((float)(x / r), (float)(y / r), (float)(z / r));
}

// Edge test only: true if the ray passes the UVW sign test.
FLG_HD bool pluecker_uvw(V3 v0, V3 v1, V3 v2, V3 D) {
  const V3 e0 = v2 - v0, e1 = v0 - v1, e2 = v1 - v2;
  const float U = dot(cross(e0, v2 + v0), D);
  const float V = dot(cross(e1, v0 + v1), D);
  const float W = dot(cross(e2, v1 + v2), D);
  const float UVW = U + V + W;
  const float eps = 1.1920928955078125e-07f * fabsf(UVW);
  return smin(U, smin(V, W)) >= -eps || smax(U, smax(V, W)) <= eps;
}

// The part of the test after the edge test: returns true and t / Ng on a hit
// (t >= 0, den != 0).
FLG_HD bool pluecker_t(V3 a, V3 b, V3 c, V3 O, V3 D, bool compat, float* thit, V3* ng) {
  const V3 v0 = a - O, v1 = b - O, v2 = c - O;
  const V3 e0 = v2 - v0, e1 = v0 - v1, e2 = v1 - v2;
  const V3 Ng = stable_normalize(stable_triangle_normal(e0, e1, e2), compat);
  const float dd = dot(Ng, D);
  const float den = dd + dd;
  const float tt = dot(v0, Ng);
  const float T = tt + tt;
  const float t = T / den;
  if (!(0.0f <= t)) return false;
  if (!(den != 0.0f)) return false;
  *thit = t;
  *ng = Ng;
  return true;
}

// Full test (PlueckerTriangleIntersect): the edge test, then t and Ng.
FLG_HD bool pluecker(V3 a, V3 b, V3 c, V3 O, V3 D, bool compat, float* thit, V3* ng) {
  if (!pluecker_uvw(a - O, b - O, c - O, D)) return false;
  return pluecker_t(a, b, c, O, D, compat, thit, ng);
}

// OffsetRayOrigin (src/common/ray.h:64-93)
FLG_HD V3 offset_ray_origin(V3 p, V3 n, V3 dir) {
  const float origin = 1.0f / 32.0f, float_scale = 1.0f / 65536.0f, int_scale = 256.0f;
  V3 offset = n;
  if (dot(n, dir) <= 0) offset = -n;
  int oi0 = (int)(offset.x * int_scale), oi1 = (int)(offset.y * int_scale),
      oi2 = (int)(offset.z * int_scale);
  float px = u2f((uint32_t)((int32_t)f2u(p.x) + ((p.x < 0) ? -oi0 : oi0)));
  float py = u2f((uint32_t)((int32_t)f2u(p.y) + ((p.y < 0) ? -oi1 : oi1)));
  float pz = u2f((uint32_t)((int32_t)f2u(p.z) + ((p.z < 0) ? -oi2 : oi2)));
  return v3(fabsf(p.x) < origin ? p.x + float_scale * offset.x : px,
            fabsf(p.y) < origin ? p.y + float_scale * offset.y : py,
            fabsf(p.z) < origin ? p.z + float_scale * offset.z : pz);
}

// BoundIntersect (intersector.hpp:103-120) with a precomputed 1/d (the
// reference computes the same IEEE quotient per call).  The reference returns
// as soon as t0 > t1 after an axis; t0 only grows and t1 only shrinks from
// one axis to the next (each update keeps the old value unless the new one
// compares past it, NaN included), so one test after the three axes gives the
// same answer and the same t0, without a branch per axis.  t0 and t1 are never
// NaN, so `tn > t0 ? tn : t0` is fmaxf(t0, tn) (a NaN operand yields the
// other) up to the sign of a zero result, which no comparison sees; the swap
// keeps the reference's comparison, under which a NaN bound is not swapped.
FLG_HD bool slab(float lox, float loy, float loz, float hix, float hiy, float hiz, V3 o, V3 inv,
                 float* tnear) {
  float t0 = 0.0f, t1 = 3.402823466e+38f;
  float tn = (lox - o.x) * inv.x, tf = (hix - o.x) * inv.x;
  if (tn > tf) { float t = tn; tn = tf; tf = t; }
  t0 = fmaxf(t0, tn);
  t1 = fminf(t1, tf);
  tn = (loy - o.y) * inv.y;
  tf = (hiy - o.y) * inv.y;
  if (tn > tf) { float t = tn; tn = tf; tf = t; }
  t0 = fmaxf(t0, tn);
  t1 = fminf(t1, tf);
  tn = (loz - o.z) * inv.z;
  tf = (hiz - o.z) * inv.z;
  if (tn > tf) { float t = tn; tn = tf; tf = t; }
  t0 = fmaxf(t0, tn);
  t1 = fminf(t1, tf);
  *tnear = t0;
  return !(t0 > t1);
}

// ------------------------------------------------------------ wide nodes --
struct WEntry {
  float b[6];  // lo.xyz, hi.xyz
  int32_t ref;
};

// The entries that stand for binary node nd with box `own`: its leaf group,
// then its inner children.
FLG_HD int wide_contents(const BNode& nd, const float* own, WEntry& e0, WEntry& e1) {
  const int32_t l = nd.d.x, r = nd.d.y;
  const float bl[6] = {nd.a.x, nd.a.y, nd.a.z, nd.a.w, nd.b.x, nd.b.y};
  const float br[6] = {nd.b.z, nd.b.w, nd.c.x, nd.c.y, nd.c.z, nd.c.w};
  const bool leaf = (l | r) < 0;
  for (int k = 0; k < 6; ++k) {
    e0.b[k] = leaf ? own[k] : bl[k];
    e1.b[k] = r < 0 ? bl[k] : br[k];
  }
  e0.ref = leaf ? (l < 0 ? l : r) : l;
  if ((l & r) < 0) e0.ref |= (int32_t)kPairBit;
  e1.ref = r < 0 ? l : r;
  return (l & r) < 0 ? 1 : 2;
}

// The wide node of binary node i: its leaf group and the contents of its inner
// children (two binary levels), an inner entry whose node has two leaves being
// that leaf group.  Filling free slots with deeper nodes (the largest box
// first) measured 1.5% fewer visits, and would leave no simple rule for which
// binary nodes start a wide node.  get(k) is binary node k; a child that is not
// open(k) keeps its own entry.
template <class Get, class Open>
FLG_HD WNode wide_node(Get get, Open open, int32_t i) {
  WEntry e[4], top[2];
  const BNode nd = get(i);
  // the node's own box (the grid's extent): the union of its children's
  float own[6];
  {
    const float l[6] = {nd.a.x, nd.a.y, nd.a.z, nd.a.w, nd.b.x, nd.b.y};
    const float r[6] = {nd.b.z, nd.b.w, nd.c.x, nd.c.y, nd.c.z, nd.c.w};
    for (int k = 0; k < 3; ++k) {
      own[k] = fminf(l[k], r[k]);
      own[3 + k] = fmaxf(l[3 + k], r[3 + k]);
    }
  }
  const int nt = wide_contents(nd, own, top[0], top[1]);
  bool used[4];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    used[2 * h] = h < nt;
    used[2 * h + 1] = false;
    e[2 * h] = e[2 * h + 1] = top[h];
    if (h < nt && top[h].ref >= 0 && open(top[h].ref))
      used[2 * h + 1] = wide_contents(get(top[h].ref), top[h].b, e[2 * h], e[2 * h + 1]) == 2;
  }
  int32_t ref[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    ref[k] = used[k] ? e[k].ref : 0;
    if (ref[k] > 0) {
      const int4 d = get(ref[k]).d;
      if ((d.x & d.y) < 0) ref[k] = d.x | (int32_t)kPairBit;
    }
  }
  WNode w;
  w.px = own[0];
  w.py = own[1];
  w.pz = own[2];
  w.exps = 0;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    // the step: the power of two above extent / 254 (at least 2^-60), so that
    // the extent takes at most 254 of them
    uint32_t ex = (f2u((own[3 + c] - own[c]) * (1.0f / 254.0f)) >> 23) + 1u;
    ex = ex < 67u ? 67u : ex > 200u ? 200u : ex;
    w.exps |= ex << (8 * c);
    const float per = u2f((254u - ex) << 23);  // 1 / step
    uint32_t lo = 0, hi = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      // the difference is within 2^-24 of its value, a 2^-16 of a step, which
      // the traversal's margin covers; NaN bounds become the whole extent
      const float a = floorf((e[k].b[c] - own[c]) * per), b = ceilf((e[k].b[3 + c] - own[c]) * per);
      lo |= (uint32_t)fminf(fmaxf(a, 0.0f), 255.0f) << (8 * k);
      hi |= (uint32_t)fmaxf(fminf(b, 255.0f), 0.0f) << (8 * k);
    }
    w.lo[c] = lo;
    w.hi[c] = hi;
  }
  w.unused[0] = w.unused[1] = 0;
  w.ref = make_int4(ref[0], ref[1], ref[2], ref[3]);
  return w;
}

}  // namespace flg
