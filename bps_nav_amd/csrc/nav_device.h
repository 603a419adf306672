// Device-side navmesh queries on PolyRec records: the geometry primitives and the
// per-lane queries (nearest polygon, move along surface, height) of the step path.
// Compile with -ffp-contract=off: polygon ids must equal the reference's bit for bit, so
// every expression keeps Detour's fp32 operation order and is never fused.
//
// Reference semantics followed (read, not copied):
//   DetourCommon.cpp:170-184 (point-segment distance), :204-233 (height on triangle),
//   :238-270 (point in polygon, edge distances), :332-369 (random point in polygon);
//   DetourNavMesh.cpp:619-758 (height mesh queries); DetourNavMeshQuery.cpp:538-586
//   (boundary clamp), :642-826 (nearest polygon over the BV tree), :2016-2255 (move along
//   surface); PathFinder.cpp:24-44, 543-584 (snapPoint / tryStep conventions).
#pragma once
#include <hip/hip_runtime.h>

#include "device_types.h"

namespace bpsx {

#define BPSX_DEV __device__ __forceinline__

struct NavPt {
  float x, y, z;
  uint32_t ref;
};

BPSX_DEV bool finite3(float x, float y, float z) { return isfinite(x) && isfinite(y) && isfinite(z); }

BPSX_DEV float dist_pt_seg_sqr2d(float px, float pz, const float* p, const float* q, float& t) {
  const float pqx = q[0] - p[0], pqz = q[2] - p[2];
  float dx = px - p[0], dz = pz - p[2];
  const float d = pqx * pqx + pqz * pqz;
  t = pqx * dx + pqz * dz;
  if (d > 0) t /= d;
  if (t < 0) t = 0;
  else if (t > 1) t = 1;
  dx = p[0] + t * pqx - px;
  dz = p[2] + t * pqz - pz;
  return dx * dx + dz * dz;
}

BPSX_DEV bool point_in_poly(float px, float pz, const PolyRec& r) {
  bool c = false;
  const int nv = r.nv;
  for (int i = 0, j = nv - 1; i < nv; j = i++) {
    const float* vi = r.v[i];
    const float* vj = r.v[j];
    if (((vi[2] > pz) != (vj[2] > pz)) && (px < (vj[0] - vi[0]) * (pz - vi[2]) / (vj[2] - vi[2]) + vi[0])) c = !c;
  }
  return c;
}

BPSX_DEV bool height_on_triangle(float px, float pz, const float* a, const float* b, const float* c, float& h) {
  const float EPS = 1e-6f;
  const float v0x = c[0] - a[0], v0y = c[1] - a[1], v0z = c[2] - a[2];
  const float v1x = b[0] - a[0], v1y = b[1] - a[1], v1z = b[2] - a[2];
  const float v2x = px - a[0], v2z = pz - a[2];
  float denom = v0x * v1z - v0z * v1x;
  if (fabsf(denom) < EPS) return false;
  float u = v1z * v2x - v1x * v2z;
  float v = v0x * v2z - v0z * v2x;
  if (denom < 0) { denom = -denom; u = -u; v = -v; }
  if (u >= 0.0f && v >= 0.0f && (u + v) <= denom) {
    h = a[1] + (v0y * u + v1y * v) / denom;
    return true;
  }
  return false;
}

BPSX_DEV const float* detail_vert(const NavData& nav, const PolyRec& r, int k) {
  return k < r.nv ? r.v[k] : &nav.dverts[(size_t)(r.dvert_base + (uint32_t)(k - r.nv)) * 3];
}

template <bool kOnlyBoundary>
BPSX_DEV void closest_on_detail_edges(const NavData& nav, const PolyRec& r, float px, float py, float pz, float* out) {
  float dmin = 3.402823466e+38f, tmin = 0;
  const float* pmin = nullptr;
  const float* pmax = nullptr;
  for (int i = 0; i < r.tri_count; ++i) {
    const uint8_t* tris = &nav.dtris[(size_t)(r.tri_base + i) * 4];
    const uint8_t tf = tris[3];
    if (kOnlyBoundary && (tf & 0x15) == 0) continue;
    const float* v[3] = {detail_vert(nav, r, tris[0]), detail_vert(nav, r, tris[1]), detail_vert(nav, r, tris[2])};
    for (int k = 0, j = 2; k < 3; j = k++) {
      if ((((tf >> (j * 2)) & 1) == 0) && (kOnlyBoundary || tris[j] < tris[k])) continue;
      float t;
      const float d = dist_pt_seg_sqr2d(px, pz, v[j], v[k], t);
      if (d < dmin) { dmin = d; tmin = t; pmin = v[j]; pmax = v[k]; }
    }
  }
  if (!pmin) { out[0] = px; out[1] = py; out[2] = pz; return; }
  out[0] = pmin[0] + (pmax[0] - pmin[0]) * tmin;
  out[1] = pmin[1] + (pmax[1] - pmin[1]) * tmin;
  out[2] = pmin[2] + (pmax[2] - pmin[2]) * tmin;
}

// dtNavMesh::getPolyHeight: false when (px,pz) is outside the polygon.
BPSX_DEV bool poly_height(const NavData& nav, const PolyRec& r, float px, float py, float pz, float& h) {
  if (r.type != 0) return false;
  if (!point_in_poly(px, pz, r)) return false;
  for (int j = 0; j < r.tri_count; ++j) {
    const uint8_t* t = &nav.dtris[(size_t)(r.tri_base + j) * 4];
    if (height_on_triangle(px, pz, detail_vert(nav, r, t[0]), detail_vert(nav, r, t[1]), detail_vert(nav, r, t[2]), h))
      return true;
  }
  float c[3];
  closest_on_detail_edges<false>(nav, r, px, py, pz, c);
  h = c[1];
  return true;
}

// closestPointOnPolyBoundary: the point itself when inside (xz), else its projection onto
// the nearest polygon edge.
BPSX_DEV void closest_on_poly_boundary(const PolyRec& r, const float* pos, float* out) {
  float ed[kNvp], et[kNvp];
  bool c = false;
  const int nv = r.nv;
  for (int i = 0, j = nv - 1; i < nv; j = i++) {
    const float* vi = r.v[i];
    const float* vj = r.v[j];
    if (((vi[2] > pos[2]) != (vj[2] > pos[2])) &&
        (pos[0] < (vj[0] - vi[0]) * (pos[2] - vi[2]) / (vj[2] - vi[2]) + vi[0]))
      c = !c;
    ed[j] = dist_pt_seg_sqr2d(pos[0], pos[2], vj, vi, et[j]);
  }
  if (c) { out[0] = pos[0]; out[1] = pos[1]; out[2] = pos[2]; return; }
  float dmin = ed[0];
  int imin = 0;
  for (int i = 1; i < nv; ++i)
    if (ed[i] < dmin) { dmin = ed[i]; imin = i; }
  const float* va = r.v[imin];
  const float* vb = r.v[(imin + 1) % nv];
  const float t = et[imin];
  out[0] = va[0] + (vb[0] - va[0]) * t;
  out[1] = va[1] + (vb[1] - va[1]) * t;
  out[2] = va[2] + (vb[2] - va[2]) * t;
}

// Polygon index of a ref within its scene, or kInvalidPoly (dtNavMesh::isValidPolyRef).
BPSX_DEV uint32_t decode_ref(const SceneDev& s, uint32_t ref) {
  if (!ref) return kInvalidPoly;
  const uint32_t ip = ref & s.poly_mask;
  if ((ref & ~s.poly_mask) != s.ref_base || ip >= s.poly_count) return kInvalidPoly;
  return ip;
}

// One candidate of the nearest-polygon search: distance rule of dtFindNearestPolyQuery.
BPSX_DEV float snap_candidate(const NavData& nav, const SceneDev& s, const PolyRec& r, float px, float py, float pz,
                              float* cp) {
  float h;
  if (poly_height(nav, r, px, py, pz, h)) {
    cp[0] = px; cp[1] = h; cp[2] = pz;
    float d = fabsf(py - h) - s.climb;
    return d > 0 ? d * d : 0;
  }
  closest_on_detail_edges<true>(nav, r, px, py, pz, cp);
  const float dx = px - cp[0], dy = py - cp[1], dz = pz - cp[2];
  return dx * dx + dy * dy + dz * dz;
}

constexpr float kSnapHalf = 2.0f;
// A box in the tree's units as it is compared with a node's bounds, two 16-bit numbers a word: no number of the first two may be
// below that of the node's first two words, nor one of the third above that of the node's third, where what stands for
// the greater end of an interval in a word of smaller ends (bmin x in w1) is there as its complement.
struct SnapBox {
  uint32_t w0, w1, w2;   // bmax x, y; bmax z, ~bmin x; bmin y, z
  bool hit_tile;
};
BPSX_DEV float clampf(float v, float lo, float hi) { return v < lo ? lo : (v > hi ? hi : v); }
// the query box around a point: the reference's has a half extent of 2 m in x and z
BPSX_DEV SnapBox snap_box(const SceneDev& s, float px, float py, float pz, float half) {
  SnapBox b;
  const float qmin[3] = {px - half, py - 4.0f, pz - half};
  const float qmax[3] = {px + half, py + 4.0f, pz + half};
  const int minx = (int)floorf((qmin[0] - s.orig[0]) / s.tile_w), miny = (int)floorf((qmin[2] - s.orig[2]) / s.tile_h);
  const int maxx = (int)floorf((qmax[0] - s.orig[0]) / s.tile_w), maxy = (int)floorf((qmax[2] - s.orig[2]) / s.tile_h);
  b.hit_tile = !(s.tx < minx || s.tx > maxx || s.ty < miny || s.ty > maxy);
  uint32_t lo16[3], hi16[3];
  for (int k = 0; k < 3; ++k) {
    const float lo = clampf(qmin[k], s.bmin[k], s.bmax[k]) - s.bmin[k];
    const float hi = clampf(qmax[k], s.bmin[k], s.bmax[k]) - s.bmin[k];
    lo16[k] = (uint16_t)((uint16_t)(int)(s.qfac * lo) & 0xfffe);
    hi16[k] = (uint16_t)((uint16_t)(int)(s.qfac * hi + 1) | 1);
  }
  b.w0 = hi16[0] | (hi16[1] << 16);
  b.w1 = hi16[2] | ((lo16[0] ^ 0xffffu) << 16);
  b.w2 = lo16[1] | (lo16[2] << 16);
  return b;
}
// by how much the 16-bit halves of a are above those of b, each 0 if it is not
BPSX_DEV uint32_t above16(uint32_t a, uint32_t b) {
  uint32_t d;
  asm("v_pk_sub_u16 %0, %1, %2 clamp" : "=v"(d) : "v"(a), "v"(b));
  return d;
}
// (Number by number the test is some twenty instructions, this way six.)
struct BVBounds { uint32_t w0, w1, w2, ab; };   // a node's words
static_assert(sizeof(BVBounds) == sizeof(BVNodeDev) && offsetof(BVNodeDev, bmax) == 6 && offsetof(BVNodeDev, a) == 12, "bmin x, y; bmin z, bmax x; bmax y, z");
BPSX_DEV bool box_overlaps(const SnapBox& box, uint32_t w0, uint32_t w1, uint32_t w2) {
  return (above16(w0, box.w0) | above16(w1 ^ 0xffff0000u, box.w1) | above16(box.w2, w2)) == 0;
}
BPSX_DEV bool box_overlaps(const SnapBox& box, const BVBounds& nd) { return box_overlaps(box, nd.w0, nd.w1, nd.w2); }
BPSX_DEV BVBounds bv_node(const BVNodeDev* nodes, uint32_t i) {
  const uint4 v = reinterpret_cast<const uint4*>(nodes)[i];
  return {v.x, v.y, v.z, v.w};
}

// snapPoint, one lane per point: BV-tree walk with escape indices, candidates taken in tree
// order with a strict '<' so the first of equally near polygons wins.  For trees whose inner nodes do
// not bound what lies below them (see SceneDev::snap_leaves).
BPSX_DEV NavPt snap_point(const NavData& nav, const SceneDev& s, float px, float py, float pz, uint32_t* ncand) {
  const float qnan = __int_as_float(0x7fc00000);
  NavPt out{qnan, qnan, qnan, 0};
  if (!finite3(px, py, pz)) return out;
  const SnapBox box = snap_box(s, px, py, pz, kSnapHalf);
  if (!box.hit_tile) return out;
  float best = 3.402823466e+38f;
  float bp[3] = {0, 0, 0};
  uint32_t bestIp = kInvalidPoly;
  uint32_t i = 0;
  while (i < s.bv_count) {
    const BVBounds nd = bv_node(nav.bv, s.bv_base + i);
    const bool overlap = box_overlaps(box, nd);
    const uint32_t a = nd.ab & 0xffffu;
    const bool leaf = nd.ab >> 16 == kBVLeaf;
    if (leaf && overlap) {
      const PolyRec& r = nav.polys[s.poly_base + a];
      if (r.flags & 1) {
        float cp[3];
        const float d = snap_candidate(nav, s, r, px, py, pz, cp);
        (*ncand)++;
        if (d < best) { best = d; bestIp = a; bp[0] = cp[0]; bp[1] = cp[1]; bp[2] = cp[2]; }
      }
    }
    if (overlap || leaf) i++;
    else i += a;
  }
  if (bestIp == kInvalidPoly || isnan(bp[0])) return out;
  out.x = bp[0]; out.y = bp[1]; out.z = bp[2];
  out.ref = s.ref_base | bestIp;
  return out;
}

// A polygon record in registers, for the move of one agent per lane: its first 112 bytes arrive
// with seven 16-byte loads that go out together, where the loops over a record in memory pay a
// load and a wait for every field as they come to it (a forward move is one chain of dependent
// loads: state, scene, polygon, neighbour polygon, height mesh).  Every index into the words is
// a compile-time constant: loops over vertices are unrolled in the source (static_for), and a
// vertex or neighbour code with a run-time index is picked by a chain of selects whose operands
// the optimiser cannot trace back to the array (PolyRegs::reg), because either an index that
// is still a loop variable or a select between two loads of the array makes it an array in
// scratch memory again.  Same float operations in the same order as the versions on records
// in memory above.
// (lambdas handed to static_for are marked BPSX_INLINE_LAMBDA: inlined together with the functions
// around them, before the optimiser first looks at the record)
#define BPSX_INLINE_LAMBDA __attribute__((always_inline))
template <int I> struct Idx { static constexpr int value = I; };
template <int B, int E, class F> BPSX_DEV void static_for(F&& f) {
  if constexpr (B < E) {
    f(Idx<B>{});
    static_for<B + 1, E>(f);
  }
}
struct PolyRegs {
  uint32_t w[28];
  BPSX_DEV void load(const PolyRec* p) {
    const uint4* s = reinterpret_cast<const uint4*>(p);
    static_for<0, 7>([&](auto K) BPSX_INLINE_LAMBDA {
      constexpr int k = decltype(K)::value;
      const uint4 q = s[k];
      w[4 * k] = q.x; w[4 * k + 1] = q.y; w[4 * k + 2] = q.z; w[4 * k + 3] = q.w;
    });
  }
  static_assert(offsetof(PolyRec, nei) == 72 && offsetof(PolyRec, walk) == 84 && offsetof(PolyRec, flags) == 96 &&
                offsetof(PolyRec, nv) == 98 && offsetof(PolyRec, type) == 99 && offsetof(PolyRec, tri_base) == 100 &&
                offsetof(PolyRec, dvert_base) == 104 && offsetof(PolyRec, tri_count) == 108, "PolyRegs follows PolyRec's layout");
  template <int I> BPSX_DEV float x() const { return __uint_as_float(w[3 * I]); }
  template <int I> BPSX_DEV float y() const { return __uint_as_float(w[3 * I + 1]); }
  template <int I> BPSX_DEV float z() const { return __uint_as_float(w[3 * I + 2]); }
  template <int J> BPSX_DEV uint32_t nei() const { return (w[18 + (J >> 1)] >> (16 * (J & 1))) & 0xffffu; }
  template <int J> BPSX_DEV uint32_t walk() const { return (w[21 + (J >> 1)] >> (16 * (J & 1))) & 0xffffu; }
  BPSX_DEV int nv() const { return (int)((w[24] >> 16) & 0xffu); }
  BPSX_DEV uint32_t type() const { return w[24] >> 24; }
  BPSX_DEV uint32_t tri_base() const { return w[25]; }
  BPSX_DEV uint32_t dvert_base() const { return w[26]; }
  BPSX_DEV int tri_count() const { return (int)(w[27] & 0xffu); }
  // vertex k, k known at run time only.  The words pass through an empty asm first: selects
  // between loads of the array would be folded into one load at a selected address, and the
  // record would have to live in (scratch) memory for it.
  static BPSX_DEV uint32_t reg(uint32_t v) { asm("" : "+v"(v)); return v; }
  BPSX_DEV uint32_t word(int k, int stride, int base) const {   // w[base + stride * k], k in 0..5
    const uint32_t a0 = reg(w[base]), a1 = reg(w[base + stride]), a2 = reg(w[base + 2 * stride]), a3 = reg(w[base + 3 * stride]),
                   a4 = reg(w[base + 4 * stride]), a5 = reg(w[base + 5 * stride]);
    return k == 5 ? a5 : k == 4 ? a4 : k == 3 ? a3 : k == 2 ? a2 : k == 1 ? a1 : a0;
  }
  BPSX_DEV void vertex(int k, float* o) const {
    o[0] = __uint_as_float(word(k, 3, 0));
    o[1] = __uint_as_float(word(k, 3, 1));
    o[2] = __uint_as_float(word(k, 3, 2));
  }
  BPSX_DEV void codes(int k, uint32_t* nei_k, uint32_t* walk_k) const {
    const uint32_t n = word(k >> 1, 1, 18), wk = word(k >> 1, 1, 21);   // two 16-bit codes per word; k >> 1 in 0..2
    *nei_k = (n >> (16 * (k & 1))) & 0xffffu;
    *walk_k = (wk >> (16 * (k & 1))) & 0xffffu;
  }
};

BPSX_DEV bool point_in_poly(float px, float pz, const PolyRegs& P) {
  bool c = false;
  const int nv = P.nv();
  float vj[3];
  P.vertex(nv - 1, vj);
  float jx = vj[0], jz = vj[2];
  static_for<0, kNvp>([&](auto I) BPSX_INLINE_LAMBDA {
    constexpr int i = decltype(I)::value;
    const float ix = P.x<i>(), iz = P.z<i>();
    const bool crosses = ((iz > pz) != (jz > pz)) && (px < (jx - ix) * (pz - iz) / (jz - iz) + ix);
    c ^= (i < nv) && crosses;
    jx = ix; jz = iz;
  });
  return c;
}

// dtNavMesh::getPolyHeight on a record in registers (`mem`: the same record in memory, for the
// rare fall-back to the detail edges).  The index words of the first four detail triangles go
// out together.
BPSX_DEV bool poly_over(const PolyRegs& P, float px, float pz) { return P.type() == 0 && point_in_poly(px, pz, P); }
BPSX_DEV float height_over(const NavData& nav, const PolyRegs& P, const PolyRec& mem, float px, float py, float pz) {   // of a polygon that it is over
  float h;
  const int tc = P.tri_count(), nv = P.nv();
  const uint32_t* tris = reinterpret_cast<const uint32_t*>(nav.dtris) + P.tri_base();   // four bytes per triangle
  const uint32_t t0 = 0 < tc ? tris[0] : 0u, t1 = 1 < tc ? tris[1] : 0u, t2 = 2 < tc ? tris[2] : 0u, t3 = 3 < tc ? tris[3] : 0u;
  auto corner = [&](uint32_t k, float* o) BPSX_INLINE_LAMBDA {
    if ((int)k < nv) P.vertex((int)k, o);
    else {
      const float* d = &nav.dverts[(size_t)(P.dvert_base() + (k - (uint32_t)nv)) * 3];
      o[0] = d[0]; o[1] = d[1]; o[2] = d[2];
    }
  };
  auto inside = [&](uint32_t t) BPSX_INLINE_LAMBDA {
    float a[3], b[3], c[3];
    corner(t & 0xffu, a); corner((t >> 8) & 0xffu, b); corner((t >> 16) & 0xffu, c);
    return height_on_triangle(px, pz, a, b, c, h);
  };
  if (0 < tc && inside(t0)) return h;
  if (1 < tc && inside(t1)) return h;
  if (2 < tc && inside(t2)) return h;
  if (3 < tc && inside(t3)) return h;
  for (int j = 4; j < tc; ++j)
    if (inside(tris[j])) return h;
  float c[3];
  closest_on_detail_edges<false>(nav, mem, px, py, pz, c);
  return c[1];
}
BPSX_DEV bool poly_height(const NavData& nav, const PolyRegs& P, const PolyRec& mem, float px, float py, float pz, float& h) {
  if (!poly_over(P, px, pz)) return false;
  h = height_over(nav, P, mem, px, py, pz);
  return true;
}

// the smallest v of a wavefront, known to be uniform (the totals of a row of 16 lanes through quad
// permutes and mirrors, then across the rows)
BPSX_DEV uint32_t wave_umin(uint32_t v) {
  auto take = [&v](uint32_t o) BPSX_INLINE_LAMBDA { v = o < v ? o : v; };
  take((uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0xb1 /* quad_perm [1,0,3,2] */, 0xf, 0xf, false));
  take((uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x4e /* quad_perm [2,3,0,1] */, 0xf, 0xf, false));
  take((uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x141 /* row_half_mirror */, 0xf, 0xf, false));
  take((uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x140 /* row_mirror */, 0xf, 0xf, false));
  take((uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x142 /* row_bcast:15 */, 0xa, 0xf, false));
  take((uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x143 /* row_bcast:31 */, 0xc, 0xf, false));
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// closest_on_detail_edges<true> on a record in registers.
BPSX_DEV void closest_on_boundary(const NavData& nav, const PolyRegs& P, float px, float py, float pz, float* out) {
  float dmin = 3.402823466e+38f, tmin = 0;
  float lo[3] = {px, py, pz}, hi[3] = {px, py, pz};   // without an edge the point itself
  const int tc = P.tri_count(), nv = P.nv();
  const uint32_t* tris = reinterpret_cast<const uint32_t*>(nav.dtris) + P.tri_base();
  auto corner = [&](uint32_t k, float* o) BPSX_INLINE_LAMBDA {
    if ((int)k < nv) P.vertex((int)k, o);
    else {
      const float* d = &nav.dverts[(size_t)(P.dvert_base() + (k - (uint32_t)nv)) * 3];
      o[0] = d[0]; o[1] = d[1]; o[2] = d[2];
    }
  };
  uint32_t next = 0 < tc ? tris[0] : 0u;
  for (int i = 0; i < tc; ++i) {
    const uint32_t t = next;
    next = i + 1 < tc ? tris[i + 1] : 0u;
    if ((t & 0x15000000u) == 0) continue;
    float v[3][3];
    corner(t & 0xffu, v[0]); corner((t >> 8) & 0xffu, v[1]); corner((t >> 16) & 0xffu, v[2]);
    auto edge = [&](uint32_t flag, const float* a, const float* b) BPSX_INLINE_LAMBDA {
      if (!(t & flag)) return;
      float u;
      const float d = dist_pt_seg_sqr2d(px, pz, a, b, u);
      if (d < dmin) {
        dmin = d; tmin = u;
        lo[0] = a[0]; lo[1] = a[1]; lo[2] = a[2];
        hi[0] = b[0]; hi[1] = b[1]; hi[2] = b[2];
      }
    };
    edge(0x10000000u, v[2], v[0]);
    edge(0x01000000u, v[0], v[1]);
    edge(0x04000000u, v[1], v[2]);
  }
  if (dmin == 3.402823466e+38f) { out[0] = px; out[1] = py; out[2] = pz; return; }
  out[0] = lo[0] + (hi[0] - lo[0]) * tmin;
  out[1] = lo[1] + (hi[1] - lo[1]) * tmin;
  out[2] = lo[2] + (hi[2] - lo[2]) * tmin;
}

// snapPoint by a whole wavefront.  The reference takes every walkable polygon whose bounds overlap a
// box of 4 x 8 x 4 m in the order of the BV tree's array and keeps the first of the nearest ones: the
// smallest (distance, place in the array).
//
// The walkable leaves lie in one array in that order, with the bounds of every 64 of them in another
// (a run of the tree's in-order array is a compact part of the mesh): all groups' bounds are read at
// once, then the leaves of four groups that overlap, 64 in one load, then one polygon per lane.  That
// is four dependent loads where a descent of the binary tree has seventeen.  (One load of groups and
// one of leaves after the other, a batch evaluated as soon as it was full, and registers for three
// instead of four wavefronts per SIMD: 277 us instead of 238 for 50000 points over a cluttered plan,
// 31 instead of 20 for the 4096 of a reset over mazes.)
//
// Where the scene allows it (SceneDev::snap_prune) the box begins with a half extent of kSnapFirst and
// grows: a polygon outside a box of half extent r is at least r - kSnapSlack away, so once the best
// distance is below that, the reference's box holds no better one and none as good.  In a batch, the
// polygons that the point is above or below come first, and the boundary of the others is looked at
// only if their bounds are no farther away than the best so far.
//
// Bound by the latency of those loads and by the divide-heavy edge distances of the candidates: most
// points are on the mesh, and of the 200 polygons of a cluttered plan in the full box five remain.
// (50000 points over a cluttered plan of 20k polygons: 1730 -> 277 us, then 238; 4096 points there, a wavefront
// each, 64 -> 14 us; snaps of 165 new episodes there next to the searches 135 -> 24 us.  The descent
// tested one level per load and evaluated the whole box, a field of a record at a time.)
constexpr float kSnapFirst = 0.25f;
// above the rounding of interpolated points, distances and boxes at coordinates up to kSnapCoord, and
// what height samples may lie outside of their polygon's bounds (kSnapOverhang, checked at load)
constexpr float kSnapSlack = 1e-3f;
static_assert(kSnapGroup == 64, "a lane per leaf of a group");
constexpr int kSnapGroupLoads = 8, kSnapLeafLoads = 4;   // groups' bounds, 64 each, and groups' leaves that are asked for at once
struct SnapLds {
  uint16_t group[64 * kSnapGroupLoads];   // the groups that overlap the box
  // candidates waiting: less than a batch is left when the leaves of further groups join
  uint16_t cand_rank[64 * (kSnapLeafLoads + 1)];   // place among the leaves
  uint16_t cand_poly[64 * (kSnapLeafLoads + 1)];
};
// the square of how far a point is at least from a polygon that it is not above or below
BPSX_DEV float snap_bounds_dist2(const PolyRegs& P, float px, float pz) {
  float x0 = P.x<0>(), x1 = x0, z0 = P.z<0>(), z1 = z0;
  const int nv = P.nv();
  static_for<1, kNvp>([&](auto I) BPSX_INLINE_LAMBDA {
    constexpr int i = decltype(I)::value;
    if (i < nv) {
      x0 = fminf(x0, P.x<i>()); x1 = fmaxf(x1, P.x<i>());
      z0 = fminf(z0, P.z<i>()); z1 = fmaxf(z1, P.z<i>());
    }
  });
  const float bx = fmaxf(fmaxf(x0 - px, px - x1) - kSnapSlack, 0.0f), bz = fmaxf(fmaxf(z0 - pz, pz - z1) - kSnapSlack, 0.0f);
  return bx * bx + bz * bz;
}
// The polygons of leaves that overlap `box`, without those that overlap `before` if that has been looked
// at (grown), join the candidates: put(c, leaf, polygon) for the c-th.  flush() takes up to 64 of them out;
// it is called while there are that many, and with `all` until none is left.
template <class Put, class Flush>
BPSX_DEV void snap_candidates(const BVNodeDev* leaves, uint32_t nleaves, uint16_t* list, const SnapBox& box, const SnapBox& before, bool grown,
                              bool all, int lane, int& ncands, Put put, Flush flush) {
  const uint32_t ngroups = (nleaves + 63u) / 64u;
  const BVNodeDev* groups = leaves + nleaves;
  for (uint32_t g0 = 0; g0 < ngroups; g0 += 64 * kSnapGroupLoads) {
    BVBounds gr[kSnapGroupLoads];
#pragma unroll
    for (int k = 0; k < kSnapGroupLoads; ++k) {
      const uint32_t g = g0 + (uint32_t)(64 * k + lane);
      gr[k] = bv_node(groups, g < ngroups ? g : ngroups - 1u);
    }
    int ng = 0;
#pragma unroll
    for (int k = 0; k < kSnapGroupLoads; ++k) {
      const uint32_t g = g0 + (uint32_t)(64 * k + lane);
      const bool over = g < ngroups && box_overlaps(box, gr[k]);
      const unsigned long long m = __ballot(over);
      if (over) list[ng + __popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)g;
      ng += (int)__popcll(m);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const bool last = all && g0 + 64 * kSnapGroupLoads >= ngroups;
    for (int j = 0;; j += kSnapLeafLoads) {
      if (j < ng) {
        BVBounds nd[kSnapLeafLoads];
        uint32_t at[kSnapLeafLoads];
#pragma unroll
        for (int k = 0; k < kSnapLeafLoads; ++k) {
          const int gk = __builtin_amdgcn_readfirstlane((int)list[j + k < ng ? j + k : j]);
          at[k] = (uint32_t)gk * kSnapGroup + (uint32_t)lane;
          nd[k] = bv_node(leaves, at[k] < nleaves ? at[k] : nleaves - 1u);
        }
#pragma unroll
        for (int k = 0; k < kSnapLeafLoads; ++k) {
          // they join the candidates
          const bool isCand = j + k < ng && at[k] < nleaves && box_overlaps(box, nd[k]) && !(grown && box_overlaps(before, nd[k]));
          const unsigned long long m = __ballot(isCand);
          if (isCand) put(ncands + (int)__popcll(m & ((1ull << lane) - 1ull)), at[k], (uint16_t)nd[k].ab);
          ncands += (int)__popcll(m);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
      const bool end = j + kSnapLeafLoads >= ng;
      while (ncands >= (end && last ? 1 : 64)) flush();   // full batches, and what is left at the end
      if (end) break;
    }
  }
}
BPSX_DEV NavPt snap_point_wave(const NavData& nav, const SceneDev& s, float px, float py, float pz, SnapLds& L,
                               uint32_t* ncand) {
  const int lane = (int)(threadIdx.x & 63);
  const float qnan = __int_as_float(0x7fc00000);
  constexpr float kNone = 3.402823466e+38f;
  NavPt out{qnan, qnan, qnan, 0};
  if (!finite3(px, py, pz)) return out;
  if (!snap_box(s, px, py, pz, kSnapHalf).hit_tile || s.bv_count == 0) return out;
  if (!s.snap_leaves) return snap_point(nav, s, px, py, pz, ncand);  // every lane walks the same tree
  const uint32_t nleaves = s.snap_leaves;
  const BVNodeDev* leaves = nav.bv + s.bv_base + s.bv_count;
  const bool prune = s.snap_prune && fabsf(px) <= 2.0f * kSnapCoord && fabsf(pz) <= 2.0f * kSnapCoord;
  float best = kNone;              // per-lane running best
  uint32_t bestKey = 0xffffffffu;  // place of the lane's best candidate
  uint32_t bestIp = kInvalidPoly;
  float bp[3] = {0, 0, 0};
  int ncands = 0;  // candidates waiting (uniform)
  auto flush = [&]() {
    const int fit = ncands < 64 ? ncands : 64;
    ncands -= fit;
    const bool have = lane < fit;
    *ncand += (uint32_t)fit;
    uint32_t ip = 0, key = 0;
    PolyRegs P;
    const PolyRec* rec = nullptr;
    bool inside = false;
    float h = 0;
    auto take = [&](float d, float x, float y, float z) BPSX_INLINE_LAMBDA {
      if (d < best || (d == best && d < kNone && key < bestKey)) {
        best = d; bestKey = key; bestIp = ip; bp[0] = x; bp[1] = y; bp[2] = z;
      }
    };
    if (have) {
      ip = L.cand_poly[ncands + lane];
      key = L.cand_rank[ncands + lane];
      rec = &nav.polys[s.poly_base + ip];
      P.load(rec);
      inside = poly_height(nav, P, *rec, px, py, pz, h);
      if (inside) {
        const float d = fabsf(py - h) - s.climb;
        take(d > 0 ? d * d : 0, px, h, pz);
      }
    }
    const float reached = __uint_as_float(wave_umin(__float_as_uint(best)));
    if (have && !inside) {
      if (!(prune && snap_bounds_dist2(P, px, pz) > reached)) {
        float cp[3];
        closest_on_boundary(nav, P, px, py, pz, cp);
        const float dx = px - cp[0], dy = py - cp[1], dz = pz - cp[2];
        take(dx * dx + dy * dy + dz * dz, cp[0], cp[1], cp[2]);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  float half = prune ? kSnapFirst : kSnapHalf;
  SnapBox box = snap_box(s, px, py, pz, half), before = box;
  bool grown = false;   // what overlaps `before` has been looked at
  for (;;) {
    snap_candidates(leaves, nleaves, L.group, box, before, grown, true, lane, ncands, [&](int c, uint32_t at, uint16_t ip) BPSX_INLINE_LAMBDA {
      L.cand_rank[c] = (uint16_t)at;
      L.cand_poly[c] = ip;
    }, flush);
    if (half >= kSnapHalf) break;
    const float reached = __uint_as_float(wave_umin(__float_as_uint(best)));
    const float clear = half - kSnapSlack;
    if (reached < clear * clear) break;
    // the next box reaches as far as the best so far, or is three times as wide
    half = fminf(reached < kNone ? sqrtf(reached) * 1.0001f + 2.0f * kSnapSlack : 3.0f * half, kSnapHalf);
    before = box;
    grown = true;
    box = snap_box(s, px, py, pz, half);
  }
  // the smallest (distance, place in the array)
  const uint32_t dist = wave_umin(__float_as_uint(best));
  const bool nearest = bestIp != kInvalidPoly && __float_as_uint(best) == dist;
  const uint32_t key = wave_umin(nearest ? bestKey : 0xffffffffu);
  const unsigned long long won = __ballot(nearest && bestKey == key);
  if (!won) return out;
  const int w = __builtin_ctzll(won);
  const float x = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(bp[0]), w));
  if (isnan(x)) return out;
  out.x = x;
  out.y = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(bp[1]), w));
  out.z = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(bp[2]), w));
  out.ref = s.ref_base | (uint32_t)__builtin_amdgcn_readlane((int)bestIp, w);
  return out;
}

// The same for up to kSnapBatch points of one scene by one wavefront.  A point has about five candidates in the first box and some
// twenty in all, so evaluating each point's on their own leaves most lanes idle: here the points' boxes are scanned one after the
// other and their candidates are looked at together, 64 at a time, whichever points they belong to.  Point p's state is lane p's;
// the smallest (distance, place in the array) of each point is found by atomics in LDS.  The groups' bounds are read once for all
// points, and the leaves of four groups at a time, whichever points' boxes those overlap.
//
// The candidates are first only sorted: whether their points are over them takes a tenth of the instructions that a distance
// does.  The few that are (one or two of a point's) are evaluated together, and then, with what those have reached, the others
// that may still be nearer.  So full wavefronts evaluate heights and edges, each once or twice in a round of boxes, where 64
// candidates as they came had some of either kind.  Bound by the sorting's and the scan's instructions.
// (50000 points over a cluttered plan, read and written in pinned memory: 168 us with the groups scanned anew for every
// point, their list read back from LDS before their leaves were asked for, and boxes compared number by number; 155 with five
// batches of 64 candidates evaluated as they came; 127 now.  In device memory 238 us by a wavefront for each, 150, 136, 106.)
constexpr int kSnapBatch = 16;
constexpr int kSnapBeside = 256;   // 13 points' candidates of a round
constexpr int kSnapPairs = 1024, kSnapPairShift = 12;   // all groups of a round for one point more fit
static_assert(kSnapPairs > 64 * kSnapGroupLoads && kSnapBatch <= (1 << (16 - kSnapPairShift)) && 0x8000u / kSnapGroup <= (1u << kSnapPairShift), "a pair has 16 bits, and a tile up to 32767 polygons");
struct SnapBatchLds {
  SnapLds snap;
  uint8_t cand_point[64 * (kSnapLeafLoads + 1)];
  uint16_t pair[kSnapPairs];             // a group that overlaps a point's box, the point
  unsigned long long best[kSnapBatch];   // bits of the smallest distance, place of its polygon
  float pt[kSnapBatch][4];               // the point; whether its box grows
  float at[kSnapBatch][4];               // the nearest point so far, its polygon
  // candidates, place and polygon, whose points are over them, and the others with a bound of their squared distances
  uint32_t over[128], beside[kSnapBeside];
  float beside_dist2[kSnapBeside];
  uint8_t over_point[128], beside_point[kSnapBeside];
};
BPSX_DEV NavPt snap_points_batch(const NavData& nav, const SceneDev& s, bool mine, float px, float py, float pz, SnapBatchLds& B) {
  const int lane = (int)(threadIdx.x & 63);
  const float qnan = __int_as_float(0x7fc00000);
  constexpr float kNone = 3.402823466e+38f;
  NavPt out{qnan, qnan, qnan, 0};
  uint32_t unused = 0;
  if (!s.snap_leaves) return mine ? snap_point(nav, s, px, py, pz, &unused) : out;
  auto sync = [&]() BPSX_INLINE_LAMBDA {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  mine = mine && finite3(px, py, pz);
  mine = mine && snap_box(s, px, py, pz, kSnapHalf).hit_tile && s.bv_count != 0;
  const bool prune = s.snap_prune && fabsf(px) <= 2.0f * kSnapCoord && fabsf(pz) <= 2.0f * kSnapCoord;
  if (lane < kSnapBatch) {
    B.best[lane] = ((unsigned long long)__float_as_uint(kNone) << 32) | 0xffffffffu;
    B.pt[lane][0] = px; B.pt[lane][1] = py; B.pt[lane][2] = pz; B.pt[lane][3] = prune ? 1.0f : 0.0f;
  }
  sync();
  const BVNodeDev* leaves = nav.bv + s.bv_base + s.bv_count;
  int ncands = 0;
  int nover = 0, nbeside = 0;
  const auto before_me = [](unsigned long long m) BPSX_INLINE_LAMBDA {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
  };
  const auto reached_by = [&](uint32_t p) BPSX_INLINE_LAMBDA { return __uint_as_float((uint32_t)(B.best[p] >> 32)); };
  // a candidate (place << 16 | polygon) of point p lies at cp, the square root of d away
  auto offer = [&](bool have, uint32_t cand, uint32_t p, float d, float x, float y, float z) BPSX_INLINE_LAMBDA {
    const bool counts = have && d < kNone;
    const unsigned long long found = ((unsigned long long)__float_as_uint(d) << 32) | (cand >> 16);
    if (counts) atomicMin(&B.best[p], found);
    sync();
    if (counts && B.best[p] == found) {   // one lane at most: a point meets each leaf once
      B.at[p][0] = x; B.at[p][1] = y; B.at[p][2] = z; B.at[p][3] = __uint_as_float(cand & 0xffffu);
    }
    sync();
  };
  // 64 candidates become ones over which their points are and ones beside them
  auto sort_out = [&]() BPSX_INLINE_LAMBDA {
    const int fit = ncands < 64 ? ncands : 64;
    ncands -= fit;
    uint32_t cand = 0, p = 0;
    bool over = false, beside = false;
    float dist2 = 0;
    if (lane < fit) {
      cand = ((uint32_t)B.snap.cand_rank[ncands + lane] << 16) | B.snap.cand_poly[ncands + lane];
      p = B.cand_point[ncands + lane];
      const float qx = B.pt[p][0], qz = B.pt[p][2];
      PolyRegs P;
      P.load(&nav.polys[s.poly_base + (cand & 0xffffu)]);
      over = poly_over(P, qx, qz);
      if (B.pt[p][3] != 0) dist2 = snap_bounds_dist2(P, qx, qz);
      beside = !over && !(dist2 > reached_by(p));
    }
    const unsigned long long o = __ballot(over), b = __ballot(beside);
    if (over) { const int at = nover + before_me(o); B.over[at] = cand; B.over_point[at] = (uint8_t)p; }
    if (beside) { const int at = nbeside + before_me(b); B.beside[at] = cand; B.beside_point[at] = (uint8_t)p; B.beside_dist2[at] = dist2; }
    nover += (int)__popcll(o); nbeside += (int)__popcll(b);
    sync();
  };
  auto heights = [&]() BPSX_INLINE_LAMBDA {
    const int fit = nover < 64 ? nover : 64;
    nover -= fit;
    const bool have = lane < fit;
    uint32_t cand = 0, p = 0;
    float d = 0, qx = 0, qz = 0, h = 0;
    if (have) {
      cand = B.over[nover + lane]; p = B.over_point[nover + lane];
      const PolyRec* rec = &nav.polys[s.poly_base + (cand & 0xffffu)];
      PolyRegs P;
      P.load(rec);
      const float qy = B.pt[p][1];
      qx = B.pt[p][0]; qz = B.pt[p][2];
      h = height_over(nav, P, *rec, qx, qy, qz);
      const float e = fabsf(qy - h) - s.climb;
      d = e > 0 ? e * e : 0;
    }
    offer(have, cand, p, d, qx, h, qz);
  };
  auto boundaries = [&]() BPSX_INLINE_LAMBDA {
    const int fit = nbeside < 64 ? nbeside : 64;
    nbeside -= fit;
    bool have = lane < fit;
    uint32_t cand = 0, p = 0;
    float d = 0, cp[3] = {0, 0, 0};
    if (have) {
      cand = B.beside[nbeside + lane]; p = B.beside_point[nbeside + lane];
      have = !(B.beside_dist2[nbeside + lane] > reached_by(p));
    }
    if (have) {
      PolyRegs P;
      P.load(&nav.polys[s.poly_base + (cand & 0xffffu)]);
      const float qx = B.pt[p][0], qy = B.pt[p][1], qz = B.pt[p][2];
      closest_on_boundary(nav, P, qx, qy, qz, cp);
      const float dx = qx - cp[0], dy = qy - cp[1], dz = qz - cp[2];
      d = dx * dx + dy * dy + dz * dz;
    }
    offer(have, cand, p, d, cp[0], cp[1], cp[2]);
  };
  // Makes room for another sort_out, or evaluates all: the heights first, then of the candidates beside their points those
  // that may still be nearer.
  auto evaluate = [&](bool all) BPSX_INLINE_LAMBDA {
    const bool full = all || nbeside > kSnapBeside - 64;
    while (nover >= (full ? 1 : 64)) heights();
    if (!full) return;
    int left = 0;
    for (int j = 0; j < nbeside; j += 64) {
      uint32_t cand = 0, p = 0;
      float dist2 = 0;
      bool stays = false;
      if (j + lane < nbeside) {
        cand = B.beside[j + lane]; p = B.beside_point[j + lane]; dist2 = B.beside_dist2[j + lane];
        stays = !(dist2 > reached_by(p));
      }
      const unsigned long long m = __ballot(stays);
      sync();
      if (stays) { const int at = left + before_me(m); B.beside[at] = cand; B.beside_point[at] = (uint8_t)p; B.beside_dist2[at] = dist2; }
      left += (int)__popcll(m);
      sync();
    }
    nbeside = left;
    while (nbeside > (all ? 0 : kSnapBeside - 64)) boundaries();
  };
  float half = prune ? kSnapFirst : kSnapHalf;
  SnapBox box = snap_box(s, px, py, pz, half), before = box;
  bool grown = false;   // of all points that are still looked at alike: what overlaps `before` has been looked at
  auto of_lane = [&](const SnapBox& b, int l) BPSX_INLINE_LAMBDA {
    SnapBox r;
    r.w0 = (uint32_t)__builtin_amdgcn_readlane((int)b.w0, l);
    r.w1 = (uint32_t)__builtin_amdgcn_readlane((int)b.w1, l);
    r.w2 = (uint32_t)__builtin_amdgcn_readlane((int)b.w2, l);
    r.hit_tile = true;
    return r;
  };
  const uint32_t nleaves = s.snap_leaves, ngroups = (nleaves + 63u) / 64u;
  const BVNodeDev* groups = leaves + nleaves;
  int npairs = 0;
  // the leaves of the pairs' groups that overlap their points' boxes join the candidates; with `last` all of those are evaluated
  auto look = [&](bool last) {
    sync();
    uint32_t pairs = 0;
    for (int j = 0;; j += kSnapLeafLoads) {
      if (j < npairs) {
        if ((j & 63) == 0) pairs = B.pair[j + lane < npairs ? j + lane : npairs - 1];
        BVBounds nd[kSnapLeafLoads];
        uint32_t at[kSnapLeafLoads];
        int pt[kSnapLeafLoads];
#pragma unroll
        for (int k = 0; k < kSnapLeafLoads; ++k) {
          const uint32_t pair = (uint32_t)__builtin_amdgcn_readlane((int)pairs, (j + k < npairs ? j + k : j) & 63);
          pt[k] = (int)(pair >> kSnapPairShift);
          at[k] = (pair & ((1u << kSnapPairShift) - 1u)) * kSnapGroup + (uint32_t)lane;
          nd[k] = bv_node(leaves, at[k] < nleaves ? at[k] : nleaves - 1u);
        }
#pragma unroll
        for (int k = 0; k < kSnapLeafLoads; ++k) {
          const bool isCand = j + k < npairs && at[k] < nleaves && box_overlaps(of_lane(box, pt[k]), nd[k]) && !(grown && box_overlaps(of_lane(before, pt[k]), nd[k]));
          const unsigned long long m = __ballot(isCand);
          if (isCand) {
            const int c = ncands + before_me(m);
            B.snap.cand_rank[c] = (uint16_t)at[k];
            B.snap.cand_poly[c] = (uint16_t)nd[k].ab;
            B.cand_point[c] = (uint8_t)pt[k];
          }
          ncands += (int)__popcll(m);
        }
        sync();
      }
      const bool end = j + kSnapLeafLoads >= npairs;
      for (const int least = end && last ? 1 : 64;;) {
        if (ncands >= least) sort_out();
        const bool more = ncands >= least;
        evaluate(end && last && !more);
        if (!more) break;
      }
      if (end) break;
    }
    npairs = 0;
  };
  static_assert(64 % kSnapLeafLoads == 0);
  bool open = mine;
  for (unsigned long long todo = __ballot(open); todo;) {
    for (uint32_t g0 = 0; g0 < ngroups; g0 += 64 * kSnapGroupLoads) {
      for (unsigned long long rest = todo; rest;) {
        // the groups' bounds are read once for all points, if the pairs have room
        uint32_t g_w0[kSnapGroupLoads], g_w1[kSnapGroupLoads], g_w2[kSnapGroupLoads];
#pragma unroll
        for (int k = 0; k < kSnapGroupLoads; ++k) {
          const uint32_t g = g0 + (uint32_t)(64 * k + lane);
          const BVBounds v = bv_node(groups, g < ngroups ? g : ngroups - 1u);
          g_w0[k] = v.w0; g_w1[k] = v.w1; g_w2[k] = v.w2;
        }
        do {
          const int p = __builtin_ctzll(rest);
          rest &= rest - 1ull;
          const SnapBox pb = of_lane(box, p);
#pragma unroll
          for (int k = 0; k < kSnapGroupLoads; ++k) {
            if (g0 + 64u * (uint32_t)k >= ngroups) break;
            const uint32_t g = g0 + (uint32_t)(64 * k + lane);
            const bool over = g < ngroups && box_overlaps(pb, g_w0[k], g_w1[k], g_w2[k]);
            const unsigned long long m = __ballot(over);
            if (over)
              B.pair[npairs + before_me(m)] = (uint16_t)(g | ((uint32_t)p << kSnapPairShift));
            npairs += (int)__popcll(m);
          }
        } while (rest && npairs <= kSnapPairs - 64 * kSnapGroupLoads);
        look(!rest && g0 + 64 * kSnapGroupLoads >= ngroups);
      }
    }
    if (open) {
      const float reached = __uint_as_float((uint32_t)(B.best[lane] >> 32)), clear = half - kSnapSlack;
      if (half >= kSnapHalf || reached < clear * clear) open = false;
      else {
        half = fminf(reached < kNone ? sqrtf(reached) * 1.0001f + 2.0f * kSnapSlack : 3.0f * half, kSnapHalf);
        before = box;
        box = snap_box(s, px, py, pz, half);
      }
    }
    grown = true;
    todo = __ballot(open);
  }
  if (!mine || (uint32_t)B.best[lane] == 0xffffffffu) return out;
  const float x = B.at[lane][0];
  if (isnan(x)) return out;
  out.x = x;
  out.y = B.at[lane][1];
  out.z = B.at[lane][2];
  out.ref = s.ref_base | __float_as_uint(B.at[lane][3]);
  return out;
}

// The tiny node pool and the queue of moveAlongSurface, one column per agent of a block, in
// LDS: they are indexed at run time, which in private memory means a trip to scratch (HBM
// behind the vector caches) per access.  A node enters the queue at most once, so the queue
// needs no more entries than there are nodes and is never shifted: `head` moves instead.
constexpr int kMoveItems = 32;   // agents of a block, a row of eight lanes each
struct MoveLds {
  uint16_t node_id[kTinyNodes][kMoveItems];
  uint8_t queue[kTinyNodes][kMoveItems];
};

// tryStep with sliding by one lane, with the reference's node pool as it is: `lane` is its column.
BPSX_DEV NavPt try_step(const NavData& nav, const SceneDev& s, const NavPt& start, float ex, float ey, float ez,
                        uint32_t* npolys, MoveLds& M, int lane) {
  const uint32_t startIp = decode_ref(s, start.ref);
  if (startIp == kInvalidPoly || !finite3(start.x, start.y, start.z) || !finite3(ex, ey, ez)) return start;
  uint64_t closed = 1ull;
  int nnodes = 1;
  int qhead = 0, qtail = 1;   // the reference's stack holds entries [qhead, qtail)
  M.node_id[0][lane] = (uint16_t)startIp;
  M.queue[0][lane] = 0;
  float bx = start.x, by = start.y, bz = start.z;
  float bestDist = 3.402823466e+38f;
  int bestNode = -1;
  const float sx = start.x + (ex - start.x) * 0.5f, sz = start.z + (ez - start.z) * 0.5f;
  const float ddx = ex - start.x, ddy = ey - start.y, ddz = ez - start.z;
  const float sr = sqrtf(ddx * ddx + ddy * ddy + ddz * ddz) / 2.0f + 0.001f;
  const float searchRadSqr = sr * sr;
  PolyRegs P;
  uint32_t loaded = kInvalidPoly;   // the polygon P holds
  while (qhead < qtail) {
    const int cur = M.queue[qhead++][lane];
    loaded = M.node_id[cur][lane];
    P.load(&nav.polys[s.poly_base + loaded]);
    (*npolys)++;
    if (point_in_poly(ex, ez, P)) {
      bestNode = cur;
      bx = ex; by = ey; bz = ez;
      break;
    }
    const int nv = P.nv();
    // edge j -> i with j the vertex before i: (nv - 1, 0), (0, 1), ...
    float vj[3];
    uint32_t neij, walkj;
    P.vertex(nv - 1, vj);
    P.codes(nv - 1, &neij, &walkj);
    static_for<0, kNvp>([&](auto I) BPSX_INLINE_LAMBDA {
      constexpr int i = decltype(I)::value;
      const float vi[3] = {P.x<i>(), P.y<i>(), P.z<i>()};
      if (i < nv) {
        // single-tile meshes carry no tile-border links, so a border edge is a wall
        const uint32_t nb = (neij & 0x8000u) ? 0u : walkj;
        if (!nb) {
          float t;
          const float d = dist_pt_seg_sqr2d(ex, ez, vj, vi, t);
          if (d < bestDist) {
            bx = vj[0] + (vi[0] - vj[0]) * t;
            by = vj[1] + (vi[1] - vj[1]) * t;
            bz = vj[2] + (vi[2] - vj[2]) * t;
            bestDist = d;
            bestNode = cur;
          }
        } else {
          const uint16_t ip = (uint16_t)(nb - 1);
          int nn = -1;
          for (int k = 0; k < nnodes; ++k)
            if (M.node_id[k][lane] == ip) { nn = k; break; }
          bool fits = true;
          if (nn < 0) {
            if (nnodes >= kTinyNodes) fits = false;
            else {
              nn = nnodes++;
              M.node_id[nn][lane] = ip;
            }
          }
          if (fits && !((closed >> nn) & 1ull)) {
            float t;
            const float d = dist_pt_seg_sqr2d(sx, sz, vj, vi, t);
            if (!(d > searchRadSqr) && qtail - qhead < kMoveQueue) {
              closed |= 1ull << nn;
              M.queue[qtail++][lane] = (uint8_t)nn;
            }
          }
        }
      }
      vj[0] = vi[0]; vj[1] = vi[1]; vj[2] = vi[2];
      neij = P.nei<i>(); walkj = P.walk<i>();
    });
  }
  if (bestNode < 0) return start;
  const uint32_t bestIp = M.node_id[bestNode][lane];
  NavPt out{bx, by, bz, s.ref_base | bestIp};
  if (isfinite(bx) && isfinite(bz)) {
    const PolyRec& mem = nav.polys[s.poly_base + bestIp];
    if (bestIp != loaded) P.load(&mem);
    float h;
    if (poly_height(nav, P, mem, bx, by, bz, h)) out.y = h;
  }
  return out;
}

// ---- queries by a row of eight lanes (lanes 8r .. 8r + 7 of a wavefront), which run in step: lane i
// has edge i (the one that ends at vertex i) of the polygon at hand, or one of eight triangles or pivots.
// All lanes of a row take the same branches and hold the same results.
struct Row {
  int el, first;   // lane within the row, the row's first lane in the wavefront
  BPSX_DEV Row() : el((int)(threadIdx.x & 7u)), first((int)(threadIdx.x & 56u)) {}
  BPSX_DEV uint32_t mask(bool b) const { return (uint32_t)(__ballot(b) >> first) & 0xffu; }
  BPSX_DEV float get(float v, int k) const { return __shfl(v, first + k); }
  BPSX_DEV uint32_t get(uint32_t v, int k) const { return (uint32_t)__shfl((int)v, first + k); }
  static BPSX_DEV uint32_t umin(uint32_t v) {
    auto take = [&v](uint32_t o) BPSX_INLINE_LAMBDA { v = o < v ? o : v; };
    take((uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0xb1 /* quad_perm [1,0,3,2] */, 0xf, 0xf, false));
    take((uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x4e /* quad_perm [2,3,0,1] */, 0xf, 0xf, false));
    take((uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x141 /* row_half_mirror */, 0xf, 0xf, false));
    return v;
  }
};
// The edge from vertex j to vertex i = el of a polygon; idle lanes have on == false.
struct RowEdge {
  float i[3], j[3];
  bool on;
  int from;   // j
  BPSX_DEV void load(const Row& row, const PolyRec* r, int nv) {
    const float* v = r->v[row.el < kNvp ? row.el : 0];
    i[0] = v[0]; i[1] = v[1]; i[2] = v[2];
    on = row.el < nv;
    from = row.el == 0 ? nv - 1 : row.el - 1;
    for (int k = 0; k < 3; ++k) j[k] = row.get(i[k], from);
  }
  BPSX_DEV bool inside(const Row& row, float px, float pz) const {
    const bool crosses = on && ((i[2] > pz) != (j[2] > pz)) && (px < (j[0] - i[0]) * (pz - i[2]) / (j[2] - i[2]) + i[0]);
    return __popc(row.mask(crosses)) & 1;
  }
};

// dtNavMesh::getPolyHeight; known_inside: (px, pz) is known to be inside the polygon.
BPSX_DEV bool poly_height_row(const Row& row, const NavData& nav, const PolyRec& r, float px, float py, float pz, bool known_inside,
                              float& h) {
  if (r.type != 0) return false;
  const int tc = r.tri_count;
  const uint32_t* tris = reinterpret_cast<const uint32_t*>(nav.dtris) + r.tri_base;   // four bytes per triangle
  uint32_t t = row.el < tc ? tris[row.el] : 0u;
  if (!known_inside) {
    RowEdge e;
    e.load(row, &r, r.nv);
    if (!e.inside(row, px, pz)) return false;
  }
  for (int j = row.el;; j += 8) {
    float mine = 0;
    const bool hit = j < tc && height_on_triangle(px, pz, detail_vert(nav, r, (int)(t & 0xffu)), detail_vert(nav, r, (int)((t >> 8) & 0xffu)),
                                                  detail_vert(nav, r, (int)((t >> 16) & 0xffu)), mine);
    const uint32_t m = row.mask(hit);
    if (m) { h = row.get(mine, __ffs((int)m) - 1); return true; }
    if (j - row.el + 8 >= tc) break;
    t = j + 8 < tc ? tris[j + 8] : 0u;
  }
  float c[3];
  closest_on_detail_edges<false>(nav, r, px, py, pz, c);
  h = c[1];
  return true;
}

// tryStep with sliding, a row per agent.  One lane per agent walked over six edges one after the other,
// with a search of the node pool in LDS for each neighbour: 51 of the 55 thousand cycles of a move
// kernel that lasts as long as its slowest lane.  Here a polygon's edges are looked at together, and a
// neighbour is looked up only if it is near enough to be entered, among the polygons that have
// been entered (`list`, 64 entries; the reference's nodes of the others are never read again).  The
// reference's limits, a pool of 64 nodes and 48 in the queue, cannot be met while the neighbours seen
// and the list stay below them; a move that could meet them (none of a step's 0.25 m in the measured
// scenes, most of several metres) is done again by the row's first lane as the reference does it.
// (50000 moves of up to half a metre over a cluttered plan: 132 -> 30 us.)
BPSX_DEV NavPt try_step_row(const Row& row, const NavData& nav, const SceneDev& s, const NavPt& start, float ex, float ey, float ez,
                            uint32_t* npolys, uint16_t* list, MoveLds& M, int column) {
  const uint32_t startIp = decode_ref(s, start.ref);
  if (startIp == kInvalidPoly || !finite3(start.x, start.y, start.z) || !finite3(ex, ey, ez)) return start;
  uint4* list4 = reinterpret_cast<uint4*>(list);
  constexpr uint32_t kUnused = 0xffffffffu;   // no polygon index: those have 15 bits
  list4[row.el] = make_uint4(row.el == 0 ? (kUnused << 16) | startIp : kUnused, kUnused, kUnused, kUnused);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  int entered = 1, head = 0, seen = 1;
  float bx = start.x, by = start.y, bz = start.z;
  float bestDist = 3.402823466e+38f;
  uint32_t bestIp = kInvalidPoly, visits = 0;
  bool reached = false, redo = false;
  const float sx = start.x + (ex - start.x) * 0.5f, sz = start.z + (ez - start.z) * 0.5f;
  const float ddx = ex - start.x, ddy = ey - start.y, ddz = ez - start.z;
  const float sr = sqrtf(ddx * ddx + ddy * ddy + ddz * ddz) / 2.0f + 0.001f;
  const float searchRadSqr = sr * sr;
  while (head < entered) {
    const uint32_t cur = list[head++];
    const PolyRec* r = &nav.polys[s.poly_base + cur];
    const int k = row.el < kNvp ? row.el : 0;
    const uint32_t nei = r->nei[k], walk = r->walk[k];
    RowEdge e;
    e.load(row, r, r->nv);
    visits++;
    if (e.inside(row, ex, ez)) {
      bestIp = cur;
      bx = ex; by = ey; bz = ez;
      reached = true;
      break;
    }
    // single-tile meshes carry no tile-border links, so a border edge is a wall
    const uint32_t nb = row.get((nei & 0x8000u) ? 0u : walk, e.from);
    const bool wall = e.on && !nb;
    float t;
    const float d = dist_pt_seg_sqr2d(wall ? ex : sx, wall ? ez : sz, e.j, e.i, t);
    // the nearest wall, the first of equal ones, if it is nearer than those before
    const uint32_t key = wall && d < bestDist ? __float_as_uint(d) : kUnused;
    const uint32_t nearest = Row::umin(key);
    if (nearest != kUnused) {
      const int w = __ffs((int)row.mask(key == nearest)) - 1;
      bx = row.get(e.j[0] + (e.i[0] - e.j[0]) * t, w);
      by = row.get(e.j[1] + (e.i[1] - e.j[1]) * t, w);
      bz = row.get(e.j[2] + (e.i[2] - e.j[2]) * t, w);
      bestDist = __uint_as_float(nearest);
      bestIp = cur;
    }
    seen += __popc(row.mask(e.on && nb));
    bool enter = e.on && nb && !(d > searchRadSqr);
    if (row.mask(enter)) {
      const uint32_t ip = nb - 1u;
      for (int q = 0; q * 8 < entered; ++q) {
        const uint4 l = list4[q];
        for (const uint32_t w : {l.x, l.y, l.z, l.w}) enter = enter && (w & 0xffffu) != ip && (w >> 16) != ip;
      }
      // two edges to one neighbour: the first enters it
      const uint32_t mine = enter ? ip : kUnused;
      static_for<1, kNvp>([&](auto K) BPSX_INLINE_LAMBDA {
        constexpr int k = decltype(K)::value;
        const uint32_t other = (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)mine, 0x110 + k /* row_shr */, 0xf, 0xf, false);
        enter = enter && !(row.el >= k && other == ip);
      });
      const uint32_t m = row.mask(enter);
      const int at = entered + __popc(m & ((1u << row.el) - 1u));
      if (enter && at < kTinyNodes) list[at] = (uint16_t)ip;
      entered += __popc(m);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    if (seen > kTinyNodes || entered - head > kMoveQueue) { redo = true; break; }
  }
  if (redo) {
    NavPt o = start;
    uint32_t n = 0;
    if (row.el == 0) o = try_step(nav, s, start, ex, ey, ez, &n, M, column);
    *npolys += row.get(n, 0);
    return NavPt{row.get(o.x, 0), row.get(o.y, 0), row.get(o.z, 0), row.get(o.ref, 0)};
  }
  *npolys += visits;
  if (bestIp == kInvalidPoly) return start;
  NavPt out{bx, by, bz, s.ref_base | bestIp};
  float h;
  if (isfinite(bx) && isfinite(bz) && poly_height_row(row, nav, nav.polys[s.poly_base + bestIp], bx, by, bz, reached, h)) out.y = h;
  return out;
}

// dtRandomPointInConvexPoly on a polygon record.
BPSX_DEV void random_point_in_poly(const PolyRec& r, float sv, float tv, float* out) {
  float areas[kNvp];
  float areasum = 0.0f;
  const int n = r.nv;
  for (int i = 2; i < n; i++) {
    const float abx = r.v[i - 1][0] - r.v[0][0], abz = r.v[i - 1][2] - r.v[0][2];
    const float acx = r.v[i][0] - r.v[0][0], acz = r.v[i][2] - r.v[0][2];
    areas[i] = acx * abz - abx * acz;
    areasum += areas[i] > 0.001f ? areas[i] : 0.001f;
  }
  const float thr = sv * areasum;
  float acc = 0.0f, u = 1.0f;
  int tri = n - 1;
  for (int i = 2; i < n; i++) {
    const float dacc = areas[i];
    if (thr >= acc && thr < (acc + dacc)) { u = (thr - acc) / dacc; tri = i; break; }
    acc += dacc;
  }
  const float v = sqrtf(tv);
  const float a = 1 - v, b = (1 - u) * v, c = u * v;
  const float* pa = r.v[0];
  const float* pb = r.v[tri - 1];
  const float* pc = r.v[tri];
  out[0] = a * pa[0] + b * pb[0] + c * pc[0];
  out[1] = a * pa[1] + b * pb[1] + c * pc[1];
  out[2] = a * pa[2] + b * pb[2] + c * pc[2];
}

// Area-weighted polygon pick + point by a row: first polygon whose inclusive area prefix sum exceeds
// u0 * total, then a point inside it, y from the height mesh.  The sums never fall, so eight pivots at
// once narrow the range to a ninth: five dependent reads among 20k polygons instead of fifteen.
BPSX_DEV bool sample_point_row(const Row& row, const NavData& nav, const SceneDev& s, float u0, float sv, float tv, float* out,
                               uint32_t* out_ip) {
  if (!(s.area_total > 0.0f)) return false;
  const float target = u0 * s.area_total;
  uint32_t lo = 0, hi = s.poly_count - 1;
  while (lo < hi) {
    const uint32_t step = (hi - lo + 8u) / 9u, at = lo + ((uint32_t)row.el + 1u) * step - 1u;
    const bool below = at < hi && !(nav.polys[s.poly_base + (at < hi ? at : hi)].area_cum > target);
    const uint32_t k = (uint32_t)__popc(row.mask(below));   // pivots 0 .. k - 1 lie before the polygon
    const uint32_t next = lo + (k + 1u) * step - 1u;
    lo = lo + k * step;
    hi = k < 8u && next < hi ? next : hi;
    lo = lo < hi ? lo : hi;
  }
  const PolyRec& r = nav.polys[s.poly_base + lo];
  random_point_in_poly(r, sv, tv, out);
  float h;
  if (isfinite(out[0]) && isfinite(out[2]) && poly_height_row(row, nav, r, out[0], out[1], out[2], false, h)) out[1] = h;
  *out_ip = lo;
  return true;
}

}  // namespace bpsx
