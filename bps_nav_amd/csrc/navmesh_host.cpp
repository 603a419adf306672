// Navmesh upload, host half.  Does what PathFinder::loadNavMesh does before the first query
// (PathFinder.cpp:330-408): read the MSET container, place the tile (dtNavMesh::init/addTile,
// DetourNavMesh.cpp:224-265, 908-1048), disable zero-area polygons (:276-328), label connected
// components (IslandSystem :53-170) — and writes the result as flat arrays for the GPU
// instead of Detour's pointer-linked tile.  Only single-tile meshes are accepted.
#include "navmesh_host.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <initializer_list>

#include "../../include/bpsx.h"
#include "dt_format.h"
#include "errors.h"

namespace bpsx {

namespace {

// The walkable leaves of the BV tree in the order of its array, then the bounds of every kSnapGroup of
// them, behind the nodes.  Testing each leaf finds what the in-order walk finds when no inner node
// hides a leaf from a box that the leaf overlaps, i.e. when every node lies within the bounds of the
// inner nodes around it; the builder's trees do, and where one does not the kernels walk it.  (The
// builder reserves 2N nodes and uses 2N - 1: the last is a zero leaf outside the tree, which the
// in-order walk visits, so it is among the leaves here.)
// snap_prune: a polygon's own extents quantise to within its leaf's bounds, the way the query's box is
// quantised, and so do its height samples up to kSnapOverhang; it has a boundary edge (without one
// the reference calls it 0 away from everywhere); and coordinates are small enough for kSnapSlack.
void append_snap_leaves(HostScene& s) {
  SceneDev& d = s.dev;
  d.snap_leaves = d.snap_prune = 0;
  const size_t n = s.bv.size();
  // quantised coordinates must neither wrap nor fall where coordinates grow
  bool prune = d.qfac > 0;
  for (int k = 0; k < 3; k += 2)
    prune = prune && std::fabs(d.bmin[k]) <= kSnapCoord && std::fabs(d.bmax[k]) <= kSnapCoord && d.bmin[k] <= d.bmax[k] &&
            d.qfac * (d.bmax[k] - d.bmin[k]) + 1 < 65535.0f;
  auto quantised = [&](float v, int k, float add) {
    const float c = v < d.bmin[k] ? d.bmin[k] : (v > d.bmax[k] ? d.bmax[k] : v);
    return (uint16_t)(int)(d.qfac * (c - d.bmin[k]) + add);
  };
  std::vector<bool> bounded(s.polys.size(), false);
  auto leaf_bounds = [&](const BVNodeDev& nd, const PolyRec& r) {
    float lo[3], hi[3];
    for (int k = 0; k < 3; ++k) lo[k] = hi[k] = r.v[0][k];
    bool finite = true;
    for (int i = 0; i < r.nv; ++i)
      for (int k = 0; k < 3; ++k) {
        finite &= std::fabs(r.v[i][k]) <= kSnapCoord;
        lo[k] = std::min(lo[k], r.v[i][k]);
        hi[k] = std::max(hi[k], r.v[i][k]);
      }
    if (!finite) return false;
    for (int i = 0; i < r.dvert_count; ++i)
      for (int k = 0; k < 3; ++k) {
        const float v = s.dverts[(size_t)(r.dvert_base + i) * 3 + k];
        if (!(std::fabs(v) <= kSnapCoord)) return false;
        if (k != 1 && !(v >= lo[k] - kSnapOverhang && v <= hi[k] + kSnapOverhang)) return false;
      }
    bool boundary = false;
    for (int j = 0; j < r.tri_count && !boundary; ++j) boundary = (s.dtris[(size_t)(r.tri_base + j) * 4 + 3] & 0x15) != 0;
    if (!boundary) return false;
    // (a further leaf of a polygon, like the zero leaf, never wins where the first one is looked at)
    if (bounded[nd.a]) return true;
    bounded[nd.a] = true;
    for (int k = 0; k < 3; k += 2)
      if (nd.bmax[k] < (quantised(hi[k], k, 0.0f) & 0xfffe) || nd.bmin[k] > (quantised(lo[k], k, 1.0f) | 1)) return false;
    return true;
  };
  auto within = [](const BVNodeDev& in, const BVNodeDev& out) {
    bool ok = true;
    for (int k = 0; k < 3; ++k) ok &= in.bmin[k] >= out.bmin[k] && in.bmax[k] <= out.bmax[k];
    return ok;
  };
  auto nodes_of = [&](size_t i) { return s.bv[i].b == kBVLeaf ? (size_t)1 : (size_t)s.bv[i].a; };
  std::vector<BVNodeDev> groups;
  size_t count = 0;
  for (size_t i = 0; i < n; ++i) {
    const BVNodeDev nd = s.bv[i];
    if (nd.b != kBVLeaf) {
      // two children that fill the node's range, each within its bounds
      const size_t left = i + 1, end = i + nd.a, right = left < n ? left + nodes_of(left) : n;
      if (right >= end || right >= n || right + nodes_of(right) != end || !within(s.bv[left], nd) || !within(s.bv[right], nd)) {
        s.bv.resize(n);
        return;
      }
      continue;
    }
    const PolyRec& r = s.polys[nd.a];
    if (!(r.flags & kPolyFlagWalk)) continue;
    s.bv.push_back(nd);
    if (count++ % kSnapGroup == 0) groups.push_back(nd);
    BVNodeDev& g = groups.back();
    for (int k = 0; k < 3; ++k) {
      g.bmin[k] = std::min(g.bmin[k], nd.bmin[k]);
      g.bmax[k] = std::max(g.bmax[k], nd.bmax[k]);
    }
    prune = prune && leaf_bounds(nd, r);
  }
  if (!count || count > 0xffff) { s.bv.resize(n); return; }
  s.bv.insert(s.bv.end(), groups.begin(), groups.end());
  d.snap_leaves = (uint32_t)count;
  d.snap_prune = prune ? 1u : 0u;
}

}  // namespace

int parse_navmesh(const uint8_t* b, size_t n, HostScene* out) {
  if (!b || !out) return fail(BPSX_E_INVAL, "navmesh: null argument");
  if (n < sizeof(MsetHeader)) return fail(BPSX_E_INVAL, "navmesh: truncated MSET header");
  MsetHeader mh;
  memcpy(&mh, b, sizeof(mh));
  if (mh.magic != kMsetMagic) return fail(BPSX_E_INVAL, "navmesh: bad MSET magic");
  if (mh.version != kMsetVersion) return fail(BPSX_E_INVAL, "navmesh: bad MSET version");
  if (mh.params.maxTiles < 1 || mh.params.maxPolys < 1) return fail(BPSX_E_INVAL, "navmesh: bad params");
  const uint32_t tileBits = ilog2(nextPow2((uint32_t)mh.params.maxTiles));
  const uint32_t polyBits = ilog2(nextPow2((uint32_t)mh.params.maxPolys));
  if (tileBits + polyBits > 22) return fail(BPSX_E_INVAL, "navmesh: params leave fewer than 10 salt bits");
  const uint32_t saltBits = std::min(31u, 32 - tileBits - polyBits);

  size_t off = sizeof(MsetHeader);
  const uint8_t* tileData = nullptr;
  MsetTileHeader th{};
  int tiles = 0;
  for (int t = 0; t < mh.numTiles; ++t) {
    if (off + sizeof(MsetTileHeader) > n) return fail(BPSX_E_INVAL, "navmesh: truncated tile header");
    MsetTileHeader cur;
    memcpy(&cur, b + off, sizeof(cur));
    off += sizeof(cur);
    if (!cur.tileRef || !cur.dataSize) break;
    if (cur.dataSize < (int)sizeof(TileHeader) || off + (size_t)cur.dataSize > n)
      return fail(BPSX_E_INVAL, "navmesh: truncated tile data");
    if (tiles == 0) { tileData = b + off; th = cur; }
    tiles++;
    off += (size_t)cur.dataSize;
  }
  if (tiles == 0) return fail(BPSX_E_INVAL, "navmesh: holds no tile");
  // The reference cannot load these either: PathFinder builds polygon refs with salt and tile
  // index swapped (PathFinder.cpp:67, 318), which only cancels out for a one-tile mesh.
  if (tiles > 1) return fail(BPSX_E_UNSUPPORTED, "navmesh: multi-tile meshes are not supported (nor by the reference's PathFinder)");

  TileHeader h;
  memcpy(&h, tileData, sizeof(h));
  if (h.magic != kTileMagic) return fail(BPSX_E_INVAL, "navmesh: bad tile magic");
  if (h.version != kTileVersion) return fail(BPSX_E_INVAL, "navmesh: bad tile version");
  if (h.offMeshConCount != 0) return fail(BPSX_E_UNSUPPORTED, "navmesh: off-mesh connections are not supported");
  if (h.polyCount < 1 || h.polyCount > 0x7fff || h.vertCount < 1 || h.detailMeshCount != h.polyCount ||
      h.maxLinkCount < 0 || h.detailVertCount < 0 || h.detailTriCount < 0 || h.bvNodeCount < 0)
    return fail(BPSX_E_INVAL, "navmesh: inconsistent tile header");
  if ((uint32_t)h.polyCount > (1u << polyBits)) return fail(BPSX_E_INVAL, "navmesh: polyCount exceeds maxPolys bits");
  // the device tree names its right children and leaves in 16 bits, 0xffff marks a leaf
  if (h.bvNodeCount > 0xfffe) return fail(BPSX_E_INVAL, "navmesh: more BV nodes than a tile of 32767 polygons can have");
  // no section can hold more elements than the tile has bytes: checked before the counts are
  // multiplied, and the sizes are computed in size_t
  const size_t tileBytes = (size_t)th.dataSize;
  for (const int count : {h.vertCount, h.polyCount, h.maxLinkCount, h.detailMeshCount, h.detailVertCount, h.detailTriCount,
                          h.bvNodeCount})
    if ((size_t)count > tileBytes) return fail(BPSX_E_INVAL, "navmesh: a section count exceeds the tile size");
  const size_t headerSize = align4(sizeof(TileHeader));
  const size_t vertsSize = align4((size_t)12 * (size_t)h.vertCount);
  const size_t polysSize = align4((size_t)32 * (size_t)h.polyCount);
  const size_t linksSize = align4((size_t)12 * (size_t)h.maxLinkCount);
  const size_t dmSize = align4((size_t)12 * (size_t)h.detailMeshCount);
  const size_t dvSize = align4((size_t)12 * (size_t)h.detailVertCount);
  const size_t dtSize = align4((size_t)4 * (size_t)h.detailTriCount);
  const size_t bvSize = align4((size_t)16 * (size_t)h.bvNodeCount);
  if (headerSize + vertsSize + polysSize + linksSize + dmSize + dvSize + dtSize + bvSize > (size_t)th.dataSize)
    return fail(BPSX_E_INVAL, "navmesh: tile sections exceed tile size");
  const float* verts = reinterpret_cast<const float*>(tileData + headerSize);
  const uint8_t* pp = tileData + headerSize + vertsSize;
  const uint8_t* dm = pp + polysSize + linksSize;
  const uint8_t* dv = dm + dmSize;
  const uint8_t* dt = dv + dvSize;
  const uint8_t* bvp = dt + dtSize;

  const uint32_t tileIndex = (th.tileRef >> polyBits) & ((1u << tileBits) - 1);
  const uint32_t salt = (th.tileRef >> (polyBits + tileBits)) & ((1u << saltBits) - 1);
  if (tileIndex >= (uint32_t)mh.params.maxTiles) return fail(BPSX_E_INVAL, "navmesh: tile index out of range");

  HostScene& s = *out;
  const int np = h.polyCount;
  s.polys.assign((size_t)np, PolyRec{});
  s.dverts.assign((const float*)dv, (const float*)dv + (size_t)h.detailVertCount * 3);
  s.dtris.assign(dt, dt + (size_t)h.detailTriCount * 4);
  std::vector<TilePoly> tp((size_t)np);
  memcpy(tp.data(), pp, (size_t)np * sizeof(TilePoly));
  std::vector<TilePolyDetail> td((size_t)np);
  memcpy(td.data(), dm, (size_t)np * sizeof(TilePolyDetail));

  for (int i = 0; i < np; ++i) {
    const TilePoly& p = tp[i];
    PolyRec& r = s.polys[i];
    if (p.vertCount < 3 || p.vertCount > kNvp) return fail(BPSX_E_INVAL, "navmesh: polygon vertex count out of range");
    r.nv = p.vertCount;
    r.type = p.areaAndType >> 6;
    if (r.type != 0) return fail(BPSX_E_UNSUPPORTED, "navmesh: off-mesh polygons are not supported");
    r.flags = p.flags;
    for (int k = 0; k < p.vertCount; ++k) {
      if (p.verts[k] >= h.vertCount) return fail(BPSX_E_INVAL, "navmesh: vertex index out of range");
      memcpy(r.v[k], &verts[(size_t)p.verts[k] * 3], 12);
      r.nei[k] = p.neis[k];
      if (p.neis[k] && !(p.neis[k] & kExtLink) && p.neis[k] - 1 >= np)
        return fail(BPSX_E_INVAL, "navmesh: neighbour index out of range");
    }
    const TilePolyDetail& d = td[i];
    if ((size_t)d.triBase + d.triCount > (size_t)h.detailTriCount ||
        (size_t)d.vertBase + d.vertCount > (size_t)h.detailVertCount)
      return fail(BPSX_E_INVAL, "navmesh: detail mesh out of range");
    for (int j = 0; j < d.triCount; ++j)
      for (int k = 0; k < 3; ++k)
        if (s.dtris[(size_t)(d.triBase + j) * 4 + k] >= p.vertCount + d.vertCount)
          return fail(BPSX_E_INVAL, "navmesh: detail triangle vertex out of range");
    r.tri_base = d.triBase;
    r.dvert_base = d.vertBase;
    r.tri_count = d.triCount;
    r.dvert_count = d.vertCount;
  }

  // removeZeroAreaPolys: 3-D area of the detail triangles, accumulated the way the
  // reference's mixed float/double expression does.
  for (int i = 0; i < np; ++i) {
    PolyRec& r = s.polys[i];
    float area = 0;
    for (int j = 0; j < r.tri_count; ++j) {
      const uint8_t* t = &s.dtris[(size_t)(r.tri_base + j) * 4];
      const float* v[3];
      for (int k = 0; k < 3; ++k)
        v[k] = t[k] < r.nv ? r.v[t[k]] : &s.dverts[(size_t)(r.dvert_base + (t[k] - r.nv)) * 3];
      float w1[3], w2[3];
      for (int k = 0; k < 3; ++k) { w1[k] = v[1][k] - v[0][k]; w2[k] = v[2][k] - v[0][k]; }
      const float cx = w1[1] * w2[2] - w1[2] * w2[1];
      const float cy = w1[2] * w2[0] - w1[0] * w2[2];
      const float cz = w1[0] * w2[1] - w1[1] * w2[0];
      const float norm = sqrtf(cx * cx + (cy * cy + cz * cz));
      area = (float)((double)area + 0.5 * (double)norm);
    }
    if ((double)area < 1e-5) r.flags = kPolyFlagDisabled;
  }
  // What depends on which polygons pass the query filter (include WALK, exclude nothing), polygon by
  // polygon: the neighbours that do; the per-edge records of the path search; the prefix sums of the fan
  // areas that findRandomPoint weighs polygons by
  s.aedges.reserve((size_t)np * kEdgeStride);
  float acc = 0.0f;
  for (int i = 0; i < np; ++i) {
    PolyRec& r = s.polys[i];
    AEdge e[kEdgeStride];
    for (AEdge& x : e) x = AEdge{{0, 0, 0}, kNoNb};
    for (int k = 0; k < r.nv; ++k) {
      const uint16_t ne = r.nei[k];
      r.walk[k] = (ne && !(ne & kExtLink) && (s.polys[ne - 1].flags & kPolyFlagWalk)) ? ne : 0;
      const float* l = r.v[k];
      const float* rt = r.v[k + 1 < r.nv ? k + 1 : 0];
      for (int c = 0; c < 3; ++c) {
        const float mid = (l[c] + rt[c]) * 0.5f;
        e[k].mid[c] = std::isfinite(mid) ? mid : kFarMid;
      }
      if (!r.walk[k]) continue;
      // a polygon behind two edges: expanding through the second never changes its node (same
      // position, not a lower cost), so only the first edge leads there
      bool first = true;
      for (int j = 0; j < k; ++j) first &= r.walk[j] != r.walk[k];
      if (first) e[k].nb = (uint32_t)(r.walk[k] - 1);
    }
    s.aedges.insert(s.aedges.end(), e, e + kEdgeStride);
    if (r.type == 0 && (r.flags & kPolyFlagWalk)) {
      float a = 0.0f;
      for (int j = 2; j < r.nv; ++j) {
        const float abx = r.v[j - 1][0] - r.v[0][0], abz = r.v[j - 1][2] - r.v[0][2];
        const float acx = r.v[j][0] - r.v[0][0], acz = r.v[j][2] - r.v[0][2];
        a += acx * abz - abx * acz;
      }
      if (a > 0.0f) acc += a;
    }
    r.area_cum = acc;
  }
  // connected components: polygons are seeded in index order, the seed is not filter-checked,
  // neighbours are entered in ascending edge order and popped last-in first-out
  {
    constexpr uint32_t kUnlabelled = 0xffffffffu;
    for (PolyRec& r : s.polys) r.island = kUnlabelled;
    std::vector<uint16_t> stack((size_t)np);   // a polygon is entered once
    uint32_t next = 0;
    for (int sd = 0; sd < np; ++sd) {
      if (s.polys[sd].island != kUnlabelled) continue;
      const uint32_t id = next++;
      s.polys[sd].island = id;
      size_t top = 0;
      stack[top++] = (uint16_t)sd;
      while (top) {
        const PolyRec& r = s.polys[stack[--top]];
        for (int k = 0; k < r.nv; ++k) {
          if (!r.walk[k]) continue;
          PolyRec& to = s.polys[r.walk[k] - 1];
          if (to.island != kUnlabelled) continue;
          to.island = id;
          stack[top++] = (uint16_t)(r.walk[k] - 1);
        }
      }
    }
  }

  // BV tree: repack dtBVNode (bounds + int) into BVNodeDev.  Leaves must name valid polygons.
  s.bv.reserve((size_t)h.bvNodeCount + (size_t)h.bvNodeCount / 2 + (size_t)h.bvNodeCount / (2 * kSnapGroup) + 2);   // and its leaves
  s.bv.resize((size_t)h.bvNodeCount);
  for (size_t i = 0; i < s.bv.size(); ++i) {
    TileBVNode r;
    memcpy(&r, bvp + i * sizeof(r), sizeof(r));
    BVNodeDev& o = s.bv[i];
    memcpy(o.bmin, r.bmin, 6);
    memcpy(o.bmax, r.bmax, 6);
    if (r.i >= 0) {
      if (r.i >= np) return fail(BPSX_E_INVAL, "navmesh: BV leaf out of range");
      o.a = (uint16_t)r.i;
      o.b = kBVLeaf;
    } else {
      const int64_t e = -(int64_t)r.i;
      if (e < 1 || e > 0xfffe) return fail(BPSX_E_INVAL, "navmesh: BV escape offset out of range");
      o.a = (uint16_t)e;
      o.b = 0;
    }
  }

  SceneDev& d = s.dev;
  d.poly_count = (uint32_t)np;
  d.bv_count = (uint32_t)h.bvNodeCount;
  d.ref_base = (salt << (polyBits + tileBits)) | (tileIndex << polyBits);
  d.poly_mask = (1u << polyBits) - 1;
  memcpy(d.orig, mh.params.orig, 12);
  d.tile_w = mh.params.tileWidth;
  d.tile_h = mh.params.tileHeight;
  d.tx = h.x;
  d.ty = h.y;
  memcpy(d.bmin, h.bmin, 12);
  memcpy(d.bmax, h.bmax, 12);
  d.qfac = h.bvQuantFactor;
  d.climb = h.walkableClimb;
  d.area_total = acc;
  append_snap_leaves(s);
  return BPSX_OK;
}

}  // namespace bpsx
