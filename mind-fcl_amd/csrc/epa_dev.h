// Device EPA (include/fcl/cvx_collide/epa.hpp, epa_polytope*.hpp,
// epa_simplex2polytope.hpp, epa_polytope_utils.h).
//
// GPU representation: one wavefront per pair; the polytope lives in that
// wavefront's LDS slice as slot arrays of vertices, edges and faces (16-bit
// indices, FP64 geometry), visited by the 64 lanes in parallel; creation
// stamps stand in for the reference's newest-first element lists.
//
// The loop is a chain of one pair's dependent steps; three wavefronts a SIMD
// (epaQueueKernel) keep the vector units 66 % busy, the few long pairs of the
// full-capacity pass 5 %.  What a step keeps between its phases lives in LDS
// and the support search is one out-of-line function (wave_dev.h), so that no
// value of the loop spills: the kernels' scratch (208 bytes a lane in
// epaQueueKernel, 64 in the full-capacity pass) holds the registers that the
// out-of-line functions save at their entry.  GJK in waveKernel, in front of
// it, has 54 spills (400 bytes a lane) to stay at three wavefronts a SIMD.
#pragma once

#include <type_traits>

#include "wave_dev.h"

namespace mfcl {

constexpr int16_t kNil = -1;

// A condition that every lane of the wavefront evaluates on identical
// values (the polytope code runs one pair per wavefront in lock step), taken
// as a scalar so that the branch on it is a scalar branch.
MFCL_D bool ub(bool c) { return __builtin_amdgcn_readfirstlane(c ? 1 : 0) != 0; }

struct EVertCore {
  double vx, vy, vz;  // vertex on the Minkowski difference
  double dx, dy, dz;  // direction that produced it
  int32_t h0, h1;     // the support vertices of the two hulls (-1: primitive or unknown)
  int32_t stamp;      // creation order; < 0: free slot
  int16_t new_edge;
  uint8_t remove, pad0;
};
struct EEdgeCore {
  double d2, wx, wy, wz;  // squared distance to origin, witness
  int32_t stamp;
  int16_t v0, v1, f0, f1;
  uint8_t in, vis;
  uint16_t pad0;
};
struct EFaceCore {
  double d2, wx, wy, wz;
  int32_t stamp;
  int16_t e0, e1, e2;
  uint8_t in, vis;
  int16_t a;     // the first edge's first vertex
  uint8_t cls;   // NormalClass (kNormals polytopes)
  uint8_t pad0;
};
// A face with its outward unit normal, which does not change while the face
// lives -- unless the origin lies close to its plane: then n is the plane's
// normal of either sign, and the side is decided by the vertices of the
// moment.
enum NormalClass : uint8_t { kNormalOut = 0, kNormalClose = 1, kNormalNone = 2 };
struct EFaceNormal : EFaceCore {
  double nx, ny, nz;
};
// PAD: records of an odd number of 8-byte words, so that the 64 lanes'
// accesses to one field of consecutive slots spread over the LDS banks
// (64- and 48-byte records put every fourth slot on the same bank).
template <class R, bool PAD>
struct Rec : R {};
template <class R>
struct Rec<R, true> : R {
  int32_t spread[2];
};
static_assert(sizeof(Rec<EVertCore, true>) == 72 && sizeof(Rec<EEdgeCore, true>) == 56 &&
                  sizeof(Rec<EVertCore, false>) == 64 && sizeof(EFaceCore) == 48 && sizeof(EFaceNormal) == 72,
              "record sizes");

// Where a polytope's slot arrays live and how an expansion marks its faces:
// kWords 64-bit masks (64 kWords faces at most, kWords faces per lane; the
// faces keep their normals), or, with 0, marks in the records.  Small: the
// wavefront's share of a block's LDS.  Mid and Large: LDS at the request's
// full capacity, up to 256 faces and beyond.  Global: device memory, a
// capacity beyond the LDS.  sync() orders one lane's writes
// before other lanes' reads of the same wavefront: LDS executes a
// wavefront's operations in order, so a compiler barrier suffices there;
// device memory needs a workgroup-scope fence.
template <int WORDS>
struct MaskMem {
  static constexpr int kWords = WORDS;
  static constexpr bool kPad = true;
  using Face = EFaceNormal;
  template <class T>
  using P = MFCL_LDS T*;
  static MFCL_D void sync() { __builtin_amdgcn_wave_barrier(); }
};
using SmallMem = MaskMem<1>;
using MidMem = MaskMem<4>;
struct LargeMem {
  static constexpr int kWords = 0;
  static constexpr bool kPad = false;
  using Face = EFaceCore;
  template <class T>
  using P = MFCL_LDS T*;
  static MFCL_D void sync() { __builtin_amdgcn_wave_barrier(); }
};
struct GlobalMem {
  static constexpr int kWords = 0;
  static constexpr bool kPad = false;
  using Face = EFaceCore;
  template <class T>
  using P = T*;
  static MFCL_D void sync() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup"); }
};
constexpr int kSmallFaces = 64, kMidFaces = 256;

// Arena sizing for a given face capacity: vertices = edges = floor(1.51 F)
// (epa_polytope.hpp:90-95).
struct ArenaDims {
  int nv, nf;
};
__host__ __device__ inline ArenaDims arenaDims(int max_faces) {
  ArenaDims d;
  d.nv = static_cast<int>(1.51 * static_cast<double>(max_faces));
  d.nf = max_faces;
  return d;
}
// Scratch record per border edge of one expansion (see coverBorder).
struct BorderRec {
  int16_t pre;     // elements (edges and faces) created before this edge's face
  int16_t e, rank; // edge slot, rank in descending stamp order
  int16_t fe, ff;  // the list of free edge / face slots (entry k: the k-th free slot)
  int8_t t0, t1;   // lower-ranked border edges sharing endpoint v0 / v1
};
template <class M>
__host__ __device__ inline size_t polyBytes(int max_faces) {
  const ArenaDims d = arenaDims(max_faces);
  return (sizeof(Rec<EVertCore, M::kPad>) + sizeof(Rec<EEdgeCore, M::kPad>)) * d.nv +
         sizeof(typename M::Face) * d.nf;
}
template <class M>
__host__ __device__ inline size_t arenaBytes(int max_faces) {
  const size_t b = polyBytes<M>(max_faces) + sizeof(BorderRec) * arenaDims(max_faces).nv;
  return (b + 255) & ~static_cast<size_t>(255);
}

enum EVis : uint8_t { kUnknown = 0, kBorder = 1, kInternal = 2 };
enum FVis : uint8_t { kFUnknown = 0, kVisible = 1, kHidden = 2 };
enum EpaStatus : int { kEpaFailed = 0, kEpaOK = 1, kEpaTouching = 2, kEpaIterLimit = 3, kEpaMallocFailed = 4 };

struct MinD {
  bool in;
  double d2;
  d3 w;
};

// epa_polytope_utils.h:19-52
MFCL_D void segDist(d3 p, d3 x0, d3 x1, MinD& o) {
  const d3 d = x1 - x0;
  const d3 a = x0 - p;
  const double l2 = sqnorm(d);
  const double t = -1.0 * dot(a, d) / l2;
  if (t <= 0.0) {
    o.w = x0;
    o.in = false;
    o.d2 = sqnorm(x0 - p);
  } else if (t >= 1.0) {
    o.w = x1;
    o.in = false;
    o.d2 = sqnorm(x1 - p);
  } else {
    o.w = x0 + t * d;
    o.in = true;
    o.d2 = sqnorm(o.w);
  }
}
MFCL_D double lineDist(d3 p, d3 a, d3 b) {
  const d3 ab = b - a;
  const double l = norm(ab);
  if (l <= 0.0) return norm(p - a);
  return norm(cross(p - a, ab)) / l;
}
MFCL_D double planeDist(d3 p, d3 a, d3 b, d3 c) {
  const d3 n = cross(a - b, b - c);
  const double l = norm(n);
  if (l <= 0.0) return lineDist(p, a, b);
  return fabs(dot(n / l, a - p));
}
// epa_polytope_utils.h:92-166 with p = origin.
MFCL_D void triDist0(d3 a, d3 b, d3 c, MinD& o) {
  const d3 dl0 = a - b, dl1 = b - c, dl2 = c - a;
  const d3 n = cross(dl0, dl1);
  const double n2 = sqnorm(n);
  const double area = sqrt(n2);
  bool sub = fabs(area) <= 1e-16;
  if (!sub) {
    const d3 proj = n * (dot(a, n) / n2);  // p + n * ((a - p).n / n2) with p = 0
    const double w0 = norm(cross(dl1, b - proj)) / area;
    const double w1 = norm(cross(dl2, c - proj)) / area;
    const double w2 = 1.0 - w0 - w1;
    bool in = !(w0 < 0.0 || w0 > 1.0) && !(w1 < 0.0 || w1 > 1.0) && !(w2 < 0.0 || w2 > 1.0);
    const double chk = norm(cross(dl0, a - proj)) / area;
    if (fabs(chk - w2) > 1e-3) in = false;
    if (in) {
      o.in = true;
      o.d2 = sqnorm(proj);
      o.w = a * w0 + b * w1 + c * w2;
      return;
    }
    sub = true;
  }
  const d3 z = {0, 0, 0};
  MinD s0, s1, s2;
  segDist(z, a, b, s0);
  segDist(z, b, c, s1);
  segDist(z, c, a, s2);
  MinD best = s0;
  if (s1.d2 < best.d2) best = s1;
  if (s2.d2 < best.d2) best = s2;
  o.in = false;
  o.d2 = best.d2;
  o.w = best.w;
}

// The polytope, processed by the 64 lanes of one wavefront together.
// Elements live in fixed slot arrays (slot s is visited by lane s % 64);
// a slot is free when its stamp is negative.  Every element gets a creation
// stamp from one counter, and the reference's element lists are
// newest-first (epa_polytope.hpp:127-290), so "earlier in the list" is
// "larger stamp": scans that the reference runs sequentially over its lists
// run here as parallel passes plus wavefront reductions ordered by stamp,
// which reproduces its tie-breaking exactly.  Slot numbers themselves never
// influence a result.  Every member function must be called by all 64 lanes
// with identical arguments.
template <class M>
struct PolyT {
  using EVert = Rec<EVertCore, M::kPad>;
  using EEdge = Rec<EEdgeCore, M::kPad>;
  using EFace = typename M::Face;
  using Base = typename M::template P<char>;
  typename M::template P<EVert> V;
  typename M::template P<EEdge> E;
  typename M::template P<EFace> F;
  typename M::template P<BorderRec> BL;  // nv records
  int nv, nf;   // slot capacities: vertices and edges nv, faces nf
  // slots in use lie below these (the lowest free ones are taken first);
  // those beyond are free and not initialised
  int hv, he, hf;
  int stamp;    // creation counter

  MFCL_D PolyT(Base base, int cap_faces) {
    const ArenaDims d = arenaDims(cap_faces);
    V = (typename M::template P<EVert>)(base);
    E = (typename M::template P<EEdge>)(base + sizeof(EVert) * d.nv);
    F = (typename M::template P<EFace>)(base + (sizeof(EVert) + sizeof(EEdge)) * d.nv);
    BL = (typename M::template P<BorderRec>)(base + (sizeof(EVert) + sizeof(EEdge)) * d.nv + sizeof(EFace) * d.nf);
    nv = d.nv;
    nf = d.nf;
    hv = he = hf = stamp = 0;
  }
  MFCL_D d3 vloc(int i) const { return {V[i].vx, V[i].vy, V[i].vz}; }

  // the initial polytope: vertices V[0 .. n_v) (written by the caller),
  // edges and faces from 4-bit tables (entry k at bits 4 k); stamps in the
  // order vertices, edges, faces; an edge's first face is its f0, the second
  // its f1.  false: it does not fit.
  MFCL_D bool build(int n_v, int n_e, int n_f, uint64_t v0, uint64_t v1, uint64_t e0, uint64_t e1, uint64_t e2) {
    const int l = __lane_id();
    if (n_v > nv || n_e > nv || n_f > nf) return false;
    if (l < n_v) V[l].stamp = l;
    hv = n_v;
    he = n_e;
    hf = n_f;
    auto nib = [](uint64_t t, int k) { return static_cast<int16_t>((t >> (4 * k)) & 15u); };
    if (l < n_e) {
      auto& e = E[l];
      e.v0 = nib(v0, l);
      e.v1 = nib(v1, l);
      int16_t f0 = kNil, f1 = kNil;
      for (int k = 0; k < n_f; ++k)
        if (nib(e0, k) == l || nib(e1, k) == l || nib(e2, k) == l) {
          if (f0 == kNil) f0 = static_cast<int16_t>(k);
          else f1 = static_cast<int16_t>(k);
        }
      e.f0 = f0;
      e.f1 = f1;
      MinD m;
      segDist(d3{0, 0, 0}, vloc(e.v0), vloc(e.v1), m);
      e.in = m.in; e.d2 = m.d2; e.wx = m.w.x; e.wy = m.w.y; e.wz = m.w.z;
      e.stamp = n_v + l;
    }
    M::sync();
    if (l < n_f) {
      auto& f = F[l];
      f.e0 = nib(e0, l); f.e1 = nib(e1, l); f.e2 = nib(e2, l);
      int16_t a, b, c;
      faceVerts(l, a, b, c);
      setFace(f, a, vloc(a), vloc(b), vloc(c));
      f.stamp = n_v + n_e + l;
    }
    stamp = n_v + n_e + n_f;
    M::sync();
    return true;
  }
  MFCL_D void faceVerts(int fi, int16_t& a, int16_t& b, int16_t& c) const {
    const auto& f = F[fi];
    a = E[f.e0].v0;
    b = E[f.e0].v1;
    const int16_t p = E[f.e1].v0, q = E[f.e1].v1;
    c = (p != a && p != b) ? p : q;
  }

  // A new face's distance record and, where faces keep it, its normal
  // (epa_polytope.hpp:347-405: outward when the origin is at least 1e-4 from
  // the plane).  a, b, c in faceVerts' order.
  template <class FR>
  MFCL_D void setFace(FR& f, int ia, d3 a, d3 b, d3 c) const {
    MinD m;
    triDist0(a, b, c, m);
    f.in = m.in; f.d2 = m.d2; f.wx = m.w.x; f.wy = m.w.y; f.wz = m.w.z;
    f.a = static_cast<int16_t>(ia);
    if constexpr (M::kWords > 0) {
      const d3 n = cross(a - b, b - c);
      const double nn = norm(n);
      const d3 dir = n / nn;
      const double od = dot(a, dir);
      const bool close = !(fabs(od) >= 1e-4);
      const d3 out = close || od > 0 ? dir : -dir;
      f.cls = nn <= 0.0 ? kNormalNone : (close ? kNormalClose : kNormalOut);
      f.nx = out.x; f.ny = out.y; f.nz = out.z;
    }
  }
  // Whether a plane near the origin has its outward side against dir (the
  // same in all lanes): away from the farther vertices.  max / min over the
  // vertices: order-free, so a parallel pass.
  MFCL_D bool closeFlips(d3 dir) const {
    double maxp = 0.0, minn = 0.0;
    for (int s = __lane_id(); s < hv; s += 64) {
      if (V[s].stamp < 0) continue;
      const double dv = dot(vloc(s), dir);
      if (dv > maxp) maxp = dv;
      if (dv < minn) minn = dv;
    }
#pragma nounroll
    for (int off = 32; off > 0; off >>= 1) {
      const double om = __shfl_xor(maxp, off), on = __shfl_xor(minn, off);
      if (om > maxp) maxp = om;
      if (on < minn) minn = on;
    }
    return ub(fabs(maxp) > fabs(minn));
  }

  // Better in the order (d2, kind, newest first) -- the first element of
  // the reference's vertex, edge, face scans with strict '<'.  rank: kind
  // and age, smaller first.
  MFCL_D static bool better(double d2, uint32_t rank, double bd, uint32_t br) {
    return d2 < bd || (d2 == bd && rank < br);
  }
  MFCL_D static uint32_t rankOf(int kind, int st) {
    return (static_cast<uint32_t>(kind) << 28) | (0x0FFFFFFFu - static_cast<uint32_t>(st));
  }
  // epa_polytope.hpp:292-345; kind: 0 none, 1 vertex, 2 edge, 3 face
  MFCL_D void minToOrigin(bool excl_vertex, int& kind, int& idx) const {
    const int l = __lane_id();
    double bd = INFINITY;
    uint32_t br = 0xFFFFFFFFu;
    int bi = kNil;
    if (!excl_vertex)
#pragma nounroll
      for (int s = l; s < hv; s += 64) {
        const int st = V[s].stamp;
        const double d2 = sqnorm(vloc(s));
        const uint32_t r = rankOf(1, st);
        if (st >= 0 && better(d2, r, bd, br)) { bd = d2; br = r; bi = s; }
      }
#pragma nounroll
    for (int s = l; s < he; s += 64) {
      const auto& e = E[s];
      const int st = e.stamp;
      const double d2 = e.d2;
      const uint32_t r = rankOf(2, st);
      if (st >= 0 && (excl_vertex || e.in) && better(d2, r, bd, br)) { bd = d2; br = r; bi = s; }
    }
#pragma nounroll
    for (int s = l; s < hf; s += 64) {
      const auto& f = F[s];
      const int st = f.stamp;
      const double d2 = f.d2;
      const uint32_t r = rankOf(3, st);
      if (st >= 0 && f.in && better(d2, r, bd, br)) { bd = d2; br = r; bi = s; }
    }
    // the smallest d2 over the wavefront, then the first rank among the
    // lanes that hold it (usually one)
    double m = -max8(-bd);
    m = fmin(m, dppD<kDppMirror>(m));
    m = fmin(fmin(readLaneF64(m, 0), readLaneF64(m, 16)), fmin(readLaneF64(m, 32), readLaneF64(m, 48)));
    unsigned long long who = __ballot(bd == m && br != 0xFFFFFFFFu);
    // only finite candidates beat the reference's initial INFINITY
    if (who == 0ull || !ub(m < INFINITY)) {
      kind = 0;
      idx = kNil;
      return;
    }
    int w = __builtin_ctzll(who);
    uint32_t r = __builtin_amdgcn_readlane(br, w);
    for (who &= who - 1; who; who &= who - 1) {
      const int o = __builtin_ctzll(who);
      const uint32_t ro = __builtin_amdgcn_readlane(br, o);
      if (ro < r) {
        r = ro;
        w = o;
      }
    }
    kind = static_cast<int>(r >> 28);
    idx = __builtin_amdgcn_readlane(bi, w);
  }

  // epa_polytope.hpp:347-405: a face's outward normal; ok: the face is not
  // degenerate (area > 0).
  struct Normal {
    d3 n;
    bool ok;
  };
  MFCL_D Normal normalOut(int fi) const {
    Normal r;
    int cls;
    if constexpr (M::kWords > 0) {
      const auto& f = F[fi];
      r.n = d3{f.nx, f.ny, f.nz};
      cls = f.cls;
    } else {
      int16_t ia, ib, ic;
      faceVerts(fi, ia, ib, ic);
      const d3 a = vloc(ia), b = vloc(ib), c = vloc(ic);
      const d3 n = cross(a - b, b - c);
      const double nn = norm(n);
      const d3 dir = n / nn;
      const double od = dot(a, dir);
      const bool close = !(fabs(od) >= 1e-4);
      r.n = close || od > 0 ? dir : -dir;
      cls = nn <= 0.0 ? kNormalNone : (close ? kNormalClose : kNormalOut);
    }
    cls = __builtin_amdgcn_readfirstlane(cls);
    r.ok = cls != kNormalNone;
    if (cls == kNormalClose && closeFlips(r.n)) r.n = -r.n;
    return r;
  }
  MFCL_D d3 faceAnchor(int fi) const { return vloc(F[fi].a); }
  MFCL_D bool anyLane(bool b) const { return __ballot(b) != 0ull; }

  // Slot of the new vertex (the lowest free one), kNil when there is none.
  MFCL_D int addVertex(d3 v, d3 d, int h0, int h1) {
    const int l = __lane_id();
    int i = kNil;
    for (int base = 0; base < hv && i == kNil; base += 64) {
      const int s = base + l;
      const unsigned long long m = __ballot(s < hv && V[s].stamp < 0);
      if (m) i = base + __builtin_ctzll(m);
    }
    if (i == kNil) {
      if (hv >= nv) return kNil;
      i = hv++;
    }
    auto& x = V[i];
    x.vx = v.x; x.vy = v.y; x.vz = v.z;
    x.dx = d.x; x.dy = d.y; x.dz = d.z;
    x.h0 = h0; x.h1 = h1;
    x.stamp = stamp++;
    M::sync();
    return i;
  }

  // Whether face fi sees p (epa_polytope_expand.hpp:12-30), evaluated by
  // one lane for its own face; the vertex fallback of the normal is scanned
  // by that lane alone.
  MFCL_D bool outsideLane(int fi, d3 p) const {
    int16_t ia, ib, ic;
    faceVerts(fi, ia, ib, ic);
    const d3 a = vloc(ia), b = vloc(ib), c = vloc(ic);
    const d3 n = cross(a - b, b - c);
    const double nn = norm(n);
    if (nn <= 0.0) return true;
    const d3 dir = n / nn;
    const double od = dot(a, dir);
    d3 normal;
    if (fabs(od) >= 1e-4) {
      normal = od > 0 ? dir : -dir;
    } else {
      double maxp = 0.0, minn = 0.0;
#pragma nounroll
      for (int s = 0; s < hv; ++s) {
        if (V[s].stamp < 0) continue;
        const double dv = dot(vloc(s), dir);
        if (dv > maxp) maxp = dv;
        if (dv < minn) minn = dv;
      }
      normal = fabs(maxp) > fabs(minn) ? -dir : dir;
    }
    return dot(normal, p - a) >= 0.0;
  }

  // epa_polytope_expand.hpp:32-281. 0 ok, 1 failed, 2 malloc failed,
  // 3 (only when may_spill) this polytope's capacity might not hold the
  // expansion -- nothing has been changed then, and the caller continues
  // in a polytope of the full capacity.
  // The reference's depth-first flood fill marks the faces reachable from
  // `start` through faces that see nv; that set, and the border / internal
  // edge marks, do not depend on the visiting order.  kWords faces per lane,
  // the visible set as bit masks: every face's test of nv runs first, all at
  // once (with the normals that the faces keep, a dot product); the fill's
  // rounds are then a few scalar instructions each.
  // One word: the mask itself; more: a flag per face (a lookup in several
  // words costs more instructions than the LDS read).
  MFCL_D bool isVisible(unsigned long long mask, int k) const {
    if (k == kNil) return false;
    if constexpr (M::kWords == 1) return ((mask >> (k & 63)) & 1ull) != 0;
    else return F[k].vis == kVisible;
  }
  MFCL_D int expandMask(d3 nv_, d3 nd, int nh0, int nh1, int start, bool may_spill) {
    constexpr int W = M::kWords;
    const int l = __lane_id();
    const unsigned long long below = (1ull << l) - 1;
    bool live[W], out[W], open[W];
    int g[W][3];
#pragma unroll
    for (int i = 0; i < W; ++i) {
      const int s = 64 * i + l;
      live[i] = out[i] = open[i] = false;
      g[i][0] = g[i][1] = g[i][2] = kNil;
      if (64 * i >= hf) continue;
      live[i] = s < hf && F[s < hf ? s : 0].stamp >= 0;
      int cls = kNormalOut;
      d3 n = {0, 0, 0}, a = {0, 0, 0};
      if (live[i]) {
        auto& f = F[s];
        const int es[3] = {f.e0, f.e1, f.e2};
        n = d3{f.nx, f.ny, f.nz};
        cls = f.cls;
        a = vloc(f.a);
        if (W > 1) f.vis = kFUnknown;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const int x = E[es[k]].f0, y = E[es[k]].f1;
          g[i][k] = x == s ? y : x;
          open[i] = open[i] || g[i][k] == kNil;
        }
      }
      for (unsigned long long m = __ballot(live[i] && cls == kNormalClose); m; m &= m - 1) {
        const int w = __builtin_ctzll(m);
        const bool flip = closeFlips(d3{readLaneF64(n.x, w), readLaneF64(n.y, w), readLaneF64(n.z, w)});
        if (l == w && flip) n = -n;
      }
      // epa_polytope_expand.hpp:12-30
      out[i] = live[i] && (cls == kNormalNone || dot(n, nv_ - a) >= 0.0);
    }
    unsigned long long vis = 1ull << (start & 63);
    bool mine[W];
    if constexpr (W == 1) {
      while (true) {
        const unsigned long long more =
            __ballot(out[0] && (isVisible(vis, g[0][0]) || isVisible(vis, g[0][1]) || isVisible(vis, g[0][2]))) & ~vis;
        if (!more) break;
        vis |= more;
      }
      mine[0] = live[0] && ((vis >> l) & 1ull) != 0;
    } else {
      M::sync();
      F[start].vis = kVisible;
      M::sync();
#pragma unroll
      for (int i = 0; i < W; ++i) mine[i] = 64 * i + l == start;
      while (true) {
        bool grew = false;
#pragma unroll
        for (int i = 0; i < W; ++i) {
          if (64 * i >= hf) continue;
          if (out[i] && !mine[i] && (isVisible(0, g[i][0]) || isVisible(0, g[i][1]) || isVisible(0, g[i][2]))) {
            mine[i] = grew = true;
            F[64 * i + l].vis = kVisible;
          }
        }
        M::sync();
        if (!anyLane(grew)) break;
      }
    }
    bool bad = false;
    int below_f = 0;  // free face slots below hf, those of the visible faces included
#pragma unroll
    for (int i = 0; i < W; ++i) {
      bad = bad || (mine[i] && open[i]);
      if (64 * i < hf) below_f += __popcll(__ballot(64 * i + l < hf && (!live[i] || mine[i])));
    }
    // an open edge on a visible face is a malformed polytope
    if (anyLane(bad)) return 1;
    // edge marks from the face classes; border edges compacted into BL
    int nb = 0, below_e = 0, free_v = nv - hv;
    for (int base = 0; base < he; base += 64) {
      const int s = base + l;
      bool border = false, fr = false;
      if (s < he) {
        auto& e = E[s];
        const bool alive = e.stamp >= 0;
        const bool a = alive && isVisible(vis, e.f0), b = alive && isVisible(vis, e.f1);
        border = a != b;
        fr = !alive || (a && b);
        e.vis = border ? kBorder : (a ? kInternal : kUnknown);
      }
      const unsigned long long m = __ballot(border);
      if (border) BL[nb + __popcll(m & below)].e = static_cast<int16_t>(s);
      nb += __popcll(m);
      below_e += __popcll(__ballot(fr));
    }
    for (int base = 0; base < hv; base += 64) {
      const int s = base + l;
      if (s < hv) V[s].remove = 1;
      free_v += __popcll(__ballot(s < hv && V[s < hv ? s : 0].stamp < 0));
    }
    const int free_e = below_e + nv - he, free_f = below_f + nf - hf;
    // Whether the expansion certainly fits: one vertex, at most two new
    // edges per border edge and one face per border edge must find slots.
    // Vertices that the expansion removes are not counted as free.
    if (may_spill && !(free_v >= 1 && free_e >= 2 * nb && free_f >= nb)) return 3;
    M::sync();
    // drop the visible faces (detaching them from their border edges), the
    // internal edges and the vertices left without a non-internal edge
#pragma unroll
    for (int i = 0; i < W; ++i)
      if (mine[i]) F[64 * i + l].stamp = -1;
    for (int s = l; s < he; s += 64) {
      auto& e = E[s];
      if (e.stamp < 0) continue;
      if (e.vis == kInternal) {
        e.stamp = -1;
        continue;
      }
      V[e.v0].remove = 0;
      V[e.v1].remove = 0;
      if (e.vis == kBorder) {
        if (isVisible(vis, e.f0)) e.f0 = e.f1;
        e.f1 = kNil;
      }
    }
    M::sync();
    for (int s = l; s < hv; s += 64)
      if (V[s].remove) V[s].stamp = -1;
    M::sync();
    const int nvi = addVertex(nv_, nd, nh0, nh1);
    if (nvi == kNil) return 2;
    if (W > 1 && nb > 64) return coverBorder(static_cast<int16_t>(nvi));
    // New faces over the border edges, one border edge per lane (with at
    // most 64 faces there are at most 49: k connected visible faces have at
    // most k + 2 border edges, the others at most 3 (64 - k)); see
    // coverBorder for the order.
    int be = 0, bst = -1, ba = 0, bb = 0;
    if (l < nb) {
      be = BL[l].e;
      const auto& e = E[be];
      bst = e.stamp;
      ba = e.v0;
      bb = e.v1;
    }
    int rank = 0, t0 = 0, t1 = 0;
    for (int k = 0; k < nb; ++k) {
      const int sk = __builtin_amdgcn_readlane(bst, k);
      const int ak = __builtin_amdgcn_readlane(ba, k), bk = __builtin_amdgcn_readlane(bb, k);
      if (sk > bst) {
        ++rank;
        t0 += ak == ba || bk == ba;
        t1 += ak == bb || bk == bb;
      }
    }
    if (anyLane(l < nb && (t0 > 1 || t1 > 1))) return 2;  // a third face on a new edge
    const int made = 1 + (t0 == 0) + (t1 == 0);
    int pre = 0, total = 0;
    for (int k = 0; k < nb; ++k) {
      const int sk = __builtin_amdgcn_readlane(bst, k), mk = __builtin_amdgcn_readlane(made, k);
      total += mk;
      if (sk > bst) pre += mk;
    }
    const int new_edges = total - nb;
    if (new_edges > free_e || nb > free_f) return 2;
    // the free slot lists (before any slot is taken)
    for (int k = below_e + l; k < new_edges; k += 64) BL[k].fe = static_cast<int16_t>(he + k - below_e);
    for (int k = below_f + l; k < nb; k += 64) BL[k].ff = static_cast<int16_t>(hf + k - below_f);
    for (int base = 0, c = 0; base < he && c < new_edges; base += 64) {
      const int s = base + l;
      const bool fr = s < he && E[s < he ? s : 0].stamp < 0;
      const unsigned long long m = __ballot(fr);
      const int pos = c + __popcll(m & below);
      if (fr && pos < new_edges) BL[pos].fe = static_cast<int16_t>(s);
      c += __popcll(m);
    }
    {
      int c = 0;
#pragma unroll
      for (int i = 0; i < W; ++i) {
        if (64 * i >= hf) continue;
        const bool fr = 64 * i + l < hf && (!live[i] || mine[i]);
        const unsigned long long m = __ballot(fr);
        const int pos = c + __popcll(m & below);
        if (fr && pos < nb) BL[pos].ff = static_cast<int16_t>(64 * i + l);
        c += __popcll(m);
      }
    }
    M::sync();
    // new edges: the k-th created edge takes the k-th free edge slot
    const d3 va = vloc(ba), vb = vloc(bb);
    if (l < nb) {
      int q = 0;
#pragma nounroll
      for (int side = 0; side < 2; ++side) {
        if ((side ? t1 : t0) != 0) continue;
        const int vq = side ? bb : ba;
        const int16_t slot = BL[pre - rank + q].fe;
        auto& x = E[slot];
        x.v0 = static_cast<int16_t>(nvi);
        x.v1 = static_cast<int16_t>(vq);
        x.f0 = x.f1 = kNil;
        MinD m;
        segDist(d3{0, 0, 0}, nv_, d3{side ? vb.x : va.x, side ? vb.y : va.y, side ? vb.z : va.z}, m);
        x.in = m.in; x.d2 = m.d2; x.wx = m.w.x; x.wy = m.w.y; x.wz = m.w.z;
        x.stamp = stamp + pre + q;
        V[vq].new_edge = slot;
        ++q;
      }
    }
    M::sync();
    // faces: the face of rank r takes the r-th free face slot; the border
    // edge keeps its hidden face as f0; each new edge gets its lower-ranked
    // face as f0 and the other as f1
    bool clash = false;
    if (l < nb) {
      const int16_t slot = BL[rank].ff;
      const int ne0 = V[ba].new_edge, ne1 = V[bb].new_edge;
      auto& f = F[slot];
      f.e0 = static_cast<int16_t>(be);
      f.e1 = static_cast<int16_t>(ne0);
      f.e2 = static_cast<int16_t>(ne1);
      setFace(f, ba, va, vb, nv_);
      f.stamp = stamp + pre + (t0 == 0) + (t1 == 0);
      auto& ej = E[be];
      if (ej.f0 == kNil) ej.f0 = slot;
      else if (ej.f1 != kNil) clash = true;
      else ej.f1 = slot;
      if (t0 == 0) E[ne0].f0 = slot; else E[ne0].f1 = slot;
      if (t1 == 0) E[ne1].f0 = slot; else E[ne1].f1 = slot;
    }
    stamp += total;
    he += max(0, new_edges - below_e);
    hf += max(0, nb - below_f);
    M::sync();
    return anyLane(clash) ? 2 : 0;
  }

  // The same for any capacity, the face classes marked in LDS and the
  // border edges in BL (polytopes beyond kSmallFaces).
  MFCL_D int expandLarge(d3 nv_, d3 nd, int nh0, int nh1, int start) {
    const int l = __lane_id();
    for (int s = l; s < hv; s += 64) V[s].remove = 1;
    for (int s = l; s < he; s += 64) E[s].vis = kUnknown;
    // a face that does not see the new vertex is never visible, unless the
    // fill starts from it
    for (int s = l; s < hf; s += 64) F[s].vis = F[s].stamp >= 0 && outsideLane(s, nv_) ? kFUnknown : kHidden;
    M::sync();
    F[start].vis = kVisible;
    M::sync();
    while (true) {
      bool changed = false;
      for (int s = l; s < hf; s += 64) {
        const auto& f = F[s];
        if (f.stamp < 0 || f.vis != kFUnknown) continue;
        const int16_t es[3] = {f.e0, f.e1, f.e2};
        bool near_visible = false;
        for (int k = 0; k < 3; ++k) {
          const auto& e = E[es[k]];
          const int16_t g = e.f0 == s ? e.f1 : e.f0;
          if (g != kNil && F[g].vis == kVisible) near_visible = true;
        }
        if (!near_visible) continue;
        F[s].vis = kVisible;
        changed = true;
      }
      M::sync();
      if (!anyLane(changed)) break;
    }
    // an open edge on a visible face is a malformed polytope
    bool bad = false;
    for (int s = l; s < hf; s += 64) {
      const auto& f = F[s];
      if (f.stamp < 0 || f.vis != kVisible) continue;
      const int16_t es[3] = {f.e0, f.e1, f.e2};
      for (int k = 0; k < 3; ++k) {
        const auto& e = E[es[k]];
        const int16_t g = e.f0 == s ? e.f1 : e.f0;
        if (g == kNil) bad = true;
      }
    }
    if (anyLane(bad)) return 1;
    // edge marks from the final face classes
    for (int s = l; s < he; s += 64) {
      auto& e = E[s];
      if (e.stamp < 0) continue;
      const bool v0 = e.f0 != kNil && F[e.f0].vis == kVisible;
      const bool v1 = e.f1 != kNil && F[e.f1].vis == kVisible;
      if (v0 && v1) {
        e.vis = kInternal;
      } else if (v0 || v1) {
        e.vis = kBorder;
        if (v0) e.f0 = e.f1;
        e.f1 = kNil;
      }
    }
    M::sync();
    for (int s = l; s < he; s += 64) {
      const auto& e = E[s];
      if (e.stamp < 0 || e.vis == kInternal) continue;
      V[e.v0].remove = 0;
      V[e.v1].remove = 0;
    }
    M::sync();
    // drop the visible faces, the internal edges and the vertices left
    // without a non-internal edge
    for (int s = l; s < hf; s += 64)
      if (F[s].stamp >= 0 && F[s].vis == kVisible) F[s].stamp = -1;
    for (int s = l; s < he; s += 64)
      if (E[s].vis == kInternal) E[s].stamp = -1;
    for (int s = l; s < hv; s += 64)
      if (V[s].remove) V[s].stamp = -1;
    M::sync();
    const int nvi = addVertex(nv_, nd, nh0, nh1);
    if (nvi == kNil) return 2;
    return coverBorder(static_cast<int16_t>(nvi));
  }

  // New faces over the border edges (epa_polytope_expand.hpp:233-281).  The
  // reference walks the border edges newest first; for each it creates the
  // edge (new vertex, endpoint) unless an earlier border edge already did,
  // then the face, each taking the next creation stamp; a new edge's first
  // face becomes its f0, the second its f1, a third is an error.  All of
  // that follows from each border edge's rank in that order, so the lanes
  // build the faces together: rank and sharing counts by comparison with the
  // other border edges, creation positions by a prefix over the ranks, slots
  // from the free lists (which free slot is used does not matter).  A slot
  // shortage fails the expansion as the reference's allocation failure does.
  MFCL_D int coverBorder(int16_t nvi) {
    const int l = __lane_id();
    const unsigned long long below = (1ull << l) - 1;
    int nb = 0;
    for (int base = 0; base < he; base += 64) {
      const int s = base + l;
      const bool isb = s < he && E[s].stamp >= 0 && E[s].vis == kBorder;
      const unsigned long long m = __ballot(isb);
      if (isb) BL[nb + __popcll(m & below)].e = static_cast<int16_t>(s);
      nb += __popcll(m);
    }
    M::sync();
    for (int j = l; j < nb; j += 64) {
      const int st = E[BL[j].e].stamp;
      int rank = 0;
      for (int k = 0; k < nb; ++k) rank += E[BL[k].e].stamp > st;
      BL[j].rank = static_cast<int16_t>(rank);
    }
    M::sync();
    bool bad = false;
    int new_edges = 0;
    for (int j = l; j < nb; j += 64) {
      const auto& ej = E[BL[j].e];
      const int r = BL[j].rank, a = ej.v0, b = ej.v1;
      int t0 = 0, t1 = 0;
      for (int k = 0; k < nb; ++k) {
        if (BL[k].rank >= r) continue;
        const auto& ek = E[BL[k].e];
        t0 += ek.v0 == a || ek.v1 == a;
        t1 += ek.v0 == b || ek.v1 == b;
      }
      if (t0 > 1 || t1 > 1) bad = true;  // a third face on a new edge
      BL[j].t0 = static_cast<int8_t>(t0 > 1 ? 2 : t0);
      BL[j].t1 = static_cast<int8_t>(t1 > 1 ? 2 : t1);
      new_edges += (t0 == 0) + (t1 == 0);
    }
    if (anyLane(bad)) return 2;
    M::sync();
    for (int j = l; j < nb; j += 64) {
      const int r = BL[j].rank;
      int pre = 0;
      for (int k = 0; k < nb; ++k)
        if (BL[k].rank < r) pre += 1 + (BL[k].t0 == 0) + (BL[k].t1 == 0);
      BL[j].pre = static_cast<int16_t>(pre);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) new_edges += __shfl_xor(new_edges, off);
    // capacity
    int below_e = 0, below_f = 0;
    for (int base = 0; base < he; base += 64) below_e += __popcll(__ballot(base + l < he && E[base + l].stamp < 0));
    for (int base = 0; base < hf; base += 64) below_f += __popcll(__ballot(base + l < hf && F[base + l].stamp < 0));
    new_edges = __builtin_amdgcn_readfirstlane(new_edges);
    if (new_edges > below_e + nv - he || nb > below_f + nf - hf) return 2;
    // the free slot lists (before any slot is taken)
    {
      for (int k = below_e + l; k < new_edges; k += 64) BL[k].fe = static_cast<int16_t>(he + k - below_e);
      for (int k = below_f + l; k < nb; k += 64) BL[k].ff = static_cast<int16_t>(hf + k - below_f);
      int ce = 0, cf = 0;
      for (int base = 0; base < he; base += 64) {
        const int s = base + l;
        const bool fr = s < he && E[s].stamp < 0;
        const unsigned long long m = __ballot(fr);
        const int pos = ce + __popcll(m & below);
        if (fr && pos < new_edges) BL[pos].fe = static_cast<int16_t>(s);
        ce += __popcll(m);
      }
      for (int base = 0; base < hf; base += 64) {
        const int s = base + l;
        const bool fr = s < hf && F[s].stamp < 0;
        const unsigned long long m = __ballot(fr);
        const int pos = cf + __popcll(m & below);
        if (fr && pos < nb) BL[pos].ff = static_cast<int16_t>(s);
        cf += __popcll(m);
      }
    }
    M::sync();
    // new edges: the k-th created edge takes the k-th free edge slot
    for (int j = l; j < nb; j += 64) {
      const auto& bj = BL[j];
      const auto& ej = E[bj.e];
      const int edges_before = bj.pre - bj.rank;
      int q = 0;
      for (int side = 0; side < 2; ++side) {
        if ((side ? bj.t1 : bj.t0) != 0) continue;
        const int16_t vq = side ? ej.v1 : ej.v0;
        const int16_t slot = BL[edges_before + q].fe;
        auto& x = E[slot];
        x.v0 = nvi;
        x.v1 = vq;
        x.f0 = x.f1 = kNil;
        x.vis = kUnknown;
        MinD m;
        segDist(d3{0, 0, 0}, vloc(nvi), vloc(vq), m);
        x.in = m.in; x.d2 = m.d2; x.wx = m.w.x; x.wy = m.w.y; x.wz = m.w.z;
        x.stamp = stamp + bj.pre + q;
        V[vq].new_edge = slot;
        ++q;
      }
    }
    M::sync();
    // faces: the face of rank r takes the r-th free face slot
    for (int j = l; j < nb; j += 64) {
      const auto& bj = BL[j];
      const int16_t ei = bj.e;
      auto& ej = E[ei];
      const int16_t a = ej.v0, b = ej.v1;
      const int16_t ne0 = V[a].new_edge, ne1 = V[b].new_edge;
      const int16_t slot = BL[bj.rank].ff;
      auto& f = F[slot];
      f.e0 = ei; f.e1 = ne0; f.e2 = ne1;
      f.vis = kFUnknown;
      setFace(f, a, vloc(a), vloc(b), vloc(nvi));
      f.stamp = stamp + bj.pre + (bj.t0 == 0) + (bj.t1 == 0);
    }
    M::sync();
    // links: the border edge keeps its hidden face as f0; each new edge gets
    // its lower-ranked face as f0 and the other as f1
    bool clash = false;
    for (int j = l; j < nb; j += 64) {
      const auto& bj = BL[j];
      auto& ej = E[bj.e];
      const int16_t slot = BL[bj.rank].ff;
      if (ej.f0 == kNil) ej.f0 = slot;
      else if (ej.f1 != kNil) clash = true;
      else ej.f1 = slot;
      auto& x0 = E[V[ej.v0].new_edge];
      auto& x1 = E[V[ej.v1].new_edge];
      if (bj.t0 == 0) x0.f0 = slot; else x0.f1 = slot;
      if (bj.t1 == 0) x1.f0 = slot; else x1.f1 = slot;
    }
    stamp += new_edges + nb;
    he += max(0, new_edges - below_e);
    hf += max(0, nb - below_f);
    M::sync();
    return anyLane(clash) ? 2 : 0;
  }

};

// The closest feature of one iteration: what the witness points are formed
// from.
struct RawF {
  double m[4];     // d2, then the witness
  double v[3][6];  // vertex and direction of a, b, c
  int h[3][2];     // support vertices of a, b, c (-1: primitive or unknown)
  int kind, pad;
};
// Where a pair that outgrows its polytope continues: the expansion it is at.
struct EpaResume {
  d3 nv, nd;
  int it, stamp, nh0, nh1, start, item, hv, he, hf, pad;
};
// The result in shape-0 frame (status: EpaStatus, or kEpaSpill).
struct EpaOut {
  double depth;
  d3 p0, p1;
  int iters, scanned;
};
// A wavefront's LDS slice: the pair's configuration and simplex, the records
// above, then the polytope arena at kEpaHeadBytes.
struct EpaLds {
  WaveCfg cfg;
  SmpD s;
  RawF raw;
  EpaResume res;
  EpaOut out;
};
constexpr int kEpaSpill = 5;
constexpr size_t kEpaHeadBytes = (sizeof(EpaLds) + 15) & ~static_cast<size_t>(15);
template <class M>
__host__ __device__ inline size_t epaSliceBytes(int cap_faces) {
  return kEpaHeadBytes + arenaBytes<M>(cap_faces);
}
// A dumped pair in device memory: RawF, EpaResume and the slot arrays.
constexpr size_t kEpaDumpHead = sizeof(RawF) + sizeof(EpaResume);
__host__ __device__ inline size_t epaDumpBytes(int cap_faces) {
  return (kEpaDumpHead + polyBytes<SmallMem>(cap_faces) + 255) & ~static_cast<size_t>(255);
}
static_assert(sizeof(RawF) % 8 == 0 && sizeof(EpaResume) % 8 == 0, "dumped as 8-byte words");

MFCL_D d3 ldsGet(const MFCL_LDS d3& o) { return d3{o.x, o.y, o.z}; }
MFCL_D d3 ldsGet(const MFCL_LDS double* o) { return d3{o[0], o[1], o[2]}; }
MFCL_D void ldsSet(MFCL_LDS d3& o, d3 v) { o.x = v.x; o.y = v.y; o.z = v.z; }
MFCL_D const MFCL_LDS MVD& smpVert(const MFCL_LDS SmpD& s, int k) {
  return k == 0 ? s.a : (k == 1 ? s.b : (k == 2 ? s.c : s.e));
}
MFCL_D void ldsSync() { __builtin_amdgcn_wave_barrier(); }
MFCL_D MFCL_LDS char* ldsArena(MFCL_LDS EpaLds* L) { return (MFCL_LDS char*)(L) + kEpaHeadBytes; }

// Vertex i of an initial polytope (every lane writes the same).
template <class M>
MFCL_D void putVertex(PolyT<M>& P, int i, d3 v, d3 d) {
  auto& x = P.V[i];
  x.vx = v.x; x.vy = v.y; x.vz = v.z;
  x.dx = d.x; x.dy = d.y; x.dz = d.z;
  x.h0 = x.h1 = -1;
}
template <class M>
MFCL_D void putVertex(PolyT<M>& P, int i, const MFCL_LDS MVD& m) { putVertex(P, i, ldsGet(m.v), ldsGet(m.d)); }
// epa_simplex2polytope.hpp:184-217 (a capacity of 4 faces, the least there
// is, holds it)
template <class M>
MFCL_D bool buildTetra(PolyT<M>& P) {
  M::sync();
  return P.build(4, 6, 4, 0x333210ull, 0x210021ull, 0x5430ull, 0x3541ull, 0x2102ull);
}

// simplexToPolytope's status: failed, touching (the points in out), or the
// initial polytope that was built.
constexpr int kS2pFailed = -1, kS2pTouching = 0, kS2pTetra = 4, kS2pOcta = 6;

MFCL_D int touchingPoint(MinkW& md, d3 d, MFCL_LDS EpaLds* L) {
  const WaveSup a = md.sup(d);
  const d3 mid = (a.p0 + a.p1) / 2;
  ldsSet(L->out.p0, mid);
  ldsSet(L->out.p1, mid);
  return kS2pTouching;
}

// Out of line: few pairs start from a triangle or a segment.  tri: the
// simplex vertices that form the triangle, (a, b, c), (a, c, e), (a, b, e)
// or (b, c, e).
template <class M>
__device__ __attribute__((noinline)) int s2p3(MFCL_LDS EpaLds* L, typename M::template P<char> arena, int cap_faces,
                                              int tri, double thr) {
  PolyT<M> P(arena, cap_faces);
  MinkW md{&L->cfg, 0};
  const MFCL_LDS MVD& va = smpVert(L->s, tri == 3 ? 1 : 0);
  const MFCL_LDS MVD& vb = smpVert(L->s, tri == 1 || tri == 3 ? 2 : 1);
  const MFCL_LDS MVD& vc = smpVert(L->s, tri == 0 ? 2 : 3);
  const d3 a = ldsGet(va.v), b = ldsGet(vb.v), c = ldsGet(vc.v);
  int r = kS2pFailed;
  d3 n = cross(b - a, c - a);
  if (!ub(sqnorm(n) <= 0.0)) {
    n = normalized(n);
    const d3 d0 = md.support(n);
    const double t0 = planeDist(d0, a, b, c);
    const d3 dir1 = -n;
    const d3 d1 = md.support(dir1);
    const double t1 = planeDist(d1, a, b, c);
    if (ub(t0 <= thr)) {
      r = touchingPoint(md, n, L);
    } else if (ub(t1 <= thr)) {
      r = touchingPoint(md, dir1, L);
    } else {
      const bool up = ub(t0 > t1);
      putVertex(P, 0, va);
      putVertex(P, 1, vb);
      putVertex(P, 2, vc);
      putVertex(P, 3, up ? d0 : d1, up ? n : dir1);
      if (buildTetra(P)) r = kS2pTetra;
    }
  }
  L->out.scanned += md.scanned;
  return r;
}

template <class M>
MFCL_D int s2p2Run(PolyT<M>& P, MinkW& md, MFCL_LDS EpaLds* L, double thr) {
  const double thr2 = thr * thr;
  const d3 a = ldsGet(L->s.a.v), b = ldsGet(L->s.b.v);
  const d3 ab = b - a;
  if (ub(sqnorm(ab) < thr2)) return kS2pFailed;
  const d3 abu = normalized(ab);
  d3 dinit = {abu.y, -abu.x, 0};
  bool valid = sqnorm(dinit) > thr2;
  if (!valid) { dinit = d3{abu.z, 0, -abu.x}; valid = sqnorm(dinit) > thr2; }
  if (!valid) { dinit = d3{0, abu.z, -abu.y}; valid = sqnorm(dinit) > thr2; }
  if (ub(!valid)) return kS2pFailed;
  dinit = normalized(dinit);
  d3 d = dinit, v = {0, 0, 0};
  bool found = false;
#pragma nounroll
  for (int i = 0; i < 72; ++i) {
    v = md.support(d);
    if (ub(lineDist(v, a, b) > thr)) {
      found = true;
      break;
    }
    const double step = 2.0 * 3.145926 / 72;  // the reference's pi constant (sic)
    d = normalized(d + step * cross(abu, v));
  }
  if (!found) return touchingPoint(md, dinit, L);
  // the octahedron a, v0, b, v1, v2, v3: v1 opposite v0, v2 and v3 along
  // the normal of (a, v0, v1).  Too small a capacity fails as the
  // reference's allocation does, after the searches.
  const bool room = P.nv >= 12 && P.nf >= 8;
  if (room) {
    putVertex(P, 0, L->s.a);
    putVertex(P, 2, L->s.b);
  }
  d3 v0 = v;
#pragma nounroll
  for (int k = 0; k < 4; ++k) {
    if (k == 2) {
      const d3 n = cross(v0 - a, v - a);
      if (ub(sqnorm(n) < thr2)) return kS2pFailed;
      d = normalized(n);
    } else if (k > 0) {
      d = -d;
    }
    if (k > 0) {
      v = md.support(d);
      if (ub(lineDist(v, a, b) < thr)) return touchingPoint(md, d, L);
    }
    if (room) putVertex(P, k == 0 ? 1 : k + 2, v, d);
  }
  if (!room) return kS2pFailed;
  M::sync();
  P.build(6, 12, 8, 0x555544443210ull, 0x321032100321ull, 0xBA987654ull, 0x8BA94765ull, 0x32103210ull);
  return kS2pOcta;
}
template <class M>
__device__ __attribute__((noinline)) int s2p2(MFCL_LDS EpaLds* L, typename M::template P<char> arena, int cap_faces,
                                              double thr) {
  PolyT<M> P(arena, cap_faces);
  MinkW md{&L->cfg, 0};
  const int r = s2p2Run(P, md, L, thr);
  L->out.scanned += md.scanned;
  return r;
}

// epa_simplex2polytope.hpp:46-110 on the simplex in LDS.
template <class M>
MFCL_D int simplexToPolytope(PolyT<M>& P, MinkW& md, MFCL_LDS EpaLds* L, typename M::template P<char> arena,
                             int cap_faces, double thr) {
  const MFCL_LDS SmpD& s = L->s;
  const double thr2 = thr * thr;
  const int rank = __builtin_amdgcn_readfirstlane(s.rank);
  const int q = __lane_id() & 3;
  // a simplex vertex at the origin, one vertex per lane
  const unsigned long long at = __ballot(q < rank && sqnorm(ldsGet(smpVert(s, q).v)) <= thr2) & 15ull;
  if (at) return touchingPoint(md, ldsGet(smpVert(s, __builtin_ctzll(at)).d), L);
  if (rank <= 1) {
    const WaveSup a = md.sup(ldsGet(s.a.d));
    ldsSet(L->out.p0, a.p0);
    ldsSet(L->out.p1, a.p1);
    return kS2pTouching;
  }
  if (rank == 2) return s2p2<M>(L, arena, cap_faces, thr);
  if (rank == 3) return s2p3<M>(L, arena, cap_faces, 0, thr);
  // the distances of the faces (a, b, c), (a, c, e), (a, b, e), (b, c, e)
  // from the origin, one per lane
  const d3 x = ldsGet(smpVert(s, q == 3 ? 1 : 0).v), y = ldsGet(smpVert(s, q & 1 ? 2 : 1).v),
           w = ldsGet(smpVert(s, q == 0 ? 2 : 3).v);
  const unsigned long long flat = __ballot(planeDist(d3{0, 0, 0}, x, y, w) < thr) & 15ull;
  if (flat) return s2p3<M>(L, arena, cap_faces, __builtin_ctzll(flat), thr);
  putVertex(P, 0, s.a);
  putVertex(P, 1, s.b);
  putVertex(P, 2, s.c);
  putVertex(P, 3, s.e);
  return buildTetra(P) ? kS2pTetra : kS2pFailed;
}

// The closest feature's record, one word or double per lane.
template <class M>
MFCL_D void toRaw(const PolyT<M>& P, int kind, int i, MFCL_LDS RawF& r) {
  using D = typename M::template P<const double>;
  const int l = __lane_id();
  int16_t ia, ib, ic;
  D rec;
  if (kind == 2) {
    ia = P.E[i].v0;
    ib = ic = P.E[i].v1;
    rec = (D)(&P.E[i]);
  } else {
    P.faceVerts(i, ia, ib, ic);
    rec = (D)(&P.F[i]);
  }
  const int k = l < 18 ? l / 6 : (l - 22) >> 1;
  const int v = k == 0 ? ia : (k == 1 ? ib : ic);
  if (l < 18) ((MFCL_LDS double*)r.v)[l] = ((D)(&P.V[v]))[l - 6 * k];
  else if (l < 22) r.m[l - 18] = rec[l - 18];
  else if (l < 28) r.h[k][l & 1] = l & 1 ? P.V[v].h1 : P.V[v].h0;
  else if (l == 28) r.kind = kind;
  ldsSync();
}

// epa.hpp:341-498: depth and witness points into L->out.
// support0 / support1 of a recorded direction come from the recorded
// support vertices when there are (the same points the support searches
// returned when the polytope vertex was created).
__device__ __attribute__((noinline)) static void assignPair(MFCL_LDS EpaLds* L, double cx, double cy, double cz, int ch0,
                                                            int ch1) {
  MinkW md{&L->cfg, 0};
  const MFCL_LDS RawF& f = L->raw;
  MFCL_LDS EpaOut& o = L->out;
  const int kind = __builtin_amdgcn_readfirstlane(f.kind);
  const d3 a = ldsGet(f.v[0]), b = ldsGet(f.v[1]), p = ldsGet(f.m + 1);
  double w[3] = {1, 0, 0};
  int n = 0;         // blended vertices
  bool one = false;  // the first vertex's points as they are
  double depth = sqrt(f.m[0]);
  if (kind == 2) {
    const d3 ab = b - a;
    int ax = 0;
    double mx = fabs(ab.x);
    if (fabs(ab.y) > mx) { ax = 1; mx = fabs(ab.y); }
    if (fabs(ab.z) > mx) { ax = 2; mx = fabs(ab.z); }
    if (ub(mx <= 1e-10)) {
      one = true;
    } else {
      const double s = (comp(p, ax) - comp(a, ax)) / (comp(b, ax) - comp(a, ax));
      if (ub(!(s < 0 || s > 1.0))) {
        w[0] = 1.0 - s;
        w[1] = s;
        n = 2;
      }
    }
  } else {
    const d3 c = ldsGet(f.v[2]);
    const d3 dl0 = a - b, dl1 = b - c, dl2 = c - a;
    const double area = sqrt(sqnorm(cross(dl0, dl1)));
    w[0] = norm(cross(dl1, b - p)) / area;
    w[1] = norm(cross(dl2, c - p)) / area;
    const double chk = norm(cross(dl0, a - p)) / area;
    w[2] = 1.0 - w[0] - w[1];
    if (ub(!(fabs(chk - w[2]) > 0.01))) n = 3;
  }
  d3 q0 = {0, 0, 0}, q1 = q0;
  const bool cand = n == 0 && !one;
#pragma nounroll
  for (int k = 0; k < (n ? n : 1); ++k) {
    const int h0 = cand ? ch0 : f.h[k][0], h1 = cand ? ch1 : f.h[k][1];
    const d3 d = cand ? d3{cx, cy, cz} : ldsGet(f.v[k] + 3);
    d3 a0, a1;
    md.pointsAt(h0, h1, d, a0, a1);
    if (n == 0) {
      q0 = a0;
      q1 = a1;
    } else {
      const double wk = k == 0 ? w[0] : (k == 1 ? w[1] : w[2]);
      q0 = k == 0 ? wk * a0 : q0 + wk * a0;
      q1 = k == 0 ? wk * a1 : q1 + wk * a1;
    }
  }
  if (cand) depth = norm(q0 - q1);
  ldsSet(o.p0, q0);
  ldsSet(o.p1, q1);
  o.depth = depth;
  o.scanned += md.scanned;
}

// epa.hpp:137-257 on the pair and simplex in L (resume: from the expansion
// in L->res, the polytope in L already).  Returns the status; depth, points,
// iterations and vertices scanned in L->out.  may_spill: the request's
// capacity is larger than this polytope's; a pair whose expansion might not
// fit stops before it (kEpaSpill, L->res filled in).
template <class M>
__device__ __attribute__((noinline)) int epaRun(MFCL_LDS EpaLds* L, typename M::template P<char> arena, int cap_faces,
                                                double tol, int max_iter, bool may_spill, bool resume) {
  constexpr double kOuter = 1e-3 * 1e-3;
  constexpr double kRatio = 1.0 - 1e-3;
  PolyT<M> P(arena, cap_faces);
  MinkW md{&L->cfg, 0};
  MFCL_LDS EpaOut& o = L->out;
  o.iters = 0;
  o.scanned = 0;
  o.depth = 0;
  ldsSet(o.p0, d3{0, 0, 0});
  ldsSet(o.p1, d3{0, 0, 0});
  int it = 0, start = kNil, nh0 = -1, nh1 = -1, status = kEpaFailed;
  d3 nd = {0, 0, 0}, nv = {0, 0, 0};
  if (resume) {
    it = __builtin_amdgcn_readfirstlane(L->res.it);
    start = __builtin_amdgcn_readfirstlane(L->res.start);
    nh0 = __builtin_amdgcn_readfirstlane(L->res.nh0);
    nh1 = __builtin_amdgcn_readfirstlane(L->res.nh1);
    P.stamp = __builtin_amdgcn_readfirstlane(L->res.stamp);
    P.hv = __builtin_amdgcn_readfirstlane(L->res.hv);
    P.he = __builtin_amdgcn_readfirstlane(L->res.he);
    P.hf = __builtin_amdgcn_readfirstlane(L->res.hf);
    nv = ldsGet(L->res.nv);
    nd = ldsGet(L->res.nd);
  } else {
    const int s2p = __builtin_amdgcn_readfirstlane(simplexToPolytope(P, md, L, arena, cap_faces, tol));
    o.scanned += md.scanned;
    md.scanned = 0;
    if (s2p < 0) return kEpaFailed;
    if (s2p == kS2pTouching) return kEpaTouching;
    // (the octahedron's and the triangle's builders work on copies of P)
    P.hv = s2p;
    P.he = s2p == kS2pTetra ? 6 : 12;
    P.hf = s2p == kS2pTetra ? 4 : 8;
    P.stamp = P.hv + P.he + P.hf;
  }
  bool pending = resume;
  while (true) {
    if (!pending) {
      int kind, fi;
      P.minToOrigin(false, kind, fi);
      if (kind == 1) {
        const double vd2 = sqnorm(P.vloc(fi));
        int k2, i2;
        P.minToOrigin(true, k2, i2);
        if (k2 == 0) break;
        const double d2 = k2 == 2 ? P.E[i2].d2 : P.F[i2].d2;
        if (ub(kRatio * d2 < vd2)) { kind = k2; fi = i2; }
      }
      if (kind != 2 && kind != 3) break;
      toRaw(P, kind, fi, L->raw);
      // epa.hpp:11-113: candidate directions -- the witness's (phase 0,
      // when it is far enough from the origin), then the normal of the face
      // or of the edge's first and second face (phases 1, 2) -- until a
      // support point lies beyond its face
      int fa = fi, fb = fi;
      if (kind == 2) {
        fa = __builtin_amdgcn_readfirstlane(P.E[fi].f0);
        fb = __builtin_amdgcn_readfirstlane(P.E[fi].f1);
        if (fa == kNil || fb == kNil) break;  // open edge: malformed polytope
      }
      const typename PolyT<M>::Normal na = P.normalOut(fa), nb = kind == 2 ? P.normalOut(fb) : na;
      if (kind == 3 && !na.ok) break;
      int ph = ub(L->raw.m[0] > kOuter) ? 0 : 1, ds = -1;
      double ba = 0;
      start = kNil;
      nh0 = nh1 = -1;
      while (ds < 0) {
        if (ph == 1 && !na.ok) ph = 2;  // an edge's degenerate first face
        if (ph == 2 && !nb.ok) {
          ds = 1;
          break;
        }
        nd = ph == 0 ? normalized(ldsGet(L->raw.m + 1)) : (ph == 1 ? na.n : nb.n);
        const WaveSup s = md.sup(nd);
        nv = s.p0 - s.p1;
        nh0 = s.i0;
        nh1 = s.i1;
        ba = dot(na.n, nv - P.faceAnchor(fa));
        const double bb = kind == 2 ? dot(nb.n, nv - P.faceAnchor(fb)) : 0.0;
        if (ph == 0) {
          // a degenerate face counts as seen (its area is not positive)
          if (ub(!na.ok || ba >= 0.0)) { start = fa; ds = 0; }
          else if (kind == 2 && ub(!nb.ok || bb >= 0.0)) { start = fb; ds = 0; }
          else ph = 1;
        } else if (ub((ph == 1 ? ba : bb) > tol)) {
          start = ph == 1 ? fa : fb;
          ds = 0;
        } else if (kind == 3 || ph == 2) {
          ds = 2;
        } else {
          ph = 2;
        }
      }
      if (ds == 1) break;
      // epa.hpp:269-299: converged when the support point is within tol of
      // the closest feature -- a face's plane (ba is that distance, signed;
      // the face is not degenerate here), or a segment (the squared norm of
      // the projection, as in the reference)
      double d2 = ba * ba;
      if (kind == 2) {
        MinD m;
        segDist(nv, ldsGet(L->raw.v[0]), ldsGet(L->raw.v[1]), m);
        d2 = m.d2;
      }
      if (ds == 2 || ub(d2 < tol * tol)) {
        status = kEpaOK;
        break;
      }
    }
    pending = false;
    int ex;
    if constexpr (M::kWords > 0) ex = P.expandMask(nv, nd, nh0, nh1, start, may_spill);
    else ex = P.expandLarge(nv, nd, nh0, nh1, start);
    ex = __builtin_amdgcn_readfirstlane(ex);
    if (M::kWords > 0 && ex == 3) {
      ldsSet(L->res.nv, nv);
      ldsSet(L->res.nd, nd);
      L->res.it = it;
      L->res.stamp = P.stamp;
      L->res.hv = P.hv;
      L->res.he = P.he;
      L->res.hf = P.hf;
      L->res.nh0 = nh0;
      L->res.nh1 = nh1;
      L->res.start = start;
      o.scanned += md.scanned;
      return kEpaSpill;
    }
    if (ex == 1) break;
    if (ex == 2) {
      status = kEpaMallocFailed;
      break;
    }
    ++it;
    if (it >= max_iter) {
      status = kEpaIterLimit;
      break;
    }
  }
  o.scanned += md.scanned;
  if (status != kEpaFailed) {
    o.iters = it;
    assignPair(L, nd.x, nd.y, nd.z, nh0, nh1);
  }
  return status;
}

// A dumped pair to / from device memory: the records keep their slot
// numbers, the larger polytope's extra slots are free.  Slot numbers never
// influence a result, so continuing there equals a run at the larger
// capacity from the start.
MFCL_D void copyOut(char* dst, const MFCL_LDS char* src, size_t bytes) {
  uint64_t* d = reinterpret_cast<uint64_t*>(dst);
  const MFCL_LDS uint64_t* s = (const MFCL_LDS uint64_t*)(src);
  for (uint32_t k = __lane_id(); k < bytes / 8; k += 64) d[k] = s[k];
}
MFCL_D void epaDump(char* dst, MFCL_LDS EpaLds* L, int cap_faces, int item) {
  L->res.item = item;
  ldsSync();
  copyOut(dst, (const MFCL_LDS char*)(&L->raw), sizeof(RawF));
  copyOut(dst + sizeof(RawF), (const MFCL_LDS char*)(&L->res), sizeof(EpaResume));
  copyOut(dst + kEpaDumpHead, ldsArena(L), polyBytes<SmallMem>(cap_faces));
}
MFCL_D int epaDumpItem(const char* src) {
  return reinterpret_cast<const EpaResume*>(src + sizeof(RawF))->item;
}
// n records of type FROM into records that are FROM or a prefix of it
template <class FROM, class P>
MFCL_D void copyRecs(P dst, const char* src, int n) {
  using To = std::remove_reference_t<decltype(*dst)>;
  constexpr int kWords = sizeof(To) / 8, kFrom = sizeof(FROM) / 8;
  static_assert(kWords <= kFrom, "a prefix");
  using Wp = std::conditional_t<std::is_same<P, To*>::value && std::is_pointer<P>::value && sizeof(P) == 8, uint64_t*,
                                MFCL_LDS uint64_t*>;
  Wp d = (Wp)(dst);
  const uint64_t* s = reinterpret_cast<const uint64_t*>(src);
  for (int k = static_cast<int>(__lane_id()); k < n * kWords; k += 64) d[k] = s[k / kWords * kFrom + k % kWords];
}
template <class M>
MFCL_D void epaLoad(MFCL_LDS EpaLds* L, typename M::template P<char> arena, int cap_faces, const char* src,
                    int small_faces) {
  const ArenaDims sd = arenaDims(small_faces);
  PolyT<M> P(arena, cap_faces);
  const uint64_t* w = reinterpret_cast<const uint64_t*>(src);
  for (uint32_t k = __lane_id(); k < kEpaDumpHead / 8; k += 64) {
    if (k < sizeof(RawF) / 8) ((MFCL_LDS uint64_t*)(&L->raw))[k] = w[k];
    else ((MFCL_LDS uint64_t*)(&L->res))[k - sizeof(RawF) / 8] = w[k];
  }
  src += kEpaDumpHead;
  using S = PolyT<SmallMem>;
  copyRecs<S::EVert>(P.V, src, sd.nv);
  src += sizeof(S::EVert) * sd.nv;
  copyRecs<S::EEdge>(P.E, src, sd.nv);
  src += sizeof(S::EEdge) * sd.nv;
  copyRecs<S::EFace>(P.F, src, sd.nf);
  M::sync();
  ldsSync();
}

}  // namespace mfcl
