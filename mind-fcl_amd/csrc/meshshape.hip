// Mesh-shape collision (fcl::collide(BVHModel<OBBRSS>, shape), penetration
// disabled, and enabled below): OrientedNodeBVHSolver::MeshShapeIntersect
// (include/fcl/narrowphase/detail/traversal/collision/bvh_solver-inl.h:6-72)
// tests the mesh's tree against the shape's volume and every reached leaf
// triangle against the shape (ShapeSimplexIntersect, shape_pair_intersect-
// inl.h:133-172 -> GJKSolver::shapeTriangleIntersect, gjk_solver-inl.h:
// 545-563: sphereTriangleIntersect, boxTriangleIntersect, else MPR on the
// shape and the triangle).
//
// Three launches: (1) one wavefront per query walks the mesh's OBB tree
// against the shape's box (its frame, FP32 test with the conservative
// margin of the mesh-mesh traversal), 64 nodes per step off an LDS stack,
// and appends every reached leaf as a (query, triangle) candidate; (2) the
// leaf tests in FP64 exactly as the reference orders them, closed forms one
// per lane and searches one per wavefront, counting and recording colliding
// triangles; (3) one wavefront per query writes the result and its kept
// triangles in ascending order.  The set of
// colliding triangles does not depend on the tree, so booleans and complete
// sets equal the reference's; which ones are kept when more than
// max_contacts collide follows the traversal here, not the reference's
// depth-first order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>
#include <vector>

#include "ctx.h"
#include "epa_dev.h"
#include "narrow_dev.h"
#include "obb_dev.h"

namespace mfcl {

constexpr int kMsStack = 2048;  // node ids per wavefront (LDS)

struct MeshShapeArgs {
  ShapeTables T;
  const double4* interior;
  const ObbNode* nodes;
  const float4* tris;
  const uint32_t* node_base;
  const uint32_t* tri_base;
  const uint32_t* mesh_ids;
  const uint32_t* shape_ids;
  const float* pose_m;
  const float* pose_s;
  uint64_t n;
  uint64_t* cand;
  uint64_t cand_cap;
  unsigned long long* cand_count;
  uint32_t* counts;    // per query: colliding triangles
  uint32_t* leaves;    // per query: candidate leaves
  uint32_t* bv_tests;  // per query: OBB tests
  uint32_t* overflow;  // per query: 1 when the LDS stack would overflow
  int max_contacts;
  int32_t* tri_out;    // colliding triangles: in the order of arrival, then ascending
  int gjk_max_it;
  double gjk_tol;
};

// The shape's box in its own frame: half extents that contain it.
MFCL_D ObbNode shapeBox(int type, float4 p) {
  ObbNode b;
  for (int k = 0; k < 9; ++k) b.ax[k] = (k % 4 == 0) ? 1.f : 0.f;
  b.c[0] = b.c[1] = b.c[2] = 0.f;
  float e0, e1, e2;
  if (type == kBox) { e0 = 0.5f * p.x; e1 = 0.5f * p.y; e2 = 0.5f * p.z; }
  else if (type == kSphere) { e0 = e1 = e2 = p.x; }
  else if (type == kCapsule) { e0 = e1 = p.x; e2 = 0.5f * p.y + p.x; }
  else if (type == kCylinder) { e0 = e1 = p.x; e2 = 0.5f * p.y; }
  else { e0 = e1 = e2 = p.w; }  // convex: max |coordinate|
  b.e[0] = e0; b.e[1] = e1; b.e[2] = e2;
  b.child = 0;
  return b;
}

__global__ void __launch_bounds__(64) msCandKernel(MeshShapeArgs A) {
  __shared__ int32_t stk[kMsStack];
  const uint64_t q = blockIdx.x;
  if (q >= A.n) return;
  const int l = threadIdx.x;
  const uint32_t mesh = A.mesh_ids[q], shp = A.shape_ids[q];
  const ObbNode sb = shapeBox(A.T.type[shp], A.T.param[shp]);
  const tf3 tm = poseFromQuat(A.pose_m + 7 * q), ts = poseFromQuat(A.pose_s + 7 * q);
  const tf3 rel = relTf(tm, ts);  // shape frame in the mesh frame
  const float Rq[9] = {static_cast<float>(rel.R.m00), static_cast<float>(rel.R.m01), static_cast<float>(rel.R.m02),
                       static_cast<float>(rel.R.m10), static_cast<float>(rel.R.m11), static_cast<float>(rel.R.m12),
                       static_cast<float>(rel.R.m20), static_cast<float>(rel.R.m21), static_cast<float>(rel.R.m22)};
  const float Tq[3] = {static_cast<float>(rel.t.x), static_cast<float>(rel.t.y), static_cast<float>(rel.t.z)};
  const ObbNode* nodes = A.nodes + A.node_base[mesh];
  const unsigned long long below = (1ull << l) - 1;
  if (l == 0) stk[0] = 0;
  int top = 1;
  uint32_t tests = 0, leaves = 0;
  bool ovf = false;
  __builtin_amdgcn_wave_barrier();
  while (top > 0) {
    const int take = top < 64 ? top : 64;
    const int base = top - take;
    const int node = l < take ? stk[base + l] : -1;
    __builtin_amdgcn_wave_barrier();
    top = base;
    bool leaf = false, inner = false;
    int child = 0;
    if (node >= 0) {
      const ObbNode a = nodes[node];
      ++tests;
      if (obbOverlapF(Rq, Tq, a, sb, kObbScaleErr)) {
        child = a.child;
        leaf = child < 0;
        inner = child >= 0;
      }
    }
    const unsigned long long lm = __ballot(leaf);
    if (lm) {
      unsigned long long b0 = 0;
      if (l == 0) b0 = atomicAdd(A.cand_count, static_cast<unsigned long long>(__popcll(lm)));
      b0 = __shfl(b0, 0);
      if (leaf) {
        const uint64_t slot = b0 + __popcll(lm & below);
        if (slot < A.cand_cap) A.cand[slot] = (q << 32) | static_cast<uint32_t>(-(child + 1));
        ++leaves;
      }
    }
    const unsigned long long pm = __ballot(inner);
    const int total = 2 * __popcll(pm);
    if (top + total > kMsStack) {  // uniform: every lane sees the same counts
      ovf = true;
      break;
    }
    if (inner) {
      const int r = 2 * __popcll(pm & below);
      stk[top + r] = child;
      stk[top + r + 1] = child + 1;
    }
    top += total;
    __builtin_amdgcn_wave_barrier();
  }
  for (int off = 32; off > 0; off >>= 1) {
    tests += __shfl_xor(tests, off);
    leaves += __shfl_xor(leaves, off);
  }
  if (l == 0) {
    A.bv_tests[q] = tests;
    A.leaves[q] = leaves;
    A.overflow[q] = ovf ? 1u : 0u;
  }
}

#pragma clang fp contract(off)
// sphere_triangle-inl.h:52-74
MFCL_D double segSqrDist(d3 from, d3 to, d3 p, d3& nearest) {
  d3 diff = p - from;
  const d3 v = to - from;
  double t = dot(v, diff);
  if (t > 0) {
    const double vv = dot(v, v);
    if (t < vv) {
      t /= vv;
      diff = diff - v * t;
    } else {
      t = 1;
      diff = diff - v;
    }
  } else {
    t = 0;
  }
  nearest = from + v * t;
  return dot(diff, diff);
}

// sphere_triangle-inl.h:107-187: sphere of radius r centred at c against
// the world triangle (P1, P2, P3).  c_out (optional) receives the contact as
// the reference writes it: pos = the nearest point found, normal = that
// point minus the centre, normalised (the flipped plane normal when they
// coincide), depth = -(r - distance) (-r when they coincide).
struct SphereTriContact {
  d3 pos, normal;
  double depth;
};
MFCL_D bool sphereTriContact(double r, d3 c, d3 P1, d3 P2, d3 P3, SphereTriContact* c_out) {
  d3 n = cross(P2 - P1, P3 - P1);
  const double nn = norm(n);
  if (nn > 0) n = n / nn;
  const double rt = r + 2.220446049250313e-16;
  double dist = dot(c - P1, n);
  if (dist < 0) {
    dist *= -1;
    n = n * -1.0;
  }
  if (!(dist < rt)) return false;
  bool has = false;
  d3 cp = {0, 0, 0};
  const double r1 = dot(cross(P2 - P1, n), c - P1);
  const double r2 = dot(cross(P3 - P2, n), c - P2);
  const double r3 = dot(cross(P1 - P3, n), c - P3);
  if ((r1 > 0 && r2 > 0 && r3 > 0) || (r1 <= 0 && r2 <= 0 && r3 <= 0)) {
    has = true;
    cp = c - n * dist;
  } else {
    const double cr2 = rt * rt;
    d3 q;
    if (segSqrDist(P1, P2, c, q) < cr2) { has = true; cp = q; }
    if (segSqrDist(P2, P3, c, q) < cr2) { has = true; cp = q; }
    if (segSqrDist(P3, P1, c, q) < cr2) { has = true; cp = q; }
  }
  if (!has) return false;
  const d3 d = cp - c;
  const double d2 = dot(d, d);
  if (!(d2 < rt * rt)) return false;
  if (c_out) {
    c_out->pos = cp;
    if (d2 > 0) {
      c_out->normal = normalized(d);
      c_out->depth = -(r - sqrt(d2));
    } else {
      c_out->normal = n * -1.0;
      c_out->depth = -r;
    }
  }
  return true;
}
MFCL_D bool sphereTriHit(double r, d3 c, d3 P1, d3 P2, d3 P3) { return sphereTriContact(r, c, P1, P2, P3, nullptr); }

// box_triangle-inl.h:9-69
MFCL_D bool sepEdgeAxes(const double h[3], d3 e0, d3 v0, d3 v1) {
  const double ax = fabs(e0.x), ay = fabs(e0.y), az = fabs(e0.z);
  auto sep = [](double p0, double p1, double rad) {
    if (p0 < p1) return p0 > rad || p1 < -rad;
    return p1 > rad || p0 < -rad;
  };
  if (sep(v0.y * e0.z - v0.z * e0.y, v1.y * e0.z - v1.z * e0.y, h[1] * az + h[2] * ay)) return true;
  if (sep(v0.x * e0.z - v0.z * e0.x, v1.x * e0.z - v1.z * e0.x, h[0] * az + h[2] * ax)) return true;
  if (sep(v0.x * e0.y - v0.y * e0.x, v1.x * e0.y - v1.y * e0.x, h[0] * ay + h[1] * ax)) return true;
  return false;
}

MFCL_D void minMax3(double a, double b, double c, double& mn, double& mx) {
  mn = mx = a;
  if (b < mn) mn = b;
  if (b > mx) mx = b;
  if (c < mn) mn = c;
  if (c > mx) mx = c;
}

// box_triangle-inl.h:72-137: box of full sides s posed ts against the
// triangle (P1, P2, P3) posed tm.
MFCL_D bool boxTriHit(double s0, double s1, double s2, const tf3& ts, const tf3& tm, d3 P1, d3 P2, d3 P3) {
  const tf3 t = relTf(ts, tm);
  const d3 v0 = apply(t, P1), v1 = apply(t, P2), v2 = apply(t, P3);
  const double h[3] = {0.5 * s0, 0.5 * s1, 0.5 * s2};
  double mn, mx;
  minMax3(v0.x, v1.x, v2.x, mn, mx);
  if (mx < -h[0] || mn > h[0]) return false;
  minMax3(v0.y, v1.y, v2.y, mn, mx);
  if (mx < -h[1] || mn > h[1]) return false;
  minMax3(v0.z, v1.z, v2.z, mn, mx);
  if (mx < -h[2] || mn > h[2]) return false;
  const d3 e0 = v1 - v0;
  if (sepEdgeAxes(h, e0, v0, v2)) return false;
  const d3 e1 = v2 - v1;
  if (sepEdgeAxes(h, e1, v1, v0)) return false;
  const d3 e2 = v0 - v2;
  if (sepEdgeAxes(h, e2, v0, v1)) return false;
  const d3 n = cross(e0, e1);
  const double nv[3] = {n.x, n.y, n.z}, pv[3] = {v0.x, v0.y, v0.z};
  double pmin[3], pmax[3];
  for (int i = 0; i < 3; ++i) {
    if (nv[i] > 0.0) {
      pmin[i] = -h[i] - pv[i];
      pmax[i] = h[i] - pv[i];
    } else {
      pmin[i] = h[i] - pv[i];
      pmax[i] = -h[i] - pv[i];
    }
  }
  return dot(n, d3{pmin[0], pmin[1], pmin[2]}) <= 0 && dot(n, d3{pmax[0], pmax[1], pmax[2]}) >= 0;
}

// A candidate's query, triangle and poses.
struct MsItem {
  uint64_t q;
  uint32_t t, shp;
  tf3 tm, ts;
  const float4* tri;
  d3 P1, P2, P3;
};
MFCL_D MsItem msItem(const MeshShapeArgs& A, uint64_t k) {
  MsItem m;
  const uint64_t c = A.cand[k];
  m.q = c >> 32;
  m.t = static_cast<uint32_t>(c & 0xFFFFFFFFull);
  m.shp = A.shape_ids[m.q];
  m.tm = poseFromQuat(A.pose_m + 7 * m.q);
  m.ts = poseFromQuat(A.pose_s + 7 * m.q);
  m.tri = A.tris + 3 * (static_cast<uint64_t>(A.tri_base[A.mesh_ids[m.q]]) + m.t);
  m.P1 = d3{m.tri[0].x, m.tri[0].y, m.tri[0].z};
  m.P2 = d3{m.tri[1].x, m.tri[1].y, m.tri[1].z};
  m.P3 = d3{m.tri[2].x, m.tri[2].y, m.tri[2].z};
  return m;
}
// The wavefront's Minkowski difference of (shape, triangle).
MFCL_D void msCfg(const MeshShapeArgs& A, const MsItem& m, MFCL_LDS WaveCfg* cfg, d3 int0, d3 int1) {
  DevShape B;
  B.type = kTriangle;
  B.p0 = B.p1 = B.p2 = 0;
  B.verts = m.tri;
  B.nv = 3;
  B.rbound = 0.f;
  B.nbr = nullptr;
  B.seed = nullptr;
  B.wblk = nullptr;
  waveCfgSet(cfg, loadShape(A.T, m.shp), m.ts, B, m.tm, int0, int1);
}

// Leaf tests: each wavefront takes `chunk` consecutive candidates; its lanes
// run the spheres' and boxes' closed forms together, then the wavefront the
// others' MPR one after the other.
MFCL_D void msHit(const MeshShapeArgs& A, uint64_t q, uint32_t t) {
  const uint32_t slot = atomicAdd(&A.counts[q], 1u);
  if (static_cast<int>(slot) < A.max_contacts)
    A.tri_out[q * static_cast<uint64_t>(A.max_contacts) + slot] = static_cast<int32_t>(t);
}
__global__ void __launch_bounds__(256) msLeafKernel(MeshShapeArgs A, uint64_t ncand, int chunk) {
  __shared__ WaveCfg cfgs[4];
  MFCL_LDS WaveCfg* cfg = (MFCL_LDS WaveCfg*)(&cfgs[threadIdx.x >> 6]);
  const int lane = threadIdx.x & 63;
  const uint64_t base = ((static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x) >> 6) * chunk;
  bool search = false;
  if (lane < chunk && base + lane < ncand) {
    const MsItem m = msItem(A, base + lane);
    const DevShape S = loadShape(A.T, m.shp);
    if (S.type == kSphere) {
      if (sphereTriHit(S.p0, m.ts.t, apply(m.tm, m.P1), apply(m.tm, m.P2), apply(m.tm, m.P3))) msHit(A, m.q, m.t);
    } else if (S.type == kBox) {
      if (boxTriHit(S.p0, S.p1, S.p2, m.ts, m.tm, m.P1, m.P2, m.P3)) msHit(A, m.q, m.t);
    } else {
      search = true;
    }
  }
  for (unsigned long long todo = __ballot(search); todo; todo &= todo - 1) {
    const MsItem m = msItem(A, base + __builtin_ctzll(todo));
    d3 int0 = {0, 0, 0};
    if (A.T.type[m.shp] == kConvex) {
      const double4 ci = A.interior[m.shp];
      int0 = d3{ci.x, ci.y, ci.z};
    }
    msCfg(A, m, cfg, int0, (m.P1 + m.P2 + m.P3) / 3.0);
    MinkW md{cfg, 0};
    const bool hit = mprIntersect(md, A.gjk_max_it, A.gjk_tol) == kMprIntersect;
    if (hit && lane == 0) msHit(A, m.q, m.t);
  }
}

// Penetration enabled (shapeTriangleIntersect with contact outputs,
// gjk_solver-inl.h:545-563).  Spheres take sphereTriContact, one per lane;
// every other shape runs GJK from -UnitX and EPA on (shape, triangle)
// (gjk_solver-inl.h:452-527), one per wavefront, the EPA polytope in the
// wavefront's LDS slice (cap_faces faces); pairs that might outgrow it
// continue (or, out of dump slots, restart) at the request's capacity in a
// second launch.  A hit records the contact with the traversal's normal
// reversal (bvh_solver-inl.h:55-65, shape_pair_intersect-inl.h:19-26): b1 =
// the triangle, b2 = -1.
struct MsPen {
  mfcl_mesh_contact* out;  // n * max_contacts: in the order of arrival, then by triangle
  int cap_faces;           // LDS polytope capacity
  size_t slice_bytes;      // LDS bytes per wavefront
  char* dumps;             // pairs to continue
  uint32_t n_dumps;
  size_t dump_bytes;
  uint32_t* redo;          // pairs to restart
  uint32_t* cnt;           // MsCount
  char* arena;             // device-memory polytopes, one per block of the full-capacity pass (null: in LDS)
  size_t arena_slice;
  int epa_max_faces, epa_max_it;
  double epa_tol;
};
enum MsCount : int { kMsNext = 0, kMsDumps = 1, kMsRedo = 2, kMsFullNext = 3, kMsCounts = 8 };

MFCL_D void msContact(const MeshShapeArgs& A, const MsPen& E, uint64_t q, uint32_t t, d3 pos, d3 nrm, double depth) {
  const uint32_t slot = atomicAdd(&A.counts[q], 1u);
  if (static_cast<int>(slot) >= A.max_contacts) return;
  mfcl_mesh_contact& o = E.out[q * static_cast<uint64_t>(A.max_contacts) + slot];
  o.b1 = static_cast<int32_t>(t);
  o.b2 = -1;
  o.pos[0] = pos.x; o.pos[1] = pos.y; o.pos[2] = pos.z;
  o.normal[0] = -nrm.x; o.normal[1] = -nrm.y; o.normal[2] = -nrm.z;
  o.depth = depth;
}
// The contact of a pair whose EPA ended with `status` (lane 0 writes).
MFCL_D void msEpaContact(const MeshShapeArgs& A, const MsPen& E, const MsItem& m, const MFCL_LDS EpaLds* L, int status) {
  if (status == kEpaFailed || __lane_id() != 0) return;
  const d3 p0 = ldsGet(L->out.p0), p1 = ldsGet(L->out.p1);
  d3 n1 = p0 - p1;
  n1 = sqnorm(n1) <= 0 ? d3{0, 0, 1} : normalized(n1);
  msContact(A, E, m.q, m.t, apply(m.ts, 0.5 * (p0 + p1)), mul(m.ts.R, n1), L->out.depth);
}
// GJK of the configuration in L; the simplex into L->s when it intersects.
MFCL_D bool msGjk(const MeshShapeArgs& A, MFCL_LDS EpaLds* L) {
  MinkW md{&L->cfg, 0};
  Smp s;
  smpInit(s);
  GjkOut g;
  gjkEvaluate(md, s, d3{-1, 0, 0}, A.gjk_tol, A.gjk_max_it, false, g);
  if (__builtin_amdgcn_readfirstlane(g.status) != kGjkIntersect) return false;
  L->s.rank = s.rank;
  ldsSet(L->s.a.v, s.a.v); ldsSet(L->s.a.d, md.dirOf(static_cast<int>(s.a.id)));
  ldsSet(L->s.b.v, s.b.v); ldsSet(L->s.b.d, md.dirOf(static_cast<int>(s.b.id)));
  ldsSet(L->s.c.v, s.c.v); ldsSet(L->s.c.d, md.dirOf(static_cast<int>(s.c.id)));
  ldsSet(L->s.e.v, s.e.v); ldsSet(L->s.e.d, md.dirOf(static_cast<int>(s.e.id)));
  return true;
}

__global__ void __launch_bounds__(256, 3) msPenKernel(MeshShapeArgs A, MsPen E, uint64_t ncand, int chunk) {
  extern __shared__ __align__(16) char ms_lds[];
  MFCL_LDS EpaLds* L = (MFCL_LDS EpaLds*)((MFCL_LDS char*)(ms_lds) + (threadIdx.x >> 6) * E.slice_bytes);
  const int lane = threadIdx.x & 63;
  const uint64_t base = ((static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x) >> 6) * chunk;
  bool search = false;
  if (lane < chunk && base + lane < ncand) {
    const MsItem m = msItem(A, base + lane);
    if (A.T.type[m.shp] == kSphere) {
      SphereTriContact sc;
      if (sphereTriContact(A.T.param[m.shp].x, m.ts.t, apply(m.tm, m.P1), apply(m.tm, m.P2), apply(m.tm, m.P3), &sc))
        msContact(A, E, m.q, m.t, sc.pos, sc.normal, sc.depth);
    } else {
      search = true;
    }
  }
  for (unsigned long long todo = __ballot(search); todo; todo &= todo - 1) {
    const uint64_t k = base + __builtin_ctzll(todo);
    msCfg(A, msItem(A, k), &L->cfg, d3{0, 0, 0}, d3{0, 0, 0});
    if (!msGjk(A, L)) continue;
    const int st = epaRun<SmallMem>(L, ldsArena(L), E.cap_faces, E.epa_tol, E.epa_max_it, E.cap_faces < E.epa_max_faces,
                                    false);
    if (st != kEpaSpill) {
      msEpaContact(A, E, msItem(A, k), L, st);
      continue;
    }
    uint32_t slot = 0;
    if (lane == 0) slot = atomicAdd(E.cnt + kMsDumps, 1u);
    slot = __builtin_amdgcn_readfirstlane(slot);
    if (slot < E.n_dumps) epaDump(E.dumps + slot * E.dump_bytes, L, E.cap_faces, static_cast<int>(k));
    else if (lane == 0) E.redo[atomicAdd(E.cnt + kMsRedo, 1u)] = static_cast<uint32_t>(k);
  }
}

template <class M>
__global__ void __launch_bounds__(64) msPenFullKernel(MeshShapeArgs A, MsPen E) {
  extern __shared__ __align__(16) char ms_lds[];
  MFCL_LDS EpaLds* L = (MFCL_LDS EpaLds*)((MFCL_LDS char*)(ms_lds));
  typename M::template P<char> arena;
  if constexpr (std::is_same<M, GlobalMem>::value) arena = E.arena + blockIdx.x * E.arena_slice;
  else arena = ldsArena(L);
  const uint32_t asked = E.cnt[kMsDumps];
  const uint32_t dumps = asked < E.n_dumps ? asked : E.n_dumps, count = dumps + E.cnt[kMsRedo];
  for (;;) {
    uint32_t i = 0;
    if (threadIdx.x == 0) i = atomicAdd(E.cnt + kMsFullNext, 1u);
    i = __builtin_amdgcn_readfirstlane(i);
    if (i >= count) break;
    const bool resume = i < dumps;
    const char* dump = E.dumps + i * E.dump_bytes;
    const uint32_t k = __builtin_amdgcn_readfirstlane(resume ? static_cast<uint32_t>(epaDumpItem(dump)) : E.redo[i - dumps]);
    const MsItem m = msItem(A, k);
    msCfg(A, m, &L->cfg, d3{0, 0, 0}, d3{0, 0, 0});
    if (resume) epaLoad<M>(L, arena, E.epa_max_faces, dump, E.cap_faces);
    else if (!msGjk(A, L)) continue;
    const int st = epaRun<M>(L, arena, E.epa_max_faces, E.epa_tol, E.epa_max_it, false, resume);
    msEpaContact(A, E, msItem(A, k), L, st);
  }
}

// Result headers, one wavefront per query.  Kept triangles (contacts) move
// from the order of arrival to ascending triangle ids, in place: a triangle's
// place is the number of smaller ids (each triangle is a candidate once).
MFCL_D int msHeader(const MeshShapeArgs& A, uint64_t q, mfcl_mesh_result* out) {
  const uint32_t cnt = A.counts[q];
  const int kept = static_cast<int>(cnt) < A.max_contacts ? static_cast<int>(cnt) : A.max_contacts;
  if (threadIdx.x == 0) {
    mfcl_mesh_result r;
    r.hit = A.overflow[q] ? -1 : (cnt > 0 ? 1 : 0);
    r.n_contacts = kept;
    r.bv_tests = static_cast<int32_t>(A.bv_tests[q]);
    r.leaf_tests = static_cast<int32_t>(A.leaves[q]);
    out[q] = r;
  }
  return kept;
}
constexpr int kMsMaxContacts = 1024;
MFCL_D int msPlace(const MFCL_LDS int32_t* ids, int kept, int32_t id) {
  int r = 0;
  for (int j = 0; j < kept; ++j) r += ids[j] < id;
  return r;
}
// LDS: the kept records (eight 8-byte words each), their triangles, their places.
constexpr size_t kMsFinishBytes = sizeof(mfcl_mesh_contact) + 2 * sizeof(int32_t);  // a record
__global__ void __launch_bounds__(64) msFinishPenKernel(MeshShapeArgs A, mfcl_mesh_contact* contacts,
                                                        mfcl_mesh_result* out) {
  extern __shared__ __align__(16) char ms_lds[];
  static_assert(sizeof(mfcl_mesh_contact) == 64, "eight words");
  MFCL_LDS uint64_t* rec = (MFCL_LDS uint64_t*)(ms_lds);
  MFCL_LDS int32_t* ids = (MFCL_LDS int32_t*)(rec + 8 * A.max_contacts);
  MFCL_LDS int32_t* place = ids + A.max_contacts;
  const uint64_t q = blockIdx.x;
  const int kept = msHeader(A, q, out), l = threadIdx.x;
  uint64_t* w = reinterpret_cast<uint64_t*>(contacts + q * static_cast<uint64_t>(A.max_contacts));
  for (int i = l; i < 8 * kept; i += 64) {
    const uint64_t v = w[i];
    rec[i] = v;
    if (i % 8 == 0) ids[i / 8] = static_cast<int32_t>(v);  // b1
  }
  __syncthreads();
  for (int i = l; i < kept; i += 64) place[i] = msPlace(ids, kept, ids[i]);
  __syncthreads();
  for (int i = l; i < 8 * kept; i += 64) w[8 * place[i / 8] + i % 8] = rec[i];
  // the others: b1 = b2 = -1, zeros
  for (int i = 8 * kept + l; i < 8 * A.max_contacts; i += 64) w[i] = i % 8 == 0 ? ~0ull : 0ull;
}

__global__ void __launch_bounds__(64) msFinishKernel(MeshShapeArgs A, mfcl_mesh_result* out) {
  __shared__ int32_t lds_ids[kMsMaxContacts];
  MFCL_LDS int32_t* ids = (MFCL_LDS int32_t*)(lds_ids);
  const uint64_t q = blockIdx.x;
  const int kept = msHeader(A, q, out), l = threadIdx.x;
  int32_t* o = A.tri_out + q * static_cast<uint64_t>(A.max_contacts);
  for (int i = l; i < kept; i += 64) ids[i] = o[i];
  __syncthreads();
  for (int i = l; i < kept; i += 64) o[msPlace(ids, kept, ids[i])] = ids[i];
  for (int i = kept + l; i < A.max_contacts; i += 64) o[i] = -1;
}

__global__ void msZeroKernel(uint32_t* p, uint64_t n) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// Dump slots and blocks of the full-capacity pass.
constexpr uint32_t kMsDumpSlots = 2048, kMsFullBlocks = 512;

namespace {
// Device memory of one call.
struct DevTemp {
  void* p{nullptr};
  ~DevTemp() {
    if (p) (void)hipFree(p);
  }
};
// A call's workspaces stay with the context for the next call, up to this
// much each; what a call grew beyond it is given back at its end.
constexpr size_t kMsKeepBytes = 256ull << 20;
struct GiveBack {
  DevBuf& b;
  const size_t before;
  explicit GiveBack(DevBuf& buf) : b(buf), before(buf.bytes) {}
  ~GiveBack() {
    if (b.bytes <= kMsKeepBytes || b.bytes <= before) return;
    (void)hipFree(b.p);
    b = DevBuf();
  }
};
}  // namespace

int meshShapeCollide(mfcl_ctx* ctx, const uint32_t* mesh_ids, const uint32_t* shape_ids, const float* pose_m7,
                     const float* pose_s7, uint64_t n, const mfcl_request* req, mfcl_mesh_result* out,
                     int32_t* tri_ids, mfcl_mesh_contact* contacts) {
  if (ctx->n_meshes == 0 || ctx->n_shapes == 0) {
    ctx->err = "mesh-shape collision needs uploaded meshes and shapes";
    return MFCL_E_STATE;
  }
  const bool pen = req->penetration != 0;
  if (pen != (contacts != nullptr)) {
    ctx->err = pen ? "a penetration-enabled mesh-shape query writes contacts: pass a contact array"
                   : "a contact array needs a request with penetration enabled";
    return MFCL_E_INVALID;
  }
  const int maxc = req->max_contacts;
  if (maxc < 1 || maxc > 1024) {
    ctx->err = "max_contacts must be in [1, 1024]";
    return MFCL_E_INVALID;
  }
  if (pen && (req->epa_max_faces < 4 || req->epa_max_faces > 8192)) {
    ctx->err = "epa_max_faces out of range [4, 8192]";
    return MFCL_E_INVALID;
  }
  for (uint64_t i = 0; i < n; ++i) {
    if (mesh_ids[i] >= ctx->n_meshes || shape_ids[i] >= ctx->n_shapes) {
      ctx->err = "query " + std::to_string(i) + " references a mesh or shape id out of range";
      return MFCL_E_INVALID;
    }
  }
  const hipStream_t s = ctx->stream;
  // the call's buffers, carved from the context's host-call workspace; the
  // candidates, whose number is known only after the tree walk, from a
  // workspace of their own (64 per query, grown to the exact count and
  // rerun); what only some candidates need is sized by their number
  const GiveBack keep_io(ctx->ws_io), keep_cand(ctx->ws_cand);
  const uint64_t slots = n * static_cast<uint64_t>(maxc);
  int lds_faces = std::min(std::min(req->epa_max_faces, 42), kSmallFaces);
  while (lds_faces > 4 && 4 * epaSliceBytes<SmallMem>(lds_faces) > static_cast<size_t>(ctx->max_lds_per_block))
    lds_faces /= 2;
  const bool spills = pen && lds_faces < req->epa_max_faces;
  const bool mid = req->epa_max_faces <= kMidFaces;
  const size_t full_slice =
      mid ? epaSliceBytes<MidMem>(req->epa_max_faces) : epaSliceBytes<LargeMem>(req->epa_max_faces);
  const bool full_lds = full_slice <= static_cast<size_t>(ctx->max_lds_per_block);
  const size_t arena_slice = full_lds ? 0 : arenaBytes<GlobalMem>(req->epa_max_faces);
  const size_t b_out = pen ? sizeof(mfcl_mesh_contact) * slots : 4 * slots;
  const size_t sizes[] = {4 * n, 4 * n, 28 * n, 28 * n, 16 * n, 64, sizeof(mfcl_mesh_result) * n, b_out};
  constexpr int kPieces = sizeof(sizes) / sizeof(sizes[0]);
  size_t total = 0;
  for (size_t b : sizes) total += (b + 255) & ~static_cast<size_t>(255);
  if (int rc = ensure(ctx, ctx->ws_io, total)) return rc;
  char* piece[kPieces];
  {
    char* p = static_cast<char*>(ctx->ws_io.p);
    for (int k = 0; k < kPieces; ++k) {
      piece[k] = p;
      p += (sizes[k] + 255) & ~static_cast<size_t>(255);
    }
  }
  auto* dm = reinterpret_cast<uint32_t*>(piece[0]);
  auto* ds = reinterpret_cast<uint32_t*>(piece[1]);
  auto* dpm = reinterpret_cast<float*>(piece[2]);
  auto* dps = reinterpret_cast<float*>(piece[3]);
  auto* dcnt = reinterpret_cast<uint32_t*>(piece[4]);            // counts, leaves, bv tests, overflow
  auto* dcc = reinterpret_cast<unsigned long long*>(piece[5]);   // candidate count, MsCount
  auto* dout = reinterpret_cast<mfcl_mesh_result*>(piece[6]);
  MFCL_HIP_TRY(ctx, hipMemcpyAsync(dm, mesh_ids, 4 * n, hipMemcpyHostToDevice, s));
  MFCL_HIP_TRY(ctx, hipMemcpyAsync(ds, shape_ids, 4 * n, hipMemcpyHostToDevice, s));
  MFCL_HIP_TRY(ctx, hipMemcpyAsync(dpm, pose_m7, 28 * n, hipMemcpyHostToDevice, s));
  MFCL_HIP_TRY(ctx, hipMemcpyAsync(dps, pose_s7, 28 * n, hipMemcpyHostToDevice, s));
  MeshShapeArgs A;
  A.T = ShapeTables{ctx->d_type, ctx->d_param, ctx->d_voff, ctx->d_vcnt, ctx->d_verts, ctx->d_nbr, ctx->d_nbr_off,
                    ctx->d_seed, ctx->d_wblk};
  A.interior = ctx->d_interior;
  A.nodes = static_cast<const ObbNode*>(ctx->d_nodes);
  A.tris = static_cast<const float4*>(ctx->d_tris);
  A.node_base = ctx->d_mesh_node_base;
  A.tri_base = ctx->d_mesh_tri_base;
  A.mesh_ids = dm;
  A.shape_ids = ds;
  A.pose_m = dpm;
  A.pose_s = dps;
  A.n = n;
  A.counts = dcnt;
  A.leaves = dcnt + n;
  A.bv_tests = dcnt + 2 * n;
  A.overflow = dcnt + 3 * n;
  A.cand_count = dcc;
  A.max_contacts = maxc;
  A.tri_out = reinterpret_cast<int32_t*>(piece[7]);
  A.gjk_max_it = req->gjk_max_iterations;
  A.gjk_tol = req->gjk_tolerance;
  uint64_t cap = std::max<uint64_t>(64 * n, 1 << 16);
  unsigned long long ncand = 0;
  for (int attempt = 0; attempt < 2; ++attempt) {
    // 8 bytes per candidate, then 4 for the restart list
    if (int rc = ensure(ctx, ctx->ws_cand, 12 * cap)) return rc;
    cap = std::max<uint64_t>(cap, ctx->ws_cand.bytes / 12);
    A.cand = static_cast<uint64_t*>(ctx->ws_cand.p);
    A.cand_cap = cap;
    msZeroKernel<<<static_cast<unsigned>((4 * n + 255) / 256), 256, 0, s>>>(dcnt, 4 * n);
    msZeroKernel<<<1, 64, 0, s>>>(reinterpret_cast<uint32_t*>(dcc), 16);
    msCandKernel<<<static_cast<unsigned>(n), 64, 0, s>>>(A);
    MFCL_HIP_TRY(ctx, hipGetLastError());
    MFCL_HIP_TRY(ctx, hipMemcpyAsync(&ncand, dcc, 8, hipMemcpyDeviceToHost, s));
    MFCL_HIP_TRY(ctx, hipStreamSynchronize(s));
    if (ncand <= cap) break;
    cap = ncand;
  }
  if (ncand > cap) {
    ctx->err = "mesh-shape candidate count changed between runs";
    return MFCL_E_STATE;
  }
  if (pen && ncand > 0xF0000000ull) {
    ctx->err = "too many mesh-shape candidates for one penetration-enabled call";
    return MFCL_E_INVALID;
  }
  // as many candidates per wavefront as leave the chip filled a few times
  const uint64_t waves = 64ull * static_cast<uint64_t>(ctx->n_cu);
  const int chunk = static_cast<int>(std::min<uint64_t>(64, (ncand + waves - 1) / waves));
  const unsigned blocks = chunk ? static_cast<unsigned>((ncand + 4ull * chunk - 1) / (4ull * chunk)) : 0;
  if (!pen) {
    if (ncand) msLeafKernel<<<blocks, 256, 0, s>>>(A, ncand, chunk);
    msFinishKernel<<<static_cast<unsigned>(n), 64, 0, s>>>(A, dout);
    MFCL_HIP_TRY(ctx, hipGetLastError());
    MFCL_HIP_TRY(ctx, hipMemcpyAsync(out, dout, sizeof(mfcl_mesh_result) * n, hipMemcpyDeviceToHost, s));
    if (tri_ids) MFCL_HIP_TRY(ctx, hipMemcpyAsync(tri_ids, A.tri_out, 4 * slots, hipMemcpyDeviceToHost, s));
    MFCL_HIP_TRY(ctx, hipStreamSynchronize(s));
    return MFCL_OK;
  }
  MsPen E;
  E.epa_max_faces = req->epa_max_faces;
  E.epa_max_it = req->epa_max_iterations;
  E.epa_tol = req->epa_tolerance;
  E.cap_faces = lds_faces;
  E.slice_bytes = epaSliceBytes<SmallMem>(lds_faces);
  E.out = reinterpret_cast<mfcl_mesh_contact*>(piece[7]);
  E.n_dumps = spills ? static_cast<uint32_t>(std::min<uint64_t>(kMsDumpSlots, ncand)) : 0;
  E.dump_bytes = epaDumpBytes(lds_faces);
  if (E.n_dumps)
    if (int rc = ensure(ctx, ctx->ws_dump, E.n_dumps * E.dump_bytes)) return rc;
  E.dumps = static_cast<char*>(ctx->ws_dump.p);
  const unsigned fb = static_cast<unsigned>(std::min<uint64_t>(kMsFullBlocks, ncand));
  DevTemp arena;
  if (spills && !full_lds && fb && hipMalloc(&arena.p, arena_slice * fb) != hipSuccess) {
    (void)hipGetLastError();
    ctx->err = "out of device memory for the mesh-shape EPA polytopes";
    return MFCL_E_NOMEM;
  }
  E.redo = reinterpret_cast<uint32_t*>(A.cand + cap);
  E.cnt = reinterpret_cast<uint32_t*>(dcc) + 2;
  E.arena = static_cast<char*>(arena.p);
  E.arena_slice = arena_slice;
  if (ncand) {
    msPenKernel<<<blocks, 256, 4 * E.slice_bytes, s>>>(A, E, ncand, chunk);
    if (spills && full_lds && mid) msPenFullKernel<MidMem><<<fb, 64, full_slice, s>>>(A, E);
    else if (spills && full_lds) msPenFullKernel<LargeMem><<<fb, 64, full_slice, s>>>(A, E);
    else if (spills) msPenFullKernel<GlobalMem><<<fb, 64, kEpaHeadBytes, s>>>(A, E);
  }
  msFinishPenKernel<<<static_cast<unsigned>(n), 64, kMsFinishBytes * maxc, s>>>(A, E.out, dout);
  MFCL_HIP_TRY(ctx, hipGetLastError());
  MFCL_HIP_TRY(ctx, hipMemcpyAsync(out, dout, sizeof(mfcl_mesh_result) * n, hipMemcpyDeviceToHost, s));
  MFCL_HIP_TRY(ctx, hipMemcpyAsync(contacts, E.out, sizeof(mfcl_mesh_contact) * slots, hipMemcpyDeviceToHost, s));
  MFCL_HIP_TRY(ctx, hipStreamSynchronize(s));
  return MFCL_OK;
}

}  // namespace mfcl
