// What the kernels of a convex query share: the pair inputs and results, the
// EPA queue entry, the closed forms' dispatch.
#pragma once

#include "ctx.h"
#include "narrow_dev.h"
#include "prim_dev.h"

namespace mfcl {

constexpr int kBlock = 256;
constexpr int kModeBool = 0, kModePen = 1, kModeSd = 2;

struct PairIO {
  const uint32_t* pa;
  const uint32_t* pb;
  const float* posea;
  const float* poseb;
  const float* guess;
  mfcl_convex_result* out;
  mfcl_contact* contacts;  // optional: cstride records per pair
  int cstride;             // min(max_contacts, 4) when contacts is set
};

struct QEntry {
  SmpD s;
  uint32_t pair;
  uint32_t pad;
};

struct Params {
  int mode, max_contacts, penetration, gjk_max_it, epa_max_faces, epa_max_it, use_guess;
  uint32_t n_shapes;
  double gjk_tol, epa_tol;
};

MFCL_D bool closedForm(int ta, int tb) {
  if (ta == kSphere && (tb == kSphere || tb == kCapsule || tb == kBox || tb == kCylinder)) return true;
  if (tb == kSphere && (ta == kCapsule || ta == kBox || ta == kCylinder)) return true;
  return ta == kBox && tb == kBox;
}

MFCL_D void clearResult(mfcl_convex_result& r) {
  r.hit = 0;
  r.n_contacts = 0;
  r.method = 0;
  r.gjk_status = -1;
  r.epa_status = -1;
  r.ok = 0;
  r.gjk_iters = 0;
  r.epa_iters = 0;
  r.distance = 0;
  r.depth = 0;
  r.normal[0] = r.normal[1] = r.normal[2] = 0;
  r.pos[0] = r.pos[1] = r.pos[2] = 0;
  r.pa[0] = r.pa[1] = r.pa[2] = 0;
  r.pb[0] = r.pb[1] = r.pb[2] = 0;
}

// Result fields gathered in registers and stored once.
struct ResAcc {
  d3 normal, pos, pa, pb;
};
MFCL_D void storeResult(mfcl_convex_result* dst, const mfcl_convex_result& r, const ResAcc& x) {
  mfcl_convex_result o = r;
  o.normal[0] = x.normal.x; o.normal[1] = x.normal.y; o.normal[2] = x.normal.z;
  o.pos[0] = x.pos.x; o.pos[1] = x.pos.y; o.pos[2] = x.pos.z;
  o.pa[0] = x.pa.x; o.pa[1] = x.pa.y; o.pa[2] = x.pa.z;
  o.pb[0] = x.pb.x; o.pb[1] = x.pb.y; o.pb[2] = x.pb.z;
  *dst = o;
}

MFCL_D uint16_t sat16(int v) { return static_cast<uint16_t>(v > 65535 ? 65535 : v); }

// Closed-form dispatch with the reference's operand swaps and normal flips
// (gjk_solver-inl.h:158-217).  Returns hit; fills contacts if requested.
MFCL_D bool runClosedForm(const DevShape& A, const tf3& ta, const DevShape& B, const tf3& tb, PContacts* pc) {
  const int x = A.type, y = B.type;
  bool hit = false, flip = false;
  if (x == kSphere && y == kSphere) hit = primSphereSphere(A.p0, ta, B.p0, tb, pc);
  else if (x == kBox && y == kBox) hit = primBoxBox(d3{A.p0, A.p1, A.p2}, ta, d3{B.p0, B.p1, B.p2}, tb, pc) != 0;
  else if (x == kSphere && y == kCapsule) hit = primSphereCapsule(A.p0, ta, B.p0, B.p1, tb, pc);
  else if (x == kCapsule && y == kSphere) { hit = primSphereCapsule(B.p0, tb, A.p0, A.p1, ta, pc); flip = true; }
  else if (x == kSphere && y == kBox) hit = primSphereBox(A.p0, ta, d3{B.p0, B.p1, B.p2}, tb, pc);
  else if (x == kBox && y == kSphere) { hit = primSphereBox(B.p0, tb, d3{A.p0, A.p1, A.p2}, ta, pc); flip = true; }
  else if (x == kSphere && y == kCylinder) hit = primSphereCylinder(A.p0, ta, B.p0, B.p1, tb, pc);
  else if (x == kCylinder && y == kSphere) { hit = primSphereCylinder(B.p0, tb, A.p0, A.p1, ta, pc); flip = true; }
  if (flip && pc)
    for (int k = 0; k < pc->n; ++k) pc->c[k].n = -pc->c[k].n;
  return hit;
}

MFCL_D void storeContact(mfcl_contact* dst, const d3& n, const d3& p, double depth) {
  mfcl_contact c;
  c.normal[0] = n.x; c.normal[1] = n.y; c.normal[2] = n.z;
  c.pos[0] = p.x; c.pos[1] = p.y; c.pos[2] = p.z;
  c.depth = depth;
  *dst = c;
}

// Contacts of a colliding closed-form pair into the result: the deepest
// max_contacts when they do not all fit (shape_pair_intersect-inl.h:91-113),
// contact 0 into the record, all kept ones into the contact array.
MFCL_D void finishClosedForm(PContacts& pc, const Params& P, const PairIO& io, uint32_t i, mfcl_convex_result& r,
                             ResAcc& acc, bool writer) {
  int kept = pc.n;
  if (pc.n > P.max_contacts) {
    partialSortDeepest(pc.c, P.max_contacts, pc.n);
    kept = P.max_contacts;
  }
  r.n_contacts = kept;
  if (kept > 0) {
    r.depth = pc.c[0].depth;
    r.distance = -r.depth;
    acc.normal = pc.c[0].n;
    acc.pos = pc.c[0].p;
  }
  if (io.contacts && writer)
    for (int k = 0; k < kept && k < io.cstride; ++k)
      storeContact(io.contacts + static_cast<uint64_t>(i) * io.cstride + k, pc.c[k].n, pc.c[k].p, pc.c[k].depth);
}

// One query on its stream, as the launchers below take it.  misc: the
// workspace's zeroed counters (see carveConvexWs).
struct ConvexJob {
  ShapeTables T;
  const double4* interior;
  PairIO io;
  Params P;
  uint64_t n;
  int mode;                // kModeBool, kModePen, kModeSd
  uint32_t* qcount;        // EPA pairs; the words after it: see EpaCounts
  QEntry* queue;
  QEntry* oflow;
  unsigned long long* sc;  // hull vertices read: GJK / MPR, EPA
  char* arena;
  size_t arena_bytes;
  hipStream_t s;
};
// Words after ConvexJob::qcount.
enum EpaCounts : int {
  kCntQueue = 0,     // EPA pairs
  kCntRestart = 1,   // pairs that restart at full capacity
  kCntNext = 2,      // cursor over the queue
  kCntFullNext = 3,  // cursor of the full-capacity pass
  kCntSpilled = 4,   // pairs that continue at full capacity
  kCntDumps = 5,     // dump slots asked for (may exceed those there are)
  kCntLanes = 8      // the lane kernel's cursor
};

// lane.hip: GJK with one pair per lane, pairs in bucketed order
int laneLaunch(mfcl_ctx* ctx, const ConvexJob& j, const uint32_t* order, double* dirs);
// epa.hip: the queued pairs; then the pairs that outgrew their polytope
int epaQueueLaunch(mfcl_ctx* ctx, const ConvexJob& j);
int epaFullLaunch(mfcl_ctx* ctx, const ConvexJob& j);
// wave.hip: whole pairs, one wavefront each (GJK or MPR, then EPA)
int waveLaunch(mfcl_ctx* ctx, const ConvexJob& j);
// Face capacity of the LDS polytopes for a request.
int epaSmallFaces(const mfcl_ctx* ctx, const Params& P);
// LDS bytes that a request's full-capacity polytope takes.
size_t epaFullBytes(int max_faces);

}  // namespace mfcl
