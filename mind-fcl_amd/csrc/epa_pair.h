// EPA of a convex query's pair: the polytope in the wavefront's LDS slice,
// pairs that outgrow it handed to the full-capacity pass, the result record.
#pragma once

#include "epa_dev.h"
#include "pair_dev.h"

namespace mfcl {

// Where pairs that outgrow their LDS polytope go: to one of n_dumps records
// in device memory (they continue), else to the restart queue.
struct EpaSink {
  char* dumps;
  uint32_t n_dumps;
  size_t dump_bytes;
  QEntry* oflow;
  uint32_t* cnt;  // EpaCounts
};

// The pair's poses and shapes into the slice's configuration.
MFCL_D void epaCfg(const ShapeTables& T, const PairIO& io, uint32_t i, MFCL_LDS EpaLds* L) {
  const tf3 ta = poseFromQuat(io.posea + 7 * static_cast<uint64_t>(i));
  const tf3 tb = poseFromQuat(io.poseb + 7 * static_cast<uint64_t>(i));
  waveCfgSet(&L->cfg, loadShape(T, io.pa[i]), ta, loadShape(T, io.pb[i]), tb, d3{0, 0, 0}, d3{0, 0, 0});
}

// The result of pair i's EPA (lane 0 writes; the other fields of the record
// were written by GJK).
MFCL_D void epaStore(const PairIO& io, const Params& P, uint32_t i, const MFCL_LDS EpaLds* L, int status) {
  if (__lane_id() != 0) return;
  const tf3 ta = poseFromQuat(io.posea + 7 * static_cast<uint64_t>(i));
  const MFCL_LDS EpaOut& o = L->out;
  mfcl_convex_result& r = io.out[i];
  r.epa_status = static_cast<int8_t>(status);
  r.epa_iters = sat16(o.iters);
  if (status == kEpaFailed) {
    r.hit = 0;
    r.ok = 0;
    return;
  }
  r.hit = 1;
  r.ok = 1;
  const d3 p0 = ldsGet(o.p0), p1 = ldsGet(o.p1);
  r.depth = o.depth;
  r.distance = -o.depth;
  if (P.mode == MFCL_MODE_COLLIDE) {
    // gjk_solver-inl.h:117-129
    d3 n1 = p0 - p1;
    n1 = sqnorm(n1) <= 0 ? d3{0, 0, 1} : normalized(n1);
    const d3 pt = 0.5 * (p0 + p1);
    r.n_contacts = 1;
    const d3 nw = mul(ta.R, n1), pw = apply(ta, pt);
    r.normal[0] = nw.x; r.normal[1] = nw.y; r.normal[2] = nw.z;
    r.pos[0] = pw.x; r.pos[1] = pw.y; r.pos[2] = pw.z;
    if (io.contacts) storeContact(io.contacts + static_cast<uint64_t>(i) * io.cstride, nw, pw, o.depth);
  } else {
    const d3 wa = apply(ta, p0), wb = apply(ta, p1);
    r.pa[0] = wa.x; r.pa[1] = wa.y; r.pa[2] = wa.z;
    r.pb[0] = wb.x; r.pb[1] = wb.y; r.pb[2] = wb.z;
  }
}

// EPA of pair i, configuration and simplex in L.  Returns the hull vertices
// scanned.  A status MallocFailed of a pair that may spill is final: its
// capacity sufficed (an expansion that might not fit spills before it), so
// it comes from a border that is not a loop, which no capacity mends.
MFCL_D int epaPair(const PairIO& io, const Params& P, uint32_t i, MFCL_LDS EpaLds* L, int cap_faces,
                   const EpaSink& sink) {
  const int st = epaRun<SmallMem>(L, ldsArena(L), cap_faces, P.epa_tol, P.epa_max_it, cap_faces < P.epa_max_faces, false);
  if (st != kEpaSpill) {
    epaStore(io, P, i, L, st);
    return L->out.scanned;
  }
  const int l = __lane_id();
  uint32_t slot = 0;
  if (l == 0) slot = atomicAdd(sink.cnt + kCntDumps, 1u);
  slot = __builtin_amdgcn_readfirstlane(slot);
  if (slot < sink.n_dumps) {
    if (l == 0) atomicAdd(sink.cnt + kCntSpilled, 1u);
    epaDump(sink.dumps + slot * sink.dump_bytes, L, cap_faces, static_cast<int>(i));
  } else {
    uint32_t o = 0;
    if (l == 0) o = atomicAdd(sink.cnt + kCntRestart, 1u);
    o = __builtin_amdgcn_readfirstlane(o);
    QEntry* q = sink.oflow + o;
    copyOut(reinterpret_cast<char*>(&q->s), (const MFCL_LDS char*)(&L->s), sizeof(SmpD));
    q->pair = i;
  }
  return L->out.scanned;
}

inline EpaSink epaSink(const mfcl_ctx* ctx, const ConvexJob& j, int cap_faces) {
  EpaSink k;
  k.dump_bytes = epaDumpBytes(cap_faces);
  k.dumps = j.arena;
  k.n_dumps = j.arena && ctx->tune.epa_spill ? static_cast<uint32_t>(j.arena_bytes / k.dump_bytes) : 0;
  k.oflow = j.oflow;
  k.cnt = j.qcount;
  return k;
}

// One atomic per wavefront (v identical in all lanes).
MFCL_D void addScanned(unsigned long long* total, int v) {
  if (__lane_id() == 0 && v) atomicAdd(total, static_cast<unsigned long long>(v));
}

}  // namespace mfcl
