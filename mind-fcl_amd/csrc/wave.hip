// Whole pairs, one wavefront each: closed form, MPR or GJK, then EPA in the
// same kernel.  For batches too small to fill the chip with one pair per
// lane (a lane's walks and simplex cases then run one after the other, in a
// few wavefronts), and for the boolean mode.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "epa_pair.h"

namespace mfcl {

// GJK (or MPR) of pair i, its configuration in L's; returns whether EPA
// follows (its simplex then is in *smp).
template <int MODE>
MFCL_D bool wavePair(const ShapeTables& T, const double4* interior, const PairIO& io, const Params& P, uint32_t i,
                     MFCL_LDS WaveCfg* cfg, MFCL_LDS SmpD* smp, int& scanned) {
  const uint32_t ia = io.pa[i], ib = io.pb[i];
  {
    const DevShape A = loadShape(T, ia), B = loadShape(T, ib);
    d3 int0 = {0, 0, 0}, int1 = {0, 0, 0};
    if constexpr (MODE == kModeBool) {
      if (A.type == kConvex) { const double4 c = interior[ia]; int0 = d3{c.x, c.y, c.z}; }
      if (B.type == kConvex) { const double4 c = interior[ib]; int1 = d3{c.x, c.y, c.z}; }
    }
    waveCfgSet(cfg, A, poseFromQuat(io.posea + 7 * static_cast<uint64_t>(i)), B,
               poseFromQuat(io.poseb + 7 * static_cast<uint64_t>(i)), int0, int1);
  }
  mfcl_convex_result r;
  clearResult(r);
  ResAcc acc;
  acc.normal = acc.pos = acc.pa = acc.pb = d3{0, 0, 0};
  MinkW md{cfg, 0};
  bool queued = false, decided = false;
  r.method = 1;
  if constexpr (MODE == kModeBool) {
    r.method = 2;
    const int m = __builtin_amdgcn_readfirstlane(mprIntersect(md, P.gjk_max_it, P.gjk_tol));
    if (m != kMprFailed) {
      r.hit = m == kMprIntersect;
      r.n_contacts = r.hit;
      r.ok = 1;
      decided = true;
    }
  }
  if (!decided) {
    d3 guess = {1, 0, 0};
    if (P.use_guess) guess = d3{io.guess[3ull * i], io.guess[3ull * i + 1], io.guess[3ull * i + 2]};
    Smp s;
    smpInit(s);
    GjkOut g;
    gjkEvaluate(md, s, -guess, P.gjk_tol, P.gjk_max_it, MODE == kModeSd, g);
    const int status = __builtin_amdgcn_readfirstlane(g.status);
    r.gjk_status = static_cast<int8_t>(status);
    if constexpr (MODE == kModeSd) {
      r.gjk_iters = sat16(g.iters + g.dist_iters);
      if (status == kGjkSeparated && g.sep_valid) {
        const tf3 ta = poseFromQuat(io.posea + 7 * static_cast<uint64_t>(i));
        acc.pa = apply(ta, g.p0);
        acc.pb = apply(ta, g.p1);
        r.distance = norm(g.p0 - g.p1);
        r.ok = 1;
      } else if (status == kGjkIntersect) {
        queued = true;
      } else {
        r.distance = -1;
      }
    } else {
      r.gjk_iters = sat16(g.iters);
      r.ok = 1;
      if constexpr (MODE == kModeBool) {
        r.hit = status == kGjkIntersect;
        r.n_contacts = r.hit;
      } else {
        queued = status == kGjkIntersect;
      }
    }
    if constexpr (MODE != kModeBool)
      if (queued) {
        smp->rank = s.rank;
        ldsSet(smp->a.v, s.a.v); ldsSet(smp->a.d, md.dirOf(static_cast<int>(s.a.id)));
        ldsSet(smp->b.v, s.b.v); ldsSet(smp->b.d, md.dirOf(static_cast<int>(s.b.id)));
        ldsSet(smp->c.v, s.c.v); ldsSet(smp->c.d, md.dirOf(static_cast<int>(s.c.id)));
        ldsSet(smp->e.v, s.e.v); ldsSet(smp->e.d, md.dirOf(static_cast<int>(s.e.id)));
      }
  }
  scanned += md.scanned;
  // queued pairs keep their GJK status here; EPA completes them
  if (__lane_id() == 0) storeResult(&io.out[i], r, acc);
  return queued;
}

// Pairs that need no search (invalid ids, no contacts asked for, closed
// forms), one per lane; true: the pair takes a wavefront.
template <int MODE>
MFCL_D bool lanePair(const ShapeTables& T, const PairIO& io, const Params& P, uint32_t i) {
  const uint32_t ia = io.pa[i], ib = io.pb[i];
  mfcl_convex_result r;
  clearResult(r);
  ResAcc acc;
  acc.normal = acc.pos = acc.pa = acc.pb = d3{0, 0, 0};
  if (ia >= P.n_shapes || ib >= P.n_shapes) {
    r.ok = -1;  // shape id out of range
  } else if (MODE == kModeSd) {
    return true;  // no closed forms (gjk_solver-inl.h:820-874)
  } else if (P.max_contacts <= 0) {
    // the reference warns and adds nothing (collision-inl.h:81-84)
  } else if (closedForm(T.type[ia], T.type[ib])) {
    PContacts pc;
    pc.n = 0;
    const bool hit = runClosedForm(loadShape(T, ia), poseFromQuat(io.posea + 7 * static_cast<uint64_t>(i)),
                                   loadShape(T, ib), poseFromQuat(io.poseb + 7 * static_cast<uint64_t>(i)),
                                   MODE == kModePen ? &pc : nullptr);
    r.hit = hit;
    r.ok = 1;
    if (hit) {
      if constexpr (MODE == kModeBool) r.n_contacts = 1;
      else finishClosedForm(pc, P, io, i, r, acc, true);
    }
  } else {
    return true;
  }
  storeResult(&io.out[i], r, acc);
  return false;
}

// Each wavefront takes `chunk` consecutive pairs: its lanes finish those
// that need no search together, then it runs the others one after the other.
template <int MODE>
__global__ void __launch_bounds__(kBlock, 3) waveKernel(ShapeTables T, const double4* interior, PairIO io, uint64_t n,
                                                        int chunk, Params P, int cap_faces, size_t slice_bytes,
                                                        EpaSink sink, unsigned long long* scanned_total) {
  extern __shared__ __align__(16) char lds[];
  MFCL_LDS char* slice = (MFCL_LDS char*)(lds) + (threadIdx.x >> 6) * slice_bytes;
  MFCL_LDS EpaLds* L = (MFCL_LDS EpaLds*)(slice);
  const uint64_t base = ((static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x) >> 6) * chunk;
  const uint64_t mine = base + __lane_id();
  bool search = false;
  if (static_cast<int>(__lane_id()) < chunk && mine < n) search = lanePair<MODE>(T, io, P, static_cast<uint32_t>(mine));
  int scanned = 0, epa_scanned = 0;
  for (unsigned long long todo = __ballot(search); todo; todo &= todo - 1) {
    const uint32_t i = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(base)) + __builtin_ctzll(todo);
    const bool epa = wavePair<MODE>(T, interior, io, P, i, &L->cfg, &L->s, scanned);
    if constexpr (MODE != kModeBool)
      if (__builtin_amdgcn_readfirstlane(epa ? 1 : 0)) {
        if (__lane_id() == 0) atomicAdd(sink.cnt + kCntQueue, 1u);
        epa_scanned += epaPair(io, P, i, L, cap_faces, sink);
      }
  }
  addScanned(scanned_total, scanned);
  if constexpr (MODE != kModeBool) addScanned(scanned_total + 1, epa_scanned);
}

int waveLaunch(mfcl_ctx* ctx, const ConvexJob& j) {
  // enough wavefronts to fill the chip a few times over, at most one per
  // pair; the lanes of a wavefront share its closed forms
  const uint64_t waves = 64ull * static_cast<uint64_t>(ctx->n_cu);
  const int chunk = static_cast<int>(std::min<uint64_t>(64, (j.n + waves - 1) / waves));
  const unsigned nb = static_cast<unsigned>((j.n + 4ull * chunk - 1) / (4ull * chunk));
  const int cap = epaSmallFaces(ctx, j.P);
  const EpaSink sink = epaSink(ctx, j, cap);
  const size_t slice = j.mode == kModeBool ? (sizeof(WaveCfg) + 15) & ~static_cast<size_t>(15) : epaSliceBytes<SmallMem>(cap);
  if (j.mode == kModeBool)
    waveKernel<kModeBool><<<nb, kBlock, 4 * slice, j.s>>>(j.T, j.interior, j.io, j.n, chunk, j.P, cap, slice, sink, j.sc);
  else if (j.mode == kModePen)
    waveKernel<kModePen><<<nb, kBlock, 4 * slice, j.s>>>(j.T, j.interior, j.io, j.n, chunk, j.P, cap, slice, sink, j.sc);
  else
    waveKernel<kModeSd><<<nb, kBlock, 4 * slice, j.s>>>(j.T, j.interior, j.io, j.n, chunk, j.P, cap, slice, sink, j.sc);
  MFCL_HIP_TRY(ctx, hipGetLastError());
  return MFCL_OK;
}

}  // namespace mfcl
