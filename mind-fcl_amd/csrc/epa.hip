// EPA stage of a convex query: the pairs that GJK queued, then those that
// outgrew their LDS polytope.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "epa_pair.h"

namespace mfcl {

// One wavefront per queued pair.  Pairs are taken one at a time from a
// shared counter: EPA iteration counts vary widely (p99 / mean ~ 3), so a
// static share per wavefront would leave the grid waiting on its most loaded
// wavefronts.  The GJK stage queues the pairs roughly in descending cost
// order (bucketed by hull sizes), so the largest pairs, which tend to need
// the most EPA iterations, start first and the tail shortens.
__global__ void __launch_bounds__(kBlock, 3) epaQueueKernel(ShapeTables T, PairIO io, Params P, const QEntry* queue,
                                                            int cap_faces, size_t slice_bytes, EpaSink sink,
                                                            unsigned long long* scanned_total) {
  extern __shared__ __align__(16) char lds[];
  MFCL_LDS EpaLds* L = (MFCL_LDS EpaLds*)((MFCL_LDS char*)(lds) + (threadIdx.x >> 6) * slice_bytes);
  const uint32_t count = sink.cnt[kCntQueue];
  const int lane = threadIdx.x & 63;
  int scanned = 0;
  for (;;) {
    uint32_t q = 0;
    if (lane == 0) q = atomicAdd(sink.cnt + kCntNext, 1u);
    q = __builtin_amdgcn_readfirstlane(q);
    if (q >= count) break;
    const uint32_t i = __builtin_amdgcn_readfirstlane(queue[q].pair);
    const uint64_t* e = reinterpret_cast<const uint64_t*>(&queue[q].s);
    if (lane < static_cast<int>(sizeof(SmpD) / 8)) ((MFCL_LDS uint64_t*)(&L->s))[lane] = e[lane];
    epaCfg(T, io, i, L);
    scanned += epaPair(io, P, i, L, cap_faces, sink);
  }
  addScanned(scanned_total, scanned);
}

// Pairs that outgrew the LDS polytope: those with a dump continue, the
// others restart, in a polytope of the request's capacity, one wavefront per
// block.
template <class M>
__global__ void __launch_bounds__(64) epaFullKernel(ShapeTables T, PairIO io, Params P, int cap_small, EpaSink sink,
                                                    unsigned long long* scanned_total) {
  extern __shared__ __align__(16) char lds[];
  MFCL_LDS EpaLds* L = (MFCL_LDS EpaLds*)((MFCL_LDS char*)(lds));
  const uint32_t dumps = sink.cnt[kCntSpilled];
  const uint32_t count = dumps + sink.cnt[kCntRestart];
  const int lane = threadIdx.x & 63;
  int scanned = 0;
  for (;;) {
    uint32_t q = 0;
    if (lane == 0) q = atomicAdd(sink.cnt + kCntFullNext, 1u);
    q = __builtin_amdgcn_readfirstlane(q);
    if (q >= count) break;
    const bool resume = q < dumps;
    const char* dump = sink.dumps + q * sink.dump_bytes;
    const QEntry* e = sink.oflow + (q - dumps);
    const uint32_t i = __builtin_amdgcn_readfirstlane(resume ? static_cast<uint32_t>(epaDumpItem(dump)) : e->pair);
    if (resume) {
      epaLoad<M>(L, ldsArena(L), P.epa_max_faces, dump, cap_small);
    } else {
      const uint64_t* w = reinterpret_cast<const uint64_t*>(&e->s);
      if (lane < static_cast<int>(sizeof(SmpD) / 8)) ((MFCL_LDS uint64_t*)(&L->s))[lane] = w[lane];
    }
    epaCfg(T, io, i, L);
    const int st = epaRun<M>(L, ldsArena(L), P.epa_max_faces, P.epa_tol, P.epa_max_it, false, resume);
    epaStore(io, P, i, L, st);
    scanned += L->out.scanned;
  }
  addScanned(scanned_total, scanned);
}

size_t epaFullBytes(int max_faces) {
  return max_faces <= kMidFaces ? epaSliceBytes<MidMem>(max_faces) : epaSliceBytes<LargeMem>(max_faces);
}

int epaSmallFaces(const mfcl_ctx* ctx, const Params& P) {
  int cap = std::min(std::min(P.epa_max_faces, ctx->tune.epa_lds_faces), kSmallFaces);
  while (cap > 4 && 4 * epaSliceBytes<SmallMem>(cap) > static_cast<size_t>(ctx->max_lds_per_block)) cap /= 2;
  return cap;
}

int epaQueueLaunch(mfcl_ctx* ctx, const ConvexJob& j) {
  const int cap = epaSmallFaces(ctx, j.P);
  const size_t slice = epaSliceBytes<SmallMem>(cap);
  const uint64_t most = (j.n + 3) / 4;  // a wavefront per pair is enough
  const unsigned eb = static_cast<unsigned>(std::min<uint64_t>(ctx->tune.epa_threads / kBlock, most));
  epaQueueKernel<<<eb, kBlock, 4 * slice, j.s>>>(j.T, j.io, j.P, j.queue, cap, slice, epaSink(ctx, j, cap), j.sc + 1);
  MFCL_HIP_TRY(ctx, hipGetLastError());
  return MFCL_OK;
}

int epaFullLaunch(mfcl_ctx* ctx, const ConvexJob& j) {
  const int cap = epaSmallFaces(ctx, j.P);
  if (cap >= j.P.epa_max_faces) return MFCL_OK;
  const unsigned ob = static_cast<unsigned>(std::min<uint64_t>(ctx->tune.epa_overflow_waves, j.n));
  const size_t lds = epaFullBytes(j.P.epa_max_faces);
  const EpaSink sink = epaSink(ctx, j, cap);
  if (j.P.epa_max_faces <= kMidFaces) epaFullKernel<MidMem><<<ob, 64, lds, j.s>>>(j.T, j.io, j.P, cap, sink, j.sc + 1);
  else epaFullKernel<LargeMem><<<ob, 64, lds, j.s>>>(j.T, j.io, j.P, cap, sink, j.sc + 1);
  MFCL_HIP_TRY(ctx, hipGetLastError());
  return MFCL_OK;
}

}  // namespace mfcl
