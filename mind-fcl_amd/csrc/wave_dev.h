// One pair per wavefront: the Minkowski difference with its configuration in
// LDS and a support search that the 64 lanes share.
//
// Every lane runs the pair's FP64 logic on identical values; only the
// support search is divided: lanes 0-31 serve shape 0 and lanes 32-63 shape
// 1, both at once.  A walking hull's step evaluates the current vertex's
// neighbours in eight lanes (one 128-byte block read, one round trip), a
// scanned hull is read by 32 lanes.
//
// What bounds the callers (EPA, small batches, MPR penetration) is the
// latency of one pair's chain of dependent steps.  The search is therefore
// one out-of-line function that needs few registers and no stack: inlined at
// its call sites with both hulls' neighbours evaluated one after the other
// in every lane, it made the EPA loop keep 256 VGPRs and 928 B of scratch
// per lane, whose reloads (2,048 wavefronts' scratch exceeds the L2) were
// most of the loop's waits.
#pragma once

#include "narrow_dev.h"

namespace mfcl {

enum WaveKind : int { kWavePrim = 0, kWaveScan = 1, kWaveBlk = 2, kWaveTab = 3 };

// Direction that produced a simplex vertex, and the hull vertex indices its
// support points came from (-1 for a primitive shape: recomputed from the
// direction when needed).
struct DirSlot {
  double d[3];
  int i0, i1;
};
constexpr int kDirSlots = 8;

struct WaveShape {
  double q[3];          // primitive parameters
  const float4* verts;
  const float4* wblk;   // kWaveBlk: the walk blocks
  const int* nbr;       // kWaveBlk / kWaveTab: the adjacency table
  int type, kind, nv;
  int seed[6];          // walk seeds, +x -x +y -y +z -z
  int pad;
};

struct WaveCfg {
  DirSlot slot[kDirSlots];
  double r1[9];  // frame 0 -> frame 1 rotation (toshape1)
  double r0[9];  // frame 1 -> frame 0 rotation (toshape0)
  double t0[3];  // frame 1 -> frame 0 translation
  double int0[3], int1[3];
  WaveShape sh[2];
};

MFCL_D void waveShapeSet(MFCL_LDS WaveShape* o, const DevShape& s) {
  o->q[0] = s.p0; o->q[1] = s.p1; o->q[2] = s.p2;
  o->verts = s.verts;
  o->wblk = s.wblk;
  o->nbr = s.nbr;
  o->type = s.type;
  o->nv = s.nv;
  o->kind = s.type != kConvex ? kWavePrim : (!s.nbr ? kWaveScan : (s.wblk ? kWaveBlk : kWaveTab));
  if (s.nbr) {
#pragma unroll
    for (int k = 0; k < 6; ++k) o->seed[k] = s.seed[k];
  }
}

MFCL_D void waveCfgSet(MFCL_LDS WaveCfg* c, const DevShape& a, const tf3& ta, const DevShape& b, const tf3& tb, d3 int0,
                       d3 int1) {
  const m33 r1 = tmulm(tb.R, ta.R);
  const tf3 t0 = relTf(ta, tb);
  storeM33(c->r1, r1);
  storeM33(c->r0, t0.R);
  c->t0[0] = t0.t.x; c->t0[1] = t0.t.y; c->t0[2] = t0.t.z;
  c->int0[0] = int0.x; c->int0[1] = int0.y; c->int0[2] = int0.z;
  c->int1[0] = int1.x; c->int1[1] = int1.y; c->int1[2] = int1.z;
  waveShapeSet(&c->sh[0], a);
  waveShapeSet(&c->sh[1], b);
  __builtin_amdgcn_wave_barrier();
}

// Lane exchanges within groups of eight lanes (DPP: no LDS round trip).
template <int CTRL>
MFCL_D int dppI(int v) { return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false); }
template <int CTRL>
MFCL_D double dppD(double v) {
  const uint64_t u = static_cast<uint64_t>(__double_as_longlong(v));
  const uint32_t lo = static_cast<uint32_t>(dppI<CTRL>(static_cast<int>(u)));
  const uint32_t hi = static_cast<uint32_t>(dppI<CTRL>(static_cast<int>(u >> 32)));
  return __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hi) << 32) | lo));
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E;  // quad_perm(1,0,3,2), (2,3,0,1)
constexpr int kDppHalfMirror = 0x141, kDppMirror = 0x140;  // lane i <-> 7 - i, 15 - i
// xor 1, xor 2, then mirroring the eight lanes: every lane ends with the
// combination of all eight
MFCL_D double max8(double v) {
  v = fmax(v, dppD<kDppXor1>(v));
  v = fmax(v, dppD<kDppXor2>(v));
  return fmax(v, dppD<kDppHalfMirror>(v));
}
MFCL_D int min8(int v) {
  v = min(v, dppI<kDppXor1>(v));
  v = min(v, dppI<kDppXor2>(v));
  return min(v, dppI<kDppHalfMirror>(v));
}

MFCL_D double readLaneF64(double v, int src) {
  const uint64_t u = static_cast<uint64_t>(__double_as_longlong(v));
  const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(u), src);
  const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(u >> 32), src);
  return __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hi) << 32) | lo));
}

// The seed of a walk (walkInit's rule): the axis of the largest support
// value, first on ties.  A finite direction's six products with the signed
// unit axes are its signed components; with a non-finite one the sums
// mostly turn NaN, so they are formed in full.
MFCL_D int waveSeedAxis(d3 d) {
  int init = 0;
  if (d.x * 0.0 + d.y * 0.0 + d.z * 0.0 == 0.0) {
    double best = d.x;
    if (-d.x > best) { best = -d.x; init = 1; }
    if (d.y > best) { best = d.y; init = 2; }
    if (-d.y > best) { best = -d.y; init = 3; }
    if (d.z > best) { best = d.z; init = 4; }
    if (-d.z > best) init = 5;
    return init;
  }
  double best = 0;
#pragma nounroll
  for (int i = 0; i < 6; ++i) {
    const double sg = (i & 1) ? -1.0 : 1.0;
    const double ax = (i >> 1) == 0 ? sg : sg * 0.0;
    const double ay = (i >> 1) == 1 ? sg : sg * 0.0;
    const double az = (i >> 1) == 2 ? sg : sg * 0.0;
    const double dv = ax * d.x + ay * d.y + az * d.z;
    if (i == 0 || dv > best) {
      best = dv;
      init = i;
    }
  }
  return init;
}

// Support points of both shapes for direction d (frame 0): p0 = support0(d),
// p1 = support1(-d) in frame 0; i0 / i1 the hull vertices they are (-1 for a
// primitive); scanned the hull vertices evaluated: all of a scanned hull's,
// of a walked one the start and the neighbours of each vertex it stood on.
struct WaveSup {
  d3 p0, p1;
  int i0, i1, scanned;
};

// All 64 lanes call this with the same arguments and get the same result.
// Walks take the neighbour that the reference's sequential comparisons end on
// (the first of the largest values, when it exceeds the current vertex's),
// so they visit the same vertices; the two vertices a walk has just left are
// compared again here, which cannot change a step (their values are below
// the current one).  Scans return the first vertex attaining the FP64
// maximum, without an FP32 pre-scan: the 32 lanes'
// loads, not the FP64 products, take the time.
__device__ __attribute__((noinline)) static WaveSup waveSupport(const MFCL_LDS WaveCfg* c, double dx, double dy, double dz) {
  const int lane = __lane_id(), sub = lane & 31, j = lane & 7;
  const bool second = lane >= 32;
  const MFCL_LDS WaveShape* S = &c->sh[second ? 1 : 0];
  const d3 r = mul(loadM33(c->r1), -d3{dx, dy, dz});
  const d3 d = {second ? r.x : dx, second ? r.y : dy, second ? r.z : dz};
  const int kind = S->kind;
  int idx = -1, count = 0;
  d3 p = {0, 0, 0};
  if (__ballot(kind == kWavePrim) != 0ull) {
    if (kind == kWavePrim) {
      DevShape s;
      s.type = S->type;
      s.p0 = S->q[0]; s.p1 = S->q[1]; s.p2 = S->q[2];
      s.verts = S->verts;
      p = primSupport(s, d);
    }
  }
  if (__ballot(kind == kWaveScan) != 0ull) {
    if (kind == kWaveScan) {
      const float4* v = S->verts;
      const int nv = S->nv;
      double bv = -INFINITY;
      int bi = 0x7fffffff;
      for (int i0 = sub; i0 < nv; i0 += 128) {
        float4 q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = v[min(i0 + 32 * u, nv - 1)];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int i = i0 + 32 * u;
          const double val = d.x * static_cast<double>(q[u].x) + d.y * static_cast<double>(q[u].y) +
                             d.z * static_cast<double>(q[u].z);
          if (i < nv && val > bv) {
            bv = val;
            bi = i;
          }
        }
      }
#pragma nounroll
      for (int off = 16; off > 0; off >>= 1) {
        const double ov = __shfl_xor(bv, off);
        const int oi = __shfl_xor(bi, off);
        if (ov > bv || (ov == bv && oi < bi)) {
          bv = ov;
          bi = oi;
        }
      }
      // a NaN direction or vertex leaves no candidate: vertex 0
      idx = bi < nv ? bi : 0;
      count = nv;
      const float4 q = v[idx];
      p = d3{q.x, q.y, q.z};
    }
  }
  if (__ballot(kind >= kWaveBlk) != 0ull) {
    bool act = kind >= kWaveBlk;
    const float4* v = S->verts;
    const char* blk = reinterpret_cast<const char*>(S->wblk);
    const int* nbr = S->nbr;
    double ev = 0;
    bool first = true;
    if (act) idx = S->seed[waveSeedAxis(d)];
    while (true) {
      // the current vertex's neighbours, eight at a time: lane j of each
      // eight holds neighbour base + j; the first eight of a block-walked
      // hull come with the block
      int cnt = 0, rec = 0, nid = 0;
      float nx = 0, ny = 0, nz = 0, sx = 0, sy = 0, sz = 0;
      bool have = false;
      if (act) {
        if (kind == kWaveBlk) {
          const char* b = blk + 128 * static_cast<uint64_t>(idx);
          const float4 q = *reinterpret_cast<const float4*>(b);
          nid = *reinterpret_cast<const uint16_t*>(b + 16 + 2 * j);
          const float* f = reinterpret_cast<const float*>(b + 32 + 12 * j);
          nx = f[0]; ny = f[1]; nz = f[2];
          sx = q.x; sy = q.y; sz = q.z;
          cnt = __float_as_int(q.w);
          have = true;
          if (cnt > 8) rec = __float_as_int(v[idx].w);
        } else {
          const float4 q = v[idx];
          sx = q.x; sy = q.y; sz = q.z;
          rec = __float_as_int(q.w);
          cnt = nbr[rec];
        }
        p = d3{sx, sy, sz};
        if (first) {
          ev = d.x * p.x + d.y * p.y + d.z * p.z;
          count = 1;
        }
        count += cnt;
      }
      first = false;
      double bv = -INFINITY;
      int bk = 0x7fffffff, bid = 0;
      for (int base = 0;; base += 8) {
        const bool in = act && base + j < cnt;
        if (in && !(have && base == 0)) {
          nid = nbr[rec + 1 + base + j];
          const float4 q = v[nid];
          nx = q.x; ny = q.y; nz = q.z;
        }
        const double val = d.x * static_cast<double>(nx) + d.y * static_cast<double>(ny) + d.z * static_cast<double>(nz);
        if (in && val > bv) {
          bv = val;
          bk = base + j;
          bid = nid;
        }
        if (__ballot(act && base + 8 < cnt) == 0ull) break;
      }
      const double m = max8(bv);
      const int k = min8(bv == m ? bk : 0x7fffffff);
      const bool better = act && m > ev;
      const unsigned long long win = __ballot(better && bv == m && bk == k);
      if (win == 0ull) break;
      // the winner's id (its eight lanes repeat within each half)
      const uint32_t w0 = static_cast<uint32_t>(win), w1 = static_cast<uint32_t>(win >> 32);
      const int id0 = __builtin_amdgcn_readlane(bid, w0 ? __builtin_ctz(w0) : 0);
      const int id1 = __builtin_amdgcn_readlane(bid, w1 ? 32 + __builtin_ctz(w1) : 32);
      act = better;
      if (act) {
        ev = m;
        idx = second ? id1 : id0;
      }
    }
  }
  WaveSup o;
  o.i0 = __builtin_amdgcn_readlane(idx, 0);
  o.i1 = __builtin_amdgcn_readlane(idx, 32);
  o.scanned = __builtin_amdgcn_readlane(count, 0) + __builtin_amdgcn_readlane(count, 32);
  o.p0 = d3{readLaneF64(p.x, 0), readLaneF64(p.y, 0), readLaneF64(p.z, 0)};
  const d3 x = {readLaneF64(p.x, 32), readLaneF64(p.y, 32), readLaneF64(p.z, 32)};
  tf3 t0;
  t0.R = loadM33(c->r0);
  t0.t = d3{c->t0[0], c->t0[1], c->t0[2]};
  o.p1 = apply(t0, x);
  return o;
}

// The Minkowski difference of the wavefront's pair, with the interface of
// the lanes' MinkLane.
struct MinkW {
  MFCL_LDS WaveCfg* c;
  int scanned;
  MFCL_D WaveSup sup(d3 d) {
    const WaveSup s = waveSupport(c, d.x, d.y, d.z);
    scanned += s.scanned;
    return s;
  }
  MFCL_D d3 support0(d3 d) { return sup(d).p0; }
  MFCL_D d3 support1(d3 d) { return sup(-d).p1; }
  MFCL_D d3 support(d3 d) {
    const WaveSup s = sup(d);
    return s.p0 - s.p1;
  }
  MFCL_D d3 supportNew(d3 d, int id) {
    const WaveSup s = sup(d);
    MFCL_LDS DirSlot& sl = c->slot[id & (kDirSlots - 1)];
    sl.d[0] = d.x; sl.d[1] = d.y; sl.d[2] = d.z;
    sl.i0 = s.i0; sl.i1 = s.i1;
    return s.p0 - s.p1;
  }
  MFCL_D d3 dirOf(int id) const {
    const MFCL_LDS DirSlot& sl = c->slot[id & (kDirSlots - 1)];
    return d3{sl.d[0], sl.d[1], sl.d[2]};
  }
  MFCL_D d3 interior() const {
    return d3{c->int0[0], c->int0[1], c->int0[2]} - toFrame0(d3{c->int1[0], c->int1[1], c->int1[2]});
  }
  MFCL_D d3 toFrame0(d3 x) const {
    tf3 t0;
    t0.R = loadM33(c->r0);
    t0.t = d3{c->t0[0], c->t0[1], c->t0[2]};
    return apply(t0, x);
  }
  // shape k's support for direction d of its own frame: a primitive's
  // closed form, or the hull vertex i
  MFCL_D d3 ownPoint(int k, int i, d3 d) const {
    const MFCL_LDS WaveShape& S = c->sh[k];
    if (__builtin_amdgcn_readfirstlane(i) >= 0) {
      const float4 q = S.verts[i];
      return d3{q.x, q.y, q.z};
    }
    DevShape s;
    s.type = S.type;
    s.p0 = S.q[0]; s.p1 = S.q[1]; s.p2 = S.q[2];
    s.verts = S.verts;
    return primSupport(s, d);
  }
  // support0(d) and support1(-d) from the recorded support vertices of that
  // direction (-1: a primitive's, or not recorded)
  MFCL_D void pointsAt(int i0, int i1, d3 d, d3& a, d3& b) {
    const bool k0 = i0 >= 0 || c->sh[0].kind == kWavePrim, k1 = i1 >= 0 || c->sh[1].kind == kWavePrim;
    if (__builtin_amdgcn_readfirstlane(k0 && k1 ? 1 : 0)) {
      a = ownPoint(0, i0, d);
      b = toFrame0(ownPoint(1, i1, mul(loadM33(c->r1), -d)));
      return;
    }
    const WaveSup s = sup(d);
    a = s.p0;
    b = s.p1;
  }
  MFCL_D d3 point0(int id) const {
    return ownPoint(0, c->slot[id & (kDirSlots - 1)].i0, dirOf(id));
  }
  MFCL_D d3 point1(int id) const {
    return toFrame0(ownPoint(1, c->slot[id & (kDirSlots - 1)].i1, mul(loadM33(c->r1), -dirOf(id))));
  }
};

}  // namespace mfcl
