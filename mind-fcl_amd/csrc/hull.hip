// Convex hulls of point sets on the device, and the convex shape table built
// from them without a host round trip.
//
// The reference takes a hull's vertices and faces from its caller
// (fcl::Convex's constructor, include/fcl/geometry/shape/convex-inl.h:50-73)
// and derives the vertex adjacency of its support walk from the faces
// (convex-inl.h:293-409).  Here the hull itself is computed on the GPU:
// one wavefront per point set runs an incremental hull in its LDS slice
// (points, triangles with their three edge neighbours, conflict faces),
// inserting outside points in index order: the faces a point sees form a
// connected cap found by a flood fill from its conflict face, the cap's
// border becomes a fan of new triangles to the point, and the points that
// saw the removed faces look for a new face they see among the fan.
// Orientation tests run in FP64 on the FP32 coordinates, after an FP32 test
// that leaves to them what it is not sure of (hull_orient.h); a point within a
// relative 1e-12 of a face's plane does not see it, so (near-)coplanar
// points are left out of the hull as qhull leaves out coplanar points.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "ctx.h"
#include "dmath.h"
#include "hull_orient.h"

namespace mfcl {

constexpr int kHullMaxPoints = 768;
constexpr int kHullMaxHorizon = 192;

enum HullStatus : int32_t { kHullOk = 0, kHullDegenerate = 1, kHullTooLarge = 2, kHullFailed = 3 };

// A face in one word: its three vertices (10 bits each), whether this step's
// flood fill has been at it, and whether the inserted point sees it.
constexpr uint32_t kFaceTouched = 1u << 30, kFaceVisible = 1u << 31, kFaceVerts = kFaceTouched - 1;
constexpr uint32_t kFaceFree = ~0u;  // vertices 1023: no point has that number

struct alignas(8) HullEdge {  // border edge (a, b) of this step's cap; outer = 4 * face beyond it + edge number there
  int16_t a, b, outer, pad;
};

// LDS slice of one wavefront for point sets of up to cap points (faces: 2
// cap, a triangulated sphere over n vertices has 2 n - 4).  The slice decides
// how many wavefronts a CU holds (each is one chain of dependent LDS reads,
// so the throughput follows their number): 23,040 B at 512 points, seven a
// CU; face state, vertices and visible list in separate words took 35,000,
// four a CU.
struct HullLds {
  float* xyz;         // [cap][3]
  uint32_t* fv;       // [F] faces
  HullEdge* hor;      // border of this step's cap
  int16_t* conf;      // per point: conflict face, -1 inside, -2 hull vertex
  int16_t* fnb;       // [3][F] neighbour across edge (v_k, v_k+1)
  int16_t* start;     // per point: border edge starting at it (-1 none); reused as new vertex ids at the end
  int16_t* endv;      // per point: border edge ending at it
  int16_t* freel;     // stack of free face slots; this step's visible faces are listed above its top
  int F;
};

__host__ __device__ inline int hullHorizon(int cap) { return cap < kHullMaxHorizon ? cap : kHullMaxHorizon; }
__host__ __device__ inline size_t hullLdsBytes(int cap) {
  const size_t c = (static_cast<size_t>(cap) + 3) & ~static_cast<size_t>(3);
  return 12 * c + 8 * c + sizeof(HullEdge) * hullHorizon(static_cast<int>(c)) + 2 * c + 12 * c + 4 * c + 4 * c;
}

MFCL_D HullLds hullCarve(char* base, int cap) {
  HullLds L;
  const int c = (cap + 3) & ~3;
  L.F = 2 * c;
  L.xyz = reinterpret_cast<float*>(base);
  L.fv = reinterpret_cast<uint32_t*>(base + 12 * c);
  L.hor = reinterpret_cast<HullEdge*>(base + 20 * c);
  L.conf = reinterpret_cast<int16_t*>(base + 20 * c + sizeof(HullEdge) * hullHorizon(c));
  L.fnb = L.conf + c;
  L.start = L.fnb + 3 * L.F;
  L.endv = L.start + c;
  L.freel = L.endv + c;
  return L;
}

MFCL_D d3 hp(const HullLds& L, int i) { return d3{L.xyz[3 * i], L.xyz[3 * i + 1], L.xyz[3 * i + 2]}; }

// Signed volume test of point P against face (A, B, C), normal (B-A)x(C-A),
// in 64 bits: true outside, beyond 1e-12 of the square root of the edges'
// square lengths.
MFCL_D bool sees64(d3 A, d3 B, d3 C, d3 P) {
  const d3 u = B - A, v = C - A, w = P - A;
  const d3 n = cross(u, v);
  const double o = dot(n, w);
  if (!(o > 0)) return false;
  return o > 1e-12 * sqrt(sqnorm(u) * sqnorm(v) * sqnorm(w));
}
MFCL_D bool sees(const HullLds& L, int a, int b, int c, int p) {
  const int s = sees32(planeOf(L.xyz + 3 * a, L.xyz + 3 * b, L.xyz + 3 * c), L.xyz + 3 * p);
  return s >= 0 ? s != 0 : sees64(hp(L, a), hp(L, b), hp(L, c), hp(L, p));
}
MFCL_D bool faceSees(const HullLds& L, uint32_t v, int p) {
  return sees(L, v & 1023, v >> 10 & 1023, v >> 20 & 1023, p);
}

MFCL_D int laneId64() { return threadIdx.x & 63; }
// What one lane writes before it, the others read after it (no instructions:
// the LDS runs one wavefront's accesses in order).
MFCL_D void wsync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

MFCL_D uint32_t faceWord(int a, int b, int c) {
  return static_cast<uint32_t>(a) | static_cast<uint32_t>(b) << 10 | static_cast<uint32_t>(c) << 20;
}
MFCL_D int below(unsigned long long m, int l) { return __popcll(m & ((1ull << l) - 1)); }

// Wave argmax of val (first index on ties); all lanes get (index, value).
MFCL_D void waveArgmax(double& val, int& idx) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const double ov = __shfl_xor(val, off);
    const int oi = __shfl_xor(idx, off);
    if (ov > val || (ov == val && oi < idx)) {
      val = ov;
      idx = oi;
    }
  }
}

// One wavefront per set (set order[b] for block b when order is given, else
// set b, skipped if its size is not in (lo, cap] and another launch takes
// it), in an LDS slice for sets of up to cap points; the slots a set's
// faces take do not depend on cap, so neither does its result.  Outputs
// (per set i, points at pt_off[i]):
// hull_idx[pt_off + k] = index (within the set) of the k-th hull vertex in
// ascending order, hull_cnt[i]; tris[6 pt_off + 3 t + j] = triangle t over
// those k-numbered vertices (outward orientation), tri_cnt[i]; status[i].
//
// An insertion is a chain of dependent LDS reads and FP64 tests.  Its longest
// part was the points that lost their conflict face: each lane tried the
// fan's faces one after another for a point of its own, so every group of 64
// points with one such point cost a whole fan of tests.  They are gathered
// from all groups instead and tested (point, face) pair per lane, each lane
// with one fan face's plane in registers.  20,011 sets of 8..512 points, back
// to back: 18.7 ms before; 5.5 with that and the smaller slices, 5.2 with a
// frontier and a border that stay in registers, 4.8 with the test in 32 bits
// first (a wavefront's insertion is then about 3 LDS round trips for each of
// 3 frontiers and as many again for the rest, 10,000 cycles).
__global__ void __launch_bounds__(64) hullKernel(const float* pts, const uint64_t* pt_off, const uint32_t* pt_cnt,
                                                 const uint32_t* order, uint32_t n_sets, int lo, int cap, int top,
                                                 uint32_t* hull_cnt, uint32_t* hull_idx, uint32_t* tri_cnt,
                                                 int32_t* tris, int32_t* status) {
  extern __shared__ __align__(16) char hull_lds[];
  if (blockIdx.x >= n_sets) return;
  const uint32_t set = order ? order[blockIdx.x] : blockIdx.x;
  const int l = laneId64();
  const uint32_t cnt = pt_cnt[set];
  if (static_cast<int64_t>(cnt) <= lo || (cnt > static_cast<uint32_t>(cap) && cap < top)) return;
  const uint64_t o = pt_off[set];
  auto finish = [&](int st) {
    if (l == 0) {
      status[set] = st;
      hull_cnt[set] = 0;
      tri_cnt[set] = 0;
    }
  };
  if (cnt > static_cast<uint32_t>(cap)) { finish(kHullTooLarge); return; }
  const int n = static_cast<int>(cnt);
  if (n < 4) { finish(kHullDegenerate); return; }
  HullLds L = hullCarve(hull_lds, cap);
  const int F = L.F;
  for (int i = l; i < 3 * n; i += 64) L.xyz[i] = pts[3 * o + i];
  for (int i = l; i < n; i += 64) L.conf[i] = L.start[i] = L.endv[i] = -1;
  for (int f = l; f < F; f += 64) L.fv[f] = kFaceFree;
  wsync();
  // ---- initial tetrahedron: extreme x, farthest point, farthest from the
  // line, farthest from the plane (relative tolerances against the extent)
  int i0 = 0;
  {
    double v = -INFINITY;
    int idx = 0x7fffffff;
    for (int i = l; i < n; i += 64)
      if (-static_cast<double>(L.xyz[3 * i]) > v) { v = -static_cast<double>(L.xyz[3 * i]); idx = i; }
    waveArgmax(v, idx);
    i0 = idx;
  }
  const d3 P0 = hp(L, i0);
  int i1 = 0;
  double ext2 = 0;
  {
    double v = -1;
    int idx = 0x7fffffff;
    for (int i = l; i < n; i += 64) {
      const double d = sqnorm(hp(L, i) - P0);
      if (d > v) { v = d; idx = i; }
    }
    waveArgmax(v, idx);
    i1 = idx;
    ext2 = v;
  }
  if (!(ext2 > 0)) { finish(kHullDegenerate); return; }
  const d3 dir = hp(L, i1) - P0;
  int i2 = 0;
  {
    double v = -1;
    int idx = 0x7fffffff;
    for (int i = l; i < n; i += 64) {
      const double d = sqnorm(cross(dir, hp(L, i) - P0));
      if (d > v) { v = d; idx = i; }
    }
    waveArgmax(v, idx);
    i2 = idx;
    if (!(v > 1e-24 * ext2 * ext2)) { finish(kHullDegenerate); return; }
  }
  const d3 nrm = cross(dir, hp(L, i2) - P0);
  int i3 = 0;
  double vol = 0;
  {
    double v = -1;
    int idx = 0x7fffffff;
    for (int i = l; i < n; i += 64) {
      const double d = fabs(dot(nrm, hp(L, i) - P0));
      if (d > v) { v = d; idx = i; }
    }
    waveArgmax(v, idx);
    i3 = idx;
    vol = v;
    if (!(vol > 1e-12 * sqrt(sqnorm(nrm)) * sqrt(ext2))) { finish(kHullDegenerate); return; }
  }
  // faces oriented outward: the fourth vertex lies below each face
  int a = i0, b = i1, c = i2;
  const int d = i3;
  if (dot(cross(hp(L, b) - hp(L, a), hp(L, c) - hp(L, a)), hp(L, d) - hp(L, a)) > 0) {
    const int t = b;
    b = c;
    c = t;
  }
  if (l == 0) {
    L.fv[0] = faceWord(a, b, c);
    L.fv[1] = faceWord(a, d, b);
    L.fv[2] = faceWord(b, d, c);
    L.fv[3] = faceWord(c, d, a);
    L.conf[a] = L.conf[b] = L.conf[c] = L.conf[d] = -2;
  }
  wsync();
  auto vertOf = [&](uint32_t w, int k) -> int { return w >> (10 * k) & 1023; };
  // number of the edge of face word w that runs from eb to ea, -1 none
  auto edgeOf = [&](uint32_t w, int ea, int eb) -> int {
    int kk = -1;
    for (int j = 0; j < 3; ++j)
      if (vertOf(w, j) == eb && vertOf(w, j < 2 ? j + 1 : 0) == ea) kk = j;
    return kk;
  };
  // neighbours of the four faces by edge matching
  if (l < 12) {
    const int f = l / 3, k = l % 3;
    const uint32_t w = L.fv[f];
    for (int g = 0; g < 4; ++g)
      if (edgeOf(L.fv[g], vertOf(w, k), vertOf(w, k < 2 ? k + 1 : 0)) >= 0) L.fnb[k * F + f] = static_cast<int16_t>(g);
  }
  int nf_used = 4, free_top = 0;
  wsync();
  // conflict faces of the other points
  for (int i = l; i < n; i += 64) {
    if (L.conf[i] == -2) continue;
    int cf = -1;
    for (int f = 0; f < 4 && cf < 0; ++f)
      if (faceSees(L, L.fv[f], i)) cf = f;
    L.conf[i] = static_cast<int16_t>(cf);
  }
  wsync();
  const int max_hor = hullHorizon(F / 2), list_max = max_hor < 64 ? max_hor : 64, l3 = l % 3;
  int cursor = 0;
  bool failed = false;
  while (true) {
    // next outside point in index order
    int p = -1, f0 = 0;
    while (cursor < n) {
      const int i = cursor + l;
      const int cf = i < n ? L.conf[i] : -1;
      const unsigned long long m = __ballot(cf >= 0);
      if (m) {
        const int at = __ffsll(m) - 1;
        p = cursor + at;
        f0 = __builtin_amdgcn_readlane(cf, at);
        break;
      }
      cursor += 64;
    }
    if (p < 0) break;
    cursor = p + 1;
    // Flood fill of the faces p sees, from its conflict face.  A frontier of
    // up to 21 faces stays in the lanes: lane 3 j + k has the k-th neighbour
    // of the frontier's j-th face, and whoever finds one that p sees hands
    // its neighbours on.
    int16_t* vis = L.freel + free_top;
    if (l == 0) {
      vis[0] = static_cast<int16_t>(f0);
      L.fv[f0] |= kFaceTouched | kFaceVisible;
    }
    wsync();
    int nvis = 1, last = 1;  // last: faces of the newest frontier
    int g = L.fnb[l3 * F + f0];
    while (last > 0 && last <= 21) {
      bool s = false;
      int nb[3] = {0, 0, 0};
      if (l < 3 * last) {
        const uint32_t w = atomicOr(&L.fv[g], kFaceTouched);
        for (int k = 0; k < 3; ++k) nb[k] = L.fnb[k * F + g];
        if (!(w & kFaceTouched)) {
          s = faceSees(L, w, p);
          if (s) L.fv[g] = w | kFaceTouched | kFaceVisible;
        }
      }
      const unsigned long long m = __ballot(s);
      const int rank = below(m, l);
      if (s) vis[nvis + rank] = static_cast<int16_t>(g);
      last = __popcll(m);
      nvis += last;
      const int to = s && rank < 21 ? 3 * rank : 63;
      const int g0 = __builtin_amdgcn_ds_permute(4 * to, nb[0]);
      const int g1 = __builtin_amdgcn_ds_permute(to < 63 ? 4 * to + 4 : 252, nb[1]);
      const int g2 = __builtin_amdgcn_ds_permute(to < 63 ? 4 * to + 8 : 252, nb[2]);
      g = l3 == 0 ? g0 : l3 == 1 ? g1 : g2;
    }
    wsync();
    for (int fr0 = nvis - last; fr0 < nvis;) {  // wider frontiers, from the list
      const int fr1 = nvis;
      for (int base = fr0 * 3; base < fr1 * 3; base += 64) {
        const int e = base + l;
        bool s = false;
        int f = 0;
        if (e < fr1 * 3) {
          const int at = e / 3;
          f = L.fnb[(e - 3 * at) * F + vis[at]];
          const uint32_t w = atomicOr(&L.fv[f], kFaceTouched);
          if (!(w & kFaceTouched)) {
            s = faceSees(L, w, p);
            if (s) L.fv[f] = w | kFaceTouched | kFaceVisible;
          }
        }
        const unsigned long long m = __ballot(s);
        if (s) vis[nvis + below(m, l)] = static_cast<int16_t>(f);
        nvis += __popcll(m);
      }
      wsync();
      fr0 = fr1;
    }
    // Border: edges of visible faces whose neighbour is not visible.  What a
    // lane found last stays in its registers: all of a border of a cap of up
    // to 21 faces.
    int nh = 0, h1 = 0;
    HullEdge e1{0, 0, 0, 0};
    bool edge1 = false;
    for (int base = 0; base < nvis * 3; base += 63) {
      const int at = base / 3 + l / 3;
      bool s = false;
      int ea = 0, eb = 0, kk = -1, out = 0;
      if (l < 63 && at < nvis) {
        const int f = vis[at];
        out = L.fnb[l3 * F + f];
        const uint32_t wf = L.fv[f], wg = L.fv[out];
        s = !(wg & kFaceVisible);
        ea = vertOf(wf, l3);
        eb = vertOf(wf, l3 < 2 ? l3 + 1 : 0);
        kk = edgeOf(wg, ea, eb);
      }
      const unsigned long long m = __ballot(s);
      h1 = nh + below(m, l);
      edge1 = s;
      const bool fits = h1 < max_hor && kk >= 0;
      if (s && fits) {
        e1 = HullEdge{static_cast<int16_t>(ea), static_cast<int16_t>(eb), static_cast<int16_t>(4 * out + kk), 0};
        L.hor[h1] = e1;
        L.start[ea] = static_cast<int16_t>(h1);
        L.endv[eb] = static_cast<int16_t>(h1);
      }
      failed |= __ballot(s && !fits) != 0;
      nh += __popcll(m);
    }
    if (failed || nh < 3) {
      failed = true;
      break;
    }
    wsync();
    const bool small = nvis <= 21;
    const int n_free = free_top + nvis;
    // slot of the new face (a, b, p) at border edge h: freed visible faces
    // first, then fresh ones
    auto slotOf = [&](int h) -> int { return h < n_free ? L.freel[n_free - 1 - h] : nf_used + (h - n_free); };
    // The border must be one loop: each vertex starts and ends one edge (of
    // two edges that start at a vertex one finds the other's number).
    bool bad = false;
    int slot1 = 0, slot_b = 0, slot_a = 0;  // slots of the edge's own face and of the next and the one before
    auto check = [&](const HullEdge& e, int h) {
      const int eb = L.start[e.b], ea = L.endv[e.a];
      bad |= L.start[e.a] != h || L.endv[e.b] != h || ea < 0 || eb < 0;
      slot1 = slotOf(h);
      slot_b = slotOf(eb > 0 ? eb : 0);
      slot_a = slotOf(ea > 0 ? ea : 0);
    };
    if (small) {
      if (edge1) check(e1, h1);
    } else {
      for (int h = l; h < nh; h += 64) check(L.hor[h], h);
    }
    // (the fan never needs more than the slots left: checked before any write)
    if (__ballot(bad) || nh > n_free + (F - nf_used)) {
      failed = true;
      break;
    }
    // points that saw a removed face look for the first new face they see
    {
      const int lg = nh > 32 ? 6 : 32 - __clz(nh - 1);  // lanes a point: the border's length, to a power of two
      const int G = 1 << lg, lead = l & ~(G - 1), h0 = l - lead, j0 = l >> lg, per = 64 >> lg;
      const int hl = h0 < nh ? h0 : 0;
      const HullEdge e0 = L.hor[hl];
      const HullPlane plane = planeOf(L.xyz + 3 * e0.a, L.xyz + 3 * e0.b, L.xyz + 3 * p);
      const int slot0 = slotOf(hl);
      int n_lost = 0;  // gathered points, in the border entries' spare fields
      auto flush = [&] {
        wsync();
        for (int j = 0; j < n_lost; j += per) {
          const bool mine = j + j0 < n_lost;
          const int i = L.hor[mine ? j + j0 : 0].pad;
          int sure = 0;
          if (mine && h0 < nh) {
            sure = sees32(plane, L.xyz + 3 * i);
            if (sure < 0) sure = sees64(hp(L, e0.a), hp(L, e0.b), hp(L, p), hp(L, i));
          }
          unsigned long long m = __ballot(sure != 0);
          if (G < 64) m = m >> lead & ((1ull << G) - 1);
          int nc = -1;
          if (m) nc = __shfl(slot0, lead + __ffsll(m) - 1);
          for (int hb = 64; hb < nh && nc < 0; hb += 64) {  // borders beyond 64 edges (one point at a time here)
            const int h = hb + l;
            const HullEdge e = L.hor[h < nh ? h : 0];
            const unsigned long long m2 = __ballot(h < nh && sees(L, e.a, e.b, p, i));
            if (m2) nc = slotOf(hb + __ffsll(m2) - 1);
          }
          if (mine && h0 == 0) L.conf[i] = static_cast<int16_t>(nc);
        }
        n_lost = 0;
        wsync();
      };
      for (int base = p + 1; base < n; base += 256) {
        int cf[4];
        uint32_t w[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int i = base + 64 * k + l;
          cf[k] = i < n ? L.conf[i] : -1;
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) w[k] = cf[k] >= 0 ? L.fv[cf[k]] : 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const bool s = (w[k] & kFaceVisible) != 0;
          const unsigned long long m = __ballot(s);
          if (!m) continue;
          const int c = __popcll(m);
          if (n_lost + c > list_max) flush();
          if (s) L.hor[n_lost + below(m, l)].pad = static_cast<int16_t>(base + 64 * k + l);
          n_lost += c;
        }
      }
      flush();
    }
    // the cap's faces go, the fan comes
    const int taken = nh < n_free ? nh : n_free;
    for (int j = l; j < nvis; j += 64) L.fv[vis[j]] = kFaceFree;
    wsync();
    auto place = [&](const HullEdge& e) {
      const int out = e.outer >> 2, kk = e.outer & 3;
      L.fv[slot1] = faceWord(e.a, e.b, p);
      L.fv[out] &= kFaceVerts;
      L.fnb[slot1] = static_cast<int16_t>(out);         // across (a, b)
      L.fnb[F + slot1] = static_cast<int16_t>(slot_b);  // across (b, p)
      L.fnb[2 * F + slot1] = static_cast<int16_t>(slot_a);  // across (p, a)
      L.fnb[kk * F + out] = static_cast<int16_t>(slot1);
    };
    if (small) {
      if (edge1) {
        place(e1);
        L.start[e1.a] = -1;
        L.endv[e1.b] = -1;
      }
    } else {
      for (int h = l; h < nh; h += 64) {
        const HullEdge e = L.hor[h];
        check(e, h);
        place(e);
      }
      wsync();
      for (int h = l; h < nh; h += 64) {
        const HullEdge e = L.hor[h];
        L.start[e.a] = -1;
        L.endv[e.b] = -1;
      }
    }
    if (l == 0) L.conf[p] = -2;
    free_top = n_free - taken;
    nf_used += nh - taken;
    wsync();
  }
  if (failed) { finish(kHullFailed); return; }
  // hull vertices are the points the remaining faces use (a point inserted
  // earlier is no longer one once every face around it was removed)
  for (int f = l; f < nf_used; f += 64) {
    const uint32_t w = L.fv[f];
    if (w != kFaceFree) L.start[vertOf(w, 0)] = L.start[vertOf(w, 1)] = L.start[vertOf(w, 2)] = -3;
  }
  wsync();
  // renumber the hull vertices in ascending point order
  int nv = 0;
  for (int base = 0; base < n; base += 64) {
    const int i = base + l;
    const bool v = i < n && L.start[i] == -3;
    const unsigned long long m = __ballot(v);
    if (v) {
      const int id = nv + below(m, l);
      L.start[i] = static_cast<int16_t>(id);
      hull_idx[o + id] = static_cast<uint32_t>(i);
    }
    nv += __popcll(m);
  }
  wsync();
  int nt = 0;
  for (int base = 0; base < nf_used; base += 64) {
    const int f = base + l;
    const uint32_t w = f < nf_used ? L.fv[f] : kFaceFree;
    const bool alive = w != kFaceFree;
    const unsigned long long m = __ballot(alive);
    if (alive) {
      int32_t* tp = tris + 6 * o + 3 * static_cast<uint64_t>(nt + below(m, l));
      for (int k = 0; k < 3; ++k) tp[k] = L.start[vertOf(w, k)];
    }
    nt += __popcll(m);
  }
  if (l == 0) {
    status[set] = kHullOk;
    hull_cnt[set] = static_cast<uint32_t>(nv);
    tri_cnt[set] = static_cast<uint32_t>(nt);
  }
}

int hullsLaunch(mfcl_ctx* ctx, const float* pts, const uint64_t* pt_off, const uint32_t* pt_cnt, uint32_t n_sets,
                int max_points, uint32_t* hull_cnt, uint32_t* hull_idx, uint32_t* tri_cnt, int32_t* tris,
                int32_t* status, hipStream_t s) {
  if (n_sets == 0) return MFCL_OK;
  if (max_points < 4 || max_points > kHullMaxPoints) {
    ctx->err = "max_points out of range [4, " + std::to_string(kHullMaxPoints) + "]";
    return MFCL_E_INVALID;
  }
  if (hullLdsBytes(max_points) > static_cast<size_t>(ctx->max_lds_per_block)) {
    ctx->err = "hull workspace exceeds the LDS of a workgroup";
    return MFCL_E_UNSUPPORTED;
  }
  // The sizes are on the device: each of two classes is a launch over all
  // sets whose blocks leave at once if their set is of the other one, the
  // longer sets first.  (20,011 sets of 8..512 points: one launch 6.98 ms, a
  // line at 256 points 6.72, two at 128 and 256 6.85, three 7.00: what finer
  // slices gain in wavefronts goes into the ends of the launches.)
  constexpr int kClasses = 2;
  const int caps[kClasses] = {256, kHullMaxPoints};
  for (int c = kClasses - 1; c >= 0; --c) {
    const int lo = c ? caps[c - 1] : -1;
    if (c && lo >= max_points) continue;
    const int cap = std::min(caps[c], max_points);
    hullKernel<<<n_sets, 64, hullLdsBytes(cap), s>>>(pts, pt_off, pt_cnt, nullptr, n_sets, lo, cap, max_points,
                                                     hull_cnt, hull_idx, tri_cnt, tris, status);
  }
  MFCL_HIP_TRY(ctx, hipGetLastError());
  return MFCL_OK;
}

// The same with the point counts also on the host: sets are grouped by size
// class (up to 32, 64, 128, 256, 512, 768 points) and each class runs in LDS
// slices of its own size, so small sets are not held to the largest set's
// slice (more wavefronts per CU).  order_dev: n_sets device words for the
// grouped set list (filled here, read by the kernels).
int hullsLaunchClassed(mfcl_ctx* ctx, const float* pts, const uint64_t* pt_off, const uint32_t* pt_cnt,
                       const uint32_t* pt_cnt_host, uint32_t n_sets, uint32_t* order_dev, uint32_t* hull_cnt,
                       uint32_t* hull_idx, uint32_t* tri_cnt, int32_t* tris, int32_t* status, hipStream_t s) {
  if (n_sets == 0) return MFCL_OK;
  constexpr int kClasses = 6;
  const int caps[kClasses] = {32, 64, 128, 256, 512, kHullMaxPoints};
  std::vector<uint32_t> order(n_sets);
  uint32_t count[kClasses] = {}, start[kClasses] = {};
  auto cls = [&](uint32_t n) {
    int c = 0;
    while (c < kClasses - 1 && static_cast<uint32_t>(caps[c]) < n) ++c;
    return c;
  };
  for (uint32_t i = 0; i < n_sets; ++i) ++count[cls(pt_cnt_host[i])];
  for (int c = 1; c < kClasses; ++c) start[c] = start[c - 1] + count[c - 1];
  uint32_t fill[kClasses];
  for (int c = 0; c < kClasses; ++c) fill[c] = start[c];
  // largest classes first, so the longest sets do not start last
  for (uint32_t i = 0; i < n_sets; ++i) order[fill[cls(pt_cnt_host[i])]++] = i;
  MFCL_HIP_TRY(ctx, hipMemcpyAsync(order_dev, order.data(), 4 * static_cast<size_t>(n_sets), hipMemcpyHostToDevice, s));
  for (int c = kClasses - 1; c >= 0; --c) {
    if (count[c] == 0) continue;
    const size_t lds = hullLdsBytes(caps[c]);
    if (lds > static_cast<size_t>(ctx->max_lds_per_block)) {
      ctx->err = "hull workspace exceeds the LDS of a workgroup";
      return MFCL_E_UNSUPPORTED;
    }
    hullKernel<<<count[c], 64, lds, s>>>(pts, pt_off, pt_cnt, order_dev + start[c], count[c], -1, caps[c],
                                         caps[c], hull_cnt, hull_idx, tri_cnt, tris, status);
  }
  MFCL_HIP_TRY(ctx, hipGetLastError());
  // the order list is read by the kernels: keep it until they have run
  MFCL_HIP_TRY(ctx, hipStreamSynchronize(s));
  return MFCL_OK;
}

// ---- shape table of the hulls (mfcl_upload_convex_points) ----------------
//
// One wavefront per hull, after hullKernel: gathers the hull vertices in
// ascending point order into the vertex table, and computes what
// mfcl_upload_shapes computes on the host for a convex shape (interior point
// = vertex mean, convex-inl.h:64-70; the largest |coordinate| for the FP32
// support-scan bound; the 16-float descriptor of the warm-start network) and
// what mfcl_upload_convex_faces builds from the faces for hulls of more than
// 32 vertices (the sorted neighbour list of every vertex in the reference's
// encoding, Convex::FindVertexNeighbors, convex-inl.h:377-409).  Sums run
// sequentially in vertex order, one lane per sum, so they round as the
// host's loops do.
__global__ void __launch_bounds__(64) convexTableKernel(const float* pts, const uint64_t* pt_off,
                                                        const uint32_t* hull_cnt, const uint32_t* hull_idx,
                                                        const uint32_t* tri_cnt, const int32_t* tris,
                                                        const uint32_t* voff, const int64_t* nbr_off, int cap,
                                                        float4* verts, float4* param, double4* interior, float* desc,
                                                        int32_t* nbr) {
#pragma clang fp contract(off)
  extern __shared__ __align__(16) char tab_lds[];
  const uint32_t set = blockIdx.x;
  const int l = laneId64();
  const int nv = static_cast<int>(hull_cnt[set]);
  const int nt = static_cast<int>(tri_cnt[set]);
  const uint64_t o = pt_off[set];
  double* sums = reinterpret_cast<double*>(tab_lds);  // 16 doubles
  float* x = reinterpret_cast<float*>(sums + 16);
  float* y = x + cap;
  float* z = y + cap;
  int32_t* rec = reinterpret_cast<int32_t*>(z + cap);
  int32_t* cur = rec + cap;
  float4* vo = verts + voff[set];
  float rb = 0.f;
  for (int k = l; k < nv; k += 64) {
    const uint64_t q = o + hull_idx[o + k];
    const float px = pts[3 * q], py = pts[3 * q + 1], pz = pts[3 * q + 2];
    x[k] = px;
    y[k] = py;
    z[k] = pz;
    vo[k] = make_float4(px, py, pz, 0.f);
    rb = fmaxf(rb, fmaxf(fabsf(px), fmaxf(fabsf(py), fabsf(pz))));
  }
  float mx[3] = {0.f, 0.f, 0.f};
  for (int k = l; k < nv; k += 64) {
    mx[0] = fmaxf(mx[0], fabsf(x[k]));
    mx[1] = fmaxf(mx[1], fabsf(y[k]));
    mx[2] = fmaxf(mx[2], fabsf(z[k]));
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    rb = fmaxf(rb, __shfl_xor(rb, off));
    mx[0] = fmaxf(mx[0], __shfl_xor(mx[0], off));
    mx[1] = fmaxf(mx[1], __shfl_xor(mx[1], off));
    mx[2] = fmaxf(mx[2], __shfl_xor(mx[2], off));
  }
  __syncthreads();
  // coordinate sums (lanes 0-2), radius sum and maximum (lane 3)
  if (l < 3) {
    const float* c = l == 0 ? x : (l == 1 ? y : z);
    double sacc = 0;
    for (int k = 0; k < nv; ++k) sacc += c[k];
    sums[l] = sacc;
  } else if (l == 3) {
    double rmax = 0, rsum = 0;
    for (int k = 0; k < nv; ++k) {
      const double px = x[k], py = y[k], pz = z[k];
      const double r = sqrt(px * px + py * py + pz * pz);
      rmax = fmax(rmax, r);
      rsum += r;
    }
    sums[3] = rmax;
    sums[4] = rsum;
  }
  __syncthreads();
  const double mean[3] = {sums[0] / nv, sums[1] / nv, sums[2] / nv};
  // second moments about the mean (lanes 0-5)
  if (l < 6) {
    const int i0 = l < 3 ? l : (l == 5 ? 1 : 0);
    const int i1 = l < 3 ? l : (l == 3 ? 1 : 2);
    const float* c0 = i0 == 0 ? x : (i0 == 1 ? y : z);
    const float* c1 = i1 == 0 ? x : (i1 == 1 ? y : z);
    double m = 0;
    for (int k = 0; k < nv; ++k) {
      const double u = c0[k] - mean[i0], w = c1[k] - mean[i1];
      m += u * w;
    }
    sums[8 + l] = m;
  }
  __syncthreads();
  if (l == 0) {
    const double inv = 1.0 / nv;
    interior[set] = double4{sums[0] * inv, sums[1] * inv, sums[2] * inv, 0};
    param[set] = make_float4(0.f, 0.f, 0.f, rb);
  }
  if (l < 16) {
    float d;
    if (l < 3) d = l == 0 ? mx[0] : (l == 1 ? mx[1] : mx[2]);
    else if (l < 6) d = static_cast<float>(mean[l - 3]);
    else if (l < 12) d = static_cast<float>(sums[8 + l - 6] / nv);
    else if (l == 12) d = static_cast<float>(log2(static_cast<double>(nv)) / 9.0);
    else if (l == 13) d = static_cast<float>(sums[3]);
    else if (l == 14) d = static_cast<float>(sums[4] / nv);
    else d = 1.f;
    desc[16 * static_cast<uint64_t>(set) + l] = d;
  }
  const int64_t no = nbr_off[set];
  if (no < 0) return;
  // neighbour records: on a closed, consistently oriented triangulation the
  // neighbours of a vertex are the successors of it in its triangles, each
  // once, so its degree is its triangle count
  int32_t* tab = nbr + no;
  const int32_t* tr = tris + 6 * o;
  for (int v = l; v < nv; v += 64) cur[v] = 0;
  __syncthreads();
  for (int t = l; t < nt; t += 64) {
    atomicAdd(&cur[tr[3 * t]], 1);
    atomicAdd(&cur[tr[3 * t + 1]], 1);
    atomicAdd(&cur[tr[3 * t + 2]], 1);
  }
  __syncthreads();
  int run = nv;
  for (int base = 0; base < nv; base += 64) {
    const int v = base + l;
    const int deg = v < nv ? cur[v] : 0;
    const int len = v < nv ? 1 + deg : 0;
    int incl = len;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int t = __shfl_up(incl, off);
      if (l >= off) incl += t;
    }
    if (v < nv) {
      const int r = run + incl - len;
      rec[v] = r;
      tab[v] = r;
      tab[r] = deg;
    }
    run += __shfl(incl, 63);
  }
  __syncthreads();
  for (int v = l; v < nv; v += 64) cur[v] = 0;
  __syncthreads();
  for (int t = l; t < nt; t += 64) {
    const int a = tr[3 * t], b = tr[3 * t + 1], c = tr[3 * t + 2];
    tab[rec[a] + 1 + atomicAdd(&cur[a], 1)] = b;
    tab[rec[b] + 1 + atomicAdd(&cur[b], 1)] = c;
    tab[rec[c] + 1 + atomicAdd(&cur[c], 1)] = a;
  }
  __syncthreads();
  for (int v = l; v < nv; v += 64) {
    int32_t* r = tab + rec[v] + 1;
    const int deg = cur[v];
    for (int i = 1; i < deg; ++i) {
      const int32_t key = r[i];
      int j = i - 1;
      while (j >= 0 && r[j] > key) {
        r[j + 1] = r[j];
        --j;
      }
      r[j + 1] = key;
    }
  }
}

namespace {
// Device allocations of one call, released on every return.
struct TempDev {
  std::vector<void*> p;
  ~TempDev() {
    for (void* q : p) (void)hipFree(q);
  }
  template <class T>
  T* get(mfcl_ctx* ctx, size_t count, int& rc) {
    void* q = nullptr;
    if (hipMalloc(&q, std::max<size_t>(count, 1) * sizeof(T)) != hipSuccess) {
      (void)hipGetLastError();
      ctx->err = "out of device memory building the convex shape table";
      rc = MFCL_E_NOMEM;
      return nullptr;
    }
    p.push_back(q);
    return static_cast<T*>(q);
  }
};

template <class T>
int allocTable(mfcl_ctx* ctx, T** dst, size_t count) {
  void* q = nullptr;
  if (hipMalloc(&q, std::max<size_t>(count, 1) * sizeof(T)) != hipSuccess) {
    (void)hipGetLastError();
    ctx->err = "out of device memory building the convex shape table";
    return MFCL_E_NOMEM;
  }
  *dst = static_cast<T*>(q);
  return MFCL_OK;
}
}  // namespace

int uploadConvexPoints(mfcl_ctx* ctx, const float* points, const uint64_t* pt_off, const uint32_t* pt_cnt,
                       uint32_t n_sets, uint32_t* hull_cnt_out) {
  uint64_t total = 0;
  uint32_t maxp = 4;
  for (uint32_t i = 0; i < n_sets; ++i) {
    if (pt_cnt[i] > static_cast<uint32_t>(kHullMaxPoints)) {
      ctx->err = "point set " + std::to_string(i) + " has more than " + std::to_string(kHullMaxPoints) + " points";
      return MFCL_E_INVALID;
    }
    total = std::max<uint64_t>(total, pt_off[i] + pt_cnt[i]);
    maxp = std::max(maxp, pt_cnt[i]);
  }
  const hipStream_t s = ctx->stream;
  int rc = MFCL_OK;
  TempDev tmp;
  float* dp = tmp.get<float>(ctx, 3 * total, rc);
  uint64_t* doff = rc ? nullptr : tmp.get<uint64_t>(ctx, n_sets, rc);
  uint32_t* dcnt = rc ? nullptr : tmp.get<uint32_t>(ctx, n_sets, rc);
  uint32_t* dhc = rc ? nullptr : tmp.get<uint32_t>(ctx, n_sets, rc);
  uint32_t* dtc = rc ? nullptr : tmp.get<uint32_t>(ctx, n_sets, rc);
  int32_t* dst = rc ? nullptr : tmp.get<int32_t>(ctx, n_sets, rc);
  uint32_t* dhi = rc ? nullptr : tmp.get<uint32_t>(ctx, total, rc);
  int32_t* dtr = rc ? nullptr : tmp.get<int32_t>(ctx, 6 * total, rc);
  uint32_t* dord = rc ? nullptr : tmp.get<uint32_t>(ctx, n_sets, rc);
  if (rc) return rc;
  MFCL_HIP_TRY(ctx, hipMemcpyAsync(dp, points, 12 * total, hipMemcpyHostToDevice, s));
  MFCL_HIP_TRY(ctx, hipMemcpyAsync(doff, pt_off, 8 * static_cast<size_t>(n_sets), hipMemcpyHostToDevice, s));
  MFCL_HIP_TRY(ctx, hipMemcpyAsync(dcnt, pt_cnt, 4 * static_cast<size_t>(n_sets), hipMemcpyHostToDevice, s));
  if ((rc = hullsLaunchClassed(ctx, dp, doff, dcnt, pt_cnt, n_sets, dord, dhc, dhi, dtc, dtr, dst, s))) return rc;
  std::vector<uint32_t> hc(n_sets), tc(n_sets);
  std::vector<int32_t> st(n_sets);
  MFCL_HIP_TRY(ctx, hipMemcpyAsync(hc.data(), dhc, 4 * static_cast<size_t>(n_sets), hipMemcpyDeviceToHost, s));
  MFCL_HIP_TRY(ctx, hipMemcpyAsync(tc.data(), dtc, 4 * static_cast<size_t>(n_sets), hipMemcpyDeviceToHost, s));
  MFCL_HIP_TRY(ctx, hipMemcpyAsync(st.data(), dst, 4 * static_cast<size_t>(n_sets), hipMemcpyDeviceToHost, s));
  MFCL_HIP_TRY(ctx, hipStreamSynchronize(s));
  for (uint32_t i = 0; i < n_sets; ++i) {
    if (st[i] == kHullOk) continue;
    static const char* why[] = {"", "is degenerate (fewer than 4 points, or all on one plane)",
                                "has too many points", "has no hull within the tolerance (near-degenerate input)"};
    ctx->err = "point set " + std::to_string(i) + " " + why[st[i] >= 1 && st[i] <= 3 ? st[i] : 3];
    return MFCL_E_INVALID;
  }
  // vertex and adjacency offsets; a hull's record area holds nv offsets and
  // nv records of 1 + degree entries, and the degrees sum to 3 nt
  std::vector<uint32_t> voff(n_sets);
  std::vector<int64_t> noff(n_sets, -1);
  uint64_t nverts = 0, nnbr = 0;
  for (uint32_t i = 0; i < n_sets; ++i) {
    voff[i] = static_cast<uint32_t>(nverts);
    nverts += hc[i];
    if (hc[i] > 32) {
      noff[i] = static_cast<int64_t>(nnbr);
      nnbr += 2 * static_cast<uint64_t>(hc[i]) + 3 * static_cast<uint64_t>(tc[i]);
    }
  }
  if (nverts > 0xFFFFFFFFull || nnbr > 0x7FFFFFFFull) {
    ctx->err = "convex tables exceed 2^32 vertices or 2^31 adjacency entries";
    return MFCL_E_INVALID;
  }
  uint32_t* dvoff = tmp.get<uint32_t>(ctx, n_sets, rc);
  if (rc) return rc;
  MFCL_HIP_TRY(ctx, hipMemcpyAsync(dvoff, voff.data(), 4 * static_cast<size_t>(n_sets), hipMemcpyHostToDevice, s));
  freeShapes(ctx);
  const std::vector<int32_t> type(n_sets, MFCL_SHAPE_CONVEX);
  auto fail = [&](int r) {
    freeShapes(ctx);
    return r;
  };
  if ((rc = allocTable(ctx, &ctx->d_type, n_sets)) || (rc = allocTable(ctx, &ctx->d_param, n_sets)) ||
      (rc = allocTable(ctx, &ctx->d_voff, n_sets)) || (rc = allocTable(ctx, &ctx->d_vcnt, n_sets)) ||
      (rc = allocTable(ctx, &ctx->d_verts, nverts)) || (rc = allocTable(ctx, &ctx->d_interior, n_sets)) ||
      (rc = allocTable(ctx, &ctx->d_desc, 16 * static_cast<size_t>(n_sets))) ||
      (rc = allocTable(ctx, &ctx->d_nbr, nnbr + 32)) || (rc = allocTable(ctx, &ctx->d_nbr_off, n_sets)) ||
      (rc = allocTable(ctx, &ctx->d_seed, 8 * static_cast<size_t>(n_sets))))
    return fail(rc);
  // walk blocks: 128 B per vertex; when the device cannot hold them the
  // walks read the adjacency table instead (same results, slower)
  if (hipMalloc(reinterpret_cast<void**>(&ctx->d_wblk), 8 * sizeof(float4) * std::max<uint64_t>(nverts, 1)) !=
      hipSuccess) {
    ctx->d_wblk = nullptr;
    (void)hipGetLastError();
  }
  auto chk = [&](hipError_t e) {
    if (e == hipSuccess) return MFCL_OK;
    ctx->err = std::string("HIP error: ") + hipGetErrorString(e);
    return MFCL_E_HIP;
  };
  if ((rc = chk(hipMemcpyAsync(ctx->d_type, type.data(), 4 * static_cast<size_t>(n_sets), hipMemcpyHostToDevice, s))) ||
      (rc = chk(hipMemcpyAsync(ctx->d_voff, voff.data(), 4 * static_cast<size_t>(n_sets), hipMemcpyHostToDevice, s))) ||
      (rc = chk(hipMemcpyAsync(ctx->d_vcnt, dhc, 4 * static_cast<size_t>(n_sets), hipMemcpyDeviceToDevice, s))) ||
      (rc = chk(hipMemcpyAsync(ctx->d_nbr_off, noff.data(), 8 * static_cast<size_t>(n_sets), hipMemcpyHostToDevice,
                               s))) ||
      (rc = chk(hipMemsetAsync(ctx->d_nbr + nnbr, 0, 32 * sizeof(int32_t), s))))
    return fail(rc);
  const size_t lds = 20 * static_cast<size_t>(maxp) + 16 * sizeof(double) + 64;
  convexTableKernel<<<n_sets, 64, lds, s>>>(dp, doff, dhc, dhi, dtc, dtr, dvoff, ctx->d_nbr_off,
                                             static_cast<int>(maxp), ctx->d_verts, ctx->d_param, ctx->d_interior,
                                             ctx->d_desc, ctx->d_nbr);
  if ((rc = chk(hipGetLastError()))) return fail(rc);
  ctx->n_shapes = n_sets;
  ctx->n_verts_alloc = std::max<uint64_t>(nverts, 1);
  ctx->h_vcnt = hc;
  ctx->h_voff = voff;
  ctx->h_type = type;
  if ((rc = computeWalkSeeds(ctx))) return fail(rc);
  if (hull_cnt_out) std::memcpy(hull_cnt_out, hc.data(), 4 * static_cast<size_t>(n_sets));
  return MFCL_OK;
}

}  // namespace mfcl
