// Batched convex narrowphase for gfx950: the stages of a query on its
// stream (no host round trip), its workspace, and the support walk's tables.
//
//   small batches and the boolean mode: wave.hip, one wavefront per pair
//     from the closed form to EPA;
//   large ones: costKey / bucketScan / bucketScatter, a counting sort of
//     the pairs by (closed form or search, walking shapes, log2 of the hull
//     vertex count) so the lanes of a wavefront run loops of similar trip
//     count; lane.hip, GJK with one pair per lane, whose intersecting pairs
//     append their simplex to a queue; epa.hip, a wavefront per queued pair;
//   both: pairs that outgrow their LDS polytope continue at full capacity
//     (epa.hip).
#include <hip/hip_runtime.h>

#include <mutex>

#include "gjk_lane.h"
#include "pair_dev.h"

namespace mfcl {

constexpr int kBuckets = 128;

MFCL_D int shapeCost(const ShapeTables& T, uint32_t i) {
  return T.type[i] == kConvex ? static_cast<int>(T.vert_cnt[i]) : 1;
}

// Closed-form pairs first (4 buckets per octave of the summed vertex
// count), then the others by how many of the two shapes walk (0, 1, 2: a
// wavefront's walks and cooperative scans then rarely mix) and, within that,
// 3 buckets per octave of the summed vertex count.
MFCL_D uint8_t pairKey(const ShapeTables& T, const PairIO& io, uint64_t i, const Params& P) {
  const uint32_t a = io.pa[i], b = io.pb[i];
  if (a >= P.n_shapes || b >= P.n_shapes) return 0;
  const bool cf = P.mode == MFCL_MODE_COLLIDE && closedForm(T.type[a], T.type[b]);
  const int cost = shapeCost(T, a) + shapeCost(T, b);
  if (cf) return static_cast<uint8_t>(min(63, static_cast<int>(4.0f * log2f(static_cast<float>(cost)))));
  auto walks = [&](uint32_t k) { return T.type[k] == kConvex && T.nbr_off && T.nbr_off[k] >= 0; };
  const int c = (walks(a) ? 1 : 0) + (walks(b) ? 1 : 0);
  const int lvl = max(0, min(20, static_cast<int>(3.0f * log2f(static_cast<float>(cost))) - 10));
  return static_cast<uint8_t>(64 + 21 * c + lvl);
}

// Block-local histogram in LDS, one global atomic per bin per block.
__global__ void __launch_bounds__(kBlock) costKeyKernel(ShapeTables T, PairIO io, uint64_t n, Params P,
                                                        uint8_t* key, uint32_t* hist) {
  __shared__ uint32_t h[kBuckets];
  if (threadIdx.x < kBuckets) h[threadIdx.x] = 0;
  __syncthreads();
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) {
    const uint8_t k = pairKey(T, io, i, P);
    key[i] = k;
    atomicAdd(&h[k], 1u);
  }
  __syncthreads();
  if (threadIdx.x < kBuckets && h[threadIdx.x]) atomicAdd(&hist[threadIdx.x], h[threadIdx.x]);
}

__global__ void bucketScanKernel(uint32_t* hist, uint32_t* offs) {
  // single block of kBuckets threads: exclusive scan
  __shared__ uint32_t s[kBuckets];
  const int t = threadIdx.x;
  s[t] = hist[t];
  __syncthreads();
  if (t == 0) {
    uint32_t acc = 0;
    for (int k = 0; k < kBuckets; ++k) {
      const uint32_t v = s[k];
      s[k] = acc;
      acc += v;
    }
  }
  __syncthreads();
  offs[t] = s[t];
}

// Each block reserves its bins' ranges with one atomic per bin, then places
// its pairs with LDS atomics (order inside a bin is irrelevant).
__global__ void __launch_bounds__(kBlock) bucketScatterKernel(const uint8_t* key, uint64_t n, uint32_t* offs,
                                                              uint32_t* order) {
  __shared__ uint32_t cnt[kBuckets], base[kBuckets];
  if (threadIdx.x < kBuckets) cnt[threadIdx.x] = 0;
  __syncthreads();
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  uint8_t k = 0;
  uint32_t local = 0;
  if (i < n) {
    k = key[i];
    local = atomicAdd(&cnt[k], 1u);
  }
  __syncthreads();
  if (threadIdx.x < kBuckets && cnt[threadIdx.x]) base[threadIdx.x] = atomicAdd(&offs[threadIdx.x], cnt[threadIdx.x]);
  __syncthreads();
  if (i < n) order[base[k] + local] = static_cast<uint32_t>(i);
}

__global__ void zeroKernel(uint32_t* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// Seed vertices of the support walk (convex-inl.h:151-199): per walking
// hull, the first vertex attaining the maximum of +x, -x, +y, -y, +z, -z
// (convex-inl.h:133-149; the dot product with a unit axis is the coordinate).
__global__ void walkSeedKernel(ShapeTables T, uint32_t n, int* seed) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || T.nbr_off[i] < 0) return;
  const float4* v = T.verts + T.vert_off[i];
  const int nv = static_cast<int>(T.vert_cnt[i]);
  int idx[6] = {0, 0, 0, 0, 0, 0};
  double best[6];
  {
    const float4 q = v[0];
    best[0] = q.x; best[1] = -static_cast<double>(q.x);
    best[2] = q.y; best[3] = -static_cast<double>(q.y);
    best[4] = q.z; best[5] = -static_cast<double>(q.z);
  }
  for (int k = 1; k < nv; ++k) {
    const float4 q = v[k];
    const double c[6] = {q.x, -static_cast<double>(q.x), q.y, -static_cast<double>(q.y), q.z,
                         -static_cast<double>(q.z)};
#pragma unroll
    for (int a = 0; a < 6; ++a)
      if (c[a] > best[a]) {
        best[a] = c[a];
        idx[a] = k;
      }
  }
#pragma unroll
  for (int a = 0; a < 6; ++a) seed[8 * static_cast<uint64_t>(i) + a] = idx[a];
  seed[8 * static_cast<uint64_t>(i) + 6] = seed[8 * static_cast<uint64_t>(i) + 7] = 0;
}

// Per walking hull (one block each, its threads over the vertices): every
// vertex's neighbour-record offset goes into the vertex's fourth word (read
// together with the vertex by the table walk).
__global__ void walkRecKernel(ShapeTables T, float4* verts_rw) {
  const uint32_t i = blockIdx.x;
  if (T.nbr_off[i] < 0) return;
  const int nv = static_cast<int>(T.vert_cnt[i]);
  const int* tab = T.nbr + T.nbr_off[i];
  for (int k = threadIdx.x; k < nv; k += blockDim.x) {
    const uint64_t g = T.vert_off[i] + static_cast<uint64_t>(k);
    verts_rw[g].w = __int_as_float(tab[k]);
  }
}

// Walk blocks (one block of threads per walking hull of at most 65535
// vertices): per vertex 8 float4 = (x, y, z, neighbour count), the first
// eight neighbour ids as 16-bit pairs, then those neighbours' x, y, z
// (24 floats, zero past the count).  Runs after walkRecKernel has written
// the vertices' fourth words; reads only their coordinates.
__global__ void walkBlkKernel(ShapeTables T, float4* wblk) {
  const uint32_t i = blockIdx.x;
  if (T.nbr_off[i] < 0) return;
  const int nv = static_cast<int>(T.vert_cnt[i]);
  if (nv > 65535) return;
  const int* tab = T.nbr + T.nbr_off[i];
  const float4* v = T.verts + T.vert_off[i];
  for (int k = threadIdx.x; k < nv; k += blockDim.x) {
    const uint64_t g = T.vert_off[i] + static_cast<uint64_t>(k);
    const int* rec = tab + tab[k];
    const int cnt = rec[0];
    uint32_t u[4] = {0, 0, 0, 0};
    float f[24];
#pragma unroll
    for (int j = 0; j < 24; ++j) f[j] = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j >= cnt) break;
      const int nb = rec[1 + j];
      u[j >> 1] |= static_cast<uint32_t>(nb) << (16 * (j & 1));
      const float4 q = v[nb];
      f[3 * j] = q.x;
      f[3 * j + 1] = q.y;
      f[3 * j + 2] = q.z;
    }
    const float4 self = v[k];
    float4* o = wblk + 8 * g;
    o[0] = make_float4(self.x, self.y, self.z, __int_as_float(cnt));
    o[1] = make_float4(__uint_as_float(u[0]), __uint_as_float(u[1]), __uint_as_float(u[2]), __uint_as_float(u[3]));
#pragma unroll
    for (int j = 0; j < 6; ++j) o[2 + j] = make_float4(f[4 * j], f[4 * j + 1], f[4 * j + 2], f[4 * j + 3]);
  }
}

int computeWalkSeeds(mfcl_ctx* ctx) {
  ShapeTables T{ctx->d_type, ctx->d_param, ctx->d_voff, ctx->d_vcnt, ctx->d_verts, ctx->d_nbr, ctx->d_nbr_off,
                ctx->d_seed, ctx->d_wblk};
  const uint32_t n = ctx->n_shapes;
  walkSeedKernel<<<(n + 255) / 256, 256, 0, ctx->stream>>>(T, n, ctx->d_seed);
  walkRecKernel<<<n, 64, 0, ctx->stream>>>(T, ctx->d_verts);
  if (ctx->d_wblk) walkBlkKernel<<<n, 64, 0, ctx->stream>>>(T, ctx->d_wblk);
  MFCL_HIP_TRY(ctx, hipGetLastError());
  MFCL_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
  return MFCL_OK;
}

// Workspace of one convex query over n pairs, carved from one device buffer
// (256-byte aligned pieces): the counters block (2 KB: bucket histogram and
// offsets, EpaCounts at byte 1024, 64-bit work counters at 1536), the bucket order (4n B) and
// keys (n B), the EPA queue and overflow queue (one QEntry per pair each,
// the most that can be queued) and the lane kernel's direction slots
// (kLaneDirDoubles doubles per wavefront of its grid).
static size_t align256(size_t b) { return (b + 255) & ~static_cast<size_t>(255); }
static size_t laneDirBytes(uint64_t n) {
  const uint64_t waves = (n + kBlock - 1) / kBlock * (kBlock / 64);
  return static_cast<size_t>(waves) * kLaneDirDoubles * sizeof(double);
}
size_t epaArenaBytes(int slices) { return static_cast<size_t>(slices) * kEpaArenaSlice; }
size_t convexWsBytes(uint64_t n, size_t arena_bytes) {
  if (n == 0) n = 1;
  return align256(2048) + align256(4 * n) + align256(n) + 2 * align256(n * sizeof(QEntry)) +
         align256(laneDirBytes(n)) + align256(arena_bytes);
}
uint64_t convexWsMaxPairs(size_t bytes, size_t arena_bytes) {
  // convexWsBytes grows by at least sizeof(QEntry) per pair: bisect
  uint64_t lo = 0, hi = bytes / (2 * sizeof(QEntry)) + 1;
  while (lo < hi) {
    const uint64_t mid = (lo + hi + 1) / 2;
    if (convexWsBytes(mid, arena_bytes) <= bytes) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}
bool carveConvexWs(void* base, size_t bytes, uint64_t n, size_t arena_bytes, ConvexWs& w) {
  if (!base || convexWsBytes(n, arena_bytes) > bytes) return false;
  char* p = static_cast<char*>(base);
  auto take = [&](size_t b) {
    char* r = p;
    p += align256(b);
    return r;
  };
  w.misc = reinterpret_cast<uint32_t*>(take(2048));
  w.order = reinterpret_cast<uint32_t*>(take(4 * (n ? n : 1)));
  w.key = reinterpret_cast<uint8_t*>(take(n ? n : 1));
  w.queue = take((n ? n : 1) * sizeof(QEntry));
  w.oflow = take((n ? n : 1) * sizeof(QEntry));
  w.lane_dirs = reinterpret_cast<double*>(take(laneDirBytes(n ? n : 1)));
  w.arena = arena_bytes ? take(arena_bytes) : nullptr;
  w.arena_bytes = arena_bytes;
  return true;
}

// Workspace of mfcl_convex_query_static_dev, for callers that cannot
// allocate: a file-scope device array, one copy per GPU (its own address on
// each), held until the process ends.  Host code never passes the array's
// name to a kernel (on the host it is only a stand-in for the symbol): it
// uses the device address that staticScratch() looked up once per device.
static __device__ __align__(256) char scratch[kStaticScratchBytes];

namespace {
constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxScratchDevices] = {};
}  // namespace

int staticScratch(int device, void** out) {
  *out = nullptr;
  if (device < 0 || device >= kMaxScratchDevices) return MFCL_E_INVALID;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[device]) {
    // the caller has made `device` current
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || p == nullptr) return MFCL_E_HIP;
    g_scratch_ptr[device] = p;
  }
  *out = g_scratch_ptr[device];
  return MFCL_OK;
}

uint64_t staticScratchMaxPairs() {
  return convexWsMaxPairs(kStaticScratchBytes, epaArenaBytes(kStaticArenaSlices));
}


// Batches of at most this many pairs run one pair per wavefront (wave.hip);
// larger ones fill the chip with one pair per lane.  A lane's pair takes
// 1.1-1.5 ms however few there are, a wavefront's 40-100 us.  The lines lie
// where the wavefronts win both alone and with two other batches beside them
// (us per batch on 256 CUs, lane / wave; hulls of 8..512 vertices, contacts
// 8..256); alone they win to beyond them:
//   distance    24,576 pairs: alone 1413 / 868, beside others 560 / 500
//               32,768 pairs: alone 1550 / 1120, beside others 574 / 677
//   penetration  8,192 pairs: alone 1663 / 1298, beside others 747 / 699
//               16,384 pairs: alone 1668 / 1494, beside others 773 / 892
constexpr uint64_t kWavePairsSd = 24576, kWavePairsPen = 8192;

int convexQueryLaunch(mfcl_ctx* ctx, const uint32_t* pa, const uint32_t* pb, const float* posea,
                      const float* poseb, const float* guess, uint64_t n, const mfcl_request* req,
                      mfcl_convex_result* out, mfcl_contact* contacts, const ConvexWs& ws, hipStream_t s) {
  if (n == 0) return MFCL_OK;
  if (ctx->n_shapes == 0) {
    ctx->err = "no shapes uploaded";
    return MFCL_E_STATE;
  }
  if (n > 0xFFFFFFFFull) {
    ctx->err = "too many pairs in one query";
    return MFCL_E_INVALID;
  }
  if (req->epa_max_faces < 4 || req->epa_max_faces > 8192) {
    ctx->err = "epa_max_faces out of range [4, 8192]";
    return MFCL_E_INVALID;
  }
  if (req->use_guess && guess == nullptr) {
    ctx->err = "use_guess set but guess3 is NULL";
    return MFCL_E_INVALID;
  }
  Params P;
  P.mode = req->mode;
  P.max_contacts = req->max_contacts;
  P.penetration = req->penetration;
  P.gjk_max_it = req->gjk_max_iterations;
  P.gjk_tol = req->gjk_tolerance;
  P.epa_max_faces = req->epa_max_faces;
  P.epa_max_it = req->epa_max_iterations;
  P.epa_tol = req->epa_tolerance;
  P.use_guess = req->use_guess;
  P.n_shapes = ctx->n_shapes;

  if (contacts && !(P.mode == MFCL_MODE_COLLIDE && P.penetration)) {
    ctx->err = "a contact array needs a collide request with penetration";
    return MFCL_E_INVALID;
  }
  // the line of the error is part of the interface: 674 faces of 241 bytes
  // each (1.51 vertices and edges a face), also where records take less
  constexpr int kMaxFaces = 674;
  if (req->epa_max_faces > kMaxFaces) {
    ctx->err = "epa_max_faces = " + std::to_string(req->epa_max_faces) + ": the LDS of a wavefront holds at most " +
               std::to_string(kMaxFaces);
    return MFCL_E_UNSUPPORTED;
  }
  const size_t full_slice = epaFullBytes(req->epa_max_faces);
  if (full_slice > static_cast<size_t>(ctx->max_lds_per_block)) {
    ctx->err = "epa_max_faces = " + std::to_string(req->epa_max_faces) + " needs " + std::to_string(full_slice) +
               " bytes of LDS per wavefront; this device allows " + std::to_string(ctx->max_lds_per_block);
    return MFCL_E_UNSUPPORTED;
  }
  uint32_t* hist = ws.misc;
  uint32_t* offs = hist + kBuckets;
  ConvexJob j;
  j.qcount = offs + kBuckets;
  j.sc = reinterpret_cast<unsigned long long*>(reinterpret_cast<char*>(ws.misc) + 1536);
  ctx->d_counters = reinterpret_cast<uint64_t*>(j.sc);
  ctx->d_qcounts = j.qcount;
  j.queue = static_cast<QEntry*>(ws.queue);
  j.oflow = static_cast<QEntry*>(ws.oflow);
  j.arena = static_cast<char*>(ws.arena);
  j.arena_bytes = ws.arena_bytes;
  j.T = ShapeTables{ctx->d_type, ctx->d_param, ctx->d_voff, ctx->d_vcnt, ctx->d_verts, ctx->d_nbr, ctx->d_nbr_off,
                    ctx->d_seed, ctx->d_wblk};
  j.interior = ctx->d_interior;
  j.io = PairIO{pa, pb, posea, poseb, guess, out, contacts, contacts ? (P.max_contacts < 4 ? P.max_contacts : 4) : 0};
  j.P = P;
  j.n = n;
  j.mode = P.mode == MFCL_MODE_SIGNED_DISTANCE ? kModeSd : (P.penetration ? kModePen : kModeBool);
  j.s = s;
  // the boolean mode (MPR first) always takes a wavefront per pair; knob
  // values above 1 force it, 1 forces one lane per pair
  const int group = ctx->tune.gjk_group;
  const bool waves = j.mode == kModeBool || group > 1 || 
                     (group == 0 && n <= (j.mode == kModeSd ? kWavePairsSd : kWavePairsPen));
  const unsigned nb = static_cast<unsigned>((n + kBlock - 1) / kBlock);
  if (ctx->timing) MFCL_HIP_TRY(ctx, hipEventRecord(ctx->ev[0], s));
  zeroKernel<<<1, 512, 0, s>>>(hist, 512);
  if (!waves) {
    costKeyKernel<<<nb, kBlock, 0, s>>>(j.T, j.io, n, P, ws.key, hist);
    bucketScanKernel<<<1, kBuckets, 0, s>>>(hist, offs);
    bucketScatterKernel<<<nb, kBlock, 0, s>>>(ws.key, n, offs, ws.order);
  }
  MFCL_HIP_TRY(ctx, hipGetLastError());
  if (ctx->timing) MFCL_HIP_TRY(ctx, hipEventRecord(ctx->ev[1], s));
  if (int rc = waves ? waveLaunch(ctx, j) : laneLaunch(ctx, j, ws.order, ws.lane_dirs)) return rc;
  if (ctx->timing) MFCL_HIP_TRY(ctx, hipEventRecord(ctx->ev[2], s));
  if (!waves)
    if (int rc = epaQueueLaunch(ctx, j)) return rc;
  if (j.mode != kModeBool)
    if (int rc = epaFullLaunch(ctx, j)) return rc;
  if (ctx->timing) MFCL_HIP_TRY(ctx, hipEventRecord(ctx->ev[3], s));
  return MFCL_OK;
}

}  // namespace mfcl
