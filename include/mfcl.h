/*
 * mfcl -- MI355X-native batched narrowphase / BVH collision library, C ABI.
 *
 * The boundary replaces per-pair calls into mind-fcl's C++ API with batched
 * calls over device-resident data.  Every entry point names the reference
 * interface it stands in for.  No C++ or HIP types cross this ABI: plain
 * pointers, sizes and PODs only; streams are passed as void* (hipStream_t).
 *
 * Conventions
 *  - every function returns 0 (MFCL_OK) or a negative MFCL_E_* code; the
 *    message of the last failure is available from mfcl_last_error();
 *  - "_dev" entry points take device pointers and enqueue on the given
 *    stream without synchronising and without allocating: their workspace
 *    is sized beforehand by mfcl_reserve / mfcl_reserve_arm (or at upload),
 *    and a query larger than it fails with MFCL_E_STATE; the others take
 *    host pointers, size their workspace themselves, copy in, run, copy out
 *    and synchronise;
 *  - a context owns its geometry and workspace; one context per stream;
 *    distinct contexts may be used from distinct threads.
 *  - poses are FP32 (tx, ty, tz, qw, qx, qy, qz); the quaternion is
 *    renormalised in FP64 on the device.
 */
#ifndef MFCL_H_
#define MFCL_H_

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define MFCL_OK 0
#define MFCL_E_INVALID (-1)
#define MFCL_E_HIP (-2)
#define MFCL_E_NOMEM (-3)
#define MFCL_E_UNSUPPORTED (-4)
#define MFCL_E_STATE (-5)

/* Shape type codes, equal to cvx_collide::GJKShapeType
 * (include/fcl/cvx_collide/gjk_shape.h:12-28). */
#define MFCL_SHAPE_BOX 0      /* params: full side lengths x, y, z (fcl::Box::side) */
#define MFCL_SHAPE_SPHERE 1   /* params: radius */
#define MFCL_SHAPE_CAPSULE 3  /* params: radius, full length lz (fcl::Capsule) */
#define MFCL_SHAPE_CYLINDER 5 /* params: radius, full length lz (fcl::Cylinder) */
#define MFCL_SHAPE_CONVEX 100 /* vertices in vert_off/vert_cnt (fcl::Convex) */

#define MFCL_MODE_COLLIDE 0         /* fcl::collide semantics */
#define MFCL_MODE_SIGNED_DISTANCE 1 /* GJKSolver::shapeSignedDistance semantics */

typedef struct mfcl_ctx mfcl_ctx;

/* Query parameters.  Mirrors CollisionRequest (include/fcl/narrowphase/
 * collision_request.h:51-95) plus the GJKSolver fields that fcl::collide
 * fills from it (include/fcl/narrowphase/collision_interface-inl.h:18-20,
 * gjk_solver-inl.h:1121-1130). */
typedef struct mfcl_request {
  int32_t mode;               /* MFCL_MODE_* */
  int32_t max_contacts;       /* collide mode; 0 returns no results (reference warns and returns 0) */
  int32_t penetration;        /* collide mode: 1 = useDefaultPenetration (GJK/EPA), 0 = boolean only */
  int32_t gjk_max_iterations; /* default 128 */
  double gjk_tolerance;       /* default 1e-6 (binaryCollisionTolerance) */
  int32_t epa_max_faces;      /* default 256 */
  int32_t epa_max_iterations; /* default 255 */
  double epa_tolerance;       /* default 1e-6 (distanceTolerance) */
  int32_t use_guess;          /* 1: per-pair initial GJK guess supplied (GJKSolver::gjk_guess) */
  int32_t reserved;
} mfcl_request;

/* Fills *req with the reference defaults for the given mode. */
void mfcl_request_defaults(mfcl_request* req, int32_t mode);

/* Per-pair result (128 bytes).  World frame throughout.
 *  collide mode: hit, n_contacts (<= max_contacts), and contact 0 as the
 *    reference's CollisionResult would hold it first (normal from shape a to
 *    shape b, pos, depth); distance = -depth when hit.
 *  signed-distance mode: hit = (distance < 0); distance > 0 separation,
 *    < 0 minus penetration depth; pa, pb witness points on a and b;
 *    status codes tell failures apart (ok = 0 means the reference's call
 *    returned false). */
typedef struct mfcl_convex_result {
  int32_t hit;
  int32_t n_contacts;
  int8_t method;     /* 0 closed form, 1 GJK/EPA, 2 MPR */
  int8_t gjk_status; /* cvx_collide::GJK_Status, -1 if not run */
  int8_t epa_status; /* cvx_collide::EPA_Status, -1 if not run */
  int8_t ok;
  uint16_t gjk_iters; /* boolean + distance iterations */
  uint16_t epa_iters;
  double distance;
  double depth;
  double normal[3];
  double pos[3];
  double pa[3];
  double pb[3];
} mfcl_convex_result;

/* One contact of a collide query (mfcl_convex_collide_contacts): the
 * reference's Contact fields normal, pos and penetration_depth
 * (include/fcl/narrowphase/contact.h:47-98), world frame, normal from shape
 * a to shape b.  56 bytes. */
typedef struct mfcl_contact {
  double normal[3];
  double pos[3];
  double depth;
} mfcl_contact;
/* Most contacts one convex pair produces (boxBox2's maxc,
 * box_box-inl.h:823-841; every other pair type produces one). */
#define MFCL_MAX_PAIR_CONTACTS 4

/* A contact of a penetration-enabled mesh-mesh query
 * (mfcl_mesh_collide_contacts): the triangle ids b1, b2 and the Contact
 * fields pos, normal and penetration_depth as the reference computes them
 * (shape_pair_intersect-inl.h:226-254, intersect-inl.h:796-842).  64 bytes. */
typedef struct mfcl_mesh_contact {
  int32_t b1, b2;
  double pos[3];
  double normal[3];
  double depth;
} mfcl_mesh_contact;

/* Mesh query result header, one per pair; contacts go to a separate
 * (n_pairs x max_contacts) array of (b1, b2) triangle index pairs. */
typedef struct mfcl_mesh_result {
  int32_t hit;
  int32_t n_contacts;
  int32_t bv_tests;   /* OBB overlap tests performed */
  int32_t leaf_tests; /* triangle-triangle tests performed */
} mfcl_mesh_result;

/* ---- context ------------------------------------------------------------ */
int mfcl_create(mfcl_ctx** out, int device);
int mfcl_destroy(mfcl_ctx* ctx);
const char* mfcl_last_error(const mfcl_ctx* ctx);
int mfcl_sync(mfcl_ctx* ctx);
/* Records HIP events around each kernel on its stream when enabled; the
 * durations of the last query are read back with mfcl_last_timing(). */
int mfcl_set_timing(mfcl_ctx* ctx, int enabled);
/* ms[0] order/bucketing kernels, ms[1] GJK/closed-form stage, ms[2] EPA
 * stage, ms[3] mesh traversal, ms[4] broadphase, ms[5] MLP.  Where a
 * wavefront takes a whole pair (small batches, boolean queries) ms[1] holds
 * its EPA too and ms[2] only the pairs that continue at full capacity. */
int mfcl_last_timing(mfcl_ctx* ctx, float* ms6);
/* Work counters of the last convex query: [0] pairs, [1] hull vertices
 * evaluated by support mapping, [2] EPA pairs, [3] EPA pairs restarted at full
 * polytope capacity after exhausting the first LDS polytope.  A support search
 * evaluates every vertex of a hull that it scans (counted once, also where a
 * rounding tie has it read them again in FP64) and, of a hull that it walks,
 * the start and all neighbours of each vertex it stood on (all are read, also
 * the two it has just left).  The counts do not depend on the launch shape. */
int mfcl_last_counters(mfcl_ctx* ctx, uint64_t* c4);
/* The same counters and more, the first n of: [0..3] as above, [4] hull
 * vertices evaluated by the EPA stage alone, [5] EPA pairs that outgrew the
 * first LDS polytope and continued, from a dump, in one of full
 * capacity (entries beyond 5 read 0). */
int mfcl_last_counters_n(mfcl_ctx* ctx, uint64_t* c, int32_t n);

/* Launch-shape knobs (no counterpart in the reference: GPU scheduling
 * parameters, chosen by the autotuner in mind-fcl_amd/mfcl/autotune.py). */
#define MFCL_TUNE_GJK_GROUP 1         /* lanes per pair in the GJK stage: 0 (default) by batch size; 1
                                         (penetration and signed-distance modes; cooperative hull scans);
                                         16, 32, 64: one wavefront per pair */
#define MFCL_TUNE_EPA_THREADS 2       /* persistent EPA lanes (64 per pair), multiple of 256 */
#define MFCL_TUNE_MESH_BLOCKS_PER_CU 3 /* persistent traversal blocks (4 wavefronts) per CU, 1..16 */
#define MFCL_TUNE_MESH_STACK 4        /* node-pair stack entries per block, 1024..262144 */
#define MFCL_TUNE_EPA_LDS_FACES 5     /* face capacity of the first LDS polytope, 16..128 (64 from there on) */
#define MFCL_TUNE_GUESS_POLICY 6      /* mfcl_mlp_guess_dev: 0 the MLP direction for every pair; 1 (default)
                                         the default guess where the MLP predicts penetration */
#define MFCL_TUNE_EPA_SPILL 7         /* 1 (default): a pair that outgrows the first LDS polytope is dumped and
                                         continues at full capacity; 0: it restarts there */
#define MFCL_TUNE_MLP_WAVES 8         /* wavefronts per block of the fused warm-start inference (4, 8 or 16; 0,
                                         the default, by batch size), sharing one LDS copy of the weights;
                                         one block per CU */
#define MFCL_TUNE_LANE_REFILL 9       /* GJK lane kernel (signed distance and penetration): 0 one pair per
                                         lane over a grid of all pairs; k in 1..63 (default 48) a persistent
                                         grid whose finished lanes take new pairs once at most k lanes of
                                         their wavefront still run */
int mfcl_tune(mfcl_ctx* ctx, int32_t knob, int32_t value);

/* Workspace sizing (no counterpart in the reference, whose calls allocate
 * per call).  Grows the context's workspace of the given kind so that later
 * "_dev" queries of up to `count` items run without allocating; never
 * shrinks it.  Synchronises the device when it grows.
 *   MFCL_WS_CONVEX: pairs per mfcl_convex_query_dev /
 *                   mfcl_convex_collide_contacts_dev call;
 *   MFCL_WS_MLP:    rows per mfcl_mlp_train_step_dev call
 *                   (mfcl_mlp_forward_dev and mfcl_mlp_guess_dev need none).
 * The mesh traversal's stacks are sized at mfcl_upload_meshes and by
 * mfcl_tune's mesh knobs; the broadphase query needs no workspace. */
#define MFCL_WS_CONVEX 1
#define MFCL_WS_MLP 2
int mfcl_reserve(mfcl_ctx* ctx, int32_t kind, uint64_t count);
/* Pairs the convex workspace holds now (0 before any reservation). */
int mfcl_reserved_pairs(mfcl_ctx* ctx, uint64_t* pairs);

/* ---- captured query sequences ------------------------------------------- */
/* No counterpart in the reference.  Between mfcl_graph_begin and
 * mfcl_graph_end, the "_dev" query calls made on this context with a NULL
 * stream (mfcl_convex_query_dev, mfcl_convex_collide_contacts_dev,
 * mfcl_mesh_collide_dev, mfcl_mesh_collide_contacts_dev,
 * mfcl_aabbtree_query_dev, mfcl_mlp_guess_dev) are recorded into a HIP
 * graph instead of running; mfcl_graph_launch replays the whole sequence
 * with one launch.  The recorded calls keep their arguments (device
 * pointers, sizes, requests, knobs): replays read the buffers' current
 * contents.  While recording, per-kernel timing is off and calls that
 * synchronise, allocate or copy host memory (uploads, mfcl_reserve*, the
 * host-pointer queries, mfcl_arm_query_dev, training) fail with
 * MFCL_E_STATE.  Sizes stay within the workspace reserved before
 * mfcl_graph_begin. */
typedef struct mfcl_graph mfcl_graph;
int mfcl_graph_begin(mfcl_ctx* ctx);
int mfcl_graph_end(mfcl_ctx* ctx, mfcl_graph** out);
/* Enqueues the recorded sequence on stream (hipStream_t, NULL: the
 * context's stream). */
int mfcl_graph_launch(mfcl_graph* g, void* stream);
int mfcl_graph_destroy(mfcl_graph* g);

/* ---- device memory helpers (so callers need no HIP runtime) ------------- */
int mfcl_dev_alloc(mfcl_ctx* ctx, uint64_t bytes, void** dptr);
int mfcl_dev_free(mfcl_ctx* ctx, void* dptr);
int mfcl_h2d(mfcl_ctx* ctx, void* dst, const void* src, uint64_t bytes);
int mfcl_d2h(mfcl_ctx* ctx, void* dst, const void* src, uint64_t bytes);

/* ---- convex / primitive narrowphase ------------------------------------ */
/* Uploads the shape table (replaces constructing fcl::Box/Sphere/Capsule/
 * Cylinder/Convex objects, include/fcl/geometry/shape/ headers; the convex
 * vertex set is fcl::Convex::getVertices()).  params: 4 floats per shape
 * (unused entries ignored).  verts: xyz triples, shape i owns
 * verts[vert_off[i] .. vert_off[i] + vert_cnt[i]).  Replaces any previous
 * shape table. */
int mfcl_upload_shapes(mfcl_ctx* ctx, const int32_t* type, const float* params4,
                       const uint64_t* vert_off, const uint32_t* vert_cnt, uint32_t n_shapes,
                       const float* verts_xyz, uint64_t n_verts);

/* Attaches faces to the convex shapes of the current shape table (the faces
 * argument of fcl::Convex's constructor, include/fcl/geometry/shape/
 * convex-inl.h:50-73).  Shape i owns num_faces[i] faces starting at
 * faces[face_off[i]], each in the reference's encoding: the vertex count,
 * then that many indices into the shape's vertices.  As in the reference, a
 * hull of more than 32 vertices whose faces are watertight and cover every
 * vertex (convex-inl.h:293-375) then finds support points by the vertex-
 * adjacency walk (convex-inl.h:202-290); other hulls, and all hulls before
 * this call or with num_faces[i] == 0, by the naive scan (convex-inl.h:
 * 133-149).  Shapes with equal (face_off, num_faces, vertex count) share one
 * adjacency table, as Convex objects built from one shared face vector do.
 * faces_len: int32 entries in faces.  Errors: a face with fewer than 3
 * vertices or an index outside its hull (MFCL_E_INVALID). */
int mfcl_upload_convex_faces(mfcl_ctx* ctx, const int32_t* faces, uint64_t faces_len,
                             const uint64_t* face_off, const uint32_t* num_faces);

/* Batched fcl::collide / GJKSolver::shapeSignedDistance over shape pairs
 * (include/fcl/narrowphase/collision_interface-inl.h:13-32,
 * gjk_solver-inl.h:820-874).  pair_a/pair_b: shape ids; pose_a/pose_b: 7
 * floats per pair; guess3: optional per-pair GJK guess (3 floats, used when
 * req->use_guess).  Host pointers. */
int mfcl_convex_query(mfcl_ctx* ctx, const uint32_t* pair_a, const uint32_t* pair_b,
                      const float* pose_a7, const float* pose_b7, const float* guess3, uint64_t n,
                      const mfcl_request* req, mfcl_convex_result* out);
/* Same over device pointers, enqueued on stream (hipStream_t or NULL).
 * Needs mfcl_reserve(ctx, MFCL_WS_CONVEX, >= n). */
int mfcl_convex_query_dev(mfcl_ctx* ctx, const uint32_t* pair_a, const uint32_t* pair_b,
                          const float* pose_a7, const float* pose_b7, const float* guess3,
                          uint64_t n, const mfcl_request* req, mfcl_convex_result* out,
                          void* stream);
/* No counterpart in the reference: mfcl_convex_query_dev for callers that
 * cannot allocate device memory (code under HIP graph capture, tight
 * serving loops, harnesses that forbid hipMalloc).  Same arguments and
 * results; needs no mfcl_reserve: the workspace is a static 64 MiB device
 * array per GPU, so one call takes at most
 * mfcl_convex_query_static_dev_max_pairs() pairs (larger calls fail with
 * MFCL_E_INVALID).  Every call on a GPU shares that GPU's array: calls that
 * overlap on one GPU (concurrent streams, threads or contexts) race; order
 * them on one stream. */
int mfcl_convex_query_static_dev(mfcl_ctx* ctx, const uint32_t* pair_a, const uint32_t* pair_b,
                                 const float* pose_a7, const float* pose_b7, const float* guess3,
                                 uint64_t n, const mfcl_request* req, mfcl_convex_result* out,
                                 void* stream);
int mfcl_convex_query_static_dev_max_pairs(uint64_t* max_pairs);
/* fcl::collide with every contact the CollisionResult would receive
 * (collide mode with penetration only): up to min(max_contacts, 4) per pair
 * -- boxBox2 yields up to 4 (box_box-inl.h:823-841), the other pair types
 * one -- truncated to the deepest by the reference's partial sort when they
 * do not all fit (shape_pair_intersect-inl.h:91-113), in CollisionResult
 * order.  contacts: n * min(max_contacts, 4) records, pair i's k-th contact
 * at contacts[i * min(max_contacts, 4) + k] for k < out[i].n_contacts
 * (other records untouched); out[i] holds contact 0 as in
 * mfcl_convex_query.  Host pointers. */
int mfcl_convex_collide_contacts(mfcl_ctx* ctx, const uint32_t* pair_a, const uint32_t* pair_b,
                                 const float* pose_a7, const float* pose_b7, const float* guess3, uint64_t n,
                                 const mfcl_request* req, mfcl_convex_result* out, mfcl_contact* contacts);
int mfcl_convex_collide_contacts_dev(mfcl_ctx* ctx, const uint32_t* pair_a, const uint32_t* pair_b,
                                     const float* pose_a7, const float* pose_b7, const float* guess3,
                                     uint64_t n, const mfcl_request* req, mfcl_convex_result* out,
                                     mfcl_contact* contacts, void* stream);

/* fcl::collisionPenetration with CollisionPenetrationMode DirectedPenetration
 * (include/fcl/narrowphase/collision_penetration-inl.h:196-244) over shape
 * pairs: the boolean collide of req (penetration disabled), then for each
 * colliding pair the MPR penetration search along dir3[i] -- a world unit
 * vector, the direction shape b escapes along -- (MPR::
 * RunDirectedPenetration, include/fcl/cvx_collide/mpr.hpp:496-704; MPR(128,
 * req->epa_tolerance) as there).  The pair's contact: depth = the distance
 * along dir3 that separates the shapes (-1 when the search fails), pos =
 * the witness midpoint (0 on failure), normal = dir3 (computePenetrationMPR,
 * :105-194); distance = -depth; epa_status = MPR::DirectedPenetrationStatus
 * (0 OK, 1 Failed, 2 FailedNoIntersect, 3 FailedRefinementIterationLimit),
 * epa_iters = its refinement iterations.  req->mode must be
 * MFCL_MODE_COLLIDE.  Host pointers; the _dev form takes device pointers and
 * needs mfcl_reserve(ctx, MFCL_WS_CONVEX, >= n). */
int mfcl_convex_directed_penetration(mfcl_ctx* ctx, const uint32_t* pair_a, const uint32_t* pair_b,
                                     const float* pose_a7, const float* pose_b7, const float* dir3, uint64_t n,
                                     const mfcl_request* req, mfcl_convex_result* out);
int mfcl_convex_directed_penetration_dev(mfcl_ctx* ctx, const uint32_t* pair_a, const uint32_t* pair_b,
                                         const float* pose_a7, const float* pose_b7, const float* dir3,
                                         uint64_t n, const mfcl_request* req, mfcl_convex_result* out,
                                         void* stream);
/* The same with CollisionPenetrationMode IncrementalMinimumPenetration:
 * from the hint hint3[i] (world unit vector) the MPR search refines the
 * direction of minimum penetration (MPR::
 * RunIncrementalMinimumPenetrationDistance, include/fcl/cvx_collide/
 * mpr_incremental_penetration.hpp:10-337).  depth = the minimum
 * penetration found, normal = its direction in the world (shape b's escape
 * direction), pos = the witness midpoint; an iteration-limit result counts
 * as found; failures as above.  epa_status = MPR::
 * IncrementalPenetrationStatus (0 OK, 1 Failed, 2 FailedNoIntersect, 4
 * IterationLimit), epa_iters = its outer iterations. */
int mfcl_convex_incremental_penetration(mfcl_ctx* ctx, const uint32_t* pair_a, const uint32_t* pair_b,
                                        const float* pose_a7, const float* pose_b7, const float* hint3, uint64_t n,
                                        const mfcl_request* req, mfcl_convex_result* out);
int mfcl_convex_incremental_penetration_dev(mfcl_ctx* ctx, const uint32_t* pair_a, const uint32_t* pair_b,
                                            const float* pose_a7, const float* pose_b7, const float* hint3,
                                            uint64_t n, const mfcl_request* req, mfcl_convex_result* out,
                                            void* stream);

/* ---- convex hulls on the device ----------------------------------------- */
/* The convex hull of each point set (what a caller of fcl::Convex computes
 * before constructing it from the hull's vertices and faces,
 * include/fcl/geometry/shape/convex-inl.h:50-73).  Set i is
 * points[pt_off[i] .. pt_off[i] + pt_cnt[i]) (xyz triples, 4 to
 * max_points <= 768 points).  Per set: status[i] (0 ok, 1 degenerate: fewer
 * than 4 points or all (nearly) coplanar, 2 more than max_points points,
 * 3 inconsistent orientation tests), hull_cnt[i] hull vertices whose indices
 * within the set are hull_idx[pt_off[i] + k] in ascending order, and
 * tri_cnt[i] triangles (outward orientation) over those k-numbered
 * vertices at tris[6 pt_off[i] + 3 t + j].  Points within a relative 1e-12
 * of a face's plane are left out of the hull.  Device pointers. */
int mfcl_convex_hulls_dev(mfcl_ctx* ctx, const float* points_xyz, const uint64_t* pt_off, const uint32_t* pt_cnt,
                          uint32_t n_sets, int32_t max_points, uint32_t* hull_cnt, uint32_t* hull_idx,
                          uint32_t* tri_cnt, int32_t* tris, int32_t* status, void* stream);
/* The same with host pointers (copies in, runs, copies out, synchronises). */
int mfcl_convex_hulls(mfcl_ctx* ctx, const float* points_xyz, const uint64_t* pt_off, const uint32_t* pt_cnt,
                      uint32_t n_sets, uint32_t* hull_cnt, uint32_t* hull_idx, uint32_t* tri_cnt, int32_t* tris,
                      int32_t* status);
/* Builds the shape table from point sets without a host pass over the
 * hulls: shape i is the convex hull of set i (as mfcl_convex_hulls, 4..768
 * points), with the hull's vertices in ascending point order and its
 * triangles as faces.  The result equals mfcl_upload_shapes (every shape
 * MFCL_SHAPE_CONVEX, zero params) with those vertices followed by
 * mfcl_upload_convex_faces with those triangles -- what the reference's
 * callers do when they construct fcl::Convex from a hull
 * (convex-inl.h:50-73, adjacency convex-inl.h:293-409) -- and replaces any
 * previous shape table.  hull_cnt: optional host output, hull vertices per
 * shape.  A set without a hull fails the call (MFCL_E_INVALID; the message
 * names the set).  Host pointers. */
int mfcl_upload_convex_points(mfcl_ctx* ctx, const float* points_xyz, const uint64_t* pt_off,
                              const uint32_t* pt_cnt, uint32_t n_sets, uint32_t* hull_cnt);

/* ---- OBBRSS mesh-mesh --------------------------------------------------- */
/* Builds one OBB tree per mesh on the host and uploads node and triangle
 * arrays (replaces BVHModel<OBBRSS>::beginModel/addSubModel/endModel,
 * include/fcl/geometry/bvh/BVH_model-inl.h:136-305).  tris: 3 vertex ids per
 * triangle, local to the mesh.  Replaces any previous mesh set. */
int mfcl_upload_meshes(mfcl_ctx* ctx, const float* verts_xyz, const uint64_t* vert_off,
                       const uint32_t* vert_cnt, const uint32_t* tris, const uint64_t* tri_off,
                       const uint32_t* tri_cnt, uint32_t n_meshes);
/* Number of BVH nodes of mesh i (host query). */
int mfcl_mesh_num_nodes(mfcl_ctx* ctx, uint32_t mesh, uint32_t* n_nodes);
/* Batched fcl::collide(BVHModel<OBBRSS>, shape) with penetration disabled
 * (OrientedNodeBVHSolver::MeshShapeIntersect, include/fcl/narrowphase/
 * detail/traversal/collision/bvh_solver-inl.h:6-72): query i tests mesh
 * mesh_ids[i] posed pose_mesh7 against shape shape_ids[i] of the shape
 * table posed pose_shape7; leaf tests as GJKSolver::shapeTriangleIntersect
 * (gjk_solver-inl.h:545-563: sphere and box closed forms, else MPR with
 * req's GJK iteration cap and tolerance).  out: hit (-1: the traversal's
 * stack overflowed), n_contacts = min(colliding triangles, max_contacts),
 * bv_tests, leaf_tests; tri_ids (optional): n x max_contacts triangle ids
 * (the reference's Contact::b1; b2 is Contact::NONE), ascending, -1 past
 * n_contacts.  When more than max_contacts triangles collide, which ones are
 * kept is not the reference's depth-first choice.  req->penetration must be
 * 0 (mfcl_mesh_shape_collide_contacts takes the penetration-enabled form).
 * Host pointers; synchronises. */
int mfcl_mesh_shape_collide(mfcl_ctx* ctx, const uint32_t* mesh_ids, const uint32_t* shape_ids,
                            const float* pose_mesh7, const float* pose_shape7, uint64_t n,
                            const mfcl_request* req, mfcl_mesh_result* out, int32_t* tri_ids);
/* The same with penetration enabled (req->penetration = 1; the same
 * traversal, bvh_solver-inl.h:6-72, with the leaf test's contact outputs,
 * shape_pair_intersect-inl.h:133-172): each colliding triangle adds one
 * contact from GJKSolver::shapeTriangleIntersect (gjk_solver-inl.h:545-563):
 * sphereTriangleIntersect's contact for spheres (sphere_triangle-inl.h:
 * 107-187: pos = the nearest point found, depth = -(r - distance)), else GJK
 * from -UnitX and EPA on (shape, triangle) with req's GJK and EPA caps and
 * tolerances (gjk_solver-inl.h:452-527: a hit unless EPA fails; pos = the
 * witness midpoint in the world, normal from the witnesses, depth = the
 * EPA depth) -- boxes included, whose closed form is boolean only.  Each
 * contact has b1 = the triangle, b2 = -1 and the normal reversed as the
 * traversal writes it (ContactMeta::reverse_normal, bvh_solver-inl.h:
 * 55-65).  contacts: n x max_contacts records, ascending b1, b1 = -1 past
 * n_contacts; which contacts of a larger set are kept follows the traversal
 * here.  Host pointers; synchronises. */
int mfcl_mesh_shape_collide_contacts(mfcl_ctx* ctx, const uint32_t* mesh_ids, const uint32_t* shape_ids,
                                     const float* pose_mesh7, const float* pose_shape7, uint64_t n,
                                     const mfcl_request* req, mfcl_mesh_result* out,
                                     mfcl_mesh_contact* contacts);
/* Copies mesh i's tree to host memory: mfcl_mesh_num_nodes() nodes of 64
 * bytes, breadth-first (float axes[9], column-major; float centre[3]; float
 * half extents[3]; int32 child: >= 0 first child, its sibling next; < 0 leaf
 * of triangle -(child + 1)). */
int mfcl_mesh_get_nodes(mfcl_ctx* ctx, uint32_t mesh, void* nodes);
/* Deforming meshes: BVHModel::beginReplaceModel / replaceSubModel /
 * endReplaceModel(refit) (include/fcl/geometry/bvh/BVH_model-inl.h:
 * 306-375) with every vertex of mesh i replaced (vert_cnt[i] xyz triples,
 * the triangles kept).  refit != 0: the tree is refitted on the device
 * (refitTree, BVH_model-inl.h:572-640) -- every node keeps its axes and
 * triangles and gets the centre and extents that contain them; refit == 0:
 * the tree is rebuilt (on the host, as mfcl_upload_meshes builds it).  Host
 * pointer; synchronises. */
int mfcl_mesh_replace_vertices(mfcl_ctx* ctx, uint32_t mesh, const float* verts_xyz, int32_t refit);
/* The refit with a device pointer, enqueued on stream (hipStream_t or
 * NULL): a vertex copy and three kernels, no allocation, capturable. */
int mfcl_mesh_replace_vertices_dev(mfcl_ctx* ctx, uint32_t mesh, const float* verts_xyz, void* stream);
/* Mesh files.  mfcl_load_obj reads a Wavefront OBJ file as the reference's
 * tests do (test/test_fcl_utility.h:250-316, loadOBJFile): "v" lines give
 * vertices, "f" lines 1-based vertex ids (each token's integer prefix); a
 * face of k ids gives k - 2 triangles, the fan (0, t+1, t+2) once a "vn" or
 * "vt" line was read and otherwise k - 2 copies of (0, 1, 2), as there.
 * Call it with verts_xyz = tris = NULL to get *n_verts / *n_tris, then with
 * buffers of those sizes.  No context needed. */
int mfcl_load_obj(const char* path, float* verts_xyz, uint64_t* n_verts, uint32_t* tris, uint64_t* n_tris);
/* No counterpart in the reference (which builds every tree from vertex and
 * triangle data): the uploaded mesh set -- current vertices, triangles and
 * built trees -- written to a flat binary file, and read back into a
 * context without a tree build.  mfcl_load_meshes replaces the mesh set and
 * rejects files that are truncated, corrupted (checksum) or malformed
 * (MFCL_E_INVALID). */
int mfcl_save_meshes(mfcl_ctx* ctx, const char* path);
int mfcl_load_meshes(mfcl_ctx* ctx, const char* path);
/* The same file built on the host alone (trees built as mfcl_upload_meshes
 * builds them), e.g. offline, and its header read back after a full check
 * (counts; MFCL_E_INVALID for a damaged file).  No context or GPU needed;
 * mfcl_host_last_error() describes the last failure of these and of
 * mfcl_load_obj on the calling thread. */
int mfcl_build_mesh_file(const char* path, const float* verts_xyz, const uint64_t* vert_off,
                         const uint32_t* vert_cnt, const uint32_t* tris, const uint64_t* tri_off,
                         const uint32_t* tri_cnt, uint32_t n_meshes);
int mfcl_mesh_file_info(const char* path, uint32_t* n_meshes, uint64_t* n_tris, uint64_t* n_nodes);
const char* mfcl_host_last_error(void);
/* Batched fcl::collide(BVHModel<OBBRSS>, BVHModel<OBBRSS>) with
 * CollisionRequest(max_contacts), penetration disabled
 * (narrowphase/detail/traversal/collision/bvh_solver-inl.h:75-164).
 * contacts: n * max_contacts * 2 int32 (b1, b2).  Host pointers. */
int mfcl_mesh_collide(mfcl_ctx* ctx, const uint32_t* pair_a, const uint32_t* pair_b,
                      const float* pose_a7, const float* pose_b7, uint64_t n, int32_t max_contacts,
                      mfcl_mesh_result* out, int32_t* contacts);
int mfcl_mesh_collide_dev(mfcl_ctx* ctx, const uint32_t* pair_a, const uint32_t* pair_b,
                          const float* pose_a7, const float* pose_b7, uint64_t n,
                          int32_t max_contacts, mfcl_mesh_result* out, int32_t* contacts,
                          void* stream);
/* The same with penetration enabled (CollisionRequest(max_contacts,
 * enable_contact = true)): each colliding triangle pair adds as many
 * contacts as intersect_Triangle's deepest points, 0 to 2
 * (intersect-inl.h:796-842), truncated to the free slots
 * (shape_pair_intersect-inl.h:226-254); the reference maps their position
 * and normal to the world with the second mesh's transform (SimplexIntersect
 * passes tf2 for both, shape_pair_intersect-inl.h:269), and so does this
 * call.  out[i].hit = 1 when pair i has a contact.  contacts: n *
 * max_contacts records; which contacts of a larger set are kept depends on
 * the traversal order.  Host pointers. */
int mfcl_mesh_collide_contacts(mfcl_ctx* ctx, const uint32_t* pair_a, const uint32_t* pair_b,
                               const float* pose_a7, const float* pose_b7, uint64_t n, int32_t max_contacts,
                               mfcl_mesh_result* out, mfcl_mesh_contact* contacts);
int mfcl_mesh_collide_contacts_dev(mfcl_ctx* ctx, const uint32_t* pair_a, const uint32_t* pair_b,
                                   const float* pose_a7, const float* pose_b7, uint64_t n, int32_t max_contacts,
                                   mfcl_mesh_result* out, mfcl_mesh_contact* contacts, void* stream);

/* ---- broadphase AABB tree ----------------------------------------------- */
/* Builds a flattened breadth-first AABB tree over n boxes (replaces
 * BinaryAABB_Tree::Rebuild, include/fcl/broadphase/binary_AABB_tree-inl.h:19-25). */
int mfcl_aabbtree_build(mfcl_ctx* ctx, const float* mn3, const float* mx3, const int64_t* ids,
                        uint32_t n);
/* For each query box, the ids of the overlapping leaves (up to cap, in no
 * particular order) and their count (replaces
 * BinaryAABB_Tree::SingleObjectCollision, binary_AABB_tree-inl.h:400-440).
 * counts may exceed cap (then only cap ids are written).  Host pointers. */
int mfcl_aabbtree_query(mfcl_ctx* ctx, const float* qmn3, const float* qmx3, uint64_t nq,
                        int32_t cap, int32_t* counts, int64_t* ids);
int mfcl_aabbtree_query_dev(mfcl_ctx* ctx, const float* qmn3, const float* qmx3, uint64_t nq,
                            int32_t cap, int32_t* counts, int64_t* ids, void* stream);

/* ---- robot-arm configurations ------------------------------------------- */
/* No counterpart in the reference (it has no arm model): forward kinematics
 * of a serial chain, then per link BinaryAABB_Tree::SingleObjectCollision
 * against the tree built by mfcl_aabbtree_build (binary_AABB_tree-inl.h:
 * 400-440) and per candidate pair GJKSolver::shapeSignedDistance
 * (gjk_solver-inl.h:820-874), reduced per configuration.  Joint i turns
 * about z (even i) or y (odd i); link i runs along its local x over
 * link_len[i], its shape centred at link_len[i] / 2; the base is the world
 * origin.  Obstacle k is shape box_shape0 + k with world pose box_pose7[k]
 * and leaf id k in the AABB tree. */
#define MFCL_ARM_MAX_LINKS 16
typedef struct mfcl_arm {
  int32_t n_links;
  uint32_t link_shape[MFCL_ARM_MAX_LINKS];  /* shape id of each link */
  float link_len[MFCL_ARM_MAX_LINKS];
  float link_radius[MFCL_ARM_MAX_LINKS];    /* bound on |x| over the link shape (broadphase sphere) */
  uint32_t box_shape0, n_boxes;
  int32_t broadphase_cap;                   /* candidates kept per link, 1..512 */
  int32_t gjk_max_iterations;               /* 0: the default */
  uint64_t max_pairs;                       /* candidate pair capacity, 0: 8 per link */
  /* heightmap (mfcl_upload_heightmap), 0: none.  Pixel (x, y) of the bottom
   * layer is shape hm_box_shape0 + y * full_x + x, a box of sides
   * (res_x, res_y, height); the map's frame has world pose hm_pose7. */
  int32_t use_heightmap;
  uint32_t hm_box_shape0;
  int32_t hm_cap;                           /* candidate pixels kept per link, 1..65536 */
  float hm_pose7[7];
} mfcl_arm;
/* q: n_configs x n_links joint angles (device).  Per configuration:
 * any_hit bit 0 = some candidate pair has signed distance < 0 or some link
 * collides with the heightmap, bit 1 = some candidate was dropped
 * (broadphase cap, pair capacity) or its query failed;
 * min_dist = the minimum signed distance over the candidates (+inf when no
 * obstacle is within `margin` of a link's bounding sphere).  n_pairs: the
 * candidate pairs queried (host, may be NULL).  Synchronises the stream once
 * (the pair count sizes the narrowphase launch).  Needs
 * mfcl_reserve_arm(ctx, arm, >= n_configs). */
int mfcl_arm_query_dev(mfcl_ctx* ctx, const mfcl_arm* arm, const float* q, uint64_t n_configs, float margin,
                       const float* box_pose7, int32_t* any_hit, float* min_dist, uint64_t* n_pairs,
                       void* stream);

/* Sizes the arm query's workspace (link poses, broadphase hits, candidate
 * pairs and their convex-query workspace) for up to n_configs
 * configurations of this arm description. */
int mfcl_reserve_arm(mfcl_ctx* ctx, const mfcl_arm* arm, uint64_t n_configs);

/* Replaces heightmap::LayeredHeightMap (layered_heightmap.h:33-36, built
 * from the bottom layer as layered_heightmap-inl.h:8-51 and :76-101: each
 * upper pixel holds the maximum of its 2 x 2 children).  heights_mm: the
 * bottom layer, (2 half_x) x (2 half_y) uint16 millimetres, pixel (x, y) at
 * y * 2 half_x + x (flat_heightmap-inl.h pixelToFlatIndex); half_x and
 * half_y powers of two.  A link of mfcl_arm_query_dev collides with the map
 * when it collides with the box of some pixel of non-zero height
 * (HeightMapCollisionSolver::HeightMapShapeIntersect, heightmap_solver_
 * traverse-inl.h:17-120: candidate pixels are those whose box overlaps the
 * link's AABB in the map frame, then ShapeIntersect(Box, Convex) per pixel,
 * heightmap_solver_leaf-inl.h:6-28).  The reference has no distance to a
 * heightmap, so min_dist covers the obstacle boxes only. */
int mfcl_upload_heightmap(mfcl_ctx* ctx, const uint16_t* heights_mm, uint16_t half_x, uint16_t half_y, float res_x,
                          float res_y);
/* No counterpart in the reference: the heightmap candidate pairs (link, pixel
 * box) that the last mfcl_arm_query_dev sent to the narrowphase. */
int mfcl_arm_last_heightmap_pairs(mfcl_ctx* ctx, uint64_t* n_pairs);

/* ---- learned GJK warm start --------------------------------------------- */
/* No counterpart in the reference: a 39-128-128-128-4 GELU MLP whose output
 * direction is passed as the per-pair GJK guess (the reference's hook
 * GJKSolver::gjk_guess / enable_cached_guess, include/fcl/narrowphase/
 * detail/gjk_solver.h:140-163, consumed at gjk_solver-inl.h:77-78,103).
 * Inputs per pair: relative pose of b in a's frame (translation 3,
 * quaternion 4) and a 16-float descriptor of each shape (computed at
 * mfcl_upload_shapes); feature rows are 64 floats (39 used).  Outputs per
 * pair: 4 floats = unnormalised direction in a's frame (3) + signed
 * distance estimate (1).  BF16 MFMA products with FP32 accumulation; FP32
 * master parameters trained with Adam. */
int mfcl_mlp_num_params(void);
/* Xavier-uniform initialisation (std::mt19937_64 seeded) and Adam reset. */
int mfcl_mlp_init(mfcl_ctx* ctx, uint64_t seed);
/* Host FP32 parameter vector of mfcl_mlp_num_params() floats (layout:
 * W1[128][64], b1[128], W2[128][128], b2, W3[128][128], b3, W4[32][128],
 * b4[32]; padding entries zero).  set_params also resets Adam. */
int mfcl_mlp_set_params(mfcl_ctx* ctx, const float* params, int32_t n);
/* Copies parameters and/or the gradients of the last training step to host
 * (either pointer may be NULL). */
int mfcl_mlp_get_params(mfcl_ctx* ctx, float* params, float* grads, int32_t n);
/* Feature rows (n x 64 FP32, device) for pairs of uploaded shapes. */
int mfcl_mlp_features_dev(mfcl_ctx* ctx, const uint32_t* pair_a, const uint32_t* pair_b,
                          const float* pose_a7, const float* pose_b7, uint64_t n, float* feat64,
                          void* stream);
/* Features + forward pass + normalisation: unit guess directions (n x 3,
 * a's frame) ready for mfcl_convex_query_dev(..., guess3, ...) with
 * req->use_guess = 1, and optional distance estimates (n, may be NULL). */
int mfcl_mlp_guess_dev(mfcl_ctx* ctx, const uint32_t* pair_a, const uint32_t* pair_b,
                       const float* pose_a7, const float* pose_b7, uint64_t n, float* guess3,
                       float* dist_estimate, void* stream);
/* Forward pass on given feature rows (device): out4 is n x 4. */
int mfcl_mlp_forward_dev(mfcl_ctx* ctx, const float* feat64, uint64_t n, float* out4, void* stream);
/* One training step on a batch (device feature rows, targets n x 4 =
 * unit direction + signed distance; rows with a zero direction are
 * ignored).  hyper6 = {lr, beta1, beta2, eps, unused, distance weight} or
 * NULL for {1e-3, 0.9, 0.999, 1e-8, 0, 1}.  apply_update = 0 computes the
 * loss and gradients only (read them with mfcl_mlp_get_params).
 * loss_host (may be NULL) receives the mean loss after synchronising. */
int mfcl_mlp_train_step_dev(mfcl_ctx* ctx, const float* feat64, const float* target4, uint64_t n,
                            const float* hyper6, int32_t apply_update, float* loss_host, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* MFCL_H_ */
