"""GPU: convex hulls with faces -- the reference's vertex-adjacency support
walk (convex-inl.h:202-290) -- against the oracle, which restates the same
walk.

Hulls of more than 32 vertices with watertight, connected faces walk; the
rest (32 or fewer vertices, faces withheld, or a face removed so the mesh is
not watertight) scan every vertex.  The device walk visits the same
neighbours in the same order with the same FP64 comparisons, so results are
compared field by field for exact equality, in signed-distance and
penetration modes, for one lane and one wavefront per pair.
"""
import numpy as np
import pytest

from common import knobs
from mfcl import autotune
from mfcl import workloads as W
import mfcl


def _setup(oracle, n_pairs, seed):
    h = W.hull_pairs(n_pairs, seed, nmin=8, nmax=512, faces=True)
    n = len(h["types"])
    tri_cnt = h["tri_cnt"].copy()
    rng = np.random.default_rng(seed + 100)
    kind = rng.integers(0, 4, size=n)  # 0, 1: faces; 2: faces minus one triangle; 3: no faces
    tri_cnt[kind == 2] -= 1
    tri_cnt[kind == 3] = 0
    S = oracle.ShapeSet(h["types"], h["params"], h["verts"], h["vert_off"], h["vert_cnt"], h["tris"],
                        h["tri_off"], tri_cnt)
    faces = mfcl.faces_from_triangles(h["tris"], h["tri_off"], tri_cnt)
    return h, S, faces, kind


def _run(ctx, h, req, group):
    with knobs(ctx, {autotune.GJK_GROUP: group}):
        return ctx.convex_query(h["pair_a"], h["pair_b"], h["pose_a"], h["pose_b"], req)


FIELDS_SD = ("ok", "gjk_status", "epa_status", "gjk_iters", "epa_iters", "distance", "pa", "pb")
FIELDS_PEN = ("hit", "ok", "gjk_status", "epa_status", "gjk_iters", "epa_iters", "depth", "normal", "pos")


@pytest.mark.gpu
@pytest.mark.parametrize("group", [0, 1, 32])
def test_walk_signed_distance_bit_exact(oracle, gpu_ctx, group):
    h, S, faces, kind = _setup(oracle, 4096, 7)
    walks = np.array([S.walks(i) for i in range(len(h["types"]))])
    assert walks[(kind <= 1) & (h["vert_cnt"] > 32)].all() and not walks[kind >= 2].any()
    assert not walks[h["vert_cnt"] <= 32].any()
    ta, tb = oracle.pose12(h["pose_a"]), oracle.pose12(h["pose_b"])
    ref, _ = S.signed_distance(h["pair_a"], h["pair_b"], ta, tb, threads=8)
    gpu_ctx.upload_shapes(h["types"], h["params"], h["vert_off"], h["vert_cnt"], h["verts"], faces=faces)
    out = _run(gpu_ctx, h, mfcl.request(mfcl.MODE_SIGNED_DISTANCE), group)
    diff = {f: int((out[f] != ref[f]).reshape(len(out), -1).any(1).sum()) for f in FIELDS_SD}
    print(f"\n[walk sd, group {group}] pairs={len(out)} walking hulls={int(walks.sum())} "
          f"intersecting={int((ref['distance'] < 0).sum())} differing per field {diff}")
    assert all(v == 0 for v in diff.values())


@pytest.mark.gpu
@pytest.mark.parametrize("group", [0, 1, 32])
def test_walk_penetration_bit_exact(oracle, gpu_ctx, group):
    h, S, faces, _ = _setup(oracle, 4096, 8)
    ta, tb = oracle.pose12(h["pose_a"]), oracle.pose12(h["pose_b"])
    ref, _ = S.collide(h["pair_a"], h["pair_b"], ta, tb, 1, True, threads=8)
    gpu_ctx.upload_shapes(h["types"], h["params"], h["vert_off"], h["vert_cnt"], h["verts"], faces=faces)
    out = _run(gpu_ctx, h, mfcl.request(mfcl.MODE_COLLIDE, max_contacts=1, penetration=1), group)
    fields = [f for f in FIELDS_PEN if f in ref.dtype.names]
    diff = {f: int((out[f] != ref[f]).reshape(len(out), -1).any(1).sum()) for f in fields}
    print(f"\n[walk collide, group {group}] pairs={len(out)} hits={int(ref['hit'].sum())} differing per field {diff}")
    assert all(v == 0 for v in diff.values())


@pytest.mark.gpu
@pytest.mark.parametrize("group", [0, 1])
@pytest.mark.parametrize("pen", [0, 1])
def test_table_walk_beyond_16_bit_ids(oracle, gpu_ctx, pen, group):
    """A hull of more than 65,535 vertices has no walk blocks (16-bit ids) and
    walks over the adjacency table, beside hulls that have blocks, are scanned
    or are primitives."""
    rng = np.random.default_rng(9)
    u = rng.normal(size=(66000, 3))
    keep, tri = W.hull_faces((0.4 * u / np.linalg.norm(u, axis=1, keepdims=True)).astype(np.float32))
    big = (0.4 * u / np.linalg.norm(u, axis=1, keepdims=True)).astype(np.float32)[keep]
    assert len(big) > 65535
    h = W.hull_pairs(32, 10, nmin=8, nmax=512, faces=True)
    prim = W.primitive_pairs(8, 11)
    nh, npr = len(h["types"]), len(prim["types"])
    types = np.concatenate([h["types"], [h["types"][0]], prim["types"]]).astype(np.int32)
    params = np.concatenate([h["params"], np.zeros((1, 4)), prim["params"]]).astype(np.float32)
    verts = np.concatenate([h["verts"], big])
    off = np.concatenate([h["vert_off"], [len(h["verts"])], np.zeros(npr)]).astype(np.uint64)
    cnt = np.concatenate([h["vert_cnt"], [len(big)], np.zeros(npr)]).astype(np.uint32)
    tris = np.concatenate([h["tris"].reshape(-1, 3), tri]).astype(np.int32)
    toff = np.concatenate([h["tri_off"], [len(tris) - len(tri)], np.zeros(npr)]).astype(np.int64)
    tcnt = np.concatenate([h["tri_cnt"], [len(tri)], np.zeros(npr)]).astype(np.int64)
    hull_of_shape = np.concatenate([np.arange(nh + 1), np.full(npr, -1)]).astype(np.int32)
    S = oracle.ShapeSet(types, params[:, :3], verts, off[:nh + 1], cnt[:nh + 1], tris, toff[:nh + 1], tcnt[:nh + 1],
                        hull_of_shape=hull_of_shape)
    assert S.walks(nh)
    gpu_ctx.upload_shapes(types, params, off, cnt, verts, faces=mfcl.faces_from_triangles(tris, toff, tcnt))
    n = 384
    a, b = rng.integers(0, len(types), n).astype(np.uint32), rng.integers(0, len(types), n).astype(np.uint32)
    a[::3], b[1::3] = nh, nh
    a[::9] = b[::9] = nh
    qa, qb = W.poses(rng, n, 0.0, 0.6), W.poses(rng, n, 0.0, 0.6)
    q = dict(pair_a=a, pair_b=b, pose_a=qa, pose_b=qb)
    ta, tb = oracle.pose12(qa), oracle.pose12(qb)
    if pen:
        ref, _ = S.collide(a, b, ta, tb, 1, True, threads=8)
        out = _run(gpu_ctx, q, mfcl.request(mfcl.MODE_COLLIDE, max_contacts=1, penetration=1), group)
    else:
        ref, _ = S.signed_distance(a, b, ta, tb, threads=8)
        out = _run(gpu_ctx, q, mfcl.request(mfcl.MODE_SIGNED_DISTANCE), group)
    fields = [f for f in (FIELDS_PEN if pen else FIELDS_SD) if f in ref.dtype.names]
    diff = {f: int((out[f] != ref[f]).reshape(len(out), -1).any(1).sum()) for f in fields}
    print(f"\n[table walk pen={pen} group={group}] vertices {len(big)} differing per field {diff}")
    assert all(v == 0 for v in diff.values())


@pytest.mark.gpu
def test_walk_faces_rejected(gpu_ctx):
    h = W.hull_pairs(64, 3, faces=True)
    gpu_ctx.upload_shapes(h["types"], h["params"], h["vert_off"], h["vert_cnt"], h["verts"])
    faces, off, cnt = mfcl.faces_from_triangles(h["tris"], h["tri_off"], h["tri_cnt"])
    bad = faces.copy()
    bad[off[5] + 1] = int(h["vert_cnt"][5])  # a vertex index one past the hull's last vertex
    with pytest.raises(RuntimeError, match="outside the hull"):
        gpu_ctx.upload_convex_faces(bad, off, cnt)
    bad = faces.copy()
    bad[off[7]] = 2  # a two-vertex face
    with pytest.raises(RuntimeError, match="invalid vertex count"):
        gpu_ctx.upload_convex_faces(bad, off, cnt)
    gpu_ctx.upload_convex_faces(faces, off, cnt)  # the valid faces are accepted afterwards
