"""GPU: the lines at which a query takes another kernel or another memory,
on both sides of each line.

* one wavefront per pair below a batch size, one lane per pair above it:
  every record of the default route, of lanes and of wavefronts is the same;
* the EPA polytope in 64-face masks in LDS, 256-face masks in LDS or longer
  lists in LDS (device memory beyond that for shapes on meshes), by the
  request's capacity; and pairs that outgrow the first continued from a dump or
  restarted: every field equals the oracle's at that capacity;
* the warm-start network's training step at row counts around its tiles and
  blocks, against the 64-bit reference.
"""
import numpy as np
import pytest

import mlp_ref as R
import mfcl
from common import knobs
from mfcl import autotune
from mfcl import workloads as W
from test_gpu_edge import _compare, setup  # noqa: F401  (fixture)
from test_gpu_lane import _mixed, _run
from test_gpu_mesh_shape import _setup as mesh_shape_setup
from test_gpu_mlp import BLOCKS, _problem


def _bytes(a):
    return np.ascontiguousarray(a).view(np.uint8).reshape(len(a), -1)


@pytest.mark.gpu
@pytest.mark.parametrize("mode,n", [("sd", 24576), ("sd", 24577), ("pen", 8192), ("pen", 8193), ("pen", 5)])
def test_lane_and_wave_routes_agree(gpu_ctx, mode, n):
    w = _mixed(31, n)
    gpu_ctx.upload_shapes(w["types"], w["params"], w["vert_off"], w["vert_cnt"], w["verts"])
    req = mfcl.request(mfcl.MODE_SIGNED_DISTANCE) if mode == "sd" else mfcl.request(mfcl.MODE_COLLIDE, max_contacts=4,
                                                                                   penetration=1)
    out = [_bytes(_run(gpu_ctx, w, req, group, False)[0]) for group in (0, 1, 64)]
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])


@pytest.mark.gpu
@pytest.mark.parametrize("group", [1, 64])
@pytest.mark.parametrize("faces,lds_faces,spill", [(64, 64, 1), (65, 64, 1), (256, 16, 1), (256, 16, 0), (257, 16, 1),
                                                   (257, 42, 0), (674, 16, 1), (674, 16, 0)])
def test_epa_capacities(oracle, gpu_ctx, setup, faces, lds_faces, spill, group):  # noqa: F811
    h, S, _, tri = setup
    gpu_ctx.upload_shapes(h["types"], h["params"], h["vert_off"], h["vert_cnt"], h["verts"], faces=tri)
    ta, tb = oracle.pose12(h["pose_a"]), oracle.pose12(h["pose_b"])
    sp = np.array([128, 1e-6, faces, 255, 1e-6, 0], np.float64)
    ref, _ = S.signed_distance(h["pair_a"], h["pair_b"], ta, tb, solver=sp, threads=8)
    with knobs(gpu_ctx, {autotune.GJK_GROUP: group, autotune.EPA_LDS_FACES: lds_faces, autotune.EPA_SPILL: spill}):
        out = gpu_ctx.convex_query(h["pair_a"], h["pair_b"], h["pose_a"], h["pose_b"],
                                   mfcl.request(mfcl.MODE_SIGNED_DISTANCE, epa_max_faces=faces))
        c = gpu_ctx.last_counters()
    assert all(v == 0 for v in _compare(out, ref).values())
    with pytest.raises(RuntimeError, match="675"):
        gpu_ctx.convex_query(h["pair_a"], h["pair_b"], h["pose_a"], h["pose_b"],
                             mfcl.request(mfcl.MODE_SIGNED_DISTANCE, epa_max_faces=675))
    if lds_faces == 16:
        assert (c[5] if spill else c[3]) > 0


@pytest.mark.gpu
def test_mesh_shape_epa_memories(oracle, gpu_ctx):
    """255 iterations make at most 4 + 2 * 255 faces, so every capacity above
    that gives the same contacts: lists in LDS, and in device memory.  (Which
    contacts of more than the cap are kept is left to the traversal: queries
    that reach it are compared by their count.)"""
    S, M, types, mesh_ids, shape_ids, pm, ps = mesh_shape_setup(oracle, gpu_ctx, 95, 96)
    got = []
    for faces in (520, 1500, 8192):
        req = mfcl.request(mfcl.MODE_COLLIDE, max_contacts=64, penetration=1, epa_max_faces=faces)
        got.append(gpu_ctx.mesh_shape_collide_contacts(mesh_ids, shape_ids, pm, ps, req))
    for out, cont in got[1:]:
        assert np.array_equal(out["n_contacts"], got[0][0]["n_contacts"])
        free = out["n_contacts"] < 64
        assert free.sum() > 48 and out["n_contacts"][free].sum() > 100
        assert np.array_equal(_bytes(cont[free]), _bytes(got[0][1][free]))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 31, 32, 33, 127, 129, 4097])
def test_mlp_training_rows(gpu_ctx, n):
    """A path of forward and backward rounds about eight times to bfloat16
    (2^-9 of a value each): 1.6e-2 if all add up, against which few rows do
    not average."""
    p, X, T = _problem(5, n + 1)
    X, T = X[1:].copy(), T[1:].copy()  # the first row's direction is masked
    gpu_ctx.mlp_set_params(p)
    loss = gpu_ctx.mlp_train_step_dev(gpu_ctx.to_device(X), gpu_ctx.to_device(T), n, apply_update=False)
    _, g = gpu_ctx.mlp_get_params(grads=True)
    y, saved = R.forward(p.astype(np.float64), X.astype(np.float64))
    ref_loss, dy = R.loss_grad(y, T.astype(np.float64))
    gr = R.backward(p.astype(np.float64), saved, dy)
    assert abs(loss - ref_loss) <= 1e-2 * (1 + abs(ref_loss))
    for name, lo, hi in BLOCKS:
        a, b = g[lo:hi].astype(np.float64), gr[lo:hi]
        assert np.linalg.norm(a - b) <= 3.2e-2 * np.linalg.norm(b), name


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 31, 33, 65535, 65537, 131073])
def test_guess_block_sizes_by_batch(gpu_ctx, n):
    """The block size follows the batch (on 256 CUs the lines are at 65,536
    and 131,072 pairs); what a tile of 32 pairs computes does not."""
    h = W.hull_pairs(200, 13, nmin=8, nmax=64)
    gpu_ctx.upload_shapes(h["types"], h["params"], h["vert_off"], h["vert_cnt"], h["verts"])
    p, _, _ = _problem(4, 2)
    gpu_ctx.mlp_set_params(p)
    rng = np.random.default_rng(14)
    dev = [gpu_ctx.to_device(a) for a in (rng.integers(0, len(h["types"]), n).astype(np.uint32),
                                          rng.integers(0, len(h["types"]), n).astype(np.uint32),
                                          W.poses(rng, n, 0.0, 1.0), W.poses(rng, n, 0.0, 1.0))]
    out = []
    for waves in (0, 4, 16):
        with knobs(gpu_ctx, {autotune.MLP_WAVES: waves}):
            dg, dd = gpu_ctx.to_device(np.full((n, 3), np.nan, np.float32)), gpu_ctx.alloc(n * 4)
            gpu_ctx.mlp_guess_dev(*dev, n, dg, dd)
            out.append((dg.download(np.zeros((n, 3), np.float32)), dd.download(np.zeros(n, np.float32))))
    assert np.all(np.isfinite(out[0][0]))
    for g, d in out[1:]:
        assert np.array_equal(g, out[0][0]) and np.array_equal(d, out[0][1])


@pytest.mark.gpu
@pytest.mark.parametrize("faces", [True, False])
@pytest.mark.parametrize("pen", [0, 1])
def test_work_counters_do_not_depend_on_the_route(gpu_ctx, pen, faces):
    """Pairs, hull vertices evaluated (GJK's and EPA's), EPA pairs: the same for
    one lane and one wavefront per pair, on hulls that walk and hulls that are
    scanned."""
    h = W.hull_pairs(3000, 33, nmin=8, nmax=512, faces=True)
    tri = mfcl.faces_from_triangles(h["tris"], h["tri_off"], h["tri_cnt"]) if faces else None
    gpu_ctx.upload_shapes(h["types"], h["params"], h["vert_off"], h["vert_cnt"], h["verts"], faces=tri)
    w = dict(h, guess=np.zeros((len(h["pair_a"]), 3), np.float32))
    req = mfcl.request(mfcl.MODE_COLLIDE, max_contacts=1, penetration=1) if pen else mfcl.request(
        mfcl.MODE_SIGNED_DISTANCE)
    (lane, cl), (wave, cw) = _run(gpu_ctx, w, req, 1, False), _run(gpu_ctx, w, req, 64, False)
    assert np.array_equal(_bytes(lane), _bytes(wave))
    print(f"\n[counters pen={pen} faces={faces}] lane {cl.tolist()} wavefront {cw.tolist()}")
    assert cl[1] > cl[4] > 0 and cl[2] > 100
    assert np.array_equal(cl[[0, 1, 2, 4]], cw[[0, 1, 2, 4]])
