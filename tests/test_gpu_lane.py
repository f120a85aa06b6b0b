"""GPU: the one-lane-per-pair GJK kernel (cooperative hull scans) against the
one-wavefront-per-pair kernel and the oracle.

The lane kernel runs the same FP64 operations in the same order as the wavefront
kernel, only scheduled differently, so the bar between them is bit equality
of every result record (and equal work counters), on a mixed
workload (hull-hull, hull-primitive and primitive-primitive pairs, hulls of
4..1500 points so scans span 1..24 wavefront chunks, out-of-range shape ids,
zero and non-zero guesses) in signed-distance and penetration modes.  Both
kernels also equal the oracle bit for bit on hulls given as vertex sets.
"""
import numpy as np
import pytest

from common import knobs
from mfcl import autotune
from mfcl import workloads as W
import mfcl


def _mixed(seed, n_pairs=6000):
    rng = np.random.default_rng(seed)
    h = W.hull_pairs(700, seed, nmin=4, nmax=1500)
    p = W.primitive_pairs(700, seed + 1)
    nh = len(h["types"])
    types = np.concatenate([h["types"], p["types"]]).astype(np.int32)
    params = np.concatenate([h["params"], p["params"]]).astype(np.float32)
    vert_off = np.concatenate([h["vert_off"], np.zeros(len(p["types"]), np.uint64)])
    vert_cnt = np.concatenate([h["vert_cnt"], np.zeros(len(p["types"]), np.uint32)])
    n = len(types)
    pa = rng.integers(0, n, size=n_pairs).astype(np.uint32)
    pb = rng.integers(0, n, size=n_pairs).astype(np.uint32)
    pa[::97] = n + 5  # out-of-range ids are reported, not read
    qa = W.poses(rng, n_pairs, 0.0, 0.6)
    qb = W.poses(rng, n_pairs, 0.0, 0.6)
    guess = rng.normal(size=(n_pairs, 3)).astype(np.float32)
    guess[::7] = 0
    return dict(types=types, params=params, verts=h["verts"], vert_off=vert_off, vert_cnt=vert_cnt,
                pair_a=pa, pair_b=pb, pose_a=qa, pose_b=qb, guess=guess, n_hull_shapes=nh)


def _run(ctx, w, req, group, guess):
    """Device-buffer entry point (the host-buffer one rejects out-of-range
    ids before launching; the kernels must report them per pair)."""
    n = len(w["pair_a"])
    dev = [ctx.to_device(np.ascontiguousarray(w[k])) for k in ("pair_a", "pair_b", "pose_a", "pose_b", "guess")]
    dout = ctx.alloc(n * mfcl.CONVEX_RESULT_DTYPE.itemsize)
    with knobs(ctx, {autotune.GJK_GROUP: group}):
        ctx.convex_query_dev(dev[0], dev[1], dev[2], dev[3], n, req, dout, guess=dev[4] if guess else None)
        ctx.sync()
        cnt = ctx.last_counters().copy()
    out = np.zeros(n, mfcl.CONVEX_RESULT_DTYPE)
    dout.download(out)
    for d in dev + [dout]:
        d.free()
    return out, cnt


@pytest.mark.gpu
@pytest.mark.parametrize("mode,pen,guess", [("sd", 0, False), ("sd", 0, True), ("collide", 1, False),
                                            ("collide", 1, True), ("collide", 0, False)])
def test_lane_kernel_equals_group_kernel(gpu_ctx, mode, pen, guess):
    w = _mixed(21)
    gpu_ctx.upload_shapes(w["types"], w["params"], w["vert_off"], w["vert_cnt"], w["verts"])
    if mode == "sd":
        req = mfcl.request(mfcl.MODE_SIGNED_DISTANCE, use_guess=int(guess))
    else:
        req = mfcl.request(mfcl.MODE_COLLIDE, max_contacts=4, penetration=pen, use_guess=int(guess))
    ref, cref = _run(gpu_ctx, w, req, 32, guess)
    out, cout = _run(gpu_ctx, w, req, 1, guess)
    diff = out.view(np.uint8).reshape(len(out), -1) != ref.view(np.uint8).reshape(len(ref), -1)
    bad = np.nonzero(diff.any(1))[0]
    print(f"\n[lane vs wavefront {mode} guess={guess}] pairs={len(out)} differing={len(bad)} "
          f"gjk statuses {np.bincount(out['gjk_status'].astype(np.int64) + 1).tolist()} "
          f"epa queued {int((out['epa_status'] >= 0).sum())} counters lane {cout[:3].tolist()} wavefront {cref[:3].tolist()}")
    assert len(bad) == 0, (bad[:10], out[bad[:3]], ref[bad[:3]])
    # pairs, vertices evaluated, EPA pairs, EPA restarts and EPA vertices
    assert np.array_equal(cout[:5], cref[:5])
    assert (out["ok"] == -1).sum() == len(out[::97])


@pytest.mark.gpu
@pytest.mark.parametrize("group", [0, 1, 32])
def test_hull_signed_distance_bit_exact_vs_naive_oracle(oracle, gpu_ctx, group):
    """Hulls given as bare vertex sets use the naive support scan
    (convex-inl.h:133-149) in the reference, the oracle and both GPU kernels;
    GJK, EPA and the witness extraction then perform the same FP64
    operations, so every field must agree exactly."""
    h = W.hull_pairs(4096, 5)
    S = oracle.ShapeSet(h["types"], h["params"], h["verts"], h["vert_off"], h["vert_cnt"])
    ta, tb = oracle.pose12(h["pose_a"]), oracle.pose12(h["pose_b"])
    ref, _ = S.signed_distance(h["pair_a"], h["pair_b"], ta, tb, threads=8)
    gpu_ctx.upload_shapes(h["types"], h["params"], h["vert_off"], h["vert_cnt"], h["verts"])
    req = mfcl.request(mfcl.MODE_SIGNED_DISTANCE)
    with knobs(gpu_ctx, {autotune.GJK_GROUP: group}):
        out = gpu_ctx.convex_query(h["pair_a"], h["pair_b"], h["pose_a"], h["pose_b"], req)
    fields = ("ok", "gjk_status", "epa_status", "gjk_iters", "epa_iters", "distance", "pa", "pb")
    diff = {f: int((out[f] != ref[f]).reshape(len(out), -1).any(1).sum()) for f in fields}
    print(f"\n[naive oracle, group {group}] pairs={len(out)} intersecting={int((ref['distance'] < 0).sum())} "
          f"differing per field {diff}")
    assert all(v == 0 for v in diff.values())


@pytest.mark.gpu
@pytest.mark.parametrize("walking,guess,pen", [(False, False, False), (False, True, False), (True, False, False),
                                              (False, True, True), (True, False, True)])
def test_lane_refill_thresholds_identical(gpu_ctx, walking, guess, pen):
    """The refilled lane grid (finished lanes take new pairs once at most k
    lanes of their wavefront still run), signed distance and penetration
    (closed forms among the pairs): every result record is byte-identical
    for k = 1, 48, 63 and without refill (one pair per lane), on scanning and
    on walking hulls; so are the work counters."""
    if walking:
        h = W.hull_pairs(3000, 24, faces=True)
        gpu_ctx.upload_shapes(h["types"], h["params"], h["vert_off"], h["vert_cnt"], h["verts"],
                              faces=mfcl.faces_from_triangles(h["tris"], h["tri_off"], h["tri_cnt"]))
        w = dict(pair_a=h["pair_a"], pair_b=h["pair_b"], pose_a=h["pose_a"], pose_b=h["pose_b"],
                 guess=np.zeros((len(h["pair_a"]), 3), np.float32))
    else:
        w = _mixed(23)
        gpu_ctx.upload_shapes(w["types"], w["params"], w["vert_off"], w["vert_cnt"], w["verts"])
    if pen:
        req = mfcl.request(mfcl.MODE_COLLIDE, max_contacts=4, penetration=1, use_guess=int(guess))
    else:
        req = mfcl.request(mfcl.MODE_SIGNED_DISTANCE, use_guess=int(guess))
    runs = []
    for k in (0, 1, 48, 63):
        with knobs(gpu_ctx, {autotune.LANE_REFILL: k}):
            runs.append(_run(gpu_ctx, w, req, 1, guess))
    ref, cref = runs[0]
    print(f"\n[lane refill walking={walking} guess={guess} pen={pen}] pairs={len(ref)} "
          f"EPA queued {int((ref['epa_status'] >= 0).sum())} counters {cref[:5].tolist()}")
    for out, cnt in runs[1:]:
        assert out.tobytes() == ref.tobytes()
        assert np.array_equal(cnt[:5], cref[:5])
