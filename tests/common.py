"""Shared helpers for the parity tests (workload setup for oracle and device)."""
from contextlib import contextmanager

import numpy as np

from mfcl import autotune
from mfcl import workloads as W


@contextmanager
def knobs(ctx, values):
    """Launch knobs {knob: value} for a block of a test; back to the defaults
    after it (the suites share one context)."""
    try:
        for k, v in values.items():
            autotune.set_knob(ctx, k, v)
        yield
    finally:
        for k in values:
            autotune.set_knob(ctx, k, autotune.DEFAULTS[k])


def hull_shapes_for_oracle(h, idx_hulls):
    """Faces (qhull) for the listed hulls; returns oracle ShapeSet arguments
    covering only those hulls, and the map shape -> local hull id."""
    vs, ts, vo, vc, to, tc = [], [], [], [], [], []
    o = q = 0
    for i in idx_hulls:
        pts = h["verts"][h["vert_off"][i]:h["vert_off"][i] + h["vert_cnt"][i]]
        keep, tri = W.hull_faces(pts)
        v = pts[keep]
        vs.append(v)
        ts.append(tri)
        vo.append(o)
        vc.append(len(v))
        to.append(q)
        tc.append(len(tri))
        o += len(v)
        q += len(tri)
    return (np.concatenate(vs), np.array(vo), np.array(vc), np.concatenate(ts), np.array(to), np.array(tc))


def scale_of(types, params, pa, pb, verts=None, vert_off=None, vert_cnt=None):
    r = W.bounding_radius(types, params, vert_cnt, verts, vert_off)
    return r[pa] + r[pb]
