"""Remeshing at resolutions around the sizes of its blocks (bricks of 8
samples, words of 64): the outside mask, the vertices and the triangle count
from the context's own distance field by numpy, and one context used for a
large grid and then a smaller one."""
import numpy as np
import pytest
import torch
from scipy import ndimage

import test_gpu_stage1 as t1
from pamo_amd import _hip, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case,R", [("icosphere", 8), ("boxes", 9), ("sheet", 15), ("boxes", 33), ("icosphere", 65),
                                    ("boxes", 71)])
def test_steps_after_the_field(case, R):
    print(f"case: remesh {case}, R {R}", flush=True)
    V, F = synth.icosphere_sh(3, 3) if case == "icosphere" else (t1._sheet() if case == "sheet" else t1._boxes())
    r = t1._remesher()
    Vd, Fd = t1._dev(V, F)
    v, f = r.remesh(Vd, Fd, t1._mean(V, F), R)
    u = r.debug(_hip.PAMO_S1_DBG_FIELD, np.uint32, R ** 3).view(np.float32).reshape(R, R, R)  # z, y, x
    outside = r.debug(_hip.PAMO_S1_DBG_OUTSIDE, np.uint8, R ** 3).reshape(R, R, R).astype(bool)
    iso = r.debug(_hip.PAMO_S1_DBG_FRAME, np.float32, 8)[7]
    # outside: the 6-connected passable regions that reach the border
    lab, _ = ndimage.label(u > np.float32(0.55) / np.float32(R))
    edge = np.ones((R, R, R), bool)
    edge[1:-1, 1:-1, 1:-1] = False
    reach = np.unique(lab[edge & (lab > 0)])
    assert np.array_equal(outside, np.isin(lab, reach) & (lab > 0))
    # one vertex for each crossing grid edge, x edges first, in sample order
    d = np.where(outside, u, -u)
    inside = d < iso
    pts = []
    for ax in (2, 1, 0):
        a = np.take(d, range(R - 1), ax), np.take(d, range(1, R), ax)
        z, y, x = np.nonzero(np.take(inside, range(R - 1), ax) != np.take(inside, range(1, R), ax))
        d0, d1 = a[0][z, y, x], a[1][z, y, x]
        p = np.stack([x, y, z], 1).astype(np.float32)
        p[:, 2 - ax] += (iso - d0) / (d1 - d0)
        pts.append(p)
    vi = r.debug(_hip.PAMO_S1_DBG_VERTS, np.float32, 4 * max(len(v), 1)).reshape(-1, 4)[:len(v), :3]
    assert np.array_equal(vi, np.concatenate(pts))
    ntri = r.debug(_hip.PAMO_S1_DBG_CASES, np.int8, 256 * 18).reshape(256, 18)[:, 17]
    c = sum(np.take(np.take(np.take(inside, range(k >> 2, R - 1 + (k >> 2)), 0), range((k >> 1) & 1, R - 1 + ((k >> 1) & 1)), 1),
                    range(k & 1, R - 1 + (k & 1)), 2).astype(int) << k for k in range(8))
    assert len(f) == ntri[c].sum()
    t1._check_closed_manifold(f.cpu().numpy(), len(v))


def test_smaller_grid_after_a_larger_one():
    print("case: remesh R 72 then 20 on one context", flush=True)
    V, F = t1._boxes()
    Vd, Fd = t1._dev(V, F)
    mean = t1._mean(V, F)
    used = t1._remesher()
    used.remesh(Vd, Fd, mean, 72)
    v, f = used.remesh(Vd, Fd, mean, 20)
    v0, f0 = t1._remesher().remesh(Vd, Fd, mean, 20)
    assert torch.equal(v, v0) and torch.equal(f, f0)
