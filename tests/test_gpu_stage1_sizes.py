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


@pytest.mark.parametrize("R", [64, 72, 128])
def test_faces_along_the_grid(R):
    """Flat faces along the grid: words whose 64 samples all cross, and (R = 72)
    words that end inside a row."""
    test_steps_after_the_field("boxes", R)


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


def _cube():
    V = t1._box_tris((0.0, 0.0, 0.0), (1.0, 1.0, 1.0)).reshape(-1, 3).astype(np.float32)
    return V, np.arange(36, dtype=np.int32).reshape(-1, 3)


def _turned_cube():
    V, F = _cube()
    q, _ = np.linalg.qr(np.random.default_rng(1).standard_normal((3, 3)))
    return (V @ q).astype(np.float32), F


@pytest.mark.parametrize("times,R", [(1, 33), (1, 70), (1400, 70)])
def test_field_of_large_triangles(times, R):
    """Triangles whose rows have up to R columns, more than a work item takes
    (rows of every remainder among them), against the oracle's field; the same
    faces many times over take the dense meshes' longer segments."""
    from oracle import stage1 as o
    V, F = _turned_cube()
    print(f"case: field of {len(F)} large triangles, {times} times, R {R}", flush=True)
    r = t1._remesher()
    r.remesh(*t1._dev(V, np.tile(F, (times, 1))), t1._mean(V, F), R)
    tris = r.debug(_hip.PAMO_S1_DBG_NORMALIZED, np.float32, 12 * len(F) * times).reshape(-1, 3, 4)[:len(F), :, :3]
    field = r.debug(_hip.PAMO_S1_DBG_FIELD, np.uint32, R ** 3).view(np.float32).reshape(R, R, R)
    ref = o.udf(tris, R, 3.0 / R)
    assert np.array_equal(np.isfinite(field), np.isfinite(ref))
    fin = np.isfinite(ref)
    assert np.abs(field[fin] - ref[fin]).max() <= 2e-7


def test_few_large_triangles_spread_over_the_chip():
    """12 triangles across the grid are no more work than 5120 small ones on a
    surface of that size (their samples are the same): the call takes no
    longer, with room for noise (2.5 times as long with a row of columns a
    lane, 0.7 with a column a lane, 0.9 now)."""
    import time
    print("case: remesh 12 and 5120 triangles, R 128", flush=True)
    r = t1._remesher()
    meshes = [t1._dev(*m) for m in (_cube(), synth.icosphere_sh(4, 3))]
    times = [[], []]
    for _ in range(25):
        for k, (V, F) in enumerate(meshes):
            t = time.perf_counter()
            r.remesh(V, F, (0.0, 0.0, 0.0), 128)
            torch.cuda.synchronize()
            times[k].append(time.perf_counter() - t)
    few, many = (float(np.median(t[5:])) for t in times)
    print(f"few {few * 1e3:.3f} ms, many {many * 1e3:.3f} ms", flush=True)
    assert few < 1.7 * many, (few, many)
