"""Nearest-face walks at the sizes where their launch changes: one face, two,
points around the wave size, the sort's threshold and the step budget's, and
trees deeper than a lane's stack; against the brute-force oracle."""
import numpy as np
import pytest
import torch

from oracle import metrics as om
from pamo_amd import _hip, metrics, synth

pytestmark = pytest.mark.gpu


def _check(P, V, F):
    sq, idx, C = metrics.point_mesh_squared_distance(P, V, F)
    so, io = om.point_mesh_sqdist(P, V, F)
    # the same arithmetic for each face; where rounding parts two faces that share the nearest point, the smaller
    # distance may differ by a few units in the last place
    assert np.all(np.abs(sq - so) <= 1e-12 * so + 1e-30)
    for i in np.flatnonzero(idx != io):
        assert om.point_tri_sqdist(P[i], *V[F[idx[i]]]) == pytest.approx(so[i], rel=1e-12, abs=1e-30)
    assert np.all(np.abs(((C - P) ** 2).sum(1) - sq) <= 1e-12 * sq + 1e-30)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 4095, 4096, 32768, 32769])
def test_point_counts_around_the_thresholds(n):
    print(f"case: {n} points", flush=True)
    V, F = synth.icosphere_sh(level=2, seed=4)
    V = V.astype(np.float64)
    rng = np.random.default_rng(n)
    # half near the surface, half far off or inside (long walks)
    P = V[rng.integers(0, len(V), n)] * rng.choice([1.001, 0.0, 0.3, 4.0], n)[:, None] + 1e-3 * rng.standard_normal((n, 3))
    _check(P, V, F)


@pytest.mark.parametrize("faces", [1, 2, 3])
def test_smallest_trees(faces):
    print(f"case: {faces} faces", flush=True)
    rng = np.random.default_rng(faces)
    V = rng.standard_normal((3 * faces, 3))
    F = np.arange(3 * faces, dtype=np.int32).reshape(-1, 3)
    _check(rng.standard_normal((100, 3)) * 3, V, F)


def test_tree_deeper_than_the_stack():
    """30 places whose Morton codes differ bit by bit, 64 equal triangles at
    each: from near the origin a walk passes 36 levels before its first face."""
    print("case: deep tree", flush=True)
    at = [np.eye(3)[d] * 2.0 ** -k for k in range(10) for d in range(3)]
    tri = np.array([[0, 0, 0], [1e-5, 0, 0], [0, 1e-5, 0]])
    V = np.concatenate([a + tri for a in at for _ in range(64)])
    F = np.arange(len(V), dtype=np.int32).reshape(-1, 3)
    rng = np.random.default_rng(1)
    P = np.concatenate([1e-4 * rng.standard_normal((40, 3)), rng.uniform(-1, 2, (40, 3))])
    _check(P, V, F)


def test_points_without_a_distance():
    """A point with a NaN or infinite coordinate has no nearest face; the
    others of its wave keep theirs."""
    print("case: NaN and infinite points", flush=True)
    V, F = synth.icosphere_sh(level=3, seed=2)
    V = V.astype(np.float64)
    P = np.random.default_rng(3).standard_normal((130, 3))
    bad = [0, 70, 129]
    P[bad] = [[np.nan, 0, 0], [np.inf, 0, 0], [0, np.nan, np.nan]]
    sq, idx, _ = metrics.point_mesh_squared_distance(P, V, F)
    assert np.all(np.isinf(sq[bad])) and np.all(idx[bad] == -1)
    ok = np.setdiff1d(np.arange(len(P)), bad)
    so, _ = om.point_mesh_sqdist(P[ok], V, F)
    assert np.all(np.abs(sq[ok] - so) <= 1e-12 * so)


@pytest.mark.parametrize("n", [300, 5000, 33000])
@pytest.mark.parametrize("scale", [1e18, 1e20])
def test_distances_beyond_single_precision(scale, n):
    """Coordinates that 32-bit boxes hold, squared distances that 32 bits do
    not (above 3.4e38 from 1.8e19 on): each point count takes another launch."""
    print(f"case: scale {scale:g}, {n} points", flush=True)
    V, F = synth.icosphere_sh(level=3, seed=2)
    V = V.astype(np.float64) * scale
    rng = np.random.default_rng(n)
    _check(rng.uniform(-3.0, 3.0, (n, 3)) * scale, V, F)


def test_hausdorff_beyond_single_precision():
    print("case: Hausdorff at 1e20", flush=True)
    (VA, FA), (VB, FB) = synth.icosphere_sh(level=3, seed=2), synth.icosphere_sh(level=2, seed=5)
    VA, VB = VA.astype(np.float64) * 1e20, VB.astype(np.float64) * 3e20
    assert metrics.hausdorff(VA, FA, VB, FB) == pytest.approx(om.hausdorff(VA, FA, VB, FB), rel=1e-12)


def test_buffers_of_a_large_call_are_bounded():
    """A context keeps order and leftover buffers for 2^24 points at most (24
    bytes each, and the sort's histograms), and points past that number are
    walked as in calls of their own."""
    n, cut = 40_000_000, 1 << 24
    print(f"case: {n} points", flush=True)
    V, F = synth.icosphere_sh(level=2, seed=4)
    m = metrics._Metrics(0)
    Vd, Fd = torch.from_numpy(V.astype(np.float64)).cuda(), torch.from_numpy(F).cuda()
    P = torch.rand((n, 3), dtype=torch.float64, device="cuda", generator=torch.Generator("cuda").manual_seed(1)) * 4 - 2

    def call(P):
        k = len(P)
        out = (torch.empty(k, dtype=torch.float64, device="cuda"), torch.empty(k, dtype=torch.int32, device="cuda"),
               torch.empty((k, 3), dtype=torch.float64, device="cuda"))
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        _hip.check(_hip.lib().pamo_point_mesh_sqdist(m.ptr, P.data_ptr(), k, Vd.data_ptr(), len(V), Fd.data_ptr(),
                                                     len(F), *(t.data_ptr() for t in out)), "pamo_point_mesh_sqdist")
        return out, free - torch.cuda.mem_get_info()[0]

    whole, kept = call(P)
    assert kept < 640 << 20, kept
    for a, b in ((0, 5000), (cut - 3000, cut + 3000), (2 * cut - 70000, 2 * cut + 70000), (n - 100, n)):
        part, _ = call(P[a:b].contiguous())
        assert all(torch.equal(w[a:b], p) for w, p in zip(whole, part))
