"""Nearest-face walks at the sizes where their launch changes: one face, two,
points around the wave size, the sort's threshold and the step budget's, and
trees deeper than a lane's stack; against the brute-force oracle."""
import numpy as np
import pytest
import torch

from oracle import metrics as om
from pamo_amd import _hip, metrics, stage3, synth

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
    each: from near the origin a walk passes 36 levels before its first face, so a
    lane meets none within its steps and leaves the query to a wave, whose stack
    holds it (the walks that run out of stack: below)."""
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


def _deep_mesh():
    """The mesh of test_tree_deeper_than_the_stack, and points near its
    origin: the way down to their first face leaves 30 places behind, all of
    them still to visit, on a stack of 24."""
    at = [np.eye(3)[d] * 2.0 ** -k for k in range(10) for d in range(3)]
    tri = np.array([[0, 0, 0], [1e-5, 0, 0], [0, 1e-5, 0]])
    V = np.concatenate([a + tri for a in at for _ in range(64)])
    P = 1e-4 * np.random.default_rng(1).standard_normal((100, 3))
    return P, V, np.arange(len(V), dtype=np.int32).reshape(-1, 3)


def test_lane_finishes_by_links_when_its_stack_ran_out():
    """The allocation-free form has no buffer for leftover queries, so every
    lane finishes its own: here with nodes that found no place on its stack."""
    print("case: deep tree, no leftovers", flush=True)
    P, V, F = _deep_mesh()
    Pd, Vd, Fd = (torch.from_numpy(a).cuda() for a in (P, V, F))
    sq = torch.empty(len(P), dtype=torch.float64, device="cuda")
    idx = torch.empty(len(P), dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    _hip.check(_hip.lib().pamo_point_mesh_sqdist_noalloc(Pd.data_ptr(), len(P), Vd.data_ptr(), len(V), Fd.data_ptr(),
                                                         len(F), sq.data_ptr(), idx.data_ptr(), None,
                                                         torch.cuda.current_stream().cuda_stream), "noalloc")
    torch.cuda.synchronize()
    so, io = om.point_mesh_sqdist(P, V, F)
    assert np.all(np.abs(sq.cpu().numpy() - so) <= 1e-12 * so)
    assert np.array_equal(idx.cpu().numpy(), io)  # the places' 64 equal triangles: the smallest number


def test_stage3_targets_when_the_stack_ran_out():
    """Stage 3's closest points over the same tree (its lanes have the same
    stack and no second kernel)."""
    print("case: deep tree as a stage-3 target", flush=True)
    _, gV, gF = _deep_mesh()
    V, F = synth.icosphere(1)
    V = (V * 1e-4).astype(np.float32)
    s = stage3.Stage3System()
    s.register_mesh(gV.astype(np.float32), gF, V, F)
    got = s.debug(_hip.PAMO_S3_DBG_TARGET).reshape(-1, 3)
    P = V.astype(np.float64)
    so, _ = om.point_mesh_sqdist(P, gV.astype(np.float32).astype(np.float64), gF)
    # 32-bit coordinates below 1: a distance's error is below 1e-6
    assert np.abs(np.sqrt(((got - P) ** 2).sum(1)) - np.sqrt(so)).max() < 1e-6
    on, _ = om.point_mesh_sqdist(got, gV.astype(np.float32).astype(np.float64), gF)
    assert np.sqrt(on).max() < 1e-6


def _expand(v):
    out = np.zeros_like(v)
    for b in range(10):
        out |= ((v >> b) & 1) << (3 * b)
    return out


def test_wave_walk_beyond_its_stack(oracle_lib):
    """64 cells, each with a chain of 24 places that split off one by one from
    the corner where most triangles are: a wave's walk goes down all chains at
    once (the right children, last pushed) and leaves 64 nodes behind a step, more
    than 1024 before its first face; a lane meets no face within its 32 steps,
    so nothing is pruned."""
    print("case: wide frontier", flush=True)
    cells = np.stack(np.meshgrid(*[np.arange(4)] * 3, indexing="ij"), -1).reshape(-1, 3) * 256
    ones = np.array([255, 255, 255])
    places = [ones - np.eye(3, dtype=int)[d] * (1 << b) for b in range(8) for d in range(3)]
    at = np.concatenate([np.repeat([c + p for p in places], 2, 0) for c in cells] +
                        [np.repeat([c + ones], 64, 0) for c in cells] + [[[0, 0, 0]]])
    centre = at / 1023.0  # place x of 1024 along an axis of the whole box, which is the unit cube
    tri = np.array([[1, 0, 0], [-1, 0, 0], [0, 0, 0]]) * 1e-6
    V = (centre[:, None] + tri).reshape(-1, 3)
    F = np.arange(len(V), dtype=np.int32).reshape(-1, 3)
    # the frontier, over the same hierarchy
    code = (_expand(at[:, 0]) * 4 + _expand(at[:, 1]) * 2 + _expand(at[:, 2])).astype(np.uint32)
    by = np.argsort(code, kind="stable")
    left, right = oracle_lib.karras(code[by], by.astype(np.int32))
    inner, stack, faces = len(F) - 1, [0], False
    while not faces:
        top, stack = stack[-64:], stack[:-64]
        kids = [left[x] for x in top] + [right[x] for x in top]
        faces = any(k >= inner for k in kids)
        stack += [k for k in kids if k < inner]
    assert len(stack) > 1024, len(stack)
    depth, x = 0, 0  # a lane's way down to the corner that is nearest to (2, 2, 2)
    while x < inner:
        x, depth = right[x], depth + 1
    assert depth > 32, depth
    P = 2.0 + 1e-3 * np.random.default_rng(2).standard_normal((40, 3))
    _check(P, V, F)
