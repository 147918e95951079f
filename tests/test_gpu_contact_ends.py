"""Contacts at the ends of the detection's range: a mesh of one face (a tree of
one leaf, whose box is tested like any other leaf's), and a frontier that
fills."""
import numpy as np
import pytest
import torch

from pamo_amd import _hip, stage3
from test_gpu_walks import _expand

pytestmark = pytest.mark.gpu


def _contacts(V, F):
    s = stage3.Stage3System()
    s.set_target(torch.from_numpy(V[:3].copy()).cuda(), torch.from_numpy(F[:1].copy()).cuda(), 1.0, np.zeros(3))
    s.set_mesh_prepared(V, F, stage3.edges_unique(F), np.zeros((0, 4), np.int32), np.ones(len(V), np.float32), False,
                        1.0, np.zeros(3))
    return {tuple(r) for r in s.debug(_hip.PAMO_S3_DBG_CONTACTS).astype(np.int64).tolist()}


def test_box_decides_as_beside_a_second_face():
    """Vertices around 2 r + d_hat from the edge of a face, a few units in the
    last place on either side: the computed distance of some is within it
    while the boxes are apart.  With a second face far away the tree has
    two leaves, and the contacts of the first face are the same."""
    print("case: one face, vertices at the threshold", flush=True)
    cfg = stage3.Stage3Config()
    rng = np.random.default_rng(5)
    thr = np.float32(2) * np.float32(cfg.contact_detection_radius) + np.float32(cfg.d_hat)
    n = 20000
    y = np.full(n, -thr, np.float32).view(np.int32) + rng.integers(-4, 5, n).astype(np.int32)
    P = np.stack([rng.uniform(0.3, 0.6, n).astype(np.float32), y.view(np.float32), np.zeros(n, np.float32)], 1)
    face = np.array([[0.25, 0, 0], [0.7, 0, 0], [0.4, 0.3, 0]], np.float32)
    far = face + np.float32(5.0)
    one = _contacts(np.concatenate([face, P]), np.array([[0, 1, 2]], np.int32))
    two = _contacts(np.concatenate([face, P, far]), np.array([[0, 1, 2], [n + 3, n + 4, n + 5]], np.int32))
    # (a vertex whose box is apart from the face's has no contact; some are that far by rounding alone)
    assert 0 < len(two) < n
    assert one == two


def test_frontier_full_lists_every_pair(oracle_lib):
    """60 vertices within reach of each other and every face over them: a
    query meets all 34,220 leaves, so a wave's frontier of 512 nodes fills and
    lanes walk the rest of their subtrees by themselves; every vertex against
    every face without it, every two edges without a common vertex, once."""
    from itertools import combinations
    print("case: every face over 60 vertices", flush=True)
    n = 60
    V = (0.3 + 0.01 * np.random.default_rng(3).random((n, 3))).astype(np.float32)
    F = np.array(list(combinations(range(n), 3)), np.int32)
    E = np.array(list(combinations(range(n), 2)), np.int32)
    # the frontier of a wave's four queries, over the same hierarchy
    T = V[F]
    c, lo, hi = (T.min(1) + T.max(1)) * np.float32(0.5), T.min((0, 1)), T.max((0, 1))
    q = np.minimum(((c - lo) / (hi - lo) * 1024).astype(np.int64), 1023)
    code = (_expand(q[:, 0]) * 4 + _expand(q[:, 1]) * 2 + _expand(q[:, 2])).astype(np.uint32)
    by = np.argsort(code, kind="stable")
    left, right = oracle_lib.karras(code[by], by.astype(np.int32))
    stack, most = [0] * 4, 0
    while stack:
        top, stack = stack[-64:], stack[:-64]
        stack += [k for x in top if x < len(F) - 1 for k in (left[x], right[x])]
        most = max(most, len(stack))
    assert most > 512, most
    s = stage3.Stage3System()
    s.set_target(torch.from_numpy(V).cuda(), torch.from_numpy(F[:1].copy()).cuda(), 1.0, np.zeros(3))
    s.set_mesh_prepared(V, F, E, np.zeros((0, 4), np.int32), np.ones(n, np.float32), False, 1.0, np.zeros(3))
    got = s.debug(_hip.PAMO_S3_DBG_CONTACTS)
    key = lambda a: np.sort((a * np.array([n ** 3, n ** 2, n, 1])).sum(1))
    kinds = [key(got[got[:, 4] == k, :4]) for k in np.unique(got[:, 4])]
    v, f = np.divmod(np.arange(n * len(F)), len(F))
    pt = np.concatenate([v[:, None], F[f]], 1)[(F[f] != v[:, None]).all(1)]
    a, b = np.triu_indices(len(E), 1)
    ee = np.concatenate([E[a], E[b]], 1)
    ee = ee[(ee[:, :2, None] != ee[:, None, 2:]).all((1, 2))]
    assert len(kinds) == 2 and sorted(map(len, kinds)) == sorted([len(pt), len(ee)])
    for want in (key(pt), key(ee)):
        assert any(np.array_equal(want, k) for k in kinds)
