"""Contacts against a mesh of one face: a tree of one leaf, whose box is tested
like any other leaf's."""
import numpy as np
import pytest
import torch

from pamo_amd import _hip, stage3

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
