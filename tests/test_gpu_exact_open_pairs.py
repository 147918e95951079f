"""The exact guard where filtered signs decide little: flat regions, whose
neighbouring faces lie in one plane, against the oracle's exact mode."""
import numpy as np
import pytest

from stage2_helpers import centred

pytestmark = pytest.mark.gpu


def cube(n, shear):
    """A cube of 12 n^2 faces; sheared, its planes hold no common coordinate
    and their corners only nearly lie in them."""
    ids, V, F = {}, [], []

    def vid(p):
        if p not in ids:
            ids[p] = len(V)
            V.append(p)
        return ids[p]

    for axis in range(3):
        for side in (0, n):
            for a in range(n):
                for b in range(n):
                    q = []
                    for da, db in ((0, 0), (1, 0), (1, 1), (0, 1)):
                        p = [0, 0, 0]
                        p[axis], p[(axis + 1) % 3], p[(axis + 2) % 3] = side, a + da, b + db
                        q.append(vid(tuple(p)))
                    if side == 0:
                        q.reverse()
                    F += [[q[0], q[1], q[2]], [q[0], q[2], q[3]]]
    V = np.array(V, np.float32) / np.float32(n)
    if shear:
        V = (V @ np.array([[1, 0.13, 0.29], [0.37, 1, 0.11], [0.23, 0.41, 1]], np.float32)).astype(np.float32)
    return V, np.array(F, np.int32)


@pytest.mark.parametrize("n,shear", [(1, False), (8, False), (8, True), (70, False)])
def test_flat_faces_match_oracle(oracle_lib, n, shear):
    """n = 70: 58,800 faces leave more pairs open in a round than the list
    first holds (2.4 a face of the capacity), so it grows and the round asks
    again."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from pamo_amd import _hip
    from pamo_amd.pamo import simplify_device
    V, F = cube(n, shear)
    Vc = centred(V, F)
    print(f"case: exact guard, cube of {len(F)} faces, shear {shear}", flush=True)
    ctx = _hip.Context(0)
    _hip.check(_hip.lib().pamo_ctx_set_option(ctx.ptr, _hip.PAMO_OPT_EXACT_GUARD, 1), "set_option")
    iters = 2 if n == 70 else 30
    vg, fg, hg = simplify_device(ctx, torch.from_numpy(Vc).cuda(), torch.from_numpy(F).cuda(), 0.05, iters=iters,
                                 min_verts=0)
    vo, fo, ho = oracle_lib.run(Vc, F, 0.05, iters=iters, min_verts=0, pred_mode=1)
    assert np.array_equal(hg, ho)
    assert np.array_equal(fg.cpu().numpy(), fo)
    assert np.array_equal(vg.cpu().numpy().view(np.uint32), vo.view(np.uint32))
