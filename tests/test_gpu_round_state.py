"""What a context keeps between rounds: the point map that an undo reads, the
stored edge costs and the edge capacity, over calls whose meshes shrink and
grow again on one context; bit for bit against the CPU oracle."""
import numpy as np
import pytest

from stage2_helpers import centred

pytestmark = pytest.mark.gpu

NAMES = ["verts", "tris", "occ", "map", "undo"]


@pytest.mark.parametrize("levels", [(3, 1, 2, 3), (3, 0, 0, 3), (1, 2, 4, 1)])
def test_rounds_of_changing_size_on_one_context(oracle_lib, levels):
    """Sheets 1e-3 apart, so that rounds undo collapses and read the map of
    the call before, also its entries past that call's points; the edge list
    (1.5 a face) passes the capacity on the growing calls only."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from pamo_amd import synth
    from pamo_amd.pamo import CUDSP_Free
    op, ref = CUDSP_Free(0), oracle_lib.Round()
    undos = 0
    for it, level in enumerate(levels):
        V, F = synth.icosphere_sh(level, 3)
        V, F = synth.offset_sheets(V, F, rel_offset=1e-3)
        V = centred(V, F)
        scale = float((V.max(0) - V.min(0)).max())
        none = np.zeros(0, np.int32)
        print(f"case: call {it}, {len(V)} points, {len(F)} faces", flush=True)
        a = op.forward(torch.from_numpy(V).cuda(), torch.from_numpy(F).cuda(), torch.from_numpy(none).cuda(), 0, scale,
                       1e-3, 0, it == 0)
        b = ref.forward(V, F, none, 0, scale, 1e-3, 0, it == 0)
        undos += len(ref.undo_iters())
        for n, x, y in zip(NAMES, a, b):
            x = x.cpu().numpy()
            assert x.shape == y.shape and x.tobytes() == y.tobytes(), f"call {it}: {n}"
    assert undos > 0 or 3 not in levels, "the case undid nothing"
