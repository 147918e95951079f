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


@pytest.mark.parametrize("threshold", [1e-3, 1e-9])
def test_records_of_a_one_leaf_tree(threshold):
    """One face: the tree is one leaf, which no child pair holds; its record is
    the face's box (an empty one where the round removed the face) with the
    face and no escape, as any leaf's."""
    import ctypes

    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from pamo_amd import _hip
    from pamo_amd.pamo import CUDSP_Free
    print(f"case: one face, threshold {threshold}", flush=True)
    V = np.array([[0.5, -0.25, 1.0], [-1.0, 0.125, 0.75], [0.25, 2.0, -0.5]], np.float32)
    F = np.array([[0, 1, 2]], np.int32)
    op = CUDSP_Free(0)
    p, t, *_ = op.forward(torch.from_numpy(V).cuda(), torch.from_numpy(F).cuda(),
                          torch.zeros(0, dtype=torch.int32, device="cuda"), 0, 3.0, threshold, 0, True)
    p, t = p.cpu().numpy(), t.cpu().numpy()
    assert op.debug(_hip.PAMO_DBG_BVH_N) == 1
    buf = torch.full((8,), 7.0, dtype=torch.float32, device="cuda")
    n = ctypes.c_longlong(0)
    _hip.check(_hip.lib().pamo_round_debug(op.ctx.ptr, _hip.PAMO_DBG_BVH_BOXES, buf.data_ptr(), 8, ctypes.byref(n)),
               "pamo_round_debug")
    assert n.value == 8
    box, at = buf.cpu().numpy(), p[t[0]]
    if t[0, 0] < 0:
        assert np.all(box[:3] == np.inf) and np.all(box[4:7] == -np.inf)
    else:
        assert np.array_equal(box[:3], at.min(0)) and np.array_equal(box[4:7], at.max(0))
    assert box.view(np.int32)[[3, 7]].tolist() == [0, -1]


def test_byte_models_count_a_closed_meshs_edges():
    """The launch profiler's bytes: launches over the edges cover a bound (two
    a face), their compulsory traffic is that of the edges (1.5 a face)."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from pamo_amd import _hip, synth
    from pamo_amd.pamo import CUDSP_Free
    V, F = synth.icosphere_sh(3, 3)
    V = centred(V, F)
    print(f"case: byte models, {len(F)} faces", flush=True)
    op = CUDSP_Free(0)
    prof = _hip.Profiler(op.ctx)
    prof.enable()
    op.forward(torch.from_numpy(V).cuda(), torch.from_numpy(F).cuda(), torch.zeros(0, dtype=torch.int32, device="cuda"),
               0, float((V.max(0) - V.min(0)).max()), 1e-3, 0, True)
    by = {s["name"]: s["bytes"] for s in prof.stats()}
    nP, nT = len(V), len(F)
    nE = op.debug(_hip.PAMO_DBG_EDGES).numel() // 2
    assert nE == 1.5 * nT
    assert by["edge_cost"] == 16 * nE + 85 * nP + 48 * nT
    assert by["select_collapse"] == 16 * nE + 12 * nP + 48 * nT
    assert by["line_flag"] == 12 * nE + 16 * nP + 12 * nT
