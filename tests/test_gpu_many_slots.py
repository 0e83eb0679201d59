"""Trees of more leaf slots than the cooperative tracers address (2^32 / 48):
the lane-per-ray tracers and canvas take them.  A small tree with its prim
indices padded past that line: records, counters and canvas bytes bit-exact
against the oracle's on the tree as it was."""
import numpy as np
import pytest

from test_gpu_parity import assert_same_hits, dev

pytestmark = pytest.mark.gpu

SLOTS = (1 << 32) // 48 + 1


@pytest.fixture(scope="module")
def scene(pm, orc, scenes):
    import torch
    from test_gpu_extras import shading_scene
    tris, _, normals, col, light = shading_scene(scenes)
    ref = orc.build(tris, orc.build_params("reference"))
    a = dict(ref.arrays())
    at = a["prim_indices"].shape[0]
    # half of the slots stay in front, half move to the end
    pad = np.zeros(SLOTS + 5, np.int32)
    half = at // 2
    pad[:at] = a["prim_indices"]
    pad[-at:] = a["prim_indices"]
    first = a["primitive_index"].copy()
    bits = a["primitive_bitmap"].view(np.uint64)
    leaf = (a["info"] & 3) == 0
    moved = leaf & (first >= half) & (bits != 0)
    first[moved] += pad.shape[0] - at
    a["prim_indices"], a["primitive_index"] = pad, first
    ctx = pm.Context(0)
    P = [dev(torch, t) for t in tris]
    ctx.set_tree(a, *P)
    assert ctx.view().num_prim_indices >= SLOTS and moved.any()
    yield ctx, ref, tris, normals, col, light, P
    ctx.close()


@pytest.mark.parametrize("algo,stack", [("SHORT_STACK", 3), ("SHORT_STACK", 8), ("SHORT_STACK", 16), ("KD_RESTART", 4)])
@pytest.mark.parametrize("test", ["MOELLER", "WOOP"])
@pytest.mark.parametrize("skip", [0, 1])
def test_traces_bit_exact(pm, orc, scenes, scene, algo, stack, test, skip):
    import torch
    ctx, ref, tris = scene[:3]
    a, ix = getattr(pm, algo), getattr(pm, test)
    org, dirs = scenes.random_rays(70001, seed=4, lo=-2.0, hi=2.0, target_lo=-1.0, target_hi=1.0)
    dirs[:9, :3] = 0.0
    for n in (1, 65, 70001):
        o, d = org[-n:].copy(), dirs[-n:].copy()
        O, D = dev(torch, o), dev(torch, d)
        want, wc = orc.trace(ref, tris, o, d, a, leaf_skipping=bool(skip), stack_size=stack, counters=True, threads=8,
                             intersection=ix)
        for order in (pm.RAY_ORDER_INPUT, pm.RAY_ORDER_COHERENT):
            tp = pm.trace_params(stack_size=stack, intersection=ix, leaf_skipping=skip, ray_order=order, step_cap=4)
            assert_same_hits(pm.hits_to_numpy(ctx.trace(a, O, D, tp)), want, f"{n}")
            cnt = torch.full((n, 4), -7, dtype=torch.int32, device="cuda:0")
            assert_same_hits(pm.hits_to_numpy(ctx.trace(a, O, D, tp, counters=cnt)), want, f"{n} counted")
            assert np.array_equal(cnt.cpu().numpy(), wc)
    assert (want["id"] >= 0).mean() > 0.2


@pytest.mark.parametrize("algo,stack", [("SHORT_STACK", 1), ("SHORT_STACK", 13), ("KD_RESTART", 4)])
@pytest.mark.parametrize("test", ["MOELLER", "WOOP"])
@pytest.mark.parametrize("skip", [0, 1])
def test_canvas_bit_exact(pm, orc, scenes, scene, algo, stack, test, skip):
    import torch
    ctx, ref, tris, normals, col, light, _ = scene
    org, dirs = scenes.pinhole_rays(120, 90, (0.0, 0.0, 3.5), (0.0, 0.0, 0.0), fov_deg=45.0, seed=9)
    a, ix = getattr(pm, algo), getattr(pm, test)
    for bounces in (1, 64):
        got = ctx.trace_canvas(a, dev(torch, org), dev(torch, dirs), [dev(torch, x) for x in normals],
                               dev(torch, col), light, max_bounces=bounces,
                               params=pm.trace_params(stack_size=stack, intersection=ix, leaf_skipping=skip)).cpu().numpy()
        want = orc.trace_canvas(ref, tris, org, dirs, a, normals, col, light, max_bounces=bounces, stack_size=stack,
                                threads=8, intersection=ix)
        assert np.array_equal(got, want), (bounces, np.nonzero((got != want).any(1))[0][:5])


def test_allocation_free_trace(pm, orc, scenes, scene):
    import ctypes as C
    import torch
    ctx, ref, tris = scene[:3]
    org, dirs = scenes.random_rays(30000, seed=4, lo=-2.0, hi=2.0, target_lo=-1.0, target_hi=1.0)
    O, D = dev(torch, org), dev(torch, dirs)
    H = torch.full((30000, 4), -7.0, device="cuda:0")
    for a in (pm.SHORT_STACK, pm.KD_RESTART):
        tp = pm.trace_params(stack_size=8)
        assert ctx._L.pm_trace_noalloc(ctx.h, a, O.data_ptr(), D.data_ptr(), 30000, H.data_ptr(), C.byref(tp), None,
                                       pm._stream_ptr(None)) == 0
        want = orc.trace(ref, tris, org, dirs, a, stack_size=8, threads=8)
        assert_same_hits(pm.hits_to_numpy(H), want, f"{a}")
