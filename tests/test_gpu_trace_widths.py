"""Tree tracers at the ray counts where a launch changes the number of rays a
wave holds (powers of two around the device's resident waves, one ray, odd
remainders), at leaf bitmaps on both sides of 32 slots, and on trees whose
root is a leaf.  Bar: bit-exact hits and per-ray counters against the oracle.
"""
import numpy as np
import pytest

from test_gpu_parity import assert_same_hits, dev, orc_params

pytestmark = pytest.mark.gpu

# around 4 x 256 CUs x 4..6 blocks x {1, 2, 4, ... 64} rays
COUNTS = [1, 2, 63, 64, 65, 4095, 4097, 6143, 6145, 12289, 24577, 49153, 98303, 98305, 196609, 393217]


@pytest.fixture(scope="module")
def torch():
    import torch as T
    assert T.cuda.is_available(), "these tests need the GPU"
    return T


@pytest.mark.parametrize("lower_size", [32, 33, 48])
@pytest.mark.parametrize("algo,test", [("SHORT_STACK", "MOELLER"), ("KD_RESTART", "MOELLER"),
                                       ("SHORT_STACK", "WOOP"), ("KD_RESTART", "WOOP")])
def test_ray_counts_bit_exact(pm, orc, scenes, torch, lower_size, algo, test):
    tris = scenes.random_soup(1500, seed=lower_size, size=0.15)
    org, dirs = scenes.random_rays(max(COUNTS), seed=17)
    bp = pm.build_params("reference", lower_size=lower_size)
    ctx = pm.Context(0)
    ctx.build(*[dev(torch, t) for t in tris], bp)
    ref = orc.build(tris, orc_params(orc, bp))
    a = getattr(pm, algo)
    want, wc = orc.trace(ref, tris, org, dirs, a, stack_size=4, counters=True, threads=8,
                         intersection=getattr(pm, test))
    O, D = dev(torch, org), dev(torch, dirs)
    for n in COUNTS:
        for cap in (0, 4):
            tp = pm.trace_params(stack_size=4, intersection=getattr(pm, test), step_cap=cap)
            h = pm.hits_to_numpy(ctx.trace(a, O[:n].contiguous(), D[:n].contiguous(), tp))
            assert_same_hits(h, want[:n], f"{n} rays, cap {cap}")
        cnt = torch.zeros((n, 4), dtype=torch.int32, device="cuda:0")
        h = pm.hits_to_numpy(ctx.trace(a, O[:n].contiguous(), D[:n].contiguous(), tp, counters=cnt))
        assert_same_hits(h, want[:n], f"{n} rays, counted")
        assert np.array_equal(cnt.cpu().numpy(), wc[:n]), n
    ctx.close()


@pytest.mark.parametrize("ntris", [1, 31, 40, 64])
@pytest.mark.parametrize("boxes", [True, False])
def test_root_leaf_bit_exact(pm, orc, scenes, torch, ntris, boxes):
    """an uploaded tree that is one leaf, with and without boxes"""
    tris = scenes.random_soup(ntris, seed=3, size=0.5)
    org, dirs = scenes.random_rays(777, seed=5)
    v = np.concatenate([t[:, :3] for t in tris])
    a = dict(info=np.zeros(1, np.int8), split_pos=np.zeros(1, np.float32),
             aabb_min=np.append(v.min(0), 0).astype(np.float32)[None],
             aabb_max=np.append(v.max(0), 0).astype(np.float32)[None],
             primitive_index=np.zeros(1, np.int32), primitive_bitmap=np.array([(1 << ntris) - 1], np.uint64).view(np.int64),
             children=np.zeros((1, 2), np.int32), prim_indices=np.arange(ntris, dtype=np.int32))
    ctx = pm.Context(0)
    ctx.set_tree(a, *[dev(torch, t) for t in tris], has_boxes=boxes)
    ref = orc.tree_from_arrays(a)
    for algo in (pm.SHORT_STACK, pm.KD_RESTART):
        want = orc.trace(ref, tris, org, dirs, algo, leaf_skipping=boxes)
        h = pm.hits_to_numpy(ctx.trace(algo, dev(torch, org), dev(torch, dirs), pm.trace_params()))
        assert_same_hits(h, want, f"{ntris} triangles, algo {algo}")
    ctx.close()


@pytest.mark.parametrize("algo,stack", [("SHORT_STACK", 1), ("SHORT_STACK", 5), ("SHORT_STACK", 13), ("KD_RESTART", 4)])
@pytest.mark.parametrize("woop", [False, True])
def test_canvas_ray_counts_bit_exact(pm, orc, scenes, torch, algo, stack, woop):
    """canvas bytes at ray counts that fill part of a wave, one and many, and at
    bounce limits met by some rays"""
    from test_gpu_extras import shading_scene
    tris, _, normals, col, light = shading_scene(scenes)
    org, dirs = scenes.pinhole_rays(300, 240, (0.0, 0.0, 3.5), (0.0, 0.0, 0.0), fov_deg=45.0, seed=9)
    test = pm.WOOP if woop else pm.MOELLER
    ctx = pm.Context(0)
    ctx.build(*[dev(torch, t) for t in tris], pm.build_params("reference"))
    ref = orc.build(tris, orc.build_params("reference"))
    a = getattr(pm, algo)
    N, C = [dev(torch, x) for x in normals], dev(torch, col)
    for n, bounces in ((1, 64), (63, 64), (65, 1), (7001, 3), (72000, 64), (72000, 2)):
        o, d = org[-n:].copy(), dirs[-n:].copy()
        got = ctx.trace_canvas(a, dev(torch, o), dev(torch, d), N, C, light, max_bounces=bounces,
                               params=pm.trace_params(stack_size=stack, intersection=test)).cpu().numpy()
        want = orc.trace_canvas(ref, tris, o, d, a, normals, col, light, max_bounces=bounces, stack_size=stack,
                                threads=8, intersection=test)
        assert np.array_equal(got, want), (n, bounces, np.nonzero((got != want).any(1))[0][:5])
    ctx.close()
