"""The coherent order on both sides of the sizes from which a trace uses it
(1,835,008 rays, 524,288 leaf slots): the records are the input order's, and a
sample's are the oracle's; rays without a direction or far outside among them,
and a forest's rays shuffled over its meshes."""
import numpy as np
import pytest

from test_gpu_parity import assert_same_hits, dev, orc_params

pytestmark = pytest.mark.gpu

RAYS = 7 << 18


@pytest.fixture(scope="module")
def torch():
    import torch as T
    assert T.cuda.is_available(), "these tests need the GPU"
    return T


@pytest.fixture(scope="module")
def rays(scenes):
    org, dirs = scenes.random_rays(RAYS, seed=9)
    dirs[:64, :3] = 0.0
    org[64:128, :3] = 1e6
    return org, dirs


@pytest.mark.parametrize("ntris", [60000, 300000])
@pytest.mark.parametrize("algo", ["SHORT_STACK", "KD_RESTART"])
@pytest.mark.parametrize("n", [RAYS - 1, RAYS])
def test_orders_agree(pm, orc, scenes, torch, rays, ntris, algo, n):
    tris = scenes.random_soup(ntris, seed=4, size=0.02)
    org, dirs = rays
    ctx = pm.Context(0)
    bp = pm.build_params("reference")
    ctx.build(*[dev(torch, t) for t in tris], bp)
    assert (ctx.view().num_prim_indices >= 1 << 19) == (ntris == 300000)
    O, D = dev(torch, org[:n]), dev(torch, dirs[:n])
    a = getattr(pm, algo)
    h = [pm.hits_to_numpy(ctx.trace(a, O, D, pm.trace_params(stack_size=8, ray_order=q)))
         for q in (pm.RAY_ORDER_INPUT, pm.RAY_ORDER_COHERENT)]
    assert_same_hits(h[1], h[0], f"{ntris} {algo} {n}")
    pick = np.concatenate([np.arange(128), np.arange(128, n, 1999)])
    ref = orc.build(tris, orc_params(orc, bp))
    want = orc.trace(ref, tris, org[pick], dirs[pick], a, stack_size=8, threads=8)
    assert_same_hits(h[1][pick], want, "oracle")
    ctx.close()


def test_shuffled_forest(pm, orc, scenes, torch, rays):
    off = np.concatenate([[0], np.cumsum([1500 + 211 * (m % 90) for m in range(60)])]).astype(np.int32)
    tris = scenes.random_soup(int(off[-1]), seed=6, size=0.05)
    org, dirs = rays
    mesh = np.random.default_rng(3).integers(0, 60, RAYS).astype(np.int32)
    ctx = pm.Context(0)
    bp = pm.build_params("reference")
    ctx.build_batched(*[dev(torch, t) for t in tris], off, bp)
    assert ctx.view().num_prim_indices >= 1 << 19
    O, D, M = dev(torch, org), dev(torch, dirs), dev(torch, mesh)
    h = [pm.hits_to_numpy(ctx.trace_batched(pm.SHORT_STACK, O, D, M, pm.trace_params(stack_size=8, ray_order=q)))
         for q in (pm.RAY_ORDER_INPUT, pm.RAY_ORDER_COHERENT)]
    assert_same_hits(h[1], h[0], "shuffled")
    pick = np.arange(0, RAYS, 1999)
    ref = orc.build_batched(tris, off, orc_params(orc, bp))
    want = orc.trace_batched(ref, tris, org[pick], dirs[pick], mesh[pick], orc.SHORT_STACK, stack_size=8, threads=8)
    assert_same_hits(h[1][pick], want, "oracle")
    ctx.close()
