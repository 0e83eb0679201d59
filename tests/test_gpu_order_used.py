"""Traces that are really sorted (more than 2^20 rays on a tree of 2^17 leaf
slots or more): that they are, and that traces on the other side of either
line are not, is seen in the memory the sort's buffers take; records and
counters are the oracle's, with step caps, with the Woop intersection, for
forests with empty meshes and rays of meshes that do not exist, and in a
captured batch."""
import numpy as np
import pytest

from test_gpu_parity import assert_same_hits, dev, orc_params

pytestmark = pytest.mark.gpu

LINE = 1 << 20
SORT_BYTES = 16 * LINE                 # two arrays of keys, two of ray indices


@pytest.fixture(scope="module")
def torch():
    import torch as T
    assert T.cuda.is_available(), "these tests need the GPU"
    return T


@pytest.fixture(scope="module")
def rays(scenes):
    org, dirs = scenes.random_rays(LINE + 1, seed=19)
    dirs[:64, :3] = 0.0
    org[64:128, :3] = 1e6
    return org, dirs


def sorted_by(torch, f) -> bool:
    """whether f(), a context's first call that may sort, took the sort's buffers"""
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    f()
    torch.cuda.synchronize()
    return before - torch.cuda.mem_get_info()[0] >= SORT_BYTES // 2


def coherent(pm, **kw):
    return pm.trace_params(stack_size=8, ray_order=pm.RAY_ORDER_COHERENT, **kw)


@pytest.mark.parametrize("ntris,n,used", [(60000, LINE + 1, False), (120000, LINE, False), (120000, LINE + 1, True)])
def test_lines(pm, orc, scenes, torch, rays, ntris, n, used):
    tris = scenes.random_soup(ntris, seed=4, size=0.02)
    org, dirs = rays[0][:n], rays[1][:n]
    ctx = pm.Context(0)
    bp = pm.build_params("reference")
    ctx.build(*[dev(torch, t) for t in tris], bp)
    assert (ctx.view().num_prim_indices >= 1 << 17) == (ntris == 120000)
    O, D = dev(torch, org), dev(torch, dirs)
    H = torch.empty((n, 4), dtype=torch.float32, device="cuda:0")
    cnt = torch.empty((n, 4), dtype=torch.int32, device="cuda:0")
    assert sorted_by(torch, lambda: ctx.trace(pm.SHORT_STACK, O, D, coherent(pm), out=H)) == used
    ref = orc.build(tris, orc_params(orc, bp))
    for algo in (pm.SHORT_STACK, pm.KD_RESTART):
        want, wc = orc.trace(ref, tris, org, dirs, algo, stack_size=8, counters=True, threads=8)
        for cap in (0, 1, 4):
            ctx.trace(algo, O, D, coherent(pm, step_cap=cap), out=H)
            assert_same_hits(pm.hits_to_numpy(H), want, f"{algo} cap {cap}")
            H.fill_(-7.0)
            ctx.trace(algo, O, D, coherent(pm, step_cap=cap), out=H, counters=cnt)
            assert_same_hits(pm.hits_to_numpy(H), want, f"{algo} cap {cap} counted")
            assert np.array_equal(cnt.cpu().numpy(), wc), (algo, cap)
        woop = [pm.hits_to_numpy(ctx.trace(algo, O, D, pm.trace_params(stack_size=8, intersection=pm.WOOP,
                                                                       ray_order=q)))
                for q in (pm.RAY_ORDER_INPUT, pm.RAY_ORDER_COHERENT)]
        assert_same_hits(woop[1], woop[0], f"{algo} woop")
    ctx.close()


def forest(scenes, rays):
    off = np.concatenate([[0], np.cumsum([0 if m == 3 else 2000 + 211 * (m % 9) for m in range(40)])]).astype(np.int32)
    tris = scenes.random_soup(int(off[-1]), seed=6, size=0.04)
    mesh = np.random.default_rng(3).integers(0, 40, rays[0].shape[0]).astype(np.int32)
    return off, tris, mesh


def test_forest(pm, orc, scenes, torch, rays):
    off, tris, mesh = forest(scenes, rays)
    org, dirs = rays
    mesh[::97] = 40                      # no such mesh
    mesh[1::89] = -1
    mesh[2::83] = 3                      # the empty mesh
    ctx = pm.Context(0)
    bp = pm.build_params("reference")
    ctx.build_batched(*[dev(torch, t) for t in tris], off, bp)
    O, D, M = dev(torch, org), dev(torch, dirs), dev(torch, mesh)
    H = torch.empty((LINE + 1, 4), dtype=torch.float32, device="cuda:0")
    cnt = [torch.empty((LINE + 1, 4), dtype=torch.int32, device="cuda:0") for _ in range(2)]
    assert sorted_by(torch, lambda: ctx.trace_batched(pm.SHORT_STACK, O, D, M, coherent(pm), out=H))
    ref = orc.build_batched(tris, off, orc_params(orc, bp))
    for algo in (pm.SHORT_STACK, pm.KD_RESTART):
        want = orc.trace_batched(ref, tris, org, dirs, mesh, algo, stack_size=8, threads=8)
        for cap in (0, 4):
            for c, q in zip(cnt, (pm.RAY_ORDER_INPUT, pm.RAY_ORDER_COHERENT)):
                H.fill_(-7.0)
                ctx.trace_batched(algo, O, D, M, pm.trace_params(stack_size=8, ray_order=q, step_cap=cap), out=H,
                                  counters=c)
                assert_same_hits(pm.hits_to_numpy(H), want, f"{algo} cap {cap} order {q}")
            assert torch.equal(*cnt), (algo, cap)
    ctx.close()


def test_captured_batch(pm, orc, scenes, torch, rays):
    """every replay sorts; the program's own work on the same arrays between them"""
    off, tris, mesh = forest(scenes, rays)
    org, dirs = rays
    bp = pm.build_params("reference")
    P = [dev(torch, t) for t in tris]
    O, D, M = dev(torch, org), dev(torch, dirs), dev(torch, mesh)
    H = torch.empty((LINE + 1, 4), dtype=torch.float32, device="cuda:0")
    want = orc.trace_batched(orc.build_batched(tris, off, orc_params(orc, bp)), tris, org, dirs, mesh,
                             orc.SHORT_STACK, stack_size=8, threads=8)
    ctx = pm.Context(0)
    ctx.batch_graph_capture(*P, off, O, D, M, H, pm.SHORT_STACK, bp, pm.trace_params(stack_size=8))
    assert sorted_by(torch, lambda: ctx.batch_graph_capture(*P, off, O, D, M, H, pm.SHORT_STACK, bp, coherent(pm)))
    for i in range(4):
        H.zero_()
        torch.cuda.synchronize()
        ctx.batch_graph_launch()
        assert ctx.batch_graph_status() == 0
        assert_same_hits(pm.hits_to_numpy(H), want, f"replay {i}")
        if i == 1:                       # an eager, sorted trace in the same context
            H.fill_(-7.0)
            ctx.trace_batched(pm.SHORT_STACK, O, D, M, coherent(pm), out=H)
            assert_same_hits(pm.hits_to_numpy(H), want, "eager")
    ctx.close()


def test_autotune_keeps_no_order_that_is_not_used(pm, scenes, torch):
    """a trace too small, or of too small a tree, to be sorted times the input
    order twice: noise between the two never picks the coherent order"""
    tris = scenes.random_soup(4000, seed=4, size=0.02)
    org, dirs = scenes.random_rays(1 << 17, seed=5)
    ctx = pm.Context(0)
    P = [dev(torch, t) for t in tris]
    O, D = dev(torch, org), dev(torch, dirs)
    got = [ctx.autotune(*P, O, D, base=pm.build_params("reference"), reps=1)["ray_order"] for _ in range(6)]
    assert got == [pm.RAY_ORDER_INPUT] * 6
    ctx.close()
