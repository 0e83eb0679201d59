"""Small builds, whose upper stage ends in subtrees built a block each: trees
bit-exact against the oracle at the sizes where a node goes to the other kind
of block or to the level passes, from the roots on and after some levels, for
forests with empty meshes, the options that change what a node's record holds,
and scenes whose refs outgrow a subtree's room (the level passes then build
them)."""
import numpy as np
import pytest

from test_gpu_parity import assert_same_tree, dev, orc_params

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as T
    assert T.cuda.is_available(), "these tests need the GPU"
    return T


@pytest.fixture(scope="module")
def ctx(pm, torch):
    c = pm.Context(0)
    yield c
    c.close()


OPTIONS = {
    "reference": dict(preset="reference"),
    "default": dict(preset="default"),
    "balanced": dict(preset="balanced"),
    "no_empty_space": dict(preset="reference", empty_space_splitting=0),
    "no_boxes": dict(preset="default", empty_space_splitting=0, propagate_aabbs=0),
    "lower16": dict(preset="reference", lower_size=16),
    "lower64_chunk128": dict(preset="reference", lower_size=64, chunk_size=128),
}


def check(pm, orc, torch, ctx, tris, bp, off=None, label=""):
    P = [dev(torch, t) for t in tris]
    if off is None:
        ctx.build(*P, bp)
        ref = orc.build(tris, orc_params(orc, bp))
    else:
        ctx.build_batched(*P, off, bp)
        ref = orc.build_batched(tris, off, orc_params(orc, bp))
    assert_same_tree(ctx.tree_arrays(), ref.arrays(), label)
    st, rs = ctx.stats(), ref.stats()
    for k in ("upper_levels", "lower_levels", "num_nodes", "num_prim_indices"):
        assert st[k] == rs[k], (label, k)


@pytest.mark.parametrize("name", list(OPTIONS))
@pytest.mark.parametrize("n", [1, 31, 64, 65, 128, 129, 512, 513, 1280, 1281, 2600, 40000])
def test_sizes(pm, orc, scenes, torch, ctx, n, name):
    opt = dict(OPTIONS[name])
    tris = scenes.random_soup(n, seed=n, size=0.4 / max(1.0, n ** (1 / 3)))
    check(pm, orc, torch, ctx, tris, pm.build_params(opt.pop("preset"), **opt), label=f"{name} {n}")


@pytest.mark.parametrize("n,size", [(600, 0.9), (1280, 0.6), (4000, 0.5), (600, 0.3), (1280, 0.2)])
def test_refs_that_outgrow_a_subtree(pm, orc, scenes, torch, ctx, n, size):
    """large triangles: most refs straddle every plane; where the oracle gives
    the build up, so does the GPU, with the same words"""
    tris = scenes.random_soup(n, seed=n, size=size)
    small = tuple(t[:200].copy() for t in tris)
    bp = pm.build_params("default")
    for t in (tris, small, tris, small):
        try:
            orc.build(t, orc_params(orc, bp))
        except RuntimeError as e:
            with pytest.raises(pm.PmError) as g:
                ctx.build(*[dev(torch, x) for x in t], bp)
            assert str(e).split(": ", 1)[1] in str(g.value)
        else:
            check(pm, orc, torch, ctx, t, bp, label=f"{n} {size}")


@pytest.mark.parametrize("name", ["reference", "no_boxes"])
@pytest.mark.parametrize("sizes", [[0, 512, 513, 0, 1], [1280, 40, 700, 0], [5000, 0, 300, 31, 1281], [64] * 300])
def test_forests(pm, orc, scenes, torch, ctx, sizes, name):
    opt = dict(OPTIONS[name])
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    tris = scenes.random_soup(int(off[-1]), seed=len(sizes), size=0.05)
    check(pm, orc, torch, ctx, tris, pm.build_params(opt.pop("preset"), **opt), off, f"{name} {sizes[:6]}")
