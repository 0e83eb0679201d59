"""A context's first build, at sizes on both sides of the lines where its
buffers are sized and where small levels are launched ahead of their state:
trees bit-exact against the oracle, a second, larger and a smaller build in
the same context too, with levels counted as the oracle counts them."""
import numpy as np
import pytest

from test_gpu_parity import assert_same_tree, dev, orc_params

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as T
    assert T.cuda.is_available(), "these tests need the GPU"
    return T


@pytest.mark.parametrize("n", [0, 1, 40, 3000, 16385, 60000, 131072, 131073, 200000])
@pytest.mark.parametrize("preset", ["reference", "config", "balanced", "default"])
def test_first_build_bit_exact(pm, orc, scenes, torch, n, preset):
    if preset != "reference" and n > 20000:
        pytest.skip("sizes beyond the lower stage's lines are covered by one preset")
    ctx = pm.Context(0)
    bp = pm.build_params(preset)
    for m in (n, n + n // 2 + 7, n // 3):
        tris = scenes.random_soup(max(m, 1), seed=m % 97, size=0.6 / max(1.0, m ** (1 / 3)))
        tris = tuple(t[:m].copy() for t in tris)
        P = [dev(torch, t if m else np.zeros((1, 4), np.float32))[:m] for t in tris]
        ctx.build(*P, bp)
        ref = orc.build(tris, orc_params(orc, bp))
        assert_same_tree(ctx.tree_arrays(), ref.arrays(), f"{preset} {m}")
        st, rs = ctx.stats(), ref.stats()
        for k in ("upper_levels", "lower_levels", "num_nodes", "num_prim_indices"):
            assert st[k] == rs[k], (k, m)
    ctx.close()


def test_build_after_capture_keeps_the_graph(pm, orc, scenes, torch):
    """an eager build of the captured size leaves the captured batch's buffers alone"""
    tris = scenes.random_soup(9000, seed=5, size=0.05)
    P = [dev(torch, t) for t in tris]
    bp = pm.build_params("reference")
    ctx = pm.Context(0)
    off = np.array([0, 4000, 9000], np.int32)
    ctx.batch_graph_capture(*P, off, None, None, None, None, build=bp)
    ref = orc.build_batched(tris, off, orc_params(orc, bp))
    for _ in range(3):
        ctx.build_batched(*P, off, bp)
        assert_same_tree(ctx.tree_arrays(), ref.arrays(), "eager")
        ctx.batch_graph_launch()
        assert ctx.batch_graph_status() == 0
        assert_same_tree(ctx.tree_arrays(), ref.arrays(), "replay")
    ctx.close()
