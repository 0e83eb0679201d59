"""Lower levels with forced splits, on both sides of the level size (4,096 nodes)
up to which screen and search are one launch: trees bit-exact against the
oracle, for leaves of one triangle to almost full ones, bitmaps of up to 32 and
of more bits, and a bonus that settles forced and unforced nodes in one level."""
import pytest

from test_gpu_parity import assert_same_tree, dev, orc_params

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as T
    assert T.cuda.is_available(), "these tests need the GPU"
    return T


@pytest.mark.parametrize("leaf_max,bonus,ct", [(1, 1.0, 24.0), (8, 0.8, 24.0), (8, 0.5, 2.0), (30, 0.8, 1.0)])
@pytest.mark.parametrize("lower_size", [32, 64])
@pytest.mark.parametrize("n", [40, 700, 20000, 60000])
def test_forced_levels_bit_exact(pm, orc, scenes, torch, n, lower_size, leaf_max, bonus, ct):
    tris = scenes.random_soup(n, seed=n + leaf_max, size=0.3 / n ** (1 / 3))
    bp = pm.build_params("config", lower_size=lower_size, sah_leaf_max=leaf_max, sah_empty_bonus=bonus,
                         traversal_cost=ct)
    ctx = pm.Context(0)
    ref = orc.build(tris, orc_params(orc, bp))
    for _ in range(2):
        ctx.build(*[dev(torch, t) for t in tris], bp)
        assert_same_tree(ctx.tree_arrays(), ref.arrays(), f"{n} {lower_size} {leaf_max}")
    st, rs = ctx.stats(), ref.stats()
    for k in ("lower_levels", "num_nodes"):
        assert st[k] == rs[k], k
    ctx.close()
