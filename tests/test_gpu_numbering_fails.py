"""A subtree numbering whose look-back gives up (its bounded wait set to give
up at once, which a build with more than one tile of nodes then does): the
build reports it with every lower creator, the context holds no tree, and the
next build in it is the oracle's."""
import numpy as np
import pytest

from test_gpu_parity import assert_same_tree, dev, orc_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("preset", ["default", "reference", "balanced"])
@pytest.mark.parametrize("n", [20000, 100000])
def test_status_reaches_the_caller(pm, orc, scenes, monkeypatch, n, preset):
    import torch
    tris = scenes.random_soup(n, seed=2, size=0.02)
    P = [dev(torch, t) for t in tris]
    bp = pm.build_params(preset)
    ref = orc.build(tris, orc_params(orc, bp))
    org, dirs = scenes.random_rays(100, seed=1)
    O, D = dev(torch, org), dev(torch, dirs)
    ctx = pm.Context(0)
    for _ in range(2):
        monkeypatch.setenv("PMKD_LOOKBACK_SPINS", "-1")
        with pytest.raises(pm.PmError) as e:
            ctx.build(*P, bp)
        assert e.value.code == 4
        with pytest.raises(pm.PmError):
            ctx.trace(pm.SHORT_STACK, O, D)
        monkeypatch.delenv("PMKD_LOOKBACK_SPINS")
        ctx.build(*P, bp)
        assert_same_tree(ctx.tree_arrays(), ref.arrays(), preset)
    torch.cuda.synchronize()
    ctx.close()
