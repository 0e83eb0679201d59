"""Forests of very many tiny or empty meshes, alone and beside larger ones:
trees bit-exact against the oracle, and the memory a context takes for them
bounded by what their nodes and refs need (subtrees keep records per node, and
are not for roots without refs)."""
import numpy as np
import pytest

from test_gpu_parity import assert_same_tree, dev, orc_params

pytestmark = pytest.mark.gpu

FORESTS = {
    "one each": [1] * 5000,
    "below a node": [31] * 700,
    "one level": [32, 33, 63] * 200,
    "two levels": [64, 65, 0] * 150,
    "empty beside one": [0] * 3000 + [1200] + [0] * 3000,
    "empty beside many": [700, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0] * 60,
    "small beside large": [3, 1280] * 40,
    "empty": [0] * 4000,
}


@pytest.mark.parametrize("preset", ["reference", "default"])
@pytest.mark.parametrize("name", list(FORESTS))
def test_bit_exact(pm, orc, scenes, name, preset):
    import torch
    off = np.concatenate([[0], np.cumsum(FORESTS[name])]).astype(np.int32)
    n = int(off[-1])
    tris = tuple(t[:n].copy() for t in scenes.random_soup(max(n, 1), seed=3, size=0.03))
    bp = pm.build_params(preset)
    ctx = pm.Context(0)
    P = [dev(torch, t if n else np.zeros((1, 4), np.float32))[:n] for t in tris]
    ref = orc.build_batched(tris, off, orc_params(orc, bp))
    for _ in range(2):
        ctx.build_batched(*P, off, bp)
        assert_same_tree(ctx.tree_arrays(), ref.arrays(), name)
        assert ctx.stats()["upper_levels"] == ref.stats()["upper_levels"]
    ctx.close()


@pytest.mark.parametrize("size", [0, 1])
def test_memory(pm, scenes, size):
    """131,072 meshes: what the level passes take (the DIVIDE split has no
    subtrees), no record beside it"""
    import torch
    M = 1 << 17
    off = (np.arange(M + 1) * size).astype(np.int32)
    P = [dev(torch, t)[:M * size] for t in scenes.random_soup(M, seed=3, size=0.01)]
    taken = []
    for split in (pm.SPLIT_BOX, pm.SPLIT_DIVIDE):
        ctx = pm.Context(0)
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        ctx.build_batched(*P, off, pm.build_params("default", split_method=split))
        torch.cuda.synchronize()
        taken.append(before - torch.cuda.mem_get_info()[0])
        ctx.close()
    assert taken[0] <= taken[1], taken
