"""kd-restart, which goes on from a ring of far children where that is what a
restart would reach: records bit-exact against the oracle's restarts where a
leaf's exit passes several planes at once (rays from far away: the exit's
relative step spans nodes), where rays lie in planes or along axes, and where
a descent from the root would spend its bound of 4096 nodes."""
import numpy as np
import pytest

from test_gpu_parity import assert_same_hits, dev, orc_params

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as T
    assert T.cuda.is_available(), "these tests need the GPU"
    return T


@pytest.mark.parametrize("test", ["MOELLER", "WOOP"])
@pytest.mark.parametrize("away", [0.0, 30.0, 1e3, 1e4, 1e5])
def test_far_rays_bit_exact(pm, orc, scenes, torch, away, test):
    tris = scenes.random_soup(6000, seed=11, size=0.05)
    org, dirs = scenes.random_rays(5000, seed=int(away) + 1)
    org[:, :3] -= np.float32(away) * dirs[:, :3]
    grid = np.arange(500) % 21 / np.float32(20)          # rays along axes, from planes of a grid
    org[:500, :3] = np.stack([grid, np.roll(grid, 7), np.full(500, -1.0 - away)], 1)
    dirs[:500, :3] = (0.0, 0.0, 1.0)
    ctx = pm.Context(0)
    bp = pm.build_params("reference")
    ctx.build(*[dev(torch, t) for t in tris], bp)
    ref = orc.build(tris, orc_params(orc, bp))
    want = orc.trace(ref, tris, org, dirs, orc.KD_RESTART, threads=8, intersection=getattr(pm, test))
    for cap in (0, 3):
        tp = pm.trace_params(step_cap=cap, intersection=getattr(pm, test))
        h = pm.hits_to_numpy(ctx.trace(pm.KD_RESTART, dev(torch, org), dev(torch, dirs), tp))
        assert_same_hits(h, want, f"away {away} cap {cap}")
    ctx.close()


@pytest.mark.parametrize("nodes", [40, 4090, 4096, 4200])
def test_chain_bit_exact(pm, orc, scenes, torch, nodes):
    """an uploaded chain of x splits, one leaf beside each: a leaf's depth is its number"""
    n = 2 * nodes + 1
    x = (np.arange(nodes) + 1) / np.float32(nodes + 1)
    tris = scenes.random_soup(nodes + 1, seed=3, size=0.0)
    at = (np.arange(nodes + 1) + 0.5) / (nodes + 1)       # a triangle across x in the middle of each leaf
    for t, (y, z) in zip(tris, ((-1.0, -1.0), (3.0, -1.0), (-1.0, 3.0))):
        t[:, 0], t[:, 1], t[:, 2] = at, y, z
    keep = np.arange(nodes + 1) % 37 == 36                # most leaves are empty
    keep[nodes] = True
    a = dict(info=np.zeros(n, np.int8), split_pos=np.zeros(n, np.float32),
             aabb_min=np.zeros((n, 4), np.float32), aabb_max=np.zeros((n, 4), np.float32),
             primitive_index=np.zeros(n, np.int32), primitive_bitmap=np.zeros(n, np.int64),
             children=np.zeros((n, 2), np.int32), prim_indices=np.arange(nodes + 1, dtype=np.int32))
    inner = 2 * np.arange(nodes)                          # node 2k splits at x[k]; its leaf is 2k + 1
    a["info"][inner], a["split_pos"][inner] = 1, x
    a["children"][inner] = np.stack([inner + 1, inner + 2], 1)
    leaf = np.append(inner + 1, n - 1)
    a["primitive_index"][leaf] = np.arange(nodes + 1)
    a["primitive_bitmap"][leaf] = keep
    org = np.zeros((96, 4), np.float32)
    dirs = np.zeros((96, 4), np.float32)
    org[:, 0] = np.where(np.arange(96) % 3 == 2, 2.0, -0.5 + np.arange(96) / 64.0)
    org[:, 1:3] = 0.3
    dirs[:, 0] = np.where(np.arange(96) % 3 == 2, -1.0, 1.0)
    dirs[:, 1] = np.arange(96) % 5 * 1e-3
    ctx = pm.Context(0)
    ctx.set_tree(a, *[dev(torch, t) for t in tris], has_boxes=False)
    ref = orc.tree_from_arrays(a)
    want = orc.trace(ref, tris, org, dirs, orc.KD_RESTART, leaf_skipping=False, threads=8)
    for cap in (0, 5):
        h = pm.hits_to_numpy(ctx.trace(pm.KD_RESTART, dev(torch, org), dev(torch, dirs), pm.trace_params(step_cap=cap)))
        assert_same_hits(h, want, f"{nodes} nodes, cap {cap}")
    ctx.close()
